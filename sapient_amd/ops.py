"""Device-resident op calls on torch tensors, through the C ABI.

torch supplies device memory and the current HIP stream; every op runs in the
HIP kernels of ``libsapient_hip.so``. Inputs must be contiguous device
tensors. Errors from the ABI raise :class:`SapientHipError`.

The checks and calls are native (``binding/torch_ops.cpp``): the host's part of a
call, beside the launch itself, is what a decode step's small kernels wait for.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _lib
from ._lib import check, lib

_DT = {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def dtype_code(t: torch.dtype) -> int:
    try:
        return _DT[t]
    except KeyError:
        raise TypeError(f"unsupported dtype {t}") from None


class _Unloaded:
    """Stands for the native module until its first use; loading fails loudly if it has not been built."""

    def __getattr__(self, name):
        global _native
        lib()  # the library first, with its own message when it is missing
        try:
            from . import _torch_ops
        except ImportError as e:
            raise RuntimeError(f"_torch_ops.so is not built or does not load ({e}); run `python -m sapient_amd.build`") from e
        built = (_torch_ops.torch_version, _torch_ops.abi_version)
        if built != (str(torch.__version__), lib().sph_abi_version()):
            raise RuntimeError(f"_torch_ops.so is built for torch {built[0]} and ABI {built[1]}, not torch {torch.__version__} "
                               f"and ABI {lib().sph_abi_version()}; run `python -m sapient_amd.build`")
        _torch_ops.set_check(check)
        _native = _torch_ops
        return getattr(_torch_ops, name)


_native = _Unloaded()


def init(device: Optional[torch.device] = None) -> None:
    """Per-device set-up (GELU tables); optional, done lazily otherwise."""
    with torch.cuda.device(device or torch.cuda.current_device()):
        check(lib().sph_init(torch.cuda.current_stream().cuda_stream), "init")


def rms_norm(x: torch.Tensor, weight: Optional[torch.Tensor], eps: float,
             out: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """RMSNorm over the last dim (layernorm.rs:75-106). out_dtype: f32 (the
    reference's output type) or x's dtype; defaults to x's dtype."""
    return _native.rms_norm(x, weight, eps, out, out_dtype)


def layer_norm(x: torch.Tensor, weight: Optional[torch.Tensor], bias: Optional[torch.Tensor], eps: float,
               out: Optional[torch.Tensor] = None, out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """LayerNorm over the last dim (layernorm.rs:17-69, axis -1; common.rs:575-577).
    weight and bias are optional and share one dtype (f32 or x's)."""
    return _native.layer_norm(x, weight, bias, eps, out, out_dtype)


def add_rms_norm(x: torch.Tensor, residual: torch.Tensor, weight: Optional[torch.Tensor], eps: float,
                 out: Optional[torch.Tensor] = None,
                 out_dtype: Optional[torch.dtype] = None,
                 sum_out: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Fused add (llama.rs:508) + rms_norm (llama.rs:515). `residual` is
    updated in place with x + residual, or, given `sum_out`, left as it is while
    the sum goes to `sum_out` (as the trait's add returns a new tensor); returns
    (normed, sum)."""
    return _native.add_rms_norm(x, residual, weight, eps, out, out_dtype, sum_out)


def add(a: torch.Tensor, b: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """a + b with the reference's length-1 broadcast (elementwise.rs:27-63)."""
    return _native.add(a, b, out)


def mul(a: torch.Tensor, b: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """a * b with the reference's length-1 broadcast (elementwise.rs:27-57, :67-69)."""
    return _native.mul(a, b, out)


def silu(x: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    return _native.silu(x, out)


def swiglu(gate: torch.Tensor, up: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """silu(gate) * up, fused (llama.rs:531-532)."""
    return _native.swiglu(gate, up, out)


def gelu_tanh(x: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """GELU tanh form (elementwise.rs:120-127), bit-exact with the reference."""
    return _native.gelu_tanh(x, out)


def gelu_erf(x: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """GELU erf form (elementwise.rs:135-138, :163-174), bit-exact with the reference."""
    return _native.gelu_erf(x, out)


def add_bias(y: torch.Tensor, bias: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """y + bias over the last dim (common.rs:556-569); bias may be f32 or a half type."""
    return _native.add_bias(y, bias, out)


def rope_(q: torch.Tensor, k: Optional[torch.Tensor], positions: torch.Tensor, base: float,
          rotary_dim: Optional[int] = None, pos_scale: float = 1.0, interleaved: bool = False) -> None:
    """RoPE in place on q [B, Hq, S, D] and optionally k [B, Hk, S, D]
    (rope.rs:18-62 / :83-136). positions: int32 device tensor [S]."""
    _native.rope_(q, k, positions, base, rotary_dim, pos_scale, interleaved)


def rope_table(positions, rotary_dim: int, base: float, pos_scale: float = 1.0, n: Optional[int] = None):
    """Host cos / sin tables [n, rotary_dim / 2] (float32 numpy) of the RoPE angles of `positions` (a
    sequence of ints, row r for positions[r]) or, with positions None, of 0 .. n - 1 — the layout of
    rope_cos_sin_cache (rope.rs:140-153), evaluated by the library with the host libm (rope.rs:48-50)."""
    import numpy as np
    if positions is None:
        if n is None:
            raise ValueError("give positions or n")
        pos, count = None, int(n)
    else:
        pos = np.ascontiguousarray(positions, dtype=np.int64)
        count = pos.size
    if rotary_dim <= 0 or rotary_dim % 2:
        raise ValueError("rotary_dim must be even and positive")
    cs = np.empty((count, rotary_dim // 2), np.float32)
    sn = np.empty((count, rotary_dim // 2), np.float32)
    check(lib().sph_rope_table(None if pos is None else pos.ctypes.data, count, rotary_dim, float(base),
                               float(pos_scale), cs.ctypes.data, sn.ctypes.data), "rope_table")
    return cs, sn


def rope_cached_(q: torch.Tensor, k: Optional[torch.Tensor], cos_table: torch.Tensor, sin_table: torch.Tensor,
                 positions: Optional[torch.Tensor] = None, rotary_dim: Optional[int] = None,
                 interleaved: bool = False, bad_pos_flag: Optional[torch.Tensor] = None) -> None:
    """RoPE in place on q [B, Hq, S, D] (and k) with the angles read from device f32 tables
    [rows, rotary_dim / 2]: token s uses row positions[s] (int32 device tensor [S]), or row s when
    positions is None."""
    _native.rope_cached_(q, k, cos_table, sin_table, positions, rotary_dim, interleaved, bad_pos_flag)


def rope_host_positions_(q: torch.Tensor, k: Optional[torch.Tensor], positions, base: float,
                         rotary_dim: Optional[int] = None, pos_scale: float = 1.0, interleaved: bool = False) -> None:
    """The trait path's RoPE (apply_rope_positions, backend.rs:84): positions on the host, angles evaluated
    on the host for exactly those positions (rope_table), uploaded, and applied by rope_cached_."""
    rd = q.shape[-1] if rotary_dim is None else rotary_dim
    cs, sn = rope_table(positions, rd, base, pos_scale)
    cs_d = torch.from_numpy(cs).to(q.device, non_blocking=False)
    sn_d = torch.from_numpy(sn).to(q.device, non_blocking=False)
    rope_cached_(q, k, cs_d, sn_d, None, rd, interleaved)


def embed(table: torch.Tensor, table_dtype: int, vocab: int, hidden: int, ids: torch.Tensor,
          out: Optional[torch.Tensor] = None, bad_id_flag: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Row gather + dequant of a raw GGUF table (common.rs:164-217) into f32
    [n_ids, hidden]. `table` holds the raw tensor bytes (any dtype, contiguous);
    ids: int32/uint32 device tensor (ids are read as uint32)."""
    return _native.embed(table, table_dtype, vocab, hidden, ids, out, bad_id_flag)


def transpose_heads(x: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """[outer, inner, head_dim] -> [inner, outer, head_dim] (resident.rs:420-458), bit for bit."""
    return _native.transpose_heads(x, out)


def kv_append(src: torch.Tensor, cache: torch.Tensor, pos: int) -> None:
    """Write src [n_kv, seq, head_dim] into cache [n_kv, max_seq, head_dim] at
    positions pos..pos+seq, converted to the cache's dtype (resident.rs:645-711).
    A uint8 cache [n_kv, max_seq, head_dim / 32 * 34] is a Q8_0 cache, quantized
    on append (common.rs:336-348, :449-508)."""
    _native.kv_append(src, cache, pos)


def kv_cache_update(src: torch.Tensor, cache: torch.Tensor, cur_len: int) -> int:
    """Append src [n_kv, seq, head_dim] after the cur_len valid rows of each head
    of cache [n_kv, max_seq, row], sliding the window left first when the rows
    would not fit, and return the new valid length min(cur_len + seq, max_seq):
    common::update_kv_cache / update_kv_cache_q8 (common.rs:355-434, :449-508).
    Cache dtypes as kv_append (a uint8 cache is Q8_0)."""
    return _native.kv_cache_update(src, cache, cur_len)


def kv_cache_update_into(src: torch.Tensor, cache: torch.Tensor, out: torch.Tensor, cur_len: int) -> int:
    """kv_cache_update into a second cache: `out` (cache's shape and dtype) receives rows [0, new_len) of the
    updated cache — cache's kept rows moved once, then src — and `cache` is only read. The caller then uses
    `out` as its cache (common.rs:355-434, :449-508 take the cache as &mut Tensor). Returns new_len."""
    return _native.kv_cache_update_into(src, cache, out, cur_len)


def rope_kv_append(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, positions: torch.Tensor, base: float,
                   kcache: torch.Tensor, vcache: torch.Tensor, pos_scale: float = 1.0, interleaved: bool = False,
                   bad_pos_flag: Optional[torch.Tensor] = None, bq: Optional[torch.Tensor] = None,
                   bk: Optional[torch.Tensor] = None, bv: Optional[torch.Tensor] = None) -> None:
    """Fused decode step: optional q/k/v biases, RoPE on q in place; rotated k and v written to
    the caches at rows positions[s] (wgpu_engine.rs:397-432). q [Hq, S, D], k/v [Hkv, S, D],
    caches [Hkv, max_seq, D], biases [Hq·D] / [Hkv·D] of one dtype."""
    _native.rope_kv_append(q, k, v, positions, base, kcache, vcache, pos_scale, interleaved, bad_pos_flag,
                           bq, bk, bv)


def rope_kv_append_tokens(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, positions: torch.Tensor, base: float,
                          kcache: torch.Tensor, vcache: torch.Tensor, pos_scale: float = 1.0,
                          interleaved: bool = False, bad_pos_flag: Optional[torch.Tensor] = None,
                          bq: Optional[torch.Tensor] = None, bk: Optional[torch.Tensor] = None,
                          bv: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The fused step on a chunk in the projections' layout: q [S, Hq, D], k/v [S, Hkv, D] token-major
    (read only); returns the rotated q heads-major [Hq, S, D] (wgpu_engine.rs:525-573 without the
    transposes); k and v rows go to the caches as in rope_kv_append."""
    return _native.rope_kv_append_tokens(q, k, v, positions, base, kcache, vcache, pos_scale, interleaved,
                                         bad_pos_flag, bq, bk, bv, out)