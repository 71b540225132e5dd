"""GPU parity where no 16-byte vector fits: widths that the vector does not divide and tensors that
are only element-aligned, at the edges of the launch shapes (a run, a wave, the widest row held in
registers, the cached / non-temporal bound).

Norms: the fixed tests' bars (f32 <= 1e-5 relative, halves <= 1 ulp, LayerNorm the summation-order
bound; the residual sum bit for bit). Reference: layernorm.rs:17-69, :75-106.
"""
import numpy as np
import pytest
import torch

from helpers import (assert_bits16_equal, assert_bits_equal, assert_ulp16, check_layer_norm, max_rel, narrow_bits,
                     to_np, widen)

import sapient_amd.ops as ops

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.float16, torch.bfloat16]
DT_ID = lambda d: str(d).split(".")[-1]


def _gen(shape, seed, dev, dtype, off=0, std=1.0, mean=0.0):
    """Seeded values `off` elements into an allocation, so element-aligned only when off is odd."""
    n = int(np.prod(shape))
    g = torch.Generator(device=dev).manual_seed(seed)
    return (torch.randn(n + off, generator=g, device=dev) * std + mean).to(dtype)[off:].view(shape)


def _same(got, want32, dtype, orc, what):
    if dtype == torch.float32:
        assert_bits_equal(to_np(got), want32, what)
    else:
        assert_bits16_equal(to_np(got), narrow_bits(want32, dtype, orc), what)


def _close(got, want32, orc, what):
    if got.dtype == torch.float32:
        assert max_rel(to_np(got), want32) <= 1e-5, what
    else:
        assert_ulp16(to_np(got), narrow_bits(want32, got.dtype, orc), got.dtype, 1, what)


# One element; a run of 8 / 4 and one either side; one and two waves' spans; 16 waves at one and at two
# runs per lane (f32 4096 / 8192, halves 8192 / 16384) and one past them; 65536 x 515: past the cached bound; narrow
# rows both few (the kernel of element accesses) and more than 3072.
@pytest.mark.parametrize("dtype", DTYPES, ids=DT_ID)
@pytest.mark.parametrize("rows,dim,off", [(3, 1, 0), (5, 7, 0), (5, 9, 1), (4, 255, 0), (4, 257, 0), (3, 513, 3),
                                          (700, 1025, 0), (2100, 1023, 0), (5, 4095, 0), (5, 4097, 1), (3, 8191, 0),
                                          (3, 8193, 0), (2, 16383, 0), (2, 16385, 0), (65536, 515, 0), (9, 512, 1),
                                          (3073, 1, 0), (3073, 7, 1), (3073, 9, 0), (3073, 255, 1), (3073, 257, 0)])
def test_ragged_norms(dev, orc, dtype, rows, dim, off):
    print(f"case ragged norms {dtype} {rows}x{dim} offset {off}", flush=True)
    x = _gen((rows, dim), 1, dev, dtype, off, mean=0.25)
    r = _gen((rows, dim), 2, dev, dtype, off)
    for wdt in {torch.float32, dtype}:
        w, b = _gen((dim,), 3, dev, wdt, off, 0.1, 1.0), _gen((dim,), 4, dev, wdt, 0, 0.1)
        w32, b32 = widen(w, orc), widen(b, orc)
        y = ops.rms_norm(x, w, 1e-5)
        ln = ops.layer_norm(x, w, b, 1e-5, out_dtype=torch.float32)
        r2 = r.clone()
        ya, r2 = ops.add_rms_norm(x, r2, w, 1e-5)
        yt, st = ops.add_rms_norm(x, r, w, 1e-5, sum_out=torch.empty_like(r))
        torch.cuda.synchronize()
        assert torch.equal(st.view(torch.uint8), r2.view(torch.uint8))
        # The rows at both ends and in the middle against the oracle: rows are independent.
        pick = sorted({i for i in (0, 1, rows // 2, rows - 2, rows - 1) if 0 <= i < rows})
        x32, r32 = widen(x[pick], orc), widen(r[pick], orc)
        _close(y[pick], orc.rms_norm(x32, w32, 1e-5), orc, "rms_norm")
        check_layer_norm(ln[pick], orc.layer_norm(x32, w32, b32, 1e-5), x32, w32, b32, orc, "layer_norm")
        ref, ref_r = orc.add_rms_norm(x32, r32, w32, 1e-5)
        _same(r2[pick], ref_r, dtype, orc, "residual")
        _close(ya[pick], ref, orc, "add_rms_norm")
        _close(yt[pick], ref, orc, "add_rms_norm_to")
        # No row is skipped: every row's RMS is 1 where the weight is 1.
        u = ops.rms_norm(x, None, 0.0, out_dtype=torch.float32)
        assert (u.square().mean(-1) - 1).abs().max().item() < 1e-4


# Element-wise launches around every bound of their dispatch (2^18 .. 2^21 elements, 2^20 vectors, 16 and 128 MB of
# traffic), a few elements past each (short last runs) and at odd addresses. Every element against the same op over
# pieces of at most 2^18 elements at aligned addresses, which take the one-element kernel (f32 SiLU and SwiGLU pieces
# below 2048 elements, adds and products in f32 as well: runs); the first and last elements, where a launch's short runs
# are, against the oracle; adds and products against torch throughout.
def _pieces(fn, *xs):
    step = 1 << 18
    n = max(x.numel() for x in xs)
    cut = lambda x, i: x if x.numel() == 1 else x.reshape(-1)[i:i + step].clone()
    return torch.cat([fn(*[cut(x, i) for x in xs]).reshape(-1) for i in range(0, n, step)])


@pytest.mark.parametrize("dtype", DTYPES, ids=DT_ID)
@pytest.mark.parametrize("n", [1, 2049, (1 << 18) + 1, (1 << 19) - 3, (1 << 19) + 8, (1 << 20) + 5, (1 << 21) + 2,
                               (1 << 22) + 4, (1 << 22) + 7, (1 << 23) + 1, 23_000_000])
@pytest.mark.parametrize("off", [0, 1])
def test_elementwise_launch_bounds(dev, orc, dtype, n, off):
    print(f"case elementwise {dtype} n {n} offset {off}", flush=True)
    x, u = _gen((n,), 11, dev, dtype, off, 2.0), _gen((n,), 12, dev, dtype, off, 2.0)
    one = _gen((1,), 13, dev, dtype)
    same = lambda a, b, what: torch.equal(a.reshape(-1).view(torch.uint8), b.reshape(-1).view(torch.uint8)) or pytest.fail(what)
    for name, fn in (("silu", ops.silu), ("gelu_tanh", ops.gelu_tanh), ("gelu_erf", ops.gelu_erf)):
        same(fn(x), _pieces(fn, x), name)
    for name, fn in (("swiglu", ops.swiglu), ("add", ops.add), ("mul", ops.mul)):
        same(fn(x, u), _pieces(fn, x, u), name)
    if n > 1:
        same(ops.add(x, one), _pieces(ops.add, x, one), "add scalar")
        same(ops.mul(one, x), _pieces(ops.mul, one, x), "scalar mul")
    for fn, tf in ((ops.add, torch.add), (ops.mul, torch.mul)):  # in f32, rounded once
        same(fn(x, u), tf(x.float(), u.float()).to(dtype), "against torch")
        same(fn(x, one), tf(x.float(), one.float()).to(dtype), "by a scalar, against torch")
    ends = torch.cat([x[:1100], x[-1100:]]), torch.cat([u[:1100], u[-1100:]])
    x32, u32 = (widen(t, orc) for t in ends)
    pick = lambda y: torch.cat([y[:1100], y[-1100:]])
    _same(pick(ops.silu(x)), orc.silu(x32), dtype, orc, "silu ends")
    _same(pick(ops.swiglu(x, u)), orc.swiglu(x32, u32), dtype, orc, "swiglu ends")
    _same(pick(ops.gelu_tanh(x)), orc.gelu(x32), dtype, orc, "gelu_tanh ends")
    _same(pick(ops.gelu_erf(x)), orc.gelu_erf(x32), dtype, orc, "gelu_erf ends")
    want = _pieces(ops.swiglu, x, u)
    assert ops.swiglu(x, u, out=x) is x  # in place
    same(x, want, "swiglu in place")


# Half GELU at the bounds of its table kernel's trips on a 256-CU device (2^21, 2^22, 2^23 elements), and of the
# element kernel's sizes (2^18; 9 x 2^18 at unaligned addresses).
@pytest.mark.parametrize("dtype", DTYPES[1:], ids=DT_ID)
@pytest.mark.parametrize("n", [(1 << 18) + 1, (9 << 18) + 1, 1 << 21, (1 << 21) + 1, (1 << 22) - 7, (1 << 22) + 8, 1 << 23, (1 << 23) + 9])
def test_half_gelu_trip_bounds(dev, dtype, n):
    print(f"case half gelu {dtype} n {n}", flush=True)
    for off in (0, 3):
        x = _gen((n,), 14, dev, dtype, off, 2.0)
        for fn in (ops.gelu_tanh, ops.gelu_erf):
            want = _pieces(fn, x)
            assert torch.equal(fn(x).view(torch.uint8), want.view(torch.uint8))
        y = x.clone()
        assert ops.gelu_erf(y, out=y) is y  # in place
        assert torch.equal(y.view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("dtype", DTYPES, ids=DT_ID)
@pytest.mark.parametrize("rows,n,off", [(3, 1, 0), (5, 7, 1), (1, 2049, 0), (1100, 1001, 0), (1100, 1001, 1), (1048, 1000, 1),
                                        (2049, 2048, 3), (700, 4097, 0), (4000, 9001, 0), (1100000, 1, 0), (400001, 3, 1),
                                        (200000, 7, 0), (150000, 9, 1), (5000, 256, 1), (5000, 257, 0), (5000, 289, 0)])
def test_ragged_bias(dev, orc, dtype, rows, n, off):
    print(f"case ragged bias {dtype} {rows}x{n} offset {off}", flush=True)
    y = _gen((rows, n), 21, dev, dtype, off)
    for bdt in {torch.float32, torch.float16, dtype}:
        b = _gen((n,), 22, dev, bdt, off)
        got = ops.add_bias(y, b)
        # y + b in f32, rounded once
        assert torch.equal(got.view(torch.uint8), (y.float() + b.float()).to(dtype).view(torch.uint8))


# Every length of a short last run (a run is 4 or 8 elements), alone in its row and after full runs; and what
# lies past the tensor's end is left alone.
@pytest.mark.parametrize("dtype", DTYPES, ids=DT_ID)
@pytest.mark.parametrize("k", range(1, 8))
def test_short_runs(dev, orc, dtype, k):
    for dim, off in ((k, 0), (8 + k, 1), (248 + k, 0)):
        test_ragged_norms(dev, orc, dtype, 3073, dim, off)  # (fewer narrow rows take the element kernel)
    print(f"case short runs {dtype} {k}", flush=True)
    n = (1 << 21) + k
    x, u = _gen((n,), 31, dev, dtype, 0, 2.0), _gen((n,), 32, dev, dtype, 0, 2.0)
    guarded = lambda m: torch.full((m + 8,), 7.0, device=dev, dtype=dtype)
    buf = guarded(n)
    got = ops.add(x, u, out=buf[:n])
    assert torch.equal(got, (x.float() + u.float()).to(dtype)) and (buf[n:] == 7).all()  # in f32, rounded once
    for fn in (ops.swiglu, lambda a, b: ops.gelu_tanh(a)):
        assert torch.equal(fn(x, u).view(torch.uint8), _pieces(fn, x, u).view(torch.uint8))
    rows, w = 1100, 1000 + k
    y, b, buf = _gen((rows, w), 33, dev, dtype), _gen((w,), 34, dev, torch.float32), guarded(rows * w)
    got = ops.add_bias(y, b, out=buf[:rows * w].view(rows, w))
    assert torch.equal(got, (y.float() + b).to(dtype)) and (buf[rows * w:] == 7).all()
