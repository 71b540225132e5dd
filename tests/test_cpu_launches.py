"""CPU: the launches of C ABI calls at sizes no test machine's memory has to hold. The library runs in a child
process under tests/native/launch_recorder.cpp, which stands in for the HIP runtime: it refuses a launch as HIP does
(2^32 work-items and more) and names the kernel, grid and block of every other. Nothing is run, so the pointers are
addresses of nothing."""
import json
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
RECORDER = ROOT / "tests" / "native" / "_build" / "launch_recorder.so"
CHILD = """
import ctypes, json, sys
rec = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the library: its symbols come first
rec.take_launches.restype = ctypes.c_char_p
from sapient_amd._lib import lib
n = ctypes.c_int64()
for name, args in json.load(sys.stdin):
    st = getattr(lib(), name)(*[ctypes.addressof(n) if a == "host int64" else a for a in args])
    print(json.dumps([st, [l.split() for l in rec.take_launches().decode().splitlines()]]))
"""
F32, F16 = 0, 1
A, B, C, D, E, G, H, I = ((i + 1) << 42 for i in range(8))  # 16-byte aligned, 4 TiB apart


@pytest.fixture(scope="module")
def launches():
    """launches(*calls): (status, [(kernel, grid x, grid y, block x)]) of each (function, *arguments)."""
    import sapient_amd
    if not sapient_amd.LIB_PATH.exists():
        from sapient_amd import build
        build.build()
    if not RECORDER.exists():
        import importlib.util
        spec = importlib.util.spec_from_file_location("native_build", RECORDER.parents[1] / "build.py")
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        mod.build()

    def go(*calls):
        res = subprocess.run([sys.executable, "-c", CHILD, str(RECORDER)], input=json.dumps([[c[0], c[1:]] for c in calls]),
                             capture_output=True, text=True, cwd=ROOT, timeout=120)
        assert res.returncode == 0, res.stderr
        got = [json.loads(line) for line in res.stdout.splitlines()]
        return [(st, [(k, int(x), int(y), int(b)) for k, x, y, b in ls]) for st, ls in got]
    return go


@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 63, 1001, 4096])
def test_add_bias_at_any_row_count(launches, n):
    """Narrow rows by the 2^27 and more, and the largest tensors: one launch within HIP's limit."""
    calls = [("sph_add_bias", A + off, B, F32, C + off, dt, rows * n, n, None)
             for dt in (F32, F16) for off in (0, 4 - 2 * dt) for rows in (1, (1 << 27) + 1, (1 << 36) // n)]
    for call, (st, ls) in zip(calls, launches(*calls)):
        assert st == 0 and len(ls) == 1, (call, st, ls)


@pytest.mark.parametrize("hd,il", [(8, 0), (64, 1), (128, 0), (512, 0)])
def test_fused_rope_step_at_any_token_count(launches, hd, il):
    """Chunks past what one launch holds are split by tokens, each launch as full as HIP allows."""
    for seq in (1, (1 << 24) + 5, (1 << 33) // hd):
        tail = [F32, il, D, seq, hd, 1e4, 1.0, E, G, F16, seq, None, None, None, F32, None, None]
        calls = [("sph_rope_kv_append", A, 2, B, C, 1, *tail), ("sph_rope_kv_append_tokens", A, H, 2, B, C, 1, *tail)]
        for st, ls in launches(*calls):
            assert st == 0 and all(k.startswith("rope_kv_kernel<") for k, *_ in ls), (seq, st, ls)
            assert len(ls) == 1 or all(x * b > (1 << 32) - 512 for _, x, _, b in ls[:-1]), ls


@pytest.mark.parametrize("heads", [1, 2, 3, 16])
def test_fused_rope_step_fills_its_blocks(launches, heads):
    """A 256-thread block takes 256 angles' tokens, also where few heads make few lanes of many tokens."""
    seq, hd = 16384, 64
    (st, [(_, x, y, b)]), = launches(("sph_rope_kv_append", A, heads - heads // 2, B, C, heads // 2, F16, 0, D, seq, hd, 1e4,
                                      1.0, E, G, F16, seq, None, None, None, F16, None, None))
    assert st == 0 and b == 256 and seq // x == 256 // (hd // 2), (x, y, b)


@pytest.mark.parametrize("dt", [F32, F16])
@pytest.mark.parametrize("dim", [7, 2049, 4096, 4097, 8193, 8200, 16383, 16384, 20001])
def test_norms_at_any_row_count(launches, dt, dim):
    """The widest blocks (16 waves a row) and the most rows a launch takes: each launch within HIP's limit, no row lost."""
    rows = (1 << 22) + 3
    w = [G, F32]
    calls = [("sph_rms_norm", A, dt, *w, C, dt, rows, dim, 1e-5, None),
             ("sph_layer_norm", A, dt, G, H, F32, C, dt, rows, dim, 1e-5, None),
             ("sph_add_rms_norm", A, B, dt, *w, C, dt, rows, dim, 1e-5, None),
             ("sph_add_rms_norm_to", A, B, D, dt, *w, C, dt, rows, dim, 1e-5, None)]
    for call, (st, ls) in zip(calls, launches(*calls)):
        assert st == 0, (call, st, ls)
        if all(k.startswith("rms_rows_generic<") for k, *_ in ls):
            assert sum(x for _, x, _, _ in ls) == rows


# The kernel of element accesses is the quicker one for a few narrow rows, the ragged one from there on.
@pytest.mark.parametrize("dt,rows,dim,kernel", [(F16, 1, 7, "generic"), (F16, 300, 127, "generic"), (F16, 514, 511, "ragged"),
                                                (F16, 3073, 7, "ragged"), (F16, 2100, 127, "ragged"), (F16, 1, 513, "ragged"), (F32, 300, 17, "generic"),
                                                (F32, 1, 65, "ragged"), (F32, 3073, 7, "ragged")])
def test_few_narrow_norm_rows(launches, dt, rows, dim, kernel):
    for call in (("sph_rms_norm", A, dt, G, F32, C, dt, rows, dim, 1e-5, None),
                 ("sph_add_rms_norm", A, B, dt, G, dt, C, F32, rows, dim, 1e-5, None),
                 ("sph_layer_norm", A, dt, G, H, F32, C, dt, rows, dim, 1e-5, None)):
        (st, [(k, *_)]), = launches(call)
        assert st == 0 and k.startswith(f"rms_rows_{kernel}<"), k


# Rows no aligned vector fits: element by element in small launches and where they are narrow, else in runs.
@pytest.mark.parametrize("dt,off,total,n,kernel", [(F32, 0, 1 << 24, 1, "scalar"), (F32, 0, 1 << 24, 255, "scalar"),
                                                   (F32, 4, 1 << 24, 256, "scalar"), (F32, 0, 1 << 24, 257, "rows"),
                                                   (F16, 0, 1 << 24, 7, "scalar"), (F16, 2, 1 << 24, 288, "scalar"),
                                                   (F16, 0, 1 << 24, 289, "rows"), (F16, 0, 1 << 20, 1001, "scalar"),
                                                   (F16, 0, 1 << 20, 1000, "rows")])
def test_ragged_bias_kernel(launches, dt, off, total, n, kernel):
    (st, [(k, *_)]), = launches(("sph_add_bias", A + off, B, F32, C + off, dt, total // n * n, n, None))
    assert st == 0 and k.startswith(f"bias_{kernel}<"), k


# Half GELU: single elements in small launches, and longer at addresses without 16-byte alignment.
@pytest.mark.parametrize("off,n,kernel", [(0, 1 << 18, "_scalar"), (0, (1 << 18) + 8, ""), (2, (1 << 18) + 1, "_scalar"),
                                          (8, 9 << 18, "_scalar"), (2, (9 << 18) + 1, "")])
@pytest.mark.parametrize("fn", ["sph_gelu_tanh", "sph_gelu_erf"])
def test_half_gelu_kernel(launches, fn, off, n, kernel):
    for a, c in ((A + off, C), (A, C + off)):
        (st, ls), = launches((fn, a, c, F16, n, None))
        assert st == 0 and ls[-1][0].startswith(f"gelu_lut_apply{kernel}<"), ls[-1]  # (the first call builds the tables)


# An in-place slide: windows where one block holds a head, and from 5 MB of valid rows on (up to 4096 windows a head);
# by reversal else. Float caches append in the last launch, others in a launch of their own.
@pytest.mark.parametrize("heads,hd,dt,cur,shift,kernels", [
    (2, 128, F16, 64, 31, ["kv_rotate_append"]), (2, 128, F16, 65, 31, ["kv_reverse_rows", "kv_reverse_append"]),
    (2, 64, F16, 4096, 16, ["kv_reverse_rows", "kv_reverse_append"]), (8, 128, F16, 2560, 1, ["kv_shift_slots", "kv_rotate_append"]),
    (8, 128, F16, 2559, 1, ["kv_reverse_rows", "kv_reverse_append"]), (8, 128, F16, 8192, 32, ["kv_reverse_rows", "kv_reverse_append"]),
    (8, 128, 8, 8192, 1, ["kv_shift_slots", "kv_rotate_windows", "kv_append_q8_0"]),
    (2, 64, 8, 4096, 4, ["kv_reverse_rows", "kv_reverse_rows", "kv_append_q8_0"]),
    (1, 8, F16, 4096 << 10, 3, ["kv_shift_slots", "kv_rotate_append"]),
    (1, 8, F16, (4096 << 10) + 1, 3, ["kv_reverse_rows", "kv_reverse_append"])])
def test_kv_slide_form(launches, heads, hd, dt, cur, shift, kernels):
    (st, ls), = launches(("sph_kv_cache_update", A, F16, B, dt, heads, shift, hd, cur, cur, "host int64", None))
    assert st == 0 and [k.split("<")[0] for k, *_ in ls] == kernels, ls


def test_kv_slide_at_the_most_rows_a_launch_takes(launches):
    """Rows past cur_len ride in the launch of the windows: within HIP's limit, else an append of its own."""
    for seq in range((1 << 32) - 300, (1 << 32) - 256, 3):
        (st, ls), = launches(("sph_kv_cache_update", A, F16, B, F16, 1, seq, 8, seq + 1, 2, "host int64", None))
        assert st == 0 and ls, (seq, st)


# One element a thread: f32 GELU to 2^18 elements, to 5 x 2^18 at addresses without 16-byte alignment.
@pytest.mark.parametrize("off,n,kernel", [(0, 1 << 18, "scalar"), (0, (1 << 18) + 4, "runs"), (4, 5 << 18, "scalar"),
                                          (4, (5 << 18) + 4, "runs")])
def test_f32_gelu_kernel(launches, off, n, kernel):
    for a, c in ((A + off, C), (A, C + off)):
        (st, [(k, *_)]), = launches(("sph_gelu_tanh", a, c, F32, n, None))
        assert st == 0 and k.startswith(f"ew_{kernel}<float,4,"), k


# Half SiLU and SwiGLU: one element a thread to 2^19 elements (5 x 2^18 unaligned), else whole runs.
@pytest.mark.parametrize("off,n,kernel", [(0, 1 << 19, "scalar"), (0, (1 << 19) + 8, "runs"), (2, 5 << 18, "scalar"),
                                          (8, (5 << 18) + 8, "runs")])
def test_half_silu_kernel(launches, off, n, kernel):
    calls = [("sph_silu", A + off, C, F16, n, None), ("sph_swiglu", A, B + off, C, F16, n, None)]
    for call in calls:
        (st, [(k, x, _, b)]), = launches(call)
        assert st == 0 and k.startswith(f"ew_{kernel}<"), k
        assert kernel == "scalar" or x * b >= n // 8 > x * b - b, (k, x, b)


# Where one run a thread covers a launch: cached below 16 MB of traffic (policy 0), from there on non-temporal stores
# (1), for adds and products loads as well (2).
@pytest.mark.parametrize("n", [(1 << 20) + 4, 1 << 21, 1 << 22])
def test_element_wise_cache_policy(launches, n):
    large = n >= 1 << 21
    for call, want in ((("sph_add", A, n, B, n, C, F32, None), 2 * large), (("sph_mul", A, n, B, 1, C, F32, None), 2 * large),
                       (("sph_swiglu", A, B, C, F32, n, None), large), (("sph_gelu_erf", A, C, F32, n, None), large)):
        (st, [(k, *_)]), = launches(call)
        u, p = map(int, k.split(",")[3:5])
        assert st == 0 and (u, p) == (1, want), k
