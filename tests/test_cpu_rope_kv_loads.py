"""CPU: what a decode step waits for, in the code built for gfx950. A fused RoPE + KV step is a few hundred threads
whose time is its chain of memory round trips, so rope_kv_kernel asks for its arguments in one batch and for the
position, the supplied angles, the rows and the biases before it waits for any of them; only per-position angles,
whose address is the position, come after. Held here on the library's own code objects."""
import re
import struct
import subprocess

import pytest

import sapient_amd

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
T = {"f32": "f", "f16": "NS_3f16E", "bf16": "NS_4bf16E"}


@pytest.fixture(scope="module")
def rope_object(tmp_path_factory):
    """The gfx950 code object that holds the fused step's kernels, out of the library's bundles."""
    if not sapient_amd.LIB_PATH.exists():
        from sapient_amd import build
        build.build()
    lib = sapient_amd.LIB_PATH.read_bytes()
    for at in (m.start() for m in re.finditer(MAGIC, lib)):
        n, = struct.unpack_from("<Q", lib, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        if n > 8:
            continue
        for _ in range(n):
            off, size, k = struct.unpack_from("<QQQ", lib, p)
            triple = lib[p + 24:p + 24 + k]
            p += 24 + k
            code = lib[at + off:at + off + size]
            if b"gfx950" in triple and b"rope_kv_kernel" in code:
                f = tmp_path_factory.mktemp("code") / "rope.co"
                f.write_bytes(code)
                return f
    pytest.fail("no gfx950 code object with rope_kv_kernel in the library")


# storage type, cache type, pairs per thread of a one-token step (half of the widest run)
@pytest.mark.parametrize("t,tc,pairs", [("f32", "f16", 2), ("f32", "f32", 2), ("f16", "f16", 4), ("bf16", "bf16", 4)])
@pytest.mark.parametrize("tokens_major", [0, 1])
@pytest.mark.parametrize("bias", [0, 1])
def test_one_wait_on_memory(rope_object, t, tc, pairs, tokens_major, bias):
    c = "S2_" if t == tc != "f32" else T[tc]
    name = f"_ZN3sph12_GLOBAL__N_114rope_kv_kernelI{T[t]}{c}Li{pairs}ELb0ELb{tokens_major}ELi1ELb{bias}ELb0EEE"
    syms = subprocess.run([OBJDUMP, "-t", str(rope_object)], capture_output=True, text=True, check=True).stdout
    full = [s for s in re.findall(r"(\S+)$", syms, flags=re.M) if s.startswith(name) and "." not in s]
    assert len(full) == 1, (name, full)
    text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={full[0]}", str(rope_object)], capture_output=True,
                          text=True, check=True).stdout
    code = re.findall(r"^\t(\S.*?)\s*//", text, flags=re.M)
    loads = [i for i, l in enumerate(code) if l.startswith("global_load")]
    first = next(i for i, l in enumerate(code) if l.startswith("s_waitcnt") and "vmcnt" in l)
    by_position = 2 * pairs * 4 // 16
    assert loads and sum(i > first for i in loads) <= by_position, "a load is asked for after a wait"
    # Scalar loads of the arguments (base s[0:1]): the first batch reaches every 64-byte line that is read at all.
    first = next(i for i, l in enumerate(code) if l.startswith("s_waitcnt") and "lgkmcnt" in l)
    args = [(i, int(m.group(1), 16) // 64) for i, l in enumerate(code)
            if (m := re.match(r"s_load_dword\w* \S+ s\[0:1\], (0x[0-9a-f]+)", l))]
    assert {ln for _, ln in args} == {ln for i, ln in args if i < first}, "an argument is asked for after a wait"
