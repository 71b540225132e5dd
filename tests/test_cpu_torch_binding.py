"""The native op calls (binding/torch_ops.cpp) without a GPU: every function of ops.py reaches its argument
checks with the arguments it documents, and refuses what is not a contiguous device tensor."""
import subprocess
import sys
from pathlib import Path

import pytest
import torch

import sapient_amd.ops as ops

X, I = torch.zeros(1, 2, 3, 4), torch.zeros(3, dtype=torch.int32)
CALLS = {
    "rms_norm": lambda t: ops.rms_norm(t, None, 1e-5, out_dtype=torch.float32),
    "layer_norm": lambda t: ops.layer_norm(t, None, None, 1e-5),
    "add_rms_norm": lambda t: ops.add_rms_norm(t, t, None, 1e-5, sum_out=t),
    "add": lambda t: ops.add(t, t), "mul": lambda t: ops.mul(t, t, out=t), "silu": ops.silu,
    "swiglu": lambda t: ops.swiglu(t, t), "gelu_tanh": ops.gelu_tanh, "gelu_erf": lambda t: ops.gelu_erf(t, out=t),
    "add_bias": lambda t: ops.add_bias(t, t),
    "rope_": lambda t: ops.rope_(t, None, I, 1e4, rotary_dim=2, interleaved=True),
    "rope_cached_": lambda t: ops.rope_cached_(t, t, t, t, positions=I, bad_pos_flag=I),
    "embed": lambda t: ops.embed(t, 0, 3, 4, I, bad_id_flag=I), "transpose_heads": lambda t: ops.transpose_heads(t),
    "kv_append": lambda t: ops.kv_append(t, t, 0), "kv_cache_update": lambda t: ops.kv_cache_update(t, t, 0),
    "kv_cache_update_into": lambda t: ops.kv_cache_update_into(t, t, t, 0),
    "rope_kv_append": lambda t: ops.rope_kv_append(t, t, t, I, 1e4, t, t, bq=t),
    "rope_kv_append_tokens": lambda t: ops.rope_kv_append_tokens(t, t, t, I, 1e4, t, t, bv=t, out=t),
}


@pytest.mark.parametrize("name", CALLS)
def test_refuses_host_tensors_and_other_objects(name):
    with pytest.raises(ValueError, match="must be a device tensor"):
        CALLS[name](X)
    with pytest.raises(TypeError, match="must be a torch.Tensor"):
        CALLS[name](object())


def test_library_builds_without_torch(monkeypatch, tmp_path):
    """The C library needs hipcc alone: without torch the binding is left out, and none from an earlier build stays."""
    from sapient_amd import build
    stale = tmp_path / "_torch_ops.so"
    stale.write_bytes(b"an earlier build")
    monkeypatch.setattr(build, "BINDING", stale)
    monkeypatch.setattr(build.importlib.util, "find_spec", lambda name: None)
    assert build._build_binding() == "torch not found" and not stale.exists()


@pytest.mark.parametrize("what", ["torch", "abi"])
def test_refuses_a_binding_built_for_another(monkeypatch, what):
    if what == "torch":
        monkeypatch.setattr(torch, "__version__", "0.0.1")
    else:
        monkeypatch.setattr(ops, "lib", lambda: type("L", (), {"sph_abi_version": staticmethod(lambda: 99)}))
    with pytest.raises(RuntimeError, match="is built for torch .* run `python -m sapient_amd.build`"):
        ops._Unloaded().silu


CHILD = """
import ctypes, sys
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
with FakeTensorMode():
    x = torch.empty(8, device="cuda")  # passes for a device tensor; there is no memory behind it
seen = ctypes.PyDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import sapient_amd.ops as ops
try:
    ops.silu(x)
except RuntimeError as e:
    print(e, seen.empty_calls(), seen.empty_held())
"""


def test_outputs_are_allocated_without_the_gil():
    """As by torch's own calls: other Python threads run on while the allocator waits for its lock or the device."""
    root = Path(__file__).resolve().parents[1]
    so = root / "tests" / "native" / "_build" / "empty_recorder.so"
    if not so.exists():
        import importlib.util
        spec = importlib.util.spec_from_file_location("native_build", so.parents[1] / "build.py")
        mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
        mod.build()
    res = subprocess.run([sys.executable, "-c", CHILD, str(so)], capture_output=True, text=True, cwd=root, timeout=120)
    assert res.stdout.split() == ["recorded", "1", "0"], res.stdout + res.stderr
