"""A sparsifier encode whose last launch the runtime refuses: an error, and nothing lost from the residual (the pass leaves zeros
there for what that launch sends, so it has to know before).  In a process of its own, in which hipFuncSetAttribute fails."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

STUB = 'extern "C" int hipFuncSetAttribute(const void*, int, int) { return 1; }\n'   # hipErrorInvalidValue

CHILD = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before the runtime: its name is found here first
sys.path.insert(0, sys.argv[2])
import importlib, torch
c = importlib.import_module("torch-hipress-extension_amd")._capi
L = c.load()
n = 1 << 20
g, r = torch.randn(n, device="cuda"), torch.randn(n, device="cuda")
want, out = r.clone(), torch.zeros(4 + 8 * 1049, dtype=torch.uint8, device="cuda")
rc = L.hpx_gd_encode(1, c.ptr_array([g.data_ptr()]), c.i32_array([n]), c.ptr_array([r.data_ptr()]), c.ptr_array([out.data_ptr()]),
                     c.f64_array([0.01]), c.f64_array([0.999]), c.u64_array([1]), torch.cuda.current_stream().cuda_stream)
torch.cuda.synchronize()
assert rc != 0 and c.last_error(), rc
assert torch.equal(r, want), "the residual lost entries"
print("kept", flush=True)
"""


def test_the_residual_is_kept(tmp_path, capi):
    (tmp_path / "stub.cpp").write_text(STUB)
    stub = str(tmp_path / "stub.so")
    subprocess.check_call(["g++", "-shared", "-fPIC", "-o", stub, str(tmp_path / "stub.cpp")])
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, stub, root], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "kept" in r.stdout, r.stdout + r.stderr
