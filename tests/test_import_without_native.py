"""Importing the package where the native binding is absent or does not load:
the import goes on, a call raises, and a call after the build reaches the
kernel (host tensors through the device key: no GPU work is reached)."""

import os
import shutil
import subprocess
import sys
import textwrap

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                   "idempotent_llm_amd")
BUILT = [f for f in ("_native.so", "libdetllm_hip.so") if os.path.exists(os.path.join(PKG, f))]

PROGRAM = """
    import os, shutil, torch
    from idempotent_llm_amd import _lib, backends, model, plugin, torch_ops
    op = torch.ops.detllm_rocm.int_gemm.default
    key = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
    i8 = lambda *s: torch.zeros(s, dtype=torch.int8)
    for _ in range(2):
        try:
            op.redispatch(key, i8(0, 16), i8(16, 5))
        except _lib.LibraryMissing as e:
            assert "g.build()" in str(e)
        else:
            raise AssertionError("called without a kernel")
    for f in ("_native.so", "libdetllm_hip.so"):
        if os.path.exists(f"idempotent_llm_amd/{f}"):
            os.remove(f"idempotent_llm_amd/{f}")
        shutil.copy(os.path.join(os.environ["BUILT_PKG"], f), "idempotent_llm_amd")
    for _ in range(2):
        out = op.redispatch(key, i8(0, 16), i8(16, 5))
        assert out.shape == (0, 5) and out.dtype == torch.int32
        try:
            op.redispatch(key, i8(3, 16), i8(8, 5))
        except ValueError:
            pass
        else:
            raise AssertionError("the native kernel's check did not run")
    print("ok")
"""


@pytest.mark.skipif(len(BUILT) < 2, reason="library not built (run build())")
@pytest.mark.parametrize("state", ["absent", "broken", "library absent"])
def test_import_goes_on_and_a_call_raises(tmp_path, state):
    pkg = tmp_path / "idempotent_llm_amd"
    pkg.mkdir()
    for f in os.listdir(PKG):
        if f.endswith(".py"):
            shutil.copy(os.path.join(PKG, f), pkg)
    if state == "broken":
        (pkg / "_native.so").write_bytes(b"not a library")
        shutil.copy(os.path.join(PKG, "libdetllm_hip.so"), pkg)
    elif state == "library absent":
        shutil.copy(os.path.join(PKG, "_native.so"), pkg)
    p = subprocess.run([sys.executable, "-c", textwrap.dedent(PROGRAM)], cwd=tmp_path,
                       env=dict(os.environ, BUILT_PKG=PKG, PYTHONPATH=str(tmp_path)),
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0 and p.stdout.strip().endswith("ok"), p.stderr[-2000:]
