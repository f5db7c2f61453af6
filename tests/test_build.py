"""The build's view of _host.so, which is linked against torch: what it is built for, when it is built again, and what the
package does beside one that cannot be loaded.  Nothing is compiled here."""
import importlib.util
import os
import shutil
import subprocess
import sys

import pytest
import torch

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pytorch-approx-topk_amd")


@pytest.fixture
def build():
    spec = importlib.util.spec_from_file_location("atk_build", os.path.join(PKG, "build.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def test_host_module_is_built_again_for_another_torch(build, monkeypatch):
    from approx_topk import _native
    assert build._built_for() == _native.host.built_for and torch.__version__ in _native.host.built_for
    assert build._host_is_current([])
    monkeypatch.setattr(build, "_built_for", lambda: "approx_topk for torch 0.0, cpython-0;")
    assert not build._host_is_current([])


@pytest.mark.parametrize("hipcc", ["hipcc", "/opt/rocm/bin/hipcc"])
def test_headers_are_found_for_a_compiler_on_the_path(build, monkeypatch, hipcc):
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    monkeypatch.delenv("ROCM_PATH", raising=False)
    monkeypatch.setattr(build, "HIPCC", hipcc)
    command = build._host_command("x.cpp")
    assert os.path.exists(os.path.join(build._rocm_include(), "hip", "hip_runtime_api.h"))
    assert all(os.path.isdir(command[i + 1]) for i, word in enumerate(command) if word == "-isystem")


@pytest.mark.parametrize("fault", ["another torch", "broken", "missing"])
def test_package_without_a_host_module_that_loads(tmp_path, fault):
    shutil.copytree(os.path.join(PKG, "approx_topk"), tmp_path / "approx_topk", ignore=shutil.ignore_patterns("*.so", "__pycache__"))
    os.symlink(os.path.join(PKG, "approx_topk", "libapprox_topk_hip.so"), tmp_path / "approx_topk" / "libapprox_topk_hip.so")
    host = tmp_path / "approx_topk" / "_host.so"
    if fault == "another torch":
        host.write_bytes(b"approx_topk for torch 0.0, cpython-0;")
    elif fault == "broken":
        from approx_topk import _native
        host.write_bytes(_native.host.built_for.encode())
    code = """
import torch, approx_topk
from approx_topk import _native
from approx_topk.experimental import autobucket, bucketed_argmax, differentiable
x = torch.arange(64.0).view(1, 64)
exact = lambda xs, k, dim: tuple(torch.topk(xs, k, dim))
for values, _ in (bucketed_argmax.topk_torch(x, 4, -1, True), autobucket.bucket(exact, 2, 1, True)(x, 4, -1)):
    assert sorted(values[0].tolist()) == [60.0, 61.0, 62.0, 63.0]
try:
    _native.lib()
except RuntimeError as e:
    assert "build.py" in str(e) and "_host.so" in str(e), e
else:
    raise SystemExit("loaded")
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, env={**os.environ, "PYTHONPATH": str(tmp_path)},
                          capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr
