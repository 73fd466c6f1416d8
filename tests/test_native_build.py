"""_native.so is taken only if it was built from the present source, and its absence costs speed alone.  CPU only."""

import os
import shutil
import subprocess
import sys

import torch

from spio_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_a_changed_source_or_torch_makes_the_extension_stale(tmp_path, monkeypatch):
    if not build.extension_is_current():
        build.build_extension()
    assert build.extension_is_current()
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "0.0.0")
        assert not build.extension_is_current()
    with monkeypatch.context() as m:
        m.setattr(build, "EXTENSION_PATH", str(tmp_path / "absent.so"))
        assert not build.extension_is_current()
    shutil.copytree(build.CSRC_DIR, tmp_path / "csrc", ignore=shutil.ignore_patterns("*.so"))
    monkeypatch.setattr(build, "CSRC_DIR", str(tmp_path / "csrc"))
    assert build.extension_is_current()
    with open(tmp_path / "csrc" / "spio_torch.cpp", "a", encoding="utf-8") as f:
        f.write("// changed\n")
    assert not build.extension_is_current()


def test_without_the_extension_the_python_operators_run(tmp_path):
    """A tree whose _native.so is stale and cannot be built again: it warns, and every part of the package works."""
    for name in ("spio_amd", "include"):
        shutil.copytree(os.path.join(ROOT, name), tmp_path / name, ignore=shutil.ignore_patterns("__pycache__"))
    (tmp_path / "spio_amd" / "_native.so").write_bytes(b"stale")
    code = """
import warnings, torch
with warnings.catch_warnings(record=True) as caught:
    warnings.simplefilter("always")
    from spio_amd import functional, native
    from spio_amd.kernels import KernelParamsLogger
assert native._native is None and any("_native" in str(w.message) for w in caught)
with KernelParamsLogger():
    native.forget_plans()
try:
    functional.conv2d_gw8(torch.zeros(1, 8, 4, 4).half(), torch.zeros(8, 8, 1, 1).half(), groups=1)
except RuntimeError as e:
    assert "GPU only" in str(e)
else:
    raise SystemExit("a CPU tensor was taken")
"""
    env = dict(os.environ, CXX="/bin/false", PYTHONPATH=str(tmp_path))
    subprocess.run([sys.executable, "-c", code], cwd=tmp_path, env=env, check=True, timeout=300)
