"""The operators' native library (libtokserve_torch.so) where it does not fit: the package
imports, and says what is wrong when a kernel is called (CPU)."""

import os
import shutil
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from tokserve_amd.kernels import _lib, torch_ops

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "tokserve_amd" / "csrc"


def test_the_built_library_fits() -> None:
    assert torch_ops._load_native(torch_ops.NATIVE_LIBRARY) is None
    for name in torch_ops.SCHEMAS:
        assert torch._C._dispatch_has_kernel_for_dispatch_key(f"tokserve_amd::{name}", "CUDA")


def test_package_imports_beside_a_library_that_does_not_load(tmp_path) -> None:
    shutil.copytree(ROOT / "tokserve_amd", tmp_path / "tokserve_amd",
                    ignore=shutil.ignore_patterns("*.so", "csrc", "__pycache__"))
    (tmp_path / "tokserve_amd" / "libtokserve_torch.so").write_bytes(b"not a library")
    code = ("import torch\nfrom tokserve_amd.kernels import ops, torch_ops\n"
            "print(torch_ops.__file__)\n"
            "try: torch_ops._unavailable(torch_ops._load_native(torch_ops.NATIVE_LIBRARY))()\n"
            "except RuntimeError as error: print(error)\n")
    run = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True,
                         text=True, env={**os.environ, "PYTHONPATH": str(tmp_path)})
    assert run.returncode == 0, run.stderr
    assert str(tmp_path) in run.stdout and "does not load into torch" in run.stdout


@pytest.mark.parametrize(("torch_version", "abi", "message"), [
    ("1.0.0", _lib.ABI_VERSION, "was built for torch 1.0.0"),
    (torch.__version__.split("+")[0], _lib.ABI_VERSION - 1, f"ABI {_lib.ABI_VERSION - 1} does")])
def test_a_library_of_other_versions_is_not_registered(tmp_path, torch_version, abi,
                                                       message) -> None:
    (tmp_path / "stub.c").write_text(
        f'const char *tks_torch_built_for(void) {{ return "{torch_version}"; }}\n'
        f"int tks_torch_abi_version(void) {{ return {abi}; }}\n"
        'const char *tks_torch_register(void) { return "registered"; }\n')
    stub = tmp_path / "stub.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", stub, tmp_path / "stub.c"], check=True)
    error = torch_ops._load_native(stub)
    assert message in error and "registered" not in error


@pytest.mark.parametrize("version", ["2.10.0", "2.10.0+rocm7.0", "2.10.0a0+git1234",
                                     "2.10.0.dev20250101"])
def test_builds_of_one_release_fit(tmp_path, monkeypatch, version) -> None:
    (tmp_path / "stub.c").write_text(
        'const char *tks_torch_built_for(void) { return "2.10.0"; }\n'
        f"int tks_torch_abi_version(void) {{ return {_lib.ABI_VERSION}; }}\n"
        'const char *tks_torch_register(void) { return 0; }\n')
    stub = tmp_path / "stub.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", stub, tmp_path / "stub.c"], check=True)
    monkeypatch.setattr(torch, "__version__", version)
    assert torch_ops._load_native(stub) is None


def test_make_without_a_torch_builds_the_c_library_alone() -> None:
    run = subprocess.run(["make", "-n", "-C", CSRC, "PYTHON=false"], capture_output=True, text=True)
    assert run.returncode == 0, run.stderr
    assert "torch" not in run.stdout


def test_make_notices_another_torch(tmp_path) -> None:
    stamp = tmp_path / "torch_id"

    def make() -> int:
        subprocess.run(["make", "-C", CSRC, f"PYTHON={sys.executable}", f"BUILD={tmp_path}", stamp],
                       check=True, capture_output=True)
        return stamp.stat().st_mtime_ns

    first = make()
    assert torch.__version__ in stamp.read_text()
    assert make() == first
    stamp.write_text(stamp.read_text().replace(torch.__version__, "1.0.0"))
    written = stamp.stat().st_mtime_ns
    assert make() > written
