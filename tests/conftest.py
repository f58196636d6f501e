import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")


@pytest.fixture(scope="session")
def gpu():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU visible")
    return torch.device("cuda:0")


@pytest.fixture
def cpp_harness(tmp_path):
    """Builds ``tests/cpp/<name>.cpp`` against the library and runs it: ``run(name, *args)`` gives
    what it printed."""
    import shutil
    import subprocess
    from pathlib import Path

    from dmuon_amd import _C
    gxx, rocm = shutil.which("g++"), Path("/opt/rocm")
    if gxx is None or not (rocm / "include" / "hip" / "hip_runtime.h").exists():
        pytest.skip("needs g++ and the ROCm headers")
    lib_dir = _C.lib_path().parent

    def run(name, *args):
        exe = tmp_path / name
        build = subprocess.run(
            [gxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm / 'include'}",
             str(Path(__file__).resolve().parent / "cpp" / f"{name}.cpp"), f"-L{lib_dir}",
             "-ldmuon_amd", f"-L{rocm / 'lib'}", "-lamdhip64", f"-Wl,-rpath,{lib_dir}",
             f"-Wl,-rpath,{rocm / 'lib'}", "-o", str(exe)], capture_output=True, text=True)
        assert build.returncode == 0, build.stderr
        out = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True,
                             timeout=60)
        assert out.returncode == 0, out.stdout + out.stderr
        return out.stdout.strip()
    return run
