"""pytest configuration: import paths and the `gpu` marker.

Tests marked `gpu` need an MI355X (gfx950) and the built library; the rest run on any CPU.
"""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for sub in ("cuda-kernel-lab_amd", "oracle", "tests"):
    path = os.path.join(ROOT, sub)
    if path not in sys.path:
        sys.path.insert(0, path)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a gfx950 GPU and the built libpdattn.so")


@pytest.fixture(scope="session")
def oracle_lib():
    import oracle
    oracle.build()
    return oracle


@pytest.fixture(scope="session")
def host_rules(tmp_path_factory):
    """The dispatch rules and range arithmetic of csrc/, compiled with the host compiler."""
    import ctypes
    import subprocess
    so = str(tmp_path_factory.mktemp("rules") / "launch_rules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "cpp", "launch_rules.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)
