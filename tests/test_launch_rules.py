"""The host's dispatch rules (csrc/launch_rules.h, compiled here with the host compiler) -- CPU only."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rules") / "launch_rules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    os.path.join(HERE, "cpp", "launch_rules.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def test_merge_trips_fit_the_longest_row(rules):
    """A row's sources in at most four trips for up to 64 ranges, whatever the average; no trip sized past
    the number of ranges."""
    for ngroups in (1, 2, 8, 16, 32, 64):
        for B in (1, 2, 3, 8, 16, 32, 64, 128, 1023):
            n = rules.rule_merge_ranges_sources(ngroups, B)
            assert 1 <= n <= ngroups
            assert -(-ngroups // n) <= 4, (ngroups, B, n)
            assert n >= min(ngroups, ngroups // B + 2)
