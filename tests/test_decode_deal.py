"""The dealing of decode attention's keys to workgroups, on the CPU: the arithmetic that the kernel uses
(csrc/q36_deal.h) walked by tests/deal_check.cpp over equal and ragged batches in page tables from as wide as
the requests to much wider.  Every key step lies in exactly one run, and the combine reads exactly the
partials that the same call's workgroups write."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("deal") / "deal_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(HERE, "..", "bundles_amd", "csrc"), "-o", out,
                    os.path.join(HERE, "deal_check.cpp")], check=True)
    return out


@pytest.mark.parametrize("seed", [1, 2])
def test_every_step_once_and_every_partial_read_was_written(exe, seed):
    r = subprocess.run([exe, str(seed), "20000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
