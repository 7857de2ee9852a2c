"""The lane walks drop a subtree when its cylinder's lower bound exceeds the query's limit; they are exact only if that
bound, with its margins, never exceeds the limit of the distance that the subtree's own leaves have.  This builds
tests/cpp/lane_bound_fuzz.cpp (a host restatement of the records, the bound and the leaf test, with the library's margins)
and checks the claim on small flat oblique patches whose coordinates lie just above powers of two, where all roundings
add up, and on patches of any shape."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(__file__)


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_bound_never_exceeds_limit(tmp_path):
    exe = tmp_path / "lane_bound_fuzz"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(exe), f"{HERE}/cpp/lane_bound_fuzz.cpp"],
                   check=True, timeout=120)
    for seed in (1, 2):
        r = subprocess.run([str(exe), str(seed), "300000"], capture_output=True, text=True, timeout=300)
        print(r.stdout)
        assert r.returncode == 0, r.stdout
        assert "bad 0" in r.stdout
