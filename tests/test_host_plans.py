"""Rules of the library's host side over random layers: host_plans.hip compiled for the CPU alone."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plans") / "host_plans")
    r = subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-std=c++17", "-O1", "-w",
                        os.path.join(HERE, "host_plans.hip"), "-o", exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    return exe


@pytest.mark.parametrize("what", ["noalloc", "native16", "jobs", "layout", "weight64", "added"])
def test_rule(probe, what):
    r = subprocess.run([probe, what, "7", "20000"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("what", ["quad", "rows", "plain_rows", "plain_chunks", "plain"])
def test_measured_line(probe, what):
    """Which variant of a kernel a layer takes, where the times with either are known."""
    r = subprocess.run([probe, what, "7", "1"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_divisors(probe):
    r = subprocess.run([probe, "div", "7", "2000"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("kb", [None, "72", "156", "158", "160", "100000"])
def test_lds_budget(probe, kb):
    """A budget past what a workgroup can have is that: its plans launch."""
    env = dict(os.environ)
    env.pop("DCN_SCATTER_BUDGET_KB", None)
    if kb:
        env["DCN_SCATTER_BUDGET_KB"] = kb
    assert subprocess.run([probe, "budget", "7", "1"], env=env, timeout=60).returncode == 0
