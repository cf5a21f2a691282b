"""Counts that their kernel hands to the host itself, through a word of pinned
memory that holds the call's number: what the memory held before may not be
taken for the result."""
import os
import subprocess

import pytest

import oracle
import subgraphmatchgpu_amd as sme
from conftest import ROOT

EMU_DIR = os.path.join(ROOT, "tests", "emu")


@pytest.fixture(scope="module")
def publish_test():
    subprocess.run(["make", "-C", EMU_DIR, "-s", "publish_test"], check=True)
    return os.path.join(EMU_DIR, "publish_test")


@pytest.mark.parametrize("what", ["stale", "dropped"])
def test_published_sums_are_the_calls(publish_test, what):
    """stale: pinned pages that come filled with 1, 2, ..: before its launch no call is published;
    dropped: a call whose launch did not happen fails, the calls after it are right."""
    r = subprocess.run([publish_test, what], capture_output=True, text=True, timeout=120,
                       env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize("calls", [1, 2, 5])
def test_devices_opened_in_turn(calls):
    """Each device counts another small graph and is closed: the next one's first calls carry the
    same numbers, on memory that the last one may have used."""
    for k in range(8):
        g = sme.gen_er(200 + 17 * k, 900 + 101 * k, seed=k)
        dev = sme.Device(0, budget_bytes=64 << 20)
        dg = dev.upload(g)
        for q in (0, 3, 0, 7, 3)[:calls]:
            r = dev.count(dg, sme.Plan(q))
            want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
            assert (r.count, r.levels) == (want[0], want[1]), (k, q)
        dev.close()


@pytest.mark.gpu
def test_two_devices_call_by_call():
    """Two open devices whose calls carry the same numbers."""
    gs = [sme.gen_er(150, 700, seed=1), sme.gen_er(310, 2100, seed=2)]
    want = [oracle.light_count(g.row_ptrs, g.cols, 0, 3) for g in gs]
    for _ in range(3):
        devs = [sme.Device(0, budget_bytes=64 << 20) for _ in gs]
        ups = [d.upload(g) for d, g in zip(devs, gs)]
        for k in range(6):
            r = devs[k % 2].count(ups[k % 2], sme.Plan(0))
            assert (r.count, r.levels) == (want[k % 2][0], want[k % 2][1])
        for d in devs:
            d.close()
