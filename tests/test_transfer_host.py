"""The large host copies (eulersf_amd/host/esf_transfer.cpp) on the CPU,
against a stand-in for the HIP runtime (tests/native/transfer_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(HERE, "..", "eulersf_amd", "host")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    """runs a scenario: {step: {counter: value}}"""
    if shutil.which(HIPCC) is None:
        pytest.skip("no hipcc")
    tmp = tmp_path_factory.mktemp("transfer")
    objs = []
    for src in (os.path.join(HERE, "native", "transfer_check.cpp"),
                os.path.join(HOST, "esf_transfer.cpp")):
        objs.append(str(tmp / (os.path.basename(src) + ".o")))
        r = subprocess.run([HIPCC, "-O1", "-std=c++17", "-fPIC", "-x", "hip", "--offload-host-only",
                            "--offload-arch=gfx950", "-w", "-c", src, "-o", objs[-1]],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
    exe = str(tmp / "transfer_check")
    r = subprocess.run(["g++", *objs, "-lpthread", "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(scenario):
        out = subprocess.run([exe, scenario], capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, out.stdout + out.stderr
        steps = {}
        for line in out.stdout.splitlines():
            w = line.split()
            steps[w[0]] = {w[i]: int(w[i + 1]) for i in range(1, len(w), 2)}
        return steps

    return run


def test_the_callers_device_stays_current(check):
    s = check("device")
    assert s["large"]["chunks"] > 0 and s["large"]["device"] == 0
    assert s["small"]["device"] == 0 and s["end"]["device"] == 0
    assert s["end"]["events"] == 0 and s["end"]["mallocs"] == s["end"]["frees"]


def test_a_pinned_destination_is_copied_to_directly(check):
    """the link writes pinned memory itself; slots would only add a copy"""
    s = check("pinned")
    assert s["pageable"]["chunks"] > 0 and s["pageable"]["direct"] == 0
    for step in ("pinned", "inside"):
        assert s[step]["chunks"] == 0 and s[step]["direct"] == 1, step


def test_slots_are_pinned_once_the_copies_repay_it(check):
    """a set is made by the copy that brings the bytes since the first live
    context to 48 MiB, used from then on, and given back with the last one"""
    s = check("pool")
    assert s["single"]["mallocs"] == 0 and s["single"]["direct"] == 3
    assert s["big"]["chunks"] > 0 and s["big"]["mallocs"] == s["big"]["frees"] == 1
    for k in range(4):
        assert (s["copy%d" % k]["chunks"] > 0) == (k >= 2)
    assert s["end"]["mallocs"] == s["end"]["frees"] == 2
