"""The staged copies between host and device (host_copy.cpp) on a stand-in for the HIP runtime
(tests/host/runtime), for what a machine with one GPU cannot show: a caller whose current
device is another one, a runtime call that fails half way, and which way a copy takes."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MB = 1 << 20


@pytest.fixture(scope="module")
def run_copy(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_copy") / "host_copy.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-w", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "tests", "host", "runtime"), "-o", out,
                    os.path.join(ROOT, "tests", "host", "host_copy.cpp")], check=True)
    lib = ctypes.CDLL(out)

    def run(n, to_device, device=0, current=0, pinned=False, fail_record=-1):
        src = np.random.default_rng(n).integers(0, 255, n, dtype=np.uint8)
        dst = np.zeros_like(src)
        host, dev = (src, dst) if to_device else (dst, src)
        res = (ctypes.c_int * 4)()
        lib.run_copy(device, current, int(to_device), host.ctypes.data_as(ctypes.c_void_p),
                     dev.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(n), int(pinned), fail_record, res)
        return dict(error=res[0], copies=res[1], in_flight=res[2], device=res[3], equal=np.array_equal(src, dst))
    return run


@pytest.mark.parametrize("to_device", [True, False])
def test_from_another_current_device(run_copy, to_device):
    """A context's copies work from a thread whose current device is another one, and leave it
    that way."""
    r = run_copy(48 * MB + 13, to_device, device=1, current=0)
    assert r["error"] == 0 and r["equal"] and r["in_flight"] == 0
    assert r["copies"] > 1 and r["device"] == 0


@pytest.mark.parametrize("n,to_device,nth", [
    (9 * MB, False, 0), (9 * MB, False, 2), (9 * MB, False, 4),      # one thread, five chunks
    (48 * MB, False, 5), (48 * MB, True, 0), (48 * MB, True, 23),    # several threads
])
def test_failed_record_leaves_no_copy_in_flight(run_copy, n, to_device, nth):
    """A copy that the runtime took but whose event it did not is waited for before the slot is
    free for the next caller."""
    r = run_copy(n, to_device, fail_record=nth)
    assert r["error"] != 0 and r["in_flight"] == 0


@pytest.mark.parametrize("n,to_device,pinned,staged", [
    (8 * MB, True, False, False),      # the runtime's own upload is the faster one up to here
    (48 * MB, True, False, True),
    (1 * MB, False, False, False),
    (8 * MB, False, False, True),      # its download is not
    (48 * MB, True, True, False),      # pinned memory needs no staging
    (48 * MB, False, True, False),
])
def test_which_copies_are_staged(run_copy, n, to_device, pinned, staged):
    r = run_copy(n, to_device, pinned=pinned)
    assert r["error"] == 0 and r["equal"] and r["in_flight"] == 0
    assert (r["copies"] > 1) == staged
