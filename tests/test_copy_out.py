"""The copy of device results to the caller's memory (copyout.hpp) over
runtime calls on the host (tests/native/copycheck.cpp): every size's bytes,
and what a caller with several devices or a system out of memory, events or
threads is left with."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MB = 1 << 20
SIZES = [1, 4 * MB - 1, 4 * MB, 8 * MB, 8 * MB + 1, 13 * MB + 4567]   # the plain copy, its edge, the ring with and without refills


@pytest.fixture(scope="module")
def copy(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("copy") / "libcopycheck.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-pthread", os.path.join(HERE, "native", "copycheck.cpp"),
                    "-o", so], check=True)
    L = C.CDLL(so)
    L.cc_copy.argtypes = [C.c_long] + [C.c_int] * 7 + [C.POINTER(C.c_int)]

    def run(n, dev=0, caller=0, bad_event=-1, bad_thread=-1, bad_kind=0, again=1, known=0):
        out = (C.c_int * 7)()
        L.cc_copy(n, dev, caller, bad_event, bad_thread, bad_kind, again, known, out)
        return dict(zip(("error", "copied", "device", "events", "pinned", "waits", "copies"), out))
    return run


@pytest.mark.parametrize("n", SIZES)
def test_callers_device_stays(copy, n):
    """A context on device 0 called from a thread whose device is 1."""
    r = copy(n, dev=0, caller=1)
    assert (r["error"], r["copied"], r["device"]) == (0, 1, 1)
    assert r["events"] == 0 and r["pinned"] == 0


@pytest.mark.parametrize("bad", [0, 3, 7])
def test_no_events_left_when_one_cannot_be_made(copy, bad):
    """The plain copy takes over, and neither buffers nor events stay."""
    r = copy(13 * MB + 4567, bad_event=bad, again=0)
    assert (r["error"], r["copied"]) == (0, 1)
    assert (r["events"], r["pinned"]) == (0, 0)


def test_ring_opened_after_a_failed_attempt(copy):
    r = copy(13 * MB + 4567, bad_event=3, again=2)
    assert (r["error"], r["copied"]) == (0, 1)
    assert (r["events"], r["pinned"]) == (0, 0)


@pytest.mark.parametrize("kind", ["no thread", "no memory"])
@pytest.mark.parametrize("started", [0, 1, 2])
def test_threads_that_cannot_be_started(copy, kind, started):
    """The calling thread does their share; nothing leaves the C entry."""
    r = copy(13 * MB + 4567, bad_thread=started, bad_kind=["no thread", "no memory"].index(kind) + 1, again=0)
    assert (r["error"], r["copied"]) == (0, 1)
    assert (r["events"], r["pinned"]) == (0, 0)


@pytest.mark.parametrize("n", SIZES)
def test_memory_the_runtime_knows_is_copied_to_at_once(copy, n):
    """Pinned and device memory: one transfer by the runtime, no thread writes there."""
    r = copy(n, again=0, known=1)
    assert (r["error"], r["copied"], r["copies"], r["waits"]) == (0, 1, 1, 1)


@pytest.mark.parametrize("n", [2, 3200, 4 * MB])
def test_two_small_results_wait_once(copy, n):
    """The results of one call, each below the chunked copy's smallest size."""
    r = copy(n, again=-1)
    assert (r["error"], r["copied"], r["waits"]) == (0, 1, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["pinned", "device"])
@pytest.mark.parametrize("cells", [(8, 6, 6), (40, 40, 40)])
def test_results_into_pinned_and_device_memory(pkg, where, cells):
    """A state and a residual of under and over the chunked copy's smallest size (4 MB), straight into the caller's memory."""
    import torch
    case = pkg.cases.bump_case(*cells, True, True, 4, 2, 8)
    s = pkg.Solver(case)
    s.put_state(0, *case.init[0])
    s.setbc()
    f8 = C.POINTER(C.c_double)
    pv, res = s.get_state(0)[0], s.calrhs(0)[0]
    assert (res.nbytes >= 4 * MB) == (cells[0] == 40)

    def memory(n):
        t = torch.zeros(n, dtype=torch.float64)
        return t.pin_memory() if where == "pinned" else t.cuda()
    a, b = memory(pv.size), memory(res.size)
    torch.cuda.synchronize()
    assert pkg.lib().cav3d_get_state(s.h, 0, C.cast(a.data_ptr(), f8), None, None, None) == 0
    assert pkg.lib().cav3d_calrhs(s.h, 0.0, 0, C.cast(b.data_ptr(), f8), None, None, None) == 0
    assert a.cpu().numpy().tobytes() == pv.tobytes() and b.cpu().numpy().tobytes() == res.tobytes()
    s.close()
