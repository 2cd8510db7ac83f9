"""The sweeps' tile tickets: more tiles than workgroups, and two contexts
sweeping at once from two threads (each started workgroup's upstream tiles
are taken by running workgroups, so neither waits on the other), give the
bits of a context that runs alone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(pkg, size, seed):
    case = pkg.cases.config2(*size, seed=seed)
    case.params["cav_clip"] = 1
    return case


def _steps(pkg, case, n, out, key):
    s = pkg.Solver(case)
    s.put_state(0, *case.init[0])
    for it in range(n):
        s.timeinteg(1, it + 1, 0.0, want_time=False)
    l2, ijk, rm = s.residual()
    out[key] = (s.get_state(0)[0], l2, ijk, rm)
    s.close()


@pytest.mark.parametrize("size", [(4, 3, 3), (20, 9, 5), (24, 72, 70)])
def test_two_contexts_at_once_match_one_alone(pkg, size):
    cases = [_case(pkg, size, seed) for seed in (2, 3)]
    print(f"sizes {size}", flush=True)
    alone, both = {}, {}
    for q, c in enumerate(cases):
        _steps(pkg, c, 6, alone, q)
    th = [threading.Thread(target=_steps, args=(pkg, c, 6, both, q)) for q, c in enumerate(cases)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for q in range(2):
        for a, b in zip(alone[q], both[q]):
            assert np.array_equal(np.asarray(a), np.asarray(b))
