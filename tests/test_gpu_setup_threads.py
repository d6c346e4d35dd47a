"""Matrices of one context made by several threads at once: the counts that
each reads back from the device are its own."""
import threading

import numpy as np
import pytest

from faspxx_amd import fx
from faspxx_amd import problems as P

pytestmark = pytest.mark.gpu


def results(ctx, A):
    M = fx.Csr.from_problem(ctx, A)
    out = []
    for C in (M.transpose(), fx.Csr.mult(M, M), fx.Csr.add(1.0, M, 0.5, M), M.lower_tri()):
        out += [a for a in C.download() if a is not None]
    return out


def test_matrices_made_by_several_threads(ctx):
    systems = [P.poisson2d(7), P.poisson2d(40), P.poisson3d(12), P.convdiff2d(61)]
    want = [results(ctx, A) for A in systems]
    bad = []

    def work(k):
        try:
            for _ in range(20):
                got = results(ctx, systems[k])
                if not all(np.array_equal(a, b) for a, b in zip(got, want[k])):
                    bad.append(k)
        except Exception as e:  # noqa: BLE001 -- reported below
            bad.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(systems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
