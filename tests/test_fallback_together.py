"""Counting builds that fall back to sorting, several at a time.

The fallback's workgroups wait for each other's stages.  Contexts that fall back together
share the card, so a build must end with whatever part of its workgroups runs: pieces are
drawn in order and wait only for earlier ones.  Eight contexts of two replicas and 118 tiles
of keys each, driven by a thread each, with a cell of 65 beads (one more than a bucket) in
every build; the order must be the incremental re-sort's.
"""
import threading

import numpy as np
import pytest

import softmold_amd as sm
from conftest import gpu_available
from test_counting_build import _system

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs the MI355X")]

CONTEXTS, BUILDS = 8, 12


def test_contexts_fall_back_together():
    n = 120000
    print(f"case {CONTEXTS} contexts of 2 x {n} beads, {BUILDS} sorted builds each", flush=True)
    ds = [_system(n, (45, 45, 45), k) for k in (1, 2)]
    for d in ds:
        rng = np.random.default_rng(7)
        d["pos"][rng.permutation(n)[:65]] = (1.1 + 0.8 * rng.random((65, 3))) * d["cutoff"]
    pos = np.concatenate([d["pos"] for d in ds])

    ref = sm.Solver.batch(ds)
    ref.tune("sort_mode", 1)
    ref.init_forces()
    want = ref.download()
    ref.close()

    solvers = [sm.Solver.batch(ds) for _ in range(CONTEXTS)]
    out, start = [None] * CONTEXTS, threading.Barrier(CONTEXTS)

    def work(k):
        s = solvers[k]
        start.wait()
        try:
            for _ in range(BUILDS):
                s.upload(pos=pos)
                s.init_forces()
            out[k] = (s.download(), s.tune_get("sort_count_path"))
        except sm.SmError as e:
            out[k] = e

    team = [threading.Thread(target=work, args=(k,)) for k in range(CONTEXTS)]
    for t in team:
        t.start()
    for t in team:
        t.join()
    for o in out:
        assert not isinstance(o, Exception), o
        assert o[1] == 0
        for x, y in zip(o[0], want):
            assert np.array_equal(x, y)
    for s in solvers:
        s.close()
