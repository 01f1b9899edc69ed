"""Phases of one to thousands of reactions: up to 1,024 are put in order by
one workgroup and rounds of up to 2,048 proposals settled by one, larger ones
by the sort, the scans and a grid.  Whatever the size, the reactions of an
iteration come in (replica, mover id) order, their products take consecutive
ids per replica, and no reactant reacts twice."""
import os
import threading

import numpy as np
import pytest

from mcell_amd import workloads as W
from mcell_amd.engine import DiffuseReactEngine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,replicas,precision", [(40, 1, "fp64"), (3000, 1, "fp32"), (60000, 1, "fp64"),
                                                  (20000, 5, "fp32")])
def test_order_and_ids_of_batches(gpu_available, n, replicas, precision):
    wl = W.bimol_box(n_a=n, n_b=n, seed=12, num_replicas=replicas, rate=1e9)
    eng = DiffuseReactEngine.from_workload(wl, precision=precision, log_capacity=1 << 20)
    next_id = np.full(replicas, 2 * n)
    gone = [set() for _ in range(replicas)]
    sizes = []
    for it in range(60):
        st = eng.step(it, 1)
        log = eng.rxn_log()
        assert st.reactions == len(log)
        sizes.append(len(log))
        key = log["replica"].astype(np.uint64) << np.uint64(32) | log["mover_id"]
        assert np.all(key[1:] > key[:-1])  # C reacts with nothing: an iteration's reactions are one phase
        for r in range(replicas):
            e = log[log["replica"] == r]
            assert np.array_equal(e["first_product_id"], next_id[r] + np.arange(len(e)))
            next_id[r] += len(e)
            used = np.concatenate([e["mover_id"], e["partner_id"]])
            assert len(set(used.tolist())) == len(used) and not gone[r] & set(used.tolist())
            gone[r] |= set(used.tolist())
    counts = eng.count_species(replicas, 3)
    reacted = next_id - 2 * n
    assert np.array_equal(counts[:, 0], n - reacted) and np.array_equal(counts[:, 2], reacted)
    assert np.array_equal(eng.next_molecule_ids(), next_id)
    assert n < 20000 or (max(sizes) > 2048 and min(sizes) < 1024)  # both ways, and the sizes between them
    eng.close()


def test_statistics_of_short_and_long_calls(gpu_available):
    """The counters of 60 calls of one iteration add up to those of one call,
    reflections of movers that then react among them (those are counted where
    the claims are settled, the last thing an iteration does)."""
    wl = W.receptor_sphere(n_l=20000, n_r=4000, n_t=2000, iterations=60, seed=8, down_fraction=0.0)
    runs = []
    for calls in ([(it, 1) for it in range(60)], [(0, 60)]):
        eng = DiffuseReactEngine.from_workload(wl, seed=2)
        st = [eng.step_raw(it, num, 100.0 - it) for it, num in calls]
        total = {f: sum(getattr(s, f) for s in st) for f in ("molecule_steps", "wall_hits", "reactions",
                                                             "transparent_crossings", "settle_rounds")}
        m = eng.molecules()
        runs.append((total, st[-1].slow_path_last, {k: v[np.argsort(m["id"])] for k, v in m.items()}))
        eng.close()
    assert runs[0][:2] == runs[1][:2]
    assert runs[0][0]["reactions"] > 0 and runs[0][0]["wall_hits"] > 0
    for k in runs[0][2]:
        assert np.array_equal(runs[0][2][k], runs[1][2][k]), k


def test_contexts_in_threads_on_one_core(gpu_available):
    """Six contexts, each driven by a thread of its own, all on one core: each
    gives the run it gives alone."""
    wl = W.bimol_box(n_a=3000, n_b=3000, seed=9, rate=1e9)

    def run(seed):
        eng = DiffuseReactEngine.from_workload(wl, seed=seed)
        st = eng.step_raw(0, 100, 100.0)
        m = eng.molecules()
        eng.close()
        o = np.argsort(m["id"])
        return st.reactions, m["id"][o], m["pos"][o]

    alone = [run(k) for k in range(6)]
    got = [None] * 6
    cores = os.sched_getaffinity(0)

    def drive(k):
        got[k] = run(k)

    try:
        os.sched_setaffinity(0, {min(cores)})
        threads = [threading.Thread(target=drive, args=(k,)) for k in range(6)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        os.sched_setaffinity(0, cores)
    for a, b in zip(alone, got):
        assert a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
