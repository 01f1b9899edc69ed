"""Phases of one to thousands of reactions: up to 1,024 are put in order by
one workgroup and rounds of up to 2,048 proposals settled by one, larger ones
by the sort, the scans and a grid.  Whatever the size, the reactions of an
iteration come in (replica, mover id) order, their products take consecutive
ids per replica, and no reactant reacts twice."""
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
