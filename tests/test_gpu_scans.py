"""The scans of the light pass and the full step: moves across many small
subpartitions (sets of subpartitions that leave the window of the set's bits,
rows of cells in several batches, moves beyond the bit of the cells without
walls around them) and species tables too large for LDS."""
import dataclasses

import numpy as np
import pytest

from mcell_amd import model as M
from mcell_amd import workloads as W
from mcell_amd.engine import DiffuseReactEngine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge,d", [(0.02, 5e-6), (0.02, 1e-6), (0.05, 5e-6), (0.2, 1e-6)])
def test_scans_match_oracle(gpu_available, oracle_lib, edge, d):
    """Every proposal and position of three snapshot iterations equals the
    oracle's: steps of 1.4 to 3.2 units per axis, cells of 2 to 20."""
    from oracle import pyoracle as po
    wl = W.bimol_box(n_a=15000, n_b=15000, iterations=3, seed=14, rate=1.36e9, subpartition_dimension=edge, d_a=d,
                     d_b=d)
    eng = DiffuseReactEngine.from_workload(wl, seed=19, propose_only=True, log_capacity=1 << 16)
    w = po.world_from_workload(wl, draw_mode=po.DRAW_PHILOX, seed=19)
    w.set_snapshot(True)
    w.set_barrier_interval(wl.barrier_interval)
    total = 0
    for it in range(wl.iterations):
        eng.step(it, 1)
        w.run(1)
        g = eng.rxn_log()
        u, _, t = w.rxn_log()
        w.lib.orc_clear_rxn_log(w.w)
        g = g[np.argsort(g["mover_id"], kind="stable")]
        o = np.argsort(u[:, 1], kind="stable")
        assert np.array_equal(g["mover_id"], u[o, 1]) and np.array_equal(g["partner_id"], u[o, 2])
        assert np.abs(g["time"] - t[o, 0]).max(initial=0) <= 1e-12
        m = eng.molecules()
        assert np.abs(m["pos"][np.argsort(m["id"])] - w.molecules()["pos"]).max() <= 1e-10
        total += len(g)
    assert total > 30
    w.close()
    eng.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_many_species(gpu_available, precision):
    """17 species (the pair table stays in memory) give the run of three."""
    wl = W.bimol_box(n_a=4000, n_b=4000, iterations=20, seed=3, rate=1e9)
    more = dataclasses.replace(wl, species=wl.species + [M.Species("X%d" % k, 1e-6) for k in range(14)])
    more.species_steps = W._species_table(more.species, more.part, more.rxns)
    got = []
    for x in (wl, more):
        eng = DiffuseReactEngine.from_workload(x, precision=precision)
        st = eng.step(0, x.iterations)
        m = eng.molecules()
        o = np.argsort(m["id"])
        got.append((st.reactions, {k: v[o] for k, v in m.items()}))
        eng.close()
    assert got[0][0] == got[1][0] > 100
    for k in got[0][1]:
        assert np.array_equal(got[0][1][k], got[1][1][k]), k


@pytest.mark.parametrize("n_a,n_b", [(1, 0), (1, 1), (1024, 1024), (1025, 1024), (65536, 65536), (65537, 65536),
                                     (64512, 64512), (64513, 64512)])
def test_waves_shares_of_the_light_pass(gpu_available, oracle_lib, n_a, n_b):
    """One molecule a wave up to 2,048, a full wave from 129,025 on: the
    positions after two snapshot iterations equal the oracle's."""
    from oracle import pyoracle as po
    wl = W.bimol_box(n_a=n_a, n_b=n_b, iterations=2, seed=4)
    eng = DiffuseReactEngine.from_workload(wl, seed=5, propose_only=True, log_capacity=1 << 12)
    w = po.world_from_workload(wl, draw_mode=po.DRAW_PHILOX, seed=5)
    w.set_snapshot(True)
    w.set_barrier_interval(wl.barrier_interval)
    eng.step(0, 2)
    w.run(2)
    m = eng.molecules()
    assert len(m["id"]) == n_a + n_b
    assert np.abs(m["pos"][np.argsort(m["id"])] - w.molecules()["pos"]).max() <= 1e-10
    w.close()
    eng.close()


@pytest.mark.parametrize("n", [1, 100, 3000])
def test_few_molecules_in_many_bins(gpu_available, oracle_lib, n):
    """Some 4e5 bins for up to 6,000 molecules: the scatter's grid is sized by
    the bins it clears, and every iteration finds them cleared."""
    from oracle import pyoracle as po
    wl = W.bimol_box(n_a=n, n_b=n, iterations=5, seed=4, subpartition_dimension=0.02)
    eng = DiffuseReactEngine.from_workload(wl, seed=5, propose_only=True, log_capacity=1 << 12)
    w = po.world_from_workload(wl, draw_mode=po.DRAW_PHILOX, seed=5)
    w.set_snapshot(True)
    w.set_barrier_interval(wl.barrier_interval)
    st = eng.step_raw(0, 5, 5.0)
    w.run(5)
    m = eng.molecules()
    assert len(m["id"]) == 2 * n and st.molecule_steps == 10 * n
    # FP64 steps in the reference's operation order, as in the other snapshot comparisons
    assert np.abs(m["pos"][np.argsort(m["id"])] - w.molecules()["pos"]).max() <= 1e-10
    w.close()
    eng.close()


@pytest.mark.parametrize("n", [500, 16384, 16385, 20000, 300001])
def test_list_moves_short_and_long(gpu_available, oracle_lib, n):
    """Second half steps of every molecule: lists below and above the length
    up to which the list moves take the large pool at once, and those up to
    which one workgroup copies the list (16,384)."""
    from oracle import pyoracle as po
    wl = W.with_time_steps(W.free_diffusion_box(scale=n / 10000, iterations=4), [0.5])
    eng = DiffuseReactEngine.from_workload(wl)
    w = po.world_from_workload(wl, draw_mode=po.DRAW_PHILOX)
    eng.step(0, 4)
    w.run(4)
    m = eng.molecules()
    got, want = m["pos"][np.argsort(m["id"])], w.molecules()["pos"]
    assert np.abs(got - want).max() <= 1e-10
    w.close()
    eng.close()
