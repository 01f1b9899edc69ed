"""Full steps run by teams of lanes (finely meshed surfaces, wall lists of
hundreds of entries) and the light pass through the boxes of groups of
entries, which come with them.

* Every proposal and position of the snapshot mode (FP64) equals the oracle's
  with the same draws, from a handful of movers (teams of 64 lanes) to more
  than 65,536 (one lane each).
* A full run with teams equals the same run by single lanes bit for bit, in
  both precisions and both drain forms: first moves, reruns, product moves,
  deferred exact_disk steps, surface tiles.
"""
import dataclasses

import numpy as np
import pytest

from mcell_amd import model as M
from mcell_amd import workloads as W
from mcell_amd.engine import DiffuseReactEngine

pytestmark = pytest.mark.gpu


def mean_list(eng, num_walls):
    """The mean list length over the wall list entries: from 64 on the full
    steps are run by teams."""
    _, off, idx = eng.wall_data(num_walls)
    length = np.diff(off.astype(np.int64))
    return float((length * length).sum()) / len(idx)


@pytest.mark.parametrize("n", [1, 65, 3001, 120000, 700000])
def test_team_steps_match_oracle(gpu_available, oracle_lib, n):
    from oracle import pyoracle as po
    seed, iterations = 23, 3
    wl = W.crowded_spheres(n_molecules=n, n_surface=min(max(n // 4, 1), 30000), num_spheres=2, cube_um=1.0, iterations=iterations)
    wl = dataclasses.replace(wl, unimol_rxns=[], rxns=[M.BimolReaction(0, 1, 1e9, [2])],
                             volsurf_rxns=[M.VolSurfReaction(0, 3, 1e9, 4, product_orient=1, geom_vol=0, geom_surf=1)])
    eng = DiffuseReactEngine.from_workload(wl, seed=seed, propose_only=True, log_capacity=1 << 20)
    assert mean_list(eng, len(wl.walls)) >= 64  # teams
    w = po.world_from_workload(wl, draw_mode=po.DRAW_PHILOX, seed=seed)
    w.set_snapshot(True)
    w.set_barrier_interval(wl.barrier_interval)
    for it in range(iterations):
        st = eng.step(it, 1)
        print("%d molecules: %d full steps" % (n, st.slow_path_last), flush=True)
        # 2,048 waves of 64 lanes for the list: one lane a mover from 65,537 on
        assert n < 700000 or st.slow_path_last > 65536
        w.run(1)
        g = eng.rxn_log()
        u, rx, d = w.rxn_log()
        w.lib.orc_clear_rxn_log(w.w)
        g = g[np.argsort(g["mover_id"], kind="stable")]
        o = np.argsort(u[:, 1], kind="stable") if len(u) else np.zeros(0, int)
        assert len(g) == len(o)
        if len(g):
            assert np.array_equal(g["mover_id"], u[o, 1]) and np.array_equal(g["partner_id"], u[o, 2])
            assert np.array_equal(g["rxn"], rx[o].astype(np.uint32))
            assert np.abs(g["time"] - d[o, 0]).max() <= 1e-12
        m, om = eng.molecules(), w.molecules()
        live = np.nonzero(((om["flags"] & 1) == 0) & (om["species"] < 3))[0]
        oo = np.argsort(m["id"], kind="stable")
        assert np.array_equal(m["id"][oo], live)
        # FP64 steps in the reference's operation order: equal up to the C
        # library's functions in the Ziggurat's wedge and tail (1e-12 relative, positions below 1000 units)
        assert np.abs(m["pos"][oo] - om["pos"][live]).max() <= 1e-9
    w.close()
    eng.close()


def with_fine_speck(wl):
    """The workload with a sphere of 20,480 triangles and 0.03 um radius in an
    empty corner of its cube, behind all other walls: no molecule comes near
    it, but the mean wall list grows past the teams' line."""
    h = wl.vertices.max() / wl.part.rcp_length_unit
    corners = np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)]) * (h - 0.05)
    free = [min(np.linalg.norm(c - s[:3]) - s[3] for s in wl.spheres) for c in corners]
    c = corners[int(np.argmax(free))]
    assert max(free) > 0.5
    ball = M.create_icosphere("speck", 0.03, 6)
    v = (ball.vertices() + c) * wl.part.rcp_length_unit
    w = ball.walls().astype(np.uint32) + np.uint32(len(wl.vertices))
    return c, dataclasses.replace(wl, vertices=np.concatenate([wl.vertices, v]), walls=np.concatenate([wl.walls, w]),
                                  wall_class=np.concatenate([wl.wall_class, np.zeros(len(w), wl.wall_class.dtype)]))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,drain,half_steps", [(1500, "defer", False), (300000, "defer", False),
                                                (300000, "inline", False), (300000, "defer", True)])
def test_teams_give_the_run_of_single_lanes(gpu_available, n, drain, half_steps, precision):
    """half_steps: A and B step twice an iteration, so that lists of some
    270,000 movers take the small exact_disk pool and defer to the large one."""
    wl = W.crowded_spheres(n_molecules=n, n_surface=n // 10, num_spheres=8, sphere_subdivisions=5)
    if half_steps:
        wl = W.with_time_steps(wl, [0.5, 0.5, 1, 1, 1])
    corner, fine = with_fine_speck(wl)
    # nothing within 0.5 um of the speck (12 iterations: 0.05 um rms per axis)
    keep = np.linalg.norm(wl.positions / wl.part.rcp_length_unit - corner, axis=1) > 0.5
    cut = dict(ids=wl.ids[keep], mol_species=wl.mol_species[keep], positions=wl.positions[keep],
               replica=wl.replica[keep])
    runs = []
    for x, teams in ((dataclasses.replace(wl, **cut), False), (dataclasses.replace(fine, **cut), True)):
        eng = DiffuseReactEngine.from_workload(x, precision=precision, seed=6, drain=drain)
        assert (mean_list(eng, len(x.walls)) >= 64) == teams
        st = eng.step(0, 12)
        m = eng.molecules()
        o = np.argsort(m["id"], kind="stable")
        s = eng.surface_molecules()
        so = np.argsort(s["id"], kind="stable")
        print("%s %s %d, teams %d: %d reactions, %d rounds, %d reflections, %d full steps"
              % (precision, drain, n, teams, st.reactions, st.settle_rounds, st.wall_hits, st.slow_path_last), flush=True)
        runs.append(({k: v[o] for k, v in m.items()}, {k: np.asarray(v)[so] for k, v in s.items()},
                     (st.molecule_steps, st.wall_hits, st.reactions, st.settle_rounds, st.slow_path_last, st.drain_form)))
        eng.close()
    a, b = runs
    assert a[2] == b[2]
    assert n < 300000 or a[2][2] > 100
    for part in (0, 1):
        assert a[part].keys() == b[part].keys()
        for k in a[part]:
            assert np.array_equal(a[part][k], b[part][k]), k
