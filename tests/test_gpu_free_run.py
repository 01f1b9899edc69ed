"""Free diffusion taken through several iterations by one launch: the same
run, bit for bit, as the passes of single iterations (which a context that
records hit traces takes), at the edges of the waves' shares of molecules and
of the rule that chooses between the two."""
import numpy as np
import pytest

from mcell_amd import _lib
from mcell_amd import workloads as W
from mcell_amd.engine import DiffuseReactEngine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 2047, 2049, 4097, 262144, 262145])
def test_run_equals_single_iterations(gpu_available, n, precision):
    wl = W.free_diffusion_replicas(1, n, seed=31, box_um=0.3, subpartition_dimension=0.05)
    got = {}
    for trace in (False, True):
        eng = DiffuseReactEngine.from_workload(wl, precision=precision, seed=8, trace=trace)
        first = eng.step(0, 1)
        rest = eng.step(1, 24)
        got[trace] = (eng.molecules(), first.wall_hits, rest.wall_hits, first.slow_path_last, rest.slow_path_last,
                      rest.molecule_steps)
        eng.close()
    a, b = got[False], got[True]
    for k in a[0]:
        assert np.array_equal(a[0][k], b[0][k]), k
    assert a[1:] == b[1:]
    assert n < 1000 or a[2] > n // 10  # the box is small enough for steps that meet walls


@pytest.mark.parametrize("action", [1, 2])
def test_run_with_surface_classes(gpu_available, action):
    """Walls that let a species through or absorb it, an absorbed molecule
    ending its run early."""
    wl = W.sphere_in_cube(n_l=3000, n_t=3000, iterations=40, t_action=action, subpartition_dimension=0.1)
    got = []
    for trace in (False, True):
        eng = DiffuseReactEngine.from_workload(wl, trace=trace)
        st = eng.step(0, wl.iterations)
        got.append((eng.molecules(), st.wall_hits, st.transparent_crossings, eng.num_molecules()))
        eng.close()
    for k in got[0][0]:
        assert np.array_equal(got[0][0][k], got[1][0][k]), k
    assert got[0][1:] == got[1][1:]
    assert got[0][2] > 0 if action == 1 else got[0][3] < wl.num_molecules


def test_no_molecules_and_the_longest_call(gpu_available):
    """Nothing to move: a call of 2^32 - 1 iterations launches nothing, ends
    and moves the clock on; the next call is refused as for any other clock."""
    wl = W.free_diffusion_box(scale=0.01)
    eng = DiffuseReactEngine.from_workload(wl, add_molecules=False)
    st = eng.step_raw(0, 2 ** 32 - 1, 2.0 ** 32)
    assert st.molecule_steps == 0 and st.kernel_launches == 0 and eng.num_molecules() == 0
    with pytest.raises(_lib.McgError, match="clock"):
        eng.step_raw(0, 1, 1.0)
    eng.close()
