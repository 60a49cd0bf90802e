"""The force loop without the 64-entry lists: no list, and longer lists.  Same pairs,
same order of summation, so the default's bits, also where pairs reach the exact
solver and where inactive neighbours are woken."""
import numpy as np
import pytest

import gzm
import ics
import oracle as O
from parity import check_pass

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("part", [False, True])
@pytest.mark.parametrize("search", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
def test_longer_lists_and_none_give_the_default_bits(precision, search, part):
    ic = ics.random_state(14)
    ic["vel"] = 8 * ic["vel"]
    active = None
    if part:
        full, _ = gzm.run_pass(ic, params=gzm.make_params(precision=precision, search=search))
        for k in ("hsml", "num_ngb", "dhsml", "divvel", "density", "pressure", "nvt", "cn", "fce", "grad_rho", "grad_p",
                  "grad_v"):
            ic[k] = full[k]
        ic["vsig"] = 0.1 * full["vsig"]
        active = ics.random_subset(14 ** 3, 0.3)
    base, bst = gzm.run_pass(ic, active=active, params=gzm.make_params(precision=precision, search=search))
    assert bst["exact_solver_calls"] > 100
    for cap in (-1, 80, 128):
        out, st = gzm.run_pass(ic, active=active,
                               params=gzm.make_params(precision=precision, search=search, pair_list_cap=cap))
        for k in ("force_interactions", "exact_solver_calls", "riemann_retries"):
            assert st[k] == bst[k], (cap, k)
        if cap == -1 and precision == 1 and search == 1:
            continue  # r^2 is FP64's rounded there, and the rounded displacement's in the lists
        for k in ("acc", "dtu", "vsig", "wakeup"):
            np.testing.assert_array_equal(out[k], base[k], err_msg=f"{cap} {k}")
    assert part == bool(base["wakeup"].any())


def force_ms(params, ic, passes=3):
    with gzm.MFMContext(params) as ctx:
        ctx.upload(ic)
        ms = []
        for _ in range(passes):
            ctx.restore_initial_state()
            ctx.density()
            ctx.gradients()
            ctx.timing_reset()
            ctx.hydro_force()
            t = ctx.timing()
            ms.append(t["force_ms"] + t["force_deferred_ms"])
        return float(np.median(ms))


def test_fp32_force_without_lists_keeps_two_waves():
    """FP32 on the tree without lists: 33 times the force loop with them; 67 times
    where the kernel's scratch and registers leave it one wave on a SIMD."""
    ic = ics.random_state(61)
    kw = dict(precision=1, search=1)
    assert force_ms(gzm.make_params(pair_list_cap=-1, **kw), ic) < 45 * force_ms(gzm.make_params(**kw), ic)


@pytest.mark.parametrize("cell_size", [0.02, 0.06, 0.3])
def test_long_pair_sets_in_any_cells(cell_size):
    """Lists of 16 leave nearly all particles to the wavefront loop: cells of less
    than a particle, of one and of a hundred, more than 64 cells and fewer."""
    ic = ics.random_state(13)
    ref, st, _ = O.run_pass(ic)
    out, gst = gzm.run_pass(ic, params=gzm.make_params(cell_size=cell_size, pair_list_cap=16))
    assert gst["force_interactions"] == st.force_interactions
    assert gst["exact_solver_calls"] == st.exact_solver_calls
    errs, bad = check_pass(out, ref)
    assert not bad, bad


def test_long_pair_sets_in_dense_cells_cost_their_candidates():
    """Plummer spheres, thousands of particles in a grid cell: the force stage takes
    as long as with the tree; 100 times and more where a cell is tested anew for
    each 64 pairs."""
    ic = ics.plummer_clusters(32768, 50)
    grid, tree = force_ms(gzm.make_params(), ic), force_ms(gzm.make_params(search=1), ic)
    assert grid < 20 * tree
