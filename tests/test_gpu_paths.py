"""The routes that a pass takes by its sizes, each against the FP64 oracle (or, for
the downloads, against the other route): lanes per particle, candidate rows and
walks, remainders of the lane groups, rounds of deferred pairs, pinned and
ordinary memory."""
import ctypes as C

import numpy as np
import pytest
import torch

import gzm
import ics
import oracle as O
from parity import check_pass

pytestmark = pytest.mark.gpu


def params_for(ic, **kw):
    return gzm.make_params(box=tuple(ic["box"]) if "box" in ic else (1.0, 1.0, 1.0), **kw)


def counts_match(gst, st):
    assert gst["density_sweeps"] == st.iterations
    assert gst["density_interactions"] == st.dens_interactions
    assert gst["gradient_interactions"] == st.grad_interactions
    assert gst["force_interactions"] == st.force_interactions
    assert gst["exact_solver_calls"] == st.exact_solver_calls


@pytest.mark.parametrize("n_active", [65536, 65537])
def test_lanes_per_particle_on_both_sides_of_the_line(n_active):
    ic = ics.lattice_gaussian(41)
    active = np.random.default_rng(3).permutation(ic["mass"].size)[:n_active].astype(np.int32)
    ref, st, _ = O.run_pass(ic, active=active)
    out, gst = gzm.run_pass(ic, active=active)
    counts_match(gst, st)
    errs, bad = check_pass(out, ref, active)
    assert not bad, bad


@pytest.mark.parametrize("search", [0, 1])
@pytest.mark.parametrize("n_clump", [60, 97, 700, 6000])
def test_clump_in_a_sparse_set(search, n_clump):
    """Particles whose candidates pass the row cap (96), the candidate budget
    (512) and the width of a shared walk's stack: a clump in a sparse set, with
    first guesses of hsml that reach into it.  The largest clump has no mass: it
    is walked, but where thousands of masses lie just inside or outside h the
    hsml iteration turns on the rounding of their sum, in the oracle as here."""
    rng = np.random.default_rng(n_clump)
    n_bg = 2000
    pos = np.concatenate([rng.uniform(0, 1, (n_bg, 3)), 0.37 + 0.01 * rng.normal(size=(n_clump, 3))])
    n = pos.shape[0]
    ic = dict(pos=pos, vel=0.1 * rng.normal(size=(n, 3)), mass=np.full(n, 1.0 / n), u=1 + 0.1 * rng.uniform(size=n),
              hsml=ics.local_hsml(pos) * 1.4, cn=np.ones(n), box=np.ones(3))
    ic["hsml"][:3] = 0.45
    if n_clump == 6000:
        ic["mass"][n_bg:] = 0
    ref, st, _ = O.run_pass(ic)
    out, gst = gzm.run_pass(ic, params=params_for(ic, search=search))
    counts_match(gst, st)
    errs, bad = check_pass(out, ref)
    assert not bad, bad


@pytest.mark.parametrize("n_active", [1, 7, 8, 9, 63, 65])
@pytest.mark.parametrize("search", [0, 1])
def test_remainders_of_the_lane_groups(n_active, search):
    ic = ics.random_state(12)
    active = np.arange(5, 5 + n_active, dtype=np.int32)
    full, _ = gzm.run_pass(ic)
    for k in ("hsml", "num_ngb", "dhsml", "divvel", "density", "pressure", "nvt", "cn", "fce", "grad_rho", "grad_p",
              "grad_v"):
        ic[k] = full[k]
    ref, st, _ = O.run_pass(ic, active=active)
    out, gst = gzm.run_pass(ic, active=active, params=params_for(ic, search=search))
    counts_match(gst, st)
    errs, bad = check_pass(out, ref, active)
    assert not bad, bad


@pytest.mark.parametrize("precision", [0, 1])
def test_deferred_pairs_past_the_first_round(precision):
    """More exact-solver pairs than the buffer first holds (65,536): the pass
    takes a second round.  The next one, with the buffer grown, takes one, and
    gives the same bits."""
    ic = ics.random_state(42)
    ic["vel"] = 60 * ic["vel"]
    with gzm.MFMContext(params_for(ic, precision=precision)) as ctx:
        ctx.upload(ic)
        outs, calls = [], []
        for _ in range(2):
            ctx.restore_initial_state()
            ctx.density()
            ctx.gradients()
            calls.append(ctx.hydro_force().exact_solver_calls)
            outs.append(ctx.download())
    assert calls[0] == calls[1] > 65536
    for k in ("acc", "dtu", "vsig"):
        np.testing.assert_array_equal(outs[1][k], outs[0][k])
    if precision == 0:
        ref, st, _ = O.run_pass(ic)
        assert calls[0] == st.exact_solver_calls
        errs, bad = check_pass(outs[0], ref)
        assert not bad, bad


@pytest.mark.parametrize("side", [9, 50])
def test_downloads_into_pinned_and_ordinary_memory_agree(side):
    """Side 9: ordinary arrays through the context's pinned array; side 50 (37 MB
    in all): through a copy each.  Pinned arrays are written by the device."""
    rng = np.random.default_rng(side)
    n = side ** 3
    ic = ics.lattice_gaussian(side)
    for k, w in (("vsig", 1), ("num_ngb", 1), ("dhsml", 1), ("divvel", 1), ("density", 1), ("pressure", 1), ("fce", 1),
                 ("dtu", 1), ("acc", 3), ("grad_rho", 3), ("grad_p", 3)):
        ic[k] = rng.normal(size=(n, w)).squeeze(-1) if w == 1 else rng.normal(size=(n, w))
    ic["grad_v"] = rng.normal(size=(n, 3, 3))
    t = rng.normal(size=(n, 3, 3))
    ic["nvt"] = np.ascontiguousarray((t + t.transpose(0, 2, 1)).reshape(n, 9))
    fields = ("hsml", "cn", "vsig", "num_ngb", "dhsml", "divvel", "density", "pressure", "fce", "dtu", "acc", "nvt",
              "grad_rho", "grad_p", "grad_v")
    with gzm.MFMContext(params_for(ic)) as ctx:
        ctx.upload(ic)
        out = ctx.download()
        view, pinned = gzm.HostView(), {}
        view.n = n
        for q, k in enumerate(fields):
            a = torch.empty(out[k].size, dtype=torch.float64, pin_memory=q % 3 != 2).numpy()
            pinned[k] = a
            setattr(view, k, a.ctypes.data_as(C.POINTER(C.c_double)))
        assert ctx.L.gzm_download(ctx.ctx, C.byref(view)) == 0
    for k in fields:
        np.testing.assert_array_equal(pinned[k], out[k].reshape(-1), err_msg=k)
        if k in ic:
            np.testing.assert_array_equal(out[k].reshape(-1), np.asarray(ic[k]).reshape(-1), err_msg=k)


def test_download_into_device_memory_and_into_part_of_a_pinned_array():
    ic = ics.lattice_gaussian(9)
    n = 9 ** 3
    with gzm.MFMContext(params_for(ic)) as ctx:
        ctx.upload(ic)
        out = ctx.download()
        on_card = torch.zeros(n, dtype=torch.float64, device="cuda")
        pinned = torch.zeros(n + 12, dtype=torch.float64, pin_memory=True)
        torch.cuda.synchronize()
        view = gzm.HostView()
        view.n = n
        view.hsml = C.cast(C.c_void_p(on_card.data_ptr()), C.POINTER(C.c_double))
        view.cn = C.cast(C.c_void_p(pinned[5:].data_ptr()), C.POINTER(C.c_double))
        assert ctx.L.gzm_download(ctx.ctx, C.byref(view)) == 0
    np.testing.assert_array_equal(on_card.cpu().numpy(), out["hsml"])
    np.testing.assert_array_equal(pinned[5:5 + n].numpy(), out["cn"])
    assert not pinned[:5].any() and not pinned[5 + n:].any()
