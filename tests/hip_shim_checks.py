"""Checks that run in hip_shim's process, each called with the shim."""
import ctypes as C

import numpy as np

import gzm
import ics
import oracle as O
from parity import TOL32_DENSITY, TOL32_FLUX, check_mfv, check_pass, error_stats

OUT_KEYS = ("hsml", "density", "grad_v", "acc", "dtu", "vsig")


def one_pass(ctx):
    ctx.restore_initial_state()
    ctx.density()
    ctx.gradients()
    return ctx.hydro_force()


def entry_points_make_their_device_current(shim):
    """every call that may launch or copy on a context's stream sets its device first"""
    with gzm.MFMContext(gzm.make_params()) as ctx:
        calls = [lambda: ctx.upload(ics.random_state(8)), ctx.density, ctx.gradients, ctx.hydro_force,
                 ctx.restore_initial_state, lambda: ctx.run_passes(1), ctx.download, lambda: ctx.neighbor_counts(0)]
        for k, call in enumerate(calls):
            before = shim.set_device_calls
            call()
            assert shim.set_device_calls > before, k


def run_passes_probes_again_without_rows(shim):
    """The probe has no memory for its pair list until it gives up the candidate
    rows: the captured passes, without rows, are probed without them too."""
    ic = ics.random_state(32)
    n = ic["mass"].size
    with gzm.MFMContext(gzm.make_params()) as ctx:
        ctx.upload(ic)
        with_rows = shim.used
        shim.set("budget", with_rows + n)
        ctx.timing_reset()
        st = ctx.run_passes(2)
        assert shim.refused > 0 and shim.used < with_rows + n
        assert ctx.timing()["density_launches"] == 2, "one probe with rows, one without"
        out = ctx.download()
        eager = one_pass(ctx)
        ref = ctx.download()
        assert st.force_interactions == 2 * eager.force_interactions
        for k in OUT_KEYS:
            np.testing.assert_array_equal(out[k], ref[k], err_msg=k)


def run_passes_reports_what_its_probe_did_not_meet(shim, precision):
    """Velocities that rise between the probe and the graph's launch send pairs to the
    exact solver for which the graph has no room."""
    ic = ics.random_state(12)
    n = ic["mass"].size
    with gzm.MFMContext(gzm.make_params(precision=int(precision))) as ctx:
        ctx.upload(ic)
        # the velocities that the force loop reads, FP64 or FP32, after the positions
        v = np.zeros((n, 4), dtype=np.float32 if int(precision) else np.float64)
        velu = [p for p, size in shim.recent() if size == v.nbytes][1]
        copy = shim.hip.hipMemcpy
        copy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]

        def faster():
            assert copy(v.ctypes.data, velu, v.nbytes, 2) == 0
            v[:, :3] *= 60
            assert copy(velu, v.ctypes.data, v.nbytes, 1) == 0

        before = one_pass(ctx)
        shim.before_graph(faster)
        try:
            ctx.run_passes(1)
            raise AssertionError("the incomplete passes were reported as complete")
        except gzm.GzmError as e:
            assert e.status == 4 and "probe" in str(e), e
        # the context goes on with what it holds now
        after = one_pass(ctx)
        again = one_pass(ctx)
        assert after.exact_solver_calls == again.exact_solver_calls > before.exact_solver_calls
        assert after.fp64_force_particles == again.fp64_force_particles


def deferred_buffer_shrinks_before_rows_go(shim):
    """The deferred pairs' buffer, half a pair per particle, has a smaller form: no
    reason to give up the candidate rows, at first or when it has to grow."""
    ic = ics.random_state(64)
    n = ic["mass"].size
    with gzm.MFMContext(gzm.make_params()) as ctx:
        ctx.upload(ic)
        ctx.density()
        ctx.gradients()
        before = shim.used
        shim.set("budget", before + 17 * n + (48 << 16) + 4096)  # per-particle arrays and the smallest buffer
        few = ctx.hydro_force()
        assert shim.refused > 0 and shim.used >= before
        out = ctx.download()
    shim.set("budget", 1 << 62)
    ref, st = gzm.run_pass(ic)
    assert st["exact_solver_calls"] == few.exact_solver_calls > 0
    for k in OUT_KEYS:
        np.testing.assert_array_equal(out[k], ref[k], err_msg=k)


def deferred_buffer_grows_within_what_is_free(shim):
    """More pairs than the buffer holds, and no memory for all of them: rounds."""
    ic = ics.random_state(42)
    ic["vel"] = 60 * ic["vel"]
    n = ic["mass"].size
    with gzm.MFMContext(gzm.make_params()) as ctx:
        ctx.upload(ic)
        ctx.density()
        ctx.gradients()
        before = shim.used
        shim.set("budget", before + 17 * n + (48 << 16) + 4096)
        many = ctx.hydro_force()
        assert shim.refused > 0 and shim.used >= before
        out = ctx.download()
    shim.set("budget", 1 << 62)
    ref, st = gzm.run_pass(ic)
    assert st["exact_solver_calls"] == many.exact_solver_calls > 1 << 16
    for k in OUT_KEYS:
        np.testing.assert_array_equal(out[k], ref[k], err_msg=k)


def rows_come_back_with_the_memory(shim):
    """Rows given up for want of memory are there again after an upload that finds it,
    and are not asked for while it is short."""
    ic = ics.random_state(32)
    n = ic["mass"].size
    ref, _ = gzm.run_pass(ic)
    with gzm.MFMContext(gzm.make_params()) as ctx:
        ctx.upload(ic)
        with_rows = shim.used
        shim.set("budget", with_rows + n)
        one_pass(ctx)
        given_up = shim.used
        assert shim.refused > 0 and given_up < with_rows + n
        ctx.upload(ic)
        assert shim.used == given_up
        refused = shim.refused
        ctx.upload(ic)
        assert shim.used == given_up and shim.refused == refused
        shim.set("budget", 1 << 62)
        ctx.upload(ic)
        assert shim.used == given_up + 412 * n
        one_pass(ctx)
        out = ctx.download()
    for k in OUT_KEYS:
        np.testing.assert_array_equal(out[k], ref[k], err_msg=k)


def params_of(ic, method=0, **kw):
    return dict(gpu=gzm.make_params(method=method, **kw), oracle=O.make_params(method=method))


def without_rows(shim, side, search, method):
    """A context that never gets candidate rows: density from the tail's and the walk's
    kernels, gradients from walks, hsml well guessed, poorly guessed and of a part,
    against the oracle; the passes of a graph against the eager one."""
    side, search, method = int(side), int(search), int(method)
    check = check_mfv if method else check_pass
    ic = ics.random_state(side)
    n = ic["mass"].size
    shim.set("unwanted", 96 * 4 * n)
    poor = dict(ic, hsml=ic["hsml"] * (0.6 + 1.2 * ics.uniform(5, 1, n)))
    for which, s in (("good", ic), ("poor", poor)):
        p = params_of(s, method=method, search=search)
        refused = shim.refused
        ref, st, _ = O.run_pass(s, p["oracle"])
        with gzm.MFMContext(p["gpu"]) as ctx:
            ctx.upload(s)
            assert shim.refused > refused, "no rows asked for"
            d, g, f = ctx.density(), ctx.gradients(), ctx.hydro_force()
            out = ctx.download()
            assert (d.density_sweeps, d.density_interactions, g.gradient_interactions, f.force_interactions,
                    f.exact_solver_calls) == (st.iterations, st.dens_interactions, st.grad_interactions,
                                              st.force_interactions, st.exact_solver_calls), which
            errs, bad = check(out, ref)
            assert not bad, (which, bad)
            if method == 0:
                ctx.restore_initial_state()
                ctx.run_passes(2)
                again = ctx.download()
                for k in OUT_KEYS:
                    np.testing.assert_array_equal(again[k], out[k], err_msg=f"{which} {k}")
    if method:
        return
    state = dict(ic)
    for k in ("hsml", "num_ngb", "dhsml", "divvel", "density", "pressure", "nvt", "cn", "fce", "grad_rho", "grad_p",
              "grad_v"):
        state[k] = out[k]
    active = ics.random_subset(n, 0.4)
    ref, st, _ = O.run_pass(state, active=active)
    part, gst = gzm.run_pass(state, active=active, params=gzm.make_params(search=search))
    assert gst["density_interactions"] == st.dens_interactions
    assert gst["force_interactions"] == st.force_interactions
    errs, bad = check_pass(part, ref, active)
    assert not bad, bad
    ref, st, _ = O.run_pass(ic)
    half, gst = gzm.run_pass(ic, params=gzm.make_params(search=search, precision=1))
    assert gst["density_interactions"] == st.dens_interactions
    assert gst["force_interactions"] == st.force_interactions
    es = error_stats(half, ref)
    for k in ("density", "hsml", "pressure"):
        assert es[k]["max"] <= TOL32_DENSITY, (k, es[k])
    for k in ("acc", "dtu"):
        assert es[k]["max"] <= TOL32_FLUX, (k, es[k])


def rows_given_up_between_stages(shim, search):
    """Rows that served the density stage and are gone at the gradients."""
    ic = ics.random_state(32)
    n = ic["mass"].size
    ref, st, _ = O.run_pass(ic)
    with gzm.MFMContext(gzm.make_params(search=int(search))) as ctx:
        ctx.upload(ic)
        d = ctx.density()
        with_rows = shim.used
        shim.set("budget", with_rows + n)
        g = ctx.gradients()
        assert shim.refused > 0 and shim.used < with_rows
        f = ctx.hydro_force()
        out = ctx.download()
    assert d.density_interactions == st.dens_interactions
    assert g.gradient_interactions == st.grad_interactions
    assert f.force_interactions == st.force_interactions
    errs, bad = check_pass(out, ref)
    assert not bad, bad


def idle_contexts_give_their_rows(shim, search):
    """A second context fits beside one with candidate rows where it fits beside one
    without: the idle one gives them up, between its density and gradients."""
    search = int(search)
    one, two = ics.random_state(32), ics.random_state(32, seed=8)
    n = one["mass"].size
    refs = [O.run_pass(ic)[0] for ic in (one, two)]
    with gzm.MFMContext(gzm.make_params(search=search)) as a:
        empty = shim.used
        a.upload(one)
        one_pass(a)  # every array that a pass needs
        a.upload(one)
        a.density()
        full = shim.used
        rows = n * (96 * 4 + 12 + (0 if search else 16))
        budget = full + (full - empty - rows) - 100 * n  # a second set of that size, without rows, lacks 100 n
        shim.set("budget", budget)
        with gzm.MFMContext(gzm.make_params(search=search)) as b:
            b.upload(two)
            one_pass(b)
            assert shim.refused > 0 and shim.used <= budget
            a.gradients()
            a.hydro_force()
            for ctx, ref in ((a, refs[0]), (b, refs[1])):
                errs, bad = check_pass(ctx.download(), ref)
                assert not bad, bad


def contexts_of_threads_share_a_full_card(shim):
    """Threads with a context each on a card that holds the rows of one or two."""
    import threading
    sets = [ics.random_state(side) for side in (30, 28, 26)]
    refs = [O.run_pass(ic)[0] for ic in sets]
    with gzm.MFMContext(gzm.make_params()) as ctx:
        empty = shim.used
        ctx.upload(sets[0])
        one_pass(ctx)
        each = shim.used - empty
    shim.set("budget", shim.used + int(2.2 * each))
    failures = []

    def work(ic, ref):
        try:
            for _ in range(4):
                with gzm.MFMContext(gzm.make_params()) as ctx:
                    for _ in range(3):
                        ctx.upload(ic)
                        one_pass(ctx)
                        errs, bad = check_pass(ctx.download(), ref)
                        assert not bad, bad
        except gzm.GzmError as e:
            if e.status != 3:  # no memory left even without rows
                failures.append(repr(e))
        except BaseException as e:  # noqa: B902
            failures.append(repr(e))

    threads = [threading.Thread(target=work, args=a) for a in zip(sets, refs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failures and not any(t.is_alive() for t in threads), failures


def failed_allocations_leave_nothing_half_made(shim):
    """An upload without memory leaves no particles, and a force stage that ran out
    of it half-way can be called again."""
    ic = ics.random_state(12)
    n = ic["mass"].size
    ref, st = gzm.run_pass(ic, params=gzm.make_params(pair_list_cap=16))
    with gzm.MFMContext(gzm.make_params(pair_list_cap=16)) as ctx:
        ctx.upload(ic)
        shim.set("budget", shim.used)
        other = ics.random_state(14)
        for call in (lambda: ctx.upload(other), ctx.density, ctx.hydro_force):
            try:
                call()
                raise AssertionError("a context without particles worked")
            except gzm.GzmError as e:
                assert e.status == (3 if call.__name__ == "<lambda>" else 4), e
        shim.set("budget", 1 << 62)
        ctx.upload(ic)
        ctx.density()
        ctx.gradients()
        # the counts of the deferred pairs, then their total
        for unwanted in (4 * n, 4):
            shim.set("unwanted", unwanted)
            try:
                ctx.hydro_force()
                raise AssertionError("the force stage had what it was refused")
            except gzm.GzmError as e:
                assert e.status == 3, e
        shim.set("unwanted", 0)
        f = ctx.hydro_force()
        out = ctx.download()
    assert f.force_interactions == st["force_interactions"]
    for k in OUT_KEYS:
        np.testing.assert_array_equal(out[k], ref[k], err_msg=k)
