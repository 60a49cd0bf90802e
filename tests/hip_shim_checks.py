"""Checks that run in hip_shim's process, each called with the shim."""
import ctypes as C

import numpy as np

import gzm
import ics

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
