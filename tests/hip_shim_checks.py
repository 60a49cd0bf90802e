"""Checks that run in hip_shim's process, each called with the shim."""
import gzm
import ics


def entry_points_make_their_device_current(shim):
    """every call that may launch or copy on a context's stream sets its device first"""
    with gzm.MFMContext(gzm.make_params()) as ctx:
        calls = [lambda: ctx.upload(ics.random_state(8)), ctx.density, ctx.gradients, ctx.hydro_force,
                 ctx.restore_initial_state, lambda: ctx.run_passes(1), ctx.download, lambda: ctx.neighbor_counts(0)]
        for k, call in enumerate(calls):
            before = shim.set_device_calls
            call()
            assert shim.set_device_calls > before, k
