"""What the library asks of the HIP runtime, with a shim before it (hip_shim)."""
import pytest

import hip_shim

pytestmark = pytest.mark.gpu


def test_entry_points_make_their_device_current():
    hip_shim.run("entry_points_make_their_device_current")


def test_run_passes_probes_again_without_rows():
    hip_shim.run("run_passes_probes_again_without_rows")


@pytest.mark.parametrize("precision", [0, 1])
def test_run_passes_reports_what_its_probe_did_not_meet(precision):
    hip_shim.run("run_passes_reports_what_its_probe_did_not_meet", precision)


@pytest.mark.parametrize("check", ["deferred_buffer_shrinks_before_rows_go", "deferred_buffer_grows_within_what_is_free"])
def test_deferred_pairs_leave_the_rows_their_memory(check):
    hip_shim.run(check)


def test_rows_come_back_with_the_memory():
    hip_shim.run("rows_come_back_with_the_memory")


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("search", [0, 1])
@pytest.mark.parametrize("side", [12, 41])  # eight lanes and one lane per particle
def test_pass_without_candidate_rows(side, search, method):
    hip_shim.run("without_rows", side, search, method)


@pytest.mark.parametrize("search", [0, 1])
def test_rows_given_up_between_stages(search):
    hip_shim.run("rows_given_up_between_stages", search)


@pytest.mark.parametrize("search", [0, 1])
def test_idle_contexts_give_their_rows(search):
    hip_shim.run("idle_contexts_give_their_rows", search)


def test_contexts_of_threads_share_a_full_card():
    hip_shim.run("contexts_of_threads_share_a_full_card")


def test_failed_allocations_leave_nothing_half_made():
    hip_shim.run("failed_allocations_leave_nothing_half_made")
