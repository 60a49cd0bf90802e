"""The autotuner leaves alone the axes that a pass does not read (on the CPU, with the
timings replaced by a model in which noise favours them)."""
import numpy as np
import pytest

import autotune

ALL = {name for name, _ in autotune.AXES}


@pytest.mark.parametrize("precision,n,read", [
    (0, 4096, {"cell_factor", "pair_list_cap", "density_budget"}),
    (0, 65537, {"cell_factor", "pair_list_cap", "density_budget", "block_gradients"}),
    (1, 4096, ALL - {"block_density", "wave_sweep_max"}),
    (2, 4096, ALL),
])
def test_axes_that_nothing_reads_are_neither_timed_nor_chosen(monkeypatch, precision, n, read):
    timed = []

    def fake(sample, prec, setting):
        timed.append(dict(setting))
        # each axis' last candidate "gains" 10 %
        return 10.0 * np.prod([0.9 if setting[name] == cands[-1] else 1.0 for name, cands in autotune.AXES])

    monkeypatch.setattr(autotune, "time_setting", fake)
    r = autotune.tune({"pos": np.zeros((n, 3))}, precision)
    for name, cands in autotune.AXES:
        assert r["setting"][name] == (cands[-1] if name in read else autotune.DEFAULTS[name]), name
        assert {s[name] for s in timed} == (set(cands) if name in read else {autotune.DEFAULTS[name]}), name
        assert set(r["axes"][name]) == {str(v) for v in cands} and all(v > 0 for v in r["axes"][name].values())
