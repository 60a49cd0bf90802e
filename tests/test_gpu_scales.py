"""The FP64 pass in other units of length (a power of two, and mass with it so that
densities stay): sides whose squares leave the range of FP32 give the pass of the
unit box, scaled."""
import numpy as np
import pytest

import gzm
import ics

pytestmark = pytest.mark.gpu

# powers of the length unit in each output
POWERS = {"hsml": 1, "density": 0, "pressure": 0, "num_ngb": 0, "divvel": -1, "fce": 0, "grad_rho": -1, "grad_v": -1,
          "vsig": 0, "acc": -1, "dtu": -1}


@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("side", [12, 41])  # eight lanes and one lane per particle
@pytest.mark.parametrize("exponent", [70, -70])
def test_units_of_length(side, exponent, method):
    ic = ics.random_state(side)
    f = 2.0 ** exponent
    big = dict(ic, pos=ic["pos"] * f, hsml=ic["hsml"] * f, mass=ic["mass"] * f ** 3, box=ic["box"] * f)
    one, st1 = gzm.run_pass(ic, params=gzm.make_params(method=method))
    out, st = gzm.run_pass(big, params=gzm.make_params(box=tuple(big["box"]), method=method))
    for k in ("density_sweeps", "density_interactions", "gradient_interactions", "force_interactions",
              "exact_solver_calls"):
        assert st[k] == st1[k], k
    for k, p in POWERS.items():
        scale = np.abs(one[k]).max()
        assert scale > 0
        # every operation scales exactly but for library roots, which may round apart
        assert np.abs(out[k] / f ** p - one[k]).max() <= 1e-12 * scale, k
