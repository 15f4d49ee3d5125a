"""The launches at the start and the end of a TGV pass (Lipschitz bounds, scaled weights, check of the upstream gradient, stores of
the outputs), each for all samples and tensors at once: against the oracle, bit for bit, at the edges of their blocks and with the
deciding entry at the first, a middle and the last place."""
import numpy as np
import pytest
import torch

from customnetworklayers_amd.workloads import tgv_inputs

pytestmark = pytest.mark.gpu
ITS, PID = 5, 6

SIZES = [(1, 1, 1, 1), (1, 1, 4, 64), (1, 2, 5, 65), (2, 1, 3, 63), (3, 2, 33, 129), (5, 1, 7, 70), (1030, 1, 5, 3), (1, 1, 380, 700), (4, 2, 150, 300)]
PLACES = [0, 0.5, 1]


@pytest.fixture(scope="module")
def ext():
    from customnetworklayers_amd.cudaTGV import tgvInpaint_cuda_ext

    return tgvInpaint_cuda_ext


@pytest.fixture(scope="module")
def oracle():
    from oracle.oracle_lib import TGVOracle

    o = TGVOracle()
    o.set_quirks()
    return o


def at(a, place):
    return np.unravel_index(int(place * (a.size - 1)), a.shape)


@pytest.mark.parametrize("n,c,h,w", SIZES)
@pytest.mark.parametrize("place", PLACES)
def test_pass(ext, oracle, n, c, h, w, place):
    print("case", n, c, h, w, place, flush=True)
    d = tgv_inputs(n, c, h, w, seed=h + w, conf_density=0.3)
    for k in ("dx", "dy"):
        d[k][at(d[k], place)] = 40.0  # decides its sample's bound
    t = {k: torch.from_numpy(v).cuda() for k, v in d.items()}
    oracle.reset_id(PID)
    ext.reset_id(PID)

    def both(grad):
        (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], ITS, PID)
        np.testing.assert_array_equal(sol.cpu().numpy(), oracle.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], ITS, PID))
        upstream, given = torch.from_numpy(grad).cuda(), grad.copy()
        got = ext.backward(upstream, t["dx"], t["dy"], t["dc"], t["db"], ITS, PID)
        want = oracle.backward(given, d["dx"], d["dy"], d["dc"], d["db"], ITS, PID)
        for a, r in zip(got, want):
            np.testing.assert_array_equal(a.cpu().numpy(), r)
        np.testing.assert_array_equal(upstream.cpu().numpy(), np.where(np.isfinite(grad), grad, 0))
        return any(r.any() for r in want)

    both(d["grad"])
    for value in (np.nan, np.inf):
        bad = d["grad"].copy()
        bad[at(bad, place)] = value
        assert not both(bad)
    assert not both(np.zeros_like(d["grad"]))
    one = np.zeros_like(d["grad"])
    one[at(one, place)] = 1.0  # the only entry that is not zero
    both(one)
    both(d["grad"])
