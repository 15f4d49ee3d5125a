"""The reverse sweep of the TGV layer on images that do not fill the chip: strips of few rows in one, two or four wavefronts, as the
library picks them by size, against the oracle, bit for bit; the corrected gradient's pairs with one channel."""
import numpy as np
import pytest
import torch

from customnetworklayers_amd.workloads import tgv_inputs

pytestmark = pytest.mark.gpu


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


def check(ext, oracle, n, c, h, w, its, pid=5):
    print("case", n, c, h, w, its, flush=True)
    d = tgv_inputs(n, c, h, w, seed=h + w, conf_density=0.3)
    t = {k: torch.from_numpy(v).cuda() for k, v in d.items()}
    (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, pid)
    got = ext.backward(t["grad"], t["dx"], t["dy"], t["dc"], t["db"], its, pid)
    oracle.reset_id(pid)
    np.testing.assert_array_equal(sol.cpu().numpy(), oracle.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], its, pid))
    for a, r in zip(got, oracle.backward(d["grad"].copy(), d["dx"], d["dy"], d["dc"], d["db"], its, pid)):
        np.testing.assert_array_equal(a.cpu().numpy(), r)


@pytest.mark.parametrize("n,c,h,w,its", [
    (1, 1, 1, 1, 6),      # strips of one row: up to one per CU in two wavefronts,
    (1, 1, 61, 97, 12),
    (1, 1, 129, 121, 9),  # more in one wavefront
    (2, 1, 170, 121, 8),
    (1, 1, 205, 300, 8),  # 1025 strips: two rows, two wavefronts
    (1, 2, 1, 1, 6),      # two channels, strips of one row: four wavefronts
    (1, 2, 3, 62, 13),
    (1, 2, 61, 97, 12),
    (2, 2, 150, 190, 8),  # more than two workgroups of four wavefronts per CU: taller strips
    (2, 2, 129, 240, 8),  # 1032 strips: two rows, two wavefronts
    (1, 3, 20, 61, 9),    # three and four channels
    (2, 4, 30, 130, 9),
])
def test_small_images_match_the_oracle(ext, oracle, n, c, h, w, its):
    ext.reset_id(5)
    check(ext, oracle, n, c, h, w, its)


@pytest.mark.parametrize("n,c,h,w,its", [(1, 1, 40, 70, 13), (1, 1, 129, 121, 9), (1, 1, 205, 300, 8), (1, 2, 40, 70, 13)])
def test_corrected_gradient_on_small_images(ext, oracle, n, c, h, w, its):
    ext.reset_id(5)
    ext.gradient_mode(5, 1)
    oracle.set_quirks(end_uses_ckpt_y=0, skip_iter0_adjoint=0, getyk_rebuild=0, scale_factors=0, dw_div=0)
    try:
        check(ext, oracle, n, c, h, w, its)
    finally:
        oracle.set_quirks()
        ext.reset_id(5)
