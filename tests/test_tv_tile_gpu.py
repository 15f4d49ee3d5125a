"""The TV layer's register-tile kernels (several iterations per launch) against the CPU oracle, bit for bit: the tiles are
forced with INPAINT_TV_TILE / INPAINT_TV_ADJ_TILE=rows per wavefront,iterations per launch, at the sizes where a tile can go
wrong -- smaller than a tile, one pixel more or less than whole tiles, launches of unequal length, launches that end on, before
and behind a segment's first iteration."""
import numpy as np
import pytest
import torch

from customnetworklayers_amd.workloads import tv_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ext():
    from customnetworklayers_amd.cudaTV import tvInpaint_cuda_ext

    return tvInpaint_cuda_ext


def tensors(d):
    return {k: torch.from_numpy(v).to(DEV) for k, v in d.items()}


def check(ext, oracle, d, its, pid, **forward):
    t = tensors(d)
    (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, pid, **forward)
    got = ext.backward(t["grad"], t["dx"], t["dy"], t["dc"], t["db"], its, pid)
    oracle.reset_id(pid)
    want = oracle.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], its, pid)
    grads = oracle.backward(d["grad"].copy(), d["dx"], d["dy"], d["dc"], d["db"], its, pid)
    np.testing.assert_array_equal(sol.cpu().numpy(), want)
    for a, r in zip(got, grads):
        np.testing.assert_array_equal(a.cpu().numpy(), r)


@pytest.mark.parametrize("fwd,adj", [("4,2", "4,1"), ("4,5", "4,3"), ("4,7", "4,7"), ("8,6", "4,5"), ("16,12", "4,6"),
                                     ("0", "0")])  # strips
@pytest.mark.parametrize("n,c,h,w,its", [
    (1, 1, 1, 1, 4),        # one pixel
    (1, 2, 5, 3, 7),        # smaller than any tile, odd its
    (1, 2, 6, 54, 20),      # exactly one tile of 4 rows, 5 iterations; its segments start at 0, 4, 8, 12
    (2, 1, 7, 55, 20),      # one row and one column more
    (1, 2, 21, 53, 26),     # two channels: 22 columns per adjoint tile of 5 steps, one column short of the next
    (1, 3, 33, 70, 9),      # three channels (forward tiles, adjoint strips)
    (2, 2, 61, 131, 2),     # a single launch in each direction
])
def test_tiles_match_the_oracle(ext, tv_oracle, monkeypatch, n, c, h, w, its, fwd, adj):
    monkeypatch.setenv("INPAINT_TV_TILE", fwd)
    monkeypatch.setenv("INPAINT_TV_ADJ_TILE", adj)
    ext.reset_id(4)
    check(ext, tv_oracle, tv_inputs(n, c, h, w, seed=h + w, conf_density=0.3), its, 4)


@pytest.mark.parametrize("keep", [0, 1])
@pytest.mark.parametrize("its", [12, 25])
def test_forward_tiles_leave_checkpoints_for_a_recomputing_backward(ext, tv_oracle, monkeypatch, keep, its):
    monkeypatch.setenv("INPAINT_TV_TILE", "4,3")
    ext.reset_id(4)
    check(ext, tv_oracle, tv_inputs(1, 2, 40, 90, seed=5), its, 4, keep=keep)


@pytest.mark.parametrize("c,its", [(1, 20), (2, 13)])
def test_corrected_gradient_in_tiles(ext, tv_oracle, monkeypatch, c, its):
    monkeypatch.setenv("INPAINT_TV_ADJ_TILE", "4,4")
    ext.reset_id(4)
    ext.gradient_mode(4, 1)
    tv_oracle.set_quirks(end_uses_ckpt_y=0, skip_iter0_adjoint=0, getyk_rebuild=0, scale_factors=0)
    try:
        check(ext, tv_oracle, tv_inputs(1, c, 37, 75, seed=6), its, 4)
    finally:
        tv_oracle.set_quirks()
        ext.reset_id(4)


@pytest.mark.parametrize("tile,its", [("8,4", 4), ("8,4", 20)])  # one launch (reads a copy of the starting point), several
def test_allocation_free_forward_in_place(ext, monkeypatch, tile, its):
    from customnetworklayers_amd._lib import reload_env

    t = tensors(tv_inputs(2, 2, 40, 70, seed=7))
    args = (t["dx"], t["dy"], t["dc"], t["db"])
    monkeypatch.setenv("INPAINT_TV_TILE", "0")
    reload_env()
    (want,) = ext.forward(*args, t["di"], its, 4)
    monkeypatch.setenv("INPAINT_TV_TILE", tile)
    reload_env()
    x = t["di"].clone()
    ext.forward_noalloc(*args, x, its, x)
    assert torch.equal(x, want)


@pytest.mark.parametrize("n,c,h,w,its", [(1, 2, 64, 128, 20), (1, 1, 40, 70, 9), (1, 2, 30, 50, 2), (4, 2, 384, 1248, 8)])
def test_profile_times_the_reverse_sweep_that_ran(ext, n, c, h, w, its):
    # tiles (the first two), a single launch that is not an inner strip launch, strips
    import ctypes

    from customnetworklayers_amd._lib import lib

    t = tensors(tv_inputs(n, c, h, w, seed=9))
    ext.reset_id(4)
    steps = lib.tvinpaint_adjoint_tile_steps(n, c, h, w, its)
    lib.tvinpaint_profile(1)
    ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, 4)
    ext.backward(t["grad"], t["dx"], t["dy"], t["dc"], t["db"], its, 4)
    ms, launches = ctypes.c_double(0), ctypes.c_int(0)
    lib.tvinpaint_profile_read(ctypes.byref(ms), ctypes.byref(launches))
    lib.tvinpaint_profile(0)
    ext.reset_id(4)
    all_steps = 2 * (its // 2) - 1
    if steps:
        assert launches.value == -(-all_steps // steps) and 0 < ms.value < 1000
    else:
        assert launches.value <= all_steps // 2  # inner pair launches only
    assert bool(steps) == (n == 1 and its > 2)


@pytest.mark.parametrize("n,c,h,w,its", [(1, 2, 64, 128, 20), (2, 2, 112, 256, 24), (1, 1, 187, 621, 20), (1, 2, 384, 1248, 20)])
def test_default_choice_of_kernels_matches_the_oracle(ext, tv_oracle, n, c, h, w, its):
    ext.reset_id(4)
    check(ext, tv_oracle, tv_inputs(n, c, h, w, seed=8), its, 4)
    ext.reset_id(4)


@pytest.mark.parametrize("pixel", [(30, 64), (0, 20), (59, 129), (17, 0)])  # inside, and on the image's edges
@pytest.mark.parametrize("name,value", [("dx", np.inf), ("dy", np.nan), ("dc", np.inf), ("db", np.inf), ("di", -np.inf), ("di", np.nan)])
def test_non_finite_inputs_spread_as_in_strips(ext, monkeypatch, name, value, pixel):
    # What a pixel outside the image takes on from a neighbour inside must not come back sooner than it spreads inside; the
    # reverse sweep's clip turns NaN into a number, outside the image too.
    d = tv_inputs(1, 2, 60, 130, seed=9)
    d[name][0, -1, pixel[0], pixel[1]] = value
    t = tensors(d)
    out = []
    for fwd, adj in (("0", "0"), ("4,3", "4,3"), ("8,6", "4,7")):
        monkeypatch.setenv("INPAINT_TV_TILE", fwd)
        monkeypatch.setenv("INPAINT_TV_ADJ_TILE", adj)
        ext.reset_id(4)
        (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], 12, 4)
        out.append([sol] + ext.backward(t["grad"].clone(), t["dx"], t["dy"], t["dc"], t["db"], 12, 4))
    ext.reset_id(4)
    assert name != "di" or not torch.isfinite(out[0][0]).all()
    for got in out[1:]:
        for a, b in zip(out[0], got):
            np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
