"""GPU parity of the TGV layer: the HIP path through the C ABI against the CPU oracle on the same
seeded inputs.

Tolerances (the layer's contract): max-abs error / max-abs oracle value <= 1e-4 on the solution
(u, v1, v2) and <= 1e-3 on the gradients wrt the two-channel edge weights, confidence, right-hand
side and starting point.  The kernels reproduce the oracle's arithmetic operation by operation, so
the observed errors are far smaller (bit-equal is expected); the tests print them.
"""
import numpy as np
import pytest
import torch

from customnetworklayers_amd.workloads import CONFIGS, tgv_inputs

pytestmark = pytest.mark.gpu

OUT_TOL = 1e-4
GRAD_TOL = 1e-3


def rel_err(a, ref):
    return float(np.abs(a.astype(np.float64) - ref.astype(np.float64)).max() / max(np.abs(ref).max(), 1e-30))


@pytest.fixture(scope="module")
def ext():
    from customnetworklayers_amd.cudaTGV import tgvInpaint_cuda_ext

    return tgvInpaint_cuda_ext


@pytest.fixture(scope="module")
def tgv_oracle():
    from oracle.oracle_lib import TGVOracle

    o = TGVOracle()
    o.set_quirks()
    return o


def varying_inputs(n, c, h, w, seed, beta_hi=9.0):
    """Spatially varying beta (exercises the data-dependent Lipschitz branch and its neighbour
    offsets) and non-zero auxiliary starting values."""
    d = tgv_inputs(n, c, h, w, seed=seed, conf_density=0.3)
    rng = np.random.default_rng(seed + 7)
    d["dx"][:, 1] = rng.uniform(0.2, beta_hi, (n, h, w)).astype(np.float32)
    d["dy"][:, 1] = rng.uniform(0.2, beta_hi, (n, h, w)).astype(np.float32)
    d["di"][:, c:] = rng.normal(0, 0.5, (n, 2 * c, h, w)).astype(np.float32)
    return d


def run_gpu(ext, d, its, pid, fresh=True):
    dev = torch.device("cuda:0")
    t = {k: torch.from_numpy(v).to(dev) for k, v in d.items()}
    if fresh:
        ext.reset_id(pid)
    (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, pid)
    grads = ext.backward(t["grad"], t["dx"], t["dy"], t["dc"], t["db"], its, pid)
    torch.cuda.synchronize()
    return sol.cpu().numpy(), [g.cpu().numpy() for g in grads], t["grad"].cpu().numpy()


def run_oracle(o, d, its, pid, fresh=True):
    if fresh:
        o.reset_id(pid)
    sol = o.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], its, pid)
    gin = d["grad"].copy()
    grads = o.backward(gin, d["dx"], d["dy"], d["dc"], d["db"], its, pid)
    return sol, list(grads), gin


def compare(name, got, ref):
    sol, grads, _ = got
    rsol, rgrads, _ = ref
    e_out = rel_err(sol, rsol)
    errs = [rel_err(g, r) for g, r in zip(grads, rgrads)]
    exact = float((sol == rsol).mean())
    print("\n[%s] out rel %.2e (bit-equal %.4f)  gx %.2e gy %.2e gc %.2e gb %.2e gi %.2e"
          % (name, e_out, exact, *errs), flush=True)
    assert e_out <= OUT_TOL, (name, e_out)
    for nm, e in zip(("gx", "gy", "gc", "gb", "gi"), errs):
        assert e <= GRAD_TOL, (name, nm, e)
    return e_out, errs


@pytest.mark.parametrize("n,c,h,w,its", [
    (1, 1, 64, 128, 20),    # the reference's own shape: one flow channel, three state channels
    (1, 1, 16, 64, 2),      # a single pair of iterations
    (2, 3, 37, 101, 9),     # ragged, odd its, three channels, two samples
    (1, 2, 5, 3, 6),        # tiny
    (1, 2, 1, 70, 4),       # a single row
    (1, 1, 33, 1, 4),       # a single column
    (2, 2, 70, 130, 50),    # several segments of unequal length
    (1, 2, 21, 64, 6),      # exactly one wavefront wide
    (1, 2, 19, 65, 6),      # one column more
])
def test_forward_backward_match_oracle(ext, tgv_oracle, kernels, n, c, h, w, its):
    d = tgv_inputs(n, c, h, w, seed=n * 1000 + h + w + its, conf_density=0.3)
    print("case n=%d c=%d h=%d w=%d its=%d" % (n, c, h, w, its), flush=True)
    compare("%dx%dx%dx%d its=%d" % (n, c, h, w, its), run_gpu(ext, d, its, 2), run_oracle(tgv_oracle, d, its, 2))


@pytest.mark.parametrize("n,c,h,w,its", [
    (1, 3, 20, 64, 6),      # 2 + 1
    (2, 4, 37, 101, 9),     # 2 + 2, ragged, odd its
    (1, 5, 19, 126, 20),    # three groups, several segments
    (1, 3, 45, 130, 12),
])
def test_more_than_two_channels_run_in_channel_groups(ext, tgv_oracle, kernels, n, c, h, w, its):
    # the strip kernels hold up to two flow channels; more run as launches over groups of channels, whose shared
    # accumulators (confidence and weight gradients) are summed group after group in the reference's order
    d = varying_inputs(n, c, h, w, seed=300 + c)
    got, ref = run_gpu(ext, d, its, 2), run_oracle(tgv_oracle, d, its, 2)
    compare("%d channels in groups" % c, got, ref)
    assert np.array_equal(got[0], ref[0])
    for a, b in zip(got[1], ref[1]):
        assert np.array_equal(a, b)


def test_removed_kernel_path_is_refused(ext, monkeypatch):
    # INPAINT_TGV_PATH=px used to select the one-pixel-per-thread kernels written first; the library no longer contains
    # them and says so
    d = varying_inputs(1, 2, 20, 64, seed=3)
    t = {k: torch.from_numpy(v).to("cuda:0") for k, v in d.items()}
    monkeypatch.setenv("INPAINT_TGV_PATH", "px")
    try:
        ext.reset_id(2)  # (re-reads the environment)
        with pytest.raises(ValueError, match="no longer contains"):
            ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], 6, 2)
    finally:
        monkeypatch.delenv("INPAINT_TGV_PATH")
        ext.reset_id(2)
    ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], 6, 2)
    ext.reset_id(2)


@pytest.mark.parametrize("n,c,h,w,its", [
    (1, 1, 9, 62, 8),       # exactly one strip wide
    (1, 2, 11, 63, 8),      # one column more than a strip
    (2, 2, 45, 508, 14),    # several strips wide, ragged rows
    (1, 2, 40, 125, 10),    # two strips and a column
    (3, 1, 130, 200, 50),   # several segments of unequal length
])
def test_strip_edges(ext, tgv_oracle, kernels, n, c, h, w, its):
    d = varying_inputs(n, c, h, w, seed=n * 100 + h + w)
    compare("%dx%dx%dx%d its=%d" % (n, c, h, w, its), run_gpu(ext, d, its, 2), run_oracle(tgv_oracle, d, its, 2))


@pytest.mark.parametrize("n,c,h,w,its", [(2, 2, 70, 256, 20), (1, 1, 45, 130, 10)])
def test_single_iteration_strip_kernels(ext, tgv_oracle, n, c, h, w, its, monkeypatch):
    # the forward and the recompute normally run two iterations per launch; INPAINT_TGV_FUSE=0 keeps
    # the one-iteration strip kernels covered
    d = varying_inputs(n, c, h, w, seed=91 + c)
    ref = run_oracle(tgv_oracle, d, its, 2)
    monkeypatch.setenv("INPAINT_TGV_FUSE", "0")
    compare("one iteration per launch c=%d" % c, run_gpu(ext, d, its, 2), ref)


@pytest.mark.parametrize("n,c,h,w,its", [
    (1, 1, 9, 60, 8),       # exactly one fused strip wide (60 output columns)
    (1, 2, 11, 61, 8),      # one column more
    (1, 2, 3, 200, 6),      # fewer rows than the fused kernel's row lag
    (1, 2, 2, 59, 4),
    (2, 2, 18, 121, 12),    # two fused strips and a column
])
def test_fused_forward_strip_edges(ext, tgv_oracle, kernels, n, c, h, w, its):
    d = varying_inputs(n, c, h, w, seed=n * 100 + h + w)
    compare("%dx%dx%dx%d its=%d" % (n, c, h, w, its), run_gpu(ext, d, its, 2), run_oracle(tgv_oracle, d, its, 2))


@pytest.mark.parametrize("keep", ["0", "2"])
@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("n,c,h,w,its", [(2, 2, 50, 140, 12), (1, 3, 37, 121, 9), (2, 4, 20, 64, 20), (1, 2, 3, 200, 6), (1, 5, 19, 126, 10)])
def test_forward_pairs_with_one_channel_per_wavefront(ext, tgv_oracle, n, c, h, w, its, split, keep, monkeypatch):
    # the forward pairs run one channel per wavefront, all channels in one launch (the default from two channels on);
    # INPAINT_TGV_FWD_SPLIT=0 keeps the launches over groups of two channels covered; with the iterates kept (the pairs
    # rebuild their input from the x05 rows) and recomputed
    d = varying_inputs(n, c, h, w, seed=640 + c + h)
    ref = run_oracle(tgv_oracle, d, its, 2)
    monkeypatch.setenv("INPAINT_TGV_FWD_SPLIT", split)
    monkeypatch.setenv("INPAINT_KEEP", keep)
    got = run_gpu(ext, d, its, 2)
    compare("forward split %s, keep %s, %d channels" % (split, keep, c), got, ref)
    assert np.array_equal(got[0], ref[0])
    for a, b in zip(got[1], ref[1]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,c,h,w,its", [(2, 2, 70, 256, 20), (1, 1, 45, 130, 10)])
def test_single_step_adjoint_strip_kernels(ext, tgv_oracle, n, c, h, w, its, monkeypatch):
    # the reverse sweep may run two adjoint steps per launch; INPAINT_TGV_FUSE_ADJ=0 keeps the
    # one-step strip kernels covered
    d = varying_inputs(n, c, h, w, seed=93 + c)
    ref = run_oracle(tgv_oracle, d, its, 2)
    monkeypatch.setenv("INPAINT_TGV_FUSE_ADJ", "0")
    compare("one adjoint step per launch c=%d" % c, run_gpu(ext, d, its, 2), ref)


@pytest.mark.parametrize("waves", ["1", "2"])
@pytest.mark.parametrize("n,c,h,w,its", [(2, 2, 70, 256, 20), (1, 1, 45, 130, 10), (1, 2, 3, 200, 6), (2, 2, 18, 121, 12),
                                         (1, 2, 1, 70, 4), (1, 1, 33, 1, 4)])
def test_adjoint_pairs_in_one_or_two_wavefronts(ext, tgv_oracle, n, c, h, w, its, waves, monkeypatch):
    # the two steps of a pair run in one wavefront (default at one channel) or in the two wavefronts of a
    # workgroup, handed over through LDS (default at two channels); force each layout for both channel counts
    d = varying_inputs(n, c, h, w, seed=95 + c + h)
    ref = run_oracle(tgv_oracle, d, its, 2)
    monkeypatch.setenv("INPAINT_TGV_PAIR_WAVES", waves)
    compare("pair in %s wavefront(s) c=%d %dx%d" % (waves, c, h, w), run_gpu(ext, d, its, 2), ref)


@pytest.mark.parametrize("split", ["0", "1"])
@pytest.mark.parametrize("rows", ["8", "13", "64"])
def test_adjoint_pair_strip_heights(ext, tgv_oracle, rows, split, monkeypatch):
    d = varying_inputs(2, 2, 50, 140, seed=97)
    ref = run_oracle(tgv_oracle, d, 12, 2)
    monkeypatch.setenv("INPAINT_TGV_ADJ_ROWS", rows)
    monkeypatch.setenv("INPAINT_TGV_FWD_ROWS", rows)
    monkeypatch.setenv("INPAINT_TGV_FWD_SPLIT", split)
    compare("strip height %s" % rows, run_gpu(ext, d, 12, 2), ref)


@pytest.mark.parametrize("rows", ["", "1", "2", "3", "5", "8", "13", "64"])
@pytest.mark.parametrize("n,c,h,w,its", [(2, 3, 50, 140, 12), (1, 4, 37, 121, 9), (1, 4, 3, 200, 6), (2, 3, 1, 70, 4),
                                         (1, 4, 33, 1, 4)])
def test_three_and_four_channels_pair_in_four_wavefronts(ext, tgv_oracle, n, c, h, w, its, rows, monkeypatch):
    # three and four channels: the pair runs in four wavefronts of a workgroup (two channel groups; the five shared
    # accumulators travel A0 -> A1 -> B1, which applies B0's terms first); strips shorter and taller than the image,
    # strips of one interval and of several, ragged last strips, images narrower than the aprons
    d = varying_inputs(n, c, h, w, seed=131 + c + h)
    ref = run_oracle(tgv_oracle, d, its, 2)
    if rows:
        monkeypatch.setenv("INPAINT_TGV_ADJ_ROWS", rows)
    got = run_gpu(ext, d, its, 2)
    compare("four-wavefront pair c=%d %dx%d rows=%s" % (c, h, w, rows or "chosen"), got, ref)
    assert np.array_equal(got[0], ref[0])
    for a, b in zip(got[1], ref[1]):
        assert np.array_equal(a, b)


REGIMES = {
    # name: (scale of the flow, confidence values, edge-weight values, beta values)
    "large flows": (1e4, (0.0, 0.3, 1.0), (1e-3, 1.0), (2.0,)),
    "tiny flows": (1e-6, (0.0, 0.3, 1.0), (1e-3, 1.0), (2.0,)),
    "confidence from 1e-8 to 1e3": (8.0, (0.0, 1e-8, 1e-3, 1.0, 1e3), (0.2, 1.0), (2.0,)),
    "weights from 0 to 1 and beta from 1e-3 to 40": (8.0, (0.0, 0.5), (0.0, 1e-12, 1e-3, 1.0), (1e-3, 0.5, 2.0, 40.0)),
    "flat image, no data": (0.0, (0.0,), (1.0,), (2.0,)),
}


@pytest.mark.parametrize("c", [1, 2, 3])
@pytest.mark.parametrize("regime", sorted(REGIMES))
def test_unusual_magnitudes_stay_bit_equal(ext, tgv_oracle, regime, c):
    # as for the TV layer: magnitudes far from the benchmark's must leave every output bit-equal to the oracle
    scale, confs, weights, betas = REGIMES[regime]
    n, h, w, its = 2, 37, 131, 12
    d = varying_inputs(n, c, h, w, seed=900 + c)
    rng = np.random.default_rng(23 + c)
    d["db"] = (d["db"] * np.float32(scale / 8.0)).astype(np.float32)
    d["di"][:, :c] = d["db"]
    d["di"][:, c:] *= np.float32(scale / 8.0)
    d["dc"] = rng.choice(np.array(confs, np.float32), size=d["dc"].shape).astype(np.float32)
    for k in ("dx", "dy"):
        d[k][:, 0] = rng.choice(np.array(weights, np.float32), size=d[k][:, 0].shape)
        d[k][:, 1] = rng.choice(np.array(betas, np.float32), size=d[k][:, 1].shape)
    got, ref = run_gpu(ext, d, its, 2), run_oracle(tgv_oracle, d, its, 2)
    compare("%s, %d channels" % (regime, c), got, ref)
    assert np.array_equal(got[0], ref[0], equal_nan=True)
    for a, b in zip(got[1], ref[1]):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("c", [1, 2, 3, 4])
@pytest.mark.parametrize("its", [2, 3, 4, 5, 6, 8, 16, 17, 26])
def test_every_pairing_of_the_reverse_sweep(ext, tgv_oracle, c, its):
    # segment lengths 2, 4, 6 ... and their mixes: first step + pairs, first + single + pairs,
    # a pair that ends a segment, a single step that ends a segment
    d = varying_inputs(1, c, 23, 75, seed=its * 7 + c)
    compare("c=%d its=%d" % (c, its), run_gpu(ext, d, its, 2), run_oracle(tgv_oracle, d, its, 2))


@pytest.mark.parametrize("c", [1, 2, 3])
@pytest.mark.parametrize("its", [4, 5, 9, 16, 50])
def test_first_step_of_the_sweep_rides_on_the_second(ext, tgv_oracle, c, its, monkeypatch):
    # one or two channels, a last segment of at least four iterations: one launch does the sweep's first two steps
    # (its = 4, 5: the last segment has two iterations, so the two steps stay apart; c = 3 always keeps them apart);
    # INPAINT_TGV_FUSE_FIRST=0 keeps the separate launches covered
    d = varying_inputs(2, c, 37, 130, seed=600 + 10 * c + its)
    ref = run_oracle(tgv_oracle, d, its, 2)
    a = run_gpu(ext, d, its, 2)
    compare("first two steps in one launch c=%d its=%d" % (c, its), a, ref)
    monkeypatch.setenv("INPAINT_TGV_FUSE_FIRST", "0")
    b = run_gpu(ext, d, its, 2)
    compare("first step in its own launch c=%d its=%d" % (c, its), b, ref)
    for x, y in zip(a[1], b[1]):
        np.testing.assert_array_equal(x, y)


def test_gradient_mode_is_fixed_by_the_forward_pass(ext):
    # as in the TV layer: a forward that keeps every x05 row stores one half of each checkpoint, the one its mode reads
    dev = torch.device("cuda:0")
    d = {k: torch.from_numpy(v).to(dev) for k, v in varying_inputs(1, 2, 24, 70, seed=12).items()}
    try:
        ext.reset_id(3)
        ext.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], 20, 3)
        ext.gradient_mode(3, 1)
        with pytest.raises(RuntimeError, match="gradient mode"):
            ext.backward(d["grad"].clone(), d["dx"], d["dy"], d["dc"], d["db"], 20, 3)
        ext.gradient_mode(3, 0)
        ext.backward(d["grad"].clone(), d["dx"], d["dy"], d["dc"], d["db"], 20, 3)
        for keep in (0, 1):  # the same rule where both checkpoint halves exist
            ext.keep_iterates(3, keep)
            ext.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], 20, 3)
            ext.gradient_mode(3, 1)
            with pytest.raises(RuntimeError, match="gradient mode"):
                ext.backward(d["grad"].clone(), d["dx"], d["dy"], d["dc"], d["db"], 20, 3)
            ext.gradient_mode(3, 0)
            ext.backward(d["grad"].clone(), d["dx"], d["dy"], d["dc"], d["db"], 20, 3)
    finally:
        ext.reset_id(3)


def test_varying_beta_and_per_sample_lipschitz(ext, tgv_oracle):
    # sample 0: beta up to 9 (bound above 32, data dependent); sample 1: small beta (bound 32)
    d = varying_inputs(2, 2, 40, 56, seed=11)
    d["dx"][1, 1] *= 0.2
    d["dy"][1, 1] *= 0.2
    got = run_gpu(ext, d, 16, 1)
    Ls = ext.lipschitz(1, 2)
    ref_L = [tgv_oracle.lipschitz(d["dx"][s], d["dy"][s])[0] for s in range(2)]
    assert Ls == ref_L, (Ls, ref_L)
    assert Ls[0] < Ls[1] == float(np.float32(1.0 / np.float64(np.float32(np.float32(32.0) + np.float32(0.01)))))
    compare("varying beta", got, run_oracle(tgv_oracle, d, 16, 1))


def test_its_zero_and_one_return_init_and_zero_grads(ext, tgv_oracle):
    d = tgv_inputs(1, 2, 20, 30, seed=5)
    for its in (0, 1):
        sol, grads, _ = run_gpu(ext, d, its, 3)
        np.testing.assert_array_equal(sol, d["di"])
        rsol, rgrads, _ = run_oracle(tgv_oracle, d, its, 3)
        for g, r in zip(grads, rgrads):
            np.testing.assert_array_equal(g, r)
            assert not g.any()


def test_headline_shape_one_sample_short(ext, tgv_oracle):
    # one sample of the TGV configuration's shape (2 x 384 x 1248), 20 iterations
    cfg = CONFIGS[2]
    d = tgv_inputs(1, cfg["c"], cfg["h"], cfg["w"], seed=0, **cfg["gen"])
    compare("tgv-config/1 its=20", run_gpu(ext, d, 20, 0), run_oracle(tgv_oracle, d, 20, 0))


@pytest.mark.parametrize("scale,bit_equal", [(1e-20, True), (1e-30, True), (1e-36, False), (1e20, True), (1e30, True)])
def test_upstream_gradients_of_extreme_magnitude(ext, tgv_oracle, scale, bit_equal):
    # The short division (reciprocal refined once, quotient corrected once, no range fix-ups) returns the compiler's bits
    # while the correction's residual stays a normal number.  The adjoint's numerators scale with the upstream gradient:
    # down to 1e-30 and up to 1e30 (where the clamps of the adjoint iterates act) every gradient is the oracle's, bit for
    # bit; at 1e-36 the results (1e-38 and below) are denormal and agree to their last bits only (1e-7 of the largest).
    from customnetworklayers_amd.workloads import tgv_inputs as make

    d = make(1, 2, 40, 130, seed=3, conf_density=0.4)
    d["grad"] = (d["grad"].astype(np.float64) * scale).astype(np.float32)
    got, ref = run_gpu(ext, d, 12, 2), run_oracle(tgv_oracle, d, 12, 2)
    for a, b in zip(got[1], ref[1]):
        if bit_equal:
            assert np.array_equal(a, b, equal_nan=True)
        else:
            assert float(np.abs(a.astype(np.float64) - b).max()) <= 1e-6 * float(np.abs(b).max())
    ext.reset_id(2)


def test_bad_upstream_returns_zeros_and_does_not_count(ext, tgv_oracle):
    d = tgv_inputs(1, 2, 24, 40, seed=6)
    its = 8
    base = run_gpu(ext, d, its, 4)
    assert ext.get_state(4)[0] == 1 and all(g.any() for g in base[1])
    dev = torch.device("cuda:0")
    t = {k: torch.from_numpy(v).to(dev) for k, v in d.items()}
    bad = t["grad"].clone()
    bad[0, 1, 7, 9] = float("nan")
    bad[0, 0, 0, 0] = float("inf")
    grads = ext.backward(bad, t["dx"], t["dy"], t["dc"], t["db"], its, 4)
    torch.cuda.synchronize()
    assert all(not g.any().item() for g in grads)
    expect = d["grad"].copy(); expect[0, 1, 7, 9] = 0; expect[0, 0, 0, 0] = 0
    np.testing.assert_array_equal(bad.cpu().numpy(), expect)  # scrubbed in the caller's tensor
    assert ext.get_state(4)[0] == 1
    grads = ext.backward(torch.zeros_like(bad), t["dx"], t["dy"], t["dc"], t["db"], its, 4)
    torch.cuda.synchronize()
    assert all(not g.any().item() for g in grads) and ext.get_state(4)[0] == 1
    # and the slot still serves a good upstream afterwards, identically
    again = ext.backward(t["grad"], t["dx"], t["dy"], t["dc"], t["db"], its, 4)
    torch.cuda.synchronize()
    for a, b in zip(again, base[1]):
        np.testing.assert_array_equal(a.cpu().numpy(), b)
    assert ext.get_state(4)[0] == 2


def test_ids_are_independent_and_separate_from_tv(ext, tgv_oracle):
    from customnetworklayers_amd.cudaTV import tvInpaint_cuda_ext as tv_ext
    from customnetworklayers_amd.workloads import tv_inputs

    dev = torch.device("cuda:0")
    cases = [tgv_inputs(1, 1, 24 * (i + 1), 40 * (i + 1), seed=30 + i) for i in range(3)]
    its = 10
    tens = [{k: torch.from_numpy(v).to(dev) for k, v in d.items()} for d in cases]
    for i in range(3):
        ext.reset_id(i)
    sols = [ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, i)[0] for i, t in enumerate(tens)]
    # a TV forward on the same id numbers in between must not disturb the TGV slots
    tvd = {k: torch.from_numpy(v).to(dev) for k, v in tv_inputs(1, 2, 16, 16, seed=1).items()}
    for i in range(3):
        tv_ext.forward(tvd["dx"], tvd["dy"], tvd["dc"], tvd["db"], tvd["di"], 4, i)
    grads = {}
    for i in (2, 1, 0):
        t = tens[i]
        grads[i] = ext.backward(t["grad"], t["dx"], t["dy"], t["dc"], t["db"], its, i)
    torch.cuda.synchronize()
    for i, d in enumerate(cases):
        ref = run_oracle(tgv_oracle, d, its, i)
        compare("id%d" % i, (sols[i].cpu().numpy(), [g.cpu().numpy() for g in grads[i]], None), ref)


def test_guard_rescales_kills_and_touches_u_only(ext, tgv_oracle):
    c = 2
    d = tgv_inputs(1, c, 32, 48, seed=8)
    its = 8
    base = run_gpu(ext, d, its, 5)
    st0 = ext.get_state(5)
    stats = ext.guard_stats(5)
    assert all(row[4] == 0 for row in stats)
    # running means 20x below (C: rescale), 40x below (X: kill, threshold 35), 100x below (I: kill)
    state = [10, st0[1] / 20, st0[2] / 40, st0[3], st0[4], st0[5] / 100]
    ext.set_state(5, state)
    tgv_oracle.reset_id(5)
    tgv_oracle.set_state(5, state)
    got = run_gpu(ext, d, its, 5, fresh=False)
    ref = run_oracle(tgv_oracle, d, its, 5, fresh=False)
    stats = ext.guard_stats(5)
    assert [int(r[4]) for r in stats] == [1, 2, 0, 0, 2]
    assert not got[1][0].any()  # gx killed
    np.testing.assert_allclose(got[1][2], base[1][2] * 0.5, rtol=1e-5, atol=0)  # gc halved
    assert not got[1][4][0, :c].any()  # u block of gi killed
    np.testing.assert_array_equal(got[1][4][0, c:], base[1][4][0, c:])  # v1, v2 gradients pass through
    compare("guard", got, ref)
    gs, os_ = ext.get_state(5), tgv_oracle.get_state(5)
    np.testing.assert_allclose(gs, os_, rtol=1e-9)
    assert gs[0] == 11


def test_errors(ext):
    dev = torch.device("cuda:0")
    d = {k: torch.from_numpy(v).to(dev) for k, v in tgv_inputs(1, 2, 8, 8, seed=1).items()}
    with pytest.raises(IndexError):
        ext.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], 4, 10)
    with pytest.raises(TypeError):
        ext.forward(d["dx"].double(), d["dy"], d["dc"], d["db"], d["di"], 4, 0)
    with pytest.raises(RuntimeError):
        ext.forward(d["dx"].cpu(), d["dy"], d["dc"], d["db"], d["di"], 4, 0)
    with pytest.raises(ValueError):  # one-channel diffusion tensor
        ext.forward(d["dx"][:, :1].contiguous(), d["dy"], d["dc"], d["db"], d["di"], 4, 0)
    with pytest.raises(ValueError):  # starting point without the auxiliary variables
        ext.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"][:, :2].contiguous(), 4, 0)
    ext.forward(d["dx"], d["dy"], d["dc"], d["db"], d["di"], 4, 0)
    with pytest.raises(RuntimeError):  # its differs from the forward that filled the slot
        ext.backward(d["grad"], d["dx"], d["dy"], d["dc"], d["db"], 6, 0)


def test_module_surface_and_autograd(ext, tgv_oracle):
    from customnetworklayers_amd import TGVInpaint

    dev = torch.device("cuda:0")
    d = tgv_inputs(1, 1, 30, 44, seed=9)
    hwc = lambda a: torch.from_numpy(np.ascontiguousarray(a[0].transpose(1, 2, 0))).to(dev).requires_grad_(True)
    tx, ty, tc, tb, ti = (hwc(d[k]) for k in ("dx", "dy", "dc", "db", "di"))
    layer = TGVInpaint(dev, 14, pid=3)
    ext.reset_id(3)
    sol = layer(tx, ty, tc, tb, ti)
    assert tuple(sol.shape) == (30, 44, 3)
    up = torch.from_numpy(np.ascontiguousarray(d["grad"][0].transpose(1, 2, 0))).to(dev)
    sol.backward(up)
    ref = run_oracle(tgv_oracle, d, 14, 3)
    got_grads = [t.grad.permute(2, 0, 1).unsqueeze(0).cpu().numpy() for t in (tx, ty, tc, tb, ti)]
    compare("module", (sol.detach().permute(2, 0, 1).unsqueeze(0).cpu().numpy(), got_grads, None), ref)


@pytest.mark.parametrize("n,c,h,w,its", [(2, 2, 40, 130, 20), (1, 1, 30, 70, 9), (1, 3, 20, 64, 6), (1, 4, 45, 70, 20)])
def test_kept_iterates_or_recomputed_segments_give_the_same_bits(ext, tgv_oracle, n, c, h, w, its, monkeypatch):
    # keep mode 2 (default) stores every x05 row in the forward and recomputes nothing; mode 1 keeps the last
    # segment's rows, which serve one backward; mode 0 recomputes every segment as the reference does.  A second
    # backward on one forward, a too-small memory budget and the per-call `keep` argument are covered as well.
    d = varying_inputs(n, c, h, w, seed=55)
    ref = run_oracle(tgv_oracle, d, its, 2)
    dev = torch.device("cuda:0")
    t = {k: torch.from_numpy(v).to(dev) for k, v in d.items()}

    def fwd_bwd(twice=False, **kw):
        ext.reset_id(2)
        if "mode" in kw:
            ext.keep_iterates(2, kw["mode"])
        (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, 2, **{k: v for k, v in kw.items() if k == "keep"})
        grads = ext.backward(t["grad"].clone(), t["dx"], t["dy"], t["dc"], t["db"], its, 2)
        if twice:
            ext.set_state(2, [0.0] * 6)
            again = ext.backward(t["grad"].clone(), t["dx"], t["dy"], t["dc"], t["db"], its, 2)
            for a, b in zip(grads, again):
                assert torch.equal(a, b)
        nbytes = ext.slot_bytes(2) if hasattr(ext, "slot_bytes") else 0
        return sol, grads, nbytes

    sol, first, bytes_all = fwd_bwd(twice=True)
    compare("all kept", (sol.cpu().numpy(), [g.cpu().numpy() for g in first], None), ref)
    runs = {"mode 2": fwd_bwd(mode=2, twice=True), "mode 1": fwd_bwd(mode=1, twice=True),
            "mode 0": fwd_bwd(mode=0, twice=True), "keep=0 once": fwd_bwd(keep=0), "after keep=0": fwd_bwd()}
    monkeypatch.setenv("INPAINT_KEEP_GB", "0.000001")  # the rows do not fit: the last segment's are kept instead
    runs["budget"] = fwd_bwd(twice=True)
    monkeypatch.delenv("INPAINT_KEEP_GB")
    monkeypatch.setenv("INPAINT_KEEP", "0")
    runs["env 0"] = fwd_bwd()
    monkeypatch.delenv("INPAINT_KEEP")
    monkeypatch.setenv("INPAINT_KEEP_LAST", "0")
    runs["env last 0"] = fwd_bwd()
    for name, (s2, grads, _) in runs.items():
        assert torch.equal(sol, s2), name
        for a, b in zip(first, grads):
            assert torch.equal(a, b), name
    if bytes_all:  # a slot that recomputes is smaller than one that keeps every row
        assert runs["mode 0"][2] < bytes_all
    with pytest.raises(ValueError):
        ext.keep_iterates(2, 3)
    ext.reset_id(2)


# the quirk toggles of the oracle that the corrected gradient switches off (clamp and guard stay)
CORRECTED = dict(end_uses_ckpt_y=0, skip_iter0_adjoint=0, getyk_rebuild=0, scale_factors=0, clamp=1, guard=1, dw_div=0)


@pytest.mark.parametrize("n,c,h,w,its", [
    (1, 2, 64, 128, 20), (2, 1, 37, 101, 9), (1, 1, 16, 64, 2), (1, 2, 1, 70, 4), (1, 1, 33, 1, 4),
    (2, 2, 90, 200, 30), (1, 2, 21, 63, 3), (1, 3, 23, 70, 10), (2, 4, 41, 130, 20),
])
def test_corrected_gradient_matches_the_oracle_with_the_same_quirks_off(ext, tgv_oracle, n, c, h, w, its):
    # gradient_mode 1: y (all three variables) as the forward pass made it, no checkpoint stand-in at segment starts,
    # the v2 block's division replaced by the product, iteration 0 back-propagated, multipliers 1 -- the oracle with
    # exactly these toggles off is the checker; every keep mode
    d = varying_inputs(n, c, h, w, seed=n * 100 + h + w + its)
    try:
        tgv_oracle.set_quirks(**CORRECTED)
        ref = run_oracle(tgv_oracle, d, its, 2)
    finally:
        tgv_oracle.set_quirks()
    plain = run_oracle(tgv_oracle, d, its, 2)
    assert any(not np.array_equal(a, b) for a, b in zip(ref[1], plain[1]))  # the toggles do something
    dev = torch.device("cuda:0")
    t = {k: torch.from_numpy(v).to(dev) for k, v in d.items()}
    try:
        for keep in (2, 1, 0):
            ext.reset_id(2)
            ext.gradient_mode(2, 1)
            ext.keep_iterates(2, keep)
            (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, 2)
            grads = ext.backward(t["grad"].clone(), t["dx"], t["dy"], t["dc"], t["db"], its, 2)
            got = (sol.cpu().numpy(), [g.cpu().numpy() for g in grads], None)
            compare("corrected, keep %d" % keep, got, ref)
            for a, b in zip(got[1], ref[1]):
                assert np.array_equal(a, b)
    finally:
        ext.reset_id(2)  # back to the reference's gradient
    compare("plain again", run_gpu(ext, d, its, 2), plain)


def test_corrected_gradient_is_the_gradient_of_the_forward_pass(ext, tgv_oracle):
    # with the clamp and the guard idle the corrected gradient is the true one: the float64 oracle with every quirk
    # off (which the CPU pins equate with automatic differentiation of an independent forward pass) agrees to
    # float32 accuracy
    n, c, h, w, its = 1, 2, 24, 40, 12
    d = varying_inputs(n, c, h, w, seed=5)
    d64 = {k: v.astype(np.float64) for k, v in d.items()}
    try:
        tgv_oracle.set_quirks(0, 0, 0, 0, 0, 0, 0)
        tgv_oracle.reset_id(3)
        tgv_oracle.forward(d64["dx"], d64["dy"], d64["dc"], d64["db"], d64["di"], its, 3, f64=True)
        true = tgv_oracle.backward(d64["grad"].copy(), d64["dx"], d64["dy"], d64["dc"], d64["db"], its, 3, f64=True)
    finally:
        tgv_oracle.set_quirks()
    dev = torch.device("cuda:0")
    t = {k: torch.from_numpy(v).to(dev) for k, v in d.items()}
    try:
        ext.reset_id(2)
        ext.gradient_mode(2, 1)
        ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, 2)
        grads = [g.cpu().numpy() for g in ext.backward(t["grad"].clone(), t["dx"], t["dy"], t["dc"], t["db"], its, 2)]
    finally:
        ext.reset_id(2)
    errs = [rel_err(g, r) for g, r in zip(grads, true)]
    print("\ncorrected gradient vs float64 true gradient: gx %.2e gy %.2e gc %.2e gb %.2e gi %.2e" % tuple(errs), flush=True)
    for e in errs:
        assert e <= 1e-3
    plain = run_gpu(ext, d, its, 2)[1]
    assert rel_err(plain[3], true[3]) > 0.5  # the reference's gradient is a different vector


def test_gradient_mode_takes_zero_or_one(ext):
    with pytest.raises(ValueError):
        ext.gradient_mode(2, 2)
    with pytest.raises(ValueError):
        ext.gradient_mode(2, -1)


@pytest.mark.parametrize("env,c", [({"INPAINT_TGV_PAIR_WAVES": "2"}, 1), ({"INPAINT_TGV_FUSE_ADJ": "0"}, 2),
                                   ({"INPAINT_TGV_PAIR_WAVES": "1"}, 2)])
def test_corrected_gradient_on_the_other_kernel_selections(ext, tgv_oracle, env, c, monkeypatch):
    # one channel in the two-wavefront pair kernel, two channels one step per launch, and two channels with the
    # one-wavefront pair kernel selected (which has no corrected form: the layer must fall back to single steps)
    n, h, w, its = 2, 45, 130, 12
    d = varying_inputs(n, c, h, w, seed=17 + c)
    try:
        tgv_oracle.set_quirks(**CORRECTED)
        ref = run_oracle(tgv_oracle, d, its, 2)
    finally:
        tgv_oracle.set_quirks()
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    dev = torch.device("cuda:0")
    t = {k: torch.from_numpy(v).to(dev) for k, v in d.items()}
    try:
        ext.reset_id(2)
        ext.gradient_mode(2, 1)
        (sol,) = ext.forward(t["dx"], t["dy"], t["dc"], t["db"], t["di"], its, 2)
        grads = ext.backward(t["grad"].clone(), t["dx"], t["dy"], t["dc"], t["db"], its, 2)
        got = (sol.cpu().numpy(), [g.cpu().numpy() for g in grads], None)
    finally:
        ext.reset_id(2)
    compare("corrected, %s" % env, got, ref)
    for a, b in zip(got[1], ref[1]):
        assert np.array_equal(a, b)
