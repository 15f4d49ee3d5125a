"""The median's backward pass from the crossing its forward pass saved: the gradient is the one that the walk over the
histogram gives, bit for bit, over every bin count's kernels, ragged pixel counts and histograms whose running sum does not
stay above one half."""
import numpy as np
import pytest
import torch

from customnetworklayers_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def med():
    from customnetworklayers_amd.cudaMedian import median_cuda_ext

    return median_cuda_ext


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def check(med, o, vol, grad):
    print("case", vol.shape, flush=True)
    v = dev(vol)
    out, saved = med.forward_saving(v)
    (g,) = med.backward(dev(grad), v, saved)
    assert np.array_equal(out.cpu().numpy(), o.median_forward(vol), equal_nan=True)
    assert np.array_equal(g.cpu().numpy(), o.median_backward(grad, vol), equal_nan=True)
    assert torch.equal(torch.nan_to_num(g), torch.nan_to_num(med.backward(dev(grad), v)[0]))


@pytest.mark.parametrize("n,h,w", [(1, 1, 1), (1, 8, 8), (1, 5, 13), (2, 9, 31), (3, 7, 11)])
@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 6, 7, 33, 39, 40, 41, 64, 130, 255])
def test_saved_crossing_gives_the_same_gradient(med, flowaux_oracle, n, h, w, d):
    m = workloads.median_inputs(n, h, w, d, seed=n + h + w + d, empty_fraction=0.1)
    check(med, flowaux_oracle, m["vol"], m["grad"])


@pytest.mark.parametrize("d", [3, 33, 40, 64])
@pytest.mark.parametrize("which", ["one pixel", "all pixels"])
def test_sums_that_fall_below_one_half_again_or_are_not_numbers(med, flowaux_oracle, d, which):
    rng = np.random.default_rng(d)
    m = workloads.median_inputs(2, 13, 17, d, seed=d, empty_fraction=0.1)
    vol = m["vol"].copy()
    if which == "all pixels":
        vol = rng.normal(0.05, 0.3, vol.shape).astype(np.float32)
    odd = vol.reshape(-1, d)
    odd[70] = 0.0
    odd[70, 0], odd[70, d - 1] = 0.75, -0.5       # back below one half in the last bin
    odd[200, 0] = np.nan                           # no crossing, all sums NaN
    odd[201] = 0.25
    odd[201, d - 1] = np.nan                       # NaN in (or in front of) the crossing, or behind it
    odd[202, 0], odd[202, 1] = 0.5, -np.inf
    odd[203, 0] = np.inf
    odd[300, :] = -1.0
    check(med, flowaux_oracle, vol, m["grad"])


@pytest.mark.parametrize("d", [5, 6, 7, 33, 34, 35])
def test_many_tiles_side_by_side_on_a_unit(med, flowaux_oracle, d):
    # some twenty tiles of 64 pixels for every compute unit, as many as its LDS holds at once: a tile whose last load reached past
    # its own rows would be seen in a neighbour's
    m = workloads.median_inputs(2, 401, 413, d, seed=d, empty_fraction=0.05)
    check(med, flowaux_oracle, m["vol"], m["grad"])
    (plain,) = med.forward(dev(m["vol"]))
    assert np.array_equal(plain.cpu().numpy(), flowaux_oracle.median_forward(m["vol"]))


def test_saved_crossing_without_16_byte_alignment(med, flowaux_oracle):
    m = workloads.median_inputs(1, 9, 14, 21, seed=9)
    flat = torch.zeros(m["vol"].size + 3, dtype=torch.float32, device="cuda")
    for shift in (1, 2, 3):
        v = flat[shift:shift + m["vol"].size].view(m["vol"].shape)
        v.copy_(dev(m["vol"]))
        out, saved = med.forward_saving(v)
        assert np.array_equal(out.cpu().numpy(), flowaux_oracle.median_forward(m["vol"]))
        assert np.array_equal(med.backward(dev(m["grad"]), v, saved)[0].cpu().numpy(), flowaux_oracle.median_backward(m["grad"], m["vol"]))


def test_autograd_saves_the_crossing_up_to_255_bins(med, flowaux_oracle):
    from customnetworklayers_amd import MedianFunction

    for d in (255, 256):
        m = workloads.median_inputs(1, 6, 9, d, seed=d)
        v = dev(m["vol"]).requires_grad_(True)
        kept = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t.shape) or t.cpu(), lambda t: t.cuda()):
            sol = MedianFunction.apply(v)
        assert len(kept) == (2 if d == 255 else 1)
        sol.backward(dev(m["grad"]))
        assert np.array_equal(v.grad.cpu().numpy(), flowaux_oracle.median_backward(m["grad"], m["vol"]))


def test_saved_errors(med):
    m = workloads.median_inputs(1, 4, 5, 6, seed=1)
    v, g = dev(m["vol"]), dev(m["grad"])
    _, saved = med.forward_saving(v)
    with pytest.raises(ValueError):
        med.backward(g, v, saved[:2].contiguous())
    with pytest.raises(RuntimeError):
        med.backward(g, v, saved.cpu())
    with pytest.raises(TypeError):
        med.backward(g, v, saved.double())
    with pytest.raises(ValueError):
        med.forward_saving(torch.zeros(1, 2, 2, 256, dtype=torch.float32, device="cuda"))
