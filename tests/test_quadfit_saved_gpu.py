"""The fit's backward pass from the costs its forward pass saved: both outputs and the gradient wrt the first map are the ones of
the pair without, bit for bit, the gradient wrt the second map within the rounding of sums in another order.  Shapes at the edges
of the tiles (64 x 8 pixels) and of the ring of windows (channel counts below and above its depth), flows that keep a tile's taps
in its window, that leave it, and that scatter the whole tile."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SCATTER_TOL = 1e-5  # of the largest entry: the sum over the pixels that land on one, in another order


@pytest.fixture(scope="module")
def qf():
    from customnetworklayers_amd.cudaQuadFit import QuadFit_cuda_ext

    return QuadFit_cuda_ext


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def inputs(n, c, h, w, amp, seed=0, fc=3):
    rng = np.random.default_rng(seed + c + h + w)
    flow = (amp * rng.standard_normal((n, fc, h, w))).astype(np.float32)
    flow[:, :, 0, 0] = np.nan
    return (rng.standard_normal((n, c, h, w)).astype(np.float32), rng.standard_normal((n, c, h, w)).astype(np.float32), flow,
            rng.standard_normal((n, 3, h, w)).astype(np.float32))


def check(qf, o, f0, f1, flow, grad, name):
    print("case", name, flush=True)
    a = dev(f0), dev(f1), dev(flow)
    out, costs = qf.forward_saving(*a)
    g0, g1 = qf.backward(dev(grad), *a, costs=costs)
    r0, r1 = o.quadfit_backward(grad, f0, f1, flow)
    assert np.array_equal(out.cpu().numpy(), o.quadfit_forward(f0, f1, flow))
    assert np.array_equal(g0.cpu().numpy(), r0)
    assert np.abs(g1.cpu().numpy() - r1).max() <= SCATTER_TOL * max(np.abs(r1).max(), 1e-30)


@pytest.mark.parametrize("amp", [0.7, 4.0, 30.0])
@pytest.mark.parametrize("n,c,h,w", [(1, 1, 1, 1), (1, 2, 8, 64), (1, 3, 9, 65), (2, 4, 7, 63), (1, 5, 40, 130), (2, 6, 17, 100),
                                     (1, 32, 24, 200), (1, 33, 16, 129), (1, 64, 33, 90), (1, 130, 12, 70)])
def test_saved_costs_give_the_same_gradients(qf, flowaux_oracle, n, c, h, w, amp):
    check(qf, flowaux_oracle, *inputs(n, c, h, w, amp), "%dx%dx%dx%d, noise %g" % (n, c, h, w, amp))


@pytest.mark.parametrize("spread", [0, 12, 18, 40])
def test_windows_of_every_size(qf, flowaux_oracle, spread):
    # one row of every tile displaced by `spread` rows: the window grows through the ring's three sizes and past its capacity
    f0, f1, flow, grad = inputs(1, 9, 120, 192, 0.3)
    flow[:, 1, ::8] += spread
    check(qf, flowaux_oracle, f0, f1, flow, grad, "spread %d" % spread)


def test_autograd_saves_the_costs_where_it_pays(qf, flowaux_oracle):
    from customnetworklayers_amd import QuadFittingFromFlowFunction

    for (n, c, h, w), kept_tensors in (((1, 8, 200, 704), 4), ((1, 33, 192, 640), 4), ((1, 8, 192, 640), 3), ((1, 33, 40, 64), 3)):
        f0, f1, flow, grad = inputs(n, c, h, w, 1.0)
        a, b = dev(f0).requires_grad_(True), dev(f1).requires_grad_(True)
        kept = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: kept.append(t.shape) or t.cpu(), lambda t: t.cuda()):
            sol = QuadFittingFromFlowFunction.apply(a, b, dev(flow))
        assert len(kept) == kept_tensors
        sol.backward(dev(grad))
        r0, r1 = flowaux_oracle.quadfit_backward(grad, f0, f1, flow)
        assert np.array_equal(a.grad.cpu().numpy(), r0)
        assert np.abs(b.grad.cpu().numpy() - r1).max() <= SCATTER_TOL * np.abs(r1).max()


def test_saved_errors(qf):
    f0, f1, flow, grad = (dev(t) for t in inputs(1, 4, 10, 12, 1.0))
    _, costs = qf.forward_saving(f0, f1, flow)
    with pytest.raises(ValueError):
        qf.backward(grad, f0, f1, flow, costs=costs[:4].contiguous())
    with pytest.raises(ValueError):
        qf.backward(grad, f0, f1, flow, use_atomics=True, costs=costs)
    with pytest.raises(RuntimeError):
        qf.backward(grad, f0, f1, flow, costs=costs.cpu())
    with pytest.raises(TypeError):
        qf.backward(grad, f0, f1, flow, costs=costs.double())
