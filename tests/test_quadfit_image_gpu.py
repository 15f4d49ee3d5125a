"""The fit's module on one image with its channels innermost: the kernels that take this layout against the oracle on the
permuted planes -- outputs and the gradient wrt the first map bit for bit, the gradient wrt the second within the rounding of sums
in another order -- at channel counts around the vector width and the chunk of 32, pixel counts around the block's 64, and for
every layout of maps and flow that the module takes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SCATTER_TOL = 1e-5  # of the largest entry: the sum over the pixels that land on one, in another order


def inputs(c, h, w, amp, seed=0):
    rng = np.random.default_rng(seed + c + h + w)
    flow = (amp * rng.standard_normal((h, w, 3))).astype(np.float32)
    flow[0, 0] = np.nan
    return (rng.standard_normal((h, w, c)).astype(np.float32), rng.standard_normal((h, w, c)).astype(np.float32), flow,
            rng.standard_normal((h, w, 3)).astype(np.float32))


def planes(a):
    return np.ascontiguousarray(a.transpose(2, 0, 1)[None])


def expected(o, f0, f1, flow, grad):
    a = planes(f0), planes(f1), planes(flow)
    out, (g0, g1) = o.quadfit_forward(*a), o.quadfit_backward(planes(grad), *a)
    return [t[0].transpose(1, 2, 0) for t in (out, g0, g1)]


def run(f0, f1, flow, grad):
    from customnetworklayers_amd import QuadFittingFromFlow

    layer = QuadFittingFromFlow(torch.device("cuda:0"))
    f0.requires_grad_(True), f1.requires_grad_(True)
    out = layer(f0, f1, flow)
    assert out.is_contiguous()
    g0, g1 = torch.autograd.grad(out, [f0, f1], grad)
    with torch.no_grad():
        assert torch.equal(layer(f0, f1, flow), out)
    return [t.detach().cpu().numpy() for t in (out, g0, g1)]


def check(got, want):
    assert np.array_equal(got[0], want[0])
    assert np.array_equal(got[1], want[1])
    assert np.abs(got[2] - want[2]).max() <= SCATTER_TOL * max(np.abs(want[2]).max(), 1e-30)


def negative_view(t):
    """t as a view whose sign is still to be applied: the imaginary part of a conjugate."""
    view = torch.complex(torch.zeros_like(t), -t).conj().imag
    assert view.is_neg() and torch.equal(view.nan_to_num(), t.nan_to_num())
    return view


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("amp", [0.7, 5.0])
@pytest.mark.parametrize("h,w", [(1, 2), (1, 64), (7, 9), (5, 13), (16, 64), (33, 70)])
@pytest.mark.parametrize("c", [2, 3, 4, 5, 8, 31, 32, 33, 36, 64, 65, 100])
def test_image_matches_the_oracle(flowaux_oracle, c, h, w, amp):
    print("case", c, h, w, amp, flush=True)
    a = inputs(c, h, w, amp)
    check(run(*(dev(t) for t in a)), expected(flowaux_oracle, *a))


@pytest.mark.parametrize("c", [6, 32])
def test_image_many_sources_per_position(flowaux_oracle, c):
    f0, f1, flow, grad = inputs(c, 20, 50, 0.0)
    flow[..., 0] = 20 - np.arange(50)[None, :] * 0.97   # whole rows onto a few columns: full lists and the overflow
    check(run(*(dev(t) for t in (f0, f1, flow, grad))), expected(flowaux_oracle, f0, f1, flow, grad))


@pytest.mark.parametrize("h", [2, 5, 130])
@pytest.mark.parametrize("layout", ["contiguous", "a batch's only column", "planes", "wider image"])
def test_one_column(flowaux_oracle, h, layout):
    print("case", h, layout, flush=True)
    a = inputs(8, h, 1, 0.7)
    f0, f1, flow, grad = (dev(t) for t in a)
    if layout == "a batch's only column":  # (contiguous, with a stride of 3 * h between columns)
        f0, f1, flow, grad = (t.reshape(1, h, -1).transpose(0, 1) for t in (f0, f1, flow, grad))
        assert flow.is_contiguous() and flow.stride() == (3, 3 * h, 1)
    if layout == "planes":
        flow = flow.permute(2, 0, 1).contiguous().permute(1, 2, 0)
    if layout == "wider image":
        flow = torch.cat([flow, flow], 1)[:, :1]
    check(run(f0.detach(), f1.detach(), flow, grad), expected(flowaux_oracle, *a))


@pytest.mark.parametrize("layout", ["flow planes", "flow strided", "maps planes", "one map planes", "maps strided", "maps shifted", "grad strided",
                                    "flow negative", "one map negative", "grad negative"])
def test_layouts_the_module_takes(flowaux_oracle, layout):
    a = inputs(8, 12, 30, 1.0)
    f0, f1, flow, grad = (dev(t) for t in a)
    as_planes = lambda t: t.permute(2, 0, 1).contiguous().permute(1, 2, 0)  # noqa: E731
    if layout == "flow planes":
        flow = as_planes(flow)
    if layout == "flow strided":
        flow = torch.cat([flow, flow], 1)[:, :30]
    if layout in ("maps planes", "one map planes"):
        f0 = as_planes(f0)
        f1 = as_planes(f1) if layout == "maps planes" else f1
    if layout == "maps strided":
        f0 = torch.cat([f0, f0], 2)[..., :8]
    if layout == "maps shifted":  # contiguous, but not 16-byte aligned
        f0, f1 = (torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape) for t in (f0, f1))
    if layout == "grad strided":
        grad = as_planes(grad)
    if layout == "flow negative":
        flow = negative_view(flow)
    if layout == "one map negative":
        f0 = negative_view(f0)
    if layout == "grad negative":
        grad = negative_view(grad)
    check(run(f0.detach(), f1.detach(), flow, grad), expected(flowaux_oracle, *a))


@pytest.mark.parametrize("c,h,w", [(2, 512, 1023), (2, 512, 1024), (3, 512, 1024), (4, 896, 1023), (4, 896, 1024)])
def test_few_channels_on_both_sides_of_the_rule(flowaux_oracle, c, h, w):
    from customnetworklayers_amd import QuadFittingFromFlow
    from customnetworklayers_amd.cudaQuadFit import QuadFit_cuda_ext as ext

    a = inputs(c, h, w, 0.7)
    f0, f1, flow, _ = (dev(t) for t in a)
    assert ext.takes_image(f0, f1, flow) == (h * w < (7 << 17 if c == 4 else 1 << 19))
    assert ext.takes_image(f0.requires_grad_(True), f1, flow)
    with torch.no_grad():
        got = QuadFittingFromFlow(torch.device("cuda:0"))(f0, f1, flow).cpu().numpy()
    want = flowaux_oracle.quadfit_forward(*(planes(t) for t in a[:3]))[0].transpose(1, 2, 0)
    assert np.array_equal(got, want)


def test_image_refuses_what_the_planes_refuse():
    from customnetworklayers_amd import QuadFittingFromFlow

    layer = QuadFittingFromFlow(torch.device("cuda:0"))
    f0, f1, flow, _ = (dev(t) for t in inputs(4, 6, 7, 1.0))
    with pytest.raises(TypeError):
        layer(f0.double(), f1.double(), flow)
    with pytest.raises(RuntimeError):
        layer(f0.cpu(), f1, flow)
    with pytest.raises(ValueError):
        layer(f0, f1[..., :3].contiguous(), flow)
    with pytest.raises(ValueError):
        layer(f0, f1, flow[:5].contiguous())
    with pytest.raises(AssertionError):
        layer(f0, f1, flow[..., :2].contiguous())


def test_gradient_wrt_the_flow_only_is_none(flowaux_oracle):
    from customnetworklayers_amd import QuadFittingFromFlow

    f0, f1, flow, grad = (dev(t) for t in inputs(4, 6, 7, 1.0))
    out = QuadFittingFromFlow(torch.device("cuda:0"))(f0, f1, flow.requires_grad_(True))
    out.backward(grad)
    assert flow.grad is None
