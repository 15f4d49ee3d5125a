"""The work a user of this framework has it do, as a list of cases that can be timed and compared.

Every case is one pass through the public entry points: the autograd Functions for a batch, the H x W x C modules (the
drop-in surface) for a single image, float32 throughout, as the layers take nothing else.

kind      fields                            one pass
tv        n c h w its train corrected       TV inpainting layer: solution, and in training the five gradients
tgv       n c h w its train corrected       the same with the second-order layer
stack     n c h w levels its                coarse-to-fine TV layers (h, w: the coarsest level), each level's solution
                                            upsampled into the next one's right-hand side; all gradients
quadfit   n c h w train                     sub-pixel fit of a matching cost over c-channel feature maps
median    n h w d train                     median of a per-pixel histogram over d displacement bins

`corrected`: back-propagate the gradient of the forward pass itself instead of the reference's hand-derived one.
"""
import math

import torch
import torch.nn.functional as F

from customnetworklayers_amd import (Median, MedianFunction, QuadFittingFromFlow, QuadFittingFromFlowFunction, TGVInpaint,
                                     TGVInpaintingFunction, TVInpaint, TVInpaintingFunction)
from customnetworklayers_amd.cudaTGV import tgvInpaint_cuda_ext
from customnetworklayers_amd.cudaTV import tvInpaint_cuda_ext
from customnetworklayers_amd.hierarchy import next_level

DEV = "cuda"
TV_ID, TGV_ID = 6, 3  # the modules' default ids


def _tv(name, n, c, h, w, its, train=True, corrected=False, kind="tv"):
    return dict(name=name, kind=kind, n=n, c=c, h=h, w=w, its=its, train=train, corrected=corrected)


def listed():
    return [
        # the smallest problem in use, the single-sample TV workload of the benchmark: launches and host work
        _tv("tv_small", 1, 2, 64, 128, 20),
        # a flow field of odd size filled in at inference (nobody differentiates), one image at a time
        _tv("tv_infer", 1, 2, 187, 621, 50, train=False),
        # one full-size single-channel map (a disparity) in training with the corrected gradient
        _tv("tv_disparity", 1, 1, 384, 1248, 100, corrected=True),
        # the headline workload: a training batch of full-size flow fields
        _tv("tv_batch", 4, 2, 384, 1248, 100),
        # three levels coarse to fine, forward and backward through all of them
        dict(name="tv_stack", kind="stack", n=2, c=2, h=112, w=256, levels=3, its=50),
        # the second-order layer on a small, ragged disparity map
        _tv("tgv_small", 1, 1, 61, 97, 30, kind="tgv"),
        # the second-order layer at inference on one full-size image of odd width
        _tv("tgv_infer", 1, 2, 375, 1241, 100, train=False, kind="tgv"),
        # the second-order layer on a training batch
        _tv("tgv_batch", 4, 2, 384, 1248, 100, kind="tgv"),
        # the fit on a coarse level: small maps, many channels
        dict(name="quadfit_coarse", kind="quadfit", n=1, c=64, h=96, w=312, train=True),
        # the fit at full size, a training batch
        dict(name="quadfit_batch", kind="quadfit", n=4, c=32, h=384, w=1248, train=True),
        # a histogram volume with a power-of-two number of bins at inference, odd size
        dict(name="median_infer", kind="median", n=2, h=187, w=621, d=64, train=False),
        # the median at full size, a training batch
        dict(name="median_batch", kind="median", n=4, h=384, w=1248, d=33, train=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tv", "tv", "tv", "tgv", "tgv", "stack", "quadfit", "quadfit", "median"])
    n = rng.choice([1, 1, 2, 3, 4])
    while True:
        if kind in ("tv", "tgv"):
            case = dict(kind=kind, n=n, c=rng.choice([1, 1, 2, 2, 2, 3] if kind == "tv" else [1, 2, 2]),
                        h=_log_int(rng, 48, 448), w=_log_int(rng, 64, 1280), its=_log_int(rng, 10, 100),
                        train=rng.random() < 0.7, corrected=rng.random() < 0.2)
            cost = case["n"] * case["c"] * case["h"] * case["w"] * case["its"]
            limit = 4 * 2 * 384 * 1248 * 100
        elif kind == "stack":
            case = dict(kind=kind, n=min(n, 2), c=rng.choice([1, 2]), h=rng.randint(40, 112), w=rng.randint(64, 256),
                        levels=rng.choice([2, 3]), its=rng.randint(10, 50))
            cost = case["n"] * case["c"] * case["h"] * case["w"] * 4 ** case["levels"] * case["its"]
            limit = 4 * 2 * 384 * 1248 * 100
        elif kind == "quadfit":
            case = dict(kind=kind, n=n, c=rng.choice([8, 16, 24, 32, 32, 48, 64]), h=_log_int(rng, 48, 448),
                        w=_log_int(rng, 64, 1280), train=rng.random() < 0.7)
            cost, limit = case["n"] * case["c"] * case["h"] * case["w"], 4 * 32 * 384 * 1248
        else:
            case = dict(kind=kind, n=n, h=_log_int(rng, 48, 448), w=_log_int(rng, 64, 1280), d=_log_int(rng, 9, 130),
                        train=rng.random() < 0.7)
            cost, limit = case["n"] * case["h"] * case["w"] * case["d"], 4 * 384 * 1248 * 33
        if cost <= limit:
            return case


# ---- inputs: those of customnetworklayers_amd/workloads.py, made on the GPU ---------------------------------------
class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device=DEV)


def _smooth(r, n, c, h, w, step):
    """Smooth random fields: noise on a grid `step` pixels wide, interpolated."""
    coarse = r.normal(n, c, h // step + 3, w // step + 3)
    return F.interpolate(coarse, size=(h, w), mode="bicubic", align_corners=False)


def _flow(r, n, c, h, w, amplitude=8.0, noise=0.5):
    """Sum of four random low-frequency sinusoids spanning +-amplitude, plus noise."""
    yy = torch.arange(h, device=DEV).view(1, 1, h, 1) / h
    xx = torch.arange(w, device=DEV).view(1, 1, 1, w) / w
    f = torch.zeros(n, c, h, w, device=DEV)
    for _ in range(4):
        fx, fy, phase = r.uniform(n, c, 1, 1, lo=-3, hi=3), r.uniform(n, c, 1, 1, lo=-3, hi=3), r.uniform(n, c, 1, 1, hi=2 * math.pi)
        f += r.uniform(n, c, 1, 1, lo=0.5) * torch.sin(2 * math.pi * (fx * xx + fy * yy) + phase)
    f *= amplitude / f.abs().amax((2, 3), keepdim=True)
    return f + noise * r.normal(n, c, h, w)


def _image(r, n, h, w):
    img = _smooth(r, n, 1, h, w, 5)
    lo, hi = img.amin((2, 3), keepdim=True), img.amax((2, 3), keepdim=True)
    return (img - lo) / (hi - lo)


def _edge_weights(img):
    dx, dy = torch.zeros_like(img), torch.zeros_like(img)
    dx[..., :-1] = (img[..., 1:] - img[..., :-1]).abs()
    dy[..., :-1, :] = (img[..., 1:, :] - img[..., :-1, :]).abs()
    return torch.exp(-10 * dx), torch.exp(-10 * dy)


def _confidence(r, n, h, w, density=0.2):
    return (r.uniform(n, 1, h, w) < density) * r.uniform(n, 1, h, w, lo=0.2)


def _hwc(t):
    return t[0].permute(1, 2, 0).contiguous()


def _inputs(case, r):
    """(inputs, upstream gradient), batched n c h w (the histogram: n h w d), and which inputs carry a gradient."""
    kind, n, h, w = case["kind"], case["n"], case["h"], case["w"]
    if kind in ("tv", "tgv"):
        c = case["c"]
        wx, wy = _edge_weights(_image(r, n, h, w))
        conf, b = _confidence(r, n, h, w), _flow(r, n, c, h, w)
        init = b.clone()
        if kind == "tgv":  # second weight channel: beta, constant; auxiliary variables start at zero
            wx, wy = (torch.cat([t, torch.full_like(t, 2.0)], 1) for t in (wx, wy))
            init = torch.cat([b, torch.zeros(n, 2 * c, h, w, device=DEV)], 1)
        return [wx, wy, conf, b, init], r.normal(*init.shape), [True] * 5
    if kind == "quadfit":
        c = case["c"]
        feat1 = _smooth(r, n, c, h, w, 3) + 0.1 * r.normal(n, c, h, w)
        true = _flow(r, n, 2, h, w, noise=0.0)
        ys, xs = torch.meshgrid(torch.arange(h, device=DEV), torch.arange(w, device=DEV), indexing="ij")
        grid = torch.stack([(xs + true[:, 0]) * (2 / max(w - 1, 1)) - 1, (ys + true[:, 1]) * (2 / max(h - 1, 1)) - 1], -1)
        feat0 = F.grid_sample(feat1, grid, padding_mode="border", align_corners=True)
        flow = torch.cat([true + 0.6 * r.normal(n, 2, h, w), r.uniform(n, 1, h, w)], 1)
        return [feat0, feat1, flow], r.normal(n, 3, h, w), [True, True, False]
    d = case["d"]
    centre = (d - 1) * (0.5 + 0.4 * _flow(r, n, 1, h, w, amplitude=1.0, noise=0.0)[:, 0])
    bins = torch.arange(d, device=DEV, dtype=torch.float32)
    vol = torch.softmax(-0.5 * ((bins - centre[..., None]) / 2.0) ** 2 + 0.5 * r.normal(n, h, w, d), -1)
    vol = vol * (1.0 - 0.7 * (r.uniform(n, h, w, 1) < 0.02))  # a few pixels with too little mass to have a median
    return [vol], r.normal(n, 2, h, w), [True]


def _prepare_stack(case, r):
    n, c, its = case["n"], case["c"], case["its"]
    sizes = [(case["h"] << k, case["w"] << k) for k in range(case["levels"])]
    wx, wy = _edge_weights(_image(r, n, *sizes[0]))
    s = dict(case=case, sizes=sizes, its=its, wx=wx, wy=wy, b=_flow(r, n, c, *sizes[0]),
             conf=[_confidence(r, n, h, w, 0.25) for h, w in sizes], img=[None] + [_image(r, n, h, w) for h, w in sizes[1:]],
             grad=r.normal(n, c, *sizes[-1]))
    s["wanted"] = [t.requires_grad_(True) for t in [s["wx"], s["wy"], s["b"]] + s["conf"]]
    return s


def prepare(case, seed):
    r = _Rng(seed)
    kind = case["kind"]
    # training starts: the gradient guard of each id in use has seen no runs yet
    if kind == "stack":
        for pid in range(case["levels"]):
            tvInpaint_cuda_ext.set_state(pid, [0.0] * 6)
            tvInpaint_cuda_ext.gradient_mode(pid, 0)
        return _prepare_stack(case, r)
    if kind in ("tv", "tgv"):
        ext, pid = (tvInpaint_cuda_ext, TV_ID) if kind == "tv" else (tgvInpaint_cuda_ext, TGV_ID)
        ext.set_state(pid, [0.0] * 6)
        ext.gradient_mode(pid, 1 if case["corrected"] else 0)
    inputs, grad, wanted = _inputs(case, r)
    module = case["n"] == 1  # a single image goes through the module, which takes H x W x C
    layer = None
    if module and kind == "median":
        inputs, grad, layer = [inputs[0][0].contiguous()], grad[0, 0].contiguous(), Median(torch.device(DEV))
    elif module:
        inputs, grad = [_hwc(t) for t in inputs], _hwc(grad)
        if kind == "quadfit":
            layer = QuadFittingFromFlow(torch.device(DEV))
        else:
            make, pid = (TVInpaint, TV_ID) if kind == "tv" else (TGVInpaint, TGV_ID)
            layer = make(torch.device(DEV), case["its"], pid, corrected_gradient=case["corrected"])
    if case["train"]:
        for t, want in zip(inputs, wanted):
            t.requires_grad_(want)
    return dict(case=case, inputs=inputs, grad=grad, layer=layer)


# ---- one pass ------------------------------------------------------------------------------------------------------
def _apply(s):
    case, inputs = s["case"], s["inputs"]
    if s["layer"] is not None:
        return s["layer"](*inputs)
    if case["kind"] == "tv":
        return TVInpaintingFunction.apply(*inputs, case["its"], TV_ID)
    if case["kind"] == "tgv":
        return TGVInpaintingFunction.apply(*inputs, case["its"], TGV_ID)
    if case["kind"] == "quadfit":
        return QuadFittingFromFlowFunction.apply(*inputs)
    return MedianFunction.apply(*inputs)


def _run_stack(s):
    wx, wy, b = s["wx"], s["wy"], s["b"]
    for pid in range(len(s["sizes"])):
        sol = TVInpaintingFunction.apply(wx, wy, s["conf"][pid], b, b, s["its"], pid)
        if pid + 1 < len(s["sizes"]):
            b, wx, wy = next_level(sol, s["img"][pid + 1])
    return [sol.detach()] + list(torch.autograd.grad(sol, s["wanted"], s["grad"]))


def run(s):
    case = s["case"]
    if case["kind"] == "stack":
        return _run_stack(s)
    if not case["train"]:
        with torch.no_grad():
            return [_apply(s)]
    sol = _apply(s)
    return [sol.detach()] + list(torch.autograd.grad(sol, [t for t in s["inputs"] if t.requires_grad], s["grad"]))


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
# Operations of one iteration per pixel and channel, counted off the definition with each triangle's weight formed
# once (a division, a square root or a comparison is one operation): gradient step, prox and extrapolation forward;
# the y rebuild, the transposed Jacobian with its rank-one terms and the weight / confidence gradients backward.
OPS = {"tv": (38, 95), "tgv": (100, 260)}


def work(case):
    kind, n, h, w = case["kind"], case["n"], case["h"], case["w"]
    px = n * h * w
    if kind in ("tv", "tgv"):
        c, its = case["c"], case["its"] // 2 * 2
        planes_in, planes_out = (3 + 2 * c, c) if kind == "tv" else (5 + 4 * c, 3 * c)
        ops = OPS[kind][0] * c * px * its
        if case["train"]:  # the upstream gradient in, one gradient per input out
            planes_in, planes_out = planes_in + planes_out, planes_out + planes_in
            ops += OPS[kind][1] * c * px * its
        return dict(bytes=4 * px * (planes_in + planes_out), flops=ops)
    if kind == "stack":
        c, its, levels = case["c"], case["its"] // 2 * 2, case["levels"]
        every = sum(px << 2 * k for k in range(levels))
        fine = px << 2 * (levels - 1)
        # in: confidences, guidance images behind the first level, coarsest weights and flow, upstream gradient;
        # out: the solution and the gradients wrt all but the images
        planes = every + (every - px) + (2 + c) * px + c * fine + c * fine + every + (2 + c) * px
        return dict(bytes=4 * planes, flops=sum(OPS["tv"]) * c * every * its)
    if kind == "quadfit":
        c = case["c"]
        planes, ops = 2 * c + 2 + 3, 10 * c + 30
        if case["train"]:
            planes, ops = planes + 3 + 2 * c, ops + 20 * c + 30
        return dict(bytes=4 * px * planes, flops=px * ops)
    d = case["d"]
    planes, ops = d + 2, 2 * d
    if case["train"]:
        planes, ops = planes + 2 + d, ops + 2 * d
    return dict(bytes=4 * px * planes, flops=px * ops)


def tolerance(case):
    """About four times what the layers differ from themselves in 64 bits (CPU statement of the same arithmetic)."""
    kind = case["kind"]
    if kind == "tv" and not case["train"]:
        return {"rel": 1e-6, "max": 2e-5}  # 2.3e-7, 4.4e-6
    if kind == "tgv" and not case["train"]:
        return {"rel": 1.7e-6, "max": 1e-5}  # 4.2e-7, 2.6e-6
    if kind in ("tv", "stack"):
        return {"rel": 4e-3, "max": 0.99}  # 9.4e-4, 0.29: a last-bit change of an iterate flips a few Huber / prox switches
    if kind == "tgv":
        return {"rel": 9e-5, "max": 0.13}  # 2.2e-5, 3.3e-2
    if kind == "quadfit":
        # every sum that decides whether an axis is fitted runs over the channels in order; the gradient wrt the second
        # map sums over the pixels that land on one: 32-bit sums in another order
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 2.5e-7, "max": 8e-5}  # 5.3e-8, 2e-5
