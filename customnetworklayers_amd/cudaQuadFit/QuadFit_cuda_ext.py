"""Binding module of the quadratic-fit layer: same name and functions as the reference's pybind
module (cudaQuadFit/QuadFit_cuda.cpp:117-122 of the reference), on top of the C ABI in
include/flowaux.h.

Differences from the reference binding: the result has 3 channels (offset x, offset y, score) as
the kernel writes them (cudaQuadFit/cudaCode/quadFit.cu:137,315; the reference binding allocates
2, QuadFit_cuda.cpp:60); the flow may have 2 or more channels, of which the first two are read;
failures raise instead of returning an empty list (QuadFit_cuda.cpp:68-74).
"""
import ctypes

import torch

from .._lib import device_of, lib

_ERRORS = {1: IndexError, 2: ValueError, 3: ValueError, 4: RuntimeError, 5: RuntimeError}


def _last_error():
    return lib.flowaux_last_error().decode("utf-8", "replace")


def _check_input(t, name):
    # CHECK_CUDA / CHECK_CONTIGUOUS, QuadFit_cuda.cpp:21-23
    if not isinstance(t, torch.Tensor):
        raise TypeError("%s must be a tensor" % name)
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)
    if not t.is_contiguous():
        raise RuntimeError("%s must be contiguous" % name)
    if t.dtype != torch.float32:  # QuadFit_cuda.cpp:57,73
        raise TypeError("Input/Output type to the operator must be single/float (%s is %s)" % (name, t.dtype))


def _check_shapes(featureImage0, featureImage1, flow):
    if featureImage0.dim() != 4:
        raise ValueError("featureImage0 must be (n, c, h, w)")
    n, _, h, w = featureImage0.shape
    if tuple(featureImage1.shape) != tuple(featureImage0.shape):
        raise ValueError("featureImage1 must have the shape of featureImage0 %s, got %s"
                         % (tuple(featureImage0.shape), tuple(featureImage1.shape)))
    if flow.dim() != 4 or flow.shape[0] != n or flow.shape[1] < 2 or tuple(flow.shape[2:]) != (h, w):
        raise ValueError("flow must have shape (%d, >=2, %d, %d), got %s" % (n, h, w, tuple(flow.shape)))
    if len({t.device for t in (featureImage0, featureImage1, flow)}) != 1:
        raise RuntimeError("all tensors must live on one device")


def _stream(t):
    return ctypes.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


def _check_maps(featureImage0, featureImage1, flow):
    for t, name in ((featureImage0, "featureImage0"), (featureImage1, "featureImage1"), (flow, "flow")):
        _check_input(t, name)
    _check_shapes(featureImage0, featureImage1, flow)
    return featureImage0.shape


def forward(featureImage0, featureImage1, flow):
    """featureImage0/1: (n,c,h,w) feature maps; flow: (n,>=2,h,w).  Returns [(n,3,h,w)]: the offsets of the
    fitted maximum in x and y (to be added to the rounded displaced position) and the fitted score."""
    n, c, h, w = _check_maps(featureImage0, featureImage1, flow)
    flowUpdate = torch.empty((n, 3, h, w), dtype=torch.float32, device=flow.device)
    with device_of(flow):
        rc = lib.quadfit_forward(featureImage0.data_ptr(), featureImage1.data_ptr(), flow.data_ptr(),
                                 flowUpdate.data_ptr(), n, c, h, w, flow.shape[1], _stream(flow))
    if rc:
        raise _ERRORS.get(rc, RuntimeError)("FlowQuadFitting::forward failed: %s" % _last_error())
    return [flowUpdate]


def saving_pays(featureImage0):
    """Whether forward_saving followed by backward(costs=...) is the faster pair at this shape (not at small ones)."""
    return featureImage0.dim() == 4 and bool(lib.quadfit_saving_pays(*featureImage0.shape))


def forward_saving(featureImage0, featureImage1, flow):
    """forward that also returns what backward takes as `costs`: [flowUpdate, costs (5,n,h,w)]."""
    n, c, h, w = _check_maps(featureImage0, featureImage1, flow)
    flowUpdate = torch.empty((n, 3, h, w), dtype=torch.float32, device=flow.device)
    costs = torch.empty((5, n, h, w), dtype=torch.float32, device=flow.device)
    with device_of(flow):
        rc = lib.quadfit_forward_saving(featureImage0.data_ptr(), featureImage1.data_ptr(), flow.data_ptr(), flowUpdate.data_ptr(),
                                        costs.data_ptr(), n, c, h, w, flow.shape[1], _stream(flow))
    if rc:
        raise _ERRORS.get(rc, RuntimeError)("FlowQuadFitting::forward failed: %s" % _last_error())
    return [flowUpdate, costs]


def backward(d_iGf, featureImage0, featureImage1, flow, use_atomics=False, costs=None):
    """d_iGf: (n,3,h,w) gradient wrt the result.  Returns [d_oFeat0, d_oFeat1].  `use_atomics` selects the
    reference's scatter with float atomics instead of the gather through a scratch buffer.  `costs`: the second result of
    forward_saving on the same inputs; without it they are formed again."""
    n, c, h, w = _check_maps(featureImage0, featureImage1, flow)
    _check_input(d_iGf, "d_iGf")
    if tuple(d_iGf.shape) != (n, 3, h, w):
        raise ValueError("d_iGf must have shape (%d, 3, %d, %d), got %s" % (n, h, w, tuple(d_iGf.shape)))
    if costs is not None:
        _check_input(costs, "costs")
        if tuple(costs.shape) != (5, n, h, w):
            raise ValueError("costs must have shape (5, %d, %d, %d), got %s" % (n, h, w, tuple(costs.shape)))
        if costs.device != flow.device:
            raise RuntimeError("all tensors must live on one device")
        if use_atomics:
            raise ValueError("the scatter with float atomics takes no costs")
    d_oFeat0, d_oFeat1 = torch.empty_like(featureImage0), torch.empty_like(featureImage1)
    ws_bytes = 0 if use_atomics else lib.quadfit_backward_workspace_bytes(n, h, w)
    workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=flow.device) if ws_bytes else None
    maps = (featureImage0.data_ptr(), featureImage1.data_ptr(), flow.data_ptr(), d_iGf.data_ptr())
    rest = (d_oFeat0.data_ptr(), d_oFeat1.data_ptr(), n, c, h, w, flow.shape[1], workspace.data_ptr() if ws_bytes else None, ws_bytes,
            _stream(flow))
    with device_of(flow):
        rc = lib.quadfit_backward(*maps, *rest) if costs is None else lib.quadfit_backward_saved(*maps, costs.data_ptr(), *rest)
    if rc:
        raise _ERRORS.get(rc, RuntimeError)("FlowQuadFitting::backward failed: %s" % _last_error())
    return [d_oFeat0, d_oFeat1]


def image_pays(channels, pixels, differentiated):
    """Whether the kernels on one image with its channels innermost are the faster ones.  With fewer than eight channels they are not on
    large images: a block's 256 lanes work through 32 channels of 64 pixels whatever the number that exists, the copies into planes and the
    kernels there move what exists.  Copies and kernels on planes / kernels on the image, us, one image at inference:
      channels   512 x 1024    600 x 1200    750 x 1300    900 x 1600    1600 x 2560
          2      45 / 43       44 / 58       44 / 84       56 / 128      129 / 355
          4      45 / 30       48 / 46       50 / 62       80 / 90       216 / 249
          5      44 / 47       57 / 70       56 / 93       98 / 135      274 / 379
          7      44 / 53       80 / 73       76 / 97       145 / 144     412 / 458
          8      49 / 33       94 / 45       90 / 59       172 / 87      489 / 300
    (below 2^19 pixels planes wait for the host, 44 us; 384 x 1248 with 2 channels 46 / 40).  Forward and backward 2 channels 241 / 223 at
    900 x 1600, 295 / 379 at 1200 x 2000; 3 348 / 421, 4 399 / 332, 5 482 / 492, 6 561 / 515 there."""
    if channels >= 8:
        return True
    if differentiated:
        return pixels < 1 << 21 or channels not in (2, 3, 5)
    return pixels < (7 << 17 if channels == 4 else 1 << 19)


def takes_image(feat0, feat1, flow):
    """Whether image_forward / image_backward are to take these H x W x C maps and H x W x 3 flow as they are: both maps contiguous with
    more than one channel innermost, at a size where that pays.  (Maps that are views of channel planes, views whose sign is still to be
    applied (is_neg), and everything that is to be refused, go through forward / backward.)"""
    if not (_readable(feat0, feat1, flow) and not (feat0.is_neg() or feat1.is_neg() or flow.is_neg())):
        return False
    h, w, c = feat0.shape
    return (c > 1 and h * w > 1 and h * w * c < 2 ** 31
            and image_pays(c, h * w, torch.is_grad_enabled() and (feat0.requires_grad or feat1.requires_grad)))


def _readable(feat0, feat1, flow):
    """Whether the kernels on one image can read these.  (One expression: a call at inference waits for the host.)"""
    shape, of_flow = feat0.shape, flow.shape
    return (len(shape) == 3 == len(of_flow) and feat1.shape == shape and of_flow[0] == shape[0] and of_flow[1] == shape[1] and of_flow[2] >= 2
            and flow.is_cuda and feat0.device == feat1.device == flow.device
            and feat0.dtype == feat1.dtype == flow.dtype == torch.float32 and feat0.is_contiguous() and feat1.is_contiguous())


def _flow_strides(flow):
    """flow with its pixels a fixed distance apart, that distance and the one between its channels.  (The stride of a dimension of
    one element says nothing: a single column's pixels lie a row apart, and a contiguous tensor may have any number there.)"""
    h, w, channels = flow.shape
    row, pixel, channel = flow.stride()
    if w == 1:
        pixel = row
    if pixel < 1 or channel < 1 or (h > 1 and row != w * pixel):
        return flow.contiguous(), channels, 1
    return flow, pixel, channel


def _check_image(feat0, feat1, flow):
    if _readable(feat0, feat1, flow):
        return feat0.shape
    for t, name in ((feat0, "featureImage0"), (feat1, "featureImage1"), (flow.contiguous(), "flow")):
        _check_input(t, name)
    if not feat0.device == feat1.device == flow.device:
        raise RuntimeError("all tensors must live on one device")
    raise ValueError("the maps must be H x W x C, the flow H x W x 2 or more, got %s, %s and %s"
                     % (tuple(feat0.shape), tuple(feat1.shape), tuple(flow.shape)))


def _check_beside(t, name, shape, flow):
    _check_input(t, name)
    if tuple(t.shape) != shape:
        raise ValueError("%s must have shape %s, got %s" % (name, shape, tuple(t.shape)))
    if t.device != flow.device:
        raise RuntimeError("all tensors must live on one device")


def image_forward(feat0, feat1, flow, want_costs, checked=False):
    """The fit of one image, feat0, feat1 H x W x C contiguous, flow H x W x 3 anyhow.  Returns [H x W x 3, costs (5,H,W) or None].
    checked: takes_image has just said yes to these."""
    h, w, c = feat0.shape if checked else _check_image(feat0, feat1, flow)
    flow, pixel, channel = _flow_strides(flow)
    out = torch.empty((h, w, 3), dtype=torch.float32, device=flow.device)
    costs = torch.empty((5, h, w), dtype=torch.float32, device=flow.device) if want_costs else None
    with device_of(flow):
        rc = lib.quadfit_image_forward(feat0.data_ptr(), feat1.data_ptr(), flow.data_ptr(), out.data_ptr(),
                                       costs.data_ptr() if want_costs else None, c, h, w, pixel, channel, _stream(flow))
    if rc:
        raise _ERRORS.get(rc, RuntimeError)("FlowQuadFitting::forward failed: %s" % _last_error())
    return [out, costs]


def image_backward(d_iGf, feat0, feat1, flow, costs):
    """d_iGf: H x W x 3 gradient wrt the result, costs: the second result of image_forward.  Returns the two maps' gradients."""
    h, w, c = _check_image(feat0, feat1, flow)
    if not (d_iGf.shape == (h, w, 3) and costs.shape == (5, h, w) and d_iGf.dtype == costs.dtype == torch.float32
            and d_iGf.device == costs.device == flow.device and d_iGf.is_contiguous() and costs.is_contiguous()):
        _check_beside(d_iGf, "d_iGf", (h, w, 3), flow)
        _check_beside(costs, "costs", (5, h, w), flow)
    flow, pixel, channel = _flow_strides(flow)
    g0, g1 = torch.empty_like(feat0), torch.empty_like(feat1)
    ws_bytes = lib.quadfit_backward_workspace_bytes(1, h, w)
    workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=flow.device)
    with device_of(flow):
        rc = lib.quadfit_image_backward(feat0.data_ptr(), feat1.data_ptr(), flow.data_ptr(), d_iGf.data_ptr(), costs.data_ptr(),
                                        g0.data_ptr(), g1.data_ptr(), c, h, w, pixel, channel, workspace.data_ptr(), ws_bytes,
                                        _stream(flow))
    if rc:
        raise _ERRORS.get(rc, RuntimeError)("FlowQuadFitting::backward failed: %s" % _last_error())
    return [g0, g1]


def dummy():
    print("Input: not present just dummy:")
    return []


def dummy_only():
    print("Dummy call:")
