"""One H x W x C image as the layers' kernels take it: planes (1,C,H,W).  Used inside the modules' autograd nodes, so that a module
is one node and not a dozen: around a layer on a small image the nodes of the permutations took as long as the layer's own
launches (1 x 2 x 64 x 128, 20 iterations, forward + backward: 299 us with them, 243 without)."""
import ctypes

import torch

from ._lib import device_of, lib

# Three or more images change their layout in one launch if they are large: four or more of _LAUNCH_PIXELS, three of twice that.
# Setting a launch up takes 6 to 13 us of host time more than torch's copies, a launch each, and saves GPU time; it loses where the
# host is what a pass waits for, which fewer iterations make more likely.  TGV, us, torch's copies / one launch:
#   channels, pixels   inference 10   training 10   training 16   inference 100   training 100 iterations
#   1 (three images)
#     320 x 960            66 / 72     291 / 329                     285 / 280      1160 / 1144
#     375 x 1241           72 / 69     292 / 328     334 / 371       347 / 340      1484 / 1463
#     540 x 1280           84 / 77     327 / 339                     405 / 398      1851 / 1834
#     700 x 1280           99 / 91     408 / 391     543 / 528
#     768 x 1536          114 / 110    486 / 474                     634 / 628      2871 / 2856
#   2 (five images, backward four)
#     320 x 960            78 / 73     310 / 346                     390 / 384      1783 / 1760
#     384 x 1024           82 / 76     347 / 371     473 / 449
#     375 x 1241          106 / 93     406 / 376     545 / 511       549 / 534      2396 / 2362
#     768 x 1536          201 / 187    783 / 754                    1157 / 1143     4876 / 4843
#   3                      375 x 1241 inference 10 139 / 116, training 10 607 / 557;  384 x 1024 106 / 101, 511 / 494
# (The TV layer has two such images at most.)
_LAUNCH_PIXELS, _LAUNCH_IMAGES = 7 << 16, 3
_MAX_IMAGES, _MAX_CHANNELS = 8, 16  # images per launch; more channels than that are left to torch's copies


def _move(fn, sources, targets, images):
    """One launch: sources[i] -> targets[i]; images: the sides of the pairs that are H x W x C."""
    n, (h, w, _) = len(images), images[0].shape
    pointers = ctypes.c_void_p * n
    strides = (ctypes.c_longlong * (3 * n))(*[s for t in images for s in t.stride()])
    device = images[0].device
    with device_of(images[0]):
        rc = fn(pointers(*[t.data_ptr() for t in sources]), pointers(*[t.data_ptr() for t in targets]),
                (ctypes.c_int * n)(*[t.shape[2] for t in images]), strides, n, h, w,
                ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream))
    if rc:
        raise RuntimeError("layout copy failed: %s" % lib.layout_last_error().decode("utf-8", "replace"))


def _movable(images):
    first = images[0]
    if not _LAUNCH_IMAGES <= len(images) <= _MAX_IMAGES:
        return False
    return (first.is_cuda and first.shape[0] * first.shape[1] >= _LAUNCH_PIXELS * (2 if len(images) == 3 else 1)
            and all(t.dtype == torch.float32 and not t.is_neg() and t.device == first.device and t.shape[:2] == first.shape[:2]
                    and 1 <= t.shape[2] <= _MAX_CHANNELS for t in images))


def planes(*images):
    """(H,W,C) images -> contiguous (1,C,H,W) tensors; no copy of a single channel or a view of planes."""
    views = [t.permute(2, 0, 1).unsqueeze(0) for t in images]
    if images[0].numel() >= _LAUNCH_PIXELS:
        todo = [i for i, v in enumerate(views) if not v.is_contiguous()]
        if todo and _movable([images[i] for i in todo]):
            for i in todo:
                views[i] = torch.empty(views[i].shape, dtype=torch.float32, device=images[i].device)
            _move(lib.layout_to_planes, [images[i] for i in todo], [views[i] for i in todo], [images[i] for i in todo])
    return [v.contiguous() for v in views]


def images(tensors):
    """(1,C,H,W) planes -> contiguous (H,W,C) images; no copy of a single channel."""
    views = [t.squeeze(0).permute(1, 2, 0) for t in tensors]
    if views and views[0].numel() >= _LAUNCH_PIXELS:
        todo = [i for i, v in enumerate(views) if not v.is_contiguous()]
        if todo and _movable([views[i] for i in todo]) and all(tensors[i].is_contiguous() for i in todo):
            for i in todo:
                views[i] = torch.empty(views[i].shape, dtype=torch.float32, device=views[i].device)
            _move(lib.layout_to_images, [tensors[i] for i in todo], [views[i] for i in todo], [views[i] for i in todo])
    return [v.contiguous() for v in views]


def result(planes):
    """The image of planes that the caller has just made and gives up: never a view, which autograd would not let a program change
    in place as the output of a node (and not by resize_, after which a trace has lost the value)."""
    _, c, h, w = planes.shape
    return planes.as_strided_((h, w, 1), (w, 1, 1)) if c == 1 else planes.squeeze(0).permute(1, 2, 0).contiguous()


def gradients(tensors, wanted):
    """The gradients of a node's inputs as images, None for inputs nobody asked one for."""
    done = iter(images([t for t, want in zip(tensors, wanted) if want]))
    return tuple(next(done) if want else None for _, want in zip(tensors, wanted))
