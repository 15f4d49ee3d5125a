"""Python surface of the TV inpainting layer: the names, signatures and tensor conventions of the
reference's cudaTV/TVInpainting.py (TVInpaintingFunction at lines 11-29, TVInpaint at 32-55)."""
import numpy as np
import torch
from torch import nn
from torch.autograd import Function

from .._image import gradients, planes, result
from . import tvInpaint_cuda_ext


class TVInpaintingFunction(Function):

    @staticmethod
    def forward(ctx, dx, dy, dc, db, di, its, pid):
        # a forward nobody differentiates keeps no intermediate iterates
        outputs = tvInpaint_cuda_ext.forward(dx.contiguous(), dy.contiguous(), dc.contiguous(),
                                             db.contiguous(), di.contiguous(), its, pid,
                                             keep=None if any(ctx.needs_input_grad[:5]) else 0)
        sol = outputs[0]
        # di is not saved: backward takes the starting point from the id's first checkpoint
        variables = [dx, dy, dc, db, torch.from_numpy(np.array([its, pid]))]
        ctx.save_for_backward(*variables)
        return sol

    @staticmethod
    def backward(ctx, grad_sol):
        dx, dy, dc, db, ii = ctx.saved_tensors
        its, pid = (int(v) for v in ii.tolist())
        outputs = tvInpaint_cuda_ext.backward(grad_sol.contiguous(), dx.contiguous(), dy.contiguous(),
                                              dc.contiguous(), db.contiguous(), its, pid)
        d_oGx, d_oGy, d_oGc, d_oGb, d_oGi = outputs
        return d_oGx, d_oGy, d_oGc, d_oGb, d_oGi, None, None


class _TVInpaintImage(Function):
    """TVInpaintingFunction of one image with its channels innermost; the permutations are part of the node."""

    @staticmethod
    def forward(ctx, dx, dy, dc, db, di, its, pid):
        (sol,) = tvInpaint_cuda_ext.forward(*planes(dx, dy, dc, db, di), its, pid, keep=None if any(ctx.needs_input_grad[:5]) else 0)
        ctx.its, ctx.pid = int(its), int(pid)
        ctx.save_for_backward(dx, dy, dc, db)
        return result(sol)

    @staticmethod
    def backward(ctx, grad_sol):
        dx, dy, dc, db = ctx.saved_tensors
        outputs = tvInpaint_cuda_ext.backward(*planes(grad_sol, dx, dy, dc, db), ctx.its, ctx.pid)
        return gradients(outputs, ctx.needs_input_grad) + (None, None)


class TVInpaint(nn.Module):
    """Unbatched H x W x C interface of the reference module (cudaTV/TVInpainting.py:32-55)."""

    def __init__(self, device, its, pid=6, corrected_gradient=False):
        super(TVInpaint, self).__init__()
        self.its = its
        self.id = pid
        self.device = device
        # not in the reference: back-propagate the corrected gradient instead of the reference's (gradient_mode)
        self.corrected_gradient = bool(corrected_gradient)

    def forward(self, t_dx, t_dy, t_dc, t_db, t_di):
        tvInpaint_cuda_ext.gradient_mode(self.id, 1 if self.corrected_gradient else 0)
        Yx, Xx, Lx = t_dx.shape  # no batches here
        assert Lx == 1, "diffusion tensors should have 1 channel\n"

        return _TVInpaintImage.apply(t_dx, t_dy, t_dc, t_db, t_di, self.its, self.id)

    def init(self):
        pass
