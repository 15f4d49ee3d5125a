"""Autograd surface of the median layer: the names, arguments and tensor layouts of the reference's
cudaMedian/median.py (MedianFunction, Median)."""
import torch
from torch import nn
from torch.autograd import Function

from . import median_cuda_ext


class MedianFunction(Function):
    @staticmethod
    def forward(ctx, in_vol):  # median.py:18-44
        vol = in_vol.contiguous()
        if ctx.needs_input_grad[0] and vol.dim() == 4 and vol.shape[3] <= median_cuda_ext.MAX_SAVED_BINS:
            solution, saved = median_cuda_ext.forward_saving(vol)
            ctx.save_for_backward(in_vol, saved)
            return solution
        outputs = median_cuda_ext.forward(vol)
        ctx.save_for_backward(in_vol)
        return outputs[0]

    @staticmethod
    def backward(ctx, grad_sol):  # median.py:47-56
        in_vol, *saved = ctx.saved_tensors
        outputs = median_cuda_ext.backward(grad_sol.contiguous(), in_vol.contiguous(), *saved)
        return outputs[0]


class _MedianImage(Function):
    """The position plane of MedianFunction for one H x W x D volume, as a node of its own: the mass plane, which the module drops,
    gets no gradient of zeros."""

    @staticmethod
    def forward(ctx, in_vol):
        h, w, _ = in_vol.shape
        if ctx.needs_input_grad[0] and in_vol.shape[2] <= median_cuda_ext.MAX_SAVED_BINS:
            solution, saved = median_cuda_ext.forward_saving(in_vol.unsqueeze(0).contiguous())
            ctx.save_for_backward(in_vol, saved)
        else:
            (solution,) = median_cuda_ext.forward(in_vol.unsqueeze(0).contiguous())
            ctx.save_for_backward(in_vol)
        # (the first plane, not as a view so that it may be changed in place; the second stays behind it in the storage, as it did behind
        # the view of both planes that the permutations gave)
        return solution.as_strided_((h, w), (w, 1))

    @staticmethod
    def backward(ctx, grad_sol):
        in_vol, *saved = ctx.saved_tensors
        grad_sol = grad_sol[None, None].contiguous().resolve_neg()
        if not saved:  # (more bins than a crossing is saved for)
            grad_sol = torch.cat([grad_sol, torch.zeros_like(grad_sol)], 1)
        (gradient,) = median_cuda_ext.backward(grad_sol, in_vol.unsqueeze(0).contiguous(), *saved)
        return gradient[0]


class Median(nn.Module):
    def __init__(self, device):
        super(Median, self).__init__()
        self.device = device

    def forward(self, t_vol):
        """t_vol: H x W x D histogram per pixel.  Returns the H x W map of median positions (median.py:69-80
        drops the second output channel, the mass of the median's bin)."""
        return _MedianImage.apply(t_vol)

    def init(self):
        pass
