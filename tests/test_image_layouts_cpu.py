"""What the single-image modules hand to the kernels of a tensor they do not copy: where its elements lie."""
import pytest
import torch

from customnetworklayers_amd.cudaQuadFit import QuadFit_cuda_ext


def flows(h, w):
    t = torch.arange(h * w * 3, dtype=torch.float32).view(h, w, 3)
    yield "contiguous", t
    yield "planes", t.permute(2, 0, 1).contiguous().permute(1, 2, 0)
    yield "columns of a wider image", torch.cat([t, t], 1)[:, :w]
    yield "rows of a taller image", torch.cat([t, t], 0)[:h]
    yield "channels of a deeper image", torch.cat([t, t], 2)[..., :3]
    yield "transposed", t.transpose(0, 1).contiguous().transpose(0, 1)
    yield "the only column of a batch of rows", t.reshape(1, h * w, 3).transpose(0, 1)
    yield "the only row of a batch of columns", t.reshape(h * w, 1, 3).transpose(0, 1)
    yield "every other pixel", t.reshape(1, h * w, 3).repeat_interleave(2, 1)[:, ::2]
    yield "one row for all", t[:1].expand(h, w, 3)
    yield "one pixel for all", t[:1, :1].expand(h, w, 3)


@pytest.mark.parametrize("h,w", [(1, 1), (1, 5), (5, 1), (2, 1), (4, 7)])
def test_flow_is_read_where_it_lies(h, w):
    for name, flow in flows(h, w):
        given, pixel, channel = QuadFit_cuda_ext._flow_strides(flow)
        assert pixel >= 1 and channel >= 1, name
        pixels = flow.shape[0] * flow.shape[1]
        last = given.storage_offset() + (pixels - 1) * pixel + 2 * channel
        assert last < given.untyped_storage().nbytes() // 4, name
        read = given.as_strided((pixels, 3), (pixel, channel))
        assert torch.equal(read, flow.reshape(pixels, 3)), name
