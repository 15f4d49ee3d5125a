"""The copies between an image with its channels innermost and channel planes, several images per launch: torch's permutations, bit
for bit, at the edges of the launch (one pixel, a block of 256, one more), for every layout of the image, and repeatedly.  planes()
and images() launch only for views that are not contiguous, which an image of one pixel or one channel never is; launched() hands any
image to the kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def every_size(monkeypatch):
    from customnetworklayers_amd import _image

    monkeypatch.setattr(_image, "_LAUNCH_PIXELS", 1)
    monkeypatch.setattr(_image, "_LAUNCH_IMAGES", 1)


LAYOUTS = ("contiguous", "planes", "wide", "deep", "transposed", "negative")


def image(h, w, c, layout, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.randn((h, w, c), generator=g, device="cuda", dtype=torch.float32)
    if layout == "planes":
        return t.permute(2, 0, 1).contiguous().permute(1, 2, 0)
    if layout == "wide":
        return torch.cat([t, t], 1)[:, :w]
    if layout == "deep":
        return torch.cat([t, t], 2)[..., :c]
    if layout == "negative":  # a view whose sign is still to be applied
        return torch.complex(torch.zeros_like(t), -t).conj().imag
    if layout == "transposed":
        return t.transpose(0, 1).contiguous().transpose(0, 1)
    return t


@pytest.mark.parametrize("h,w", [(1, 1), (1, 2), (2, 1), (1, 255), (16, 16), (1, 257), (33, 70), (375, 1241)])
@pytest.mark.parametrize("channels", [(1,), (2,), (3, 2), (2, 2, 1, 2, 6), (16, 17, 4)])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_images_to_planes_and_back(h, w, channels, layout):
    from customnetworklayers_amd import _image

    given = [image(h, w, c, layout, seed=i) for i, c in enumerate(channels)]
    there = _image.planes(*given)
    for t, g in zip(there, given):
        assert t.is_contiguous() and torch.equal(t, g.permute(2, 0, 1).unsqueeze(0))
    back = _image.images(there)
    for t, g in zip(back, given):
        assert t.is_contiguous() and torch.equal(t, g)


def launched(given):
    """The images through both kernels, whatever their layout: (planes, images)."""
    from customnetworklayers_amd import _image
    from customnetworklayers_amd._lib import lib

    there = [torch.full((1, t.shape[2]) + t.shape[:2], float("nan"), device="cuda", dtype=torch.float32) for t in given]
    _image._move(lib.layout_to_planes, given, there, given)
    back = [torch.full(t.shape, float("nan"), device="cuda", dtype=torch.float32) for t in given]
    _image._move(lib.layout_to_images, there, back, back)
    return there, back


@pytest.mark.parametrize("h,w", [(1, 1), (1, 2), (2, 1), (16, 16), (1, 257), (33, 70)])
@pytest.mark.parametrize("channels", [(1,), (2,), (1, 2, 1), (2, 2, 1, 2, 6), (1, 16, 17)])
@pytest.mark.parametrize("layout", LAYOUTS[:-1])  # (a negative view is not handed to the kernels)
def test_kernels_on_every_image(h, w, channels, layout):
    given = [image(h, w, c, layout, seed=i) for i, c in enumerate(channels)]
    there, back = launched(given)
    for t, b, g in zip(there, back, given):
        assert torch.equal(t, g.permute(2, 0, 1).unsqueeze(0)) and torch.equal(b, g)


def test_images_of_two_values_many_times():
    for k in range(300):
        a, b = torch.randn(1, 1, 2, device="cuda", dtype=torch.float32), torch.randn(1, 2, 1, device="cuda", dtype=torch.float32)
        c = torch.randn(1, 2, 2, device="cuda", dtype=torch.float32)
        for given in ([a], [b], [c], [b, c[..., :1]]):
            there, back = launched(given)
            assert all(torch.equal(t, g.permute(2, 0, 1).unsqueeze(0)) for t, g in zip(there, given))
            assert all(torch.equal(t, g) for t, g in zip(back, given))


def test_result_is_no_view():
    from customnetworklayers_amd import _image

    for c in (1, 3):
        t = torch.randn(1, c, 5, 7, device="cuda", dtype=torch.float32)
        want = t.clone().squeeze(0).permute(1, 2, 0)
        got = _image.result(t)
        assert got._base is None and got.is_contiguous() and torch.equal(got, want)


def test_large_images_as_the_modules_pass_them(monkeypatch):
    from customnetworklayers_amd import _image

    monkeypatch.undo()  # the sizes and numbers of images that the modules send this way
    calls = []
    move = _image._move
    monkeypatch.setattr(_image, "_move", lambda *a: (calls.append(len(a[3])), move(*a)))
    three, four = (2, 2, 1, 1, 3), (2, 2, 1, 2, 6)  # the layer's images at one and at two channels; those of one channel are no copy
    for h, w, channels, sent in ((1023, 896, three, []), (1024, 896, three, [3, 3]), (511, 896, four, []), (512, 896, four, [4, 4])):
        calls.clear()
        given = [image(h, w, c, "contiguous", seed=c) for c in channels]
        there = _image.planes(*given)
        back = _image.images(there)
        assert calls == sent
        assert all(torch.equal(t, g.permute(2, 0, 1).unsqueeze(0)) for t, g in zip(there, given))
        assert all(torch.equal(t, g) for t, g in zip(back, given))


def test_layout_errors():
    from customnetworklayers_amd._lib import lib

    assert lib.layout_to_planes(None, None, None, None, 1, 4, 4, None) != 0
    assert b"null" in lib.layout_last_error()
