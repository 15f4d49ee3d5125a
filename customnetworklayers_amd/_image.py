"""One H x W x C image as the layers' kernels take it: planes (1,C,H,W).  Used inside the modules' autograd nodes, so that a module
is one node and not a dozen: around a layer on a small image the nodes of the permutations took as long as the layer's own
launches (1 x 2 x 64 x 128, 20 iterations, forward + backward: 299 us with them, 243 without)."""


def planes(image):
    """(H,W,C) -> contiguous (1,C,H,W); no copy for a single channel or a view of planes."""
    return image.permute(2, 0, 1).unsqueeze(0).contiguous()


def image(planes):
    """(1,C,H,W) -> contiguous (H,W,C); no copy for a single channel."""
    return planes.squeeze(0).permute(1, 2, 0).contiguous()


def result(planes):
    """image() of a tensor the caller has just made and gives up: never a view, which autograd would not let a program change in
    place as the output of a node."""
    _, c, h, w = planes.shape
    return planes.resize_(h, w, 1) if c == 1 else image(planes)


def images(gradients, wanted):
    """The gradients of a node's inputs as images, None for inputs nobody asked one for."""
    return tuple(image(g) if want else None for g, want in zip(gradients, wanted))
