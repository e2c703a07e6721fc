"""Input gradient of the plain L2 Similarity on its matrix kernel, workgroups of eight waves beside those of four
(csrc/similarity_split.hip): single, even and odd numbers of channel chunks, chunks of eight, remainders of pixels and of
channels, several images and more staged pixels than are requested ahead in a tile, rows in two groups.
Reference: torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# A factor in three pieces keeps 24 bits and a product loses what lies below 2^-24 of it; K products of either sign add up to
# sqrt(K) roundings of a sum whose terms add up to as much: 2 x 2^-24 each for the two sums and their difference, 4e-7, and
# twice that for x against t's centre.
TOL = 8e-7


@pytest.mark.parametrize("shape,templates,block", [
    ((32, 128, 28, 28), 128, 3),       # 196 workgroups of eight waves
    ((22, 128, 28, 28), 40, 3),        # three chunks, the last of eight channels
    ((33, 97, 27, 23), 24, 3),         # 97 rows: four tiles; two chunks, no multiples
    ((30, 256, 24, 24), 16, 3),        # one chunk, two groups of rows
    ((23, 128, 28, 28), 128, 1),       # a step a chunk
    ((4, 128, 20, 250), 33, 3),        # wide rows
    ((3, 128, 80, 100), 33, 5),        # chunks of eight
    ((400, 112, 7, 7), 64, 3),         # three images to a tile
    ((32, 64, 28, 28), 40, 3),         # two tiles of rows to a workgroup
    ((12, 100, 28, 28), 33, 3),        # ... two groups of them
    ((32, 50, 28, 28), 33, 5),         # chunks of eight: four waves
    ((25, 48, 32, 32), 64, 1),         # ... a step a chunk
    ((44, 128, 28, 28), 30, 3),        # 270 tiles: four waves
    ((32, 96, 28, 28), 30, 3),         # three tiles of rows: four waves
    ((32, 32, 28, 28), 7, 1),          # eight templates or fewer, in a chunk of sixteen: four waves
    ((32, 64, 28, 28), 8, 1),          # ... eight
    ((32, 64, 28, 28), 9, 1),
])
def test_input_gradient(pkg, shape, templates, block):
    gen = torch.Generator(device="cuda").manual_seed(43)
    kw = dict(blocks=[block] * 2, strides=[1, 1], padding=[block // 2] * 2)
    x = torch.randn(shape, generator=gen, device="cuda")
    t = torch.randn(templates, shape[1], block, block, generator=gen, device="cuda")
    w = torch.rand(t.shape, generator=gen, device="cuda") * 1.9 + 0.1
    go = torch.randn((shape[0], templates) + shape[2:], generator=gen, device="cuda")
    got = pkg.similarity_input_grad(x, t, w, go, **kw)
    a, b = (torch.nn.functional.conv_transpose2d(go.cpu().double(), 2 * v.cpu().double(), padding=block // 2)
            for v in (w * t.double(), w))
    want = a - x.cpu().double() * b
    error = float((got.cpu().double() - want).norm() / want.norm())
    print("%.2g" % error)
    assert error <= TOL
