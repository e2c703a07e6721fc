"""L1 forward and input gradient on the lane tiles whose four waves split the contraction (csrc/similarity_direct.hip,
csrc/similarity_grad.hip): channels and templates that do not divide among the waves, chunks with idle waves, ragged rows,
strides.  Reference: torch in 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

GEOMS = [
    dict(shape=(20, 13, 28, 28), O=60, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),    # 13 channels among four waves
    dict(shape=(33, 8, 31, 30), O=64, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),     # two channels each
    dict(shape=(16, 37, 45, 47), O=67, blocks=[3, 3], strides=[1, 1], padding=[1, 0]),    # odd chunks, ragged rows
    dict(shape=(20, 21, 33, 29), O=57, blocks=[5, 5], strides=[1, 1], padding=[2, 2]),    # the table-driven loop
    dict(shape=(30, 17, 57, 61), O=43, blocks=[3, 4], strides=[2, 2], padding=[1, 1]),    # stride 2
]


@pytest.mark.parametrize("geom", GEOMS)
def test_l1_with_the_contraction_split_over_waves(pkg, geom):
    g = torch.Generator(device="cuda").manual_seed(37)
    shape, O, blocks = geom["shape"], geom["O"], geom["blocks"]
    kw = dict(similarity_function="L1", blocks=blocks, strides=geom["strides"], padding=geom["padding"],
              out_of_bounds_value=0.25)
    x = torch.randn(shape, generator=g, device="cuda")
    t = torch.randn((O, shape[1], *blocks), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    t[4] = x[1, :, 2:2 + blocks[0], 3:3 + blocks[1]]   # ties
    got = pkg.similarity(x, t, w, **kw)
    go = torch.randn(got.shape, generator=g, device="cuda")
    dx = pkg.similarity_input_grad(x, t, w, go, **kw)
    (ph, pw), (sh, sw) = geom["padding"], geom["strides"]
    K = shape[1] * blocks[0] * blocks[1]
    for b in (0, 1, shape[0] - 1):                  # images in 64 bits, one at a time
        xb = x[b:b + 1].double().requires_grad_()
        xp = torch.nn.functional.pad(xb, (pw, pw, ph, ph), value=0.25)
        cols = xp.unfold(2, blocks[0], sh).unfold(3, blocks[1], sw).permute(0, 1, 4, 5, 2, 3)
        cols = cols.reshape(1, K, -1)
        want = torch.cat([-(w[m].reshape(1, K, 1) * (t[m].reshape(1, K, 1).double() - cols).abs()).sum(1, keepdim=True)
                          for m in range(O)], 1).reshape(1, *got.shape[1:])
        # terms of one sign, each rounded twice and their sum K times at most
        err = float(((got[b:b + 1].double() - want.detach()).abs() / want.detach().abs().clamp_min(1e-3)).max())
        assert err <= (K + 2) * 2.0 ** -24, err
        ref = torch.autograd.grad(want, xb, go[b:b + 1].double())[0]
        n = O * blocks[0] * blocks[1]
        err = float((dx[b:b + 1].double() - ref).norm() / ref.norm())
        assert err <= 4 * math.sqrt(n) * 2.0 ** -24, err
    assert torch.equal(pkg.similarity_prepare(shape, t, w, **kw)(x), got)


@pytest.mark.parametrize("geom", [
    dict(shape=(33, 13, 28, 28), O=60, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),     # 2 x 14 columns, split channels
    dict(shape=(40, 9, 24, 23), O=64, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),      # 2 x 12, the last column empty
    dict(shape=(64, 17, 36, 36), O=40, blocks=[5, 5], strides=[1, 1], padding=[2, 2]),     # 3 x 12, the table-driven loop
    dict(shape=(200, 5, 53, 55), O=33, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),     # 4 x 14, whole channels
    dict(shape=(150, 9, 83, 84), O=40, blocks=[3, 3], strides=[2, 2], padding=[1, 1]),     # 3 x 14 at stride 2
    dict(shape=(220, 4, 38, 36), O=70, blocks=[3, 4], strides=[1, 1], padding=[1, 2]),     # 37 columns, the table-driven loop
])
def test_l1_on_lane_tiles_of_14_and_12_columns(pkg, geom):
    test_l1_with_the_contraction_split_over_waves(pkg, geom)
