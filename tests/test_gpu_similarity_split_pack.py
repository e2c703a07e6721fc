"""Packing of the L2 Similarity modes' parameters into 16-bit pieces (csrc/sim_split.h): channels up to and beyond what a
packing workgroup samples at a time, rows up to and beyond what it requests ahead and keeps in LDS, fewer template elements in a
channel than are sampled, templates of one channel chunk and of eight-channel ones.  Reference: torch in 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [   # shape, templates, block
    ((32, 64, 12, 12), 40, 1),      # the shortest rows, channels sampled at once
    ((32, 65, 12, 12), 33, 1),      # one channel more
    ((32, 128, 12, 12), 19, 1),     # twice as many, a channel of 19 elements
    ((32, 193, 12, 12), 32, 1),     # four times, the last one alone
    ((40, 30, 11, 13), 64, 3),      # 270 elements: a second one for some threads
    ((24, 114, 12, 12), 64, 3),     # 1026: just more than are requested ahead
    ((24, 62, 12, 12), 64, 5),      # 1550: just more than LDS keeps
    ((24, 200, 9, 9), 70, 3),       # 1800
    ((6, 8, 30, 30), 96, 3),        # chunks of eight channels
]


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("shape,templates,block", CASES)
def test_packed_parameters(pkg, shape, templates, block, mode):
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(shape, generator=gen, device="cuda")
    # channels on scales of their own, which the packing evens out, and templates
    scale = 2.0 ** torch.randint(-3, 4, (shape[1],), generator=gen, device="cuda").float()
    x = x * scale[:, None, None] + scale[:, None, None]
    t = torch.randn(templates, shape[1], block, block, generator=gen, device="cuda") * scale[:, None, None] + scale[:, None, None]
    w = (torch.rand(t.shape, generator=gen, device="cuda") * 1.9 + 0.1) / (scale * scale)[:, None, None]
    kw = dict(blocks=[block] * 2, strides=[1, 1], padding=[block // 2] * 2)
    if mode != "l2":
        kw["normalization_term"] = True
    if mode == "missing":
        x[torch.rand(shape, generator=gen, device="cuda") < 0.25] = float("nan")
        kw.update(ignore_nan_input=True, out_of_bounds_value=float("nan"))
    got = pkg.similarity(x, t, w, **kw)
    pad = float("nan") if mode == "missing" else 0.0
    cols = torch.nn.functional.pad(x.double(), (block // 2,) * 4, value=pad).unfold(2, block, 1).unfold(3, block, 1)
    cols = cols.permute(0, 1, 4, 5, 2, 3).reshape(shape[0], -1, got.shape[2] * got.shape[3])
    keep = (cols == cols).double() if mode == "missing" else torch.ones_like(cols)
    cols = torch.where(cols == cols, cols, torch.zeros_like(cols))
    t64, w64 = t.double().flatten(1), w.double().flatten(1)
    want = -(w64 @ (cols * cols) - 2 * (w64 * t64) @ cols + (w64 * t64 * t64) @ keep)
    if mode != "l2":
        want = 0.5 * (want + (torch.log(w64 + 0.001) - math.log(2 * math.pi)) @ keep)
    error = float((got.double().flatten(2) - want).norm() / want.norm())
    print("%.2g" % error)
    # products of 22 bits and one rounding of fp32 in every 144 terms, of sums of one sign: half of what term by term sums of
    # that length show (sqrt(K) / 2 roundings of 2^-24), and 2e-7 at least
    K = shape[1] * block * block
    assert error <= max(2e-7, math.sqrt(K) / 4 * 2.0 ** -24)
