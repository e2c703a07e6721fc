"""Plain and normalized L2 Similarity forward in workgroups of eight waves (csrc/similarity_split.hip): numbers of chunks, chunks of
eight channels, remainders of templates and pixels, two groups of templates; inputs that leave the first scale, at once and
chunk by chunk; outputs that are recomputed, few, many and too many of a tile; values that are not finite.
Reference: torch in 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# An output above the guard's line has an error of 2.4e-7 of itself at the line, one below it, summed term by term, of 3.6e-7 (root mean
# square); the largest of 10^6 is five times that, and half as much again for K up to 600.
TOL = 3e-6

GEOMS = [
    ((32, 40, 28, 28), 100, 3),    # three chunks, the last of eight channels; four tiles of templates
    ((30, 45, 29, 35), 75, 3),     # three tiles: two waves idle
    ((33, 16, 25, 25), 128, 3),    # one chunk
    ((40, 70, 24, 24), 128, 1),    # a step a chunk
    ((22, 24, 28, 28), 128, 5),    # chunks of eight channels
    ((18, 32, 28, 28), 256, 3),    # two groups of templates
    ((32, 40, 28, 28), 50, 3),     # two tiles to a workgroup
    ((12, 24, 28, 28), 100, 3),    # ... and two groups of them
    ((22, 24, 28, 28), 64, 5),     # ... chunks of eight channels
]


def check(pkg, x, t, w, block, norm=False, tol=TOL):
    pad = block // 2
    out = pkg.similarity(x, t, w, blocks=[block] * 2, strides=[1, 1], padding=[pad] * 2, normalization_term=norm).cpu().double()
    x, t, w = (v.cpu().double() for v in (x, t, w))
    finite = torch.where(x.isfinite(), x, torch.zeros_like(x))

    def conv(a, b):
        return torch.nn.functional.conv2d(a, b, padding=pad)
    sums = conv(finite * finite, w) - 2 * conv(finite, w * t) + (w * t * t).sum((1, 2, 3))[:, None, None]
    touched = conv((~x.isfinite()).double(), torch.ones_like(w[:1]))[:, 0] > 0
    holds_nan = conv(x.isnan().double(), torch.ones_like(w[:1]))[:, 0] > 0
    touched, holds_nan = (v[:, None].expand_as(out) for v in (touched, holds_nan))
    want = -sums
    if norm:
        want = 0.5 * (want + (torch.log(w + 0.001) - math.log(2 * math.pi)).sum((1, 2, 3))[:, None, None])
    assert bool(out[holds_nan].isnan().all()) and bool((out[touched & ~holds_nan] == -math.inf).all())
    error = (out - want).abs()[~touched]
    # (a sum that is 0 term by term, and in 64 bits not quite)
    bound = tol * (sums.abs() if not norm else sums.abs() + (want * 2).abs())[~touched] + 1e-9 * float(sums[~touched].abs().max())
    print("%.2g" % float((error / bound).max()))
    assert bool((error <= bound).all())


def tensors(geom, seed=47):
    shape, templates, block = geom
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(shape, generator=gen, device="cuda")
    t = torch.randn(templates, shape[1], block, block, generator=gen, device="cuda")
    w = torch.rand(t.shape, generator=gen, device="cuda") * 1.9 + 0.1
    return x, t, w


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("geom", GEOMS)
def test_geometries(pkg, geom, norm):
    check(pkg, *tensors(geom), geom[2], norm)


@pytest.mark.parametrize("kind", ["all", "rising", "falling", "pixels"])
@pytest.mark.parametrize("geom", GEOMS)
def test_inputs_on_another_scale(pkg, geom, kind):
    x, t, w = tensors(geom)
    t *= 0.05
    channel = torch.arange(x.shape[1], device="cuda")[:, None, None]
    if kind == "all":
        x *= 1e3
    elif kind == "pixels":
        x[::3, :, 5, 7::11] *= 3e3
    else:
        x *= 3.0 ** (channel // 4 if kind == "rising" else (x.shape[1] - 1 - channel) // 4).float()
    # the sums hold what the scale leaves of the pieces: the line of the guard rises with the staged values
    check(pkg, x, t, w, geom[2], tol=2 * TOL)


@pytest.mark.parametrize("templates", [128, 64])
@pytest.mark.parametrize("pixels, copies", [(3, 1), (50, 1), (100, 1), (64, 2), (100, 4)])
def test_outputs_near_a_template(pkg, pixels, copies, templates):
    x, t, w = tensors((GEOMS[3][0], templates, 1))
    t[:copies] = t[40]
    t[40:40 + copies] = t[40].clone()
    flat = x.view(x.shape[0], x.shape[1], -1)
    for image in (0, 17, 39):
        flat[image, :, 30:30 + pixels] = t[40].flatten()[:, None]
    check(pkg, x, t, w, 1)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("geom", GEOMS[:4])
def test_values_that_are_not_finite(pkg, geom, value):
    x, t, w = tensors(geom)
    x[3, 1, 4, 5] = value
    x[-1, -1, -1, -1] = value
    check(pkg, x, t, w, geom[2])
