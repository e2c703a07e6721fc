"""Parameter gradients of the Similarity layer where the pixels are split over workgroups (csrc/similarity_grad.hip,
csrc/similarity_split_params.hip): splits whose sums are stored segment by segment, one and several rounds of workgroups, elements
behind the last of a row and templates behind the last of a tile in the finishing and packing launches.
Reference: torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# Sums of at most 512 terms in a row, of either sign: sqrt(512) roundings of 2^-24 of a sum that the whole one exceeds by its
# other parts' share; 1.5e-6 of the gradient's 2-norm.
TOL = 1.5e-6


@pytest.mark.parametrize("function", ["L1", "L2"])
@pytest.mark.parametrize("shape,templates,block,stride", [
    ((50, 24, 9, 9), 48, 5, 1),        # three segments to a split
    ((64, 3, 40, 40), 33, 3, 1),       # rows of 27 elements, 33 templates
    ((13, 45, 29, 35), 75, 3, 1),      # no multiple of anything, thirteen images
    ((16, 64, 14, 14), 64, 3, 1),      # two chunks to a split
    ((24, 40, 33, 31), 200, 3, 2),
    ((7, 16, 20, 21), 130, 1, 1),
    ((9, 75, 15, 14), 59, 3, 1),       # 39825 elements, one to a thread of the finish (L2)
    ((9, 75, 15, 14), 60, 3, 1),       # 40500, four; rows of 675
    ((9, 75, 15, 14), 14, 3, 1),       # 9450, one (L1)
])
def test_parameter_gradients_of_split_pixels(pkg, shape, templates, block, stride, function):
    gen = torch.Generator(device="cuda").manual_seed(41)
    kw = dict(similarity_function=function, blocks=[block] * 2, strides=[stride] * 2, padding=[block // 2] * 2)
    x = torch.randn(shape, generator=gen, device="cuda")
    t = torch.randn(templates, shape[1], block, block, generator=gen, device="cuda")
    w = torch.rand(t.shape, generator=gen, device="cuda") * 1.9 + 0.1
    out = pkg.similarity(x, t, w, **kw)
    go = torch.randn(out.shape, generator=gen, device="cuda")
    got = pkg.similarity_parameters_grad(x, t, w, go, **kw)
    want_t, want_w = torch.zeros_like(t, dtype=torch.float64), torch.zeros_like(t, dtype=torch.float64)
    t64, w64 = t.double().flatten(1), w.double().flatten(1)
    for b in range(shape[0]):
        cols = torch.nn.functional.unfold(x[b:b + 1].double(), block, padding=block // 2, stride=stride)[0]
        for m in range(templates):
            d = cols - t64[m][:, None]
            g = go[b, m].double().flatten()
            if function == "L1":
                want_t[m] += ((torch.sign(d) @ g) * w64[m]).reshape(t[m].shape)
                want_w[m] -= (d.abs() @ g).reshape(t[m].shape)
            else:
                want_t[m] += (2 * (d @ g) * w64[m]).reshape(t[m].shape)
                want_w[m] -= ((d * d) @ g).reshape(t[m].shape)
    for name, a, b in (("templates", got[0], want_t), ("weights", got[1], want_w)):
        error = float((a.double() - b).norm() / b.norm())
        print("%s %.2g" % (name, error))
        assert error <= TOL


@pytest.mark.parametrize("missing", [0.0, 0.25])
@pytest.mark.parametrize("templates", [14, 61])   # one element to a thread of the finish, and four
def test_parameter_gradients_with_normalization(pkg, templates, missing):
    gen = torch.Generator(device="cuda").manual_seed(47)
    x = torch.randn(9, 75, 15, 14, generator=gen, device="cuda")
    t = torch.randn(templates, 75, 3, 3, generator=gen, device="cuda")
    w = torch.rand(t.shape, generator=gen, device="cuda") * 1.9 + 0.1
    kw = dict(blocks=[3, 3], strides=[1, 1], padding=[1, 1], normalization_term=True)
    if missing:
        x = x.masked_fill_(torch.rand(x.shape, generator=gen, device="cuda") < missing, float("nan"))
        kw.update(ignore_nan_input=True, out_of_bounds_value=float("nan"))
    out = pkg.similarity(x, t, w, **kw)
    go = torch.randn(out.shape, generator=gen, device="cuda")
    got = pkg.similarity_parameters_grad(x, t, w, go, **kw)
    pad = torch.nn.functional.pad(x.double(), (1, 1, 1, 1), value=float("nan") if missing else 0.0)
    there = (pad == pad).double()
    x0, keep = (torch.nn.functional.unfold(v, 3) for v in (torch.nan_to_num(pad), there))
    g = go.double().flatten(2)
    s0, s1, s2 = (torch.einsum("bmp,bkp->mk", g, v) for v in (keep, x0, x0 * x0))
    t64, w64 = t.double().flatten(1), w.double().flatten(1)
    want_t = w64 * (s1 - t64 * s0)
    want_w = 0.5 * (s0 / (w64 + 0.001) - (s2 - 2 * t64 * s1 + t64 * t64 * s0))
    for a, b in zip(got, (want_t, want_w)):
        assert float((a.double().flatten(1) - b).norm() / b.norm()) <= TOL
