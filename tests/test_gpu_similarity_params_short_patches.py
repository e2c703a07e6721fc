"""Parameter gradients of Similarity layers with few templates over short patches (sim_grad_params_small_kernel,
csrc/similarity_grad.hip): sums over the lanes of 32 and fewer values, templates behind the last of a wave.
Reference: torch in 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# Sums of some thousand terms of either sign, in lanes of a dozen each: sqrt(12) roundings of 2^-24 of a lane's share and eleven of
# the sums over lanes and splits; moments about the templates' mean, whose difference costs as much again: 1e-6.
TOL = 1e-6


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("channels, block, templates", [
    (1, (1, 1), 128), (2, (1, 1), 61), (3, (1, 1), 40), (1, (2, 2), 32), (4, (1, 1), 29), (5, (1, 1), 24), (1, (2, 3), 17),
    (7, (1, 1), 16), (2, (2, 2), 13), (1, (3, 3), 12),
])
def test_parameter_gradients(pkg, channels, block, templates, mode):
    gen = torch.Generator(device="cuda").manual_seed(53)
    x = torch.rand(9, channels, 17, 15, generator=gen, device="cuda") - 0.5
    t = torch.randn(templates, channels, *block, generator=gen, device="cuda") * 0.1
    w = torch.rand(t.shape, generator=gen, device="cuda") + 0.5
    kw = dict(blocks=list(block), strides=[1, 1], padding=[0, 0])
    if mode != "l2":
        kw["normalization_term"] = True
    if mode == "missing":
        x[torch.rand(x.shape, generator=gen, device="cuda") < 0.25] = math.nan
        kw["ignore_nan_input"] = True
    out = pkg.similarity(x, t, w, **kw)
    go = torch.randn(out.shape, generator=gen, device="cuda")
    got = pkg.similarity_parameters_grad(x, t, w, go, **kw)
    cols = x.cpu().double().unfold(2, block[0], 1).unfold(3, block[1], 1).permute(0, 2, 3, 1, 4, 5)
    cols = cols.reshape(-1, t[0].numel())
    keep = (cols == cols).double()
    cols = torch.nan_to_num(cols)
    g = go.cpu().double().permute(0, 2, 3, 1).reshape(-1, templates)
    t64, w64 = t.cpu().double().reshape(templates, -1), w.cpu().double().reshape(templates, -1)
    s0, s1, s2 = g.T @ keep, g.T @ cols, g.T @ (cols * cols)
    half = 1.0 if mode == "l2" else 0.5
    want_t = half * 2 * w64 * (s1 - t64 * s0)
    want_w = -half * (s2 - 2 * t64 * s1 + t64 * t64 * s0)
    if mode != "l2":
        want_w += half * s0 / (w64 + 0.001)
    for name, a, b in (("templates", got[0], want_t), ("weights", got[1], want_w)):
        error = float((a.cpu().double().reshape(b.shape) - b).norm() / b.norm())
        print("%s %.2g" % (name, error))
        assert error <= TOL
