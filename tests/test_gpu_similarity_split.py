"""The L2 Similarity modes on the matrix cores in 16-bit pieces (csrc/similarity_split.hip): edges of its tiles, its three
modes, both chunk sizes, and what its guard hands to the term-by-term kernel.  Reference: torch in 64 bits."""
import ctypes
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def exact(x, t, w, blocks, strides, padding, mode, oob=0.0, fudge=0.001):
    x, t, w = x.double(), t.double(), w.double()
    x = torch.nn.functional.pad(x, (padding[1],) * 2 + (padding[0],) * 2, value=oob)
    cols = x.unfold(2, blocks[0], strides[0]).unfold(3, blocks[1], strides[1]).permute(0, 1, 4, 5, 2, 3)
    B, _, _, _, oh, ow = cols.shape
    cols = cols.reshape(B, -1, oh * ow)
    t, w = t.reshape(t.shape[0], -1), w.reshape(w.shape[0], -1)
    out = torch.empty(B, t.shape[0], oh * ow, dtype=torch.float64, device=x.device)
    for m in range(t.shape[0]):
        term = -w[m, :, None] * (cols - t[m, :, None]) ** 2
        if mode != "l2":
            term = 0.5 * (term + torch.log(w[m] + fudge)[:, None] - math.log(2 * math.pi))
        if mode == "missing":
            term = torch.where(cols == cols, term, torch.zeros_like(term))
        out[:, m] = term.sum(1)
    return out.reshape(B, -1, oh, ow)


def options(mode, g):
    kw = dict(blocks=g["blocks"], strides=g["strides"], padding=g["padding"])
    if mode != "l2":
        kw["normalization_term"] = True
    if mode == "missing":
        kw.update(ignore_nan_input=True, out_of_bounds_value=float("nan"))
    return kw


def pieces_used(pkg, shape, O, mode="l2", **kw):
    """Which of the operator's calls take the form in 16-bit pieces on this geometry, from their workspaces: those of the
    forms that can be asked for by name are of another size."""
    def sizes(algo, **options):
        attrs, i4 = pkg.ops.similarity_attrs(algo=algo, **options), ctypes.c_int * 4
        x, t = i4(*shape), i4(O, shape[1], *options["blocks"])
        n = [ctypes.c_size_t() for _ in range(3)]
        assert lib.simnets_hip_similarity_workspace_bytes(ctypes.byref(attrs), x, t, ctypes.byref(n[0])) == 0
        assert lib.simnets_hip_similarity_grad_workspace_bytes(ctypes.byref(attrs), x, t, ctypes.byref(n[1]),
                                                               ctypes.byref(n[2])) == 0
        return [v.value for v in n]
    lib = pkg._lib.lib()
    kw = {k: v for k, v in kw.items() if k in ("blocks", "strides", "padding")}
    norm = dict(normalization_term=mode != "l2", ignore_nan_input=mode == "missing")
    named = [sizes(algo, **kw, **norm) for algo in (["direct", "sqrtw"] if mode == "l2" else ["direct"])]
    # (the gradients' geometry rules are the same for all L2 modes)
    grads, fp32 = sizes(None, **kw), sizes("sqrtw", **kw)
    return dict(forward=all(sizes(None, **kw, **norm)[0] != n[0] for n in named), input=grads[1] != fp32[1],
                params=grads[2] != fp32[2] and mode != "missing")


GEOMS = [
    dict(shape=(5, 16, 40, 40), O=128, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),   # whole tiles, four template tiles
    dict(shape=(9, 13, 33, 31), O=75, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),    # ragged everywhere, 2 + 1 tiles
    dict(shape=(7, 45, 29, 35), O=33, blocks=[3, 3], strides=[1, 1], padding=[0, 2]),    # one template in the second tile
    dict(shape=(40, 40, 12, 11), O=225, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),  # tiles span images, 4 + 4 tiles
    dict(shape=(37, 32, 7, 7), O=160, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),    # several images to a tile
    dict(shape=(3, 20, 61, 67), O=34, blocks=[5, 5], strides=[1, 1], padding=[2, 2]),    # wide rows: chunks of 8 channels
    dict(shape=(9, 24, 62, 65), O=76, blocks=[3, 3], strides=[2, 2], padding=[1, 1]),    # stride 2
    dict(shape=(6, 100, 45, 20), O=40, blocks=[1, 1], strides=[1, 1], padding=[0, 0]),   # one tap
    dict(shape=(90, 16, 9, 9), O=32, blocks=[2, 3], strides=[3, 2], padding=[0, 0]),     # strides beyond the block
    dict(shape=(12, 66, 33, 34), O=31, blocks=[1, 3], strides=[1, 1], padding=[0, 1], out_of_bounds_value=0.5),
    dict(shape=(80, 32, 7, 7), O=160, blocks=[3, 3], strides=[1, 1], padding=[1, 1]),    # several images to a tile
    dict(shape=(20, 20, 34, 37), O=34, blocks=[5, 5], strides=[1, 1], padding=[2, 2]),   # chunks of 8 in every mode
    dict(shape=(20, 40, 41, 31), O=60, blocks=[1, 3], strides=[2, 2], padding=[0, 0]),   # a stride beyond the block
    dict(shape=(20, 40, 41, 20), O=60, blocks=[2, 2], strides=[1, 3], padding=[0, 0]),   # ... the other way
]


def test_geometries_reach_the_form(pkg):
    """The tests below would pass on any form: which of them run on this one."""
    runs = {mode: [pieces_used(pkg, mode=mode, **g) for g in GEOMS] for mode in ("l2", "norm", "missing")}
    used = lambda mode, what: [i for i, r in enumerate(runs[mode]) if r[what]]
    for mode in ("l2", "norm"):
        assert used(mode, "forward") == [0, 1, 2, 3, 5, 6, 7, 9, 10, 11, 12, 13]
        assert used(mode, "params") == [0, 1, 2, 3, 4, 6, 9, 10, 11, 12, 13]
    assert used("missing", "forward") == [0, 1, 2, 3, 7, 9, 11, 12, 13]
    assert used("l2", "input") == [0, 1, 2, 5, 7, 9, 11]    # (3: few tiles of a long contraction)


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("geom", GEOMS)
def test_split_form_matches_64_bits(pkg, geom, mode):
    g = torch.Generator(device="cuda").manual_seed(17)
    shape, O, blocks = geom["shape"], geom["O"], geom["blocks"]
    x = torch.randn(shape, generator=g, device="cuda")
    t = torch.randn((O, shape[1], *blocks), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    kw = options(mode, geom)
    oob = kw.get("out_of_bounds_value", geom.get("out_of_bounds_value", 0.0))
    kw["out_of_bounds_value"] = oob
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    got = pkg.similarity(x, t, w, **kw)
    want = exact(x, t, w, blocks, geom["strides"], geom["padding"], mode, oob)
    # an output is rounded K / 16 + 4 times at no more than its own size and once more as a sum of three of comparable
    # size; the logarithms of the normalized modes are summed at about the same size again
    K = shape[1] * blocks[0] * blocks[1]
    size = want.abs().clamp_min(float(want.abs().mean()))
    err = (got.double() - want).abs() / size
    assert float(err.max()) <= 2 * (K / 16 + 8) * 2.0 ** -24, float(err.max())
    call = pkg.similarity_prepare(shape, t, w, **kw)
    assert torch.equal(call(x), got)


@pytest.mark.parametrize("kind", ["equal", "offset", "negative", "tiny", "huge", "inf", "nan"])
@pytest.mark.parametrize("geom", [GEOMS[1], GEOMS[3], GEOMS[4], GEOMS[5]])
def test_split_form_leaves_what_it_cannot_do_to_the_direct_kernel(pkg, geom, kind):
    g = torch.Generator(device="cuda").manual_seed(23)
    shape, O, blocks = geom["shape"], geom["O"], geom["blocks"]
    kw = options("l2", geom)
    x = torch.randn(shape, generator=g, device="cuda")
    t = torch.randn((O, shape[1], *blocks), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    ph, pw = geom["padding"]
    xp = torch.nn.functional.pad(x, (pw, pw, ph, ph))
    if kind == "equal":      # templates cut out of the input: outputs of zero, and nearly zero
        for m in range(0, O, 5):
            t[m] = xp[m % shape[0], :, m % 5:m % 5 + blocks[0], m % 7:m % 7 + blocks[1]]
        t[1::10] += 1e-4
    elif kind == "offset":
        x += 1000.0
        t += 1000.0
        kw["out_of_bounds_value"] = 1000.0
    elif kind == "negative":
        w[1::4] *= -1.0
    elif kind == "tiny":
        w[2] = 1e-30
        w[3] = 0.0
    elif kind == "huge":
        w[2] = 1e30
        t[3] = 1e25
    elif kind == "inf":
        x[torch.rand(shape, generator=g, device="cuda") < 0.001] = float("inf")
    elif kind == "nan":
        x[torch.rand(shape, generator=g, device="cuda") < 0.001] = float("nan")
    got = pkg.similarity(x, t, w, **kw).cpu().numpy()
    direct = pkg.similarity(x, t, w, algo="direct", **kw).cpu().numpy()
    assert np.array_equal(np.isfinite(got), np.isfinite(direct))
    assert np.array_equal(np.isnan(got), np.isnan(direct))
    fin = np.isfinite(direct)
    # K roundings of the term-by-term sum on one side, 25 K / 16 at the guard's line on the other, and what is below it
    # is the term-by-term sum itself
    K = shape[1] * blocks[0] * blocks[1]
    with np.errstate(invalid="ignore", divide="ignore"):
        err = np.abs(got - direct)[fin] / np.maximum(np.abs(direct[fin]), 1e-37)
    assert err.max() <= 3 * K * 2.0 ** -24, err.max()
    if kind == "equal":
        assert (direct == 0).any() and np.array_equal(got[direct == 0], direct[direct == 0])
    if kind == "offset":
        assert np.array_equal(got, direct)
    if kind == "negative":
        assert np.array_equal(got[:, 1::4], direct[:, 1::4])


def test_split_form_with_everything_missing(pkg):
    geom = GEOMS[1]
    x = torch.full(geom["shape"], float("nan"), device="cuda")
    t = torch.randn((geom["O"], geom["shape"][1], 3, 3), device="cuda")
    got = pkg.similarity(x, t, t.abs() + 0.1, **options("missing", geom))
    assert torch.equal(got, torch.zeros_like(got)) and not torch.signbit(got).any()


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("geom", GEOMS)
def test_split_gradients_match_64_bits(pkg, geom, mode):
    g = torch.Generator(device="cuda").manual_seed(29)
    shape, O, blocks = geom["shape"], geom["O"], geom["blocks"]
    x = torch.randn(shape, generator=g, device="cuda") + 0.5
    t = torch.randn((O, shape[1], *blocks), generator=g, device="cuda") + 0.5
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    kw = options(mode, geom)
    kw.setdefault("out_of_bounds_value", geom.get("out_of_bounds_value", 0.0))
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    (ph, pw), (sh, sw) = geom["padding"], geom["strides"]
    # -w (x - t)^2 (halved, with 0.5 log(w + 0.001), in the normalized modes) as three convolutions in 64 bits
    leaves = [v.double().cpu().requires_grad_() for v in (x, t, w)]
    xd, td, wd = leaves
    xp = torch.nn.functional.pad(xd, (pw, pw, ph, ph), value=kw["out_of_bounds_value"])
    keep = (xp == xp).double()
    xz = torch.where(xp == xp, xp, torch.zeros_like(xp))
    conv = lambda a, b: torch.nn.functional.conv2d(a, b, stride=(sh, sw))
    out = -(conv(xz * xz, wd) - 2 * conv(xz, wd * td) + conv(keep, wd * td * td))
    if mode != "l2":
        out = 0.5 * (out + conv(keep, torch.log(wd + 0.001)))
    go = torch.randn(out.shape, generator=g, device="cuda")
    want = torch.autograd.grad(out, leaves, go.double().cpu())
    dx = pkg.similarity_input_grad(x, t, w, go, **kw)
    dt, dw = pkg.similarity_parameters_grad(x, t, w, go, **kw)
    # n terms of random sign: their sum's error is 2^-24 of the root of the sum of their squares, some n / 3 times added
    # at random, and the moments' combination cancels a few of the size of the terms: 4 sqrt(n) 2^-24 of the scale
    for got, ref, n in ((dx, want[0], O * blocks[0] * blocks[1]), (dt, want[1], go.numel() // O),
                        (dw, want[2], go.numel() // O)):
        err = (got.double().cpu() - ref).norm() / ref.norm()
        assert float(err) <= 4 * math.sqrt(n) * 2.0 ** -24, float(err)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_split_gradients_with_infinite_values(pkg, value):
    """What is not finite reaches the gradients that read it and no others."""
    geom = GEOMS[1]
    g = torch.Generator(device="cuda").manual_seed(31)
    shape, O = geom["shape"], geom["O"]
    x, t = torch.randn(shape, generator=g, device="cuda"), torch.randn((O, shape[1], 3, 3), generator=g, device="cuda")
    kw = options("l2", geom)
    go = torch.randn((shape[0], O, shape[2], shape[3]), generator=g, device="cuda")
    go[3, 7, 11, 30] = value
    dx = pkg.similarity_input_grad(x, t, t.abs() + 0.1, go, **kw)
    bad = torch.zeros_like(dx, dtype=torch.bool)
    bad[3, :, 10:13, 29:31] = True
    assert torch.equal(~torch.isfinite(dx), bad)
    dt, dw = pkg.similarity_parameters_grad(x, t, t.abs() + 0.1, go, **kw)
    for d in (dt, dw):
        rows = ~torch.isfinite(d.flatten(1))
        assert rows[7].any() and not rows[:7].any() and not rows[8:].any()
    go[3, 7, 11, 30] = 0.0
    x[8, 5, 32, 30] = value      # the last image's last corner: taps 0 and 1 of either axis read it
    dt, dw = pkg.similarity_parameters_grad(x, t, t.abs() + 0.1, go, **kw)
    for d in (dt, dw):
        bad = ~torch.isfinite(d)
        assert bad[:, 5, 1:, 1:].all()
        bad[:, 5, 1:, 1:] = False
        assert not bad.any()


def terms_64(x, t, w, go):
    """Parameter gradients of plain L2, 3 x 3, stride 1, padding 1, sum by sum in the order of values (x - t) in 32 bits, as
    the operator defines them, added in 64 bits: infinities and NaN appear where an fp32 evaluation of the terms has them."""
    O, C = t.shape[:2]
    cols = torch.nn.functional.unfold(x, 3, padding=1).permute(1, 0, 2).reshape(C * 9, -1)
    g = go.permute(1, 0, 2, 3).reshape(O, -1)
    dt, dw = (torch.empty((O, C * 9), dtype=torch.float64, device=x.device) for _ in range(2))
    for o in range(O):
        d = cols - t[o].reshape(-1, 1)
        dt[o] = (2 * w[o].reshape(-1, 1) * (g[o] * d)).double().sum(1)
        dw[o] = -((g[o] * d) * d).double().sum(1)
    return dt.reshape(t.shape), dw.reshape(t.shape)


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), 3e19])
@pytest.mark.parametrize("ones", [True, False])
def test_split_parameter_gradients_keep_infinities(pkg, value, ones):
    """An infinite input, or one whose square overflows, gives the gradients the infinities that the terms have - where the
    output gradient's lesser pieces are zero (g = 1) and where they have signs of their own."""
    geom = GEOMS[1]
    g = torch.Generator(device="cuda").manual_seed(37)
    shape, O = geom["shape"], geom["O"]
    x, t = torch.randn(shape, generator=g, device="cuda"), torch.randn((O, shape[1], 3, 3), generator=g, device="cuda")
    w = t.abs() + 0.1
    go = torch.rand((shape[0], O, shape[2], shape[3]), generator=g, device="cuda") + 0.5
    if ones:
        go = torch.ones_like(go)
    x[8, 5, 20, 30] = value
    want = terms_64(x, t, w, go)
    assert want[1][:, 5].isinf().any() and not want[0].isnan().any() and not want[1].isnan().any()
    for got, ref in zip(pkg.similarity_parameters_grad(x, t, w, go, **options("l2", geom)), want):
        inf = ref.isinf()
        assert torch.equal(got[inf].double(), ref[inf])
        err = (got.double() - ref)[~inf].norm() / ref[~inf].norm()
        assert float(err) <= 4 * math.sqrt(go.numel() // O) * 2.0 ** -24, float(err)


@pytest.mark.parametrize("geom, where", [(GEOMS[1], "g"), (GEOMS[2], "g"), (GEOMS[1], "w")])
def test_split_input_gradient_keeps_infinities(pkg, geom, where):
    """One infinite output gradient, or weight: the input gradients that it reaches are infinite with the sign of their
    term g w (t - x), whichever way the channel's centre lies."""
    g = torch.Generator(device="cuda").manual_seed(41)
    shape, O = geom["shape"], geom["O"]
    x, t = torch.randn(shape, generator=g, device="cuda"), torch.randn((O, shape[1], 3, 3), generator=g, device="cuda")
    w = t.abs() + 0.1
    kw = options("l2", geom)
    out = pkg.similarity(x, t, w, **kw).shape
    go = torch.rand(tuple(out), generator=g, device="cuda") + 0.5
    want = torch.zeros_like(x)
    ph, pw = geom["padding"]
    if where == "g":
        go[3, 7, 11, 20] = float("inf")
        r, c = 11 - ph, 20 - pw
        want[3, :, r:r + 3, c:c + 3] = t[7] - x[3, :, r:r + 3, c:c + 3]
    else:
        w[7, 3, 1, 1] = float("inf")
        want[:, 3] = t[7, 3, 1, 1] - x[:, 3]    # the padding lets the middle tap read every input pixel
    dx = pkg.similarity_input_grad(x, t, w, go, **kw)
    reached = want != 0
    assert torch.equal(torch.isfinite(dx), ~reached)
    assert torch.equal(dx[reached], torch.sign(want[reached]) * float("inf"))


@pytest.mark.parametrize("shape, O, depth", [((256, 16, 32, 32), 32, 48), ((32, 128, 28, 28), 128, 26)])
def test_split_parameter_gradients_sum_of_the_output_gradient(pkg, shape, O, depth):
    """x = 0 and t = +-1: the template gradients are +-2 G, and their error is that of G = sum g alone.  Its longest chain of
    additions: 4 within sixteen values, 12 (7) of those per thread, 3 across threads, 21 + 8 (4 + 8) of the partial sums.
    Each rounds by 0.3 ulp (root mean square; an ulp is on average 1.4 * 2^-24 of a value), of partial sums that grow like a
    random walk: 0.4 * 2^-24 sqrt(depth / 2) of the total."""
    g = torch.Generator(device="cuda").manual_seed(0)
    t = torch.randn((O, shape[1], 3, 3), generator=g, device="cuda").sign()
    go = torch.randn((shape[0], O, *shape[2:]), generator=g, device="cuda")
    dt, _ = pkg.similarity_parameters_grad(torch.zeros(shape, device="cuda"), t, torch.ones_like(t), go, padding=[1, 1],
                                           strides=[1, 1])
    want = -2 * t.double() * go.double().sum((0, 2, 3))[:, None, None, None]
    err = float((dt - want).norm() / want.norm())
    assert err <= 2 * 0.4 * 2.0 ** -24 * math.sqrt(depth / 2), err


@pytest.mark.parametrize("spread", [0.3, 0.1, 0.01])
@pytest.mark.parametrize("shape, O, blocks, strides, padding", [
    ((64, 16, 32, 32), 64, [4, 4], [4, 4], [0, 0]),
    ((70, 5, 24, 37), 200, [4, 4], [4, 4], [0, 0]),     # ragged everywhere; 4 + 3 tiles, one and a quarter groups of 64
    ((233, 40, 22, 21), 33, [2, 2], [2, 2], [0, 0]),    # one template in the second tile
    ((64, 12, 37, 38), 129, [3, 3], [3, 3], [3, 0]),    # out-of-bounds rows, 4 + 1 tiles
    ((500, 70, 3, 4), 64, [3, 3], [1, 1], [0, 0]),      # nearly whole images
])
def test_split_parameter_gradients_of_templates_that_share_a_pattern(pkg, shape, O, blocks, strides, padding, spread):
    """Templates, and patches, that are one pattern of size 1 plus differences of size `spread`: the gradients come from the
    differences, and are as exact as those of templates without a pattern (the bound of test_split_gradients_match_64_bits)."""
    g = torch.Generator(device="cuda").manual_seed(47)
    B, C, H, W = shape
    bh, bw = blocks
    pattern = torch.randn((1, C, bh, bw), generator=g, device="cuda")
    t = pattern + spread * torch.randn((O, C, bh, bw), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    tiled = pattern.repeat(1, 1, H // bh + 2, W // bw + 2)
    at = [padding[0] % bh, padding[1] % bw]    # where the first pixel lies in its block
    x = tiled[:, :, at[0]:at[0] + H, at[1]:at[1] + W] + spread * torch.randn(shape, generator=g, device="cuda")
    kw = dict(blocks=blocks, strides=strides, padding=padding)
    assert pieces_used(pkg, shape, O, **kw)["params"]
    xp = torch.nn.functional.pad(x.double(), (padding[1],) * 2 + (padding[0],) * 2)
    cols = xp.unfold(2, bh, strides[0]).unfold(3, bw, strides[1])
    oh, ow = cols.shape[2:4]
    cols = cols.permute(0, 2, 3, 1, 4, 5).reshape(B * oh * ow, -1) - pattern.double().flatten()
    td = t.double().flatten(1) - pattern.double().flatten()
    go = torch.randn((B, O, oh, ow), generator=g, device="cuda")
    gd = go.double().permute(1, 0, 2, 3).reshape(O, -1)
    s1, s2, s0 = gd @ cols, gd @ (cols * cols), gd.sum(1, keepdim=True)
    want = (2 * w.double().flatten(1) * (s1 - td * s0), -(s2 - 2 * td * s1 + td * td * s0))
    for got, ref in zip(pkg.similarity_parameters_grad(x, t, w, go, **kw), want):
        err = (got.double().flatten(1) - ref).norm() / ref.norm()
        assert float(err) <= 4 * math.sqrt(B * oh * ow) * 2.0 ** -24, float(err)


@pytest.mark.parametrize("mode", ["l2", "missing"])
@pytest.mark.parametrize("ratio", [2.0, 1.0, 0.5, 0.3])
@pytest.mark.parametrize("C, block", [(64, 3), (20, 3), (64, 1)])
def test_split_form_near_a_template(pkg, C, block, ratio, mode):
    """Outputs at a given share of sum w t^2, on either side of the guard's line: no further from the 64-bit value than the
    term-by-term sum, K additions of which each rounds by 0.4 * 2^-24 of a partial sum (root mean square, as in
    test_split_parameter_gradients_sum_of_the_output_gradient): 0.4 * 2^-24 sqrt(K / 3) for terms of one sign."""
    g = torch.Generator(device="cuda").manual_seed(53)
    K, O, n = C * block * block, 64, 28 // block
    shape = (16, C, n * block, n * block)
    t = torch.randn((O, C, block, block), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    which = torch.randint(0, O, (shape[0], n, n), generator=g, device="cuda")
    x = t[which].permute(0, 3, 1, 4, 2, 5).reshape(shape)
    x = x + math.sqrt(ratio) * torch.randn(shape, generator=g, device="cuda")
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    kw = options(mode, dict(blocks=[block, block], strides=[1, 1], padding=[0, 0]))
    assert pieces_used(pkg, shape, O, mode, **kw)["forward"]
    if mode == "missing":   # weights at which the logarithm terms vanish: the distance alone
        w = torch.full_like(w, 2 * math.pi - 0.001)
    got = pkg.similarity(x, t, w, **kw)[:, :, ::block, ::block].gather(1, which[:, None])[:, 0].double()
    cols = x.double().unfold(2, block, block).unfold(3, block, block).permute(0, 2, 3, 1, 4, 5)
    d = torch.nan_to_num(cols - t.double()[which])
    want = -(w.double()[which] * d * d).flatten(3).sum(-1) * (0.5 if mode == "missing" else 1.0)
    if mode == "missing":
        log = 0.5 * (torch.log(w.flatten()[:1].double() + 0.001) - math.log(2 * math.pi))
        want = want + log * (cols == cols).flatten(3).sum(-1)
    err = float((((got - want) / want) ** 2).mean().sqrt())
    assert err <= 1.5 * 0.4 * 2.0 ** -24 * math.sqrt(K / 3), err


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("near", [1, 3, 8])
@pytest.mark.parametrize("shape, O, block", [
    ((20, 40, 22, 21), 225, 3),    # chunks of 16 channels, the last of 8
    ((20, 20, 34, 37), 34, 5),     # chunks of 8, the last of 4
    ((20, 65, 24, 25), 33, 1),     # a single tap
])
def test_split_form_recomputes_outputs_near_a_template_alone(pkg, shape, O, block, near, mode):
    """The first image's last row of patches lies close to `near` templates, 19 to 264 outputs: they have the error of a sum
    of their terms, K roundings of at most its size; and the images that share their tiles have the values that they have
    in other company, unless there are more than 128 in a tile."""
    g = torch.Generator(device="cuda").manual_seed(59)
    C, K = shape[1], shape[1] * block * block
    kw = options(mode, dict(blocks=[block, block], strides=[1, 1], padding=[0, 0]))
    x = torch.randn(shape, generator=g, device="cuda")
    t = torch.randn((O, C, block, block), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    value = 2 * torch.randn((C, 1, 1), generator=g, device="cuda")
    t[:near] = value + 0.1 * torch.randn((near, C, block, block), generator=g, device="cuda")
    t[near:2 * near] = -value    # the channels' centres stay away from it
    other = x.clone()
    x[0, :, -block:] = value
    assert pieces_used(pkg, shape, O, mode, **kw)["forward"]
    got = pkg.similarity(x, t, w, **kw)
    want = exact(x[:1], t, w, [block, block], [1, 1], [0, 0], mode, kw.get("out_of_bounds_value", 0.0))
    size = want[0, :near, -1].abs()
    if mode != "l2":    # the terms' and the logarithms' sums have either sign
        size = size + 0.5 * (K * math.log(2 * math.pi) + torch.log(w[:near].double() + 0.001).abs().flatten(1).sum(1))[:, None]
    err = ((got[0, :near, -1].double() - want[0, :near, -1]).abs() / size).max()
    assert float(err) <= K * 2.0 ** -24, float(err)
    if near * got.shape[3] * (block + 1) // 2 <= 128:    # patches that reach half way into those rows are near, too
        assert torch.equal(pkg.similarity(other, t, w, **kw)[1:], got[1:])


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("kind", ["channels", "templates", "far", "small", "sparse", "equal"])
@pytest.mark.parametrize("geom", [GEOMS[1], GEOMS[11], GEOMS[7]])   # chunks of 16 and 8 channels, a single tap
def test_split_form_scales(pkg, geom, kind, mode):
    """Half-precision pieces of values of any size: channels and templates of very different scales, inputs far from the
    templates and close to zero, weights mostly zero, templates that tell no scale.  Bound: test_split_form_matches_64_bits;
    the size of an output is that of its logarithms' sum where that is the larger."""
    g = torch.Generator(device="cuda").manual_seed(61)
    shape, O, blocks = geom["shape"], geom["O"], geom["blocks"]
    x = torch.randn(shape, generator=g, device="cuda")
    t = torch.randn((O, shape[1], *blocks), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    if kind == "channels":
        f = 10.0 ** (torch.rand((shape[1], 1, 1), generator=g, device="cuda") * 6 - 3)
        x, t, w = x * f, t * f, w / f ** 2
    elif kind == "templates":
        w *= 10.0 ** (torch.rand((O, 1, 1, 1), generator=g, device="cuda") * 8 - 5)
    elif kind == "far":
        x *= 300.0
    elif kind == "small":
        x *= 1e-3
    elif kind == "sparse":
        w *= torch.rand(t.shape, generator=g, device="cuda") < 0.05
    elif kind == "equal":
        t.fill_(0.25)
    kw = options(mode, geom)
    oob = kw.setdefault("out_of_bounds_value", geom.get("out_of_bounds_value", 0.0))
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    got = pkg.similarity(x, t, w, **kw).double()
    want = exact(x, t, w, blocks, geom["strides"], geom["padding"], mode, oob)
    K = shape[1] * blocks[0] * blocks[1]
    size = want.abs()
    if mode != "l2":
        logs = 0.5 * (K * math.log(2 * math.pi) + torch.log(w.double() + 0.001).abs().flatten(1).sum(1))
        size = torch.maximum(size, logs[None, :, None, None])
    size = size.clamp_min(1e-30)
    assert float(((got - want).abs() / size).max()) <= 2 * (K / 16 + 8) * 2.0 ** -24


@pytest.mark.parametrize("O, block", [(64, 3), (63, 3), (23, 5), (24, 5), (144, 2)])    # 576, 567, 575, 600, 576 terms
def test_split_input_gradient_scales(pkg, O, block):
    """Images whose output gradients differ by 10^35, channels whose weights and templates differ by many orders: each image
    and channel by itself has the error of its own sums."""
    g = torch.Generator(device="cuda").manual_seed(67)
    B, C, H, W = 36, 37, 23, 30
    f = 10.0 ** (torch.rand((C, 1, 1), generator=g, device="cuda") * 6 - 3)
    x = torch.randn((B, C, H, W), generator=g, device="cuda") * f
    t = torch.randn((O, C, block, block), generator=g, device="cuda") * f
    w = (torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1) / f ** 2
    go = torch.randn((B, O, H - block + 1, W - block + 1), generator=g, device="cuda")
    go *= 10.0 ** torch.linspace(-20, 15, B, device="cuda")[:, None, None, None]
    go[5] = 0.0
    kw = dict(blocks=[block, block], strides=[1, 1], padding=[0, 0])
    assert pieces_used(pkg, (B, C, H, W), O, **kw)["input"]
    got = pkg.similarity_input_grad(x, t, w, go, **kw).double().cpu()
    xd, td, wd, gd = (v.double().cpu() for v in (x, t, w, go))
    up = lambda k: torch.nn.functional.conv_transpose2d(gd, k)
    want = 2 * (up(wd * td) - xd * up(wd))
    assert not got[5].any()
    err = (got - want).flatten(2).norm(dim=2) / want.flatten(2).norm(dim=2).clamp_min(1e-300)
    assert float(err.max()) <= 4 * math.sqrt(O * block * block) * 2.0 ** -24, float(err.max())


@pytest.mark.parametrize("kind", ["templates", "routed", "loud", "pixel"])
@pytest.mark.parametrize("O, block", [(64, 3), (32, 3), (128, 3)])    # 576, 288, 1152 terms
def test_split_input_gradient_over_templates_and_pixels_of_any_size(pkg, O, block, kind):
    """Output gradients that reach templates whose weights are small beside others', and pixels whose output gradients are
    small beside others': every element by itself has the error of a sum of its terms, whatever stands beside them."""
    g = torch.Generator(device="cuda").manual_seed(71)
    B, C, H, W = 36, 37, 23, 30
    x = torch.randn((B, C, H, W), generator=g, device="cuda")
    t = torch.randn((O, C, block, block), generator=g, device="cuda")
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    go = torch.randn((B, O, H - block + 1, W - block + 1), generator=g, device="cuda")
    clear = torch.ones((B, 1, H, W), dtype=torch.bool)
    if kind == "templates":    # ten orders of magnitude, the output gradient the larger the smaller the weights
        f = 10.0 ** (torch.rand((O, 1, 1, 1), generator=g, device="cuda") * 10 - 6)
        w, go = w * f, go / f[:, 0][None]
    elif kind == "routed":     # to four templates of small weights alone
        w[::O // 4] *= 1e-10
        go[:, torch.arange(O, device="cuda") % (O // 4) != 0] = 0.0
    elif kind == "loud":       # one template with large weights that nothing reaches
        w[5] *= 1e8
        go[:, 5] = 0.0
    else:                      # one output pixel of an image beside the others
        r, c = 7, 12
        go[:, :, r, c] *= 1e14
        clear[:, :, r:r + block, c:c + block] = False
    kw = dict(blocks=[block, block], strides=[1, 1], padding=[0, 0])
    assert pieces_used(pkg, (B, C, H, W), O, **kw)["input"]
    got = pkg.similarity_input_grad(x, t, w, go, **kw).double().cpu()
    xd, td, wd, gd = (v.double().cpu() for v in (x, t, w, go))
    up = lambda a, k: torch.nn.functional.conv_transpose2d(a, k)
    want = 2 * (up(gd, wd * td) - xd * up(gd, wd))
    # A - (x - c) B, c of the templates' size at most: each of A and B rounds 6 K / 16 times, at no more than the sum of its
    # terms' sizes
    size = 2 * (up(gd.abs(), wd * (td.abs() + 1)) + (xd.abs() + 1) * up(gd.abs(), wd))
    err = ((got - want).abs() / size.clamp_min(1e-300))[clear.expand_as(got)]
    assert float(err.max()) <= 2 * (O * block * block / 16 + 8) * 2.0 ** -24, float(err.max())


FAR = [("init", 255.0), ("init", 6e4), ("init", 1e8), ("normal", 1e4), ("similar", 1.0), ("similar", 1e-6), ("pixels", 1e3), ("border", 100.0)]


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("kind, size", FAR)
@pytest.mark.parametrize("geom", [GEOMS[i] for i in (0, 1, 3, 7, 11, 12, 13)])
def test_split_form_of_inputs_on_another_scale(pkg, geom, kind, size, mode):
    """Inputs much larger than the templates, or than what the templates differ by: bounds of test_split_form_scales, and the
    outputs are this form's own and not the term-by-term sums of the direct kernel, which agree in the last bit for some."""
    g = torch.Generator(device="cuda").manual_seed(73)
    shape, O, blocks = geom["shape"], geom["O"], geom["blocks"]
    t = torch.randn((O, shape[1], *blocks), generator=g, device="cuda")
    w = torch.ones_like(t)
    if kind == "init":         # a layer's default initialisation on unscaled images
        t = t * 0.05
        x = torch.rand(shape, generator=g, device="cuda") * size
    elif kind == "normal":
        x = torch.randn(shape, generator=g, device="cuda") * size
    elif kind == "pixels":     # one in a hundred
        x = torch.randn(shape, generator=g, device="cuda")
        x *= 1 + size * (torch.rand((shape[0], 1, *shape[2:]), generator=g, device="cuda") < 0.01)
    elif kind == "border":
        t = t * 0.05
        x = torch.randn(shape, generator=g, device="cuda") * 0.05
    else:                      # templates all nearly the same
        t = size * (1 + 1e-4 * t)
        x = torch.randn(shape, generator=g, device="cuda") * size
    kw = options(mode, geom)
    oob = kw.setdefault("out_of_bounds_value", size if kind == "border" else geom.get("out_of_bounds_value", 0.0))
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    assert pieces_used(pkg, shape, O, mode, **kw)["forward"]
    got = pkg.similarity(x, t, w, **kw)
    want = exact(x, t, w, blocks, geom["strides"], geom["padding"], mode, oob)
    K = shape[1] * blocks[0] * blocks[1]
    scale = want.abs()
    if mode != "l2":
        logs = 0.5 * (K * math.log(2 * math.pi) + torch.log(w.double() + 0.001).abs().flatten(1).sum(1))
        scale = torch.maximum(scale, logs[None, :, None, None])
    err = float(((got.double() - want).abs() / scale).max())
    assert err <= 2 * (K / 16 + 8) * 2.0 ** -24, err
    if mode == "missing" and size == 1e8 or mode == "norm" and (size == 1e-6 or kind == "border"):
        return    # beyond the levels of that mode; away from the border nothing but the logarithms' sum
    direct = pkg.similarity(x, t, w, algo="direct", **kw)
    assert float((got == direct).float().mean()) < 0.7


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("geom", [GEOMS[i] for i in (0, 1, 3, 7, 11, 12, 13)])
def test_split_form_of_inputs_on_several_scales(pkg, geom, mode):
    """Pixels, channels and whole images of inputs far from the templates beside ordinary ones: every output by itself has
    the error of a sum of its terms."""
    g = torch.Generator(device="cuda").manual_seed(79)
    shape, O, blocks = geom["shape"], geom["O"], geom["blocks"]
    t = torch.randn((O, shape[1], *blocks), generator=g, device="cuda") * 0.05
    w = torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1
    x = torch.randn(shape, generator=g, device="cuda") * 0.1
    x[:, shape[1] // 2] *= 1e3
    x[1] *= 1e5
    x[2, :, ::7, ::9] *= 1e9
    x[3, -1, 4, 5] = 1e15
    kw = options(mode, geom)
    oob = kw.setdefault("out_of_bounds_value", geom.get("out_of_bounds_value", 0.0))
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    got = pkg.similarity(x, t, w, **kw).double()
    want = exact(x, t, w, blocks, geom["strides"], geom["padding"], mode, oob)
    K = shape[1] * blocks[0] * blocks[1]
    scale = want.abs()
    if mode != "l2":
        logs = 0.5 * (K * math.log(2 * math.pi) + torch.log(w.double() + 0.001).abs().flatten(1).sum(1))
        scale = torch.maximum(scale, logs[None, :, None, None])
    err = float(((got - want).abs() / scale).max())
    assert err <= 2 * (K / 16 + 8) * 2.0 ** -24, err


@pytest.mark.parametrize("mode", ["l2", "norm", "missing"])
@pytest.mark.parametrize("factor", [1e4, 1e6, 1e8])
@pytest.mark.parametrize("geom", [GEOMS[0], GEOMS[1], GEOMS[11], GEOMS[7]])
def test_split_form_of_weights_far_below_their_templates_largest(pkg, geom, factor, mode):
    """One weight of a template is `factor` times the others', the input is on the template there and far from it
    elsewhere: the small weights' terms are all there is of the sum, and it has the error of a sum of its terms.  (The
    large weights lie where the packing kernel takes no samples.)"""
    g = torch.Generator(device="cuda").manual_seed(83)
    shape, O, (bh, bw) = geom["shape"], geom["O"], geom["blocks"]
    t = torch.full((O, shape[1], bh, bw), 0.25, device="cuda")
    w = (torch.rand(t.shape, generator=g, device="cuda") * 1.9 + 0.1) / factor
    x = torch.randn(shape, generator=g, device="cuda").sign() * 20
    rows = range(O) if bh * bw > 1 else range(32, O)
    for m in rows:
        c = 1 + m % 3 if bh * bw > 1 else m
        w[m, c, bh // 2, bw // 2] *= factor
        x[:, c] = 0.25
    kw = options(mode, geom)
    oob = kw.setdefault("out_of_bounds_value", 0.25)
    if mode == "missing":
        x[torch.rand(shape, generator=g, device="cuda") < 0.25] = float("nan")
    got = pkg.similarity(x, t, w, **kw).double()
    want = exact(x, t, w, geom["blocks"], geom["strides"], geom["padding"], mode, oob)
    K = shape[1] * bh * bw
    scale = want.abs()
    if mode != "l2":
        logs = 0.5 * (K * math.log(2 * math.pi) + torch.log(w.double() + 0.001).abs().flatten(1).sum(1))
        scale = torch.maximum(scale, logs[None, :, None, None])
    err = float(((got - want).abs() / scale.clamp_min(1e-30)).max())
    assert err <= 2 * (K / 16 + 8) * 2.0 ** -24, err
