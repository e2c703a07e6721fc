"""Both MEX gradients of layers with 2 x 2 unshared offsets over whole-channel patches on maps with power-of-two sides
(mex_grads_rows_kernel and mex_grad_offsets_rows_kernel, csrc/mex_grad.hip): maps of two columns, several chunks of pixels to a workgroup (its partial sums are
added to), 16 and 32 patch elements to a workgroup, instance groups split, rows that are no whole 16-byte pieces, few chunks on
eight dies, and regions that a wide offsets range, or one chunk's wide pixels, send to the term-by-term path.
Reference: torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# Three factors to a term, whose exponents of two are at most about 64 and known to 2^-24 of themselves: 3 * 64 * ln 2 * 2^-24
TOL = 8e-6


def reference(x, off, g):
    x, off = x.double().requires_grad_(), off.double().requires_grad_()
    n, c = off.shape[1], x.shape[1]
    out = torch.empty(g.shape, dtype=torch.float64, device=x.device)
    dx, doff = torch.zeros_like(x), torch.zeros_like(off)
    step = max(1, (1 << 25) // (n * x[0].numel()))
    for i in range(0, x.shape[0], step):
        for r in range(4):
            part = (slice(i, i + step), slice(None), slice(r // 2, None, 2), slice(r % 2, None, 2))
            y = torch.logsumexp(x[part][:, None] + off[r].reshape(1, n, c, 1, 1), 2)
            gx, go = torch.autograd.grad(y, (x, off), g[part].double())
            dx += gx
            doff += go
            out[part] = y.detach()
    return out.float(), dx, doff


def err(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("shape,n,spread,outlier", [
    ((70, 24, 2, 2), 40, 0.5, False),        # two columns, a quad of pixels is a window; the last chunk part empty
    ((9, 20, 8, 2), 33, 3.0, False),         # offsets beyond the few-instances bound: the pixels' own maxima
    ((130, 64, 2, 2), 200, 0.5, False),      # instance groups split, three chunks on eight dies
    ((3, 32, 2, 2), 64, 12.0, False),        # term by term, one chunk
    ((1030, 6, 16, 16), 5, 0.5, False),      # two chunks to a workgroup, rows of six elements
    ((1027, 8, 16, 16), 33, 0.5, False),     # ... of eight, two instance groups, an odd number of chunks
    ((1026, 8, 16, 16), 3, 4.5, True),       # ... one chunk's pixels term by term, the other's not
    ((520, 33, 8, 8), 40, 0.5, False),       # 16 elements to a workgroup, the last of 33
    ((70, 48, 4, 4), 70, 3.0, False),
    # the offsets' gradient in a kernel of its own
    ((1030, 24, 16, 16), 40, 0.5, False),    # a single tile of patch elements, two groups, two chunks to a workgroup
    ((1030, 17, 16, 16), 9, 3.0, True),      # ... one group, rows that are no whole 16-byte pieces, infinite pixels' flags
    ((515, 50, 16, 16), 20, 0.5, False),     # two tiles, the last of 18; the input's gradient beside it
    ((2100, 70, 4, 8), 40, 3.0, True),       # three, tight bounds
    ((515, 64, 16, 16), 8, 12.0, False),     # ... term by term
    ((33, 20, 8, 8), 230, 0.5, False),       # eight groups
    ((130, 256, 8, 8), 1030, 0.5, False),    # many terms
])
@pytest.mark.parametrize("normalize", [False, True])
def test_row_wise_gradients(pkg, shape, n, spread, outlier, normalize):
    gen = torch.Generator(device="cuda").manual_seed(97)
    b, c, h, w = shape
    x = torch.randn(shape, generator=gen, device="cuda")
    if outlier:
        x[1, 0, 3, 4] = 70.0
        x[1, 1, 3, 4] = -70.0
    raw = torch.randn(4, n, c, 1, 1, generator=gen, device="cuda") * spread
    used = raw - torch.logsumexp(raw.double(), 2, keepdim=True).float() if normalize else raw
    g = torch.randn(b, n, h, w, generator=gen, device="cuda")
    out, want_x, want_off = reference(x, used, g)
    if normalize:
        want_off = want_off - used.double().exp() * want_off.sum(2, keepdim=True)
    kw = dict(blocks=[c, 1, 1], strides=[c, 1, 1], unshared_offset_region=[2], softmax_mode=True,
              normalize_offsets=normalize)
    dx, doff = pkg.mex_grads(x, raw, out, g, n, **kw)
    errors = err(dx, want_x), err(doff, want_off)
    print("input %.2g, offsets %.2g" % errors)
    assert max(errors) <= TOL
    # either alone: the same bits
    assert torch.equal(dx, pkg.mex_input_grad(x, raw, out, g, n, **kw))
    assert torch.equal(doff, pkg.mex_offsets_grad(x, raw, out, g, n, **kw))
    # the gradient of the pooled output: as its expansion
    full, pooled = pkg.mex_sum_pool_both(x, raw, n, (2, 2), **kw)
    gp = torch.randn(pooled.shape, generator=gen, device="cuda")
    want = pkg.mex_grads(x, raw, full, pkg.sum_pooling_input_grad(gp, full.shape, (2, 2)), n, **kw)
    got = pkg.mex_sum_pool_grads(x, raw, full, gp, n, (2, 2), **kw)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("shape", [(65930, 6, 2, 2), (1030, 6, 16, 16)])   # two chunks to a workgroup
def test_pixels_of_one_chunk_leave_the_next_ones_alone(pkg, shape):
    """Offsets that span 29 exponents, so that each chunk's pixels decide; those of the first chunk send all four regions
    term by term.  The input's gradient of the other chunks is the same bits as without them."""
    gen = torch.Generator(device="cuda").manual_seed(101)
    b, c, h, w = shape
    n, chunk = 5, 256 // (h * w)   # (images)
    off = torch.rand(4, n, c, 1, 1, generator=gen, device="cuda") * 20
    off[:, 0, 0], off[:, 0, 1] = 0, 20
    g = torch.randn(b, n, h, w, generator=gen, device="cuda")
    kw = dict(blocks=[c, 1, 1], strides=[c, 1, 1], unshared_offset_region=[2], softmax_mode=True)
    results = []
    for outlier in (False, True):
        x = torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(103), device="cuda")
        if outlier:
            x[0, 0, :2, :2], x[0, 1, :2, :2] = 70, -70
        out, want_x, want_off = reference(x, off, g)
        dx, doff = pkg.mex_grads(x, off, out, g, n, **kw)
        assert max(err(dx, want_x), err(doff, want_off)) <= TOL
        results.append(dx)
    assert torch.equal(results[0][chunk:], results[1][chunk:])


@pytest.mark.parametrize("value", [-70, -float("inf")])
@pytest.mark.parametrize("shape", [(65930, 6, 2, 2), (1030, 6, 16, 16), (70, 24, 8, 4)])
def test_offsets_gradient_keeps_its_form_for_wide_pixels(pkg, shape, value):
    """Offsets that span 29 exponents and pixels that span more than 64: the input's gradient is formed term by term, the
    offsets' as without them - the same bits where those pixels' output gradients are zero."""
    gen = torch.Generator(device="cuda").manual_seed(107)
    b, c, h, w = shape
    n = 5
    off = torch.rand(4, n, c, 1, 1, generator=gen, device="cuda") * 20
    off[:, 0, 0], off[:, 0, 1] = 0, 20
    g = torch.randn(b, n, h, w, generator=gen, device="cuda")
    kw = dict(blocks=[c, 1, 1], strides=[c, 1, 1], unshared_offset_region=[2], softmax_mode=True)
    results = []
    for outlier in (False, True):
        x = torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(103), device="cuda")
        if outlier:
            x[::7, 0, :2, :2], x[::7, 1, :2, :2] = 70, value
        out, want_x, want_off = reference(x, off, g)
        dx, doff = pkg.mex_grads(x, off, out, g, n, **kw)
        assert max(err(dx, want_x), err(doff, want_off)) <= TOL
        quiet = g.clone()
        quiet[::7, :, :2, :2] = 0
        results.append(pkg.mex_offsets_grad(x, off, out, quiet, n, **kw))
    assert torch.equal(*results)


def test_offsets_gradient_of_an_infinite_pixel(pkg):
    """Offsets that span 29 exponents: an infinite value makes its own element's gradient NaN and leaves the others to the
    other pixels."""
    gen = torch.Generator(device="cuda").manual_seed(109)
    shape, n = (520, 64, 16, 16), 6
    x = torch.randn(shape, generator=gen, device="cuda")
    off = torch.rand(4, n, 64, 1, 1, generator=gen, device="cuda") * 20
    off[:, 0, 0], off[:, 0, 1] = 0, 20
    g = torch.randn(shape[0], n, 16, 16, generator=gen, device="cuda")
    kw = dict(blocks=[64, 1, 1], strides=[64, 1, 1], unshared_offset_region=[2], softmax_mode=True)
    plain = pkg.mex_offsets_grad(x, off, reference(x, off, g)[0], g, n, **kw)
    x[3, 7, 4, 6] = float("inf")   # region 0
    out = reference(x, off, g)[0]
    assert out[3, :, 4, 6].isinf().all()
    doff = pkg.mex_grads(x, off, out, g, n, **kw)[1]
    assert torch.equal(doff[0].isnan().nonzero()[:, 1].unique().cpu(), torch.tensor([7]))
    assert err(doff[1:], plain[1:].double()) <= TOL
    g[3, :, 4, 6] = 0
    want = reference(torch.where(x.isinf(), torch.zeros_like(x), x), off, g)[2]
    keep = [k for k in range(64) if k != 7]
    assert err(doff[:, :, keep], want[:, :, keep]) <= TOL
