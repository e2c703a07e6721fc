"""Offsets rows of MEX, normalized and packed by a wave each (mex_pack_offsets_kernel, csrc/mex.hip): rows shorter than a wave,
one element more than its registers hold at each of its sizes, rows with infinite entries.
Reference: torch in 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps", [1.0, -0.5, math.inf])
@pytest.mark.parametrize("K", [1, 5, 31, 33, 63, 64, 65, 130, 256, 257, 1024, 1025])
def test_normalized_rows(pkg, K, eps):
    gen = torch.Generator(device="cuda").manual_seed(59)
    x = torch.randn(6, K, 5, 7, generator=gen, device="cuda")
    off = torch.randn(1, 40, K, 1, 1, generator=gen, device="cuda") * 2
    if K > 4 and eps > 0:   # (an infinite extreme value makes the result of a finite epsilon NaN)
        off[0, 3, 2] = -math.inf
    kw = dict(blocks=[K, 1, 1], strides=[K, 1, 1], use_unshared_regions=False, shared_offset_region=[-1], epsilon=eps)
    got = pkg.mex(x, off, 40, normalize_offsets=True, softmax_mode=math.isfinite(eps), **kw).cpu().double()
    rows = torch.log_softmax(off.cpu().double().reshape(40, K), 1)
    terms = x.cpu().double()[:, None] + rows[None, :, :, None, None]
    if eps == math.inf:
        want = terms.amax(2)
    else:
        want = torch.logsumexp(eps * terms, 2) / eps
        # softmax mode: the sum of the exponentials, otherwise their mean
        plain = pkg.mex(x, off, 40, normalize_offsets=True, softmax_mode=False, **kw).cpu().double()
        check(plain, want - math.log(K) / eps, terms)
    check(got, want, terms)


def check(got, want, terms):
    # roundings of 2^-24 of the largest term and of the row's logsumexp, of the exponentials and of a sum of up to 1025 of one
    # sign: 1e-5 of the size of what is added
    finite = want.isfinite()
    assert bool((got[~finite] == want[~finite]).all())
    scale = float(terms[terms.isfinite()].abs().max())
    assert float((got - want)[finite].abs().max()) <= 1e-5 * max(1.0, scale)


def in_fours(batch, side, regions, K, instances):
    """mex_pack_offsets' rule: not one of the layers that run a wave to a pixel (mex_use_small, unpadded rows), instances in
    fours, and 1024 rows of 192 elements, padded to groups of 16, or more."""
    tiles = regions * -(-batch * side * side // regions // 64) * -(-instances // 16)
    rows = regions * -(-instances // 16) * 16
    return tiles >= 256 and instances % 4 == 0 and 64 < K <= 256 and rows * K >= 3 << 16


def special_rows(gen, K, instances):
    """Rows with infinite entries, of one value, of NaN."""
    off = torch.randn(4, instances, K, 1, 1, generator=gen, device="cuda") * 2
    off[0, 3, 2] = -math.inf
    off[1, 5] = 0.25
    off[2, 7] = -math.inf
    off[3, 9, 1] = math.inf
    off[3, 11] = math.nan
    return off


def same(a, b):
    return torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)) and torch.equal(a.isnan(), b.isnan())


@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("eps", [1.0, -0.5, math.inf])
@pytest.mark.parametrize("K", [65, 128, 191, 256])
def test_four_rows_to_a_wave_are_the_same_bits(pkg, K, eps, normalize):
    """Many rows in fours (mex_pack_offsets4_kernel: the forward's layout, with the gradients' beside it where it is finite) and,
    two instances fewer, not in fours: what both have, padding rows included, is equal."""
    gen = torch.Generator(device="cuda").manual_seed(67)
    x = torch.randn(40, K, 8, 8, generator=gen, device="cuda")
    off = special_rows(gen, K, 772)
    go = torch.randn(40, 772, 8, 8, generator=gen, device="cuda")
    go[:, 770:] = 0
    assert in_fours(40, 8, 4, K, 772) and not in_fours(40, 8, 4, K, 770)
    results = []
    for n in (772, 770):
        leaves = [v.clone().requires_grad_() for v in (x, off[:, :n])]
        out = pkg.layers.mex(*leaves, n, blocks=[K, 1, 1], strides=[K, 1, 1], unshared_offset_region=[2], epsilon=eps,
                             softmax_mode=math.isfinite(eps), normalize_offsets=normalize)
        grads = torch.autograd.grad(out, leaves, go[:, :n])
        results.append((out.detach()[:, :770], grads[1][:, :770]))
    for a, b in zip(*results):
        assert same(a, b)


@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("K, instances", [(65, 768), (193, 260), (256, 192)])
def test_four_rows_to_a_wave_in_every_caller(pkg, K, instances, normalize):
    """The forward's layout alone and the gradients' alone: the same bits as from the call that writes both."""
    gen = torch.Generator(device="cuda").manual_seed(71)
    x = torch.randn(70, K, 8, 8, generator=gen, device="cuda")
    off = special_rows(gen, K, instances)
    go = torch.randn(70, instances, 8, 8, generator=gen, device="cuda")
    kw = dict(blocks=[K, 1, 1], strides=[K, 1, 1], unshared_offset_region=[2], softmax_mode=True, normalize_offsets=normalize)
    assert in_fours(70, 8, 4, K, instances)
    leaves = [v.clone().requires_grad_() for v in (x, off)]
    out = pkg.layers.mex(*leaves, instances, **kw)
    want = torch.autograd.grad(out, leaves, go)
    assert same(pkg.mex(x, off, instances, **kw), out.detach())
    for a, b in zip(pkg.mex_grads(x, off, out.detach(), go, instances, **kw), want):
        assert same(a, b)
    # ... and against 64 bits, the rows without special values
    rows = off.double().reshape(4, instances, K)
    rows = torch.log_softmax(rows, 2) if normalize else rows
    for r in range(4):
        part = x.double()[:, :, r // 2::2, r % 2::2]
        exact = torch.logsumexp(part[:2, None] + rows[r, 12:44, :, None, None], 2)
        assert float((out.detach()[:2, 12:44, r // 2::2, r % 2::2] - exact).abs().max()) <= 1e-5 * 20
