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


@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("eps", [1.0, math.inf])
@pytest.mark.parametrize("K", [65, 128, 191, 256])
def test_four_rows_to_a_wave_are_the_same_bits(pkg, K, eps, normalize):
    """Many rows in fours (mex_pack_offsets4_kernel) and, two instances fewer, not in fours: what both have, padding rows
    included, is equal.  Rows with infinite entries, of one value, of NaN."""
    gen = torch.Generator(device="cuda").manual_seed(67)
    x = torch.randn(8, K, 4, 4, generator=gen, device="cuda")
    off = torch.randn(4, 732, K, 1, 1, generator=gen, device="cuda") * 2
    off[0, 3, 2] = -math.inf
    off[1, 5] = 0.25
    off[2, 7] = -math.inf
    off[3, 9, 1] = math.inf
    off[3, 11] = math.nan
    go = torch.randn(8, 732, 4, 4, generator=gen, device="cuda")
    go[:, 730:] = 0
    results = []
    for n in (732, 730):
        leaves = [v.clone().requires_grad_() for v in (x, off[:, :n])]
        out = pkg.layers.mex(*leaves, n, blocks=[K, 1, 1], strides=[K, 1, 1], unshared_offset_region=[2], epsilon=eps,
                             softmax_mode=math.isfinite(eps), normalize_offsets=normalize)
        grads = torch.autograd.grad(out, leaves, go[:, :n])
        results.append((out.detach()[:, :730], grads[1][:, :730]))
    for a, b in zip(*results):
        assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)) and torch.equal(a.isnan(), b.isnan())
