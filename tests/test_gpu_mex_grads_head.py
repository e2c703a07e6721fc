"""Gradients of MEX layers with few instances on few pixels (mex_grad_head_kernel, csrc/mex_grad.hip): one round of pixels to a
workgroup and several, remainders of pixels, elements and instances, sums of up to 128 parts.  Reference: torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# Terms of 2^-22 each (an exponential of a difference), of either sign in a gradient: 1e-6 of the 2-norm, and as much
# again for the chain rule through the normalization.
TOL = 2e-6


@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("batch, K, instances", [
    (1, 64, 10), (3, 1024, 2), (188, 1000, 9), (189, 64, 5), (255, 100, 10), (256, 512, 10), (257, 512, 3), (509, 511, 16), (513, 257, 7), (1030, 1000, 10),
])
def test_gradients(pkg, batch, K, instances, normalize):
    gen = torch.Generator(device="cuda").manual_seed(61)
    x = torch.randn(batch, K, 1, 1, generator=gen, device="cuda")
    off = torch.randn(1, instances, K, 1, 1, generator=gen, device="cuda")
    go = torch.randn(batch, instances, 1, 1, generator=gen, device="cuda")
    leaves = [v.clone().requires_grad_() for v in (x, off)]
    out = pkg.layers.mex(*leaves, instances, blocks=[K, 1, 1], strides=[K, 1, 1], softmax_mode=True, shared_offset_region=[1],
                         normalize_offsets=normalize)
    got = torch.autograd.grad(out, leaves, go)
    exact = [v.cpu().double().requires_grad_() for v in (x, off)]
    rows = exact[1].reshape(instances, K)
    rows = torch.log_softmax(rows, 1) if normalize else rows
    want = torch.autograd.grad(torch.logsumexp(exact[0].reshape(batch, 1, K) + rows, 2), exact, go.cpu().double()[:, :, 0, 0])
    for name, a, b in zip(("input", "offsets"), got, want):
        error = float((a.cpu().double() - b).norm() / b.norm())
        print("%s %.2g" % (name, error))
        assert error <= TOL


@pytest.mark.parametrize("side", [4, 16])
def test_gradients_of_many_regions(pkg, side):
    """A region to each pixel: few partial sums to a row."""
    gen = torch.Generator(device="cuda").manual_seed(63)
    batch, K, instances = 37, 66, 10
    x = torch.randn(batch, K, side, side, generator=gen, device="cuda")
    off = torch.randn(side * side, instances, K, 1, 1, generator=gen, device="cuda")
    go = torch.randn(batch, instances, side, side, generator=gen, device="cuda")
    kw = dict(blocks=[K, 1, 1], strides=[K, 1, 1], softmax_mode=True, unshared_offset_region=[side], normalize_offsets=True)
    leaves = [v.clone().requires_grad_() for v in (x, off)]
    got = torch.autograd.grad(pkg.layers.mex(*leaves, instances, **kw), leaves, go)
    exact = [v.cpu().double().requires_grad_() for v in (x, off)]
    rows = torch.log_softmax(exact[1].reshape(side * side, instances, K), 2)
    out = torch.logsumexp(exact[0].reshape(batch, 1, K, -1) + rows.permute(1, 2, 0), 2)
    want = torch.autograd.grad(out, exact, go.cpu().double().reshape(out.shape))
    for a, b in zip(got, want):
        assert float((a.cpu().double() - b).norm() / b.norm()) <= TOL
