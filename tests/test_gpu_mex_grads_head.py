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
    (1, 64, 10), (3, 1024, 2), (255, 100, 10), (256, 512, 10), (257, 512, 3), (509, 511, 16), (513, 257, 7), (1030, 1000, 10),
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
