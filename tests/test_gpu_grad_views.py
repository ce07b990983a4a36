"""Gradients and filters that reach the torch functions as views: contiguous
at any element offset, as autograd hands out the parts of a concatenation."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# the row kernel, one workgroup per signal, and the split as a pass of its own
@pytest.mark.parametrize("n,batch", [(512, 5), (32768, 2), (1 << 17, 1)])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_rfft_gradient_at_any_offset(n, batch, offset):
    """The gradient of y behind torch.cat([head, y.flatten()]) is a contiguous
    narrow() that starts `offset` halves into a buffer: the same bits as the
    gradient from an aligned copy."""
    from tcfft_amd import torch_fft
    g = torch.Generator(device="cuda").manual_seed(n + offset)
    x = (torch.rand(batch, n, generator=g, device="cuda") * 2 - 1).half().requires_grad_(True)
    up = (torch.rand(offset + batch * (n // 2 + 1) * 2, generator=g, device="cuda") * 2 - 1).half()
    head = torch.zeros(offset, dtype=torch.float16, device="cuda")
    y = torch_fft.rfft(x)
    want = torch.autograd.grad(y, x, up[offset:].clone().view(y.shape), retain_graph=True)[0]
    got = torch.autograd.grad(torch.cat([head, y.flatten()]), x, up)[0]
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_lazily_negated_gradient_and_filter():
    """A tensor whose sign flip is still pending (is_neg) counts with it."""
    from tcfft_amd import torch_fft
    g = torch.Generator(device="cuda").manual_seed(5)
    x = (torch.rand(3, 512, generator=g, device="cuda") * 2 - 1).half().requires_grad_(True)
    y = torch_fft.rfft(x)
    up = (torch.rand(y.shape, generator=g, device="cuda") * 2 - 1).half()
    want = torch.autograd.grad(y, x, -up, retain_graph=True)[0]
    got = torch.autograd.grad(y, x, torch._neg_view(up))[0]
    assert torch.equal(got, want)
    sig = (torch.rand(2, 3, 4096, 2, generator=g, device="cuda") * 2 - 1).half()
    w = torch.randn(3, 4096, 2, generator=g, device="cuda")
    want = torch_fft._FusedConv.apply(sig, -w, False)
    got = torch_fft._FusedConv.apply(sig, torch._neg_view(w), False)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
