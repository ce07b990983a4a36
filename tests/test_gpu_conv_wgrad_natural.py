"""The filter gradient in natural spectrum order against the digit-reversed
one gathered by the plan's gen_rev: the same FP32 sums in the same order, so
within 1e-6 of the gradient's rms.  Both workgroup shapes (four times the
channels below and above the CU count), one and odd batches."""
import numpy as np
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [(4096, 1, 1), (4096, 70, 3), (8192, 3, 5), (8192, 64, 2), (16384, 2, 7), (16384, 67, 1)]


@pytest.mark.parametrize("n,channels,batch", CASES, ids=[f"n{n}-c{c}-b{b}" for n, c, b in CASES])
def test_natural_filter_gradient(n, channels, batch):
    print(f"[gpu] wgrad natural n={n} C={channels} B={batch}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + channels + batch)
    xs, gs = ((torch.rand(batch, channels, n, 2, generator=g, device="cuda") * 2 - 1).half() for _ in range(2))
    plan = tcfft_amd.Plan1D(n, batch * channels)
    rev, nat = (torch.full((channels, n, 2), float("nan"), device="cuda") for _ in range(2))
    plan.conv_filter_grad(channels, xs.data_ptr(), gs.data_ptr(), rev.data_ptr())
    plan.conv_filter_grad_natural(channels, xs.data_ptr(), gs.data_ptr(), nat.data_ptr())
    torch.cuda.synchronize()
    idx = torch.as_tensor(tcfft_amd.gen_rev(n, plan.radices).astype(np.int64), device="cuda")
    want = torch.empty_like(rev).index_copy_(1, idx, rev)
    assert torch.isfinite(nat).all()
    assert float((nat - want).abs().max()) <= 1e-6 * float(want.square().mean().sqrt())
    plan.destroy()


def test_natural_filter_gradient_rejects():
    p = tcfft_amd.Plan1D(2048, 2)
    t = torch.zeros(4096 * 4, device="cuda")
    with pytest.raises(tcfft_amd.TcfftError):
        p.conv_filter_grad_natural(1, t.data_ptr(), t.data_ptr(), t.data_ptr())
    p.destroy()
    p = tcfft_amd.Plan1D(4096, 3)
    for c in (0, 2):
        with pytest.raises(tcfft_amd.TcfftError):
            p.conv_filter_grad_natural(c, t.data_ptr(), t.data_ptr(), t.data_ptr())
    p.destroy()
