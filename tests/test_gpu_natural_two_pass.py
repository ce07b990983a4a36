"""Natural-order lines of 2^17..2^20 points (two passes cut one stage earlier
than the drop-in plan's, no reversal pass): the drop-in path on the reversed
input gives the same bits, out of place and in place, both directions, one,
odd and chunked batches; and both agree with the FP64 transform (rel-L2 <=
1e-3, the plain path's bound)."""
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [(1 << 17, 1), (1 << 17, 5), (1 << 18, 1), (1 << 18, 3), (1 << 19, 1), (1 << 19, 3), (1 << 20, 1),
         (1 << 20, 3), (1 << 20, 67), (1 << 17, 515)]


@pytest.mark.parametrize("n,batch", CASES, ids=[f"n2^{n.bit_length() - 1}-b{b}" for n, b in CASES])
def test_natural_two_pass_equals_dropin(n, batch):
    print(f"[gpu] natural two pass n={n} batch={batch}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + batch)
    x = (torch.rand(batch, n, 2, generator=g, device="cuda") * 2 - 1).half()
    plan = tcfft_amd.Plan1D(n, batch)
    for direction in (tcfft_amd.FORWARD, tcfft_amd.INVERSE):
        want, got = torch.empty_like(x), torch.empty_like(x)
        plan.permute_to_dropin(x.data_ptr(), want.data_ptr(), batch)
        plan.exec(want.data_ptr(), direction)
        plan.exec_natural(x.data_ptr(), got.data_ptr(), direction)
        own = x.clone()
        plan.exec_natural(own.data_ptr(), own.data_ptr(), direction)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
        assert torch.equal(own.view(torch.int32), want.view(torch.int32))
        z = torch.view_as_complex(x[-1].cpu().double())
        ref = torch.fft.fft(z) if direction < 0 else torch.fft.ifft(z, norm="forward")
        err = float((torch.view_as_complex(got[-1].cpu().double()) - ref).norm() / ref.norm())
        print(f"  dir={direction} rel_l2={err:.3e}", flush=True)
        assert err <= 1e-3
    plan.destroy()
