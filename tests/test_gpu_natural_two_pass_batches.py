"""Natural-order lines of 2^17..2^20 points on both sides of the rule that
sends them through two passes (k_lines_nat, k_rows16r) or, with few signals,
through the reversal pass and the plan's own passes: the launches, the bits of
the drop-in path, and every signal against FP64 (rel-L2 <= 1.5e-3, the plain
path's bound above 65536 points)."""
import pytest

import tcfft_amd
from launches import launches

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# n: batches of the reversal route, batches of the two-pass route
ROUTES = {1 << 17: ((1, 4), (5, 6)), 1 << 18: ((1, 3), (4, 5)), 1 << 19: ((1, 3, 5), (2, 4, 6)),
          1 << 20: ((1, 3), (4, 5))}


@pytest.mark.parametrize("n", ROUTES, ids=[f"n2^{n.bit_length() - 1}" for n in ROUTES])
@pytest.mark.parametrize("direction", [tcfft_amd.FORWARD, tcfft_amd.INVERSE])
def test_few_and_many_signals(n, direction):
    for batch in sum(ROUTES[n], ()):
        print(f"[gpu] natural n={n} batch={batch} dir={direction}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(n + batch)
        x = (torch.rand(batch, n, 2, generator=g, device="cuda") * 2 - 1).half()
        want, got = torch.empty_like(x), torch.empty_like(x)
        plan = tcfft_amd.Plan1D(n, batch)
        call = launches(lambda st: plan.exec_natural(x.data_ptr(), got.data_ptr(), direction, st))
        assert len(call) == (2 if batch in ROUTES[n][1] else 3)
        plan.permute_to_dropin(x.data_ptr(), want.data_ptr(), batch)
        plan.exec(want.data_ptr(), direction)
        plan.exec_natural(x.data_ptr(), got.data_ptr(), direction)
        own = x.clone()
        plan.exec_natural(own.data_ptr(), own.data_ptr(), direction)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
        assert torch.equal(own.view(torch.int32), want.view(torch.int32))
        z = torch.view_as_complex(x.cpu().double())
        ref = torch.fft.fft(z) if direction < 0 else torch.fft.ifft(z, norm="forward")
        err = (torch.view_as_complex(got.cpu().double()) - ref).norm(dim=1) / ref.norm(dim=1)
        assert float(err.max()) <= 1.5e-3
        plan.destroy()


# the half-size transform of a real-input plan: n/2 points; fewest signals of
# the two-pass route
@pytest.mark.parametrize("n,edge", [(1 << 18, 5), (1 << 19, 4), (1 << 20, 2), (1 << 21, 2)])
def test_real_input_plans(n, edge):
    for batch in (edge - 1, edge):
        print(f"[gpu] real n={n} batch={batch}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(n + batch)
        x = ((torch.rand(batch, n, generator=g, device="cuda") * 2 - 1) / 8).half()
        bins = torch.empty(batch, n // 2 + 1, 2, dtype=torch.float16, device="cuda")
        plan = tcfft_amd.PlanR2C(n, batch)
        call = launches(lambda st: plan.exec_r2c(x.data_ptr(), bins.data_ptr(), st))
        assert len(call) == (3 if batch >= edge else 4)
        plan.exec_r2c(x.data_ptr(), bins.data_ptr())
        torch.cuda.synchronize()
        ref = torch.fft.rfft(x.cpu().double())
        err = (torch.view_as_complex(bins.cpu().double()) - ref).norm(dim=1) / ref.norm(dim=1)
        assert float(err.max()) <= 1.5e-3
        plan.destroy()
