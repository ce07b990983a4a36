"""Natural-order first passes: every tile count per wave and load path of the
row kernels (4, 8 and 16 tiles; two or four waves per 4096-point line, straight
from memory or through LDS), whole and ragged last waves, 1D out of place and
in place and 2D rows that fill the chip.  Reference: the drop-in path on the
reversed input, bit for bit (same arithmetic, other loads)."""
import numpy as np
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (n, batch): around 2048 waves of 16, 8 and 4 tiles on 256 CUs
CASES = [(256, 5), (256, 8192 + 3), (256, 32768 + 5), (512, 4096 + 1), (512, 8192 + 3), (512, 16384 + 5), (1024, 2049),
         (1024, 4099), (1024, 8195), (2048, 1027), (2048, 2051), (2048, 4099), (4096, 3), (4096, 513), (4096, 1025),
         (4096, 4099), (8192, 3), (8192, 130), (16384, 5), (32768, 3), (65536, 2)]


@pytest.mark.parametrize("n,batch", CASES, ids=[f"n{n}-b{b}" for n, b in CASES])
def test_natural_equals_dropin_1d(n, batch):
    print(f"[gpu] natural loads n={n} batch={batch}", flush=True)
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
        assert torch.isfinite(want).all()
        assert torch.equal(got, want) and torch.equal(own, want)
    plan.destroy()


CASES_2D = [(4, 256, 3), (64, 1024, 33), (32, 1024, 1030), (16, 2048, 260), (8, 4096, 515), (4, 8192, 65)]


@pytest.mark.parametrize("nx,ny,batch", CASES_2D, ids=[f"{a}x{n}-b{b}" for a, n, b in CASES_2D])
def test_natural_equals_dropin_2d(nx, ny, batch):
    print(f"[gpu] natural loads {nx}x{ny} batch={batch}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nx + ny + batch)
    x = (torch.rand(batch, nx, ny, 2, generator=g, device="cuda") * 2 - 1).half()
    plan = tcfft_amd.Plan2D(nx, ny, batch)
    rx, ry = (torch.as_tensor(tcfft_amd.gen_rev(n, r).astype(np.int64), device="cuda")
              for n, r in ((nx, plan.radices_x), (ny, plan.radices_y)))
    want = x.index_select(1, rx).index_select(2, ry).contiguous()
    plan.exec(want.data_ptr())
    got = torch.empty_like(x)
    plan.exec_natural(x.data_ptr(), got.data_ptr())
    plan.exec_natural(x.data_ptr(), x.data_ptr())
    torch.cuda.synchronize()
    assert torch.equal(got, want) and torch.equal(x, want)
    plan.destroy()
