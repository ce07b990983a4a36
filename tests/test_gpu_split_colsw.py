"""Split-precision column passes of radix 512..2048 (k_split_colsw): as the
row store and the last pass of 1D 2^17..2^22 and as the strided axis of 2D
shapes, one and several column groups per signal, odd batches, signals a
million times apart in scale, out of place and in place (bit-identical).
Bound: rel-L2 <= 1e-6 against FP64 for every signal."""
import numpy as np
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [(0, 1 << 17, 3), (0, 1 << 18, 1), (0, 1 << 19, 3), (0, 1 << 21, 1), (0, 1 << 22, 1), (512, 256, 3),
         (1024, 512, 3), (2048, 256, 5), (2048, 8192, 1), (512, 65536, 1)]


@pytest.mark.parametrize("nx,n,batch", CASES, ids=[f"{a}x{n}-b{b}" for a, n, b in CASES])
def test_wide_column_passes_vs_fp64(nx, n, batch):
    print(f"[gpu] split colsw {nx}x{n} batch={batch}", flush=True)
    rng = np.random.default_rng(nx + n + batch)
    shape = (batch, nx, n, 2) if nx else (batch, n, 2)
    x = rng.standard_normal(shape, dtype=np.float32)
    x *= (10.0 ** rng.uniform(-3, 3, (batch,) + (1,) * (len(shape) - 1))).astype(np.float32)
    x = torch.from_numpy(x)
    x64 = torch.view_as_complex(x.double())
    dims = (1, 2) if nx else (1,)
    plan = tcfft_amd.Plan2D(nx, n, batch) if nx else tcfft_amd.Plan1D(n, batch)
    plan.prepare_split()
    for direction in (tcfft_amd.FORWARD, tcfft_amd.INVERSE):
        src = x.cuda()
        dst = torch.empty_like(src)
        plan.exec_split(src.data_ptr(), dst.data_ptr(), direction)
        plan.exec_split(src.data_ptr(), src.data_ptr(), direction)
        torch.cuda.synchronize()
        assert torch.equal(src, dst)
        ref = torch.fft.fftn(x64, dim=dims) if direction < 0 else torch.fft.ifftn(x64, dim=dims, norm="forward")
        d = (torch.view_as_complex(dst.cpu().double()) - ref).reshape(batch, -1)
        err = float((d.norm(dim=1) / ref.reshape(batch, -1).norm(dim=1)).max())
        print(f"  dir={direction} per-signal rel_l2 max={err:.3e}", flush=True)
        assert err <= 1e-6
    plan.destroy()
