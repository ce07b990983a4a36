"""Split precision over contiguous lines in one pass (k_split_rows): the two
tile counts per wave (a chip-filling batch runs 16 tiles, the batches of
test_gpu_split_sizes.py fewer), the workgroup of four waves, ragged last
waves, signals a million times apart in one wave, in place and out of place.
Bound: rel-L2 <= 1e-6 against FP64 for every signal."""
import numpy as np
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# 2048 waves of 16 tiles fill the chip (two per SIMD): just below, at and just above
CASES = [(256, 32768 - 17), (256, 32768 + 5), (512, 16384 + 3), (1024, 8192 + 1), (2048, 4096 + 1), (4096, 2048),
         (4096, 2051)]


@pytest.mark.parametrize("n,batch", CASES, ids=[f"n{n}-b{b}" for n, b in CASES])
def test_lines_vs_fp64(n, batch):
    print(f"[gpu] split rows n={n} batch={batch}", flush=True)
    rng = np.random.default_rng(n + batch)
    x = rng.standard_normal((batch, n, 2), dtype=np.float32) * (10.0 ** rng.uniform(-3, 3, (batch, 1, 1)))
    x = torch.from_numpy(x.astype(np.float32))
    x64 = torch.view_as_complex(x.double())
    plan = tcfft_amd.Plan1D(n, batch)
    plan.prepare_split()
    src = x.cuda()
    dst = torch.empty_like(src)
    plan.exec_split(src.data_ptr(), dst.data_ptr(), tcfft_amd.FORWARD)
    plan.exec_split(src.data_ptr(), src.data_ptr(), tcfft_amd.INVERSE)
    torch.cuda.synchronize()
    for got, ref in ((dst, torch.fft.fft(x64)), (src, torch.fft.ifft(x64, norm="forward"))):
        d = torch.view_as_complex(got.cpu().double()) - ref
        err = float((d.norm(dim=1) / ref.norm(dim=1)).max())
        print(f"  per-signal rel_l2 max={err:.3e}", flush=True)
        assert err <= 1e-6
    plan.destroy()
