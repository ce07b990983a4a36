"""The adjoints of the real-input transforms (tcfft_exec_r2c_adjoint,
tcfft_exec_c2r_adjoint) against the FP64 oracle at every kernel they have:
the row kernels (n = 512..8192, ragged waves), one workgroup per signal
(16384..65536) and the split as a pass of its own (above).  They are the
transforms with exact factors 1/2 or 2 on bins 1..n/2-1, so the transforms'
own bounds hold: rel-L2 <= 1e-3 up to 65536 points, 1.5e-3 above."""
import numpy as np
import pytest

import oracle
import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [(512, 1), (512, 33), (1024, 5), (2048, 3), (4096, 3), (8192, 1), (8192, 7), (16384, 2), (32768, 1),
         (65536, 2), (1 << 17, 1), (1 << 18, 2)]


def bins_to_dev(X):
    return torch.from_numpy(np.stack([X.real, X.imag], -1).astype(np.float16)).cuda()


@pytest.mark.parametrize("n,batch", CASES, ids=[f"n{n}-b{b}" for n, b in CASES])
def test_adjoints_match_oracle(n, batch):
    print(f"[gpu] real adjoints n={n} batch={batch}", flush=True)
    tol = 1e-3 if n <= 65536 else 1.5e-3
    rng = np.random.default_rng(n + batch)
    plan = tcfft_amd.PlanR2C(n, batch)
    half = n // 2
    X = rng.uniform(-1, 1, (batch, half + 1)) + 1j * rng.uniform(-1, 1, (batch, half + 1))
    X = X.real.astype(np.float16).astype(np.float64) + 1j * X.imag.astype(np.float16).astype(np.float64)
    src, out = bins_to_dev(X), torch.empty(batch, n, dtype=torch.float16, device="cuda")
    plan.exec_r2c_adjoint(src.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    Xh = X.copy()
    Xh[:, 1:-1] *= 0.5
    want = oracle.irfft(Xh, n)
    err = float(np.linalg.norm(out.cpu().numpy().astype(np.float64) - want) / np.linalg.norm(want))
    print(f"  r2c adjoint rel_l2={err:.3e}", flush=True)
    assert err <= tol

    x = (rng.uniform(-1, 1, (batch, n)) / (4 if n > 65536 else 1)).astype(np.float16)
    src, out = torch.from_numpy(x).cuda(), torch.empty(batch, half + 1, 2, dtype=torch.float16, device="cuda")
    plan.exec_c2r_adjoint(src.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    h = out.cpu().numpy().astype(np.float64)
    want = oracle.rfft(x.astype(np.float64))
    want[:, 1:-1] *= 2
    err = oracle.rel_l2(h[..., 0] + 1j * h[..., 1], want)
    print(f"  c2r adjoint rel_l2={err:.3e}", flush=True)
    assert err <= tol
    # bins 0, n/4 and n/2 are written by single lanes: each on its own
    scale = np.sqrt(np.mean(np.abs(want) ** 2))
    for k in (0, n // 4, half):
        assert np.max(np.abs(h[:, k, 0] + 1j * h[:, k, 1] - want[:, k])) <= 8 * tol * scale
    plan.destroy()
