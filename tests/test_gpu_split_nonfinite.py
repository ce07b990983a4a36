"""Split precision with infinities, NaN and extreme magnitudes in single
signals: a wave of k_split_rows holds up to 16 lines, each with its own scale,
and k_split_colsw's scales never cross signals, so every other signal keeps its
bits; a signal with a non-finite value has no finite output, as its DFT has
none."""
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# lines with few tiles per wave, with 16 (a full chip), and two wide passes
@pytest.mark.parametrize("n,batch", [(256, 37), (256, 32768 + 5), (512, 33), (1024, 19), (1024, 8192 + 1), (2048, 9),
                                     (4096, 7), (1 << 17, 5), (1 << 20, 4)])
def test_other_signals_keep_their_bits(n, batch):
    print(f"[gpu] split non-finite n={n} batch={batch}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + batch)
    x = torch.randn(batch, n, 2, generator=g, device="cuda")
    plan = tcfft_amd.Plan1D(n, batch)
    plan.prepare_split()
    for direction in (tcfft_amd.FORWARD, tcfft_amd.INVERSE):
        clean = torch.empty_like(x)
        plan.exec_split(x.data_ptr(), clean.data_ptr(), direction)
        bad = x.clone()
        rows = (0, batch // 2, batch - 1)
        bad[rows[0], n // 3, 0] = float("inf")
        bad[rows[1], n - 1, 1] = float("nan")
        bad[rows[2], 5, 1] = -float("inf")
        bad[1] *= 1e30  # finite: scaled by a neighbour's power of two it would vanish or overflow
        bad[2] *= 1e-30
        got = torch.empty_like(x)
        plan.exec_split(bad.data_ptr(), got.data_ptr(), direction)
        plan.exec_split(bad.data_ptr(), bad.data_ptr(), direction)
        torch.cuda.synchronize()
        assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), bad.nan_to_num(7.0, 8.0, 9.0))
        for r in rows:
            assert not torch.isfinite(got[r]).any()
        keep = torch.ones(batch, dtype=torch.bool, device="cuda")
        for r in (*rows, 1, 2):
            keep[r] = False
        assert torch.equal(got[keep], clean[keep])
        for r, f in ((1, 1e30), (2, 1e-30)):
            if r in rows:
                continue
            ref = torch.view_as_complex(x[r].double() * f)
            ref = torch.fft.fft(ref) if direction < 0 else torch.fft.ifft(ref, norm="forward")
            err = (torch.view_as_complex(got[r].double()) - ref).norm() / ref.norm()
            assert float(err) <= 1e-6
    plan.destroy()
