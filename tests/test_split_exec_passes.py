"""The split-precision passes tcfft_exec_split runs (tcfft_query_split_exec,
host only): each is run in FP64 as its descriptor states, and the sequence must
give numpy's own FFT of the shape; a pass over whole lines is an R-point DFT of
every contiguous line.  This pins the radices, strides, twiddle moduli and grid
sizes that reach the kernels, without a device."""
import numpy as np
import pytest

import tcfft_amd
from test_split_passes import apply_pass


def run_model(x, passes, sign):
    total = x.size
    for p in passes:
        sig_len = p["R"] << p["q_log2"]
        signals = total // sig_len
        assert p["units"] == (signals if p["q_log2"] == 0 else signals * (1 << p["q_log2"]) // 16)
        x = apply_pass(x.reshape(signals, sig_len), p, sign)
    return x


def kernels_take(passes):
    """What launch_split_rows and launch_split_pass accept."""
    for i, p in enumerate(passes):
        if p["q_log2"] == 0:  # k_split_rows
            assert 256 <= p["R"] <= 4096 and p["qlo_log2"] == 0 and p["m_log2"] == 0
            continue
        assert p["q_log2"] >= 4
        row = p["qlo_log2"] == 0  # the transposed store
        assert (2 if not row else 64) <= p["R"] <= 2048
        assert row or p["qlo_log2"] >= 4
        if p["m_log2"]:
            assert p["qlo_log2"] < p["q_log2"]
            assert (1 << p["m_log2"]) == (p["R"] << p["q_log2"]) >> p["qlo_log2"]
            assert row or 16 <= p["R"] <= 256  # the other kernels have no twiddle in the column store
        else:
            assert p["qlo_log2"] == p["q_log2"]  # in place


@pytest.mark.parametrize("n", [1 << k for k in range(8, 23) if k != 16])
def test_1d_passes_compute_the_dft(n):
    batch = 3 if n <= (1 << 20) else 1
    passes = tcfft_amd.query_split_exec(1, n, 0, batch)
    kernels_take(passes)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((batch, n)) + 1j * rng.standard_normal((batch, n))
    for sign in (-1, 1):
        got = run_model(x.copy(), passes, sign).reshape(batch, n)
        ref = np.fft.fft(x, axis=-1) if sign < 0 else np.fft.ifft(x, axis=-1) * n
        assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 1e-12


# every radix of a strided axis, over rows of one pass and of several
@pytest.mark.parametrize("nx,ny", [(2, 256), (8, 4096), (16, 512), (32, 8192), (128, 256), (256, 2048), (512, 256),
                                   (512, 8192), (1024, 1024), (2048, 256), (2048, 1024), (4096, 256), (4, 65536)])
def test_2d_passes_compute_the_dft(nx, ny):
    batch = 2
    passes = tcfft_amd.query_split_exec(2, nx, ny, batch)
    kernels_take(passes)
    rng = np.random.default_rng(nx * ny)
    x = rng.standard_normal((batch, nx, ny)) + 1j * rng.standard_normal((batch, nx, ny))
    for sign in (-1, 1):
        got = run_model(x.copy().reshape(-1), passes, sign).reshape(batch, nx, ny)
        ref = np.fft.fft2(x) if sign < 0 else np.fft.ifft2(x) * (nx * ny)
        assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 1e-12


def test_number_of_passes():
    """Lines of 256..4096 points and strided axes of up to 2048 take one pass,
    1D 2^13..2^22 two, 2^23 and 2^24 three, above four; 65536 has its own
    kernel (no list); the passes of a shape multiply to its size."""
    for k in range(8, 28):
        passes = tcfft_amd.query_split_exec(1, 1 << k)
        kernels_take(passes)
        assert len(passes) == (0 if k == 16 else 1 if k <= 12 else 2 if k <= 22 else 3 if k <= 24 else 4), k
        assert k == 16 or sum(p["R"].bit_length() - 1 for p in passes) == k
    for kx in range(1, 17):
        for ky in range(8, 17):
            if kx + ky > 27:
                continue
            passes = tcfft_amd.query_split_exec(2, 1 << kx, 1 << ky)
            kernels_take(passes)
            assert len(passes) == (1 if ky <= 12 else 2) + (1 if kx <= 11 else 2), (kx, ky)
            assert sum(p["R"].bit_length() - 1 for p in passes) == kx + ky


def test_rejects_what_query_split_rejects():
    for args in ((1, 100, 0, 1), (1, 128, 0, 1), (1, 1 << 28, 0, 1), (2, 256, 128, 1), (3, 256, 256, 1),
                 (1, 1 << 20, 0, 4096)):
        with pytest.raises(tcfft_amd.TcfftError):
            tcfft_amd.query_split_exec(*args)
