"""tcfft_permute_to_dropin_f32: the permutation of FP32 lines rounded to fp16,
bit for bit the fp16 permutation of the lines rounded first, zeros, fp16
subnormals, values past fp16's range, infinities and ties included; and the
FFT-conv layer's filter on both routes (an offset view takes the other)."""
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lines", [(256, 3), (4096, 5), (8192, 7), (1 << 16, 2)])
def test_permute_f32_is_the_rounded_permutation(n, lines):
    print(f"[gpu] permute f32 n={n} lines={lines}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + lines)
    x = torch.randn(lines, n, 2, generator=g, device="cuda")
    x *= torch.exp2(torch.randint(-30, 20, (lines, n, 1), generator=g, device="cuda").float())
    x[0, :6, 0] = torch.tensor([0.0, -0.0, float("inf"), 65520.0, 1.0 + 2.0 ** -11, 2.0 ** -25], device="cuda")
    plan = tcfft_amd.Plan1D(n, 1)
    want, got = (torch.empty(lines, n, 2, dtype=torch.float16, device="cuda") for _ in range(2))
    h = x.half()
    plan.permute_to_dropin(h.data_ptr(), want.data_ptr(), lines)
    plan.permute_to_dropin_f32(x.data_ptr(), got.data_ptr(), lines)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # refused as the fp16 permutation refuses it: overlap over 8 bytes a point, alignment
    p = x.data_ptr()
    for args in ((p, p + n * lines * 8 - 16, lines), (p + 8, got.data_ptr(), lines), (p, got.data_ptr(), 0)):
        with pytest.raises(tcfft_amd.TcfftError):
            plan.permute_to_dropin_f32(*args)
    plan.destroy()


def test_conv_filter_routes_agree():
    from tcfft_amd import torch_fft
    n, channels, batch = 4096, 3, 2
    g = torch.Generator(device="cuda").manual_seed(3)
    x = (torch.rand(batch, channels, n, 2, generator=g, device="cuda") * 2 - 1).half()
    flat = torch.randn(channels * n * 2 + 2, generator=g, device="cuda") * 0.02
    off = flat[2:].view(channels, n, 2)  # 8-byte aligned
    ys = [torch_fft._FusedConv.apply(x, w, False) for w in (off, off.clone(), off.transpose(1, 2).contiguous().transpose(1, 2))]
    torch.cuda.synchronize()
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])
