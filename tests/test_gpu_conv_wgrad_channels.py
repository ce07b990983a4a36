"""The natural-order filter gradient on both sides of its rule (a workgroup per
compute unit from 64 channels up on 256 of them) and over the batch remainders
of both kernels (4, and 8 / W entries at a time): the same FP32 sums in the same
order as the digit-reversed call, so the same bits; and with few channels no
slower than those sums in digit-reversed order."""
import statistics

import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def setup(n, channels, batch, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    xs, gs = ((torch.rand(batch, channels, n, 2, generator=g, device="cuda") * 2 - 1).half() for _ in range(2))
    return tcfft_amd.Plan1D(n, batch * channels), xs, gs


@pytest.mark.parametrize("n", [4096, 8192, 16384])
@pytest.mark.parametrize("channels,batch", [(1, 1), (1, 3), (2, 4), (3, 5), (7, 9), (33, 6), (63, 8), (64, 1), (64, 7),
                                            (65, 10)])
def test_same_bits(n, channels, batch):
    print(f"[gpu] wgrad n={n} C={channels} B={batch}", flush=True)
    plan, xs, gs = setup(n, channels, batch, n + channels + batch)
    rev, nat = (torch.full((channels, n, 2), float("nan"), device="cuda") for _ in range(2))
    plan.conv_filter_grad(channels, xs.data_ptr(), gs.data_ptr(), rev.data_ptr())
    plan.conv_filter_grad_natural(channels, xs.data_ptr(), gs.data_ptr(), nat.data_ptr())
    torch.cuda.synchronize()
    idx = torch.as_tensor(tcfft_amd.gen_rev(n, plan.radices).astype("int64"), device="cuda")
    want = torch.empty_like(rev).index_copy_(1, idx, rev)
    assert torch.equal(nat, want)
    plan.destroy()


@pytest.mark.parametrize("n,channels,batch", [(16384, 32, 32), (8192, 48, 24)])
def test_few_channels_are_not_slower(n, channels, batch):
    """Whole cache lines per workgroup: 24.7 us against 27.5 for 32 x 16384 over
    32 entries, 51 with 64-byte reads.  The bound is half way."""
    plan, xs, gs = setup(n, channels, batch, 1)
    out = torch.empty(channels, n, 2, device="cuda")

    def timed(call):
        graph = torch.cuda.CUDAGraph()
        call(channels, xs.data_ptr(), gs.data_ptr(), out.data_ptr())
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            for _ in range(20):
                call(channels, xs.data_ptr(), gs.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        ts = []
        for _ in range(9):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            ts.append(a.elapsed_time(b))
        return statistics.median(ts)

    rev, nat = timed(plan.conv_filter_grad), timed(plan.conv_filter_grad_natural)
    print(f"  digit-reversed {rev * 50:.1f} us, natural {nat * 50:.1f} us", flush=True)
    assert nat <= 1.4 * rev
    plan.destroy()
