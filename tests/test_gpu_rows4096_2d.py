"""2D rows of 4096 points on natural-order input: which kernel form a number of
lines takes (one wave per line, 256 threads; two waves through 32 KiB of LDS or
straight into registers with 16; four waves), and that every form gives the
bits of the drop-in path, in and out of place."""
import pytest

import tcfft_amd
from launches import launches

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

KIB = 1024
# (nx, batch): (threads, dynamic LDS) of the row pass on 256 compute units
CASES = [((16, 31), (256, 16 * KIB)), ((16, 33), (128, 16 * KIB)), ((16, 47), (128, 16 * KIB)),
         ((16, 48), (128, 32 * KIB)), ((1024, 1), (128, 32 * KIB)), ((16, 65), (128, 16 * KIB)),
         ((16, 95), (128, 16 * KIB)), ((16, 96), (256, 0)), ((1024, 2), (256, 0)), ((16, 255), (256, 0)),
         ((16, 256), (128, 32 * KIB)), ((16, 257), (128, 32 * KIB)),
         ((128, 6), (128, 16 * KIB)), ((512, 4), (128, 16 * KIB)), ((256, 17), (128, 32 * KIB))]


@pytest.mark.parametrize("shape,form", CASES, ids=[f"{nx}x4096-b{b}" for (nx, b), _ in CASES])
def test_row_form_by_lines(shape, form):
    nx, batch = shape
    print(f"[gpu] natural 2D rows {nx} x 4096 x {batch}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nx + batch)
    x = (torch.rand(batch, nx, 4096, 2, generator=g, device="cuda") * 2 - 1).half()
    plan = tcfft_amd.Plan2D(nx, 4096, batch)
    got = torch.empty_like(x)
    row = launches(lambda st: plan.exec_natural(x.data_ptr(), got.data_ptr(), tcfft_amd.FORWARD, st))[0]
    assert (row.threads, row.shared) == form
    rx = torch.as_tensor(tcfft_amd.gen_rev(nx, plan.radices_x).astype("int64"), device="cuda")
    ry = torch.as_tensor(tcfft_amd.gen_rev(4096, plan.radices_y).astype("int64"), device="cuda")
    for direction in (tcfft_amd.FORWARD, tcfft_amd.INVERSE):
        want = x.index_select(1, rx).index_select(2, ry).contiguous()
        plan.exec(want.data_ptr(), direction)
        plan.exec_natural(x.data_ptr(), got.data_ptr(), direction)
        own = x.clone()
        plan.exec_natural(own.data_ptr(), own.data_ptr(), direction)
        torch.cuda.synchronize()
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
        assert torch.equal(own.view(torch.int32), want.view(torch.int32))
    plan.destroy()
