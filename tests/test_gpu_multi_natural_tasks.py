"""Uneven natural-order batches with more tasks than workgroups: the walk from
the end of the list (the default above a task per compute unit) and workgroups
that pass from one size class to the next, reusing their LDS.  The bits of
tcfft_multi_exec on the reversed signals, in both directions, in and out of
place."""
import numpy as np
import pytest

import tcfft_amd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dropin_index(sizes):
    """Flat index of the drop-in order of packed natural-order signals."""
    rev = {}
    for n in set(sizes.tolist()):
        rev[n] = tcfft_amd.gen_rev(n, tcfft_amd.query_1d(n, 1)[0]).astype(np.int64)
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    return torch.from_numpy(np.concatenate([s + rev[int(n)] for s, n in zip(starts, sizes)])).cuda()


# (signals, grid, order): grid None = the plan's defaults (walked from the end
# above 256 tasks: 2048 signals make 480); few workgroups for many tasks else
@pytest.mark.parametrize("signals,grid,order", [(2048, None, 0), (2048, 128, 0), (2048, 31, 1), (160, 5, 0),
                                                (160, 5, 1), (160, 5, 2), (160, 1, 0)])
def test_many_tasks_per_workgroup(signals, grid, order):
    print(f"[gpu] multi natural {signals} signals grid={grid} order={order}", flush=True)
    rng = np.random.default_rng(signals)
    sizes = np.concatenate([2 ** np.arange(8, 17), 2 ** rng.integers(8, 17, signals - 9)]).astype(np.int32)
    rng.shuffle(sizes)
    g = torch.Generator(device="cuda").manual_seed(signals)
    x = (torch.rand(int(sizes.sum()), 2, generator=g, device="cuda") * 2 - 1).half()
    rev = dropin_index(sizes)
    plan = tcfft_amd.MultiPlan(sizes)
    if grid is None:
        assert plan.n_tasks > 256
    else:
        assert plan.n_tasks > grid
        plan.set_schedule(grid, order)
    for direction in (tcfft_amd.FORWARD, tcfft_amd.INVERSE):
        want = x.index_select(0, rev)
        plan.exec(want.data_ptr(), direction)
        out = torch.full_like(x, float("nan"))
        plan.exec_natural(x.data_ptr(), out.data_ptr(), direction)
        own = x.clone()
        plan.exec_natural(own.data_ptr(), own.data_ptr(), direction)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))
        assert torch.equal(own.view(torch.int32), want.view(torch.int32))
    plan.destroy()
