"""What tcfft_plan_autotune and tcfft_multi_autotune choose, they choose by
timing the drop-in call: it must not reach the natural-order kernels, which
have other optima.  The launches of a tuned plan's natural-order call are
compared with an untuned plan's."""
import numpy as np
import pytest

import tcfft_amd
from launches import launches

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def natural_launches(plan, x, out, params=None):
    return launches(lambda st: plan.exec_natural(x.data_ptr(), out.data_ptr(), tcfft_amd.FORWARD, st), params)


# shapes whose drop-in optimum (tiles per wave, waves per workgroup) is not the
# natural-order one: 256-point lines (8 tiles against 4), 2D rows (1 wave
# against 4)
@pytest.mark.parametrize("shape", [(256, 16384), (1024, 1024, 8), (2048, 8192)])
def test_tuned_rows_keep_the_natural_launch(shape):
    x = (torch.rand(*(shape[::-1] if len(shape) == 2 else shape), 2, device="cuda") * 2 - 1).half()
    out = torch.empty_like(x)
    make = tcfft_amd.Plan1D if len(shape) == 2 else tcfft_amd.Plan2D
    plain, tuned = make(*shape), make(*shape)
    scratch = x.clone()
    tuned.autotune(scratch.data_ptr())
    a, b = (natural_launches(p, x, out, {0: (6,)})[0] for p in (plain, tuned))
    assert b.key == a.key and b.words == [0]  # parameter 6: the start schedule, its delay first
    # a caller's own choice holds for both calls
    tuned.set_option(tcfft_amd.OPT_ROWS_WAVES, 2)
    assert natural_launches(tuned, x, out)[0].threads == 128
    plain.destroy()
    tuned.destroy()


@pytest.mark.parametrize("n,batch", [(1 << 17, 128), (1 << 20, 16)])
def test_tuned_two_pass_lines_start_together(n, batch):
    """k_lines_nat runs without a start delay (the first word of its parameter
    6, the schedule) unless the caller sets one."""
    x = (torch.rand(batch, n, 2, device="cuda") * 2 - 1).half()
    out = torch.empty_like(x)
    plan = tcfft_amd.Plan1D(n, batch)
    scratch = x.clone()
    plan.autotune(scratch.data_ptr())
    assert natural_launches(plan, x, out, {0: (6,)})[0].words == [0]
    plan.set_option(tcfft_amd.OPT_BIG_DELAY, 2)
    assert natural_launches(plan, x, out, {0: (6,)})[0].words == [2]
    plan.destroy()


def test_uneven_natural_walk_is_kept():
    """A list of more than a task per compute unit in the default order is
    walked from its end (parameter 7 of k_multi_nat) whatever the grid, and
    also after the current schedule is set again or tuned."""
    rng = np.random.default_rng(3)
    sizes = 2 ** rng.integers(8, 17, 2048)
    plan = tcfft_amd.MultiPlan(sizes)
    assert plan.n_tasks > 256
    x = (torch.rand(int(sizes.sum()), 2, device="cuda") * 2 - 1).half()
    out = torch.empty_like(x)

    def reverse(p=plan):
        return natural_launches(p, x, out, {0: (7,)})[0].words[0]

    assert reverse() == 1
    plan.set_schedule(*plan.schedule()[:2])
    assert reverse() == 1
    for grid, order, want in ((0, 0, 1), (512, 0, 1), (128, 0, 1), (256, 2, 0), (256, 1, 0), (256, 0, 1)):
        plan.set_schedule(grid, order)
        assert reverse() == want, (grid, order)
    scratch = x.clone()
    _, order, _ = plan.autotune(scratch.data_ptr())
    assert reverse() == (order == 0)
    few = tcfft_amd.MultiPlan(sizes[:300])
    assert few.n_tasks <= 256 and reverse(few) == 0
    few.destroy()
    plan.destroy()
