"""Ragged batches that report each group's completion (done events), as the
server runs them: the bits of the launches per pass, and no group later than
with them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM, N0, UNITS = .5, 1.33, (.1, .1, .1)


def run(n, groups, how, data, reps=1):
    """(fields, sums, fastest of reps: us until each group is done)"""
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    dn, u0, H = data
    plan = B.Plan(n, n)
    try:
        B.apply_tuning(plan, n, n, 16)
        _lib.call("bpmh_plan_set_loop", plan, how)
        best = None
        for _ in range(reps):
            p, acc = u0.clone(), torch.empty(u0.shape, dtype=torch.float32, device="cuda")
            evs = [torch.cuda.Event(enable_timing=True) for _ in groups]
            e0 = torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            torch.cuda._sleep(2_000_000)  # the whole call is enqueued before it starts
            e0.record()
            B.propagate_groups(p, groups, UNITS, LAM, dn, H, groups[0][1] * n * n, out_sum=acc, plan=plan,
                               done_events=evs)
            torch.cuda.synchronize()
            us = np.array([e0.elapsed_time(e) * 1e3 for e in evs])
            best = us if best is None else np.minimum(best, us)
        return p, acc, best
    finally:
        plan.close()


@pytest.mark.parametrize("n,groups,faster", [
    (128, [(8, 200)] * 6, True), (128, [(24, 193), (17, 150), (9, 77)], True), (256, [(8, 120), (8, 90), (1, 9)], True),
    (64, [(9, 40), (2, 40), (70, 12), (1, 2)], False), (256, [(1, 100), (1, 80), (1, 60)], False),
    (512, [(12, 30), (9, 20)], False)])
def test_groups_with_events(n, groups, faster):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    rng = np.random.default_rng(n)
    tot, nz = sum(g[0] for g in groups), groups[0][1]
    dn = torch.rand((len(groups), nz, n, n), device="cuda") * .05
    u0 = torch.from_numpy(np.exp(1j * rng.uniform(0, 3, (tot, n, n))).astype(np.complex64)).cuda()
    data = dn, u0, B.propagator_table(n, n, UNITS, LAM, N0, _lib.H_F64)
    p, acc, us = run(n, groups, 0, data, 4)
    q, sums, launches = run(n, groups, 1, data, 4)
    print(n, groups, us.round(), launches.round(), flush=True)
    assert torch.equal(p, q) and torch.equal(acc, sums)
    # (a tenth and 30 us: what the step times of the rule and the clock leave open)
    assert (us <= 1.1 * launches + 30).all()
    if faster:
        assert us.max() < .85 * launches.max()
