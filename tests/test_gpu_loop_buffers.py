"""One-launch calls in flight on more streams than there are synchronisation
buffers, small and large ones in turn: the bits of the launches per pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM, N0, UNITS = .5, 1.33, (.1, .1, .1)
LAUNCHES, LOOP = 1, 2


def test_overlapping_calls_of_all_sizes():
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    rng = np.random.default_rng(2)
    work = []
    for n, nz, b in ((64, 30, 1), (64, 12, 256), (256, 9, 1), (128, 9, 70)):
        plan = B.Plan(n, n)
        dn = torch.from_numpy(rng.uniform(0, .05, (nz, n, n)).astype(np.float32)).cuda()
        u0 = torch.from_numpy(np.exp(1j * rng.uniform(0, 3, (b, n, n))).astype(np.complex64)).cuda()
        H = B.propagator_table(n, n, UNITS, LAM, N0, _lib.H_F64)

        def call(p, plan=plan, dn=dn, nz=nz, H=H):
            B.propagate_fields(p, nz, UNITS, LAM, N0, dn=dn, dn_kind=_lib.DN_F32, mean_mode="ignore",
                               H=H, tuned=False, plan=plan)

        _lib.call("bpmh_plan_set_loop", plan, LAUNCHES)
        ref = u0.clone()
        call(ref)
        torch.cuda.synchronize()
        _lib.call("bpmh_plan_set_loop", plan, LOOP)
        work.append((plan, call, u0, ref))
    try:
        streams = [torch.cuda.Stream() for _ in range(20)]
        planes = [[w[2].clone() for w in work] for _ in streams]
        torch.cuda.synchronize()
        for s in streams:
            with torch.cuda.stream(s):
                torch.cuda._sleep(2_000_000)
        for turn in range(len(work)):
            for i, s in enumerate(streams):
                k = (i + turn) % len(work)
                with torch.cuda.stream(s):
                    work[k][1](planes[i][k])
        torch.cuda.synchronize()
        for i in range(len(streams)):
            for k, w in enumerate(work):
                assert torch.equal(planes[i][k], w[3]), (i, k)
    finally:
        for w in work:
            w[0].close()
