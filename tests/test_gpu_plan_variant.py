"""A call takes its kernels and its twiddle tables from the plan's variant as it
was at one time: with another host thread setting the variant while calls
enqueue, every result is that of one pair of radix schedules."""
import itertools
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM, N0, UNITS = .5, 1.33, (.1, .1, .1)


@pytest.mark.parametrize("n,b,nz,how,mode", [(128, 3, 60, 1, "ignore"), (128, 3, 60, 1, "weighted"),
                                             (128, 3, 60, 0, "ignore"), (1024, 4, 20, 0, "ignore")])
def test_variant_set_while_calls_enqueue(n, b, nz, how, mode):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    rng = np.random.default_rng(n)
    dn = torch.from_numpy(rng.uniform(0, .05, (nz, n, n)).astype(np.float32)).cuda()
    u0 = torch.from_numpy(np.exp(1j * rng.uniform(0, 3, (b, n, n))).astype(np.complex64)).cuda()
    H = B.propagator_table(n, n, UNITS, LAM, N0, _lib.H_F64) if mode == "ignore" else None
    plan = B.Plan(n, n)

    def call():
        p = u0.clone()
        B.propagate_fields(p, nz, UNITS, LAM, N0, dn=dn, dn_kind=_lib.DN_F32, mean_mode=mode, H=H,
                           tuned=False, plan=plan)
        return p

    variants = [(r, c) for r in (1, 4) for c in (1, 6)]  # 4 or 8 points per thread of rows, columns
    stop = threading.Event()

    def turn():
        for v in itertools.cycle(variants):
            if stop.is_set():
                return
            _lib.call("bpmh_plan_set_variant", plan, *v)

    try:
        _lib.call("bpmh_plan_set_loop", plan, how)
        refs = []
        for v in variants:
            _lib.call("bpmh_plan_set_variant", plan, *v)
            refs.append(call())
        torch.cuda.synchronize()
        th = threading.Thread(target=turn)
        th.start()
        try:
            out = [call() for _ in range(40)]
            torch.cuda.synchronize()
        finally:
            stop.set()
            th.join()
        for i, p in enumerate(out):
            assert any(torch.equal(p, r) for r in refs), i
    finally:
        plan.close()
