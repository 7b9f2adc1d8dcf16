"""A mean-corrected adjoint given the workspace of one step (asked for under
another loop mode) runs as launches per pass: the same bits, nothing written
beyond it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAUNCHES, LOOP = 1, 2


@pytest.mark.parametrize("mode", [1, 2])
def test_one_step_workspace(mode):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    nx, ny, b, nseg = 128, 64, 2, 7
    rng = np.random.default_rng(6)
    cplx = lambda *s: torch.from_numpy((rng.normal(size=s) + 1j * rng.normal(size=s)).astype(np.complex64)).cuda()
    p0, g0 = cplx(b, ny, nx), cplx(b, ny, nx)
    dn = torch.from_numpy(rng.uniform(0, .05, (nseg, ny, nx)).astype(np.float32)).cuda()
    dn0 = torch.full((nseg,), .02, device="cuda")
    ne = dn0 + 1.33
    plan = B.Plan(nx, ny)

    def need(how):
        n = ctypes.c_longlong()
        _lib.call("bpmh_plan_set_loop", plan, how)
        _lib.call("bpmh_mean_segment_work", plan, b, 0, nseg - 1, 1, ctypes.byref(n))
        return n.value

    def run(how, numel):
        _lib.call("bpmh_plan_set_loop", plan, how)
        g, grad, work = g0.clone(), torch.zeros_like(dn), torch.zeros(numel + 4096, device="cuda")
        _lib.call("bpmh_mean_segment", plan, mode, b, 0, nseg - 1, _lib.ptr(p0), _lib.ptr(dn), dn.numel(),
                  _lib.ptr(ne) if mode == 1 else None, _lib.ptr(dn0) if mode == 1 else None, 1.33, 12.566,
                  .1, .1, .1, 1.26, 3, _lib.ptr(g), _lib.ptr(grad), _lib.ptr(work), numel, _lib.stream_handle())
        torch.cuda.synchronize()
        assert (work[numel:] == 0).all()
        return g, grad

    try:
        one, every = need(LAUNCHES), need(LOOP)
        assert every > one
        ref = run(LAUNCHES, one)
        for numel in (one, every - 1, every):
            for x, y in zip(run(LOOP, numel), ref):
                assert torch.equal(x, y), numel
        with pytest.raises(ValueError):
            run(LOOP, one - 1)
    finally:
        plan.close()
