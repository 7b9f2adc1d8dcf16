"""Waits of the one-launch z-loop that give up (loop mode 4: at once, whatever the
flags are): every kernel ends, all results of the call are NaN, the failure is
reported once, and the next call is right again."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM, N0, UNITS = .5, 1.33, (.1, .1, .1)
LAUNCHES, LOOP, LOST = 1, 2, 4


@pytest.mark.parametrize("b,mode", [(1, "ignore"), (300, "ignore"), (3, "weighted")])
def test_propagation_that_gives_up(b, mode):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    nx = ny = 64
    nz = 5
    rng = np.random.default_rng(4)
    dn = torch.from_numpy(rng.uniform(0, .05, (nz, ny, nx)).astype(np.float32)).cuda()
    u0 = torch.from_numpy(np.exp(1j * rng.uniform(0, 3, (b, ny, nx))).astype(np.complex64)).cuda()
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64) if mode == "ignore" else None
    plan = B.Plan(nx, ny)
    # rooms of one more item that no call may touch
    def outputs():
        return (torch.zeros((b + 1, ny, nx), dtype=torch.complex64, device="cuda"),
                torch.zeros((b + 1, ny, nx), device="cuda"),
                torch.zeros((b + 1, nz, ny, nx), dtype=torch.complex64, device="cuda"))

    def run(how):
        print("case loop failure", nx, ny, b, mode, how, flush=True)
        _lib.call("bpmh_plan_set_loop", plan, how)
        p, acc, vol = outputs()
        p[:b] = u0
        B.propagate_fields(p[:b], nz, UNITS, LAM, N0, dn=dn, dn_kind=_lib.DN_F32, mean_mode=mode, H=H,
                           out_sum=acc[:b], out_field=vol[:b], tuned=False, plan=plan)
        torch.cuda.synchronize()
        return p, acc, vol

    try:
        _lib.call("bpmh_plan_set_variant", plan, 1, 6)
        ref = run(LAUNCHES)
        for x in run(LOST):
            assert torch.isnan(torch.view_as_real(x[:b]) if x.is_complex() else x[:b]).all()
            assert (x[b] == 0).all()
        with pytest.raises(RuntimeError, match="gave up"):
            _lib.call("bpmh_loop_check")
        _lib.call("bpmh_loop_check")
        run(LOST)
        with pytest.raises(RuntimeError, match="gave up"):
            run(LOOP)
        for x, y in zip(run(LOOP), ref):
            assert torch.equal(x, y)
        p = run(LOST)[0]
        with pytest.raises(RuntimeError, match="gave up"):
            _lib.to_numpy(p)
    finally:
        plan.close()
        _lib.load().bpmh_loop_check()


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_adjoint_that_gives_up(mode):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    nx, ny, b, z_hi = 64, 64, 3, 4
    rng = np.random.default_rng(5)
    cplx = lambda *s: torch.from_numpy((rng.normal(size=s) + 1j * rng.normal(size=s)).astype(np.complex64)).cuda()
    dn = torch.from_numpy(rng.uniform(0, .05, (z_hi + 1, ny, nx)).astype(np.float32)).cuda()
    dn0 = torch.full((z_hi + 1,), .02, device="cuda")
    ne = dn0 + N0
    g0, p0, useg = cplx(b, ny, nx), cplx(b, ny, nx), cplx(b, z_hi + 1, ny, nx)
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64)
    plan = B.Plan(nx, ny)

    def run(how):
        print("case adjoint failure", mode, how, flush=True)
        _lib.call("bpmh_plan_set_loop", plan, how)
        g, p, grad, need = g0.clone(), p0.clone(), torch.zeros_like(dn), ctypes.c_longlong()
        if mode == 0:
            _lib.call("bpmh_adjoint_segment_work", plan, b, 0, z_hi, _lib.DN_F32, ctypes.byref(need))
        else:
            _lib.call("bpmh_mean_segment_work", plan, b, 0, z_hi, 1, ctypes.byref(need))
        work = torch.zeros(need.value + 1024, device="cuda")
        if mode == 0:
            _lib.call("bpmh_adjoint_segment_ws", plan, b, 0, z_hi, _lib.ptr(g), _lib.ptr(useg), useg.numel(),
                      _lib.ptr(dn), _lib.DN_F32, dn.numel(), _lib.ptr(H), 1.26, 0, _lib.ptr(grad), _lib.ptr(work),
                      need.value, _lib.stream_handle())
        else:
            _lib.call("bpmh_mean_segment", plan, mode, b, 0, z_hi, _lib.ptr(p), _lib.ptr(dn), dn.numel(),
                      _lib.ptr(ne) if mode == 1 else None, _lib.ptr(dn0) if mode == 1 else None, N0, 12.566, *UNITS,
                      1.26, 0, _lib.ptr(g), _lib.ptr(grad), _lib.ptr(work), need.value, _lib.stream_handle())
        torch.cuda.synchronize()
        assert (work[need.value:] == 0).all()
        return g, grad

    try:
        _lib.call("bpmh_plan_set_variant", plan, 1, 6)
        ref = run(LAUNCHES)
        try:
            g, grad = run(LOST)
            # (plane 0 has a gradient as the weight slice alone)
            assert torch.isnan(torch.view_as_real(g)).all() and torch.isnan(grad[1:]).all()
            with pytest.raises(RuntimeError, match="gave up"):
                _lib.call("bpmh_loop_check")
        except RuntimeError as e:  # the recorded forward had failed before the adjoint was enqueued
            assert "gave up" in str(e)
            torch.cuda.synchronize()
            _lib.load().bpmh_loop_check()
        for x, y in zip(run(LOOP), ref):
            assert torch.equal(x, y)
    finally:
        plan.close()
        _lib.load().bpmh_loop_check()
