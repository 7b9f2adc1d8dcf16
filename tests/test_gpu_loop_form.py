"""Which form a call takes: one launch wherever it is built when asked for,
launches per pass when they are, and by grid, batch and schedule by default."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEFAULT, LAUNCHES, LOOP, PART = 0, 1, 2, 3
SCHED = {"4.4": (1, 6), "4.8": (1, 1), "8.4": (4, 6), "8.8": (4, 1)}


def calls(plan):
    from bpm_amd import _lib
    n = ctypes.c_longlong()
    _lib.call("bpmh_plan_loop_calls", plan, ctypes.byref(n))
    return n.value


def forward(plan, nx, ny, b, mode, nz=4):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    dn = torch.full((nz, ny, nx), .01, device="cuda")
    H = B.propagator_table(nx, ny, (.1,) * 3, .5, 1.33, _lib.H_F64) if mode == "ignore" else None
    p = torch.ones((b, ny, nx), dtype=torch.complex64, device="cuda")
    n = calls(plan)
    B.propagate_fields(p, nz, (.1,) * 3, .5, 1.33, dn=dn, dn_kind=_lib.DN_F32, mean_mode=mode, H=H,
                       tuned=False, plan=plan)
    torch.cuda.synchronize()
    return calls(plan) - n


def adjoint(plan, nx, ny, b, mode, nseg=4):
    """(loops run, workspace in planes of the batch) of a segment's adjoint; a
    mean's call runs its forward first."""
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    n2 = nx * ny
    c = lambda *s: torch.ones(s, dtype=torch.complex64, device="cuda")
    g, p, dn, grad = c(b, ny, nx), c(b, ny, nx), torch.zeros((nseg, ny, nx), device="cuda"), torch.zeros((nseg, ny, nx), device="cuda")
    need = ctypes.c_longlong()
    n = calls(plan)
    if mode == "ignore":
        H = B.propagator_table(nx, ny, (.1,) * 3, .5, 1.33, _lib.H_F64)
        useg = c(b, nseg, ny, nx)
        _lib.call("bpmh_adjoint_segment_work", plan, b, 0, nseg - 1, _lib.DN_F32, ctypes.byref(need))
        work = torch.empty(need.value, device="cuda")
        _lib.call("bpmh_adjoint_segment_ws", plan, b, 0, nseg - 1, _lib.ptr(g), _lib.ptr(useg), useg.numel(),
                  _lib.ptr(dn), _lib.DN_F32, dn.numel(), _lib.ptr(H), 1.26, 0, _lib.ptr(grad), _lib.ptr(work),
                  work.numel(), _lib.stream_handle())
    else:
        _lib.call("bpmh_mean_segment_work", plan, b, 0, nseg - 1, 1, ctypes.byref(need))
        work = torch.empty(need.value, device="cuda")
        _lib.call("bpmh_mean_segment", plan, 2, b, 0, nseg - 1, _lib.ptr(p), _lib.ptr(dn), dn.numel(), None, None,
                  1.33, 12.566, .1, .1, .1, 1.26, 0, _lib.ptr(g), _lib.ptr(grad), _lib.ptr(work), work.numel(),
                  _lib.stream_handle())
    torch.cuda.synchronize()
    return calls(plan) - n, need.value / (b * n2)


@pytest.mark.parametrize("nx,ny", [(64, 64), (64, 512), (512, 64), (256, 128), (512, 512), (1024, 64), (32, 64)])
@pytest.mark.parametrize("sched", sorted(SCHED))
def test_form_asked_for(nx, ny, sched):
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    plan = B.Plan(nx, ny)
    try:
        _lib.call("bpmh_plan_set_variant", plan, *SCHED[sched])
        built = 64 <= nx <= 512 and 64 <= ny <= 512 and sched != "8.4"
        adj = built and nx // int(sched[0]) <= 64
        for how in (LAUNCHES, LOOP, PART):
            _lib.call("bpmh_plan_set_loop", plan, how)
            loop, back = int(built and how != LAUNCHES), int(adj and how != LAUNCHES)
            for mode in ("ignore", "weighted"):
                print("case form", nx, ny, sched, how, mode, flush=True)
                assert forward(plan, nx, ny, 2, mode) == loop
            assert adjoint(plan, nx, ny, 2, "ignore") == (back, 3 if back else 1)
            n, planes = adjoint(plan, nx, ny, 2, "weighted")
            assert n == loop + back and (round(planes) >= 20) == bool(back)
    finally:
        plan.close()


def test_form_by_default():
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    for nx, ny, sched, b, mode, loop in (
            (64, 64, "4.4", 1, "ignore", 1), (256, 256, "4.8", 40, "weighted", 1), (512, 256, "4.4", 16, "ignore", 1),
            (512, 256, "4.4", 17, "ignore", 0), (512, 512, "8.8", 1, "ignore", 0), (512, 512, "8.8", 2, "ignore", 1),
            (512, 512, "4.4", 8, "ignore", 0), (512, 512, "8.8", 17, "ignore", 0), (512, 512, "8.8", 20, "ignore", 1),
            (512, 512, "8.8", 40, "weighted", 0), (1024, 256, "4.8", 1, "ignore", 0)):
        plan = B.Plan(nx, ny)
        try:
            _lib.call("bpmh_plan_set_variant", plan, *SCHED[sched])
            print("case default form", nx, ny, sched, b, mode, flush=True)
            assert forward(plan, nx, ny, b, mode) == loop, (nx, ny, sched, b, mode)
        finally:
            plan.close()
