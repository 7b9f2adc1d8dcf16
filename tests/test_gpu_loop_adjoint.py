"""The adjoint of a segment in one launch (bpmh_plan_set_loop) against the
launches per pass: the same operations on every line and the same order of
every sum, so the same bits, for every mean mode, with complete and incomplete
teams; a workspace of one step keeps the launches."""
import ctypes
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM, N0, UNITS = .5, 1.33, (.1, .1, .1)
LAUNCHES, LOOP, PART = 1, 2, 3
SCHED = {"4.4": (1, 6), "4.8": (1, 1), "8.8": (4, 1)}


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def ignore_segment(plan, how, nx, ny, z_lo, z_hi, b, kind, absorb, small=False):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    rng = np.random.default_rng(nx + 3 * ny + b)
    cplx = lambda *s: torch.from_numpy((rng.normal(size=s) + 1j * rng.normal(size=s)).astype(np.complex64)).cuda()
    d = rng.uniform(0, 2. if kind == "far" else .05, (z_hi + 1, ny, nx))
    dn = torch.from_numpy((d - .1j * d).astype(np.complex64) if kind == "c64" else d.astype(np.float32)).cuda()
    k = _lib.DN_C64 if kind == "c64" else _lib.DN_F32
    g, useg = cplx(b, ny, nx), cplx(b, z_hi - z_lo + 1, ny, nx)
    grad = dn * 0 + .5
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64)
    _lib.call("bpmh_plan_set_loop", plan, how)
    need = ctypes.c_longlong()
    _lib.call("bpmh_adjoint_segment_work", plan, b, z_lo, z_hi, k, ctypes.byref(need))
    one = b * ny * nx * (2 if kind == "c64" else 1)
    assert need.value in (one, one * (z_hi - z_lo)) and (how != LAUNCHES or need.value == one)
    work = torch.empty(one if small else need.value, dtype=torch.float32, device="cuda")
    _lib.call("bpmh_adjoint_segment_ws", plan, b, z_lo, z_hi, _lib.ptr(g), _lib.ptr(useg), useg.numel(),
              _lib.ptr(dn), k, dn.numel(), _lib.ptr(H), 1.26, absorb, _lib.ptr(grad), _lib.ptr(work),
              work.numel(), _lib.stream_handle())
    torch.cuda.synchronize()
    return g, grad


def mean_segment(plan, how, nx, ny, z_lo, z_hi, b, mode, absorb, far):
    import torch
    from bpm_amd import _lib
    rng = np.random.default_rng(nx + 3 * ny + b)
    cplx = lambda *s: torch.from_numpy((rng.normal(size=s) + 1j * rng.normal(size=s)).astype(np.complex64)).cuda()
    f = lambda lo, hi, *s: torch.from_numpy(rng.uniform(lo, hi, s).astype(np.float32)).cuda()
    dn = f(0, 2. if far else .05, z_hi + 1, ny, nx)
    p, g = cplx(b, ny, nx), cplx(b, ny, nx)
    dn0 = f(0, .05, z_hi + 1)
    ne = dn0 + N0
    grad = torch.full_like(dn, .5)
    simple = mode == 1
    _lib.call("bpmh_plan_set_loop", plan, how)
    out = [g, grad]
    for adjoint in (0, 1):
        q = p.clone()
        need = ctypes.c_longlong()
        _lib.call("bpmh_mean_segment_work", plan, b, z_lo, z_hi, adjoint, ctypes.byref(need))
        work = torch.empty(need.value, dtype=torch.float32, device="cuda")
        _lib.call("bpmh_mean_segment", plan, mode, b, z_lo, z_hi, _lib.ptr(q), _lib.ptr(dn), dn.numel(),
                  _lib.ptr(ne) if simple else None, _lib.ptr(dn0) if simple else None, N0, 12.566, *UNITS, 1.26,
                  absorb, _lib.ptr(g) if adjoint else None, _lib.ptr(grad) if adjoint else None,
                  _lib.ptr(work), work.numel(), _lib.stream_handle())
        torch.cuda.synchronize()
        out.append(q)
    return out


@pytest.mark.parametrize("sched", sorted(SCHED))
@pytest.mark.parametrize("nx,ny", [(64, 64), (64, 512), (512, 64), (256, 128), (512, 512)])
def test_adjoint_loop_equals_launches(nx, ny, sched):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    plan = B.Plan(nx, ny)
    try:
        _lib.call("bpmh_plan_set_variant", plan, *SCHED[sched])
        for z_lo, z_hi, b, kind, absorb in ((0, 1, 1, "f32", 0), (2, 6, 9, "f32", 4), (0, 66, 2, "f32", 0),
                                            (1, 4, 3, "c64", 0), (0, 3, 2, "far", 3)):
            say("case adjoint loop", nx, ny, sched, z_lo, z_hi, b, kind)
            ref = ignore_segment(plan, LAUNCHES, nx, ny, z_lo, z_hi, b, kind, absorb)
            for how, small in ((LOOP, False), (PART, False), (LOOP, True)):
                got = ignore_segment(plan, how, nx, ny, z_lo, z_hi, b, kind, absorb, small)
                assert all(torch.equal(x, y) for x, y in zip(got, ref)), (how, small)
        for z_lo, z_hi, b, mode, absorb, far in ((0, 1, 1, 2, 0, False), (2, 6, 9, 2, 4, False),
                                                 (0, 66, 2, 2, 0, False), (1, 5, 9, 1, 3, False),
                                                 (0, 3, 2, 2, 0, True), (0, 3, 2, 1, 0, True)):
            say("case mean adjoint loop", nx, ny, sched, z_lo, z_hi, b, mode)
            ref = mean_segment(plan, LAUNCHES, nx, ny, z_lo, z_hi, b, mode, absorb, far)
            for how in (LOOP, PART):
                got = mean_segment(plan, how, nx, ny, z_lo, z_hi, b, mode, absorb, far)
                assert all(torch.equal(x, y) for x, y in zip(got, ref)), how
    finally:
        plan.close()
