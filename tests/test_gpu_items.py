"""The passes that keep a line over several items of a batch, against the same
items one by one below their size limit (the one-item passes): the same bits,
for every dn kind, mean mode and output, shared and separate volumes, chunks
that do not divide the batch, ragged groups and the adjoint."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM, N0, UNITS = .5, 1.33, (.1, .1, .1)
LAUNCHES = 1
LIMIT = 2 << 20  # points of a call from which the passes of several items run


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def plan_of(nx, ny, sched=(1, 1)):
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    plan = B.Plan(nx, ny)
    _lib.call("bpmh_plan_set_variant", plan, *sched)
    _lib.call("bpmh_plan_set_loop", plan, LAUNCHES)
    return plan


# both radix schedules of rows and columns
@pytest.mark.parametrize("sched", [(1, 1), (4, 6)])
@pytest.mark.parametrize("nx,ny,b", [(512, 512, 9), (1024, 512, 4), (512, 1024, 37), (2048, 512, 3),
                                     (256, 2048, 5), (1024, 256, 9), (512, 64, 65)])
def test_items_equal_single_fields(nx, ny, b, sched):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    assert b * nx * ny >= LIMIT > nx * ny
    plan = plan_of(nx, ny, sched)
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64)
    rng = np.random.default_rng(nx + ny + b)
    nz = 3
    f = lambda *s: torch.from_numpy(rng.uniform(0, 1, s).astype(np.float32)).cuda()
    u0 = torch.polar(torch.ones((b, ny, nx), device="cuda"), f(b, ny, nx))
    try:
        for kind, mode, absorb, own, scat in (
                ("f32", "ignore", 0, False, False), ("f16", "ignore", 7, False, False),
                ("c64", "simple", 5, False, False), ("f32", "simple", 0, False, False),
                ("none", "ignore", 0, False, False), ("f32", "ignore", 3, True, False),
                ("f32", "weighted", 4, False, False), ("f32", "ignore", 0, False, True)):
            if (own or scat) and nx * ny * b > 3 * LIMIT:
                continue
            say("case items", nx, ny, b, kind, mode, absorb, own, scat)
            d = .05 * f(*((b, nz, ny, nx) if own else (nz, ny, nx)))
            dn = {"f32": d, "f16": d.half(), "c64": torch.complex(d, -.1 * d), "none": None}[kind]
            k = {"f32": _lib.DN_F32, "f16": _lib.DN_F16, "c64": _lib.DN_C64, "none": _lib.DN_NONE}[kind]
            dn0 = .05 * f(nz) if mode == "simple" else None
            sw = (f(ny, nx), f(ny, nx), torch.polar(f(nz), f(nz))) if scat else None

            def run(u, dnv, stride):
                n = u.shape[0]
                acc = torch.empty(u.shape, device="cuda")
                vol = torch.empty((n, nz, ny, nx), dtype=torch.complex64, device="cuda")
                out = torch.zeros(n * nz * 2, device="cuda")
                p = u.clone()
                B.propagate_fields(p, nz, UNITS, LAM, N0, dn=dnv, dn_kind=k, mean_mode=mode,
                                   H=H if mode == "ignore" else None,
                                   n_eff=None if dn0 is None else (dn0 + N0).contiguous(), dn0=dn0,
                                   dn_batch_stride=stride, absorbing_width=absorb, out_sum=acc, out_field=vol,
                                   scat=sw + (out,) if scat else None, tuned=False, plan=plan)
                return p, acc, vol, out.view(n, -1)

            got = run(u0, dn, nz * ny * nx if own else 0)
            for i in range(b):
                ref = run(u0[i:i + 1], dn[i] if own else dn, 0)
                for j, (x, y) in enumerate(zip(got, ref)):
                    assert torch.equal(x[i:i + 1], y), (i, j)
    finally:
        plan.close()


@pytest.mark.parametrize("nx,ny", [(512, 1024), (1024, 512)])
def test_groups_and_adjoint_equal_single_fields(nx, ny):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    plan = plan_of(nx, ny)
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64)
    rng = np.random.default_rng(5)
    f = lambda *s: torch.from_numpy(rng.uniform(0, 1, s).astype(np.float32)).cuda()
    groups = [(3, 6), (2, 3)]
    n, nz = 5, 6
    u0 = torch.polar(torch.ones((n, ny, nx), device="cuda"), f(n, ny, nx))
    try:
        say("case items groups", nx, ny)
        dn = .05 * f(2, nz, ny, nx)
        p, acc = u0.clone(), torch.empty((n, ny, nx), device="cuda")
        B.propagate_groups(p, groups, UNITS, LAM, dn, H, nz * ny * nx, out_sum=acc, plan=plan)
        for i in range(n):
            g = int(i >= 3)
            q, s = u0[i:i + 1].clone(), torch.empty((1, ny, nx), device="cuda")
            B.propagate_fields(q, groups[g][1], UNITS, LAM, N0, dn=dn[g], dn_kind=_lib.DN_F32,
                               mean_mode="ignore", H=H, out_sum=s, tuned=False, plan=plan)
            assert torch.equal(p[i:i + 1], q) and torch.equal(acc[i:i + 1], s), i
        for kind, absorb in (("f32", 4), ("c64", 0)):
            say("case items adjoint", nx, ny, kind)
            d = .05 * f(nz, ny, nx)
            dnv = torch.complex(d, -.1 * d) if kind == "c64" else d
            k = _lib.DN_C64 if kind == "c64" else _lib.DN_F32
            useg = torch.polar(f(n, 4, ny, nx), f(n, 4, ny, nx))

            def adjoint(g, u, grad):
                w = torch.empty(g.shape[0] * ny * nx * 2, device="cuda")
                _lib.call("bpmh_adjoint_segment", plan, g.shape[0], 1, 4, _lib.ptr(g), _lib.ptr(u),
                          u.numel(), _lib.ptr(dnv), k, dnv.numel(), _lib.ptr(H), 1.26, absorb,
                          _lib.ptr(grad), _lib.ptr(w), _lib.stream_handle())
                return g

            grad, one = dnv * 0, dnv * 0
            got = adjoint(u0.clone(), useg, grad)
            for i in range(n):  # gradients added item by item, as the batch does
                ref = adjoint(u0[i:i + 1].clone(), useg[i:i + 1].contiguous(), one)
                assert torch.equal(got[i:i + 1], ref), i
            assert torch.equal(grad, one)
    finally:
        plan.close()
