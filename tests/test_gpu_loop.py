"""The one-launch z-loop (bpmh_plan_set_loop) against the launches per pass:
the same operations on every line, so the same bits, on every mean mode, dn
kind and output, with complete and incomplete teams, ragged groups, several
streams and a captured stream (which keeps the launches)."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAM, N0, UNITS = .5, 1.33, (.1, .1, .1)
LAUNCHES, LOOP, PART = 1, 2, 3


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def inputs(nx, ny, nz, b, kind, seed=0):
    import torch
    rng = np.random.default_rng(seed)
    d = rng.uniform(0, .05, (nz, ny, nx)) if kind != "far" else rng.uniform(0, 2., (nz, ny, nx))
    dt = {"f16": np.float16, "c64": np.complex64}.get(kind, np.float32)
    dn = torch.from_numpy((d - .1j * d if kind == "c64" else d).astype(dt)).cuda()
    u0 = torch.from_numpy(np.exp(1j * rng.uniform(0, 3, (b, ny, nx))).astype(np.complex64)).cuda()
    return dn, u0, rng


def propagate(plan, how, u0, nz, dn, kind, mode, absorb, extra, rng_seed=1):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    b, ny, nx = u0.shape
    rng = np.random.default_rng(rng_seed)
    _lib.call("bpmh_plan_set_loop", plan, how)
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64) if mode == "ignore" else None
    dn0 = n_eff = None
    if mode == "simple":
        dn0 = torch.from_numpy(rng.uniform(0, .05, nz).astype(np.float32)).cuda()
        n_eff = (dn0 + N0).contiguous()
    f = lambda *s: torch.from_numpy(rng.uniform(0, 1, s).astype(np.float32)).cuda()
    acc = torch.empty(u0.shape, dtype=torch.float32, device="cuda") if extra else None
    vol = torch.empty((b, nz, ny, nx), dtype=torch.complex64, device="cuda") if extra else None
    scat = None
    if extra:
        scat = (f(ny, nx), f(ny, nx), torch.polar(f(nz), f(nz)),
                torch.zeros(b * nz * 2, dtype=torch.float32, device="cuda"))
    p = u0.clone()
    k = {"f16": _lib.DN_F16, "c64": _lib.DN_C64, "none": _lib.DN_NONE}.get(kind, _lib.DN_F32)
    B.propagate_fields(p, nz, UNITS, LAM, N0, dn=None if kind == "none" else dn, dn_kind=k,
                       mean_mode=mode, H=H, n_eff=n_eff, dn0=dn0, absorbing_width=absorb,
                       out_sum=acc, out_field=vol, scat=scat, tuned=False, plan=plan)
    torch.cuda.synchronize()
    return [x for x in (p, acc, vol, scat[3] if scat else None) if x is not None]


# points per thread of rows and columns: variants of the schedules built
SCHED = {"4.4": (1, 6), "4.8": (1, 1), "8.8": (4, 1)}


@pytest.mark.parametrize("sched", sorted(SCHED))
@pytest.mark.parametrize("nx,ny", [(64, 64), (64, 512), (512, 64), (256, 128), (512, 512)])
def test_loop_equals_launches(nx, ny, sched):
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    plan = B.Plan(nx, ny)
    try:
        _lib.call("bpmh_plan_set_variant", plan, *SCHED[sched])
        for nz, b, kind, mode, absorb, extra in (
                (2, 1, "f32", "ignore", 0, False), (67, 2, "f32", "ignore", 5, True),
                (6, 19, "f16", "ignore", 3, True), (5, 9, "c64", "simple", 0, False),
                (67, 1, "f32", "weighted", 4, True), (4, 9, "far", "weighted", 0, False),
                (4, 3, "far", "ignore", 3, False), (7, 2, "none", "ignore", 0, True)):
            say("case loop", nx, ny, sched, nz, b, kind, mode)
            dn, u0, _ = inputs(nx, ny, nz, b, kind)
            ref = propagate(plan, LAUNCHES, u0, nz, dn, kind, mode, absorb, extra)
            for how in (LOOP, PART):
                got = propagate(plan, how, u0, nz, dn, kind, mode, absorb, extra)
                for i, (x, y) in enumerate(zip(got, ref)):
                    assert torch.equal(x, y), (how, i)
    finally:
        plan.close()


def test_ragged_groups():
    """Groups with and without completion events (one loop for all, or one per
    group, shallowest first), a group of depth 1 among them."""
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    nx, ny = 128, 64
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64)
    for groups in ([(3, 70), (9, 12), (2, 12)], [(2, 9), (5, 1)]):
        say("case loop groups", groups)
        nzmax, tot = groups[0][1], sum(g[0] for g in groups)
        dn, _, rng = inputs(nx, ny, nzmax * len(groups), 1, "f32", seed=3)
        u0 = torch.from_numpy(np.exp(1j * rng.uniform(0, 3, (tot, ny, nx))).astype(np.complex64)).cuda()
        plan = B.Plan(nx, ny)
        try:
            out = {}
            for how, events in ((LAUNCHES, False), (LOOP, False), (LOOP, True), (PART, True)):
                _lib.call("bpmh_plan_set_loop", plan, how)
                p, acc = u0.clone(), torch.empty((tot, ny, nx), device="cuda")
                evs = [torch.cuda.Event() for _ in groups] if events else None
                B.propagate_groups(p, groups, UNITS, LAM, dn, H, nzmax * ny * nx, out_sum=acc,
                                   plan=plan, done_events=evs)
                torch.cuda.synchronize()
                assert evs is None or all(e.query() for e in evs)
                out[how, events] = (p, acc)
            for k, v in out.items():
                assert all(torch.equal(a, b) for a, b in zip(v, out[LAUNCHES, False])), k
        finally:
            plan.close()


def test_streams_share_a_plan_and_capture_keeps_the_launches():
    """Calls of one plan on two streams at once (each takes its own
    synchronisation buffer), and a call recorded into a graph and replayed
    with other work between the replays."""
    import torch
    from bpm_amd import _lib
    from bpm_amd import bpm3d as B
    nx, ny, nz, b = 128, 128, 40, 5
    say("case loop streams and capture")
    dn, u0, rng = inputs(nx, ny, nz, b, "f32", seed=5)
    H = B.propagator_table(nx, ny, UNITS, LAM, N0, _lib.H_F64)
    plan = B.Plan(nx, ny)

    def call(p):
        B.propagate_fields(p, nz, UNITS, LAM, N0, dn=dn, dn_kind=_lib.DN_F32, mean_mode="ignore",
                           H=H, tuned=False, plan=plan)

    try:
        _lib.call("bpmh_plan_set_loop", plan, LAUNCHES)
        ref = u0.clone()
        call(ref)
        torch.cuda.synchronize()
        _lib.call("bpmh_plan_set_loop", plan, LOOP)
        streams = [torch.cuda.Stream() for _ in range(3)]
        planes = [u0.clone() for _ in range(9)]
        torch.cuda.synchronize()
        for i, p in enumerate(planes):
            with torch.cuda.stream(streams[i % 3]):
                call(p)
        torch.cuda.synchronize()
        assert all(torch.equal(p, ref) for p in planes)
        g = torch.cuda.CUDAGraph()
        p = u0.clone()
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            call(p)
        for _ in range(4):
            p.copy_(u0)
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(p, ref)
            q = u0.clone()
            call(q)
            torch.cuda.synchronize()
            assert torch.equal(q, ref)
    finally:
        plan.close()
