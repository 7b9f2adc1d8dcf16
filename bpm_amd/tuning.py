"""Autotuner for the launch shapes and radix schedules of the split-step passes.

For a grid (Nx, Ny) and batch size it times every (row, column) variant of
``bpmh_plan_set_variant`` -- work-group shapes, paired or split column
accesses, and for each pass both radix schedules (4 or 8 elements per
thread, e.g. a 1024-point line as 4.4.4.4.4 or 2.8.8.8) -- on the device
(HIP events on the current stream around a short propagation) and keeps the
fastest.  Grids that run their z-loop as one launch (bpmh_plan_set_loop) have
one time per schedule there; the schedule with the fastest loop is kept, with
the launch shapes that are its fastest as launches per pass (which timed,
captured and adjoint passes still use).  Launch shapes do not change a result's
bits, schedules do: one whose error against float64 is not smaller than that of
the one it would replace (``schedule_errors``) is not taken, however fast.
Results are cached in ``tuning_cache.json`` next to the library, keyed by
"gfx:NxxNy:batch"; ``get_plan`` applies a cached choice automatically.
"""
import ctypes
import json
import os

import numpy as np

from . import _lib

CACHE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuning_cache.json")
_cache = None


def _key(nx, ny, batch):
    return "gfx950:%dx%d:%d" % (nx, ny, batch)


def load_cache():
    global _cache
    if _cache is None:
        _cache = {}
        if os.path.exists(CACHE):
            with open(CACHE) as f:
                _cache = json.load(f)
    return _cache


def lookup(nx, ny, batch=1):
    """Cached (row_variant, col_variant) for this grid and batch, else for
    the nearest cached batch of the same grid, else None.  Read from the cache
    at each call (4 us at most): a re-tuned or replaced entry counts at once."""
    c = load_cache()
    entry = c.get(_key(nx, ny, batch))
    if entry is None:
        grid = ":%dx%d:" % (nx, ny)
        same = [(abs(int(k.rpartition(":")[2]) - batch), k) for k in c if grid in k]
        if not same:
            return None
        entry = c[min(same)[1]]
    return tuple(entry["best"])


ROW_VARIANTS, COL_VARIANTS = 6, 10  # V + 3*s, V + 5*s (s: radix schedule)


def shape_of(plan):
    """(row variant, column variant, lines per row work-group, columns per
    column tile, row elements per thread, column elements per thread)."""
    v = [ctypes.c_int() for _ in range(6)]
    _lib.call("bpmh_plan_get_variant", plan, *[ctypes.byref(x) for x in v])
    return tuple(x.value for x in v)


def schedule_errors(plan, nx, ny, variants, nz=65, volumes=8, waves=3, units=(.1, .1, .1), lam=.5,
                    n0=1.33):
    """Errors of the radix schedules of ``variants`` on this grid: for each, the
    relative L2 distance of the last fields and of the summed intensities from
    complex128, the mean over ``volumes`` sphere volumes under ``waves`` plane
    waves tilted by up to .2 rad.  (The rounding of a schedule's twiddles is the
    same at every step, so its bias grows with the steps: 74 steps of 512^2 are
    off by 4.6e-6 with 4.4 points per thread, 5.0e-6 with 4.8, 5.7e-6 with 8.8,
    their sums by 3.6e-6, 4.0e-6, 5.0e-6.  Columns of 128 points are the one
    length where 4 and 8 points are alike.)"""
    from . import bpm3d as B
    from .spheres import spheres_dn_device
    from .workloads import plane_waves, small_workload_spheres
    t = _lib.torch()
    dev = _lib.device()
    k0 = 2. * np.pi / lam
    kx, ky = (2. * np.pi * np.fft.fftfreq(n, d) for n, d in ((nx, units[0]), (ny, units[1])))
    k2 = (n0 * k0) ** 2 - (kx * kx)[None, :] - (ky * ky)[:, None]
    H64 = t.from_numpy(np.where(k2 >= 0, np.exp(-1j * units[2] * np.sqrt(np.maximum(k2, 0))), 0)).to(dev)
    H = B.propagator_table(nx, ny, units, lam, n0, _lib.H_F64)
    acc = t.empty((waves, ny, nx), dtype=t.float32, device=dev)
    off = lambda x, ref: float((x.to(ref.dtype) - ref).norm() / ref.norm())  # noqa: E731
    errs = {v: [] for v in variants}
    for seed in range(volumes):
        rng = np.random.default_rng(seed)
        dn = spheres_dn_device((nx, ny, nz), units, *small_workload_spheres(rng, (nx, ny, nz), units))
        u0 = t.from_numpy(plane_waves(nx, ny, units[0], units[1], lam, n0,
                                      rng.uniform(-.2, .2, (waves, 2)))).to(dev)
        u = u0.to(t.complex128)
        sums = u.abs().square()
        for z in range(1, nz):
            u = t.fft.ifft2(t.fft.fft2(u) * H64) * t.exp(-1j * k0 * units[2] * dn[z].double())
            sums += u.abs().square()
        for v in variants:
            _lib.call("bpmh_plan_set_variant", plan, *v)
            p = u0.clone()
            B.propagate_fields(p, nz, units, lam, n0, dn=dn, dn_kind=_lib.DN_F32, mean_mode="ignore",
                               H=H, out_sum=acc, tuned=False, plan=plan)
            errs[v].append((off(p, u), off(acc, sums)))
    return {v: tuple(float(x) for x in np.mean(e, axis=0)) for v, e in errs.items()}


def autotune(nx, ny, batch=1, nz=65, reps=3, units=(.1, .1, .1), lam=.5, n0=1.33, save=None):
    """Time all 6x10 (row, column) variants for one grid/batch (variants that
    map to an identical kernel pair are timed once) and each schedule as the
    plan runs it, and keep the fastest of the schedule in use (that of the cached
    entry of this grid and batch, else the default) and those more accurate; returns (best, table), the table of the kept
    schedule's launch shapes."""
    from . import bpm3d as B
    t = _lib.torch()
    plan = B.Plan(nx, ny)
    rng = np.random.default_rng(0)
    dn = t.from_numpy(rng.uniform(0, .05, (nz, ny, nx)).astype(np.float32)).to(_lib.device())
    u0 = t.ones((batch, ny, nx), dtype=t.complex64, device=_lib.device())
    H = B.propagator_table(nx, ny, units, lam, n0, _lib.H_F64)
    acc = t.empty((batch, ny, nx), dtype=t.float32, device=_lib.device())
    plane = t.empty_like(u0)

    def run():
        plane.copy_(u0)
        B.propagate_fields(plane, nz, units, lam, n0, dn=dn, dn_kind=_lib.DN_F32,
                           mean_mode="ignore", H=H, out_sum=acc, tuned=False, plan=plan)

    def time_ms():
        run()
        t.cuda.synchronize()
        e0, e1 = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            run()
        e1.record()
        t.cuda.synchronize()
        return e0.elapsed_time(e1) / reps

    def schedule(v):
        _lib.call("bpmh_plan_set_variant", plan, *v)
        return shape_of(plan)[4:6]

    table = {}
    _lib.call("bpmh_plan_set_loop", plan, 1)
    for rv in range(ROW_VARIANTS):
        for cv in range(COL_VARIANTS):
            _lib.call("bpmh_plan_set_variant", plan, rv, cv)
            shp = shape_of(plan)
            key = [shp[2], shp[3], shp[4], shp[5]]
            if cv % 5 in (3, 4) and 256 <= ny <= 1024:
                key.append(cv % 5)  # paired / split columns: kernels of their own
            if key in [v["shape"] for v in table.values()]:
                continue  # clamped to an identical launch shape
            ms = time_ms()
            table["%d,%d" % (rv, cv)] = {"ms": ms, "shape": key,
                                         "us_per_step": ms * 1e3 / (nz - 1)}
    _lib.call("bpmh_plan_set_loop", plan, 0)
    # the time of each schedule as it runs, at its fastest launch shapes
    runs, tries = {}, {}
    for sched in {tuple(v["shape"][2:4]) for v in table.values()}:
        k = min((k for k in table if tuple(table[k]["shape"][2:4]) == sched), key=lambda k: table[k]["ms"])
        tries[sched] = tuple(int(x) for x in k.split(","))
        _lib.call("bpmh_plan_set_variant", plan, *tries[sched])
        runs[sched] = time_ms()
    del dn, u0, acc, plane
    c = load_cache()
    now = schedule(c[_key(nx, ny, batch)]["best"] if _key(nx, ny, batch) in c else (1, 1))
    errs = schedule_errors(plan, nx, ny, list(tries.values()), units=units, lam=lam, n0=n0)
    errs = {q: errs[v] for q, v in tries.items()}
    # another schedule's errors have to be smaller by more than what the inputs leave open
    sched = min((q for q in runs if q == now or all(e < .97 * f for e, f in zip(errs[q], errs[now]))),
                key=lambda q: runs[q])
    plan.close()
    table = {k: v for k, v in table.items() if tuple(v["shape"][2:4]) == sched}
    best = min(table, key=lambda k: table[k]["ms"])
    bv = tuple(int(x) for x in best.split(","))
    _lib.call("bpmh_plan_set_variant", B.get_plan(nx, ny, None), *bv)
    c[_key(nx, ny, batch)] = {"best": list(bv), "table": table,
                              "us_per_step": {"%d.%d" % q: r * 1e3 / (nz - 1) for q, r in runs.items()},
                              "errors": {"%d.%d" % q: e for q, e in errs.items()}}
    if save:
        with open(save, "w") as f:
            json.dump(c, f, indent=1, sort_keys=True)
    return bv, table


def main(argv=None):
    import argparse
    ap = argparse.ArgumentParser(description="autotune the split-step launch shapes")
    ap.add_argument("--grids", default="1024x1024,512x512,256x256,128x128")
    ap.add_argument("--batches", default="1")
    ap.add_argument("--nz", type=int, default=65)
    ap.add_argument("--out", default=CACHE)
    a = ap.parse_args(argv)
    for g in a.grids.split(","):
        nx, ny = (int(v) for v in g.split("x"))
        for b in (int(v) for v in a.batches.split(",")):
            best, table = autotune(nx, ny, b, nz=a.nz, save=a.out)
            print("%dx%d batch %d best %s %s" % (nx, ny, b, best,
                  {k: round(v["us_per_step"], 2) for k, v in table.items()}), flush=True)


if __name__ == "__main__":
    main()
