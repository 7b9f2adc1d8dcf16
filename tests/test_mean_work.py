"""Workspace of a mean-corrected segment (bpmh_mean_segment_work): the screen
gradients of every step only where its adjoint runs as one launch."""
import ctypes

import pytest

from bpm_amd import _lib

DEFAULT, LAUNCHES, LOOP = 0, 1, 2


def work(nx, ny, variant, how, batch, nseg):
    lib = _lib.load()
    plan, n = ctypes.c_void_p(), ctypes.c_longlong()
    _lib.call("bpmh_plan_create", nx, ny, ctypes.byref(plan))
    try:
        _lib.call("bpmh_plan_set_variant", plan, *variant)
        _lib.call("bpmh_plan_set_loop", plan, how)
        _lib.call("bpmh_mean_segment_work", plan, batch, 0, nseg - 1, 1, ctypes.byref(n))
    finally:
        lib.bpmh_plan_destroy(plan)
    return n.value


@pytest.mark.parametrize("nx,ny,variant,loop", [
    (128, 64, (1, 6), True), (256, 256, (1, 1), True), (512, 512, (4, 1), True), (512, 256, (1, 6), False),
    (512, 512, (1, 6), False), (256, 256, (4, 6), False), (1024, 512, (1, 1), False)])
def test_screen_gradients_of_every_step_only_where_used(nx, ny, variant, loop):
    batch, nseg, n2 = 3, 17, nx * ny
    one = work(nx, ny, variant, LAUNCHES, batch, nseg)
    # planes of the batch: the forward plane, its fields and k-space planes, one
    # screen gradient and the weight slice's
    assert 0 <= one - batch * n2 * (2 + 2 * nseg + 2 * (nseg - 1) + 2) < 64 * batch * (nx + ny + nseg)
    more = batch * n2 * (nseg - 2) if loop else 0
    assert work(nx, ny, variant, LOOP, batch, nseg) == one + more
    assert work(nx, ny, variant, DEFAULT, batch, nseg) == one + more
