"""A gradient whose one-launch workspace does not fit the GPU runs with the least
one: the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["ignore", "weighted", "simple"])
def test_gradient_with_the_least_workspace(mode, monkeypatch):
    import torch
    from bpm_amd import adjoint
    rng = np.random.default_rng(8)
    dn = torch.from_numpy(rng.uniform(0, .05, (9, 64, 128)).astype(np.float32)).cuda().requires_grad_(True)
    u0 = torch.from_numpy(np.exp(1j * rng.uniform(0, 3, (2, 64, 128))).astype(np.complex64)).cuda()

    def gradient():
        u = adjoint.propagate(dn, u0, n0=1.33, checkpoint=4, mean_mode=mode)
        return torch.autograd.grad(u.abs().square()[:, ::3].sum(), [dn])[0]

    ref = gradient()
    empty, sizes = adjoint._empty, []

    def little(shape, *dtype):
        # (workspaces are flat, a segment's forward planes are not)
        sizes.append(shape if isinstance(shape, int) else None)
        if len(sizes) == fails:
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(shape, *dtype)

    monkeypatch.setattr(adjoint, "_empty", little)
    # the workspace, the first or the second segment's forward planes do not fit;
    # a mean's forward takes a workspace before
    for fails in ((1, 2, 3) if mode == "ignore" else (2,)):
        sizes.clear()
        assert torch.equal(gradient(), ref)
        flat = [n for n in sizes if n]
        assert len(flat) == (2 if mode == "ignore" else 3) and flat[-1] < max(flat)
