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

    def little(n):
        sizes.append(n)
        # the first allocation of the backward pass, or what it needs beside it, does not fit
        if len(sizes) == fails:
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(n)

    monkeypatch.setattr(adjoint, "_empty", little)
    for fails in ((1, 2) if mode == "ignore" else (2,)):  # (a mean's forward takes one before)
        sizes.clear()
        assert torch.equal(gradient(), ref)
        assert len(sizes) >= fails + 1 and sizes[-1] < max(sizes)
