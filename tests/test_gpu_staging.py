"""Host arrays to the GPU and back around the sizes where a copy goes through
pinned staging: one part, exactly two, a remainder, several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float16, np.float32, np.complex64])
def test_round_trip(dtype):
    import torch
    from bpm_amd import _lib
    per = _lib._STAGE // np.dtype(dtype).itemsize
    rng = np.random.default_rng(3)
    for n in (0, 1, per // 16, per // 16 + 1, per // 4 + 1, per - 1, per, per + 1, 2 * per, 4 * per + 7):
        a = rng.integers(-99, 99, n).astype(dtype)
        x = _lib.to_device(a, dtype)
        keep = a.copy()
        a[:] = 0  # the source is the caller's again once the call returns
        assert x.shape == (n,) and torch.equal(x.cpu(), torch.from_numpy(keep)), n
        y = _lib.to_numpy(x)
        assert y.dtype == keep.dtype and np.array_equal(y, keep) and y.flags.writeable, n
    x = torch.arange(6 * (1 << 20), dtype=torch.float32, device="cuda").view(6, 1024, 1024)
    for v in (x[1:5], x[2], x[:, :, ::2], x.transpose(0, 1)):
        assert np.array_equal(_lib.to_numpy(v), v.cpu().numpy())


@pytest.mark.parametrize("mib", [3, 8, 9, 40])
def test_upload_is_complete_on_return(mib):
    """Uploaded behind other work of one stream, read on another without a wait
    between the two streams."""
    import torch
    from bpm_amd import _lib
    a = np.random.default_rng(mib).random(mib << 18, dtype=np.float32)
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(one):
        torch.cuda._sleep(20_000_000)
        x = _lib.to_device(a, np.float32)
    with torch.cuda.stream(two):
        y = x.clone()
    two.synchronize()
    assert np.array_equal(y.cpu().numpy(), a)


def test_copies_without_pinned_memory(monkeypatch):
    import torch
    from bpm_amd import _lib
    a = np.random.default_rng(1).random(5 << 20, dtype=np.float32)
    empty = torch.empty

    def none_pinned(*args, pin_memory=False, **kw):
        if pin_memory:
            raise RuntimeError("no memory to pin")
        return empty(*args, **kw)

    monkeypatch.setattr(torch, "empty", none_pinned)
    x = _lib.to_device(a, np.float32)
    assert np.array_equal(_lib.to_numpy(x), a)
