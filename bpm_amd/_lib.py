"""ctypes binding of libbpmhip.so and the device-memory plumbing around it.

The library is loaded from this package directory (built in-tree by
``python -m bpm_amd.build``).  There is no fallback: if the library is
missing, or no ROCm GPU is visible, every compute call raises.
Error codes of the C ABI map onto the exception types the reference raises
(ValueError, NotImplementedError) or RuntimeError/MemoryError.
"""
import ctypes
import os

import numpy as np

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libbpmhip.so")

OK, ERR_INVALID, ERR_UNSUPPORTED, ERR_HIP, ERR_NOMEM = 0, -1, -2, -3, -4
DN_NONE, DN_F32, DN_F16, DN_C64 = 0, 1, 2, 3
MEAN_IGNORE, MEAN_SIMPLE, MEAN_WEIGHTED = 0, 1, 2
H_F32, H_F64 = 0, 1
DW_INDEX, DW_SIN, DW_GAUSS = 0, 1, 2

_P = ctypes.c_void_p
_I = ctypes.c_int
_F = ctypes.c_float
_D = ctypes.c_double
_LL = ctypes.c_longlong

# name -> (restype, argtypes); every symbol declared in include/bpm_hip.h
SIGNATURES = {
    "bpmh_version": (_I, []),
    "bpmh_last_error": (ctypes.c_char_p, []),
    "bpmh_plan_create": (_I, [_I, _I, ctypes.POINTER(_P)]),
    "bpmh_plan_destroy": (_I, [_P]),
    "bpmh_plan_set_timing": (_I, [_P, _I]),
    "bpmh_plan_kernel_times": (_I, [_P, _P, _P]),
    "bpmh_plan_set_graph": (_I, [_P, _I]),
    "bpmh_plan_set_loop": (_I, [_P, _I]),
    "bpmh_plan_loop_calls": (_I, [_P, _P]),
    "bpmh_loop_check": (_I, []),
    "bpmh_plan_set_variant": (_I, [_P, _I, _I]),
    "bpmh_plan_get_variant": (_I, [_P, _P, _P, _P, _P, _P, _P]),
    "bpmh_propagator_table": (_I, [_I, _I, _I, _D, _D, _D, _D, _D, _P, _P]),
    "bpmh_propagate": (_I, [_P, _I, _I, _P, _P, _I, _LL, _LL, _I, _P, _P, _P, _F, _F, _F, _F,
                            _F, _F, _I, _P, _P, _LL, _P, _P, _P, _P, _P, _P]),
    "bpmh_propagate_noalloc": (_I, [_P, _I, _I, _P, _P, _I, _LL, _LL, _I, _P, _P, _P, _F, _F,
                                    _F, _F, _F, _F, _I, _P, _P, _LL, _P, _P, _P, _P, _P, _P]),
    "bpmh_propagate_groups": (_I, [_P, _I, _P, _P, _P, _P, _I, _LL, _LL, _P, _F, _I, _P, _P,
                                   _P]),
    "bpmh_adjoint_segment": (_I, [_P, _I, _I, _I, _P, _P, _LL, _P, _I, _LL, _P, _F, _I, _P, _P,
                                  _P]),
    "bpmh_adjoint_segment_work": (_I, [_P, _I, _I, _I, _I, _P]),
    "bpmh_adjoint_segment_ws": (_I, [_P, _I, _I, _I, _P, _P, _LL, _P, _I, _LL, _P, _F, _I, _P, _P,
                                     _LL, _P]),
    "bpmh_mean_segment": (_I, [_P, _I, _I, _I, _I, _P, _P, _LL, _P, _P, _F, _F, _F, _F, _F, _F,
                               _I, _P, _P, _P, _LL, _P]),
    "bpmh_mean_segment_work": (_I, [_P, _I, _I, _I, _I, _P]),
    "bpmh_floor_steps": (_I, [_P, _I, _I, _P, _P, _LL, _P]),
    "bpmh_debye_wolf": (_I, [_I, _I, _I, _F, _F, _F, _F, _F, _F, _F, _P, _I, _I, _F, _F, _I,
                             _F, _I, _P, _P, _P, _P, _P]),
    "bpmh_debye_wolf_points": (_I, [_I, _P, _P, _P, _F, _P, _I, _I, _F, _F, _I, _F, _I, _P,
                                    _P, _P, _P, _P]),
    "bpmh_debye_mirror": (_I, [_I, _I, _I, _P, _P, _P, _P, _P, _P, _P, _P, _P]),
    "bpmh_focus_field_debye": (_I, [_I, _I, _I, _D, _D, _D, _F, _P, _I, _I, _P, _P, _P, _P, _P]),
    "bpmh_debye_set_timing": (_I, [_I]),
    "bpmh_debye_kernel_times": (_I, [_P, _P]),
    "bpmh_bessel_fill": (_I, [_I, _P, _P, _I, _P]),
    "bpmh_cylindrical": (_I, [_I, _I, _F, _F, _F, _F, _F, _F, _I, _I, _P, _P, _P, _P, _P]),
    "bpmh_fill_dn_coated": (_I, [_I, _I, _I, _F, _F, _F, _P, _I, _F, _F, _F, _F, _P, _P]),
    "bpmh_spheres_dn": (_I, [_I, _I, _I, _D, _D, _D, _P, _I, _P, _P]),
    "bpmh_bessel_host": (_I, [_I, _P, _P, _I]),
}

_lib = None


def load():
    """Load libbpmhip.so (once) and declare its signatures; raises if absent."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError("libbpmhip.so not found at %s: build it with "
                              "`python -m bpm_amd.build`" % LIB_PATH)
        lib = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _lib = lib
    return _lib


def check(rc):
    """Raise the Python exception that corresponds to a C-ABI return code."""
    if rc == OK:
        return
    msg = load().bpmh_last_error().decode(errors="replace")
    if rc == ERR_INVALID:
        raise ValueError(msg)
    if rc == ERR_UNSUPPORTED:
        raise NotImplementedError(msg)
    if rc == ERR_NOMEM:
        raise MemoryError(msg)
    raise RuntimeError("libbpmhip error %d: %s" % (rc, msg))


def call(name, *args):
    check(getattr(load(), name)(*args))


# ----------------------------------------------------------------------------
# device memory (torch is only the allocator / stream provider)
# ----------------------------------------------------------------------------
_torch = None


def torch():
    global _torch
    if _torch is None:
        import torch as t
        if not t.cuda.is_available():
            raise RuntimeError("bpm_amd needs a ROCm GPU: torch.cuda.is_available() is False")
        load()
        _torch = t
    return _torch


def device():
    return torch().device("cuda", torch().cuda.current_device())


def stream_handle():
    return ctypes.c_void_p(torch().cuda.current_stream().cuda_stream)


_TDT = {np.dtype(np.float32): "float32", np.dtype(np.float16): "float16",
        np.dtype(np.complex64): "complex64"}


def to_device(x, np_dtype, wait=True):
    """numpy array or torch tensor -> contiguous torch tensor on the GPU with dtype np_dtype.
    wait False: for a tensor that the current stream alone uses (a large array's
    copy may still be under way there)."""
    t = torch()
    tdt = getattr(t, _TDT[np.dtype(np_dtype)])
    if isinstance(x, t.Tensor):
        return x.to(device=device(), dtype=tdt).contiguous()
    a = np.ascontiguousarray(np.asarray(x).astype(np_dtype, copy=False))
    if not a.flags.writeable:  # torch.from_numpy wants a writable array
        a = a.copy()
    return _upload(t.from_numpy(a), wait)


def _upload(src, wait):
    """A contiguous host tensor on the GPU, staged as in to_numpy.  With wait the
    copy is complete when this returns, as the unstaged one is: the tensor may
    next be used on any stream."""
    t = torch()
    dev = device()
    n = src.numel()
    half = None if n * src.element_size() <= _STAGE_UP or src.is_pinned() else _halves(n, src.dtype)
    if half is None:
        return src.to(dev)
    out = t.empty(src.shape, dtype=src.dtype, device=dev)
    flat, dst = src.reshape(-1), out.reshape(-1)
    with t.cuda.device(out.device):
        per = half[0].numel()
        stream = t.cuda.current_stream()
        done = [None, None]
        for i in range((n + per - 1) // per):
            part = flat[i * per:(i + 1) * per]
            if done[i & 1] is not None:
                done[i & 1].synchronize()
            half[i & 1][:part.numel()].copy_(part)
            dst[i * per:(i + 1) * per].copy_(half[i & 1][:part.numel()], non_blocking=True)
            done[i & 1] = t.cuda.Event()
            done[i & 1].record(stream)
        if wait:
            done[i & 1].synchronize()
    return out


def empty(shape, np_dtype):
    t = torch()
    return t.empty(tuple(shape), dtype=getattr(t, _TDT[np.dtype(np_dtype)]), device=device())


def ptr(x):
    """Device pointer of a tensor (or None -> NULL)."""
    if x is None:
        return None
    return ctypes.c_void_p(x.data_ptr())


def is_tensor(x):
    try:
        import torch as t
    except ImportError:
        return False
    return isinstance(x, t.Tensor)


# Bytes of each half of the pinned staging memory of a copy between host arrays
# and the GPU.  A copy that HIP stages itself moves 4 GB/s to the host (53 MB:
# 12.2 ms); through pinned halves, one filled by the copy engine while all host
# threads empty the other into a fresh numpy array (whose large pages numpy asks
# for), it moves 46 GB/s (1.1 ms; halves of 1 MiB 4.4, 4 MiB 2.3).  Uploads:
# 1.8 against 1.1 ms.  Below _STAGE_DOWN and _STAGE_UP staging costs more than it
# gives (256 KB down: 44 against 25 us; 2 MB up: 86 against 86).  The memory is
# torch's pinned pool's: taken for the call and given back.
_STAGE = 8 << 20
_STAGE_DOWN, _STAGE_UP = 512 << 10, 2 << 20


def _halves(n, dtype):
    """Pinned staging for n elements: one buffer if they fit, else two halves;
    None where the host has no memory to pin (the copy is then HIP's own)."""
    t = torch()
    per = max(1, _STAGE // t.empty(0, dtype=dtype).element_size())
    try:
        return [t.empty(min(n, per), dtype=dtype, pin_memory=True) for _ in range(1 if n <= per else 2)]
    except RuntimeError:
        return None


def to_numpy(x):
    """The tensor as a numpy array; a GPU tensor is copied once what its stream
    holds has run (an error if a z-loop before it gave up)."""
    out = _to_numpy(x)
    if x.is_cuda:
        call("bpmh_loop_check")
    return out


def _to_numpy(x):
    n = x.numel()
    if (not x.is_cuda or n * x.element_size() <= _STAGE_DOWN or not x.is_contiguous() or
            x.requires_grad or x.is_conj()):
        return x.cpu().numpy()
    t = torch()
    src = x.reshape(-1)
    with t.cuda.device(x.device):
        half = _halves(n, x.dtype)
        if half is None:
            return x.cpu().numpy()
        per = half[0].numel()
        stream = t.cuda.current_stream()
        out = np.empty(tuple(x.shape), half[0].numpy().dtype)
        dst = t.from_numpy(out.reshape(-1))
        done = [t.cuda.Event(), t.cuda.Event()]

        def fetch(i):
            part = src[i * per:(i + 1) * per]
            half[i & 1][:part.numel()].copy_(part, non_blocking=True)
            done[i & 1].record(stream)

        parts = (n + per - 1) // per
        fetch(0)
        for i in range(parts):
            if i + 1 < parts:
                fetch(i + 1)
            done[i & 1].synchronize()
            part = dst[i * per:(i + 1) * per]
            part.copy_(half[i & 1][:part.numel()])
    return out
