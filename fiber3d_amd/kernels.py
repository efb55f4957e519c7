"""Drop-in replacements for the reference's Green's-function sums.

The functions named ``*_numba`` keep the names, signatures, argument meaning
and return convention of python/kernels/kernels.py: float64 NumPy arrays of 3N
values (flat or (N,3), AoS) in, a new flat float64 NumPy array out.  They run
on the GPU through libf3d.so; nothing here computes on the CPU.

``pairsum`` is the device-tensor twin used by the GPU-resident pipeline: torch
float64 CUDA tensors in and out, no host round trip.

A module-level precision (``set_precision``) selects FP64 (default, parity
path) or FP32-compensated evaluation for the drop-in names.
"""
import ctypes
import threading

import numpy as np
import torch

from . import _lib as L

_PREC = {"f64": L.F64, "f32c": L.F32C}
_KIND = {"oseen": L.OSEEN, "rotlet": L.ROTLET, "stresslet": L.STRESSLET}
_precision = "f64"
_ws = {}


def set_precision(p):
    """Select 'f64' (default) or 'f32c' for the drop-in functions."""
    global _precision
    if p not in _PREC:
        raise ValueError(f"precision must be one of {sorted(_PREC)}")
    _precision = p


def device():
    if not torch.cuda.is_available():
        raise L.F3DError("fiber3d_amd needs a ROCm GPU (torch.cuda.is_available() is False)")
    return torch.device("cuda")


_tuned = False


def _ensure_tuned():
    """Install the saved launch-shape table (fiber3d_amd/tuning.json) once; other
    threads' first sums wait for it."""
    global _tuned
    if not _tuned:
        with _ws_lock:
            if not _tuned:
                from . import autotune
                try:
                    autotune.apply()
                finally:
                    _tuned = True


# Workspace buffers replaced by a larger one stay allocated for the life of
# the process: a recorded HIP graph keeps the device address it was recorded
# with, and freeing the buffer would hand that memory to other tensors.
_ws_retired = []

# Held from the look-up of a workspace to the end of the call that launches with
# it: a sum is several launches, and those of two threads on one stream must
# not interleave.
_ws_lock = threading.RLock()


def workspace(nbytes, tag="default", at=None):
    """The device byte buffer (at least nbytes) of the current stream (`at`, where
    the caller has it): sums queued on different streams are not ordered, so
    each stream has its own, and recorded work another than the stream's eager
    work (graphs that share one: those recorded on one stream; replay them in
    order).  Grown by >= 1.5x on demand; a replaced buffer is retired, never
    freed."""
    at = at or _here()
    if at[1] and _capturing():  # (the default stream cannot be recorded)
        tag = ("recorded", tag)
    return _buffer((tag, at), nbytes)


def _buffer(key, nbytes):
    buf = _ws.get(key)
    if buf is None or buf.numel() < nbytes:
        size = max(int(nbytes), 256)
        if buf is not None:
            _ws_retired.append(buf)
            size = max(size, int(1.5 * buf.numel()))
        buf = torch.empty(size, dtype=torch.uint8, device=device())
        _ws[key] = buf
    return buf


_recording = {}


def recording_stream():
    """The stream on which HIP graphs are recorded, one per device.  Its recorded
    work has a workspace as large as the current stream's, so that recording
    what has run here allocates none."""
    dev = torch.cuda.current_device()
    with _ws_lock:
        if dev not in _recording:
            _recording[dev] = torch.cuda.Stream()
        side = _recording[dev]
        mine = _ws.get(("default", _here()))
        key = (("recorded", "default"), (dev, side.cuda_stream))
        if mine is not None and (key not in _ws or _ws[key].numel() < mine.numel()):
            with torch.cuda.stream(side):
                _buffer(key, mine.numel())
    return side


_capturing = getattr(torch._C, "_cuda_isCurrentStreamCapturing",
                     torch.cuda.is_current_stream_capturing)


# the current device and stream without their Python wrappers (0.1 us instead of
# 3, of the 14 us of host work that bounded a small sum)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_device_index = getattr(torch._C, "_cuda_getDevice", None)


def _here():
    """(device index, raw handle) of the current stream."""
    if _raw_stream is None or _device_index is None:
        return torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream
    dev = _device_index()
    return dev, _raw_stream(dev)


def _stream():
    return ctypes.c_void_p(_here()[1])


def ctypes_stream(s):
    return ctypes.c_void_p(s.cuda_stream)


def _strides3(t):
    """(sp, sc) of an (N,3)-shaped float64 tensor."""
    shape = t.shape
    if len(shape) != 2 or shape[1] != 3:
        raise ValueError(f"expected an (N,3) tensor, got shape {tuple(shape)}")
    if t.dtype != torch.float64:
        raise TypeError("expected float64")
    return t.stride()


def _addr(t):
    return None if t is None else t.data_ptr()


def _as_common(ts):
    """Make a list of (N,3) tensors (None allowed) share one (sp, sc) and device."""
    ref = next(t for t in ts if t is not None)
    st, dev = _strides3(ref), ref.get_device()
    out = []
    for t in ts:
        if t is None:
            out.append(None)
        elif _strides3(t) != st or t.get_device() != dev:
            out.append(torch.empty_strided(ref.shape, ref.stride(), dtype=ref.dtype,
                                           device=ref.device).copy_(t))
        else:
            out.append(t)
    return out, st


def pairsum(kernel, src_pos, src_den, trg_pos, src_nrm=None, src_w=None, excl=None,
            eta=1.0, reg=5e-3, eps=1e-5, precision="f64", out=None, accumulate=False,
            clamp_near=False, exclude_self=False):
    """Device pair sum (libf3d f3d_pairsum) on torch CUDA tensors.

    kernel: 'oseen' | 'rotlet' | 'stresslet'.  src_pos, src_den, src_nrm,
    trg_pos, out: (N,3) float64 CUDA tensors with any strides (an SoA buffer
    (3,N) is passed as its transpose).  src_w: (Ns,) float64 weights.
    excl: (lo, hi) int32 (Nt,) tensors of excluded source ranges.
    exclude_self: drop the pair (source i, target i) (self-sums, j != i).
    Returns out (allocated AoS if None).
    """
    k = _KIND[kernel]
    lib = L.load()
    _ensure_tuned()
    nt = trg_pos.shape[0]
    ns = src_pos.shape[0]
    dev = src_pos.get_device()
    if (src_den.shape != src_pos.shape or src_den.get_device() != dev
            or (src_nrm is not None and (src_nrm.shape != src_pos.shape
                                         or src_nrm.get_device() != dev))):
        (src_pos, src_den, src_nrm), _ = _as_common([src_pos, src_den, src_nrm])
    s_sp, s_sc = _strides3(src_pos)
    d_sp, d_sc = _strides3(src_den)
    n_sp, n_sc = (0, 0) if src_nrm is None else _strides3(src_nrm)
    t_sp, t_sc = _strides3(trg_pos)
    if out is None:
        out = torch.empty((nt, 3), dtype=torch.float64, device=trg_pos.device)
    o_sp, o_sc = _strides3(out)
    lo = hi = None
    if excl is not None:
        lo, hi = excl
        assert lo.dtype == torch.int32 and hi.dtype == torch.int32 and lo.numel() == nt
    if src_w is not None:
        assert src_w.dtype == torch.float64 and src_w.numel() == ns and src_w.is_contiguous()
    prec = _PREC[precision]
    need = lib.f3d_pairsum_workspace_size(k, prec, ns, nt)
    flags = ((L.ACCUMULATE if accumulate else 0) | (L.CLAMP_NEAR if clamp_near else 0)
             | (L.EXCLUDE_SELF if exclude_self else 0))
    at = _here()
    with _ws_lock:
        ws = workspace(need, at=at)
        rc = lib.f3d_pairsum_strided(
            k, prec, flags, ns, src_pos.data_ptr(), s_sp, s_sc, _addr(src_nrm), n_sp, n_sc,
            src_den.data_ptr(), d_sp, d_sc, _addr(src_w), nt, trg_pos.data_ptr(), t_sp, t_sc,
            _addr(lo), _addr(hi), float(eta), float(reg), float(eps), out.data_ptr(), o_sp, o_sc,
            ws.data_ptr(), ws.numel(), at[1])
    L.check(rc, "f3d_pairsum")
    return out


def periphery_apply(pos, nrm, w, ex, ey, ez, q, add=None, eta=1.0, reg=5e-3, eps=1e-5,
                    precision="f64", out=None):
    """Matrix-free shell operator (f3d_periphery_apply) on (N,3) CUDA tensors."""
    lib = L.load()
    _ensure_tuned()
    (pos, nrm, ex, ey, ez, q, add), (sp, sc) = _as_common([pos, nrm, ex, ey, ez, q, add])
    n = pos.shape[0]
    if out is None:
        out = torch.empty_strided(pos.shape, pos.stride(), dtype=torch.float64, device=pos.device)
    elif _strides3(out) != (sp, sc):
        raise ValueError("out must share the layout of the inputs")
    prec = _PREC[precision]
    need = lib.f3d_periphery_workspace_size(prec, n)
    at = _here()
    with _ws_lock:
        ws = workspace(need, at=at)
        rc = lib.f3d_periphery_apply(
            prec, n, pos.data_ptr(), _addr(nrm), _addr(w), _addr(ex), _addr(ey), _addr(ez),
            _addr(q), _addr(add), sp, sc, float(eta), float(reg), float(eps), out.data_ptr(),
            ws.data_ptr(), ws.numel(), at[1])
    L.check(rc, "f3d_periphery_apply")
    return out


def kernel_timer(enable=True):
    """Start (clearing earlier records) or stop HIP-event timing of the pair
    kernel inside every later pairsum / periphery_apply call."""
    L.check(L.load().f3d_pairsum_timer(1 if enable else 0), "f3d_pairsum_timer")


def kernel_timer_read():
    """(summed milliseconds, launch count) of the pair-kernel launches timed
    since kernel_timer(True); waits for the last one."""
    ms = ctypes.c_double()
    n = ctypes.c_int32()
    L.check(L.load().f3d_pairsum_timer_read(ctypes.byref(ms), ctypes.byref(n)),
            "f3d_pairsum_timer_read")
    return ms.value, n.value


# ---------------------------------------------------------------------------
# Drop-in names (python/kernels/kernels.py)

def _to_dev(a, n=None):
    a = np.ascontiguousarray(np.asarray(a, dtype=np.float64).reshape(-1, 3))
    if n is not None and a.shape[0] != n:
        raise ValueError(f"expected {n} points, got {a.shape[0]}")
    return torch.from_numpy(a).to(device())


def _np_pairsum(kernel, r_source, r_target, density, normal, eta, reg, eps, self_sum=False):
    s = _to_dev(r_source)
    t = s if self_sum else _to_dev(r_target)
    d = _to_dev(density, s.shape[0])
    nm = _to_dev(normal, s.shape[0]) if normal is not None else None
    u = pairsum(kernel, s, d, t, src_nrm=nm, eta=eta, reg=reg, eps=eps,
                precision=_precision, exclude_self=self_sum)
    return u.cpu().numpy().ravel()


def oseen_kernel_source_target_numba(r_source, r_target, density, eta=1.0, reg=5e-3,
                                     epsilon_distance=1e-5):
    """Drop-in for kernels.oseen_kernel_source_target_numba (kernels/kernels.py:794-846)."""
    return _np_pairsum("oseen", r_source, r_target, density, None, eta, reg, epsilon_distance)


def rotlet_kernel_source_target_numba(r_source, r_target, density, eta=1.0, reg=5e-3,
                                      epsilon_distance=1e-5):
    """Drop-in for kernels.rotlet_kernel_source_target_numba (kernels/kernels.py:856-908)."""
    return _np_pairsum("rotlet", r_source, r_target, density, None, eta, reg, epsilon_distance)


def stresslet_kernel_source_target_numba(r_source, r_target, normal, density, eta=1.0,
                                         reg=5e-3, epsilon_distance=1e-5):
    """Drop-in for kernels.stresslet_kernel_source_target_numba (kernels/kernels.py:1186-1217)."""
    return _np_pairsum("stresslet", r_source, r_target, density, normal, eta, reg,
                       epsilon_distance)


def stresslet_kernel_times_normal_times_density_numba(r_vectors, normal, density, eta=1.0,
                                                      reg=5e-3, epsilon_distance=1e-5):
    """Drop-in for kernels.stresslet_kernel_times_normal_times_density_numba
    (kernels/kernels.py:1123-1183): the self-sum over j != i (the i == j pair
    is dropped by F3D_EXCLUDE_SELF, as the reference's loop skips it)."""
    return _np_pairsum("stresslet", r_vectors, r_vectors, density, normal, eta, reg,
                       epsilon_distance, self_sum=True)


def complementary_kernel_times_density_numba(r_vectors, normal, density):
    """Drop-in for kernels.complementary_kernel_times_density_numba
    (kernels/kernels.py:1267-1283): n_i * sum_j n_j . q_j, on the GPU."""
    n = _to_dev(normal)
    q = _to_dev(density, n.shape[0])
    return (n * (n * q).sum()).cpu().numpy().ravel()


def _points(r, fmt, what):
    """Device (N, 3) view parameters of an AoS ('r') or component-block
    ('xyz') point array: (tensor, point stride, component stride, N)."""
    a = np.ascontiguousarray(np.asarray(r, dtype=np.float64).ravel())
    if a.size % 3:
        raise ValueError(f"{what}: size {a.size} is not a multiple of 3")
    n = a.size // 3
    if fmt == "r":
        return torch.from_numpy(a).to(device()), 3, 1, n
    if fmt == "xyz":
        return torch.from_numpy(a).to(device()), 1, n, n
    raise ValueError("input_format is 'r' or 'xyz'")


def oseen_tensor_source_target(r_source, r_target, eta=1.0, reg=5e-3, epsilon_distance=1e-5,
                               input_format="r"):
    """Drop-in for kernels.oseen_tensor_source_target (kernels/kernels.py:119-211):
    the dense (3 Nt, 3 Ns) Oseen tensor, built on the GPU by f3d_oseen_matrix."""
    s, ssp, ssc, ns = _points(r_source, input_format, "r_source")
    t, tsp, tsc, nt = _points(r_target, input_format, "r_target")
    G = torch.empty((3 * nt, 3 * ns), dtype=torch.float64, device=device())
    rc = L.load().f3d_oseen_matrix(ns, L.ptr(s), ssp, ssc, nt, L.ptr(t), tsp, tsc, float(eta),
                                   float(reg), float(epsilon_distance),
                                   0 if input_format == "r" else 1, L.ptr(G), 3 * ns, _stream())
    L.check(rc, "f3d_oseen_matrix")
    return G.cpu().numpy()


def oseen_tensor(r_vectors, eta=1.0, reg=5e-3, epsilon_distance=1e-5, input_format="r"):
    """Drop-in for kernels.oseen_tensor (kernels/kernels.py:31-116): the points
    as both sources and targets (diagonal blocks regularised, not zero)."""
    return oseen_tensor_source_target(r_vectors, r_vectors, eta, reg, epsilon_distance,
                                      input_format)


def stresslet_kernel_times_normal_numba(r_vectors, normal, eta=1.0, reg=5e-3,
                                        epsilon_distance=1e-5):
    """Drop-in for kernels.stresslet_kernel_times_normal_numba
    (kernels/kernels.py:1063-1120): the dense (3N, 3N) stresslet contracted with
    the normals, built on the GPU by f3d_stresslet_matrix."""
    x = _to_dev(r_vectors)
    n = _to_dev(normal, x.shape[0])
    N = x.shape[0]
    M = torch.empty((3 * N, 3 * N), dtype=torch.float64, device=device())
    rc = L.load().f3d_stresslet_matrix(N, L.ptr(x), L.ptr(n), 3, 1, float(eta), float(reg),
                                       float(epsilon_distance), L.ptr(M), 3 * N, _stream())
    L.check(rc, "f3d_stresslet_matrix")
    return M.cpu().numpy()


def complementary_kernel(r_vectors, normal):
    """Drop-in for kernels.complementary_kernel (kernels/kernels.py:1286-1295):
    the rank-one (3N, 3N) matrix n n^T, formed on the GPU."""
    n = _to_dev(normal).reshape(-1)
    return torch.outer(n, n).cpu().numpy()
