"""ctypes binding of libtq_hip.so (include/tq.h) and the device-buffer plumbing.

There is no CPU implementation behind these calls: when the shared library or
a GPU is missing the entry points raise, they never fall back.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import threading
from concurrent.futures import ThreadPoolExecutor
from contextlib import contextmanager, nullcontext

import numpy as np

_HERE = os.path.dirname(os.path.abspath(__file__))
# TQ_HIP_LIBRARY names another build of the same library (the measurement variants that
# `make KNOCKOUT=.. OUT=..` produces); unset, the product library next to this file is loaded.
LIB_PATH = os.environ.get("TQ_HIP_LIBRARY") or os.path.join(_HERE, "libtq_hip.so")

TQ_F16, TQ_F32, TQ_F64 = 0, 1, 2
ROT_DENSE, ROT_WHT = 0, 1
KIND_K, KIND_V = 0, 1
DOMAIN_ROTATED, DOMAIN_ORIGINAL = 0, 1
KFMT_TURBO, KFMT_Q8_0 = 0, 1
ERR_ARG, ERR_UNSUPPORTED, ERR_ALIGN, ERR_HIP = -1, -2, -3, -4


class TQConfig(C.Structure):
    _fields_ = [("d", C.c_int32), ("bits", C.c_int32), ("rotation", C.c_int32), ("norm_correction", C.c_int32),
                ("centroids", C.POINTER(C.c_double)), ("signs1", C.POINTER(C.c_double)),
                ("signs2", C.POINTER(C.c_double)), ("rotation_matrix", C.POINTER(C.c_double)),
                ("projection", C.POINTER(C.c_double)), ("projection_scale", C.c_double)]


class TQAttnParams(C.Structure):
    _fields_ = [("batch", C.c_int32), ("n_q_heads", C.c_int32), ("n_kv_heads", C.c_int32), ("tokens", C.c_int64),
                ("capacity", C.c_int64), ("n_splits", C.c_int32), ("k_format", C.c_int32), ("v_format", C.c_int32),
                ("scale", C.c_float), ("sparse_v_tau", C.c_float), ("tokens_dev", C.c_void_p),
                ("bias_entries", C.c_int32), ("bias_pos", C.c_void_p), ("bias_val", C.c_void_p),
                ("head_dim", C.c_int32)]


class TQAttnPlan(C.Structure):
    _fields_ = [("passes", C.c_int32), ("heads_per_pass", C.c_int32), ("wavefronts", C.c_int32), ("partials", C.c_int32),
                ("groups_per_workgroup", C.c_int32), ("lane_tables", C.c_int32), ("workgroups", C.c_int64)]


HOST_SLOTS = 8
HOST_FETCH, HOST_WIDEN, HOST_UPLOAD, HOST_NARROW = 0, 1, 2, 3


class TQHostJob(C.Structure):
    _fields_ = [("kind", C.c_int64), ("n", C.c_int64), ("n_pieces", C.c_int64), ("piece", C.c_int64), ("host", C.c_void_p),
                ("slots", C.c_void_p), ("seen", C.c_int64), ("next", C.c_int64), ("ready", C.c_int64), ("done", C.c_int64),
                ("slot_done", C.c_int32 * HOST_SLOTS)]


class TQHostDesk(C.Structure):
    _fields_ = [("job", C.c_void_p), ("users", C.c_int64), ("taken", C.c_int64)]


class TQHostBoard(C.Structure):
    _fields_ = [("desk", TQHostDesk * 16), ("state", C.c_int64), ("bell", C.c_int32), ("sleepers", C.c_int32)]


_P, _I, _L, _D = C.c_void_p, C.c_int, C.c_int64, C.c_double

# name -> (restype, argtypes); mirrors include/tq.h one to one
PROTOTYPES = {
    "tq_version": (_I, []),
    "tq_last_error": (C.c_char_p, []),
    "tq_device_count": (_I, []),
    "tq_create": (_I, [C.POINTER(_P), C.POINTER(TQConfig)]),
    "tq_destroy": (None, [_P]),
    "tq_fwht": (_I, [_P, _P, _L, C.c_int32, _I, _I, _P]),
    "tq_rotate": (_I, [_P, _P, _P, _L, _I, _I, _I, _P]),
    "tq_nearest_centroid": (_I, [_P, _L, C.POINTER(C.c_double), C.c_int32, _P, _P]),
    "tq_quantize_indices": (_I, [_P, _P, _L, _I, _P, _P, _P, _P]),
    "tq_dequantize_indices": (_I, [_P, _P, _P, _L, _P, _P, _I, _P, _P]),
    "tq_qjl_quantize": (_I, [_P, _P, _L, _I, _P, _P, _P]),
    "tq_qjl_dequantize": (_I, [_P, _P, _P, _D, _L, _P, _P]),
    "tq_qjl_dequantize_add": (_I, [_P, _P, _P, _D, _L, _P, _P]),
    "tq_pack_bits": (_I, [_P, _L, C.c_int32, _P, _P]),
    "tq_unpack_bits": (_I, [_P, _L, C.c_int32, _P, _P]),
    "tq_pack_indices": (_I, [_P, _L, C.c_int32, _P, _P]),
    "tq_packed_bytes": (_L, [C.c_int32, _L, _L]),
    "tq_store": (_I, [_P, _P, _L, _L, _I, _I, _P, _P]),
    "tq_store_kv": (_I, [_P, _P, _P, _P, _L, _L, _I, _P, _P, _P]),
    "tq_store_kv_cache": (_I, [_P, _P, _P, _P, _L, _L, _L, _I, _P, _P, _P]),
    "tq_append": (_I, [_P, _P, _L, _L, _L, _L, _I, _I, _P, _P]),
    "tq_append_kv": (_I, [_P, _P, _P, _P, _L, _L, _L, _L, _I, _P, _P, _P]),
    "tq_store_layer": (_I, [_P, _P, _P, _P, _L, _L, _L, _I, _P, _P, _P]),
    "tq_append_layer": (_I, [_P, _P, _P, _P, _L, _L, _P, _L, _L, _I, _P, _P, _P, _P]),
    "tq_append_kv_at": (_I, [_P, _P, _P, _P, _L, _P, _L, _L, _I, _P, _P, _P, _P]),
    "tq_append_at": (_I, [_P, _P, _L, _P, _L, _L, _I, _I, _P, _P, _P]),
    "tq_q8_0_append_at": (_I, [_P, _L, _P, _L, _L, _I, _I, _P, _P, _P]),
    "tq_requantize": (_I, [_P, _P, _P, _L, _L, _I, _P, _P]),
    "tq_fork_block_bytes": (_L, [C.c_int32]),
    "tq_export_fork_blocks": (_I, [_P, _P, _L, _L, _I, _P, _P]),
    "tq_import_fork_blocks": (_I, [_P, _P, _L, _L, _I, _P, _P]),
    "tq_fork_row_bytes": (_L, [C.c_int32, C.c_int32]),
    "tq_export_fork_blocks_sized": (_I, [_P, _P, _L, _L, _I, C.c_int32, _P, _P]),
    "tq_import_fork_blocks_sized": (_I, [_P, _P, _L, _L, _I, C.c_int32, _P, _P]),
    "tq_load": (_I, [_P, _P, _L, _L, _I, _P, _I, _I, _P]),
    "tq_load_kv": (_I, [_P, _P, _P, _P, _L, _L, _P, _P, _P]),
    "tq_unpack_codes": (_I, [_P, _P, _L, _L, _I, _P, _P, _P]),
    "tq_store_qjl": (_I, [_P, _P, _L, _L, _I, _P, _P, _P, _P]),
    "tq_q8_0_bytes": (_L, [_L, _L]),
    "tq_q8_0_store": (_I, [_P, _L, _L, _I, _P, _P]),
    "tq_q8_0_unpack": (_I, [_P, _L, _L, _P, _P, _P]),
    "tq_q8_0_store_v": (_I, [_P, _L, _L, _I, _P, _P]),
    "tq_q8_0_unpack_v": (_I, [_P, _L, _L, _P, _P, _P]),
    "tq_q8_0_append": (_I, [_P, _L, _L, _L, _L, _I, _I, _P, _P]),
    "tq_attn_workspace_bytes": (_L, [C.POINTER(TQAttnParams)]),
    "tq_decode_attention_plan": (_I, [C.POINTER(TQAttnParams), _I, _I, _I, _I, _L, C.POINTER(TQAttnPlan)]),
    "tq_decode_attention": (_I, [_P, _P, C.POINTER(TQAttnParams), _P, _I, _P, _P, _P, _P, _P, _P, _P, _L, _P]),
    "tq_decode_attention_static": (_I, [_P, _P, C.POINTER(TQAttnParams), _P, _I, _P, _P, _P, _P, _P, _P]),
    "tq_host_serve": (None, [C.POINTER(TQHostBoard)]),
    "tq_host_open": (_I, [C.POINTER(TQHostBoard), _I]),
    "tq_host_close": (None, [C.POINTER(TQHostBoard), _I]),
    "tq_host_drive": (_I, [C.POINTER(TQHostBoard), C.POINTER(TQHostJob), _P, _P]),
    "tq_score_tile": (_I, [_P, _P, _I, _L, _P, _P, _P, _L, _P, _I, _P, _L, _P]),
}

_lib = None


def lib():
    """The loaded library; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `make -C turboquant_plus_amd/csrc` "
                "(or __graft_entry__.build()); there is no CPU fallback")
        handle = C.CDLL(LIB_PATH)
        for name, (res, args) in PROTOTYPES.items():
            fn = getattr(handle, name)
            fn.restype, fn.argtypes = res, args
        _lib = handle
    return _lib


def last_error() -> str:
    return lib().tq_last_error().decode("utf-8", "replace")


def check(rc: int) -> None:
    """Map a C return code to the exception the reference API raises."""
    if rc == 0:
        return
    msg = last_error()
    if rc in (ERR_ARG, ERR_ALIGN):
        raise ValueError(msg)
    if rc == ERR_UNSUPPORTED:
        raise NotImplementedError(msg)
    raise RuntimeError(f"HIP error: {msg}")


_torch = None
_FLOATS = {}            # torch dtype -> code, for the three that the kernels take
_current_device = _raw_stream = None


def torch():
    global _torch, _current_device, _raw_stream
    if _torch is None:
        import torch as _t
        _FLOATS.update({_t.float16: TQ_F16, _t.float32: TQ_F32, _t.float64: TQ_F64})
        # torch's own short ways to the current device and to a stream's handle, where it has them: the public ones cost 0.3 and
        # 2.7 us of a call that launches in 3.5
        _current_device = getattr(_t._C, "_cuda_getDevice", None) or _t.cuda.current_device
        _raw_stream = getattr(_t._C, "_cuda_getCurrentRawStream", None) or (lambda d: _t.cuda.current_stream(d).cuda_stream)
        _torch = _t
    return _torch


def require_gpu():
    if lib().tq_device_count() < 1:
        raise RuntimeError("no HIP device visible: the TurboQuant kernels need an MI355X (no CPU path exists)")
    return torch().device("cuda")


def dtype_code(t) -> int:
    torch()
    code = _FLOATS.get(t.dtype)
    if code is None:
        raise TypeError(f"unsupported dtype {t.dtype}")
    return code


def torch_dtype(code: int):
    tt = torch()
    return {TQ_F16: tt.float16, TQ_F32: tt.float32, TQ_F64: tt.float64}[code]


def to_device(x, float_ok=(np.float16, np.float32, np.float64)):
    """NumPy array or torch tensor -> contiguous CUDA tensor (floats keep their
    width, everything else becomes float64 as NumPy promotion would)."""
    tt = torch()
    if isinstance(x, tt.Tensor):
        if x.is_cuda and x.dtype in _FLOATS and x.is_contiguous() and x.get_device() == _current_device():
            return x        # in place already
        t = x.to(require_gpu())
        if t.dtype not in (tt.float16, tt.float32, tt.float64):
            t = t.to(tt.float64)
        return t.contiguous()
    a = np.asarray(x)
    if a.dtype not in [np.dtype(f) for f in float_ok]:
        a = a.astype(np.float64)
    return _upload_one(np.ascontiguousarray(a), require_gpu())


# ---- results of the NumPy classes: device buffers and their way into host arrays -----------------------------------

def unchanged(obj, *methods):
    """Whether these functions are what `obj` answers to by their names: not where it is of another class or where a
    subclass, the object or a patch of its class has them replaced.  The classes take each other's device-side steps only
    then, else the public methods."""
    return all(getattr(getattr(obj, f.__name__, None), "__func__", None) is f for f in methods)


def device_block(*specs):
    """(buffer, tensors): one uint8 device buffer and views of it for the (shape, torch dtype) specs, so that small
    results travel to or from the host in one copy."""
    tt = torch()
    offs, total = [], 0
    for shape, dtype in specs:
        offs.append(total)
        total += (math.prod(shape) * dtype.itemsize + 255) // 256 * 256
    buf = tt.empty(total, dtype=tt.uint8, device=require_gpu())
    return buf, [buf[o:o + math.prod(shape) * dtype.itemsize].view(dtype).view(shape) for o, (shape, dtype) in zip(offs, specs)]


# A block up to this size travels as one pageable copy (a copy costs 14 us before its first byte).  64 rows of 384: 0.23 ms, 0.25
# with 128 KiB; a cache of 2 x 4 x 512 x 128: 1.44 and 1.55.
ONE_COPY = 1 << 19
# Bytes of the host array that a thread takes at a time (no two threads clear the same huge page), and the threads beside the
# caller's.  A cache of 2 x 4 x 4096 x 128 in float32, both ways, ms, with pieces of 1 / 2 / 4 MiB: four threads 9.6 / 8.6 / 8.5, six
# 8.9 / 8.6 / 8.0, eight 9.1 / 7.8 / 7.6, eleven 9.1 / 8.4 / 7.9 (16 CPUs); through the interpreter, which handed a share of each slot to six
# threads, 9.4 - 11.0, 16 000 rows of 128 10.1 (now 4.5 - 5.4), 2 x 4 x 2048 x 256 in float64 11.9 - 13.7 (9.0).  Never more of them than
# there are processors for beside the caller's.
STAGE = 4 << 20
COPY_THREADS = max(1, min(8, len(os.sched_getaffinity(0)) - 1))
# Host arrays from this size on are worked on by several threads: below, handing the work over costs more.
SHARED = 4 << 20
_copiers = None
_copiers_lock = threading.Lock()
# The copy threads work for every thread of the process that has large arrays under way, and go back to the pool some milliseconds
# after the last of them is done.
_board = TQHostBoard()


def _copy_pool():
    global _copiers
    with _copiers_lock:
        if _copiers is None:
            _copiers = ThreadPoolExecutor(COPY_THREADS, thread_name_prefix="tq-copy")
        return _copiers


def _forget_copiers():
    """A forked child has none of the threads, and the lock and the board as they happened to be held."""
    global _copiers, _copiers_lock, _board
    _copiers, _copiers_lock, _board = None, threading.Lock(), TQHostBoard()


os.register_at_fork(after_in_child=_forget_copiers)


_helping = threading.local()     # .board: where this thread's jobs are helped with, while it has any


_alone = nullcontext()


def helpers(nbytes):
    """A context in which the copy threads help with this thread's host arrays where those are large (`nbytes`: the largest
    one's): one handing over for all the arrays of a call.  Where there are no threads (the ending interpreter takes no more work, a
    forked child starts its own) the caller's does it all."""
    return _alone if nbytes <= SHARED or getattr(_helping, "board", None) is _board else _helped()


@contextmanager
def _helped():
    board, before = _board, getattr(_helping, "board", None)
    missing = lib().tq_host_open(board, COPY_THREADS)
    try:
        try:
            while missing > 0:
                missing -= 1    # also where the submit fails: it may have queued its work all the same
                _copy_pool().submit(lib().tq_host_serve, board)
        except RuntimeError:    # the interpreter is ending, or no thread can be started
            pass
        _helping.board = board
        yield
    finally:
        lib().tq_host_close(board, missing)
        _helping.board = before


def _host_job(kind, n, host, device):
    """A job of n elements (include/tq.h) between the contiguous array `host` and the device tensor `device`.  Returns the bits
    that HOST_NARROW saw."""
    each = 8 if kind in (HOST_WIDEN, HOST_NARROW) else 1       # host bytes of an element; one on the other side
    piece = max(min(STAGE, n * each // 4), 1 << 18) // each
    pieces = -(-n // piece)
    slots = torch().empty(min(HOST_SLOTS, pieces) * piece, dtype=torch().uint8, pin_memory=True)
    job = TQHostJob(kind=kind, n=n, n_pieces=pieces, piece=piece, host=host.ctypes.data, slots=slots.data_ptr())
    stream = stream_ptr()
    if n * each <= SHARED:
        check(lib().tq_host_drive(None, job, ptr(device), stream))
    else:
        with helpers(n * each):
            check(lib().tq_host_drive(_board, job, ptr(device), stream))
    return job.seen


def narrow_indices(indices, n_centroids):
    """Codebook indices of any type as contiguous uint8; ValueError if one is outside 0 .. n_centroids - 1 (a power of
    two).  int64 ones, what the classes return, are checked and narrowed in one go."""
    if indices.dtype != np.int64 or not indices.flags.c_contiguous:
        if indices.size and (indices.min() < 0 or indices.max() >= n_centroids):
            _refuse_indices()
        return np.ascontiguousarray(indices, dtype=np.uint8)
    out = np.empty(indices.shape, np.uint8)
    np.copyto(out, indices, casting="unsafe")
    seen = int(np.bitwise_or.reduce(indices, axis=None))
    if seen & ~(n_centroids - 1):       # a bit above the codebook's: some index is outside
        _refuse_indices()
    return out


def _refuse_indices():
    raise ValueError("indices out of range for this codebook")


def upload_indices(indices, n_centroids, *others):
    """Device tensors of codebook indices (uint8; checked as narrow_indices does) and of further arrays (upload)."""
    if indices.dtype != np.int64 or not indices.flags.c_contiguous or indices.nbytes <= SHARED:
        return upload(narrow_indices(indices, n_centroids), *others)
    t = torch().empty(indices.shape, dtype=torch().uint8, device=require_gpu())
    if _host_job(HOST_NARROW, indices.size, indices, t) & ~(n_centroids - 1):
        _refuse_indices()
    return [t, *upload(*others)]


def fetch(buf, *wanted):
    """NumPy arrays of (tensor, NumPy dtype) pairs whose tensors are views of the block `buf` (device_block)."""
    tt = torch()
    if buf.numel() <= ONE_COPY:
        raw = np.empty(buf.numel(), np.uint8)
        tt.from_numpy(raw).copy_(buf)
        base = buf.data_ptr()
        res = []
        for t, dtype in wanted:
            o = t.data_ptr() - base
            a = raw[o:o + t.nbytes].view(_NP_DTYPES[str(t.dtype)]).reshape(tuple(t.shape))
            res.append(a if a.dtype == dtype else a.astype(dtype))
        return res
    res = []
    for t, dtype in wanted:
        a = np.empty(tuple(t.shape), dtype)
        same = a.dtype == _NP_DTYPES[str(t.dtype)]
        if t.nbytes > ONE_COPY and (same or (t.dtype == tt.uint8 and dtype == np.int64)):
            # fresh host memory costs more than the transfer (64 MiB: 9.3 ms by one pageable copy, 1.2 ms of them the link)
            _host_job(HOST_FETCH if same else HOST_WIDEN, a.nbytes if same else a.size, a, t)
        else:
            src = a if same else np.empty(tuple(t.shape), _NP_DTYPES[str(t.dtype)])
            tt.from_numpy(src).copy_(t)
            if src is not a:
                np.copyto(a, src)
        res.append(a)
    return res


def _torch_dtype(dt):
    tt = torch()
    return {"u1": tt.uint8, "i1": tt.int8, "f2": tt.float16, "f4": tt.float32, "f8": tt.float64}[dt.str[1:]]


_NP_DTYPES = {"torch.uint8": np.dtype(np.uint8), "torch.int8": np.dtype(np.int8), "torch.float64": np.dtype(np.float64)}


def host_norms(norms, n):
    """The first n norms, those of n vectors, as a contiguous float64 array."""
    a = np.ascontiguousarray(np.asarray(norms, dtype=np.float64).reshape(-1)[:n])
    if a.size != n:
        raise ValueError(f"{a.size} norms for {n} vectors")
    return a


def _upload_one(a, dev):
    tt = torch()
    if a.nbytes < SHARED // 2:
        return tt.from_numpy(a if a.flags.writeable else a.copy()).to(dev)   # torch warns of read-only memory
    t = tt.empty(a.shape, dtype=_torch_dtype(a.dtype), device=dev)
    _host_job(HOST_UPLOAD, a.nbytes, a, t)
    return t


def upload(*arrays):
    """Contiguous NumPy arrays -> device tensors; small ones in one copy."""
    tt = torch()
    dev = require_gpu()
    if sum(a.nbytes for a in arrays) > ONE_COPY:
        return [_upload_one(a, dev) for a in arrays]
    offs, total = [], 0
    for a in arrays:
        offs.append(total)
        total += (a.nbytes + 255) // 256 * 256
    raw = np.empty(total, np.uint8)
    for a, o in zip(arrays, offs):
        raw[o:o + a.nbytes] = a.reshape(-1).view(np.uint8)
    buf = tt.from_numpy(raw).to(dev)
    return [buf[o:o + a.nbytes].view(_torch_dtype(a.dtype)).view(a.shape) for a, o in zip(arrays, offs)]


def stream_ptr():
    """The handle of the current device's current stream, for a void * argument."""
    if not torch().cuda.is_initialized():
        torch().cuda.init()
    return _raw_stream(_current_device())


def ptr(t):
    return t.data_ptr() if t is not None else None


def dbl_ptr(a):
    return a.ctypes.data_as(C.POINTER(C.c_double)) if a is not None else None


class Handle:
    """Owns a tq_handle*; the NumPy tables it was built from stay referenced."""

    def __init__(self, d, bits, centroids, *, signs1=None, signs2=None, rotation=None, projection=None,
                 projection_scale=0.0, norm_correction=True):
        require_gpu()
        keep = lambda a: None if a is None else np.ascontiguousarray(a, dtype=np.float64)
        self._tables = [keep(centroids), keep(signs1), keep(signs2), keep(rotation), keep(projection)]
        cfg = TQConfig(d=d, bits=bits, rotation=ROT_DENSE if rotation is not None else ROT_WHT,
                       norm_correction=int(bool(norm_correction)),
                       centroids=dbl_ptr(self._tables[0]), signs1=dbl_ptr(self._tables[1]),
                       signs2=dbl_ptr(self._tables[2]), rotation_matrix=dbl_ptr(self._tables[3]),
                       projection=dbl_ptr(self._tables[4]), projection_scale=float(projection_scale))
        h = C.c_void_p()
        check(lib().tq_create(C.byref(h), C.byref(cfg)))
        self.h = h

    def __del__(self):
        h, self.h = getattr(self, "h", None), None
        if h and _lib is not None:
            _lib.tq_destroy(h)
