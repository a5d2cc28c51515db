"""ctypes binding of ``libqlinear.so`` (declared in ``include/qlinear.h``).

The reference reaches its kernels the same way -- ctypes into a native loader
(engine/kernels/cuda_jit.py:141-289) -- so this module is the MI355X counterpart
of ``cuda_jit``: it loads one prebuilt gfx950 library instead of compiling CUDA at
run time. There is no fallback: without the library every op raises.
"""

import ctypes
import itertools
import os
import threading

import torch  # noqa: F401  (loads the HIP runtime the library then shares)

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libqlinear.so")

QLX_OK, QLX_EINVAL, QLX_EHIP = 0, -1, -2
MODE_BF16, MODE_PLANES, MODE_SWIGLU, MODE_SUM = 0, 1, 2, 3
SCALE_F16, SCALE_BF16 = 0, 1
STORE_OFFSET, STORE_SIGNED, STORE_K32 = 0, 1, 2
FMT_W8A16, FMT_W4A16, FMT_FP8, FMT_REF8, FMT_REF4, FMT_FP8WO, FMT_INT8 = range(7)


class Plan(ctypes.Structure):
    """``qlx_plan``: mode, splits, waves, kw, rw, workspace, tickets."""

    _fields_ = [
        ("mode", ctypes.c_int), ("splits", ctypes.c_int), ("waves", ctypes.c_int),
        ("kw", ctypes.c_int), ("rw", ctypes.c_int),
        ("workspace", ctypes.c_void_p), ("tickets", ctypes.c_void_p),
    ]


class StackCall(ctypes.Structure):
    """``qlx_stack_call``: one projection of a decode-step chain."""

    _fields_ = [
        ("w", ctypes.c_void_p), ("w_scale", ctypes.c_void_p), ("x", ctypes.c_void_p), ("y", ctypes.c_void_p),
        ("n", ctypes.c_int), ("k", ctypes.c_int), ("mode", ctypes.c_int), ("kw", ctypes.c_int),
    ]


class StackLaunch(ctypes.Structure):
    """``qlx_stack_launch``: grid, LDS bytes, waves, descriptor LDS offset, lanes, the LDS offset
    of the FP8 row maxima, whether row blocks are cut into K pieces, and whether the chain has
    attention stages."""

    _fields_ = [(f, ctypes.c_int) for f in ("grid", "lds_bytes", "waves", "desc_lds", "lanes", "amax_off", "pieces",
                                            "attention")]


class NormInput(ctypes.Structure):
    _fields_ = [("resid", ctypes.c_void_p), ("delta", ctypes.c_void_p), ("norm_w", ctypes.c_void_p),
                ("resid_out", ctypes.c_void_p), ("normed_out", ctypes.c_void_p), ("eps", ctypes.c_float),
                ("pad", ctypes.c_int)]


class StackAttention(ctypes.Structure):
    """``qlx_stack_attention``: what entry c of an executor chain is -- kind 0 a projection, 1
    an attention stage's splits, 2 their merge -- and the attention stage's parameters."""

    _fields_ = [("kind", ctypes.c_int), ("n_q", ctypes.c_int), ("n_kv", ctypes.c_int), ("splits", ctypes.c_int),
                ("capacity", ctypes.c_int), ("table_rows", ctypes.c_int), ("q_norm_w", ctypes.c_void_p),
                ("k_norm_w", ctypes.c_void_p), ("cos", ctypes.c_void_p), ("sin", ctypes.c_void_p),
                ("positions", ctypes.c_void_p), ("k_cache", ctypes.c_void_p), ("v_cache", ctypes.c_void_p),
                ("eps", ctypes.c_float), ("scale", ctypes.c_float)]


class RopeArgs(ctypes.Structure):
    """``qlx_rope_args``: the fused QKV head-norm + RoPE + cache write."""

    _fields_ = [("qkv", ctypes.c_void_p), ("planes", ctypes.c_void_p), ("stride", ctypes.c_longlong),
                ("splits", ctypes.c_int), ("rows", ctypes.c_int), ("n_q", ctypes.c_int), ("n_kv", ctypes.c_int),
                ("q_col", ctypes.c_int), ("k_col", ctypes.c_int), ("v_col", ctypes.c_int),
                ("seq_len", ctypes.c_int), ("capacity", ctypes.c_int), ("table_rows", ctypes.c_int),
                ("pos_int64", ctypes.c_int), ("eps", ctypes.c_float),
                ("q_norm_w", ctypes.c_void_p), ("k_norm_w", ctypes.c_void_p), ("cos", ctypes.c_void_p),
                ("sin", ctypes.c_void_p), ("positions", ctypes.c_void_p), ("q_out", ctypes.c_void_p),
                ("k_cache", ctypes.c_void_p), ("v_cache", ctypes.c_void_p), ("k_scale", ctypes.c_void_p),
                ("v_scale", ctypes.c_void_p), ("k_copy", ctypes.c_void_p), ("v_copy", ctypes.c_void_p)]


_P, _I, _F, _LL = ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_longlong
_PLAN = ctypes.POINTER(Plan)
_PI, _PLL = ctypes.POINTER(ctypes.c_int), ctypes.POINTER(ctypes.c_longlong)

#: Every exported entry point and its argument types (the header's declarations).
SIGNATURES = {
    "qlx_last_error": ([], ctypes.c_char_p),
    "qlx_abi_version": ([], _I),
    "qlx_quantize_weight": ([_P, _P, _P, _I, _I, _I, _I, _I, _I, _I, _P], _I),
    "qlx_dequantize": ([_P, _P, _P, _I, _I, _I, _I, _I, _I, _P], _I),
    "qlx_prepare_ref": ([_P, _P, _I, _I, _I, _I, _P], _I),
    "qlx_row_major_ref": ([_P, _P, _I, _I, _P], _I),
    "qlx_quantize_fp8_weight": ([_P, _P, _P, _I, _I, _I, _P], _I),
    "qlx_quantize_fp8_act": ([_P, _P, _P, _I, _I, _P], _I),
    "qlx_fp8_selfcheck": ([_P, _P], _I),
    "qlx_int8_prepare": ([_P, _P, _I, _I, _P], _I),
    "qlx_quantize_act_int8": ([_P, _P, _P, _P, _P, _I, _I, _P], _I),
    "qlx_plan_linear": ([_I, _I, _I, _I, _I, _PLAN], _I),
    "qlx_plan_tickets": ([_PLAN, _I, _I, _I, _I], _I),
    "qlx_stream_capture": ([_P], ctypes.c_ulonglong),
    "qlx_plan_fit": ([_PLAN, _I, _I, _I, _I, _I, _I], _I),
    "qlx_plan_slices": ([_I, _I, _I, _I, _I, _I], _I),
    "qlx_tile_rows": ([_P, _P, _I, _I, _P], _I),
    "qlx_linear_w8a16": ([_P, _P, _P, _P, _I, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_w4a16": ([_P, _P, _P, _P, _I, _I, _I, _I, _PLAN, _P], _I),
    "qlx_plan_skinny": ([_I, _I, _I, _I, _I, _PLAN], _I),
    "qlx_linear_skinny": ([_I, _P, _P, _P, _P, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_skinny_noalloc": ([_I, _P, _P, _P, _P, _I, _I, _I, _I, _P], _I),
    "qlx_linear_skinny_fp8": ([_P, _P, _P, _P, _P, _I, _I, _I, _PLAN, _P], _I),
    "qlx_plan_resident": ([_I, _I, _I, _I, _I, _PLAN], _I),
    "qlx_linear_resident": ([_I, _P, _P, _P, _P, _P, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_fp8_w8a8_q": ([_P, _P, _P, _P, _P, _I, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_fp8_w8a8": ([_P, _P, _P, _P, _I, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_ref": ([_P, _P, _P, _P, _I, _I, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_fp8wo": ([_P, _P, _P, _P, _I, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_int8": ([_P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _PLAN, _P], _I),
    "qlx_linear_add_norm": ([_I, _P, _P, _P, _I, _I, _I, _I, _P, _P, _F, _P, _P, _P, _P, _PLAN, _P], _I),
    "qlx_reduce_planes": ([_P, _P, _LL, _I, _P], _I),
    "qlx_residual_planes": ([_P, _P, _P, _LL, _I, _P], _I),
    "qlx_add_rms_norm": ([_P, _P, _P, _I, _P, _P, _P, _I, _I, _F, _P], _I),
    "qlx_add_norm_quant_int8": ([_P, _P, _P, _I, _P, _P, _P, _P, _I, _I, _F, _P], _I),
    "qlx_add_norm_quant_fp8": ([_P, _P, _P, _I, _P, _P, _P, _P, _P, _I, _I, _F, _P], _I),
    "qlx_swiglu": ([_P, _P, _I, _P, _I, _I, _P], _I),
    "qlx_stack_desc_size": ([], _I),
    "qlx_stack_build": ([_I, _I, ctypes.POINTER(StackCall), _I, _I, _I, _P, _PLAN, _P, _PLL,
                         ctypes.POINTER(StackLaunch)], _I),
    "qlx_stack_build_normed": ([_I, _I, ctypes.POINTER(StackCall), _I, ctypes.POINTER(NormInput), _I, _I, _P,
                                _PLAN, _P, _PLL, ctypes.POINTER(StackLaunch)], _I),
    "qlx_stack_build_step": ([_I, _I, ctypes.POINTER(StackCall), _I, ctypes.POINTER(NormInput),
                              ctypes.POINTER(StackAttention), _I, _I, _P, _PLAN, _P, _PLL, ctypes.POINTER(StackLaunch)],
                             _I),
    "qlx_stack_run": ([_I, _P, _I, ctypes.POINTER(StackLaunch), _P, _P, _LL, _P], _I),
    "qlx_stream_read": ([_P, _LL, _P, _I, _P], _I),
    "qlx_qkv_norm_rope": ([ctypes.POINTER(RopeArgs), _P], _I),
    "qlx_attention_workspace": ([_I, _I, _I, _I, _I, ctypes.POINTER(ctypes.c_size_t)], _I),
    "qlx_decode_attention": ([_P, _P, _P, _P, _P, _P, _P, _P, ctypes.c_size_t, _I, _I, _I, _I, _I, _I, _I, _F, _P],
                             _I),
}

_lib = None


def lib():
    """The loaded library; raises RuntimeError if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with __graft_entry__.build() "
                "(there is no CPU or Python fallback for these ops)")
        handle = ctypes.CDLL(LIB_PATH)
        for name, (args, res) in SIGNATURES.items():
            fn = getattr(handle, name)
            fn.argtypes = args
            fn.restype = res
        _lib = handle
    return _lib


def last_error():
    return lib().qlx_last_error().decode(errors="replace")


def check(rc, what):
    """Map a status to the reference's conventions: ValueError for contract violations,
    RuntimeError for runtime failures (engine/kernels/cuda_jit.py:43-45)."""
    if rc == QLX_OK:
        return
    msg = f"{what}: {last_error()}"
    if rc == QLX_EINVAL:
        raise ValueError(msg)
    raise RuntimeError(msg)


def call(name, *args):
    check(getattr(lib(), name)(*args), name)


# Addresses travel as plain ints (None: NULL), which ctypes converts for the declared pointer
# types, and the current stream comes without a torch.cuda.Stream object: an eager single linear is
# bound by this host path (2560 x 9728 W8A16 of one token, 10 us of kernel: 14.1 -> 10.3 us a call).
def ptr(t):
    return t.data_ptr() if t is not None else None


def stream(device):
    """The current stream of ``device`` (its handle, as an int)."""
    index = device.index
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)


def require_device(*tensors):
    """The ops run only on a ROCm device; CPU tensors are a contract violation."""
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise ValueError("quantized linear ops need tensors on a ROCm GPU (no CPU path)")
        if not t.is_contiguous():
            raise ValueError("tensors must be contiguous")


#: Counters of a slot and slots of a device (256 x 2 KB). A slot stays with its stream, or with its stream of
#: one graph capture, whose graph may be replayed at any later time; calls past the last slot, and those
#: that need more counters, zero their own.
STREAM_TICKETS = 512
STREAM_SLOTS = 256
_stream_tickets = {}


class _Local(threading.local):
    """The capture that this thread last launched into (0: none), and its counters outside the slots by
    device and stream. A buffer is memory of its stream, so it may go once the call is enqueued; a
    capture's is memory of its graph."""

    def __init__(self):
        self.capture, self.counters = 0, {}


_local = _Local()


def capture_id(stream):
    """The graph capture that ``stream`` (a handle) is in, 0 outside one."""
    return lib().qlx_stream_capture(stream)


def stream_tickets(device, stream, count=STREAM_TICKETS):
    """The address of ``count`` zeroed counters for this thread's next split-K call on ``stream``, the current
    one: calls that may overlap count apart, whether on two streams, in two graphs' replays (whatever
    stream they were captured on) or in one graph's branches. The slots are made by eager calls: inside a
    capture their zeroing would be a node of that graph. Counters zeroed in a capture cost its replays
    that node, 1 to 4 us."""
    capture = capture_id(stream)
    if _local.capture != capture:  # an ended capture's go back to its pool
        _local.capture, _local.counters = capture, {}
    index = device.index if device.index is not None else torch.cuda.current_device()
    pool = _stream_tickets.get(index)
    if pool is None and not capture:
        buf = torch.zeros(STREAM_SLOTS * STREAM_TICKETS, dtype=torch.int32, device=device)
        torch.cuda.current_stream(device).synchronize()  # once: other streams' first calls find it zeroed
        pool = _stream_tickets.setdefault(index, (buf, {}, itertools.count()))
    if pool is not None and count <= STREAM_TICKETS:
        buf, slots, numbers = pool
        slot = slots.get((stream, capture))
        if slot is None and len(slots) < STREAM_SLOTS:
            slot = slots.setdefault((stream, capture), next(numbers))
        if slot is not None and slot < STREAM_SLOTS:
            return buf.data_ptr() + slot * STREAM_TICKETS * 4
    buf = _local.counters.get((index, stream))
    if buf is None or buf.numel() < count:
        if len(_local.counters) >= 64:
            _local.counters = {}
        buf = torch.zeros(max(count, STREAM_TICKETS), dtype=torch.int32, device=device)
        _local.counters[index, stream] = buf
    return buf.data_ptr()


def tickets(device, count):
    """``stream_tickets`` for a call on ``device``'s current stream."""
    return stream_tickets(device, stream(device), count)
