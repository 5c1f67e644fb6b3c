"""FlashAttention-2 forward on MI355X (gfx950) behind the reference's Python surface.

Drop-in for ``ascend_rsfa/flash_attention_forward.py`` of Dell710000/ascend-rsfa:

==============================  ===============================================
this module                     reference (flash_attention_forward.py)
==============================  ===============================================
``get_num_compute_cores()``     ``get_num_compute_cores`` (19-21)
``_attention``                  ``class _attention(torch.autograd.Function)``
                                (547-616): same forward signature
                                ``(ctx, q, k, v, causal, sm_scale, BM, BN)``,
                                same assertions (553-554), same saved tensors
                                (612-615), no backward (calling it raises)
``attention``                   ``attention = _attention.apply`` (622)
``get_tiling(Z,H,N,D,causal)``  ``get_tiling`` (624-665): a lookup table there,
                                a gfx950 tile search here; returns
                                ``(BLOCK_M, BLOCK_N)`` for every valid shape
==============================  ===============================================

All arithmetic runs in the HIP library ``lib/librsfa.so`` (C ABI in
``include/rsfa.h``), enqueued on the current HIP stream of the tensors'
device.  There is no fallback path: without the built library, or for tensors
that are not on a GPU, the calls raise.

A ``float8_e5m2`` V with float16 Q and K runs the reference's fp8_v branch
(_attn_fwd_inner 208-211, 217): P is rounded to e5m2 for P.V while the row
sums add the unrounded P; O is float16.  The kernels read V's bytes and run
P.V on the e5m2 MFMA at every head dim (no workspace).

``BM``/``BN`` keep the reference's meaning (query rows per program, keys per
inner tile) and its validity rules: they select the tile, and the compiled
gfx950 tile nearest to the request runs (``resolve_tiling``), so a harness
that times ``attention`` per (BM, BN) candidate, as the reference's tiling
search does, times distinct kernels.  ``BM = BN = 0`` runs ``get_tiling``'s
tile.  Hint mode (``forward(..., tile_hint=True)``, or the environment
variable ``RSFA_TILE_HINT=1`` for every call, ``attention`` included) only
checks a request and runs ``get_tiling``'s tile for the shape, for callers
whose tiles were tuned for Ascend's unified buffer.

Behaviour beyond the reference (documented, deliberate):

* Causal calls with ``BN > BM``, which give NaN in the reference
  (benchmarks/run_correctness_test.py:24-25), raise ``ValueError`` instead.
* Any ``N_CTX >= 1`` works (the reference has no load masks, so it needs
  ``N_CTX`` divisible by its tiles).
* Per-tensor strides are honoured as long as the head dim is unit-stride; other
  layouts are copied to contiguous first.
"""
import ctypes
import importlib
import os
import struct
import sys

import torch


def _package_module(name):
    """``ascend_rsfa.<name>``, whether this file was imported as part of the
    package or loaded by file path under a bare module name, the way every
    reference harness loads its kernel file (benchmarks/run_correctness_test.py:
    58-65: ``spec_from_file_location(clean_name, path)``)."""
    if __package__:
        return importlib.import_module(f"{__package__}.{name}")
    here = os.path.dirname(os.path.abspath(__file__))
    parent = os.path.dirname(here)
    if parent not in sys.path:
        sys.path.insert(0, parent)
    mod = importlib.import_module(f"ascend_rsfa.{name}")
    if os.path.dirname(os.path.abspath(mod.__file__)) != here:
        raise ImportError(f"ascend_rsfa.{name} resolved to {mod.__file__}, not to the package beside "
                          f"{__file__}; put {parent} first on sys.path")
    return mod


_native = _package_module("_native")

__all__ = ["attention", "get_tiling", "get_num_compute_cores", "resolve_tiling", "forward",
           "split_workspace_bytes"]

_DTYPES = {torch.float16: _native.DTYPE_F16, torch.bfloat16: _native.DTYPE_BF16}
_FP8_E5M2 = getattr(torch, "float8_e5m2", None)


def _raise_for(status):
    """Map an rsfa_status to the exception type the reference would raise."""
    if status == _native.OK:
        return
    msg = _native.strerror(status)
    if status == _native.E_HEADDIM:
        raise AssertionError(msg)
    if status == _native.E_DTYPE:
        raise TypeError(msg)
    if status in (_native.E_TILE, _native.E_SHAPE, _native.E_WORKSPACE, _native.E_ALIGN, _native.E_NULL):
        raise ValueError(msg)
    raise RuntimeError(f"rsfa error {status}: {msg}")


def get_num_compute_cores():
    """Compute units of the current device (reference 19-21 reads num_aicore)."""
    n = _native.lib().rsfa_get_num_compute_cores(torch.cuda.current_device())
    if n < 0:
        _raise_for(n)
    return n


_TILING_MEMO = {}


def get_tiling(Z, H, N_CTX, HEAD_DIM, causal, dtype=torch.float16):
    """Return (BLOCK_M, BLOCK_N) for the shape (reference 624-665).

    The reference looks the shape up in a table of Ascend tilings and raises
    KeyError for any shape not listed.  Here a measured, correctness-gated
    tiling cache answers first when one is active (``tiling.use_cache`` or
    ``RSFA_TILING_CACHE``; entries that are not a compiled tile shape are
    ignored); otherwise the library searches the compiled gfx950 tile shapes
    with an LDS feasibility check and a makespan model of the persistent grid
    on the current device's CUs, so it answers for every valid shape.
    ``attention`` called with this tile (or with ``BM = BN = 0``) runs it.
    """
    cache = _tiling_module().active_cache()
    if cache is not None:
        entry = cache.lookup(Z, H, N_CTX, HEAD_DIM, causal, dtype)
        if entry is not None:
            try:
                if resolve_tiling(HEAD_DIM, causal, entry[0], entry[1], dtype) == tuple(entry):
                    return tuple(entry)
            except ValueError:
                pass
    # the library's answer depends only on the shape, dtype and device: memoised
    key = (int(Z), int(H), int(N_CTX), int(HEAD_DIM), bool(causal), dtype,
           torch.cuda.current_device() if torch.cuda.is_available() else -1)
    hit = _TILING_MEMO.get(key)
    if hit is None:
        bm = ctypes.c_int32()
        bn = ctypes.c_int32()
        st = _native.lib().rsfa_get_tiling(int(Z), int(H), int(N_CTX), int(HEAD_DIM), 1 if causal else 0,
                                           _DTYPES.get(dtype, _native.DTYPE_F16), ctypes.byref(bm),
                                           ctypes.byref(bn))
        _raise_for(st)
        hit = (bm.value, bn.value)
        if len(_TILING_MEMO) > 4096:
            _TILING_MEMO.clear()
        _TILING_MEMO[key] = hit
    return hit


def resolve_tiling(HEAD_DIM, causal, BM, BN, dtype=torch.float16):
    """The compiled (BLOCK_M, BLOCK_N) instantiation nearest to a request.

    Raises ValueError for a request the reference's rules reject.  This is the
    tile ``attention`` / ``forward`` run for the request (in hint mode the
    tile of ``get_tiling`` runs instead).
    """
    bm = ctypes.c_int32()
    bn = ctypes.c_int32()
    st = _native.lib().rsfa_resolve_tiling(int(HEAD_DIM), 1 if causal else 0, _DTYPES.get(dtype, -1),
                                           int(BM), int(BN), ctypes.byref(bm), ctypes.byref(bn))
    _raise_for(st)
    return (bm.value, bn.value)


def split_workspace_bytes(Z, H, N_CTX, HEAD_DIM, BM):
    """Workspace of split mode for the BLOCK_M that runs: fp32 (m, l) and the
    un-normalised fp32 accumulator of every query row of every task."""
    return int(_native.lib().rsfa_split_workspace_bytes(int(Z), int(H), int(N_CTX), int(HEAD_DIM), int(BM)))


def _meets_contract(t):
    # 16-byte rows: outer strides a multiple of 8 two-byte or 16 one-byte elements
    mult = 16 // t.element_size()
    st = t.stride()
    return st[3] == 1 and all(s % mult == 0 for s in st[:3]) and t.data_ptr() % 16 == 0


def _as_kernel_layout(t):
    if _meets_contract(t):
        return t
    t = t.contiguous()
    if not _meets_contract(t):
        t = t.clone(memory_format=torch.contiguous_format)
    return t


def _hint_mode(tile_hint, exact_tile):
    if exact_tile:
        return False
    if tile_hint is not None:
        return bool(tile_hint)
    return os.environ.get("RSFA_TILE_HINT", "").strip().lower() in ("1", "true", "yes", "on")


_PLANS = {}
_TILING = None
# rsfa_fwd_args around a plan's constant parts: the pointers and workspace size,
# and the scale, are filled in per call
_PTR_OFF, _SHAPE_OFF = _native.FwdArgs.q.offset, _native.FwdArgs.z.offset
_SCALE_OFF, _FLAGS_OFF = _native.FwdArgs.sm_scale.offset, _native.FwdArgs.causal.offset
_POINTERS = struct.Struct("=7Q")  # q, k, v, o, lse, workspace, workspace_bytes
_SCALE = struct.Struct("=f")
assert _SHAPE_OFF - _PTR_OFF == _POINTERS.size and _FLAGS_OFF - _SCALE_OFF == _SCALE.size
_LAUNCH = None


def _launch_fn():
    """rsfa_attention_fwd taking the argument struct's bytes."""
    global _LAUNCH
    if _LAUNCH is None or _LAUNCH[0] is not _native.lib():
        lib = _native.lib()
        fn = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_char_p, ctypes.c_void_p)(("rsfa_attention_fwd", lib))
        _LAUNCH = (lib, fn)
    return _LAUNCH[1]


def _tiling_module():
    global _TILING
    if _TILING is None:
        _TILING = _package_module("tiling")
    return _TILING


def _make_plan(q_, k_, v_, o, v8, causal, BM, BN, hint, exact, split, static_schedule, single_blocks):
    """The launch arguments of a call but its pointers and scale (the bytes of
    rsfa_fwd_args before, between and after them), and the workspace bytes it
    needs; on the current device, which must be the tensors' device."""
    Z, H, N, D = q_.shape
    lib = _native.lib()
    # The tile is settled here and passed as a request, so the launch runs the
    # same tile the split workspace is sized for, and a get_tiling answer from a
    # measured cache is honoured.
    if (BM or BN) and not hint:
        bm, bn = resolve_tiling(D, causal, BM, BN, q_.dtype)
    else:
        if BM or BN:
            resolve_tiling(D, causal, BM, BN, q_.dtype)  # the reference's validity rules
        bm, bn = get_tiling(Z, H, N, D, causal, q_.dtype)
    args = _native.FwdArgs()
    args.struct_size = ctypes.sizeof(_native.FwdArgs)
    args.dtype = _native.DTYPE_F16_V8E5M2 if v8 else _DTYPES[q_.dtype]
    args.z, args.h, args.n_ctx, args.head_dim = Z, H, N, D
    for name, t in (("q_stride", q_), ("k_stride", k_), ("v_stride", v_), ("o_stride", o)):
        getattr(args, name)[:] = list(t.stride())
    args.causal = 1 if causal else 0
    args.block_m = bm
    args.block_n = bn
    args.flags = (_native.FLAG_EXACT_TILE if exact else 0) | (_native.FLAG_STATIC_SCHEDULE if static_schedule else 0) | (
        _native.FLAG_CAUSAL_SPLIT if (split and causal) else 0) | (
        _native.FLAG_SINGLE_BLOCKS if single_blocks else 0)
    nbytes = int(lib.rsfa_v8_workspace_bytes(Z, H, N, D)) if v8 else 0  # 0: the kernels read the bytes
    if split and causal:
        nbytes += split_workspace_bytes(Z, H, N, D, bm)
    b = bytes(args)
    return b[:_PTR_OFF], b[_SHAPE_OFF:_SCALE_OFF], b[_FLAGS_OFF:], nbytes


def _plan_key(q, k, v, out, *options):
    return (q.shape, k.shape, v.shape, q.stride(), k.stride(), v.stride(), q.dtype, k.dtype, v.dtype,
            q.device, k.device, v.device, None if out is None else out.stride(), options)


def forward(q, k, v, causal, sm_scale, BM=0, BN=0, *, return_lse=False, split=False,
            static_schedule=False, single_blocks=False, tile_hint=None, exact_tile=False, out=None):
    """Run the forward kernel; returns ``o`` or ``(o, lse)``.

    ``BM``/``BN`` keep the reference's meaning and validity rules (ValueError
    otherwise) and select the tile: the compiled tile nearest to the request
    runs (``resolve_tiling``); ``BM = BN = 0`` runs ``get_tiling``'s tile.
    ``tile_hint=True`` (default: the ``RSFA_TILE_HINT`` environment variable)
    only checks a request and runs ``get_tiling``'s tile; ``exact_tile=True``
    overrides hint mode and runs the requested tile's own kernel, where a request
    for ``get_tiling``'s tile may run a key-split variant of it on small grids.
    ``split=True`` (causal only) runs the reference's
    two-launch prefix/diagonal split, handing (m, l, acc) over in an fp32
    workspace;
    ``static_schedule=True`` replaces the dynamic task queue by the
    reference's grid-stride order, and ``single_blocks=True`` makes every
    causal task one query block instead of the pairs of blocks (nmb-1-i, i)
    the library otherwise uses when they fill whole rounds of the grid (results
    are bitwise identical either way).  ``lse`` is
    the natural-log logsumexp of the scaled scores, fp32 [Z, H, N].
    """
    hint = _hint_mode(tile_hint, exact_tile) if (BM or BN) else False
    exact = bool(exact_tile and (BM or BN))
    options = (bool(causal), int(BM), int(BN), hint, exact, bool(split), bool(static_schedule), bool(single_blocks))
    # The launch arguments but the pointers and the scale depend only on the
    # call's shapes, strides, types, devices and options: memoised while no
    # measured tiling cache is active (its answers may change between calls).  A
    # plan is kept for tensors that passed the checks below, so tensors with its
    # key need only their addresses checked (one 64-key tile: 15.2 -> 12.4 us
    # of host time per attention() call, the library's part of it included).
    memo = _tiling_module().active_cache() is None
    plan = _PLANS.get(_plan_key(q, k, v, None, *options)) if memo and out is None else None
    if plan is not None and not (q.data_ptr() | k.data_ptr() | v.data_ptr()) & 15:
        q_, k_, v_ = q, k, v
        o = torch.empty_like(q)
    else:
        if q.dim() != 4 or k.shape != q.shape or v.shape != q.shape:
            raise ValueError(f"q, k, v must share one 4-D shape [Z, H, N_CTX, D]; got "
                             f"{tuple(q.shape)}, {tuple(k.shape)}, {tuple(v.shape)}")
        # a float8 e5m2 V with float16 Q, K takes the reference's fp8_v branch (208-211)
        v8 = v.dtype == _FP8_E5M2 and q.dtype == torch.float16 and k.dtype == torch.float16
        if not v8 and not (q.dtype == k.dtype == v.dtype):
            raise TypeError("q, k and v must have the same dtype (or float16 q, k with a float8_e5m2 v)")
        if q.dtype not in _DTYPES:
            raise TypeError(f"unsupported dtype {q.dtype}; float16 and bfloat16 are supported")
        if not (q.is_cuda and k.is_cuda and v.is_cuda) or not (q.device == k.device == v.device):
            raise ValueError("q, k and v must be GPU tensors on one device")
        q_, k_, v_ = _as_kernel_layout(q), _as_kernel_layout(k), _as_kernel_layout(v)
        if out is None:
            o = torch.empty_like(q_)
        else:
            o = out
            if o.shape != q.shape or o.dtype != q.dtype or o.device != q.device or not _meets_contract(o):
                raise ValueError("out must match q's shape, dtype and device and have a unit-stride head dim")
        key = _plan_key(q_, k_, v_, out, *options) if memo else None
        plan = _PLANS.get(key) if memo else None
        if plan is None:
            if q.device.index == torch.cuda.current_device():
                plan = _make_plan(q_, k_, v_, o, v8, causal, BM, BN, hint, exact, split, static_schedule, single_blocks)
            else:
                with torch.cuda.device(q.device):
                    plan = _make_plan(q_, k_, v_, o, v8, causal, BM, BN, hint, exact, split, static_schedule, single_blocks)
            if memo:
                if len(_PLANS) > 4096:
                    _PLANS.clear()
                _PLANS[key] = plan
    head, mid, tail, nbytes = plan
    lse = torch.empty(q.shape[:3], dtype=torch.float32, device=q.device) if return_lse else None
    # workspace: the split state (a float8 V needs none)
    ws = torch.empty(nbytes // 4, dtype=torch.float32, device=q.device) if nbytes else None
    try:
        scale = _SCALE.pack(sm_scale)
    except (OverflowError, struct.error):  # past the float32 range, or a number by conversion
        scale = bytes(ctypes.c_float(float(sm_scale)))
    args = b"".join((head, _POINTERS.pack(q_.data_ptr(), k_.data_ptr(), v_.data_ptr(), o.data_ptr(),
                                          lse.data_ptr() if return_lse else 0,
                                          ws.data_ptr() if nbytes else 0, nbytes), mid, scale, tail))
    dev = q.device.index
    # (torch.cuda.current_stream wraps the same handle in a Stream object, 1.7 us)
    stream = torch._C._cuda_getCurrentRawStream(dev)
    if dev == torch.cuda.current_device():
        st = _launch_fn()(args, stream)
    else:
        with torch.cuda.device(q.device):
            st = _launch_fn()(args, stream)
    _raise_for(st)
    if out is not None and o is not out:
        out.copy_(o)
        o = out
    return (o, lse) if return_lse else o


# ============================================================================
# Same class name and apply alias as the reference (545-546, 619-622).
# ============================================================================
class _attention(torch.autograd.Function):

    @staticmethod
    def forward(ctx, q, k, v, causal, sm_scale, BM, BN):
        HEAD_DIM_Q, HEAD_DIM_K = q.shape[-1], k.shape[-1]
        HEAD_DIM_V = v.shape[-1]
        assert HEAD_DIM_Q == HEAD_DIM_K and HEAD_DIM_K == HEAD_DIM_V
        assert HEAD_DIM_K in {16, 32, 64, 128, 256}

        Z, H, N_CTX, HEAD_DIM = q.shape
        if causal:
            # the reference keeps a (1,) placeholder for the causal path (559-560)
            o = forward(q, k, v, True, sm_scale, BM, BN)
            M = torch.empty((1,), dtype=torch.float32, device=q.device)
        else:
            # non-causal writes the row logsumexp M = m + ln(l) (400-403)
            o, M = forward(q, k, v, False, sm_scale, BM, BN, return_lse=True)

        ctx.save_for_backward(q, k, v, o, M)
        ctx.sm_scale = sm_scale
        ctx.HEAD_DIM = HEAD_DIM_K
        ctx.causal = causal
        return o


attention = _attention.apply
