"""Which kernels a call of the C ABI launches, without a GPU.

A child process loads tests/launch_recorder.cpp (the HIP entry points the library
calls, recording launches) ahead of librsfa.so, runs the given calls and prints
the recorded launches.  ``record`` returns one list of ``Launch`` per call.
"""
import collections
import json
import os
import re
import subprocess
import sys

_TESTS = os.path.dirname(os.path.abspath(__file__))
_PKG = os.path.join(os.path.dirname(_TESTS), "ascend-rsfa_amd", "ascend_rsfa")

# kernel: "fa" (d, bn, nw, causal, mode), "keysplit" (d, keys, groups, causal) or "clear"
Launch = collections.namedtuple("Launch", "kernel params grid threads pairs counters")

# FwdParams: 7 pointers, 12 strides, 7 ints (the last: pairs), c, neg, (4 bytes up to) the counters
_PAIRS_OFFSET = 7 * 8 + 12 * 8 + 6 * 4
_TICKET_OFFSET = _PAIRS_OFFSET + 3 * 4 + 4


def _parse(line):
    name, grid, threads, pairs, counters = line.rsplit(" ", 4)
    nums = [int(x) for x in re.findall(r"L[ib](\d+)E", name)]
    if "clear_words" in name:
        kind, params = "clear", {}
    elif "keysplit" in name:
        kind, params = "keysplit", dict(zip(("d", "keys", "groups", "causal"), nums))
    else:
        kind, params = "fa", dict(zip(("d", "bn", "nw", "causal", "mode"), nums))
    return Launch(kind, params, int(grid), int(threads), int(pairs), counters)


def record(calls, tmp_path, occupancy=()):
    """Runs ``calls`` in turn: dicts of rsfa_fwd_args fields, with ``heads``, ``n``
    and ``d`` for contiguous tensors and optionally ``entry``, ``capturing``,
    ``stream`` and ``tiling`` (block_m, block_n from rsfa_get_tiling).  ``occupancy``: (part of a
    kernel's mangled name, workgroups per CU).  Returns [(status, [Launch])]."""
    so = os.path.join(str(tmp_path), "librecorder.so")
    if not os.path.exists(so):
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-DRECORDER_TICKET_OFFSET={_TICKET_OFFSET}",
                        f"-DRECORDER_PAIRS_OFFSET={_PAIRS_OFFSET}", "-o", so, os.path.join(_TESTS, "launch_recorder.cpp")], check=True)
    spec = json.dumps({"so": so, "pkg": _PKG, "calls": list(calls), "occupancy": list(occupancy)})
    out = subprocess.run([sys.executable, os.path.abspath(__file__)], input=spec, text=True, capture_output=True,
                         timeout=120)
    assert out.returncode == 0, out.stderr
    return [(st, [_parse(x) for x in lines]) for st, lines in json.loads(out.stdout.splitlines()[-1])]


def _child():
    import ctypes
    import importlib.util

    spec = json.load(sys.stdin)
    rec = ctypes.CDLL(spec["so"], mode=ctypes.RTLD_GLOBAL)
    rec.recorder_lines.restype = ctypes.c_char_p
    mod = importlib.util.spec_from_file_location("_native", os.path.join(spec["pkg"], "_native.py"))
    native = importlib.util.module_from_spec(mod)
    mod.loader.exec_module(native)
    lib = native.lib()
    for part, wgs in spec["occupancy"]:
        rec.recorder_occupancy(part.encode(), wgs)
    results = []
    for call in spec["calls"]:
        heads, n, d = call.pop("heads"), call.pop("n"), call.pop("d")
        entry = call.pop("entry", "rsfa_attention_fwd")
        rec.recorder_capturing(int(call.pop("capturing", 0)))
        stream = call.pop("stream", None)
        a = native.FwdArgs()
        a.struct_size = ctypes.sizeof(a)
        a.q = a.k = a.v = a.o = a.workspace = 0x1000
        a.workspace_bytes = 1 << 40
        a.z, a.h, a.n_ctx, a.head_dim, a.sm_scale = 1, heads, n, d, 0.5
        for f in ("q_stride", "k_stride", "v_stride", "o_stride"):
            getattr(a, f)[:] = [heads * n * d, n * d, d, 1]
        tiling = call.pop("tiling", False)
        for f, x in call.items():
            if f.endswith("_stride"):
                getattr(a, f)[:] = x
            else:
                setattr(a, f, x)
        if tiling:
            bm, bn = ctypes.c_int32(), ctypes.c_int32()
            assert lib.rsfa_get_tiling(1, heads, n, d, a.causal, a.dtype, ctypes.byref(bm), ctypes.byref(bn)) == 0
            a.block_m, a.block_n = bm.value, bn.value
        rec.recorder_clear()
        st = getattr(lib, entry)(ctypes.byref(a), ctypes.c_void_p(stream))
        results.append((st, rec.recorder_lines().decode().splitlines()))
    print(json.dumps(results))


if __name__ == "__main__":
    _child()
