"""The work this framework is measured on: FlashAttention-2 forward calls.

Every case is one call of a public entry point, ``attention(q, k, v, causal,
sm_scale, BM, BN)`` with the tile ``get_tiling`` gives for the shape, or
``forward(..., return_lse=True)`` for callers that keep the row logsumexp, on
inputs resident on the GPU.  The cases are attention layers as they occur: from
a single 64-key tile, where the launch and the host call are all there is, over
short and ragged batches and batch-1 prefill, to the largest benchmark shapes;
every head dim class, both masks, float16, bfloat16 and a float8_e5m2 V,
[Z, H, N, D] tensors and [Z, N, H, D] ones seen through a transpose.

A case holds the shape (Z, H, N, D), ``causal``, ``dtype`` ("f16", "bf16", or
"f16v8" for float16 Q and K with a float8_e5m2 V), ``layout`` ("bhsd" or
"bshd"), ``lse`` (the call returns the row logsumexp too), the standard
deviation ``std`` of the inputs and the softmax ``scale``.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ascend-rsfa_amd"))

from ascend_rsfa.flash_attention_forward import attention, forward, get_tiling  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f16v8": torch.float16}


def _case(Z, H, N, D, causal, dtype="f16", layout="bhsd", lse=False, std=1.0, scale=None, name=None):
    c = {"Z": Z, "H": H, "N": N, "D": D, "causal": causal, "dtype": dtype, "layout": layout, "lse": lse,
         "std": std, "scale": 1.0 / math.sqrt(D) if scale is None else scale}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # a single key tile: the smallest call, all latency
        _case(1, 8, 64, 64, False, name="one-tile"),
        # a batch of short sequences of no round length (an encoder's layer), bfloat16
        _case(4, 32, 197, 64, False, "bf16", "bshd", name="short-ragged"),
        # two causal sequences of 1024 keys, 8 heads: a small prefill
        _case(2, 8, 1024, 128, True, scale=0.5, name="prefill-2x1024"),
        # one prompt of 2048 tokens through a 32-head layer, tensors as a projection leaves them
        _case(1, 32, 2048, 128, True, "bf16", "bshd", name="prefill-1x2048"),
        # one long prompt on few heads (one tensor-parallel shard of a layer)
        _case(1, 8, 8192, 128, True, "bf16", name="long-1x8192"),
        # a causal layer of ragged length whose caller keeps the logsumexp
        _case(8, 16, 1531, 128, True, "bf16", lse=True, name="ragged-lse"),
        # a non-causal layer with a small head dim
        _case(32, 8, 2048, 32, False, name="small-head"),
        # long causal sequences at head dim 64
        _case(4, 16, 8192, 64, True, name="long-d64"),
        # a causal layer with a wide head
        _case(64, 8, 1024, 256, True, name="wide-head"),
        # a float8 V cache
        _case(32, 8, 2048, 128, False, "f16v8", name="float8-v"),
        # the causal benchmark shape
        _case(128, 8, 2048, 128, True, scale=0.5, name="large-causal"),
        # the non-causal benchmark shape, the largest
        _case(128, 8, 2048, 128, False, name="large"),
    ]


# the largest listed case's cost, with head dims below 128 counted as 128 (their softmax costs as much)
_MAX_COST = 128 * 8 * 2048 * 2048 * 128
_MAX_ELEMS = 128 * 8 * 2048 * 128


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        D = rng.choice([16, 32, 64, 64, 128, 128, 128, 256])
        N = _log_int(rng, 33, 8192)
        if rng.random() < 0.4:  # round lengths are common, odd ones too
            N = max(64, N // 64 * 64)
        Z = _log_int(rng, 1, 128)
        H = rng.choice([4, 6, 8, 12, 16, 32])
        causal = rng.random() < 0.5
        cost = Z * H * N * N * max(D, 128) * (0.5 if causal else 1.0)
        if cost > 0.5 * _MAX_COST or Z * H * N * D > _MAX_ELEMS:
            continue
        dtype = rng.choice(["f16", "f16", "bf16", "bf16", "f16v8"])
        layout = rng.choice(["bhsd", "bshd"])
        std, scale = rng.choice([(1.0, 1.0 / math.sqrt(D)), (0.5, 0.5)])
        return _case(Z, H, N, D, causal, dtype, layout, rng.random() < 0.3, std, scale)


def _inputs(case, seed):
    Z, H, N, D = case["Z"], case["H"], case["N"], case["D"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    ts = []
    for i in range(3):
        shape = (Z, N, H, D) if case["layout"] == "bshd" else (Z, H, N, D)
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, case["std"], generator=g)
        t = t.to(torch.float8_e5m2 if i == 2 and case["dtype"] == "f16v8" else DTYPES[case["dtype"]])
        ts.append(t.transpose(1, 2) if case["layout"] == "bshd" else t)
    return ts


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    Z, H, N, D = q.shape
    return {"q": q, "k": k, "v": v, "causal": case["causal"], "scale": case["scale"], "lse": case["lse"],
            "tile": get_tiling(Z, H, N, D, case["causal"], q.dtype)}


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    if state["lse"]:
        return forward(q, k, v, state["causal"], state["scale"], return_lse=True)
    return attention(q, k, v, state["causal"], state["scale"], *state["tile"])


def work(case):
    Z, H, N, D = case["Z"], case["H"], case["N"], case["D"]
    v_bytes = 1 if case["dtype"] == "f16v8" else 2
    # Q, K, V read and O written once; attention() keeps the logsumexp of non-causal calls
    nbytes = Z * H * N * D * (6 + v_bytes) + (4 * Z * H * N if case["lse"] or not case["causal"] else 0)
    pairs = N * (N + 1) // 2 if case["causal"] else N * N
    return {"bytes": nbytes, "flops": 4 * Z * H * pairs * D}


def tolerance(case):
    # P and O are rounded to the input type (a float8_e5m2 V rounds P to 2 fraction
    # bits); against exact() the outputs differ by up to 3.0e-4 (float16), 2.2e-3
    # (bfloat16) and 5.2e-2 (float8 V): four times that
    return {"rel": {"f16": 1.2e-3, "bf16": 9e-3, "f16v8": 0.2}[case["dtype"]]}


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    Z, H, N, D = q.shape
    o = torch.empty((Z * H, N, D), dtype=torch.float64, device="cuda")
    lse = torch.empty((Z * H, N), dtype=torch.float64, device="cuda")
    q, k, v = (t.reshape(Z * H, N, D) for t in (q, k, v))
    step = max(1, (1 << 27) // (N * N))  # heads at a time: 1 GiB of scores
    hidden = torch.ones((N, N), dtype=torch.bool, device="cuda").triu_(1) if case["causal"] else None
    for i in range(0, Z * H, step):
        s = torch.bmm(q[i:i + step].double(), k[i:i + step].double().transpose(1, 2).contiguous())
        s.mul_(case["scale"])
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        lse[i:i + step] = torch.logsumexp(s, -1)
        s.sub_(lse[i:i + step, :, None]).exp_()
        o[i:i + step] = torch.bmm(s, v[i:i + step].double())
    o = o.reshape(Z, H, N, D)
    return (o, lse.reshape(Z, H, N)) if case["lse"] else o
