"""Which kernels the C ABI launches for a call, recorded on the CPU for 256 CUs
(tests/launch_recorder.py)."""
import pytest

from ascend_rsfa import _native
from launch_recorder import record

# (head dim, heads, causal) at 1024 keys: shapes whose search answers a key-split variant of (128, 64)
KEYSPLIT = [(128, 16, 1), (128, 32, 0), (128, 32, 1), (64, 16, 1), (64, 24, 0), (32, 2, 0), (32, 2, 1)]


@pytest.mark.parametrize("entry", ["rsfa_attention_fwd", "rsfa_attention_fwd_noalloc"])
def test_exact_requests_run_the_plain_kernel(tmp_path, entry):
    calls = []
    for d, heads, causal in KEYSPLIT:
        base = dict(heads=heads, n=1024, d=d, causal=causal, entry=entry)
        tile = dict(base, block_m=128, block_n=64)
        calls += [base, tile, dict(tile, flags=_native.FLAG_EXACT_TILE), dict(tile, flags=_native.FLAG_TILE_HINT),
                  dict(tile, flags=_native.FLAG_TILE_HINT | _native.FLAG_EXACT_TILE)]
    got = record(calls, tmp_path)
    assert all(st == _native.OK for st, _ in got)
    runs = [[x for x in launches if x.kernel != "clear"] for _, launches in got]
    assert all(len(r) == 1 for r in runs)
    for i, (d, heads, causal) in enumerate(KEYSPLIT):
        none, request, exact, hint, exact_hint = (r[0] for r in runs[5 * i:5 * i + 5])
        for x in (none, request, hint):
            assert x.kernel == "keysplit" and x.params["d"] == d and x.params["causal"] == causal
            assert x.params == none.params
        for x in (exact, exact_hint):
            assert x.kernel == "fa" and x.params == {"d": d, "bn": 64, "nw": 4, "causal": causal, "mode": 0}
