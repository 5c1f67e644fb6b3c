"""Which kernels the C ABI launches for a call, recorded on the CPU for 256 CUs
(tests/launch_recorder.py)."""
import pytest

import test_keysplit_gpu
import test_parity_gpu
import test_streams_gpu
import test_zz_no_alloc
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


# a split call whose prefix launch has a workgroup per task and whose diagonal launch has not,
# and the other way round, and neither
@pytest.mark.parametrize("prefix,diag", [(2, 1), (1, 2), (1, 1)])
@pytest.mark.parametrize("d", [16, 64])
def test_callers_counters_are_cleared_before_their_first_use(tmp_path, prefix, diag, d):
    call = dict(heads=160, n=200, d=d, causal=1, entry="rsfa_attention_fwd_noalloc",
                flags=_native.FLAG_CAUSAL_SPLIT, block_m=128, block_n=64)  # 320 tasks
    # (part of the kernel's mangled name: causal, mode)
    ((st, launches),) = record([call], tmp_path, [("Lb1ELi1E", prefix), ("Lb1ELi2E", diag)])
    assert st == _native.OK
    runs = [x for x in launches if x.kernel == "fa"]
    assert [x.params["mode"] for x in runs] == [1, 2]
    assert [x.counters for x in runs] == ["scratch" if 320 > 256 * w else "none" for w in (prefix, diag)]
    first = next(i for i, x in enumerate(launches) if x.kernel == "fa" and x.counters == "scratch")
    assert [x.kernel for x in launches[:first]].count("clear") == 1
    assert [x.kernel for x in launches].count("clear") == 1
    assert all(x.counters == "scratch" for x in launches if x.kernel == "clear")


def test_rows_past_a_kernels_reach_run_its_stand_in(tmp_path):
    far = 16909320   # past a 128-key tile's 32-bit offsets, within a 64-key tile's
    wide = 34087048  # past a 64-key tile's too: for Q at head dim 32 only the key-split loader's
    calls, want = [], []
    for d in (16, 32):
        near = dict(heads=64, n=2048, d=d, dtype=_native.DTYPE_F16)
        calls += [near, dict(near, k_stride=[0, 0, far, 1]), dict(near, v_stride=[0, 0, far, 1]),
                  dict(near, block_m=128, block_n=128, k_stride=[0, 0, far, 1]),
                  dict(near, block_m=128, block_n=128, v_stride=[0, 0, far, 1], flags=_native.FLAG_EXACT_TILE)]
        want += [("fa", 128)] + 4 * [("fa", 64)]
    for causal in (0, 1):
        split = dict(heads=1, n=385, d=32, causal=causal)
        calls += [split, dict(split, q_stride=[0, 0, wide, 1]),
                  dict(split, q_stride=[0, 0, wide, 1], block_m=128, block_n=64)]
        want += [("keysplit", 64), ("fa", 64), ("fa", 64)]
    got = record(calls, tmp_path)
    assert [(st, [x.kernel for x in launches]) for st, launches in got] == [(_native.OK, [k]) for k, _ in want]
    keys = [launches[0].params.get("bn", launches[0].params.get("keys")) for _, launches in got]
    assert keys == [k for _, k in want]


# at least the workgroups that fit a CU: one of 8 waves, as many of 4 as a SIMD holds waves of the smallest tiles
FULL = [("Li8ELb", 1), ("Li4ELb", 4), ("keysplit", 1)]


def _queued_calls():
    for z, h, n, d in test_parity_gpu.QUEUED + test_streams_gpu.QUEUED:
        for causal in (0, 1):
            yield dict(heads=z * h, n=n, d=d, causal=causal)
    codes = {"v8": _native.DTYPE_F16_V8E5M2, "torch.float16": _native.DTYPE_F16, "torch.bfloat16": _native.DTYPE_BF16}
    for (z, h, n, d), _, causal, dtype, flags in test_zz_no_alloc.QUEUED_CASES:
        yield dict(heads=z * h, n=n, d=d, causal=int(causal), flags=flags, dtype=codes[str(dtype)])


def test_queued_shapes_take_counters_and_captured_streams_none(tmp_path):
    calls = [dict(c, entry=e, capturing=cap, stream=stream) for c in _queued_calls()
             for e in ("rsfa_attention_fwd", "rsfa_attention_fwd_noalloc")
             for cap, stream in ((0, None), (1, None), (0, 2))]  # 2: hipStreamPerThread
    for call, (st, launches) in zip(calls, record([dict(c) for c in calls], tmp_path, FULL)):
        assert st == _native.OK, call
        runs = [x for x in launches if x.kernel != "clear"]
        assert len(runs) == (2 if call.get("flags") else 1)
        if call["entry"] == "rsfa_attention_fwd_noalloc":
            want = "scratch"  # the call's own counters: under capture too
            assert launches[0].kernel == "clear" and len(launches) == len(runs) + 1
        else:
            want = "none" if call["capturing"] or call["stream"] else "allocated"
        assert {x.counters for x in runs} == {want}, call


def test_keysplit_cases_run_the_groups_they_name(tmp_path):
    cases = test_keysplit_gpu.CASES
    calls = [dict(heads=h, n=n, d=d, causal=int(c), **tile) for d, _, c, n, h in cases
             for tile in ({}, {"block_m": 128, "block_n": 64})]
    got = record(calls, tmp_path, FULL)
    for (st, launches), case in zip(got, [c for c in cases for _ in range(2)]):
        (x,) = [x for x in launches if x.kernel != "clear"]
        assert st == _native.OK and x.kernel == "keysplit" and x.params["groups"] == case[1], case
        assert not (case in test_keysplit_gpu.PAIRS) or x.pairs, case
    assert any(x.counters != "none" for _, launches in got for x in launches)  # some of them queued


def test_two_workgroups_per_cu_for_long_pairs_in_two_rounds_only(tmp_path):
    # head dim 32, four workgroups per CU: (heads, keys, workgroups)
    cases = [(32, 8192, 1024), (64, 8192, 512), (96, 8192, 1024), (128, 8192, 1024), (128, 4096, 512), (64, 4096, 1024),
             (256, 2048, 1024), (32, 16384, 512)]
    dtypes = (_native.DTYPE_F16, _native.DTYPE_BF16, _native.DTYPE_F16_V8E5M2)
    got = record([dict(heads=h, n=n, d=32, causal=1, dtype=dt) for h, n, _ in cases for dt in dtypes], tmp_path, FULL)
    for (st, (x,)), (h, n, grid, dt) in zip(got, [c + (dt,) for c in cases for dt in dtypes]):
        assert st == _native.OK and x.pairs == 1 and x.params["nw"] == 4
        assert x.grid == (1024 if dt == _native.DTYPE_F16_V8E5M2 else grid), (h, n, dt)


def test_few_rounds_of_equal_tasks_take_no_counters(tmp_path):
    # (head dim, heads, keys, causal, takes counters), three or four workgroups per CU at head dims 16 and 32
    cases = [(32, 20, 8192, 0, False), (16, 32, 8192, 0, False), (32, 36, 6348, 0, True), (32, 40, 8192, 0, True),
             (32, 24, 8192, 0, False), (32, 256, 777, 0, False), (32, 512, 777, 0, True), (16, 1024, 333, 0, True),
             (32, 20, 16384, 1, True), (64, 20, 8192, 0, True)]
    got = record([dict(heads=h, n=n, d=d, causal=c) for d, h, n, c, _ in cases], tmp_path,
                 [("Li64ELi4ELb", 4), ("Li128ELi4ELb", 3)])
    for (st, (x,)), case in zip(got, cases):
        assert st == _native.OK and (x.counters != "none") == case[4], case
