"""Key-split kernels (a task's keys shared by the wave groups of its workgroup) around
the edges of their key steps and query blocks, against the oracle and the static order.
Head counts are chosen so that the tile search picks the named number of groups on 256
CUs; test_dispatch_cpu.py checks that it does for every case here."""
import pytest
import torch

from ascend_rsfa.flash_attention_forward import forward
from oracle import attention as oracle

pytestmark = pytest.mark.gpu

# (head dim, key groups): 64-row blocks and four groups, or 128 rows and two
KINDS = [(128, 4), (128, 2), (64, 4), (64, 2), (32, 4)]
# heads that give two groups around 1024 keys, by (head dim, causal)
TWO_GROUPS = {(128, False): 20, (128, True): 32, (64, False): 20, (64, True): 28}


def _heads(d, groups, causal):
    return 2 if groups == 4 else TWO_GROUPS[d, causal]


# (head dim, groups, causal, keys, heads)
EDGES = [(d, g, c, n, _heads(d, g, c)) for d, g in KINDS for c in (False, True)
         for n in (1023, 1024, 1025, 1088, 1153, 1200)]
SHORT = [(d, 4, c, n, 4) for d, lengths in ((128, (130, 200, 257, 300, 385, 449, 513)),
                                            (64, (200, 257, 300, 385, 449, 513)), (32, (385, 449, 513)))
         for c in (False, True) for n in lengths]
SHORT += [(128, 2, c, n, h) for c, h in ((False, 40), (True, 56)) for n in (449, 513)] + [(64, 2, False, 449, 64)]
AT_1024 = [(d, g, c, 1024, _heads(d, g, c)) for d, g in KINDS for c in (False, True)]
PAIRS = [(128, 2, True, 2048, 32), (128, 4, True, 2048, 16), (64, 4, True, 4096, 8), (32, 4, True, 4096, 16)]
CASES = EDGES + SHORT + AT_1024 + PAIRS


def _check(q, k, v, causal, scale, o, lse):
    want = oracle.reference_attention(q, k, v, causal, scale)
    assert torch.allclose(o.float().cpu(), want, atol=1e-2, rtol=1e-2)
    s = (q.double() @ k.double().transpose(-1, -2)) * scale
    if causal:
        n = q.shape[2]
        s.masked_fill_(torch.ones(n, n, dtype=torch.bool).triu_(1), float("-inf"))
    # the row sum adds P rounded to the input type: relative 2^-9 (bfloat16) at worst
    assert (lse.cpu().double() - torch.logsumexp(s, -1)).abs().max() < 2.0 ** -8


@pytest.mark.parametrize("d,groups,causal,n,heads", EDGES)
def test_step_and_block_edges(d, groups, causal, n, heads):
    dtype = torch.bfloat16 if n % 2 else torch.float16
    q, k, v = (t.to(dtype) for t in oracle.make_inputs(1, heads, n, d, seed=n))
    scale = -0.7 * d ** -0.5 if n == 1088 else d ** -0.5
    qg, kg, vg = q.cuda(), k.cuda(), v.cuda()
    o, lse = forward(qg, kg, vg, causal, scale, return_lse=True)
    sel = slice(heads - 2, heads)
    _check(q[:, sel], k[:, sel], v[:, sel], causal, scale, o[:, sel], lse[:, sel])
    assert torch.equal(forward(qg, kg, vg, causal, scale, static_schedule=True), o)
    # [B, S, H, D] storage
    qs, ks, vs = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (qg, kg, vg))
    assert torch.equal(forward(qs, ks, vs, causal, scale), o)


@pytest.mark.parametrize("d,groups,causal,n,heads", SHORT)
def test_short_rows(d, groups, causal, n, heads):
    q, k, v = oracle.make_inputs(1, heads, n, d, seed=n)
    o, lse = forward(q.cuda(), k.cuda(), v.cuda(), causal, d ** -0.5, return_lse=True)
    sel = slice(heads - 4, heads)
    _check(q[:, sel], k[:, sel], v[:, sel], causal, d ** -0.5, o[:, sel], lse[:, sel])


@pytest.mark.parametrize("d,groups,causal,n,heads", PAIRS)
def test_paired_blocks(d, groups, causal, n, heads):
    q, k, v = oracle.make_inputs(1, heads, n, d, seed=d)
    qg, kg, vg = q.cuda(), k.cuda(), v.cuda()
    o, lse = forward(qg, kg, vg, causal, d ** -0.5, return_lse=True)
    assert torch.equal(forward(qg, kg, vg, causal, d ** -0.5, single_blocks=True), o)
    assert torch.equal(forward(qg, kg, vg, causal, d ** -0.5, static_schedule=True), o)
    sel = slice(heads - 1, heads)
    _check(q[:, sel], k[:, sel], v[:, sel], causal, d ** -0.5, o[:, sel], lse[:, sel])


@pytest.mark.parametrize("d,groups,causal,n,heads", AT_1024)
def test_peaked_rows_and_rescales(d, groups, causal, n, heads):
    # scores spread over hundreds of log2 units: every group's running max moves,
    # and most groups' factors in the merge are 0
    q, k, v = oracle.make_inputs(1, heads, n, d, seed=3)
    o, lse = forward(q.cuda(), k.cuda(), v.cuda(), causal, 4.0, return_lse=True)
    want = oracle.reference_attention(q[:, -2:], k[:, -2:], v[:, -2:], causal, 4.0)
    assert torch.allclose(o[:, -2:].float().cpu(), want, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("d,groups,causal,n,heads", AT_1024)
def test_nan_stays_in_its_rows(d, groups, causal, n, heads):
    bad = 700
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, heads, n, d, seed=5))
    want = forward(q, k, v, causal, 0.125)
    q[0, 0, bad] = float("nan")
    o = forward(q, k, v, causal, 0.125)
    rows = torch.isnan(o[0, 0]).any(-1).nonzero().flatten().tolist()
    assert rows == [bad] and torch.equal(o[0, 1:], want[0, 1:])
    q[0, 0, bad] = 0.0
    k[0, 0, bad] = float("nan")
    o = forward(q, k, v, causal, 0.125)
    seen = torch.isnan(o[0, 0]).any(-1)
    assert seen[bad if causal else 0:].all() and not (causal and seen[:bad].any())


@pytest.mark.parametrize("d,groups,causal,n,heads", AT_1024)
@pytest.mark.parametrize("lo,hi", [(20, 1024), (64, 128), (40, 900)])
def test_keys_scored_minus_infinity(d, groups, causal, n, heads, lo, hi):
    # keys lo .. hi - 1 score -inf through a channel (Q's last column 1, K's -inf there):
    # whole tiles of a key group, its first ones too, while other keys score finite
    q, k, v = oracle.make_inputs(1, heads, n, d, seed=lo)
    q[..., -1], k[..., -1] = 1.0, 0.0
    k[:, :, lo:hi, -1] = float("-inf")
    o, lse = forward(q.cuda(), k.cuda(), v.cuda(), causal, d ** -0.5, return_lse=True)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    _check(q[:, :2], k[:, :2], v[:, :2], causal, d ** -0.5, o[:, :2], lse[:, :2])


@pytest.mark.parametrize("d,groups,causal,n,heads", AT_1024)
def test_exact_tile_runs_the_plain_kernel(d, groups, causal, n, heads):
    # kept plans of one shape, with and without exact_tile, stay apart
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, heads, n, d, seed=11))
    split = forward(q, k, v, causal, d ** -0.5, 128, 64)
    exact = forward(q, k, v, causal, d ** -0.5, 128, 64, exact_tile=True)
    assert torch.equal(forward(q, k, v, causal, d ** -0.5, 128, 64), split)
    assert torch.equal(forward(q, k, v, causal, d ** -0.5), split)
    assert not torch.equal(exact, split)  # another order of summation
    want = oracle.reference_attention(q[:, -2:].cpu(), k[:, -2:].cpu(), v[:, -2:].cpu(), causal, d ** -0.5)
    for o in (exact, split):
        assert torch.allclose(o[:, -2:].float().cpu(), want, atol=1e-2, rtol=1e-2)
