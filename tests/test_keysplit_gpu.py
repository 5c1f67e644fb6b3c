"""Key-split kernels (a task's keys shared by the wave groups of its workgroup): few
heads, so that get_tiling's tile runs them, with lengths around the edges of their key
steps and query blocks, against the oracle and the static order."""
import pytest
import torch

from ascend_rsfa.flash_attention_forward import forward, get_tiling
from oracle import attention as oracle

pytestmark = pytest.mark.gpu

# (head dim, heads, tile): 2 heads take 64-row blocks and four key groups, 24 and 32
# heads 128 rows and two groups
SHAPES = [(128, 2, (128, 64)), (128, 32, (128, 64)), (64, 2, (128, 64)), (64, 24, (128, 64)), (32, 2, (128, 64))]


def _check(q, k, v, causal, scale, o, lse):
    want = oracle.reference_attention(q, k, v, causal, scale)
    assert torch.allclose(o.float().cpu(), want, atol=1e-2, rtol=1e-2)
    s = (q.double() @ k.double().transpose(-1, -2)) * scale
    if causal:
        n = q.shape[2]
        s.masked_fill_(torch.ones(n, n, dtype=torch.bool).triu_(1), float("-inf"))
    # the row sum adds P rounded to the input type: relative 2^-9 (bfloat16) at worst
    assert (lse.cpu().double() - torch.logsumexp(s, -1)).abs().max() < 2.0 ** -8


@pytest.mark.parametrize("d,heads,tile", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("n", [1023, 1024, 1025, 1088, 1153, 1200])
def test_step_and_block_edges(d, heads, tile, causal, n):
    if get_tiling(1, heads, n, d, causal) != tile:
        pytest.skip("another tile runs this shape")
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


@pytest.mark.parametrize("d,heads,tile", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("n", [130, 200, 257, 300, 385, 449, 513])
def test_short_rows(d, heads, tile, causal, n):
    q, k, v = oracle.make_inputs(1, min(heads, 4), n, d, seed=n)
    o, lse = forward(q.cuda(), k.cuda(), v.cuda(), causal, d ** -0.5, return_lse=True)
    _check(q, k, v, causal, d ** -0.5, o, lse)


@pytest.mark.parametrize("d", [32, 64, 128])
def test_peaked_rows_and_rescales(d):
    # scores spread over hundreds of log2 units: every group's running max moves,
    # and most groups' factors in the merge are 0
    n = 1024
    q, k, v = oracle.make_inputs(1, 2, n, d, seed=3)
    for causal in (False, True):
        o, lse = forward(q.cuda(), k.cuda(), v.cuda(), causal, 4.0, return_lse=True)
        want = oracle.reference_attention(q, k, v, causal, 4.0)
        assert torch.allclose(o.float().cpu(), want, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("causal", [False, True])
def test_nan_stays_in_its_rows(causal):
    n, bad = 1024, 700
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, 2, n, 128, seed=5))
    want = forward(q, k, v, causal, 0.125)
    q[0, 0, bad] = float("nan")
    o = forward(q, k, v, causal, 0.125)
    rows = torch.isnan(o[0, 0]).any(-1).nonzero().flatten().tolist()
    assert rows == [bad] and torch.equal(o[0, 1], want[0, 1])
    q[0, 0, bad] = 0.0
    k[0, 0, bad] = float("nan")
    o = forward(q, k, v, causal, 0.125)
    seen = torch.isnan(o[0, 0]).any(-1)
    assert seen[bad if causal else 0:].all() and not (causal and seen[:bad].any())


@pytest.mark.parametrize("d,heads,tile", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("lo,hi", [(20, 1024), (64, 128), (40, 900)])
def test_keys_scored_minus_infinity(d, heads, tile, causal, lo, hi):
    # keys lo .. hi - 1 score -inf through a channel (Q's last column 1, K's -inf there):
    # whole tiles of a key group, its first ones too, while other keys score finite
    n = 1024
    q, k, v = oracle.make_inputs(1, heads, n, d, seed=lo)
    q[..., -1], k[..., -1] = 1.0, 0.0
    k[:, :, lo:hi, -1] = float("-inf")
    o, lse = forward(q.cuda(), k.cuda(), v.cuda(), causal, d ** -0.5, return_lse=True)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    _check(q[:, :2], k[:, :2], v[:, :2], causal, d ** -0.5, o[:, :2], lse[:, :2])


@pytest.mark.parametrize("d,heads,tile", SHAPES)
@pytest.mark.parametrize("causal", [False, True])
def test_exact_tile_runs_the_plain_kernel(d, heads, tile, causal):
    # kept plans of one shape, with and without exact_tile, stay apart
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, heads, 1024, d, seed=11))
    split = forward(q, k, v, causal, d ** -0.5, *tile)
    exact = forward(q, k, v, causal, d ** -0.5, *tile, exact_tile=True)
    assert torch.equal(forward(q, k, v, causal, d ** -0.5, *tile), split)
    assert torch.equal(forward(q, k, v, causal, d ** -0.5), split)
    assert not torch.equal(exact, split)  # another order of summation
    want = oracle.reference_attention(q[:, -2:].cpu(), k[:, -2:].cpu(), v[:, -2:].cpu(), causal, d ** -0.5)
    for o in (exact, split):
        assert torch.allclose(o[:, -2:].float().cpu(), want, atol=1e-2, rtol=1e-2)
