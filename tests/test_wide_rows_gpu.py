"""Calls whose rows lie too far apart for the 32-bit load offsets of the kernel their
shape runs: they run a kernel that reaches them, bitwise as on contiguous rows."""
import pytest
import torch

from ascend_rsfa.flash_attention_forward import forward
from oracle import attention as oracle

pytestmark = pytest.mark.gpu


def _spread(t, stride):
    """t [1, 1, N, D] with its rows `stride` elements apart."""
    n, d = t.shape[2:]
    flat = torch.empty((n - 1) * stride + d, dtype=t.dtype, device=t.device)
    return flat.as_strided(t.shape, (n * stride, n * stride, stride, 1)).copy_(t)


@pytest.mark.parametrize("d", [16, 32])
@pytest.mark.parametrize("which", [1, 2])
@pytest.mark.parametrize("v8", [False, True])
def test_128_key_tile_hands_over_to_64(d, which, v8):
    # 127 rows of 16909328 two-byte elements end past 2^32 bytes, 63 do not
    ts = [t.cuda() for t in oracle.make_inputs(1, 1, 130, d, seed=d + which)]
    if v8:
        ts[2] = ts[2].to(torch.float8_e5m2)
    want = forward(*ts, False, 0.25, 128, 64, exact_tile=True)
    ts[which] = _spread(ts[which], 16909328)
    assert torch.equal(forward(*ts, False, 0.25, 128, 128), want)
    assert torch.equal(forward(*ts, False, 0.25), want)
    assert torch.equal(forward(*ts, False, 0.25, 128, 128, exact_tile=True), want)


@pytest.mark.parametrize("causal", [False, True])
def test_key_split_hands_over_to_the_plain_tile(causal):
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs a 26 GB view")
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, 1, 385, 32, seed=3))
    want = forward(q, k, v, causal, 0.25, 128, 64, exact_tile=True)
    assert not torch.equal(forward(q, k, v, causal, 0.25), want)  # contiguous: the key-split kernel
    wide = _spread(q, 34087048)
    # (out=: the output would take Q's strides, and their size)
    for tile in ((0, 0), (128, 64)):
        assert torch.equal(forward(wide, k, v, causal, 0.25, *tile, out=torch.empty_like(v)), want)
    del wide
    torch.cuda.empty_cache()
