"""Causal calls whose last query block is partial: a NaN in the K or V of a key that a
row does not see leaves the row alone, down to the 32-key sub-tile the key is in."""
import pytest
import torch

from ascend_rsfa.flash_attention_forward import forward
from oracle import attention as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,tile", [(64, (256, 128)), (128, (256, 64)), (256, (256, 32))])
@pytest.mark.parametrize("n", [456, 650])
def test_nan_key_in_a_partial_query_block(d, tile, n):
    bad = n // tile[1] * tile[1] - 10  # in the block's last whole key tile
    first = bad // 32 * 32             # rows before it run no step of the key's sub-tile
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, 3, n, d, seed=n))
    want = forward(q, k, v, True, 0.125, *tile, exact_tile=True)
    for t in (k, v):
        keep = t[0, 1, bad].clone()
        t[0, 1, bad] = float("nan")
        o = forward(q, k, v, True, 0.125, *tile, exact_tile=True)
        assert torch.equal(o[:, 0], want[:, 0]) and torch.equal(o[:, 2], want[:, 2])
        assert torch.equal(o[0, 1, :first], want[0, 1, :first])
        assert torch.isnan(o[0, 1, bad:]).all()
        t[0, 1, bad] = keep
