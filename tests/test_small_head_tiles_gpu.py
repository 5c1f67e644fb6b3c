"""The 128-key tiles of head dims 16 and 32 (three waves per SIMD, non-causal) around
their tile edges, against the oracle."""
import pytest
import torch

from ascend_rsfa.flash_attention_forward import forward, resolve_tiling
from oracle import attention as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [16, 32])
@pytest.mark.parametrize("n", [1, 127, 128, 129, 255, 257, 520])
@pytest.mark.parametrize("dtype", ["f16", "bf16", "v8"])
def test_128_key_tile_edges(d, n, dtype):
    assert resolve_tiling(d, False, 128, 128) == (128, 128)
    q, k, v = oracle.make_inputs(1, 3, n, d, seed=n)
    if dtype == "bf16":
        q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    v_in = v.to(torch.float8_e5m2) if dtype == "v8" else v
    o, lse = forward(q.cuda(), k.cuda(), v_in.cuda(), False, d ** -0.5, 128, 128, return_lse=True)
    o = o.float().cpu()
    if dtype == "v8":
        # per element: every P rounded to two fraction bits
        want = oracle.reference_attention_fp8v(q, k, v_in, False, d ** -0.5)
        bound = oracle.fp8v_error_bound(q, k, v_in, False, d ** -0.5)
        assert ((o - want).abs() <= bound).all()
    else:
        want = oracle.reference_attention(q, k, v, False, d ** -0.5)
        assert torch.allclose(o, want, atol=1e-2, rtol=1e-2)
    s = (q.double() @ k.double().transpose(-1, -2)) * d ** -0.5
    # the row sum adds P rounded to the input type (relative 2^-9 at worst, bfloat16)
    assert (lse.cpu().double() - torch.logsumexp(s, -1)).abs().max() < 2.0 ** -8
