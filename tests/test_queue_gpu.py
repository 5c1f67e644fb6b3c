"""First tickets by rank, and launches without a queue: task counts just below, at and
just past one per workgroup, launched repeatedly on one stream (each launch must leave
the queue's counters at zero), against the static order bitwise."""
import pytest
import torch

from ascend_rsfa.flash_attention_forward import forward, get_num_compute_cores
from oracle import attention as oracle

pytestmark = pytest.mark.gpu


# (head dim, tile, workgroups per CU): the 4-wave tiles run two workgroups on a CU
@pytest.mark.parametrize("d,tile,per_cu", [(128, (256, 64), 1), (64, (256, 128), 1), (256, (256, 32), 1),
                                           (128, (128, 64), 2)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("extra", [-8, 0, 8, 3])
def test_tickets_around_one_per_workgroup(d, tile, per_cu, causal, extra):
    heads = get_num_compute_cores() * per_cu // 2 + extra  # two query blocks per head
    n = tile[0] + 24
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, heads, n, d, seed=7 + extra))
    want = forward(q, k, v, causal, 0.125, *tile, exact_tile=True, static_schedule=True)
    for _ in range(3):
        assert torch.equal(forward(q, k, v, causal, 0.125, *tile, exact_tile=True), want)
    ref = oracle.reference_attention(q[:, -2:].cpu(), k[:, -2:].cpu(), v[:, -2:].cpu(), causal, 0.125)
    assert torch.allclose(want[:, -2:].float().cpu(), ref, atol=1e-2, rtol=1e-2)
