"""Row strides that the 64-key tiles of head dims 16 and 32 address stay accepted
beside the 128-key tiles, whose 32-bit offsets span twice the rows."""
import ctypes

import pytest
import torch

from ascend_rsfa import _native


@pytest.mark.parametrize("d", [16, 32])
@pytest.mark.parametrize("field", ["k_stride", "v_stride"])
# 63 rows of 34087040 elements end 2^32 bytes past the first; 16909320 are past a 128-key tile's reach
@pytest.mark.parametrize("stride,admitted", [(16909320, True), (34087032, True), (34087048, False)])
def test_row_strides_of_small_head_dims(d, field, stride, admitted):
    if admitted and torch.cuda.is_available():
        pytest.skip("a GPU is visible; the admitted call must end at the device query")
    a = _native.FwdArgs()
    a.struct_size = ctypes.sizeof(_native.FwdArgs)
    a.q, a.k, a.v, a.o = 0x1000, 0x2000, 0x3000, 0x4000
    a.z, a.h, a.n_ctx, a.head_dim = 1, 1, 2048, d
    for f in ("q_stride", "k_stride", "v_stride", "o_stride"):
        getattr(a, f)[:] = [2048 * d, 2048 * d, d, 1]
    getattr(a, field)[:] = [0, 0, stride, 1]
    a.sm_scale = 1.0
    want = _native.E_DEVICE if admitted else _native.E_ALIGN
    assert _native.lib().rsfa_attention_fwd(ctypes.byref(a), None) == want
