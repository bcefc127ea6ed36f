"""CPU test of the sizes that ltr_attn_bwd_delta takes."""
import ctypes

import pytest
import torch

from lightron_amd import _lib as L


@pytest.mark.skipif(torch.cuda.is_available(), reason="the pointers are not memory: only without a device does the call stop before its launch")
@pytest.mark.parametrize("B,Sq,Hq,rc", [(65536, 65536, 1, -5), (1, 64, 4, -5), (3, (1 << 31) - 2, 1, -5), (1, 1 << 31, 1, -1)])
def test_more_rows_than_32_bits_count(B, Sq, Hq, rc):
    """Valid sizes get as far as the device check (batch entries may share their memory: strides of zero)."""
    a = L.DeltaArgs()
    a.o = a.d_o = a.delta = 4096
    a.B, a.Hq, a.D, a.Sq, a.o_dtype, a.do_dtype = B, Hq, 64, Sq, L.LTR_BF16, L.LTR_BF16
    assert L.load().ltr_attn_bwd_delta(ctypes.byref(a), None) == rc
