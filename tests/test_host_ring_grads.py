"""CPU tests of a ring's gradient accumulators when a caller puts tensors of its own in their place (chunks that travel take theirs along)."""
import copy

import pytest
import torch

import lightron_amd as la


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_replaced_accumulators_are_the_ones_that_count(dtype):
    kv = [tuple(torch.zeros(1, n, 2, 8, dtype=dtype) for _ in range(2)) for n in (5, 7)]
    acc = la.RingKVGrads(kv)
    acc.dk[1] = torch.full((1, 7, 2, 8), 3.0)
    acc.dv = [torch.full(v.shape, 5.0) for _, v in kv]
    acc.dk[0].fill_(2.0)
    (k0, v0), (k1, v1) = acc.finalize(assign=False)
    assert all(t.dtype == dtype for t in (k0, v0, k1, v1))
    assert (k0 == 2).all() and (k1 == 3).all() and (v0 == 5).all() and (v1 == 5).all()
    acc.zero_()
    assert all((t == 0).all() for t in (*acc.dk, *acc.dv))


def test_copies_keep_one_buffer():
    kv = [tuple(torch.zeros(1, n, 2, 8) for _ in range(2)) for n in (5, 7)]
    acc = copy.deepcopy(la.RingKVGrads(kv))
    assert acc._whole() is acc._buf
    for t in (*acc.dk, *acc.dv):
        t.fill_(1.0)
    acc.zero_()
    assert all((t == 0).all() for t in (*acc.dk, *acc.dv)) and acc.dk[1].data_ptr() > acc._buf.data_ptr()
