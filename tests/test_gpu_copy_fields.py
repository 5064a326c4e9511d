"""Several device arrays copied in one launch: lengths around a block and past
the grid's stride, arrays of different lengths, an empty one.  Exact."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (255, 256, 257), (0, 5, 1024 * 256 + 3), (7,) * 8])
def test_copy_fields(sizes):
    import torch
    from pybella_amd import _abi
    print(f"case copy fields {sizes}", flush=True)
    ctx = _abi.default_context()
    ctx.sync_stream()
    src = [torch.randn(n + 1, dtype=torch.float64, device="cuda") for n in sizes]
    dst = [torch.full((n + 1,), 7.0, dtype=torch.float64, device="cuda") for n in sizes]
    k = len(sizes)
    P = lambda ts: (C.c_void_p * k)(*[t.data_ptr() for t in ts])
    ctx.check(ctx.lib.pb_copy_fields(ctx.h, k, P(src), P(dst), (C.c_int64 * k)(*sizes)))
    for n, s, d in zip(sizes, src, dst):
        assert torch.equal(d[:n], s[:n]) and float(d[n]) == 7.0
    assert ctx.lib.pb_copy_fields(ctx.h, 9, P(src), P(dst), (C.c_int64 * k)(*sizes)) < 0
