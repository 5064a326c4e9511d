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


def test_model_copies_of_other_arrays():
    """time_update.copy_fields hands raw pointers on only for contiguous FP64
    arrays of one shape: strides and types are torch's, a size that differs is
    refused, and the arrays around stay as they are."""
    import types

    import torch
    from pybella_amd import _abi
    from pybella_amd import time_update as tu
    print("case copy fields of a model", flush=True)
    M = types.SimpleNamespace(ctx=_abi.default_context())
    M.ctx.sync_stream()
    a, b = torch.randn(7, 9, dtype=torch.float64, device="cuda"), torch.randn(9, 7, dtype=torch.float64, device="cuda")
    new = lambda *s, **k: torch.full(s, 7.0, **{"dtype": torch.float64, "device": "cuda", **k})
    for dst in ((new(7, 9), new(9, 7)), (new(7, 18)[:, ::2], new(9, 7)), (new(7, 9), new(9, 7, dtype=torch.float32)),
                (new(9, 7).t(), new(7, 9).t()), (new(7, 9, device="cpu"), new(9, 7))):
        tu.copy_fields(M, [a, b], dst)
        for s, d in zip((a, b), dst):
            assert torch.equal(d.cpu(), s.to(d.dtype).cpu())
    for bad in (new(6, 9), new(9, 7), new(7, 10)):
        keep = bad.clone()
        with pytest.raises(RuntimeError):
            tu.copy_fields(M, [a], [bad])
        assert torch.equal(bad, keep)
