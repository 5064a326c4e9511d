"""Weight and bias gradients where the pixel walk and the chunking can go
wrong: the smallest grid (its coarsest level is 2 x 2, so four consecutive
pixels cross two rows), widths that are not multiples of the 16-pixel step,
a last chunk that is cut, several images per chunk, and chunks past 128
pixels.

Tolerance: gradients pass through up to 15 layers stored in bf16 (unit
roundoff 2^-9 each): sqrt(2 * 15) * 2^-9 = 1.1 % expected, three times that
allowed; the bias of the last layer is a sum that is zero in exact
arithmetic."""
import numpy as np
import pytest

from oracle import nn as onn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 9, 9), (7, 9, 17), (3, 25, 17), (40, 33, 33)])
def test_gradient_shapes(shape):
    import torch
    from pybella_amd.nn import Network
    print(f"case nn gradients {shape}", flush=True)
    net = Network(5)
    P = net.get_params().astype(np.float64)
    rng = np.random.default_rng(sum(shape))
    X = rng.standard_normal(shape + (3,)).astype(np.float32)
    T = onn.project_null(rng.standard_normal(shape)).astype(np.float32)
    net.step(torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda(), lr=0.0)
    g = net.get_grads().astype(np.float64)
    z, cache = onn.forward(P, X.astype(np.float64), bf16=True)
    gr = onn.backward(P, cache, onn.loss(z, T.astype(np.float64))[1])
    off = 0
    for l, (ci, co, _) in enumerate(onn.LAYERS):
        nw = 9 * ci * co
        for part, sl in (("W", slice(off, off + nw)), ("b", slice(off + nw, off + nw + co))):
            if l == 14 and part == "b":
                continue
            rel = np.linalg.norm(g[sl] - gr[sl]) / np.linalg.norm(gr[sl])
            assert rel <= 0.033, (l, part, rel)
        off += nw + co
