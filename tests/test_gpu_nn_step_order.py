"""A training step's gradients and parameters, bit for bit those on record:
the sums of the weight and bias gradients have one order, fixed by the shape
alone, however their work is split over blocks.  Adam's first steps turn a
rounding difference of a near-zero gradient into a full learning rate, so a
changed order shows in the parameters at once.

Shapes: the smallest grid, chunks cut short, several images per chunk, one and
many chunks, and a coarsest level with fewer pixels than a chunk's waves."""
import hashlib
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "nn_step_digests.json")
with open(GOLDEN) as f:
    STEPS = json.load(f)["steps"]


def _digest(a):
    return hashlib.sha256(a.astype(np.float32).tobytes()).hexdigest()[:16]


@pytest.mark.parametrize("name", sorted(STEPS))
def test_step_is_bitwise_the_recorded_one(name):
    import torch
    from pybella_amd.nn import Network
    print(f"case nn step order {name}", flush=True)
    shape = tuple(int(v) for v in name.split("x"))
    net = Network(5)
    rng = np.random.default_rng(sum(shape))
    X = torch.from_numpy(rng.standard_normal(shape + (3,)).astype(np.float32)).cuda()
    T = torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).cuda()
    got = []
    for _ in range(2):
        net.step(X, T, lr=1e-3)
        got.append(_digest(net.get_grads()))
    assert got + [_digest(net.get_params())] == STEPS[name]
