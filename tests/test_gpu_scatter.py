"""The scatter kernel that takes four items a workgroup (batches of 1024 items
and more): an item's input gradient is the same sum in the same order as the
one-item kernel's, so a batch equals its halves' calls bit for bit."""
from __future__ import annotations

import pytest
import torch

from test_gpu_parity import DEV, make_pair, seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "i,o,t,c,b",
    [
        (128, 128, 136, 6, 1025),  # two lanes a feature; one item in the last workgroup
        (129, 64, 40, 5, 1027),    # one lane a feature
        (37, 96, 300, 3, 1030),    # more tables than threads, long features (many entry batches)
        (700, 34, 33, 8, 1024),    # general path, 512 threads, most features short or empty
        (1500, 16, 20, 4, 1026),   # 1024 threads, more features than threads
    ],
)
def test_batch_equals_its_halves(i, o, t, c, b):
    _, hip = make_pair(i, o, t, c, seed=b, thr_std=0.3)
    hip.input_grad = "scatter"
    x, g = seeded((b, i), seed=1).to(DEV), seeded((b, 1, o), seed=2).to(DEV)

    def grad_x(lo, hi):
        xs = x[lo:hi].clone().requires_grad_(True)
        hip.train()(xs).backward(g[lo:hi])
        return xs.grad

    whole = grad_x(0, b)
    half = b // 2 - 1
    assert torch.equal(whole, torch.cat([grad_x(0, half), grad_x(half, b)]))
    assert bool(whole.abs().sum() > 0)
