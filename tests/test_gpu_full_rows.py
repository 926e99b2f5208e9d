"""The full STE's backward of large batches: every comparison's dots in the row
kernel over the sorted slots, the per-comparison gradients from the reduce
kernel. Against the oracle, at the line's two sides and at the edges of the
column pieces, chunks and comparisons."""
from __future__ import annotations

import pytest
import torch

from test_gpu_parity import DEV, F16_TOL, F32_TOL, assert_gradients_f64, assert_train_parity, make_pair, rel_err, seeded, train_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "i,o,t,c,b,thr_std,lut_dtype",
    [
        (32, 24, 40, 6, 1023, 0.3, "f32"),   # the item kernel
        (32, 24, 40, 6, 1024, 0.3, "f32"),   # the row kernel's first with many tables
        (32, 24, 17, 5, 2047, 0.3, "f32"),   # the item kernel, fewer tables
        (32, 24, 17, 5, 2048, 0.3, "f32"),   # the row kernel's first
        (20, 1, 7, 1, 2050, 0.3, "f32"),     # one column, one comparison; items no multiple of four
        (64, 130, 9, 8, 5001, 0.3, "f16"),   # 256 rows, 2 columns a lane, three chunks; several pieces a table
        (40, 33, 5, 3, 2050, 4.0, "f32"),    # one column a lane; skewed codes, empty rows
        (64, 320, 2, 6, 8200, 0.3, "f32"),   # five chunks, several workgroups per (table, chunk)
    ],
)
def test_full_ste_row_dots(i, o, t, c, b, thr_std, lut_dtype):
    ref, hip = make_pair(i, o, t, c, seed=3, thr_std=thr_std, lut_dtype=lut_dtype, use_min_margin_ste=False)
    if lut_dtype == "f16":
        with torch.no_grad():
            ref.lut.copy_(ref.lut.half().float())  # the values the kernels read
    x, g = seeded((b, i), seed=1), seeded((b, 1, o), seed=2)
    # rows of thousands of items: the f32 oracle's own rounding of such sums
    # reaches 4e-4 of an element (sqrt(8200) eps against a cancelled sum), so
    # the usual element-wise bar is held against float64
    pair = train_step(ref, hip, x, g)
    assert_train_parity(ref, hip, *pair, tol=F16_TOL if lut_dtype == "f16" else F32_TOL, elem_rtol=1e-3)
    assert_gradients_f64(hip, x, g, pair[1][1].grad, lut_dtype=lut_dtype)
    # each parameter's gradient alone: the same sums, the LUT's over other row groups
    (thr,) = torch.autograd.grad(hip(x.to(DEV)), [hip.thresholds], g.to(DEV))
    assert torch.equal(thr, hip.thresholds.grad)
    (lut,) = torch.autograd.grad(hip(x.to(DEV)), [hip.lut], g.to(DEV))
    assert rel_err(lut.cpu(), hip.lut.grad.cpu()) <= 1e-6
