"""The general backward's row kernel when a (table, column chunk)'s sorted
batches are shared by several workgroups (few tables or chunks, large batches):
rows of the LUT gradient that cross workgroups are merged from their part sums.
Against the oracle; with large thresholds most items fall into a few rows, so
that one row spans several parts, and many rows are empty."""
from __future__ import annotations

import importlib

import pytest
import torch

from test_gpu_parity import DEV, F16_TOL, F32_TOL, assert_gradients_f64, assert_train_parity, make_pair, rel_err, seeded, train_step

ph = importlib.import_module("tropnn_amd.backends.pairwise_hip")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "i,o,t,c,b,thr_std,lut_dtype",
    [
        (64, 320, 9, 6, 4100, 0.3, "f32"),   # 45 units: four parts
        (64, 320, 2, 3, 8200, 5.0, "f32"),   # eight parts, rows spanning several of them
        (40, 1000, 1, 1, 8195, 0.3, "f32"),  # two rows, each over half the parts
        (64, 90, 5, 8, 5000, 4.0, "f16"),    # two columns per lane, 8-slot batches, f16 rows
        (33, 31, 3, 8, 9000, 0.3, "f32"),    # one column per lane, 1024-thread workgroups
    ],
)
def test_rows_split_over_parts(i, o, t, c, b, thr_std, lut_dtype):
    ref, hip = make_pair(i, o, t, c, seed=3, thr_std=thr_std, lut_dtype=lut_dtype)
    x, g = seeded((b, i), seed=1), seeded((b, 1, o), seed=2)
    # rows of thousands of items: the f32 oracle's own rounding of such sums
    # reaches 4e-4 of an element (sqrt(8200) eps against a cancelled sum), so
    # the usual element-wise bar is held against float64
    pair = train_step(ref, hip, x, g)
    assert_train_parity(ref, hip, *pair, tol=F16_TOL if lut_dtype == "f16" else F32_TOL, elem_rtol=1e-3)
    assert_gradients_f64(hip, x, g, pair[1][1].grad, lut_dtype=lut_dtype)


@pytest.mark.parametrize("o", [512, 250])  # eight columns per lane, two
def test_row_sums_are_no_chain_of_single_items(o):
    """The LUT gradient's distance from float64 against that of a plain f32 sum
    of a row's items one after the other. A chain of n roundings errs by
    sqrt(n / 2) of one, a chain of batches of 4 by half of that (and the batch
    itself by little more than one): 0.5 to 0.6 of the plain sum, at most 0.8."""
    b, i, t, c = 4096, 64, 128, 6
    _, hip = make_pair(i, o, t, c, seed=5, thr_std=0.3)
    x, g = seeded((b, i), seed=1).to(DEV), seeded((b, 1, o), seed=2)
    hip.train()(x).backward(g.to(DEV))
    rows = (g[:, 0].numpy(), g[:, 0].double().numpy())
    err = [0.0, 0.0]
    for k in range(4):
        codes = hip._last_indices[:, 0, k].cpu().numpy()
        for r in range(1 << c):
            sel = codes == r
            if not sel.any():
                continue
            chain, exact = rows[0][sel].cumsum(axis=0)[-1], rows[1][sel].sum(axis=0)  # (cumsum adds in order, in f32)
            got = hip.lut.grad[k, r].double().cpu().numpy() / hip.output_scale
            err[0] += ((got - exact) ** 2).sum()
            err[1] += ((chain - exact) ** 2).sum()
    print(f"[row sums] o={o} kernel / chain {(err[0] / err[1]) ** 0.5:.3f}", flush=True)
    assert err[0] <= 0.8**2 * err[1]


@pytest.mark.parametrize(
    "i,o,t,c,b,thr_std,lut_dtype",
    [
        (128, 128, 136, 6, 2100, 0.3, "f32"),  # three tiles a table: workgroups of one and two tables
        (64, 256, 3, 5, 4100, 4.0, "f32"),     # fewer units than CUs: every unit a workgroup, skewed codes
        (32, 32, 300, 4, 3073, 0.3, "f16"),    # more tables than CUs: several whole tables a workgroup
        (40, 26, 140, 3, 2048, 0.3, "f32"),    # two columns per lane; whole tiles
        (32, 64, 3000, 4, 2050, 0.3, "f32"),   # gu slots past the four-item scatter kernel: a merge of its own
        (20, 64, 7, 8, 5000, 0.3, "f32"),      # 256 rows
    ],
)
def test_fused_split_over_tiles(i, o, t, c, b, thr_std, lut_dtype):
    """The fused backward of several tiles whose (table, tile) units are dealt
    to the workgroups: tables shared by workgroups merged, others written."""
    ref, hip = make_pair(i, o, t, c, seed=5, thr_std=thr_std, lut_dtype=lut_dtype)
    if lut_dtype == "f16":
        with torch.no_grad():
            ref.lut.copy_(ref.lut.half().float())  # the values the kernels read
    x, g = seeded((b, i), seed=1), seeded((b, 1, o), seed=2)
    # (element-wise bar: rows of many items, as above)
    pair = train_step(ref, hip, x, g)
    assert_train_parity(ref, hip, *pair, elem_rtol=1e-3)
    assert_gradients_f64(hip, x, g, pair[1][1].grad, lut_dtype=lut_dtype, block=512 if t < 1000 else 64)
    first = [p.grad.clone() for p in (hip.thresholds, hip.lut)]
    # parameter gradients alone (the merge kernel), the same sums
    hip.zero_grad(set_to_none=True)
    hip(x.to(DEV)).backward(g.to(DEV))
    assert torch.equal(hip.thresholds.grad, first[0]) and torch.equal(hip.lut.grad, first[1])


@pytest.mark.parametrize(
    "i,o,t,c,b",
    [
        (128, 64, 136, 6, 4096),  # its split plan asks for 13 MB
        (40, 26, 60, 3, 2100),    # two columns per lane
    ],
)
def test_fused_flag_without_workspace(i, o, t, c, b):
    """INPUT_GRAD_FUSED needs no workspace, whatever the batch: without the one
    that a split launch asks for, the item role runs. The input gradient is the
    split launch's bit for bit, the parameter gradients sum in another order."""
    lib = ph.load_library()
    mode = ph.STE_MIN_MARGIN | ph.BWD_INPUT_GRAD_FUSED
    need = lib.tropnn_hip_pairwise_backward_workspace_size(b, i, o, t, c, ph.LUT_F32, mode)
    assert need > 0, "the shape must take the split launch"
    _, hip = make_pair(i, o, t, c, seed=3, thr_std=0.3)
    hip.input_grad = "fused"
    x, g = seeded((b, i), seed=1).to(DEV).requires_grad_(True), seeded((b, 1, o), seed=2).to(DEV)
    hip.train()(x).backward(g)
    _, rec, *_ = ph._route_forward(x.detach().unsqueeze(1), hip.anchors, hip.thresholds.detach(), hip.lut.detach(),
                                   output_scale=hip.output_scale, want_record=True, return_route=False)
    offsets, entries = ph.anchor_index(hip.anchors, i)
    for ws_bytes in (0, need - 1):
        ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=DEV)
        out = [torch.full(s, float("nan"), device=DEV) for s in ((b, i), (t, c), (t, 1 << c, o))]
        rc = lib.tropnn_hip_pairwise_backward(
            b, i, o, t, c, g.data_ptr(), hip.lut.data_ptr(), ph.LUT_F32, rec.data_ptr(), None, offsets.data_ptr(),
            entries.data_ptr(), hip.output_scale, mode, 0, *(v.data_ptr() for v in out),
            ws.data_ptr() if ws_bytes else None, ws_bytes, torch.cuda.current_stream(DEV).cuda_stream)
        assert rc == 0, lib.tropnn_hip_last_error()
        assert torch.equal(out[0], x.grad)
        for got, want in zip(out[1:], (hip.thresholds.grad, hip.lut.grad)):
            # two orders of sums of up to 4096 f32 terms: 2 sqrt(4096) roundings of 2^-24 at most
            assert rel_err(got.cpu(), want.cpu()) <= 2 * 4096**0.5 * 2.0**-24


@pytest.mark.parametrize(
    "i,o,t,c,b,lut_dtype",
    [
        (32, 90, 128, 4, 60, "f32"),   # row kernel: 256 (table, chunk)s, workgroups of 1024 threads
        (32, 90, 129, 4, 60, "f16"),   # 258: of 512
        (32, 33, 512, 3, 40, "f32"),   # one column per lane: 1024 threads up to 512 (table, chunk)s
        (32, 33, 513, 3, 40, "f32"),   # 512 threads
        (32, 33, 6, 7, 70, "f32"),     # the LUT chunk staged eight pieces at a time, 128 rows
        (32, 65, 4, 8, 70, "f16"),     # 256 rows, two chunks
        (32, 33, 150, 8, 1500, "f32"), # three parts: one round of workgroups
        (16, 1030, 3, 3, 968, "f32"),  # reduce kernel: at most 1024 slots, 17 chunks
        (16, 1030, 3, 3, 969, "f32"),  # more
        (16, 33, 5, 2, 900, "f32"),    # at most 1024 slots in three parts
        (16, 35, 2, 5, 3000, "f32"),   # one-column pieces of G over many copy workgroups
    ],
)
def test_general_path_by_size(i, o, t, c, b, lut_dtype):
    """Either side of the general path's lines between its launch shapes."""
    ref, hip = make_pair(i, o, t, c, seed=7, thr_std=0.3, lut_dtype=lut_dtype)
    if lut_dtype == "f16":
        with torch.no_grad():
            ref.lut.copy_(ref.lut.half().float())  # the values the kernels read
    x, g = seeded((b, i), seed=1), seeded((b, 1, o), seed=2)
    pair = train_step(ref, hip, x, g)
    assert_train_parity(ref, hip, *pair, elem_rtol=1e-3)
    assert_gradients_f64(hip, x, g, pair[1][1].grad, lut_dtype=lut_dtype, block=256)


@pytest.mark.parametrize("off", [0, 2])
def test_split_launch_with_grad_lut_off_16_bytes(off):
    """Two columns per lane (26 columns) need grad_lut aligned to two floats
    only, in the merge of the workgroups' sums too."""
    b, i, o, t, c = 2048, 40, 26, 140, 3
    lib = ph.load_library()
    _, hip = make_pair(i, o, t, c, seed=5, thr_std=0.3)
    x, g = seeded((b, i), seed=1).to(DEV).requires_grad_(True), seeded((b, 1, o), seed=2).to(DEV)
    hip.train()(x).backward(g)
    _, rec, *_ = ph._route_forward(x.detach().unsqueeze(1), hip.anchors, hip.thresholds.detach(), hip.lut.detach(),
                                   output_scale=hip.output_scale, want_record=True, return_route=False)
    ws = torch.empty(lib.tropnn_hip_pairwise_backward_workspace_size(b, i, o, t, c, ph.LUT_F32, ph.STE_MIN_MARGIN),
                     dtype=torch.uint8, device=DEV)
    n = t * (1 << c) * o
    buf = torch.full((off + n + 4,), 7.0, device=DEV)
    rc = lib.tropnn_hip_pairwise_backward(
        b, i, o, t, c, g.data_ptr(), hip.lut.data_ptr(), ph.LUT_F32, rec.data_ptr(), None, None, None,
        hip.output_scale, ph.STE_MIN_MARGIN, 0, None, None, buf[off:].data_ptr(), ws.data_ptr(), ws.numel(),
        torch.cuda.current_stream(DEV).cuda_stream)
    assert rc == 0, lib.tropnn_hip_last_error()
    assert torch.equal(buf[off : off + n].view_as(hip.lut.grad), hip.lut.grad)
    assert bool((buf[:off] == 7).all()) and bool((buf[off + n :] == 7).all())


def test_allocation_free_backward_keeps_its_range():
    """A shape whose split plan needs more than the allocation-free entry
    point's 32 MiB, but whose plain one fits: still served."""
    b, i, o, t, c = 12000, 32, 512, 16, 6
    lib = ph.load_library()
    assert lib.tropnn_hip_pairwise_backward_workspace_size(b, i, o, t, c, ph.LUT_F32, ph.STE_MIN_MARGIN) > 32 << 20
    _, hip = make_pair(i, o, t, c, seed=3, thr_std=0.3)
    x, g = seeded((b, i), seed=1).to(DEV).requires_grad_(True), seeded((b, 1, o), seed=2).to(DEV)
    hip.train()(x).backward(g)
    _, rec, *_ = ph._route_forward(x.detach().unsqueeze(1), hip.anchors, hip.thresholds.detach(), hip.lut.detach(),
                                   output_scale=hip.output_scale, want_record=True, return_route=False)
    offsets, entries = ph.anchor_index(hip.anchors, i)
    out = [torch.empty(b, i, device=DEV), torch.empty(t, c, device=DEV), torch.empty(t, 1 << c, o, device=DEV)]
    rc = lib.tropnn_hip_pairwise_backward_noalloc(
        b, i, o, t, c, g.data_ptr(), hip.lut.data_ptr(), ph.LUT_F32, rec.data_ptr(), None, offsets.data_ptr(),
        entries.data_ptr(), hip.output_scale, ph.STE_MIN_MARGIN, 0, *(v.data_ptr() for v in out),
        torch.cuda.current_stream(DEV).cuda_stream)
    assert rc == 0, lib.tropnn_hip_last_error()
    for got, want in zip(out, (x.grad, hip.thresholds.grad, hip.lut.grad)):
        assert rel_err(got.cpu(), want.cpu()) <= 1e-6  # another order of a few row sums
