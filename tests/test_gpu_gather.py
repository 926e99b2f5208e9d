"""The staged forward (tropnn_hip_pairwise_forward_ws): a route kernel that
writes packed codes to the caller's workspace, then a gather out of LDS. Its
route outputs equal the plain forward's bit for bit; the slice gather's output
too (it sums the same 16-table blocks in order), the stream gather's (LUTs of
32 MiB and more, another order of the sum over tables) to f32 rounding of a
float64 sum."""
from __future__ import annotations

import importlib

import pytest
import torch

from test_gpu_parity import DEV, make_pair, rel_err, seeded

ph = importlib.import_module("tropnn_amd.backends.pairwise_hip")

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    yield
    torch.cuda.synchronize()


def layer_tensors(i, o, t, c, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed)
    first = torch.randint(0, i, (t, c), generator=gen)
    anchors = torch.stack((first, torch.randint(0, i, (t, c), generator=gen)), dim=-1)
    thr = 0.1 * torch.randn(t, c, generator=gen)
    gpu = torch.Generator(DEV).manual_seed(seed)
    lut = (0.02 * torch.randn(t, 1 << c, o, generator=gpu, device=DEV)).to(dtype)
    return anchors.to(DEV), thr.to(DEV), lut


def forward(x, anchors, thr, lut, *, staged, record=True, debug=True, out_off=0):
    """(output, record, indices, margin bits, codes) of one C ABI call, every
    buffer filled with a value no kernel writes."""
    (b, i), (t, c, _), o = x.shape, anchors.shape, lut.shape[2]
    lib = ph.load_library()
    dt = ph.LUT_F16 if lut.dtype == torch.float16 else ph.LUT_F32
    out = torch.full((b * o + out_off,), float("nan"), device=DEV)[out_off:].view(b, o)
    rec = torch.full((t, b), -1, dtype=torch.int64, device=DEV) if record else None
    idx = torch.full((b, t), -1, dtype=torch.int64, device=DEV) if debug else None
    mar = torch.full((b, t, c), -1, dtype=torch.int32, device=DEV) if debug else None
    codes = torch.full((b, t), 255, dtype=torch.uint8, device=DEV) if debug else None
    ptr = [None if v is None else v.data_ptr() for v in (rec, idx, mar, codes)]
    n = lib.tropnn_hip_pairwise_forward_workspace_size(b, i, o, t, c, dt) if staged else 0
    assert not staged or n > 0, "the shape must take the staged forward"
    ws = torch.full((n + 16,), 255, dtype=torch.uint8, device=DEV)
    args = (b, i, o, t, c, x.data_ptr(), anchors.data_ptr(), thr.data_ptr(), lut.data_ptr(), dt, 0.25, out.data_ptr(), *ptr)
    stream = torch.cuda.current_stream(DEV).cuda_stream
    if staged:
        rc = lib.tropnn_hip_pairwise_forward_ws(*args, ws.data_ptr(), n, stream)
    else:
        rc = lib.tropnn_hip_pairwise_forward(*args, stream)
    assert rc == 0, lib.tropnn_hip_last_error()
    torch.cuda.synchronize()
    assert bool((ws[n:] == 255).all())
    return out, rec, idx, mar, codes


SLICE = [
    # b, i, o, t, c, dtype, output offset
    (12288, 128, 128, 136, 6, torch.float32, 0),  # one stage of all tables, whole waves
    (8195, 33, 250, 100, 5, torch.float32, 0),    # rows of 1000 bytes: 8-byte staging; blocks of 15 tables
    (6001, 40, 251, 100, 5, torch.float32, 1),    # 4-byte staging, ragged last slice
    (9001, 37, 250, 101, 4, torch.float16, 0),    # f16 rows of 500 bytes: 4-byte staging
    (9001, 37, 251, 100, 5, torch.float16, 1),    # 2-byte staging
    (4100, 64, 512, 128, 6, torch.float32, 4),    # several items per thread
    (24500, 64, 96, 200, 6, torch.float32, 0),    # tables in several stages
    (24001, 64, 200, 150, 7, torch.float16, 0),   # several stages, f16
    (60000, 50, 200, 37, 1, torch.float32, 0),    # one comparison, blocks of 13 and 11 tables
    (8200, 2600, 256, 120, 3, torch.float32, 0),  # 10 KB input rows: four items per route workgroup
]


@pytest.mark.parametrize("b,i,o,t,c,dtype,out_off", SLICE)
def test_slice_gather_equals_the_plain_forward(b, i, o, t, c, dtype, out_off):
    anchors, thr, lut = layer_tensors(i, o, t, c, dtype, seed=b)
    x = seeded((b, i), seed=t).to(DEV)
    plain = forward(x, anchors, thr, lut, staged=False, out_off=out_off)
    staged = forward(x, anchors, thr, lut, staged=True, out_off=out_off)
    for name, p, s in zip(("output", "record", "indices", "margins", "codes"), plain, staged):
        assert torch.equal(p, s), name
    assert torch.equal(forward(x, anchors, thr, lut, staged=True, record=False, debug=False, out_off=out_off)[0], plain[0])


@pytest.mark.parametrize(
    "b,i,o,t,c,dtype",
    [
        (4096, 64, 1024, 134, 7, torch.float16),  # two groups a stage, a tail of two tables
        (4100, 64, 512, 131, 8, torch.float16),   # one group a stage, a tail of three, a partial item block
        (9000, 24, 2048, 1033, 3, torch.float16),  # 8-row tables: 32 groups a stage, a tail of one
        (2100, 300, 2048, 128, 8, torch.float16),  # fewer items: four items per thread
    ],
)
def test_stream_gather_against_float64(b, i, o, t, c, dtype):
    anchors, thr, lut = layer_tensors(i, o, t, c, dtype, seed=b)
    x = seeded((b, i), seed=t).to(DEV)
    plain = forward(x, anchors, thr, lut, staged=False)
    staged = forward(x, anchors, thr, lut, staged=True)
    for name, p, s in list(zip(("output", "record", "indices", "margins", "codes"), plain, staged))[1:]:
        assert torch.equal(p, s), name
    exact = torch.zeros(b, o, dtype=torch.float64, device=DEV)
    for k in range(t):
        exact += lut[k].double()[plain[2][:, k]]
    exact *= 0.25
    # a sum of t terms in f32: each partial sum rounded once, at most about t
    # eps / 2 of it, and sqrt(t) eps for rounding errors of random sign
    err = (staged[0].double() - exact).norm() / exact.norm()
    assert float(err) <= 2.0**-24 * t**0.5
    # without a record the 512-column layer gains nothing and keeps the one-launch kernels
    want = forward(x, anchors, thr, lut, staged=False, record=False, debug=False) if (b, o) == (4100, 512) else staged
    assert torch.equal(forward(x, anchors, thr, lut, staged=True, record=False, debug=False)[0], want[0])


@pytest.mark.parametrize("b,o,t,c,gains", [(4096, 128, 512, 8, False), (8192, 96, 700, 8, False), (8192, 1024, 128, 8, True)])
def test_eval_takes_the_stream_gather_only_where_it_gains(b, o, t, c, gains):
    """An eval forward of few columns keeps the one-launch kernels at every
    batch size (a stream gather of 8 or 12 workgroups would take several times
    as long): the workspace, sized for training, stays untouched."""
    anchors, thr, lut = layer_tensors(64, o, t, c, torch.float16, seed=b)
    x = seeded((b, 64), seed=t).to(DEV)
    lib = ph.load_library()
    n = lib.tropnn_hip_pairwise_forward_workspace_size(b, 64, o, t, c, ph.LUT_F16)
    out, rec = torch.empty(b, o, device=DEV), torch.empty(t, b, dtype=torch.int64, device=DEV)
    for record in (False, True):
        ws = torch.full((n,), 255, dtype=torch.uint8, device=DEV)
        rc = lib.tropnn_hip_pairwise_forward_ws(
            b, 64, o, t, c, x.data_ptr(), anchors.data_ptr(), thr.data_ptr(), lut.data_ptr(), ph.LUT_F16, 0.25,
            out.data_ptr(), rec.data_ptr() if record else None, None, None, None, ws.data_ptr(), n,
            torch.cuda.current_stream(DEV).cuda_stream)
        assert rc == 0, lib.tropnn_hip_last_error()
        assert bool((ws != 255).any()) == (record or gains)


@pytest.mark.parametrize("b,o,t,c", [(4096, 512, 512, 6), (4100, 1024, 200, 7), (4096, 4096, 512, 4)])
def test_stream_gather_is_as_close_to_float64_as_the_plain_forward(b, o, t, c):
    """f16 LUT rows of unit size, whose f32 sums round: the staged forward's
    two halves of four-table groups against the plain kernels' blocks of 16
    tables (one run of all the groups would be 1.5 to 4 % further off)."""
    anchors, thr, lut = layer_tensors(64, o, t, c, torch.float16, seed=b)
    lut.copy_(torch.randn(lut.shape, generator=torch.Generator(DEV).manual_seed(1), device=DEV))
    x = seeded((b, 64), seed=t).to(DEV)
    lib = ph.load_library()
    args = (b, 64, o, t, c, x.data_ptr(), anchors.data_ptr(), thr.data_ptr(), lut.data_ptr(), ph.LUT_F16, t**-0.5)
    n = lib.tropnn_hip_pairwise_forward_workspace_size(b, 64, o, t, c, ph.LUT_F16)
    assert n > 0, "the shape must take the staged forward"
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    rec = torch.empty(t, b, dtype=torch.int64, device=DEV)
    codes = torch.empty(b, t, dtype=torch.uint8, device=DEV)
    out = [torch.empty(b, o, device=DEV) for _ in range(2)]
    stream = torch.cuda.current_stream(DEV).cuda_stream
    rc = lib.tropnn_hip_pairwise_forward(*args, out[0].data_ptr(), None, None, None, codes.data_ptr(), stream)
    assert rc == 0, lib.tropnn_hip_last_error()
    rc = lib.tropnn_hip_pairwise_forward_ws(*args, out[1].data_ptr(), rec.data_ptr(), None, None, None, ws.data_ptr(), n, stream)
    assert rc == 0, lib.tropnn_hip_last_error()
    exact = torch.zeros(b, o, dtype=torch.float64, device=DEV)
    for k in range(t):
        exact += lut[k].double()[codes[:, k].long()]
    exact *= float(torch.tensor(t**-0.5, dtype=torch.float32))
    plain, staged = (float((v.double() - exact).norm() / exact.norm()) for v in out)
    print(f"[stream gather] {b} x {o}, {t} tables: plain {plain:.4g}, staged {staged:.4g}", flush=True)
    assert 0 < staged <= plain


def test_non_finite_rows_stay_in_their_items():
    """An infinity or NaN of the LUT reaches exactly the items whose codes name
    its row: padding slots and absent tables read zeros, not other rows."""
    for b, i, o, t, c, dtype in ((8195, 33, 250, 100, 5, torch.float32), (4100, 64, 512, 131, 8, torch.float16)):
        anchors, thr, lut = layer_tensors(i, o, t, c, dtype, seed=1)
        lut[t - 1, 0] = float("inf")
        lut[0, 0] = float("nan")
        x = seeded((b, i), seed=2).to(DEV)
        out, _, idx, _, _ = forward(x, anchors, thr, lut, staged=True)
        nan, inf = idx[:, 0] == 0, (idx[:, t - 1] == 0) & (idx[:, 0] != 0)
        assert bool(nan.any()) and bool(inf.any())
        assert bool(out[nan].isnan().all()) and bool(out[inf].isinf().all())
        assert bool(out[~nan & ~inf].isfinite().all())


def test_module_uses_the_staged_forward_under_capture():
    """A captured eval forward of a staged shape replays (three replays, other
    inputs and eager work between) to the eager result."""
    ref, hip = make_pair(300, 250, 100, 5, seed=3, thr_std=0.2)
    hip.eval()
    hip.cache_route_debug = False
    x = seeded((8195, 300), seed=5).to(DEV)
    with torch.no_grad():
        assert rel_err(hip(x), ref.eval()(x.cpu())) <= 1e-5
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            hip(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = hip(x)
        for k in range(3):
            x.copy_(seeded((8195, 300), seed=10 + k))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, hip(x))
