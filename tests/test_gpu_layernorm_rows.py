"""GPU parity of LayerNorm over rows of any length and alignment, wide rows and few rows, against the
CPU oracle with the tolerances of test_gpu_elementwise.py."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import half_ulp_check, max_rel
from test_gpu_elementwise import DEV, _ln16_case, _ln_case, dev, dev16, host, say, to16

pytestmark = pytest.mark.gpu

# Both sides of: the one-launch limit (512 rows), one vector (4 fp32, 8 16-bit elements), one wave's
# row and four waves' rows (2048 and 4096 columns), each with whole and with overlapping vectors
SHAPES = [(3, 3), (3, 9), (513, 7), (513, 8), (513, 9), (512, 767), (513, 767), (514, 1025),
          (600, 2047), (513, 2049), (515, 2052), (520, 2560), (514, 3001), (513, 4095), (513, 4096),
          (70, 4097), (513, 4100), (130, 8195), (1, 4096), (512, 2560)]


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_layernorm_rows_f32(hk, orc, rows, cols):
    say("layernorm rows f32", rows, cols)
    _ln_case(hk, orc, rows, cols, (161, 162, 163, 164))


@pytest.mark.parametrize("fmt", ["bf16", "f16"])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_layernorm_rows_16bit(hk, orc, fmt, rows, cols):
    say("layernorm rows", fmt, rows, cols)
    _ln16_case(hk, orc, rows, cols, fmt, (165, 166, 167, 168))


@pytest.mark.parametrize("rows,cols", [(5, 264), (600, 264), (600, 2568), (40, 515)])
@pytest.mark.parametrize("fmt", ["f32", "bf16"])
def test_layernorm_unaligned_bases(hk, orc, fmt, rows, cols):
    # every tensor starts one element past a 16-byte boundary; what lies before and behind the
    # outputs stays as it was, and NaN around the inputs does not reach them
    say("layernorm unaligned", fmt, rows, cols)
    if fmt == "f32":
        put = lambda a: torch.from_numpy(np.ascontiguousarray(a))  # noqa: E731
        x = orc.normal(rows * cols, 171).reshape(rows, cols)
        dy = orc.normal(rows * cols, 172).reshape(rows, cols)
        gamma, beta = orc.rand_uniform(cols, 173, 0.5, 1.5), orc.normal(cols, 174, 0.0, 0.1)
        xs, dys, gs, bs = put(x), put(dy), put(gamma), put(beta)
    else:
        x16, x = to16(orc, orc.normal(rows * cols, 171).reshape(rows, cols), fmt)
        dy16, dy = to16(orc, orc.normal(rows * cols, 172).reshape(rows, cols), fmt)
        g16, gamma = to16(orc, orc.rand_uniform(cols, 173, 0.5, 1.5), fmt)
        b16, beta = to16(orc, orc.normal(cols, 174, 0.0, 0.1), fmt)
        xs, dys, gs, bs = (dev16(a, fmt) for a in (x16, dy16, g16, b16))

    def off(t, fill=float("nan")):
        t = t.to(DEV)
        buf = torch.full((t.numel() + 17,), fill, device=DEV, dtype=t.dtype)
        v = buf[1:1 + t.numel()].view(t.shape)
        v.copy_(t)
        return buf, v
    (_, X), (_, DY), (_, G), (_, B) = off(xs), off(dys), off(gs), off(bs)
    (ybuf, Y), (dbuf, DX) = off(torch.zeros_like(xs), 3.0), off(torch.zeros_like(xs), 3.0)
    yr, mr, rr = orc.layer_norm_forward(x, gamma, beta, 1e-5)
    hk.layer_norm_forward(X, G, B, 1e-5, y=Y)
    dg, db = torch.ones(cols, device=DEV), torch.ones(cols, device=DEV)  # added into
    hk.layer_norm_backward(DY, X, dev(mr), dev(rr), G, dg, db, grad_x=DX)
    dxr = orc.ln_backward_input(dy, x, mr, rr, gamma)
    dgr, dbr = orc.ln_backward_gamma_beta(dy, x, mr, rr)
    if fmt == "f32":
        assert max_rel(host(Y), yr) <= 1e-5 and max_rel(host(DX), dxr) <= 1e-5
    else:
        half_ulp_check(host(Y), yr, fmt)
        half_ulp_check(host(DX), dxr, fmt)
    assert max_rel(host(dg) - 1, dgr) <= 1e-5 and max_rel(host(db) - 1, dbr) <= 1e-5
    for buf, n in ((ybuf, Y.numel()), (dbuf, DX.numel())):
        assert float(buf[0]) == 3.0 and bool((buf[1 + n:] == 3.0).all())


@pytest.mark.parametrize("rows,cols", [(100, 768), (700, 2560), (700, 333)])
def test_layernorm_gradients_deterministic_and_optional(hk, orc, rows, cols):
    say("layernorm optional gradients", rows, cols)
    x, dy = (dev(orc.normal(rows * cols, s).reshape(rows, cols)) for s in (181, 182))
    y, m, r = hk.layer_norm_forward(x)
    out = []
    for _ in range(2):
        dg, db = torch.zeros(cols, device=DEV), torch.zeros(cols, device=DEV)
        out.append((hk.layer_norm_backward(dy, x, m, r, None, dg, db), dg, db))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    only = torch.zeros(cols, device=DEV)
    lib = hk.lib()
    p = lambda t: t.data_ptr()  # noqa: E731
    st = torch.cuda.current_stream().cuda_stream
    assert lib.hk_ln_backward_gamma_beta_f32(p(dy), p(x), p(m), p(r), None, p(only), rows, cols, st) == 0
    assert max_rel(host(only), host(out[0][2])) <= 1e-6


@pytest.mark.parametrize("rows,cols", [(600, 333), (600, 2560)])
def test_layernorm_backward_under_capture(hk, orc, rows, cols):
    # these shapes use no workspace while a graph is captured; replays stay right after eager calls
    # that need a larger one
    say("layernorm capture", rows, cols)
    x, dy = (dev(orc.normal(rows * cols, s).reshape(rows, cols)) for s in (191, 192))
    y, m, r = hk.layer_norm_forward(x)
    g = torch.zeros(2, cols, device=DEV)
    dx = hk.layer_norm_backward(dy, x, m, r, None, g[0], g[1])
    want, want_dx = g.clone(), dx.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        g.zero_()
        hk.layer_norm_backward(dy, x, m, r, None, g[0], g[1], grad_x=dx)
    big = torch.randn(4096, 4096, device=DEV)
    for _ in range(3):
        dx.zero_()
        graph.replay()
        assert max_rel(host(g), host(want)) <= 1e-5 and max_rel(host(dx), host(want_dx)) <= 1e-6
        _, bm, br = hk.layer_norm_forward(big)
        hk.layer_norm_backward(big, big, bm, br, None, torch.zeros(4096, device=DEV),
                               torch.zeros(4096, device=DEV))


@pytest.mark.parametrize("rows,cols", [(1, 1), (16, 4096), (20, 8200), (128, 5000), (129, 5000), (33, 3),
                                       (512, 17)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layernorm_gradients_alone(hk, rows, cols, dtype):
    # the gamma/beta entry point on few rows of any length, against 64 bits: fp32 sums of `rows` terms,
    # pairwise over 32 groups
    say("layernorm gradients alone", rows, cols, dtype)
    g = torch.Generator(device=DEV)
    g.manual_seed(rows + cols)
    x, dy = (torch.randn(rows, cols, generator=g, device=DEV).to(dtype) for _ in range(2))
    _, m, r = hk.layer_norm_forward(x)
    sums = torch.ones(2, cols, device=DEV)  # added into
    hk.ln_backward_gamma_beta(dy, x, m, r, sums[0], sums[1])
    xh = (x.double() - m.double()[:, None]) * r.double()[:, None]
    want = torch.stack([(dy.double() * xh).sum(0), dy.double().sum(0)]) + 1
    assert max_rel(host(sums), want.cpu().numpy()) <= 2e-6


# Both sides of the one-launch limit (512 rows) in every form of a row: whole vectors of one wave,
# overlapping vectors, four waves, a workgroup per row, less than a vector
@pytest.mark.parametrize("rows,cols", [(64, 768), (512, 768), (513, 768), (512, 333), (600, 333),
                                       (512, 2560), (600, 2560), (128, 8200), (600, 8200), (512, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("into", ["dy", "x"])
@pytest.mark.parametrize("captured", [False, True])
def test_layernorm_backward_in_place(hk, rows, cols, dtype, into, captured):
    # grad_x written over dy or x: the same grad_x and the same sums (in another order, 1e-5) as in a
    # buffer of its own
    say("layernorm in place", rows, cols, dtype, into, captured)
    g = torch.Generator(device=DEV)
    g.manual_seed(rows + cols)
    x, dy = (torch.randn(rows, cols, generator=g, device=DEV).to(dtype) for _ in range(2))
    gamma = torch.rand(cols, generator=g, device=DEV).to(dtype)
    _, m, r = hk.layer_norm_forward(x)
    want = torch.zeros(2, cols, device=DEV)
    want_dx = hk.layer_norm_backward(dy, x, m, r, gamma, want[0], want[1])
    bufs = {"x": x.clone(), "dy": dy.clone()}
    sums = torch.zeros(2, cols, device=DEV)

    def call():
        hk.layer_norm_backward(bufs["dy"], bufs["x"], m, r, gamma, sums[0], sums[1],
                               grad_x=bufs[into])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()  # also gives the stream's workspace its size before a capture
    torch.cuda.synchronize()
    run = call
    if captured:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            call()
        run = graph.replay
    for _ in range(3):
        bufs["x"].copy_(x)
        bufs["dy"].copy_(dy)
        sums.zero_()
        run()
        torch.cuda.synchronize()
        assert max_rel(host(bufs[into].float()), host(want_dx.float())) <= (
            1e-6 if dtype == torch.float32 else 2.0 ** -8)
        assert max_rel(host(sums), host(want)) <= 1e-5
