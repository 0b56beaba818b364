"""GPU parity of the attention backward where a key tile's queries are shared by several workgroups,
of query tiles that end past T anywhere in the order, and of the form that writes dQ, against the
CPU oracle with the tolerance of test_gpu_attention.py (2e-3; measured 1e-5)."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from conftest import max_rel
from test_gpu_attention import DEV, _qkv, say

pytestmark = pytest.mark.gpu


def _case(hk, orc, B, H, T, causal, seeds=(301, 302, 303, 304)):
    q, k, v, do = _qkv(orc, B, H, T, 64, seeds, normal=True)
    ro, rl = orc.attn_forward(q, k, v, 0.125, causal)
    want = orc.attn_backward(q, k, v, ro, do, rl, 0.125, causal)[1:]
    dev = [torch.from_numpy(a).to(DEV) for a in (q, k, v, do, rl)]
    D = hk.attn_bwd_precompute_D(dev[3], torch.from_numpy(ro).to(DEV))
    return dev, D, want


# few heads: split into pieces of 1 to 5 query tiles, with and without a partial last tile; the last
# shapes fill the device and stay whole
@pytest.mark.parametrize("B,H,T", [(1, 1, 128), (1, 1, 129), (1, 1, 1000), (1, 2, 1024), (2, 12, 333),
                                   (1, 3, 2031), (3, 5, 450), (4, 40, 190), (1, 1, 4000)])
@pytest.mark.parametrize("causal", [False, True])
def test_attn_backward_split_queries(hk, orc, B, H, T, causal):
    say("attn bwd split", B, H, T, causal)
    (q, k, v, do, lse), D, want = _case(hk, orc, B, H, T, causal)
    first = hk.attn_backward(q, k, v, do, lse, D, causal)
    for got, ref in zip(first, want):
        assert max_rel(got.cpu().numpy(), ref) <= 2e-3
    second = hk.attn_backward(q, k, v, do, lse, D, causal)
    # dK and dV are summed in a fixed order (dQ is accumulated with atomics)
    assert torch.equal(first[1], second[1]) and torch.equal(first[2], second[2])


@pytest.mark.parametrize("causal", [False, True])
def test_attn_backward_strided_outputs_and_set(hk, orc, causal):
    # dQ, dK, dV between NaNs with odd row strides: hk_attn_backward_set writes every element of dQ
    # and nothing else; hk_attn_backward adds to what is there
    B, H, T = 2, 3, 333
    say("attn bwd strided outputs", causal)
    (q, k, v, do, lse), D, want = _case(hk, orc, B, H, T, causal)
    for fn, start in (("hk_attn_backward_set", float("nan")), ("hk_attn_backward", 1.0)):
        bufs = [torch.full((B, H, T + 1, 67), float("nan"), device=DEV) for _ in range(3)]
        dq, dk, dv = (b[:, :, :T, 1:65] for b in bufs)
        dq.fill_(start)
        p = hk._bwd_params(q, k, v, None, do, lse, D, dq, dk, dv, causal, 0.125)
        assert getattr(hk.lib(), fn)(ctypes.byref(p), 64, torch.cuda.current_stream().cuda_stream) == 0
        got = [t.cpu().numpy() for t in (dq, dk, dv)]
        if start == 1.0:
            got[0] = got[0] - 1.0
        for g, ref in zip(got, want):
            assert max_rel(g, ref) <= 2e-3
        for b in bufs:
            outside = b.clone()
            outside[:, :, :T, 1:65] = float("nan")
            assert bool(torch.isnan(outside).all())


def test_attn_backward_set_replayed_graph(hk, orc):
    # the split form in a captured graph, replayed with other work between
    B, H, T = 1, 4, 520
    say("attn bwd graph")
    (q, k, v, do, lse), D, want = _case(hk, orc, B, H, T, True)
    out = [torch.empty_like(q) for _ in range(3)]
    p = hk._bwd_params(q, k, v, None, do, lse, D, *out, True, 0.125)
    side = torch.cuda.Stream()

    def call():
        assert hk.lib().hk_attn_backward_set(ctypes.byref(p), 64,
                                             torch.cuda.current_stream().cuda_stream) == 0
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()  # the stream's workspace has its size before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call()
    for _ in range(3):
        for t in out:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip(out, want):
            assert max_rel(got.cpu().numpy(), ref) <= 2e-3


def test_attn_backward_under_capture_in_the_workspace_it_has(hk, orc):
    # a workspace that holds the planes of 12 x 1024 queries and not the partials of shared key tiles,
    # as other shapes leave it: the captured call keeps its key tiles whole
    B, H, T = 1, 12, 1024
    say("attn bwd capture without partials")
    (q, k, v, do, lse), D, want = _case(hk, orc, B, H, T, True)
    out = [torch.empty_like(q) for _ in range(3)]
    small = [torch.randn(25, 12, 64, 64, device=DEV) for _ in range(4)]  # 19,200 rows, none shared
    so, sl = hk.fused_attn_forward(*small[:3], True)
    sd = hk.attn_bwd_precompute_D(small[3], so)
    p = hk._bwd_params(q, k, v, None, do, lse, D, *out, True, 0.125)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        hk.attn_backward(*small, sl, sd, True)
    torch.cuda.synchronize()

    def call():
        assert hk.lib().hk_attn_backward_set(ctypes.byref(p), 64,
                                             torch.cuda.current_stream().cuda_stream) == 0
    with torch.cuda.graph(graph, stream=side):
        call()
    for _ in range(3):
        for t in out:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip(out, want):
            assert max_rel(got.cpu().numpy(), ref) <= 2e-3
        with torch.cuda.stream(side):
            call()  # eager: shares the key tiles, in a larger workspace
        torch.cuda.synchronize()
