"""The stream workspace and graph capture: a captured graph keeps the workspace it was captured with when
later calls on the stream need a larger one."""
from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def say(*a):
    print("[case]", *a, flush=True)


def _grow(hk, stream, times):
    """Split products whose partials need a larger workspace each time (2 to 20 MB and more)."""
    lib = hk.lib()
    for i in range(times):
        M, N, K = 300 * (i + 1), 299, 4001
        splits = lib.hk_bgemm_split_count(0, 0, M, N, K, 1, 4)
        assert splits == 4
        a = torch.ones(M, K, device=DEV, dtype=torch.bfloat16)
        b = torch.ones(K, N, device=DEV, dtype=torch.bfloat16)
        c = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
        with torch.cuda.stream(stream):
            assert lib.hk_bgemm_core(2, splits, M, N, K, 0x3F80, a.data_ptr(), K, 0, b.data_ptr(), N, 0, 0,
                                     c.data_ptr(), N, 0, 1, stream.cuda_stream) == 0
        torch.cuda.synchronize()
        assert bool((c.float() == 4000.0).all())  # 4001 rounded to bf16


@pytest.mark.parametrize("what", ["layer norm", "sgemm", "attention"])
def test_graph_keeps_its_workspace(hk, what):
    say("workspace", what)
    g = torch.Generator(device=DEV)
    g.manual_seed(7)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    side = torch.cuda.Stream()
    if what == "layer norm":
        x, dy = rand(600, 768), rand(600, 768)
        _, m, r = hk.layer_norm_forward(x)
        dx, sums = torch.empty_like(x), torch.zeros(2, 768, device=DEV)
        out = [dx, sums]

        def call():
            sums.zero_()
            hk.layer_norm_backward(dy, x, m, r, None, sums[0], sums[1], grad_x=dx)
    elif what == "sgemm":
        a, b, c = rand(64, 96), rand(96, 128), torch.empty(64, 128, device=DEV)
        out = [c]

        def call():
            hk.call("hk_sgemm", 2, 64, 128, 96, 1.0, a.data_ptr(), 96, 0, b.data_ptr(), 128, 0, 0.0,
                    c.data_ptr(), 128, 0, None, 0, 1, 0, torch.cuda.current_stream().cuda_stream)
    else:
        q, k, v, do = (rand(1, 2, 100, 64) for _ in range(4))
        o, lse = hk.fused_attn_forward(q, k, v, True)
        D = hk.attn_bwd_precompute_D(do, o)
        out = [torch.empty_like(q) for _ in range(3)]
        p = hk._bwd_params(q, k, v, None, do, lse, D, *out, True, 0.125)

        def call():
            hk.call("hk_attn_backward_set", ctypes.byref(p), 64,
                    torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.synchronize()
    want = [t.clone() for t in out]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call()
    for times in (1, 3, 2):
        _grow(hk, side, times)
        for t in out:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip(out, want):
            # dQ is accumulated with atomics: a few fp32 roundings apart
            assert (got - ref).abs().max() <= 1e-5 * ref.abs().max()
