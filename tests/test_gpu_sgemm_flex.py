"""GPU parity of the FP32 GEMM over rows of any length and alignment and over small products
(sgemm_flex.hip; the small bf16x3 products on bgemm_flex.hip), against float64 products of the same
inputs. fp32 products and sums over K <= 4096 stay within 1e-5 of the largest output; bf16x3 within
the 2e-3 of test_gpu_gemm.py (measured 1e-5)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import max_rel
from test_gpu_gemm import DEV, SG_LAYOUT, _sg_call, _sg_operands, say

pytestmark = pytest.mark.gpu


def _ref(A, B, ta, tb, alpha=1.0, beta=0.0, C0=0.0, bias=0.0):
    a = (A.T if ta else A).astype(np.float64)
    b = (B.T if tb else B).astype(np.float64)
    return alpha * (a @ b) + beta * C0 + bias


# Edges of the 32-, 64- and 128-row tiles, k tails, k-tile counts that leave the four k groups
# unequal, 4-multiples that are no 8-multiples, and products for each tile shape
@pytest.mark.parametrize("M,N,K", [(4, 4, 4), (5, 7, 6), (31, 33, 31), (33, 31, 33), (64, 65, 97),
                                   (63, 130, 129), (129, 127, 161), (333, 77, 1111), (511, 513, 65),
                                   (1001, 1203, 203), (2049, 2047, 67), (132, 204, 268),
                                   (1028, 516, 36)])
@pytest.mark.parametrize("lay", ["NN", "NT", "TN"])
def test_sgemm_any_rows(hk, orc, M, N, K, lay):
    enum, ta, tb = SG_LAYOUT[lay]
    say("sgemm flex", lay, M, N, K)
    A, B, C0, bias = _sg_operands(orc, M, N, K, ta, tb, 31 + M)
    t = lambda x: torch.from_numpy(x.copy()).to(DEV)  # noqa: E731
    for split_k in (0, 3):
        out = _sg_call(hk, "hk_sgemm", enum, t(A), t(B), t(C0), M, N, K, 1.5, 0.5, bias=t(bias),
                       bias_stride=N, split_k=split_k)
        assert max_rel(out, _ref(A, B, ta, tb, 1.5, 0.5, C0, bias)) <= 1e-5
    same = _sg_call(hk, "hk_sgemm", enum, t(A), t(B), t(C0), M, N, K, 1.5, 0.5, bias=t(bias),
                    bias_stride=N, split_k=3)
    assert np.array_equal(out, same)


def test_sgemm_any_rows_error_not_above_fp32_sums(hk, orc):
    # against 64 bits the exact fp32 products on the MFMA are no further off than numpy's fp32 product
    for M, N, K in ((333, 301, 1111), (1023, 1025, 2047)):
        A, B, _, _ = _sg_operands(orc, M, N, K, 0, 0, 41, normal=True)
        out = _sg_call(hk, "hk_sgemm", 2, torch.from_numpy(A).to(DEV), torch.from_numpy(B).to(DEV),
                       torch.zeros(M, N, device=DEV), M, N, K, 1.0, 0.0, split_k=0)
        ref = _ref(A, B, 0, 0)
        serial = np.zeros((M, N), np.float32)
        for k in range(K):  # the k-order fp32 sum that these shapes took before
            serial += A[:, k:k + 1] * B[k]
        err = lambda x: np.linalg.norm(x - ref) / np.linalg.norm(ref)  # noqa: E731
        say("sgemm flex error", err(out), "k-order", err(serial))
        assert err(out) <= err(serial)


@pytest.mark.parametrize("M,N,K", [(132, 204, 2052), (68, 380, 2404), (260, 260, 4100),
                                   (516, 516, 8196)])
@pytest.mark.parametrize("lay", ["NN", "NT", "TN"])
def test_sgemm_multiples_of_four_error_not_above_the_split_tiles(hk, orc, M, N, K, lay):
    # few 256 x 256 tiles over a deep k ran split 8 ways; the small tiles that take them now may be no
    # further from 64 bits. Both are root mean squares over more than 20,000 outputs: 5% for chance.
    enum, ta, tb = SG_LAYOUT[lay]
    A, B, _, _ = _sg_operands(orc, M, N, K, ta, tb, 43, normal=True)
    assert hk.lib().hk_sgemm_split_count(enum, M, N, K, 1, 0) == 1
    assert hk.lib().hk_sgemm_split_count(enum, M, N, K, 1, 8) >= 7
    ref, err = _ref(A, B, ta, tb), []
    for split_k in (8, 0):
        out = _sg_call(hk, "hk_sgemm", enum, torch.from_numpy(A).to(DEV), torch.from_numpy(B).to(DEV),
                       torch.zeros(M, N, device=DEV), M, N, K, 1.0, 0.0, split_k=split_k)
        err.append(np.linalg.norm(out - ref) / np.linalg.norm(ref))
    say("sgemm flex error", lay, M, N, K, "split 8", err[0], "small tiles", err[1])
    assert err[1] <= 1.05 * err[0]


@pytest.mark.parametrize("pad,offset", [(1, 1), (2, 0), (4, 3), (0, 2)])
@pytest.mark.parametrize("lay", ["NN", "NT", "TN"])
def test_sgemm_strided_rows_between_nans(hk, orc, pad, offset, lay):
    enum, ta, tb = SG_LAYOUT[lay]
    for M, N, K in ((70, 45, 100), (131, 200, 67), (264, 136, 200)):
        say("sgemm flex strided", lay, M, N, K, pad, offset)
        A, B, C0, _ = _sg_operands(orc, M, N, K, ta, tb, 51)

        def padded(mat, fill):
            r, c = mat.shape
            buf = torch.full((offset + r * (c + pad) + 64,), fill, device=DEV)
            v = buf[offset:offset + r * (c + pad)].view(r, c + pad)[:, :c]
            v.copy_(torch.from_numpy(mat))
            return buf, v
        (_, a), (_, b), (cbuf, c) = padded(A, float("nan")), padded(B, float("nan")), padded(C0, 7.0)
        before = cbuf.clone()
        assert hk.lib().hk_sgemm(enum, M, N, K, 1.5, a.data_ptr(), a.stride(0), 0, b.data_ptr(),
                                 b.stride(0), 0, 0.5, c.data_ptr(), c.stride(0), 0, 0, 0, 1, 0,
                                 torch.cuda.current_stream().cuda_stream) == 0
        # (264, 136, 200) with pad 4 or an even base may take bf16x3: its bound
        assert max_rel(c.cpu().numpy(), _ref(A, B, ta, tb, 1.5, 0.5, C0)) <= 2e-3
        c.copy_(torch.from_numpy(C0))
        assert torch.equal(cbuf, before)


@pytest.mark.parametrize("stride", ["N", "MN", "1"])
def test_sgemm_any_rows_bias_and_batches(hk, orc, stride):
    M, N, K, batch = 35, 45, 77, 3
    say("sgemm flex bias", stride)
    ops = [_sg_operands(orc, M, N, K, 0, 0, 61 + 10 * b) for b in range(batch)]
    A, B, C = (torch.from_numpy(np.stack([o[i] for o in ops])).to(DEV) for i in range(3))
    n = {"N": N, "MN": M * N, "1": 1}[stride]
    bias = orc.splitmix_uniform(n, 69)
    out = _sg_call(hk, "hk_sgemm", 2, A, B, C, M, N, K, 1.0, -0.5, bias=torch.from_numpy(bias).to(DEV),
                   bias_stride=n, split_k=0, batch=batch, sA=M * K, sB=K * N, sC=M * N)
    for b in range(batch):
        add = bias if stride == "N" else bias[(b % M) * N:(b % M + 1) * N] if stride == "MN" else bias[0]
        assert max_rel(out[b], _ref(ops[b][0], ops[b][1], 0, 0, 1.0, -0.5, ops[b][2], add)) <= 1e-5


@pytest.mark.parametrize("M,N,K", [(64, 64, 64), (264, 136, 200), (512, 768, 2304), (1024, 2304, 768),
                                   (256, 256, 4096)])
@pytest.mark.parametrize("lay", ["NN", "NT", "TN"])
def test_sgemm_bf16x3_small_tiles(hk, orc, M, N, K, lay):
    # small bf16x3 products on the small tiles: fp32 C from the tiles or from split partials
    enum, ta, tb = SG_LAYOUT[lay]
    say("sgemm bf16x3 small", lay, M, N, K, "splits", hk.lib().hk_sgemm_split_count(enum, M, N, K, 1, 0))
    A, B, C0, bias = _sg_operands(orc, M, N, K, ta, tb, 71 + M)
    t = lambda x: torch.from_numpy(x.copy()).to(DEV)  # noqa: E731
    out = _sg_call(hk, "hk_sgemm", enum, t(A), t(B), t(C0), M, N, K, 1.5, 0.5, bias=t(bias),
                   bias_stride=N, split_k=0)
    assert max_rel(out, _ref(A, B, ta, tb, 1.5, 0.5, C0, bias)) <= 5e-5


@pytest.mark.parametrize("M,N,K", [(256, 256, 4096), (64, 128, 8192)])
def test_sgemm_bf16x3_under_capture_in_the_workspace_it_has(hk, orc, M, N, K):
    # a workspace that holds the split operands and no partials: the captured product does without
    say("sgemm capture", M, N, K)
    lib = hk.lib()
    assert lib.hk_sgemm_split_count(2, M, N, K, 1, 0) > 1
    A, B, C0, _ = _sg_operands(orc, M, N, K, 0, 0, 81)
    a, b, c = (torch.from_numpy(x.copy()).to(DEV) for x in (A, B, C0))
    side = torch.cuda.Stream()

    def call(split_k):
        assert lib.hk_sgemm(2, M, N, K, 1.0, a.data_ptr(), K, 0, b.data_ptr(), N, 0, 0.0, c.data_ptr(), N,
                            0, None, 0, 1, split_k, torch.cuda.current_stream().cuda_stream) == 0
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(1)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(0)
    for _ in range(3):
        c.zero_()
        graph.replay()
        assert max_rel(c.cpu().numpy(), _ref(A, B, 0, 0)) <= 5e-5
        with torch.cuda.stream(side):
            call(0)  # eager: grows the workspace
        torch.cuda.synchronize()
