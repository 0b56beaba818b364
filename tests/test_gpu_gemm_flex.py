"""GPU parity of the BF16 GEMM's small tiles and any-alignment tiles (bgemm_flex.hip) against the
CPU oracle's fp32-accumulated reference. Tolerance as in test_gpu_gemm.py: max|err| / max|ref| <=
1e-2 for one bf16 rounding of an fp32 sum (2^-9 of the element plus fp32 rounding)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import max_rel
from test_gpu_gemm import _check, _operands, _run, bits, say, to_dev_bf16, to_host_bits

pytestmark = pytest.mark.gpu
DEV = "cuda"
LAYOUTS = [(0, 0), (0, 1), (1, 0), (1, 1)]


# Edges of the 64-, 128- and 256-row tiles, k tails of one element up to a whole k-tile and one k
# more, k-tile counts that leave the k groups unequal, and odd extents of every operand.
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 64, 64), (65, 63, 65), (63, 65, 127),
                                   (9, 200, 129), (200, 9, 321), (127, 129, 191), (129, 257, 255),
                                   (333, 77, 1111), (255, 1001, 449)])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_bgemm_ragged_and_small(hk, orc, M, N, K, ta, tb):
    assert hk.lib().hk_bgemm_small_tile(ta, tb, M, N, K, 1, 0) in (64, 128, 256)
    say("bgemm flex", M, N, K, ta, tb)
    A, B, C0 = _operands(orc, M, N, K, ta, tb, 2000 + M + N)
    _check(orc, _run(hk, "hk_bgemm", A, B, C0, M, N, K, ta, tb, 1.5, 0.5), A, B, C0, ta, tb, 1.5,
           0.5)


# One shape per tile shape and split that the plan can pick: (rows of the tile, splits > 1)
@pytest.mark.parametrize("M,N,K,ta,tb,tile,split", [
    (512, 768, 2304, 0, 1, 64, False), (80, 136, 576, 0, 1, 64, False),
    (1024, 1024, 1024, 0, 0, 64, False), (192, 384, 4096, 0, 0, 64, True),
    (512, 2304, 768, 0, 0, 128, False), (2048, 2048, 512, 0, 0, 128, False),
    (500, 1003, 333, 1, 0, 64, False), (300, 299, 4001, 0, 0, 64, True),
    (2047, 2049, 257, 0, 1, 128, False), (4095, 4097, 65, 1, 0, None, False),
    (257, 511, 9001, 1, 1, None, True)])
def test_bgemm_plan_shapes(hk, orc, M, N, K, ta, tb, tile, split):
    lib = hk.lib()
    rows = lib.hk_bgemm_small_tile(ta, tb, M, N, K, 1, 0)
    splits = lib.hk_bgemm_split_count(ta, tb, M, N, K, 1, 0)
    say("bgemm flex plan", M, N, K, ta, tb, "tile", rows, "splits", splits)
    assert rows == tile if tile else rows > 0
    assert (splits > 1) == split
    A, B, C0 = _operands(orc, M, N, K, ta, tb, 2100 + M)
    first = _run(hk, "hk_bgemm", A, B, C0, M, N, K, ta, tb, 1.0, 0.5)
    assert np.array_equal(first, _run(hk, "hk_bgemm", A, B, C0, M, N, K, ta, tb, 1.0, 0.5))
    sel = np.unique(np.concatenate([np.arange(0, M, max(1, M // 64)), np.arange(M - 8, M)]))
    Asub = np.ascontiguousarray(A[:, sel] if ta else A[sel])
    ref = orc.bgemm(ta, tb, Asub, B, alpha=1.0, beta=0.5, C0=np.ascontiguousarray(C0[sel]))
    assert max_rel(orc.bf16_to_f32(first[sel]), ref) <= 1e-2


def _padded(rows, cols, ld, offset, fill):
    """A [rows, cols] view with leading dimension ld at element `offset` of a buffer of `fill`."""
    buf = torch.full((offset + rows * ld + 64,), fill, dtype=torch.bfloat16, device=DEV)
    return buf, buf[offset:offset + rows * ld].view(rows, ld)[:, :cols]


@pytest.mark.parametrize("M,N,K", [(70, 45, 100), (131, 200, 67), (264, 136, 200), (300, 520, 72)])
@pytest.mark.parametrize("pad,offset", [(1, 1), (3, 0), (8, 5), (0, 3)])
@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_bgemm_strided_rows_between_nans(hk, orc, M, N, K, pad, offset, ta, tb):
    # Leading dimensions and bases at any 2-byte address; everything around the operands is NaN
    # and must not reach C, and C's own surroundings must stay as they are.
    say("bgemm flex strided", M, N, K, "pad", pad, "offset", offset, ta, tb)
    A, B, C0 = _operands(orc, M, N, K, ta, tb, 2200 + M)
    bufs = []
    for mat in (A, B):
        buf, view = _padded(mat.shape[0], mat.shape[1], mat.shape[1] + pad, offset, float("nan"))
        view.copy_(to_dev_bf16(mat))
        bufs.append((buf, view))
    cbuf, cview = _padded(M, N, N + pad, offset, 7.0)
    cview.copy_(to_dev_bf16(C0))
    before = cbuf.clone()
    (_, a), (_, b) = bufs
    st = hk.lib().hk_bgemm(ta, tb, M, N, K, bits(1.5), a.data_ptr(), a.stride(0), 0, b.data_ptr(),
                           b.stride(0), 0, bits(0.5), cview.data_ptr(), cview.stride(0), 0, 1,
                           torch.cuda.current_stream().cuda_stream)
    assert st == 0
    _check(orc, to_host_bits(cview.contiguous()), A, B, C0, ta, tb, 1.5, 0.5)
    cview.copy_(to_dev_bf16(C0))
    assert torch.equal(cbuf, before)


@pytest.mark.parametrize("which", ["N", "M", "one", "MN"])
@pytest.mark.parametrize("M,N,K", [(77, 131, 95), (264, 520, 136)])
def test_bgemm_flex_bias(hk, orc, which, M, N, K):
    say("bgemm flex bias", which, M, N, K)
    A, B, _ = _operands(orc, M, N, K, 0, 0, 2300)
    n = {"N": N, "M": M, "one": 1, "MN": M * N}[which]
    bias = orc.f32_to_bf16(orc.splitmix_uniform(n, 2301, -1.0, 1.0))
    dA, dB, db = to_dev_bf16(A), to_dev_bf16(B), to_dev_bf16(bias)
    C = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)  # written, not read
    st = hk.lib().hk_bgemm_addmm(M, N, K, bits(1.0), dA.data_ptr(), K, 0, dB.data_ptr(), N, 0,
                                 bits(2.0), db.data_ptr(), n, C.data_ptr(), N, 0, 1,
                                 torch.cuda.current_stream().cuda_stream)
    assert st == 0
    ref = orc.bgemm(0, 0, A, B, alpha=1.0, beta=2.0, bias=bias.reshape(M, N) if which == "MN" else bias)
    assert max_rel(orc.bf16_to_f32(to_host_bits(C)), ref) <= 1e-2


@pytest.mark.parametrize("ta,tb", LAYOUTS)
def test_bgemm_flex_batches_and_split(hk, orc, ta, tb):
    # odd batch strides, an explicit split of rows that the 256-wide tiles do not take
    M, N, K, batch = 67, 85, 403, 3
    say("bgemm flex batches", ta, tb)
    ops = [_operands(orc, M, N, K, ta, tb, 2400 + 10 * b) for b in range(batch)]
    dA, dB, dC = (to_dev_bf16(np.stack([o[i] for o in ops])) for i in range(3))
    lda, ldb = ops[0][0].shape[1], ops[0][1].shape[1]
    st = hk.lib().hk_bgemm(ta, tb, M, N, K, bits(1.0), dA.data_ptr(), lda, M * K, dB.data_ptr(), ldb,
                           N * K, bits(0.5), dC.data_ptr(), N, M * N, batch,
                           torch.cuda.current_stream().cuda_stream)
    assert st == 0
    out = to_host_bits(dC)
    for b, (A, B, C0) in enumerate(ops):
        _check(orc, out[b], A, B, C0, ta, tb, 1.0, 0.5)
    if (ta, tb) != (1, 1):
        A, B, C0 = ops[0]
        _check(orc, _run(hk, "hk_bgemm_core", A, B, C0, M, N, K, ta, tb, 1.0, 0.5, split_k=3), A, B,
               C0, ta, tb, 1.0, 0.5)


# several matrices in a launch: tiles x batches (x splits) that are and are no multiple of the 8 XCDs
@pytest.mark.parametrize("batch,M,N,K,split", [(13, 136, 72, 96, 0), (5, 304, 200, 72, 0), (16, 64, 64, 128, 0),
                                               (7, 67, 131, 45, 0), (9, 130, 67, 403, 3),
                                               (2, 1000, 24, 40, 0), (257, 8, 16, 24, 0)])
@pytest.mark.parametrize("ta,tb", LAYOUTS[:3])
def test_bgemm_flex_matrices_in_a_launch(hk, batch, M, N, K, split, ta, tb):
    say("bgemm flex matrices", batch, M, N, K, split, ta, tb)
    assert hk.lib().hk_bgemm_small_tile(ta, tb, M, N, K, batch, split) > 0
    g = torch.Generator(device=DEV)
    g.manual_seed(M + N + K)
    rand = lambda r, c: torch.randn(batch, r, c, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    a, b = rand(*((K, M) if ta else (M, K))), rand(*((N, K) if tb else (K, N)))
    c = torch.full((batch, M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    tail = (M, N, K, bits(1.0), a.data_ptr(), a.shape[2], M * K, b.data_ptr(), b.shape[2], N * K, 0,
            c.data_ptr(), N, M * N, batch, torch.cuda.current_stream().cuda_stream)
    lay = {(0, 1): 0, (1, 0): 1, (0, 0): 2}[(ta, tb)]
    rc = hk.lib().hk_bgemm_core(lay, split, *tail) if split else hk.lib().hk_bgemm(ta, tb, *tail)
    assert rc == 0
    A = (a.transpose(1, 2) if ta else a).float().contiguous()
    B = (b.transpose(1, 2) if tb else b).float().contiguous()
    ref = torch.stack([torch.mm(A[i], B[i]) for i in range(batch)])
    assert (c.float() - ref).abs().max() <= 1e-2 * ref.abs().max()


@pytest.mark.parametrize("batch,K,split,odd_c", [(40000, 130, 2, False), (40000, 136, 2, True),
                                                 (65535, 65, 2, False), (65536, 72, 1, True),
                                                 (65537, 9, 1, False)])
def test_bgemm_flex_more_batches_than_a_grid_takes(hk, batch, K, split, odd_c):
    # batch x splits past 65535, and batches past it, of rows that are no whole vectors (of A and B, or
    # of C alone): a given split is left out
    M, N = 3, 9
    say("bgemm flex batches x splits", batch, K, split)
    g = torch.Generator(device=DEV)
    g.manual_seed(K)
    a, b = (torch.randn(batch, r, K, generator=g, device=DEV).to(torch.bfloat16) for r in (M, N))
    c = torch.full((batch, M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    assert a.shape[2] % 8 == 0 if odd_c else a.shape[2] % 8
    assert hk.lib().hk_bgemm_core(0, split, M, N, K, bits(1.0), a.data_ptr(), K, M * K, b.data_ptr(), K,
                                  N * K, 0, c.data_ptr(), N, M * N, batch,
                                  torch.cuda.current_stream().cuda_stream) == 0
    ref = (a.float()[:, :, None] * b.float()[:, None]).sum(3)
    assert (c.float() - ref).abs().max() <= 1e-2 * ref.abs().max()


@pytest.mark.parametrize("split_k", [0, 3])
@pytest.mark.parametrize("M,N,K", [(64, 33, 8192), (300, 299, 4001)])
def test_bgemm_unaligned_rows_need_no_workspace_under_capture(hk, orc, M, N, K, split_k):
    # products that split k (N odd: only the rows of C are unaligned) on a stream without a workspace
    say("bgemm capture cold", M, N, K, split_k)
    assert hk.lib().hk_bgemm_split_count(0, 1, M, N, K, 1, split_k) > 1
    A, B, C0 = _operands(orc, M, N, K, 0, 1, 2550)
    dA, dB, dC = to_dev_bf16(A), to_dev_bf16(B), to_dev_bf16(C0)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        args = (M, N, K, bits(1.0), dA.data_ptr(), K, 0, dB.data_ptr(), K, 0, 0, dC.data_ptr(), N, 0, 1,
                torch.cuda.current_stream().cuda_stream)
        rc = (hk.lib().hk_bgemm_core(0, split_k, *args) if split_k
              else hk.lib().hk_bgemm(0, 1, *args))
    assert rc == 0
    for _ in range(3):
        dC.zero_()
        graph.replay()
        _check(orc, to_host_bits(dC), A, B, C0, 0, 1, 1.0, 0.0)


@pytest.mark.parametrize("M,N,K,splits", [(256, 256, 65536, 8), (176, 312, 6152, 8)])
def test_bgemm_deep_k_keeps_the_wide_splits_under_capture(hk, orc, M, N, K, splits):
    # few aligned tiles over a deep k: eager calls split it over small tiles and leave a workspace in which
    # a captured one takes the 256-wide tiles' splits (bit for bit those of an explicit split), not one
    # chain
    lib = hk.lib()
    assert lib.hk_bgemm_small_tile(0, 0, M, N, K, 1, 0) > 0
    assert lib.hk_bgemm_split_count(0, 0, M, N, K, 1, 0) > 1
    say("bgemm capture deep k")
    A, B, C0 = _operands(orc, M, N, K, 0, 0, 2560)
    dA, dB, dC = to_dev_bf16(A), to_dev_bf16(B), to_dev_bf16(C0)
    side = torch.cuda.Stream()

    def call(stream, split_k=0):
        args = (M, N, K, bits(1.0), dA.data_ptr(), K, 0, dB.data_ptr(), N, 0, 0, dC.data_ptr(), N, 0, 1,
                stream)
        assert (lib.hk_bgemm_core(2, split_k, *args) if split_k else lib.hk_bgemm(0, 0, *args)) == 0
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(side.cuda_stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(torch.cuda.current_stream().cuda_stream)
    call(torch.cuda.current_stream().cuda_stream, splits)
    wide = to_host_bits(dC)
    for _ in range(3):
        dC.zero_()
        graph.replay()
        assert np.array_equal(to_host_bits(dC), wide)


def test_bgemm_flex_split_plan_under_capture(hk, orc):
    # A split plan takes the stream's workspace in eager calls and runs unsplit in a captured graph: the
    # replays give the bits of an explicit split of one, which are not the eager call's, also after a
    # larger call has grown the workspace.
    M, N, K = 300, 299, 4001
    lib = hk.lib()
    assert lib.hk_bgemm_split_count(0, 0, M, N, K, 1, 0) > 1
    say("bgemm flex capture")
    A, B, C0 = _operands(orc, M, N, K, 0, 0, 2500)
    dA, dB, dC = to_dev_bf16(A), to_dev_bf16(B), to_dev_bf16(C0)
    big = torch.randn(1500, K, device=DEV).to(torch.bfloat16)
    out = torch.empty(1500, N, device=DEV, dtype=torch.bfloat16)

    def call(stream, split_k=0, a=dA, c=dC, rows=M):
        args = (rows, N, K, bits(1.0), a.data_ptr(), K, 0, dB.data_ptr(), N, 0, 0, c.data_ptr(), N, 0, 1,
                stream)
        assert (lib.hk_bgemm_core(2, split_k, *args) if split_k else lib.hk_bgemm(0, 0, *args)) == 0
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    got = {}
    for name, split_k in (("whole", 1), ("eager", 0)):
        with torch.cuda.stream(side):
            call(side.cuda_stream, split_k)
        torch.cuda.synchronize()
        got[name] = to_host_bits(dC)
        _check(orc, got[name], A, B, C0, 0, 0, 1.0, 0.0)
    assert not np.array_equal(got["whole"], got["eager"])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        call(torch.cuda.current_stream().cuda_stream)
    for i in range(3):
        dC.zero_()
        graph.replay()
        assert np.array_equal(to_host_bits(dC), got["whole"])
        with torch.cuda.stream(side):
            call(side.cuda_stream)
        assert np.array_equal(to_host_bits(dC), got["eager"])
        # 8 x 1500 x 304 fp32 partials: more than the products above take (at most 32 x 300 x 304)
        with torch.cuda.stream(side):
            call(side.cuda_stream, 8, big, out, 1500)
        torch.cuda.synchronize()


# Large outputs of few k are bound by their stores: several rounds of small tiles lose to the 256-wide
# ones there (43.4 us against 28.3 for the first), one round wins.
@pytest.mark.parametrize("M,N,K,small", [(5208, 6880, 80, False), (1704, 6208, 64, False),
                                         (536, 9576, 312, False), (512, 50304, 64, False),
                                         (1024, 4096, 64, True), (2048, 2048, 16, True),
                                         (1432, 2160, 368, True)])
def test_bgemm_small_tiles_by_rounds(hk, M, N, K, small):
    assert (hk.lib().hk_bgemm_small_tile(0, 1, M, N, K, 1, 0) > 0) == small


# The 256-wide tiles at sizes that the library itself now gives to the small ones.
@pytest.mark.parametrize("M,N,K,ta,tb,rows,cols", [
    (192, 256, 64, 0, 0, 192, 256), (200, 264, 136, 0, 1, 192, 256), (400, 512, 72, 0, 0, 192, 256),
    (1000, 136, 520, 0, 1, 192, 256), (256, 160, 64, 0, 1, 256, 160), (1024, 800, 320, 0, 1, 256, 160),
    (2048, 1280, 192, 0, 1, 256, 160), (512, 384, 128, 1, 0, 256, 256), (136, 72, 200, 1, 0, 256, 256)])
def test_bgemm_wide_tiles_small_sizes(hk, orc, M, N, K, ta, tb, rows, cols):
    lib = hk.lib()
    assert lib.hk_bgemm_small_tile(ta, tb, M, N, K, 1, 1) == 0
    assert lib.hk_bgemm_tile_rows(ta, tb, M, N, K, 1, 1) == rows
    assert lib.hk_bgemm_tile_cols(ta, tb, M, N, K, 1, 1) == cols
    say("bgemm wide small", M, N, K, ta, tb)
    A, B, C0 = _operands(orc, M, N, K, ta, tb, 2600 + M)
    _check(orc, _run(hk, "hk_bgemm_core", A, B, C0, M, N, K, ta, tb, 1.5, 0.5, split_k=1), A, B, C0,
           ta, tb, 1.5, 0.5)


@pytest.mark.parametrize("N", [8185, 8191])
def test_bgemm_wide_tiles_odd_logits(hk, orc, N):
    # aligned operands, rows of C of odd length: the 256-wide tiles with the element-wise column edge
    M, K = 2048, 136
    assert hk.lib().hk_bgemm_small_tile(0, 1, M, N, K, 1, 0) == 0
    say("bgemm wide odd N", N)
    A, B, C0 = _operands(orc, M, N, K, 0, 1, 2700)
    out = _run(hk, "hk_bgemm", A, B, C0, M, N, K, 0, 1, 1.0, 0.5)
    sel = np.arange(0, M, 31)
    ref = orc.bgemm(0, 1, A[sel], B, alpha=1.0, beta=0.5, C0=np.ascontiguousarray(C0[sel]))
    assert max_rel(orc.bf16_to_f32(out[sel]), ref) <= 1e-2
