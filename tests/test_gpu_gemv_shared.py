"""GPU parity of the NT row GEMV with one matrix for all batches (stride 0): two or four vectors
share a pass over it. Every batch count that leaves a group part-filled, aligned and unaligned
rows, and a strided vector, against the oracle at the bf16 GEMM bar (1e-2 of max|ref|); each
batch equals a call for that batch alone bit for bit where both split k alike."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import max_rel

pytestmark = pytest.mark.gpu
ONE = 0x3F80


@pytest.mark.parametrize("batch", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("R,K,off", [(17, 136, 0), (1001, 768, 0), (1001, 921, 1), (16, 4099, 3),
                                     (40000, 72, 0), (3, 5, 0)])
def test_batches_of_one_matrix(hk, orc, R, K, off, batch):
    print("[case] shared gemv", R, K, off, batch, flush=True)
    sx = K + 3 if off else (K + 7) // 8 * 8  # off 0: every row 16-byte aligned where K allows it
    g = np.random.default_rng(R + K + batch)
    m = orc.f32_to_bf16(g.standard_normal((R, K)).astype(np.float32))
    x = orc.f32_to_bf16(g.standard_normal((batch, K)).astype(np.float32))
    mb = torch.full((R * K + off + 64,), 0x7FC0, dtype=torch.int16, device="cuda")
    xb = torch.full((batch * sx + 64,), 0x7FC0, dtype=torch.int16, device="cuda")
    mb[off:off + R * K] = torch.from_numpy(m.view(np.int16).reshape(-1)).cuda()
    for b in range(batch):
        xb[b * sx:b * sx + K] = torch.from_numpy(x[b].view(np.int16)).cuda()
    y = torch.full((batch, R + 1), 0x7FC0, dtype=torch.int16, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    e = 2

    def call(n, sx_from, out):
        rc = hk.lib().hk_bgemv_nt_row(R, K, ONE, xb.data_ptr() + e * sx_from * sx,
                                      mb.data_ptr() + e * off, K, 0, out.data_ptr(), n, sx, 0,
                                      R + 1, s)
        assert rc == 0

    call(batch, 0, y)
    got = y.cpu().numpy().view(np.uint16)
    assert (got[:, R] == 0x7FC0).all()
    ref = orc.bgemm(0, 1, x, m, 1.0, 0.0, np.zeros((batch, R), np.uint16))
    assert max_rel(orc.bf16_to_f32(got[:, :R]), ref) <= 1e-2
    if R >= 40000:  # enough rows that neither call splits k
        one = torch.full((1, R + 1), 0x7FC0, dtype=torch.int16, device="cuda")
        for b in range(batch):
            call(1, b, one)
            assert np.array_equal(one.cpu().numpy().view(np.uint16)[0, :R], got[b, :R])
