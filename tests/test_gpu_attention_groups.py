"""hk_fused_attn_forward on grids small enough for two key groups per workgroup (more than 128 keys) and
on fewer keys, against a float64 reference: key counts and masks that leave the second group without a
tile, with a partial one, or one tile behind; dropout, and rows whose keys one group holds alone or that keep nothing. Tolerance: the
bf16x3 products (relative 2^-16 each) summed over 64 products and T keys of weight 1 in all,
1e-4 of max|ref|. The same heads in a grid too large for it take one group and agree as closely."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, causal, mask):
    T = q.shape[2]
    s = torch.matmul(q.double().cpu(), k.double().cpu().transpose(2, 3)) / 8.0
    if causal:
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool).triu(1), float("-inf"))
    top = s.max(3, keepdim=True).values
    e = (s - top).exp()
    if mask is not None:
        e = e * mask.double().cpu()
    z = e.sum(3, keepdim=True)
    o = torch.matmul(e, v.double().cpu()) / torch.where(z > 0, z, torch.ones_like(z))
    return o, (top + z.log()).squeeze(3)


@pytest.mark.parametrize("drop", [False, True])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 63, 65, 128, 129, 160, 161, 193, 333, 516])
def test_key_groups(hk, T, causal, drop):
    print("[case] attention groups", T, causal, drop, flush=True)
    torch.manual_seed(T)
    # 700 heads fill more than one workgroup per CU; a few of them alone do not
    q, k, v = (torch.randn(350, 2, T, 64, device="cuda") * 2 for _ in range(3))
    q, k, v = (t[:350 if T <= 129 else 2] for t in (q, k, v))
    mask = None
    if drop:
        mask = (torch.rand(q.shape[0], 2, T, T, device="cuda") < 0.75).float() / 0.75
        mask[0, 0, T // 2] = 0.0
        mask[0, 1, :, 32:] = 0.0
    kw = {} if mask is None else {"dropout_p": 0.25, "dropout_mask": mask}
    few = {} if mask is None else {"dropout_p": 0.25, "dropout_mask": mask[:2].contiguous()}
    o, lse = hk.fused_attn_forward(q[:2].contiguous(), k[:2].contiguous(), v[:2].contiguous(), causal,
                                   **few)
    ro, rl = _reference(q[:2], k[:2], v[:2], causal, None if mask is None else mask[:2])
    assert (o.double().cpu() - ro).abs().max() <= 1e-4 * ro.abs().max()
    kept = torch.isfinite(rl)
    assert torch.equal(torch.isfinite(lse.cpu()), kept)
    assert (lse.double().cpu()[kept] - rl[kept]).abs().max() <= 1e-4
    if q.shape[0] > 2:
        whole, _ = hk.fused_attn_forward(q, k, v, causal, **kw)
        assert (whole[:2] - o).abs().max().item() <= 2e-4 * ro.abs().max()
