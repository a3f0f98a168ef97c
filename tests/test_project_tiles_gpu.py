"""The projection GEMMs' 128 x 128 tiles (few tokens) against the 256 x 256
ones: a token's forward row and grad_x row are the same products summed in the
same order whichever tile computes them, so the rows must be bitwise those of a
call with enough tokens for the large tiles; grad_weight, split elsewhere, stays
within the bound of an fp32 sum of the same bf16 products.

Sizes where it can go wrong: one token, one short of and one past a tile,
channel counts that cut a tile inside and leave a tile of 8 columns, feature
counts that end in a partial k-step, a reduction cut into several splits with a
ragged last one, the largest sizes of each rule and the first past it.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
BIG = 40960  # tokens: past every small-tile rule at the widths below


def _case(C, H, D, Da, M, seed):
    from nanochat_amd.ops import ltv_hm_fast as hm
    F, Fp = H * (D + Da), hm.packed_width(H, D, Da)
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(1, M, C, generator=g, device=DEV).bfloat16()
    w = torch.randn(F, C, generator=g, device=DEV) * C ** -0.5
    gc = torch.randn(1, M, Fp, generator=g, device=DEV).bfloat16()
    gc[..., F:] = 0
    return x, w, hm.pack_weight(w, H, D, Da), gc, F


@pytest.mark.parametrize("C,H,D,Da", [(768, 18, 128, 1), (136, 5, 64, 4), (1024, 9, 24, 3)],
                         ids=lambda v: str(v))
def test_rows_equal_the_large_tiles(C, H, D, Da):
    from nanochat_amd.ops import ltv_hm_fast as hm
    x, w, wp, gc, F = _case(C, H, D, Da, BIG, C)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    fcols = -(-hm.packed_width(H, D, Da) // 128)
    ccols = -(-C // 128)
    v, lg = hm.project(x, w, H, D, Da)[:2]
    gx, _ = hm.project_backward(x, wp, gc, H, D, Da, pad_zeroed=True)
    # token counts at the forward's and grad_x's lines, and one tile past them
    lines = {2 * cus // fcols * 128, cus // ccols * 128}
    for M in sorted({1, 127, 128, 129, 1000} | {m + d for m in lines for d in (0, 1)}):
        if M >= BIG:
            continue
        xs, gs = x[:, :M].contiguous(), gc[:, :M].contiguous()
        vs, ls = hm.project(xs, w, H, D, Da)[:2]
        assert torch.equal(vs, v[:, :, :M]) and torch.equal(ls, lg[:, :M]), f"forward M={M}"
        gxs, _ = hm.project_backward(xs, wp, gs, H, D, Da, pad_zeroed=True)
        assert torch.equal(gxs, gx[:, :M]), f"grad_x M={M}"


@pytest.mark.parametrize("M", [1, 64, 511, 513, 1025, 2111, 4096, 5439, 8192, 20000])
@pytest.mark.parametrize("C,H,D,Da", [(768, 18, 128, 1), (136, 5, 64, 4), (256, 4, 128, 1)],
                         ids=lambda v: str(v))
def test_grad_weight(C, H, D, Da, M):
    from nanochat_amd.ops import ltv_hm_fast as hm
    x, w, wp, gc, F = _case(C, H, D, Da, M, M)
    _, gw = hm.project_backward(x, wp, gc, H, D, Da, pad_zeroed=True)
    gcd, xd = gc[0, :, :F].double(), x[0].double()
    # packed columns: the values of all heads, then the logits
    rows = torch.cat([gcd[:, :H * D].view(M, H, D), gcd[:, H * D:].view(M, H, Da)], -1)
    rows = rows.reshape(M, F)
    want = rows.T @ xd
    # an fp32 sum of n products in any order errs by at most n 2^-24 sum |a b|;
    # n: the M products and the partial sums of the splits
    bound = (M + 64) * 2.0 ** -24 * (rows.abs().T @ xd.abs())
    err = (gw.double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound.clamp_min(1e-30)).max())
