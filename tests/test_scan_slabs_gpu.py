"""The scan backward in 64-channel slabs (one gate per channel, bf16): several
workgroups per head.

Exact integer cases where a slab can go wrong: heads of one slab, of one and a
vector (a last slab with one lane of 8), of a slab and a half, of several, the
widest; T of one step, one short of, at and past a tile of 64, several tiles;
few sequences with their time cut into chunks.  Which of these run in slabs and
which with a whole head per workgroup is the library's choice.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ltv_test_utils import (assert_close, int_combined, int_inits, int_logit_bias, np_of,
                            to_torch)
from test_scan_gpu import DEV, _expected, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 72, 96, 128, 200, 256, 512])
@pytest.mark.parametrize("T", [1, 63, 64, 65, 200, 300])
def test_slab_backward_exact(D, T, monkeypatch):
    _exact(2, D, T, monkeypatch)


@pytest.mark.parametrize("D,T", [(40, 200), (64, 65), (64, 200), (72, 65), (128, 130), (200, 65),
                                 (200, 200), (256, 65), (256, 200)])
def test_slab_backward_many_sequences(D, T, monkeypatch):
    """More sequences than compute units, where the slabs are chosen (two tiles and
    more; heads of up to one slab, of several, of a cut last one)."""
    _exact(72, D, T, monkeypatch)


def _exact(B, D, T, monkeypatch):
    from nanochat_amd import _native as N

    monkeypatch.setattr(N, "chain_workspace_for", lambda *a, **k: N._NO_CHAIN)
    NH, NKVH, r, dtype = 2, 1, 1, torch.bfloat16
    H, Da = NH + 2 * NKVH, D
    c = int_combined(B, T, NH, NKVH, Da, r)
    ini, bias = int_inits(B, NH, NKVH, Da, r), int_logit_bias(NH, NKVH, Da, False)
    gy = np.random.default_rng(D + T).integers(-2, 3, size=(B, H, T, D)).astype(np.float32)
    out, (egc, egi, egb) = _expected(c, ini, bias, NH, NKVH, Da, r, False, "bf16", gy)
    grads = [to_torch(g, dtype, DEV) for g in (gy[:, :NH], gy[:, NH:NH + NKVH], gy[:, NH + NKVH:])]
    _, gc, gi, gb = _run(to_torch(c, dtype, DEV), to_torch(ini, dtype, DEV),
                         to_torch(bias, torch.float32, DEV), NH, NKVH, Da, r, False, grads)
    assert_close(np_of(gc), egc, 0, f"grad_combined D={D} T={T}")
    assert_close(np_of(gi), egi, 0, f"grad_inits D={D} T={T}")
    # sums of B T integer terms: exact while they stay below 2**24
    assert_close(np_of(gb), egb, 1e-6, f"grad_logit_bias D={D} T={T}")
