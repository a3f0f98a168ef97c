"""The time-chunked scan backward (chunk maps, carries, then the tile kernel per
chunk), which runs where no chain workspace is given and few sequences leave the
device idle.

Exact integer cases at the chunks' edges (T one short of, at and past two
chunks, a last chunk of one step, many chunks, runs shorter than a chunk's time
lanes), for every way a lane finds its gates, 16-byte and element accesses, and
head widths that leave channel lanes idle.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ltv_test_utils import (assert_close, int_combined, int_inits, int_logit_bias, io_name, np_of,
                            to_torch)
from test_scan_gpu import DEV, DTYPES, _expected, _run

pytestmark = pytest.mark.gpu

# (head width, channels per gate): one gate per lane, whole groups in a lane, one
# per channel; D = 24 and 96 leave lanes idle, D = 10 has no 16-byte vectors
WIDTHS = [(128, 128), (64, 16), (128, 1), (32, 4), (24, 24), (96, 96), (10, 2)]


@pytest.mark.parametrize("dtype", DTYPES, ids=io_name)
@pytest.mark.parametrize("T", [129, 255, 256, 257, 385, 1153, 2049])
def test_chunked_backward_exact(dtype, T, monkeypatch):
    from nanochat_amd import _native as N

    monkeypatch.setattr(N, "chain_workspace_for", lambda *a, **k: N._NO_CHAIN)
    B, NH, NKVH = 1, 2, 1
    H = NH + 2 * NKVH
    for D, r in WIDTHS:
        Da = D // r
        c = int_combined(B, T, NH, NKVH, Da, r)
        ini, bias = int_inits(B, NH, NKVH, Da, r), int_logit_bias(NH, NKVH, Da, False)
        gy = np.random.default_rng(D + T).integers(-2, 3, size=(B, H, T, D)).astype(np.float32)
        out, (egc, egi, egb) = _expected(c, ini, bias, NH, NKVH, Da, r, False, io_name(dtype), gy)
        grads = [to_torch(g, dtype, DEV)
                 for g in (gy[:, :NH], gy[:, NH:NH + NKVH], gy[:, NH + NKVH:])]
        _, gc, gi, gb = _run(to_torch(c, dtype, DEV), to_torch(ini, dtype, DEV),
                             to_torch(bias, torch.float32, DEV), NH, NKVH, Da, r, False, grads)
        case = f"{io_name(dtype)} D={D} r={r} T={T}"
        assert_close(np_of(gc), egc, 0, "grad_combined " + case)
        assert_close(np_of(gi), egi, 0, "grad_inits " + case)
        # sums of T integer terms past 2**24: the order of the fp32 sums shows
        assert_close(np_of(gb), egb, 1e-6, "grad_logit_bias " + case)
