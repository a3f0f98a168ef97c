"""The look-back backward's fold of later windows' warm-ups into du, a 16-byte
vector per thread: exact integer cases against the oracle and, for the same
values in a layout without vectors, against the element form.

Heads of one vector and of several, one and many gates; warm-ups longer than a
chunk (several windows per step), a last window of one step, no warm-up past
the first chunk.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ltv_test_utils import int_combined, int_inits, int_logit_bias, io_name, to_torch
from test_look_back_gpu import DEV, DTYPES, _check, _expected, _grads, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES, ids=io_name)
@pytest.mark.parametrize("D,r", [(8, 8), (16, 1), (128, 128), (72, 8)])
@pytest.mark.parametrize("T,pqk", [(65, (64, 60, 21)), (70, (5, 6, 20)), (131, (30, 20, 45)),
                                   (40, (64, 60, 21))], ids=str)
def test_fold_exact(dtype, D, r, T, pqk):
    B, NH, NKVH = 2, 2, 1
    Da, H = D // r, NH + 2 * NKVH
    c = int_combined(B, T, NH, NKVH, Da, r)
    ini, bias = int_inits(B, NH, NKVH, Da, r), int_logit_bias(NH, NKVH, Da, False)
    gy = np.random.default_rng(D + T).integers(-2, 3, size=(B, H, T, D)).astype(np.float32)
    want = _expected(c, ini, bias, NH, NKVH, Da, r, pqk, False, io_name(dtype), gy)
    btf = to_torch(c, dtype, DEV)
    bft = to_torch(np.ascontiguousarray(c.transpose(0, 2, 1)), dtype, DEV).transpose(1, 2)
    for comb in (btf, bft):
        got = _run("blelloch", comb, to_torch(ini, dtype, DEV), to_torch(bias, torch.float32, DEV),
                   NH, NKVH, Da, r, pqk, False, _grads(gy, NH, NKVH, dtype))
        _check(got, want, 0, f"{io_name(dtype)} D={D} r={r} T={T} pqk={pqk}")
