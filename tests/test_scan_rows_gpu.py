"""The scan's row modes: values that lie time-contiguous, one row per channel
(the transposed view of a (B, F, T) projection), read and written in quads of 4
steps.

Exact integer cases where quads can go wrong: T one quad, not a multiple of 4
(the last quad is read early and shifted), tiles and chunks with a remainder,
rows that start inside a dword (odd row pitch, odd storage offset), head widths
that leave channel lanes idle, every kernel the modes are built into (chained,
tile, tile with time chunks).  Oracle: the sequential recurrence.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ltv_test_utils import (assert_close, int_combined, int_inits, int_logit_bias, io_name, np_of,
                            to_torch)
from test_scan_gpu import DEV, DTYPES, _expected, _op

pytestmark = pytest.mark.gpu

# (steps between two rows' starts - T, elements before the first row)
PITCHES = [(0, 0), (1, 0), (3, 1), (8, 2)]


def _rows_view(a, pitch, offset, dtype):
    """a (B, T, F) as the transposed view of (B, F, T) rows, T + pitch apart."""
    B, T, F = a.shape
    buf = torch.full((offset + B * F * (T + pitch),), float("nan"), dtype=dtype, device=DEV)
    v = buf[offset:].view(B, F, T + pitch)[:, :, :T].transpose(1, 2)
    v.copy_(to_torch(a, dtype, DEV))
    return buf, v


def _check(dtype, B, NH, NKVH, D, r, T, pitch, offset):
    """Forward and backward of the op's kernels on such a view; grad_combined
    goes into another one, whose gaps must stay untouched."""
    ops = torch.ops.nanochat_cuda
    name = "ltv_fused_concat_head_major_register_cast_blelloch_scan_cuda_"
    Da, H = D // r, NH + 2 * NKVH
    c = int_combined(B, T, NH, NKVH, Da, r)
    ini, bias = int_inits(B, NH, NKVH, Da, r), int_logit_bias(NH, NKVH, Da, False)
    gy = np.random.default_rng(T).integers(-2, 3, size=(B, H, T, D)).astype(np.float32)
    out, (egc, egi, egb) = _expected(c, ini, bias, NH, NKVH, Da, r, False, io_name(dtype), gy)
    _, comb = _rows_view(c, pitch, offset, dtype)
    ini_d, bias_d = to_torch(ini, dtype, DEV), to_torch(bias, torch.float32, DEV)
    with torch.no_grad():
        h = _op()(comb, ini_d, bias_d, NH, NKVH, Da, r, 8, 8, 4, 32, 2, 8, False)
    case = f"{io_name(dtype)} B={B} D={D} r={r} T={T} pitch={pitch} offset={offset}"
    for got, want, n in zip(h, out, "qkv"):
        assert_close(np_of(got), want, 0, f"{n} {case}")
    g = [to_torch(x, dtype, DEV) for x in (gy[:, :NH], gy[:, NH:NH + NKVH], gy[:, NH + NKVH:])]
    buf, gc = _rows_view(np.zeros_like(c), pitch, offset, dtype)
    gi, gb = torch.empty_like(ini_d), torch.empty_like(bias_d)
    getattr(ops, name + "backward_kernel")(comb, ini_d, bias_d, *h, *g, gc, gi, gb, NH, NKVH, Da,
                                           r, 32, 2, 8, False)
    assert_close(np_of(gc), egc, 0, "grad_combined " + case)
    assert_close(np_of(gi), egi, 0, "grad_inits " + case)
    # sums of B T integer terms past 2**24: the order of the fp32 sums shows
    assert_close(np_of(gb), egb, 1e-6, "grad_logit_bias " + case)
    gaps = buf.numel() - gc.numel()
    assert int(torch.isnan(buf.float()).sum()) == gaps, "gaps written: " + case


@pytest.mark.parametrize("dtype", DTYPES, ids=io_name)
@pytest.mark.parametrize("T", [4, 5, 6, 7, 63, 64, 65, 130, 259, 1030])
def test_rows_few_sequences(dtype, T):
    """The forward's tile kernel; the backward chained from two chunks on (up to
    16), the tile kernels below and above."""
    for D, r in ((128, 128), (64, 16), (32, 32)):
        for pitch, offset in PITCHES:
            _check(dtype, 1, 2, 1, D, r, T, pitch, offset)


@pytest.mark.parametrize("dtype", DTYPES, ids=io_name)
@pytest.mark.parametrize("T", [3585, 4096, 4099, 4606])
def test_rows_chained_forward(dtype, T):
    """The chained forward, two quads of steps per lane: it takes sequences from 8
    chunks of 512 steps on (a last chunk of one step, a whole one, one of
    three steps, one whose last quad is cut)."""
    from nanochat_amd import _native as N

    for D, r, NH, NKVH in ((128, 128, 1, 1), (64, 16, 2, 1)):
        assert N.lib().ltv_hm_scan_forward_chain_workspace_size(
            N.dtype_code(dtype), 1, T, NH, NKVH, D // r, r) > 0
        for pitch, offset in PITCHES:
            _check(dtype, 1, NH, NKVH, D, r, T, pitch, offset)


@pytest.mark.parametrize("dtype", DTYPES, ids=io_name)
@pytest.mark.parametrize("T", [9, 64, 131, 300])
def test_rows_many_sequences(dtype, T):
    """256 sequences and more: the tile kernels over several tiles; a head of
    96 channels leaves a quarter of its channel lanes idle."""
    for D, r in ((128, 128), (96, 32), (64, 64)):
        for pitch, offset in PITCHES[:3]:
            _check(dtype, 26, 4, 3, D, r, T, pitch, offset)


@pytest.mark.parametrize("dtype", DTYPES, ids=io_name)
@pytest.mark.parametrize("T", [200, 517])
def test_rows_time_chunks(dtype, T, monkeypatch):
    """Without a chain workspace few sequences run in time chunks, each
    entered from its chunk map."""
    from nanochat_amd import _native as N

    monkeypatch.setattr(N, "chain_workspace_for", lambda *a, **k: N._NO_CHAIN)
    for pitch, offset in PITCHES:
        _check(dtype, 2, 2, 1, 128, 128, T, pitch, offset)
