"""The strided bf16-MFMA GEMM behind ``fused_linear_transpose``: fp32 operands
as three bf16 pieces each, bf16 operands of any alignment.

Sizes where it can go wrong: reductions of no, one, an even and an odd number of
whole k-steps (16 or 32 indices) with and without a partial one, rows cut inside
a chunk of 8 (fewer than 8, one past, one short of a chunk and of a tile), odd
row pitches, both tile sizes (128 x 128 where those fill the device), several
reduction splits.  Bounds: the worst case of an fp32 sum, as for the op.
Infinities, NaNs and values past the largest bf16 come out as fp32 arithmetic
gives them.
"""

from __future__ import annotations

import pytest
import torch

from test_linear_transpose_f32_gpu import DEV, _check, _operands, _ops

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]


def _run(B, T, K, F, dtype, btf, seed=0):
    ops = _ops().nanochat_cuda
    x, w, go = _operands(B, T, K, F, dtype, seed)
    if btf:
        go = go.transpose(1, 2).contiguous().transpose(1, 2)
    bf = dtype == torch.bfloat16
    case = f"B={B} T={T} K={K} F={F} {dtype} btf={btf}"
    out = ops.fused_linear_transpose_cuda_op(x, w)
    gx, gw = torch.empty_like(x), torch.empty_like(w)
    ops.fused_linear_transpose_backward_kernel(x, w, go, gx, gw)
    _check(out, w.unsqueeze(0).expand(B, F, K), x.transpose(1, 2), K, "out " + case, bf)
    _check(gx, go.transpose(1, 2), w.unsqueeze(0).expand(B, F, K), F, "grad_x " + case, bf)
    _check(gw, go.permute(1, 0, 2).reshape(F, B * T), x.reshape(B * T, K), B * T + 32,
           "grad_weight " + case, bf)


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16"])
@pytest.mark.parametrize("btf", [False, True], ids=["bft", "btf"])
@pytest.mark.parametrize("K,F", [(8, 16), (15, 31), (16, 47), (33, 64), (71, 129), (128, 97)])
def test_small_tiles(dtype, btf, K, F):
    for T in (3, 7, 9, 16, 31, 33, 65, 127, 135):
        _run(2, T, K, F, dtype, btf, seed=T)


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16"])
@pytest.mark.parametrize("btf", [False, True], ids=["bft", "btf"])
@pytest.mark.parametrize("T,K,F", [(129, 100, 333), (257, 72, 1041), (1000, 129, 161)])
def test_large_tiles_and_splits(dtype, btf, T, K, F):
    _run(40, T, K, F, dtype, btf, seed=T)


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16"])
@pytest.mark.parametrize("btf", [False, True], ids=["bft", "btf"])
@pytest.mark.parametrize("B", [1, 13, 700])
def test_short_inner_reductions(B, btf, dtype):
    """grad_weight over many sequences whose lengths leave 1 to 31 indices past the
    whole k-steps: the packed steps, in one split and in several."""
    for T in (1, 2, 5, 15, 17, 31, 33):
        _run(B, T, 40, 50, dtype, btf, seed=T)


@pytest.mark.parametrize("fill", [float("nan"), float("inf"), 2.0 ** 110])
def test_f32_operands_past_the_split_range(fill):
    """A tensor with no element in the range that is split."""
    B, T, K, F = 3, 150, 64, 200
    x, w, go = _operands(B, T, K, F, torch.float32, 6)
    x = x.sign() * fill
    ops = _ops().nanochat_cuda
    out = ops.fused_linear_transpose_cuda_op(x, w)
    gx, gw = torch.empty_like(x), torch.empty_like(w)
    ops.fused_linear_transpose_backward_kernel(x, w, go, gx, gw)
    xd, gd = x.double(), go.double().permute(1, 0, 2).reshape(F, B * T)
    for got, want, mag in (
            (out, torch.matmul(w.double().unsqueeze(0), xd.transpose(1, 2).contiguous()),
             torch.matmul(w.double().abs().unsqueeze(0), xd.abs().transpose(1, 2).contiguous())),
            (gw, gd @ xd.reshape(B * T, K), gd.abs() @ xd.abs().reshape(B * T, K))):
        fin = torch.isfinite(want)
        assert bool(fin.all()) == (fill == 2.0 ** 110)
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(got.double()[torch.isinf(want)], want[torch.isinf(want)])
        err = (got.double() - want).abs()[fin]
        assert bool((err <= (B * T + 4) * 2.0 ** -24 * mag[fin]).all())


@pytest.mark.parametrize("T", [40, 1024])
def test_f32_non_finite(T):
    """Every element of the result that an infinity, a NaN or a value past the
    largest bf16 takes part in equals the fp32 arithmetic's class; the others
    stay within the bound."""
    B, K, F = 8, 96, 200
    x, w, _ = _operands(B, T, K, F, torch.float32, 5)
    big = 3.4e38  # rounds to infinity in bf16
    x[0, 3, 5], x[1, 0, 0], x[2, 7, 95], x[3, 1, 2] = float("inf"), float("nan"), -float("inf"), big
    w[17] = w[17].abs() * 2.0 ** -10  # positive: one sign per product with x[0, 3, 5]
    w[18] = 0.0                        # 0 * inf
    out = _ops().nanochat_cuda.fused_linear_transpose_cuda_op(x, w)
    want = torch.matmul(w.double().unsqueeze(0), x.double().transpose(1, 2))
    assert torch.equal(torch.isnan(out), torch.isnan(want))
    inf = torch.isinf(want)
    assert bool(inf.any()) and torch.equal(out.double()[inf], want[inf])
    fin = torch.isfinite(want)
    mag = torch.matmul(w.double().abs().unsqueeze(0), x.double().abs().transpose(1, 2))
    assert bool(((out.double() - want).abs()[fin] <= (K + 4) * 2.0 ** -24 * mag[fin]).all())
    assert float(out[3, 17, 1]) > 1e30


@pytest.mark.parametrize("dtype", DTYPES, ids=["f32", "bf16"])
@pytest.mark.parametrize("T,K,F", [(1024, 64, 98), (1024, 64, 97), (1024, 9, 33), (4096, 32, 257)])
def test_split_reduction_widths(dtype, T, K, F):
    """grad_weight's partials summed 4 elements per thread and (F K not a
    multiple of 4) one by one; one to many splits."""
    for B in (1, 3, 24):
        _run(B, T, K, F, dtype, False, seed=F)


def _scaled(t, e):
    """t 2^e in fp32, subnormals included."""
    return (t.double() * 2.0 ** e).float()


@pytest.mark.parametrize("other", [0, 60, 90])
@pytest.mark.parametrize("e", [-100, -109, -113, -118, -124, -130, -140])
def test_f32_small_operands(e, other):
    """Operands down to the smallest subnormals keep every bit, against ordinary
    and against large ones.  Bound: one fp32 rounding per term of the products
    (as for any magnitude) and one of 2^-150 per term where results are subnormal."""
    B, T, K, F = 2, 150, 40, 70
    x, w, go = _operands(B, T, K, F, torch.float32, 11)
    x, w = _scaled(x, e), _scaled(w, other)
    ops = _ops().nanochat_cuda
    # the small operand on either side: x w^T, and w x^T
    for a, b in ((x, w), (w.expand(2, F, K).contiguous(), x[0])):
        out = ops.fused_linear_transpose_cuda_op(a, b)
        want = torch.matmul(b.double().unsqueeze(0), a.double().transpose(1, 2).contiguous())
        mag = torch.matmul(b.double().abs().unsqueeze(0),
                           a.double().abs().transpose(1, 2).contiguous())
        err = (out.double() - want).abs()
        assert bool((err <= (K + 1) * (2.0 ** -24 * mag + 2.0 ** -150)).all()), float((err / mag).max())
    # gradients of the same
    gx, gw = torch.empty_like(x), torch.empty_like(w)
    go = _scaled(go, other)
    ops.fused_linear_transpose_backward_kernel(x, w, go, gx, gw)
    gd = go.double().permute(1, 0, 2).reshape(F, B * T)
    xd = x.double().reshape(B * T, K)
    err, mag = (gw.double() - gd @ xd).abs(), gd.abs() @ xd.abs()
    assert bool((err <= (B * T + 1) * (2.0 ** -24 * mag + 2.0 ** -150)).all()), float((err / mag).max())


@pytest.mark.parametrize("K", [1, 2, 3, 7, 16])
def test_f32_short_reductions(K):
    """Up to 16 indices: the fp32 arithmetic's bound, and for one index its value,
    the product rounded once -- of the outputs and, over B T = K tokens, of the
    weight's gradient."""
    F, T = 131, 70
    x, w, _ = _operands(1, T, K, F, torch.float32, 13)
    w[0] = 1 + 2.0 ** -8 + 2.0 ** -17  # (all of its low pieces at their largest)
    x[0, 0] = 1 + 2.0 ** -8 + 2.0 ** -17
    ops = _ops().nanochat_cuda
    out = ops.fused_linear_transpose_cuda_op(x, w)[0]
    # tokens as the reduction: x and grad_out with K of them
    x2, go = x[0].t().contiguous().unsqueeze(0), w.unsqueeze(0)
    gx, gw = torch.empty_like(x2), torch.empty(F, T, device=DEV)
    ops.fused_linear_transpose_backward_kernel(x2, torch.zeros(F, T, device=DEV), go, gx, gw)
    want, mag = w.double() @ x[0].double().t(), w.double().abs() @ x[0].double().abs().t()
    for got in (out, gw):
        assert bool(((got.double() - want).abs() <= K * 2.0 ** -24 * mag).all())
        if K == 1:
            assert torch.equal(got, w * x[0].t())


@pytest.mark.parametrize("B,T,K,F", [(3, 40, 17, 130), (3, 40, 96, 130), (8, 1024, 640, 258)])
def test_f32_errors_are_those_of_fp32_sums_or_less(B, T, K, F):
    """Worst case (K / 16 + 8) 2^-24 of the products' magnitudes.  In 2-norm no more
    than fp32 sums over pairs of products in order; where every product is the same
    and its dropped terms at their largest, no more than those, 2^-24, and one
    rounding of the result, 2^-24."""
    def check(got, a, b, what, const):
        # got = a @ b.T over the last axes
        n = a.shape[1]
        want, mag = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
        assert bool(((got.double() - want).abs() <= (n / 16 + 8) * 2.0 ** -24 * mag).all()), what
        err = float((got.double() - want).norm())
        if const:
            assert err <= 2 * 2.0 ** -24 * float(want.norm()), what
            return
        seq = torch.zeros_like(want, dtype=torch.float32)
        for k in range(0, n, 2):
            seq += a[:, k:k + 2] @ b[:, k:k + 2].t()
        assert err <= float((seq.double() - want).norm()), what

    ops = _ops().nanochat_cuda
    for const in (False, True):
        x, w, go = _operands(B, T, K, F, torch.float32, 14)
        if const:
            for t in (x, w, go):
                t.fill_(1 + 2.0 ** -8 + 2.0 ** -17)
        gx, gw = torch.empty_like(x), torch.empty_like(w)
        out = ops.fused_linear_transpose_cuda_op(x, w)
        ops.fused_linear_transpose_backward_kernel(x, w, go, gx, gw)
        xt, gt = x.reshape(B * T, K), go.transpose(1, 2).reshape(B * T, F)
        check(out.transpose(1, 2).reshape(B * T, F), xt, w, "out", const)
        check(gx.reshape(B * T, K), gt, w.t().contiguous(), "grad_x", const)
        check(gw, gt.t().contiguous(), xt.t().contiguous(), "grad_weight", const)


def test_f32_values_that_the_scale_overflows():
    """Finite operands and results past the scaled range come out as usual."""
    B, T, K, F = 2, 40, 24, 70
    x, w, _ = _operands(B, T, K, F, torch.float32, 12)
    for ex, ew in ((105, 0), (60, 40), (0, 81), (103, -90)):
        a, b = _scaled(x, ex), _scaled(w, ew)
        out = _ops().nanochat_cuda.fused_linear_transpose_cuda_op(a, b)
        want = torch.matmul(b.double().unsqueeze(0), a.double().transpose(1, 2).contiguous())
        mag = torch.matmul(b.double().abs().unsqueeze(0),
                           a.double().abs().transpose(1, 2).contiguous())
        assert bool(((out.double() - want).abs() <= (K + 1) * 2.0 ** -24 * mag).all())
