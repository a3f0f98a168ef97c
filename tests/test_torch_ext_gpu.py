"""The native host path of the bf16 filter (``_ltv_torch.so``) against the Python
autograd function and decode call over the same library entries: bitwise equal
results for every kind of scan behind it, and the inputs it must leave to Python.
"""

from __future__ import annotations

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _hm():
    from nanochat_amd.ops import ltv_hm_fast as hm
    return hm


def _case(B, T, shared, inits_dtype, weight_dtype=torch.float32, seed=0):
    NH, NKVH, D, r = 2, 1, 64, 16
    H, Da, C = NH + 2 * NKVH, D // r, NH * D
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(B, T, C, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(H * (D + Da), C, generator=g) / C ** 0.5).to(weight_dtype).to(DEV)
    i = torch.randn(H, D, generator=g) if shared else torch.randn(B, H, D, generator=g)
    b = (torch.rand(H, Da, generator=g) - 0.5).to(DEV)
    gs = [torch.randn(B, T, n, D, generator=g).to(torch.bfloat16).to(DEV).transpose(1, 2)
          for n in (NH, NKVH, NKVH)]
    return (x, w, i.to(inits_dtype).to(DEV), b), gs, (NH, NKVH, Da, r)


def _step(fn, tensors, gs, dims, pqk=(2 ** 31 - 1, 1, 1), skip=()):
    ts = [t.detach().clone().requires_grad_(True) for t in tensors]
    out = fn(*ts, *dims, *pqk)[:3]
    pairs = [(o, g) for n, (o, g) in enumerate(zip(out, gs)) if n not in skip]
    torch.autograd.backward([o for o, _ in pairs], [g for _, g in pairs])
    return [o.detach() for o in out] + [t.grad for t in ts]


def _same(a, b, label):
    for n, (x, y) in enumerate(zip(a, b)):
        assert x.dtype == y.dtype and torch.equal(x, y), f"{label}: output {n}"


@pytest.mark.parametrize("B,T,pqk", [
    (2, 1, (2 ** 31 - 1, 1, 1)), (3, 150, (2 ** 31 - 1, 1, 1)), (70, 33, (2 ** 31 - 1, 1, 1)),
    (1, 5000, (2 ** 31 - 1, 1, 1)),                    # chained forward
    (2, 300, (16, 16, 9)), (2, 300, (64, 60, 37)),     # short and general windows
])
def test_equals_python_function(B, T, pqk):
    hm = _hm()
    full = pqk[0] > T
    for shared, idt in ((True, torch.float32), (False, torch.bfloat16)):
        if shared and not full and pqk != (16, 16, 9):
            continue  # general windows take per-sequence bf16 inits
        tensors, gs, dims = _case(B, T, shared, idt, seed=T)
        native = hm.N.torch_ext().qkv_filter(*tensors, *dims, *pqk)
        assert native is not None, "the plain case goes through the native function"
        _same(_step(hm.qkv_filter_call, tensors, gs, dims, pqk),
              _step(hm._QkvFilterEager.apply, tensors, gs, dims, pqk), f"B={B} T={T} {pqk}")
        # an output that takes no part in the loss; a bf16 weight
        tensors, gs, dims = _case(B, T, shared, idt, torch.bfloat16, seed=T + 1)
        _same(_step(hm.qkv_filter_call, tensors, gs, dims, pqk, skip=(1,)),
              _step(hm._QkvFilterEager.apply, tensors, gs, dims, pqk, skip=(1,)), "k unused")


def test_saved_tensor_hooks_streams_and_threads():
    hm = _hm()
    tensors, gs, dims = _case(2, 257, True, torch.float32)
    want = _step(hm._QkvFilterEager.apply, tensors, gs, dims)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(0) or t.cpu(),
                                                  lambda t: t.to(DEV)):
        _same(_step(hm.qkv_filter_call, tensors, gs, dims), want, "saved-tensor hooks")
    assert len(packed) == 9
    torch.cuda.synchronize()
    results = {}

    def work(n):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(5):
                results[n] = _step(hm.qkv_filter_call, tensors, gs, dims)
        s.synchronize()

    threads = [threading.Thread(target=work, args=(n,)) for n in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for n in range(3):
        _same(results[n], want, f"thread {n}")


def test_saved_tensors_in_another_layout():
    """Hooks may hand tensors back with the same values and other strides: x is
    made contiguous and the scan reads any strides, as from Python."""
    hm = _hm()
    tensors, gs, dims = _case(3, 70, False, torch.bfloat16)

    def other_layout(t):
        return t.transpose(0, -1).contiguous().transpose(0, -1) if t.dim() > 2 else t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, other_layout):
        want = _step(hm._QkvFilterEager.apply, tensors, gs, dims)
        _same(_step(hm.qkv_filter_call, tensors, gs, dims), want, "restrided")
    for a, b in zip(want, _step(hm._QkvFilterEager.apply, tensors, gs, dims)):
        assert float((a.double() - b.double()).norm()) <= 2.0 ** -7 * float(b.double().norm())


def test_inputs_left_to_python():
    """Refused by the native entry, so that Python's own checks and paths apply."""
    hm = _hm()
    ext = hm.N.torch_ext()
    (x, w, i, b), _, dims = _case(2, 40, False, torch.bfloat16)
    full = (2 ** 31 - 1, 1, 1)
    for bad in ((x.float(), w, i, b), (x.transpose(0, 1), w, i, b), (x, w[:-1], i, b),
                (x, w.t().contiguous().t(), i, b), (x, w, i[:1], b), (x, w, i, b.bfloat16()),
                (x.cpu(), w, i, b), (x[:0], w, i, b), (x, w.double(), i, b)):
        assert ext.qkv_filter(*bad, *dims, *full) is None
    with pytest.raises(RuntimeError, match="weight must be"):
        hm.qkv_filter_call(x, w[:-1], i, b, *dims)
    with pytest.raises(RuntimeError, match="GPU tensors"):
        hm.qkv_filter_call(x.cpu(), w.cpu(), i.cpu(), b.cpu(), *dims)
    with pytest.raises(RuntimeError, match="LTV_ERR_UNSUPPORTED"):  # fp32 inits, general windows
        hm.qkv_filter_call(x, w, i.float(), b, *dims, 16, 80, 40)


@pytest.mark.parametrize("B", [1, 33])
def test_decode_rows_equals_decode_step(B):
    hm = _hm()
    (x, w, _, b), _, (NH, NKVH, Da, r) = _case(B, 1, True, torch.float32, seed=B)
    g = torch.Generator().manual_seed(B)
    rows = [torch.randn(B, n, Da * r, generator=g).to(torch.bfloat16).to(DEV)
            for n in (NH, NKVH, NKVH)]
    wpack = hm.pack_weight(w, NH + 2 * NKVH, Da * r, Da)
    mine, theirs = [t.clone() for t in rows], [t.clone() for t in rows]
    ext = hm.N.torch_ext()
    out = ext.decode_rows(x, wpack, *mine, b, NH, NKVH, Da, r)
    want = hm.decode_step(x, wpack, theirs, b, NH, NKVH, Da, r, rows=theirs)
    _same([torch.cat(out, 2)[:, 0], *mine], [want, *theirs], f"B={B}")
    assert all(o.shape == (B, 1, n, Da * r) for o, n in zip(out, (NH, NKVH, NKVH)))
    f32 = [t.float() for t in rows]
    assert ext.decode_rows(x, wpack, *f32, b, NH, NKVH, Da, r) is None
    assert ext.decode_rows(x.expand(B, 2, -1), wpack, *mine, b, NH, NKVH, Da, r) is None
