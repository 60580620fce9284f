"""GPU: the operators whose common case the host extension takes in one native call (host_ops.cpp)
against the Python form below it, which takes everything else: the same bits for the same
arguments, and the same refusals."""

import math

import pytest
import torch

from testt_amd import _ext, attention, blas, mlp, rmsnorm, rope, workloads

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
NH, NKV, D = 4, 2, 128
SCALE = 1.0 / math.sqrt(D)
LENGTHS, T = (70, 33, 1), 70
OPERATORS = ("rmsnorm_fwd", "rmsnorm_bwd", "rope_tokens", "rope_fwd", "rope_bwd", "varlen_fwd",
             "varlen_bwd", "attn_fwd", "attn_bwd", "swiglu_fwd", "gemm")


class Host:
    """The extension with its operators counted, or answering None (`python`)."""

    def __init__(self, python):
        self.real, self.python, self.taken = _ext.host(), python, set()

    def __getattr__(self, name):
        fn = getattr(self.real, name)
        if name not in OPERATORS:
            return fn

        def call(*args):
            out = None if self.python else fn(*args)
            if out is not None:
                self.taken.add(name)
            return out
        return call


def rand(*shape, dtype=torch.float16, seed=0, std=1.0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (std * torch.randn(*shape, generator=g)).to(dtype).to(DEV)


def positions():
    return workloads.ragged_positions(LENGTHS, T).to(DEV)


def tables():
    return workloads.rope_tables(T, D, workloads.ROPE_THETA, device=DEV)


def norm(rows, padded, with_delta=True, with_pad=True):
    x = rand(rows, 256, dtype=torch.float32).requires_grad_(True)
    delta = rand(rows, 256, seed=1).requires_grad_(True) if with_delta else None
    w = rand(256, dtype=torch.float32, seed=2)
    pad = torch.randperm(padded, generator=torch.Generator().manual_seed(3))[:rows].to(DEV) \
        if with_pad else None
    s, y, yp = rmsnorm.add_rmsnorm(x, delta, w, 1e-6, pad, padded if with_pad else 0)
    outs = [y] + ([yp] if with_pad else []) + ([s] if with_delta else [])
    grads = torch.autograd.grad(outs, [x] + ([delta] if with_delta else []),
                                [rand(*o.shape, dtype=o.dtype, seed=5) for o in outs])
    return [s, y, yp, *grads]


def packed(dtype, with_q=True, with_v=True):
    pos, m = positions(), sum(LENGTHS)
    qkv = rand(m, (NH + 2 * NKV) * D).requires_grad_(True)
    lq = rand(m, NH * D, dtype=dtype, seed=1).requires_grad_(True) if with_q else None
    lv = rand(m, NKV * D, dtype=dtype, seed=2).requires_grad_(True) if with_v else None
    leaves = [t for t in (qkv, lq, lv) if t is not None]
    out = rope.rope_pack(qkv, lq, lv, *tables(), pos, len(LENGTHS), T, NH, NKV, D)
    grads = torch.autograd.grad(out, leaves, [rand(*o.shape, seed=7) for o in out])
    cu = attention.cu_seqlens_of(pos, len(LENGTHS), T)
    o = attention.rope_attention(qkv, lq, lv, *tables(), pos, cu, len(LENGTHS), T, NH, NKV)
    return [*out, *grads, o, *torch.autograd.grad([o], leaves, [rand(*o.shape, seed=8)])]


def padded_attention(flags):
    B = len(LENGTHS)
    q, k, v = (rand(B, h, T, D, seed=h + i).requires_grad_(True)
               for i, h in enumerate((NH, NKV, NKV)))
    valid = (torch.arange(T, device=DEV)[None] <
             torch.tensor(LENGTHS, device=DEV)[:, None]).to(torch.uint8) if flags else None
    out = attention.causal_attention(q, k, v, valid, SCALE)
    return [out, *torch.autograd.grad([out], [q, k, v], [rand(*out.shape, seed=9)])]


def varlen(with_rope):
    pos, m = positions(), sum(LENGTHS)
    rows = rand(m, (NH + 2 * NKV) * D, seed=4)
    cu = attention.cu_seqlens_of(pos, len(LENGTHS), T)
    out, lse = attention.attention_varlen_fwd(rows, cu, NH, NKV, SCALE)
    return [out, lse, attention.attention_varlen_bwd(
        rows, cu, out, lse, rand(*out.shape, seed=3), SCALE, NH, NKV,
        rope=(*tables(), pos, len(LENGTHS), T) if with_rope else None)]


def gemm(transposed, bias=False, into=False, strided=False):
    a = rand(48, 192)[:, :128] if strided else rand(48, 128)
    w = rand(64, 128, seed=1).t() if transposed else rand(128, 64, seed=1)
    out = rand(48, 64, seed=2) if into else None
    got = blas.matmul(a, w, rand(64, seed=3) if bias else None, out, into)
    assert out is None or got is out
    return [got]


# name: (call, the operators that it takes natively)
CALLS = {
    "norm": (lambda: norm(96, 96), {"rmsnorm_fwd", "rmsnorm_bwd"}),
    "norm, padded rows": (lambda: norm(70, 128), {"rmsnorm_fwd", "rmsnorm_bwd"}),
    "norm, no delta": (lambda: norm(33, 64, with_delta=False), {"rmsnorm_fwd", "rmsnorm_bwd"}),
    "norm alone": (lambda: norm(7, 0, with_pad=False), {"rmsnorm_fwd", "rmsnorm_bwd"}),
    "rope fp16": (lambda: packed(torch.float16), {"rope_fwd", "rope_bwd", "rope_tokens"}),
    "rope fp32": (lambda: packed(torch.float32), {"rope_fwd", "rope_bwd", "rope_tokens"}),
    "rope, q alone": (lambda: packed(torch.float16, with_v=False), {"rope_fwd", "rope_tokens"}),
    "rope, no deltas": (lambda: packed(None, False, False), {"rope_fwd", "rope_tokens"}),
    "padded attention": (lambda: padded_attention(False), {"attn_fwd", "attn_bwd"}),
    "padded attention, flags": (lambda: padded_attention(True), {"attn_fwd", "attn_bwd"}),
    "varlen": (lambda: varlen(False), {"varlen_fwd", "varlen_bwd"}),
    "varlen, rope": (lambda: varlen(True), {"varlen_fwd", "varlen_bwd"}),
    "swiglu": (lambda: [mlp.gated_silu(rand(37, 512))], {"swiglu_fwd"}),
    "gemm nn": (lambda: gemm(False), {"gemm"}),
    "gemm tn, bias": (lambda: gemm(True, bias=True), {"gemm"}),
    "gemm nn, accumulate": (lambda: gemm(False, into=True), {"gemm"}),
    "gemm, strided rows": (lambda: gemm(True, strided=True), {"gemm"}),
}


def run(monkeypatch, call, python):
    host = Host(python)
    monkeypatch.setattr(_ext, "host", lambda: host)
    try:
        return host, [t.detach() for t in call()]
    finally:
        monkeypatch.undo()


@pytest.mark.parametrize("name", CALLS)
def test_native_and_python_forms_agree(monkeypatch, name):
    call, operators = CALLS[name]
    print(name, flush=True)
    host, native = run(monkeypatch, call, False)
    assert operators <= host.taken, host.taken
    host, plain = run(monkeypatch, call, True)
    assert not host.taken and len(native) == len(plain)
    for i, (a, b) in enumerate(zip(native, plain)):
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride(), i
        bits = torch.int16 if a.dtype == torch.float16 else torch.int32
        assert torch.equal(a.contiguous().view(bits), b.contiguous().view(bits)), (name, i)


def _pos(**change):
    args = dict(qkv=rand(104, (NH + 2 * NKV) * D), lq=None, lv=None, cos=tables()[0],
                sin=tables()[1], pos=positions(), batch=3, seq=T, nh=NH, nkv=NKV, hd=D)
    args.update(change)
    return rope.rope_pack(*args.values())


# Arguments outside the operators' ranges, refused on the host by both forms.
REFUSED = {
    "norm, fp64 rows": lambda: rmsnorm.add_rmsnorm(rand(4, 64).double(), None,
                                                   rand(64, dtype=torch.float32), 1e-6),
    "norm, weight of another size": lambda: rmsnorm.add_rmsnorm(
        rand(4, 64, dtype=torch.float32), None, rand(32, dtype=torch.float32), 1e-6),
    "norm, delta of another shape": lambda: rmsnorm.add_rmsnorm(
        rand(4, 64, dtype=torch.float32), rand(3, 64), rand(64, dtype=torch.float32), 1e-6),
    "norm, another pad count": lambda: rmsnorm.add_rmsnorm(
        rand(4, 64, dtype=torch.float32), None, rand(64, dtype=torch.float32), 1e-6,
        torch.arange(3, device=DEV), 8),
    "rope, fp32 rows": lambda: _pos(qkv=rand(104, (NH + 2 * NKV) * D, dtype=torch.float32)),
    "rope, width": lambda: _pos(qkv=rand(104, D)),
    "rope, positions": lambda: _pos(pos=positions()[:5]),
    "rope, short tables": lambda: _pos(cos=tables()[0][:9]),
    "rope, delta shape": lambda: _pos(lq=rand(104, D)),
    "rope, odd head dim": lambda: _pos(hd=127),
    "attention, k of another length": lambda: attention.attention_fwd(
        rand(2, NH, 64, D), rand(2, NKV, 32, D), rand(2, NKV, 64, D)),
    "attention, flags of another type": lambda: attention.attention_fwd(
        rand(2, NH, 64, D), rand(2, NKV, 64, D), rand(2, NKV, 64, D),
        torch.ones(2, 64, device=DEV)),
    "attention, head dim 64": lambda: attention.attention_fwd(
        rand(2, NH, 64, 64), rand(2, NKV, 64, 64), rand(2, NKV, 64, 64)),
    "attention, heads": lambda: attention.attention_fwd(
        rand(2, 3, 64, D), rand(2, 2, 64, D), rand(2, 2, 64, D)),
    "attention, scale": lambda: attention.attention_fwd(
        rand(2, NH, 64, D), rand(2, NKV, 64, D), rand(2, NKV, 64, D), None, -1.0),
    "varlen, width": lambda: attention.attention_varlen_fwd(
        rand(8, D), torch.tensor([0, 8], dtype=torch.int32, device=DEV), NH, NKV, SCALE),
    "varlen, int64 bounds": lambda: attention.attention_varlen_fwd(
        rand(8, (NH + 2 * NKV) * D), torch.tensor([0, 8], device=DEV), NH, NKV, SCALE),
    "swiglu, odd width": lambda: mlp.gated_silu(rand(4, 63)),
    "swiglu, fp32": lambda: mlp.gated_silu(rand(4, 64, dtype=torch.float32)),
    "gemm, sizes": lambda: blas.matmul(rand(4, 64), rand(32, 8)),
    "gemm, accumulate without out": lambda: blas.matmul(rand(8, 64), rand(64, 8), None, None, True),
}


@pytest.mark.parametrize("name", REFUSED)
def test_both_forms_refuse(monkeypatch, name):
    print(name, flush=True)
    raised = []
    for python in (False, True):
        with pytest.raises((ValueError, TypeError, RuntimeError)) as e:
            run(monkeypatch, lambda: list(REFUSED[name]()), python)
        raised.append((e.type, str(e.value)))
    assert raised[0] == raised[1]


def test_uncommon_arguments_take_the_python_form(monkeypatch):
    """Non-contiguous gradients, int32 positions, weights in fp16: converted as before."""
    def call():
        x = rand(40, 256, dtype=torch.float32).requires_grad_(True)
        w = rand(256, seed=2)                                     # fp16
        pad = torch.arange(40, dtype=torch.int32, device=DEV)
        s, y, yp = rmsnorm.add_rmsnorm(x, rand(40, 256, seed=1), w, 1e-6, pad, 64)
        g = torch.autograd.grad([s, y, yp], [x], [rand(256, 40, dtype=torch.float32).t(),
                                                  rand(256, 40).t(),
                                                  rand(1, 256, dtype=torch.float32).expand(64, 256)])
        return [s, y, yp, *g, mlp.gated_silu(rand(9, 128)),
                blas.matmul(rand(5, 24)[:, :20], rand(20, 12, seed=1))]

    (_, a), (_, b) = run(monkeypatch, call, False), run(monkeypatch, call, True)
    assert all(torch.equal(x, y) for x, y in zip(a, b))
