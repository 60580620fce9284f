"""CPU: what a call prepares for weights that it has not seen.  The launch arguments of an unpack and
of the fused products, from real NF4 states on the CPU (launches recorded, not made); a product
reads each weight's state three times at most, for its choice, its plan and its launch, and an unpack
of one product's stack leaves the plan of the layer's projections where it is."""

import ctypes

import pytest
import torch

from testt_amd import _ext, nf4, nf4_gemm
from testt_amd import workloads as wl

CPU = torch.device("cpu")


class Rows:
    """Stands in for an fp16 device tensor [rows, cols]."""

    is_cuda, dtype, device = True, torch.float16, CPU

    def __init__(self, *shape):
        self.shape = shape

    def dim(self):
        return 2

    def stride(self, d):
        return (self.shape[1], 1)[d]

    def data_ptr(self):
        return 4096


@pytest.fixture
def launches(monkeypatch):
    made, keys, empty = [], [], torch.empty
    plan_key, plan_keys = nf4._plan_key, nf4._plan_keys
    monkeypatch.setattr(torch, "empty", lambda *a, device=None, **k: empty(*a, **k))
    monkeypatch.setattr(_ext, "call", lambda name, *a: made.append((name, a)))
    monkeypatch.setattr(_ext, "stream_of", lambda t: 0)
    monkeypatch.setattr(nf4, "kernels_ok", lambda t: True)
    monkeypatch.setattr(nf4, "_hip_device", lambda d: CPU)
    monkeypatch.setattr(nf4, "_plan_key", lambda *a: (keys.append(a), plan_key(*a))[1])
    monkeypatch.setattr(nf4, "_plan_keys", lambda ws, d: (keys.extend(ws), plan_keys(ws, d))[1])
    monkeypatch.setattr(nf4_gemm, "fused_fits", lambda *a, **k: True)
    monkeypatch.setitem(nf4_gemm._cu_count.cache, CPU, 256)
    return made, keys


def weights(*rows):
    return tuple(wl.nf4_weight(n, 256, 7 + i) for i, n in enumerate(rows))


def pointers(address, n):
    return list((ctypes.c_void_p * n).from_address(address))


def test_a_product_reads_each_state_three_times_at_most(launches):
    made, keys = launches
    ws = weights(256, 128, 128)
    nf4.fused_linear(Rows(16, 256), ws, None)
    assert len(keys) <= 3 * len(ws)
    nf4.fused_grad_input(Rows(16, 512), ws)
    assert len(keys) <= 5 * len(ws) and len(made) == 2
    for name, a in made:
        assert a[2] == 3                       # parts
        assert pointers(a[3], 3) == [w.data.data_ptr() for w in ws]
        assert pointers(a[4], 3) == [w.quant_state.absmax.data_ptr() for w in ws]
        assert list((ctypes.c_int32 * 3).from_address(a[9])) == [256, 128, 128]
        assert a[10:12] == (64, 256)


@pytest.mark.parametrize("rows", [(128,), (256, 128, 128), (64,) * 8, (64,) * 9, (7, 3)])
def test_unpack_concat(launches, monkeypatch, rows):
    made, keys = launches
    read = []

    def call(name, *a):                        # (the tables live until the call returns)
        n = a[0]
        read.append((name, pointers(a[1], n), pointers(a[7], n),
                     list((ctypes.c_int64 * n).from_address(a[8])), a[9:11]))

    monkeypatch.setattr(_ext, "call", call)
    monkeypatch.setattr(_ext, "require", lambda t, *a, **k: t)
    ws = weights(*rows)
    out = nf4.unpack_concat(ws, "cuda")
    assert tuple(out.shape) == (sum(rows), 256) and out.dtype is torch.float16
    assert all(name == "soupk_nf4_unpack_multi" and blocks == (64, 256)
               for name, _, _, _, blocks in read)
    assert [p for r in read for p in r[1]] == [w.data.data_ptr() for w in ws]
    before = [sum(rows[:i]) for i in range(len(rows))]
    assert [p for r in read for p in r[2]] == [out.data_ptr() + 512 * b for b in before]
    assert [p for r in read for p in r[3]] == [128 * n for n in rows]


def test_unpack_concat_leaves_the_layers_plan(launches):
    ws = weights(256, 128, 128, 256)
    groups = (ws[:3], ws[3:])

    def layers_plan():
        return nf4._group_plan(groups, CPU, *nf4._group_layout(groups))

    plan = layers_plan()
    nf4.unpack_concat(ws[:3], "cuda")
    assert layers_plan() is plan
