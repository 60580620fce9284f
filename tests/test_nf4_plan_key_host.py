"""CPU: the key under which an NF4 weight's kernel arguments are kept (nf4._plan_key) covers all that
they are made from and checked on, so that no change of a weight's state is run on old arguments.
The arguments are built for CPU tensors here; nothing is launched."""

import copy
import ctypes

import pytest
import torch

from testt_amd import nf4, nf4_gemm
from testt_amd import workloads as wl

CPU = torch.device("cpu")


def weight(seed=1):
    return wl.nf4_weight(128, 256, seed)


def offset_of(plan):
    """The offset that the kernel would read."""
    return ctypes.c_float.from_address(plan[0][4]).value


CHANGES = {
    "quant_type": lambda w: setattr(w.quant_state, "quant_type", "fp4"),
    "nested": lambda w: setattr(w.quant_state, "nested", False),
    "blocksize": lambda w: setattr(w.quant_state, "blocksize", 32),
    "outer blocksize": lambda w: setattr(w.quant_state.state2, "blocksize", 128),
    "shape": lambda w: setattr(w.quant_state, "shape", (256, 128)),
    "data dtype": lambda w: setattr(w, "data", w.data.view(torch.int8)),
    "data size": lambda w: setattr(w, "data", w.data[:-64]),
    "absmax": lambda w: setattr(w.quant_state, "absmax", w.quant_state.absmax.clone()),
    "absmax size": lambda w: setattr(w.quant_state, "absmax", w.quant_state.absmax[:-1]),
    "absmax type": lambda w: setattr(w.quant_state, "absmax",
                                     w.quant_state.absmax.view(torch.int8)),
    "code": lambda w: setattr(w.quant_state, "code", w.quant_state.code.clone()),
    "code2 size": lambda w: setattr(w.quant_state.state2, "code", w.quant_state.state2.code[:8]),
    "offset": lambda w: setattr(w.quant_state, "offset", w.quant_state.offset + 1),
    "offset, a number": lambda w: setattr(w.quant_state, "offset", 0.25),
}


@pytest.mark.parametrize("change", CHANGES)
def test_a_changed_state_is_planned_again(change):
    w = weight()
    plan, stack = nf4._plan(w, CPU), nf4_gemm._stack((w,), CPU)
    assert nf4._plan(w, CPU) is plan and nf4_gemm._stack((w,), CPU) is stack is not None
    key = nf4._plan_key(w, CPU)
    CHANGES[change](w)
    assert nf4._plan_key(w, CPU) != key
    try:
        assert nf4._plan(w, CPU) is not plan
        assert nf4_gemm._stack((w,), CPU) is not stack
    except (TypeError, ValueError):     # refused, as the same state of a new weight is
        with pytest.raises((TypeError, ValueError)):
            nf4._plan(copy.deepcopy(wl.Params4bit(data=w.data, quant_state=w.quant_state)), CPU)


@pytest.mark.parametrize("make", [float, lambda v: torch.tensor(v), lambda v: torch.tensor([v]),
                                  lambda v: torch.tensor(v, dtype=torch.float16)])
def test_offset_replaced_in_place_of_a_freed_one(make):
    """Offsets that take turns at one object's or one tensor's memory."""
    w = weight()
    for i in range(64):
        w.quant_state.offset = None
        w.quant_state.offset = make(0.5 + i)
        assert offset_of(nf4._plan(w, CPU)) == 0.5 + i


def test_unsupported_state_is_checked_again():
    w = weight()
    w.quant_state.quant_type = "fp4"
    assert nf4_gemm._stack((w,), CPU) is None
    w.quant_state.quant_type = "nf4"
    assert nf4_gemm._stack((w,), CPU) is not None


def test_keys_of_several_weights():
    ws = [weight(i) for i in range(3)]
    both = nf4._plan_keys(ws, CPU)
    assert both[1] == b"".join(nf4._plan_key(w, CPU)[1] for w in ws)
    ws[1].quant_state.state2.blocksize = 128
    assert nf4._plan_keys(ws, CPU) != both
    assert nf4._plan_keys([*ws, object()], CPU) is None and nf4._plan_keys([], CPU) is None
