"""CPU: a weight that calls have prepared launch arguments for can still be copied and pickled, and
the copy prepares its own (addresses of its own state, not of the original's)."""

import copy
import pickle
from types import SimpleNamespace

import pytest
import torch

from testt_amd import layer_native, nf4, nf4_gemm
from testt_amd import workloads as wl

CPU = torch.device("cpu")
SHAPES = {"q": (256, 256), "k": (128, 256), "v": (128, 256), "o": (256, 256), "gate": (256, 256),
          "up": (256, 256), "down": (256, 256)}


def prepare(w, cus):
    """Every kind of argument that the operators keep on a weight."""
    q, k, v = w.q, w.k, w.v
    nf4_gemm._stack((q, k, v), CPU)
    groups = ((q, k, v), (w.o,), (w.gate, w.up), (w.down,))
    nf4._group_plan(groups, CPU, *nf4._group_layout(groups))
    return layer_native._nf4_layer(w, 16, CPU)


@pytest.mark.parametrize("again", [copy.deepcopy, lambda w: pickle.loads(pickle.dumps(w))])
def test_copies_and_pickles(monkeypatch, again):
    monkeypatch.setitem(nf4_gemm._cu_count.cache, CPU, 256)
    w = SimpleNamespace(**{n: wl.nf4_weight(*s, 3) for n, s in SHAPES.items()})
    struct = bytes(prepare(w, 256)[0])
    twin = again(w)
    for name in SHAPES:
        assert not any(getattr(getattr(twin, name), a) for a in vars(getattr(twin, name))
                       if a.startswith("_soupk_"))
    assert torch.equal(twin.q.data, w.q.data)
    assert nf4._plan(twin.q, CPU)[0] != nf4._plan(w.q, CPU)[0]
    assert nf4_gemm._stack((twin.q, twin.k, twin.v), CPU) is not \
        nf4_gemm._stack((w.q, w.k, w.v), CPU)
    assert bytes(prepare(twin, 256)[0]) != struct
    assert nf4._plan(twin.q, CPU)[0][0] == twin.q.data.data_ptr()
