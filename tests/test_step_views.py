"""Views of a layer that csrc/step.cpp makes without the dispatcher: what torch's own are, and torch's own wherever somebody looks.  Runs on the CPU."""
import struct

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from trimkv_amd import _lib

B, H, CAP, D = 2, 3, 20, 64


class _Slab:
    def __init__(self, **how):
        self.k, self.v = torch.randn(B * H, CAP, D, dtype=torch.bfloat16), torch.randn(B * H, CAP, D, dtype=torch.bfloat16)
        self.lb, self.pos = torch.randn(B * H, CAP), torch.arange(B * H * CAP).view(B * H, CAP).clone()
        self.step = bytearray(struct.pack("12q", 0, 0, 0, 0, 0, 0, B * H, H, CAP, D, 1, 0)) + bytearray(19 * 8)
        self.__dict__.update(how)


def _own(slab, n):
    if n < 0:
        return [t.view(B * H * CAP, -1) for t in (slab.k, slab.v, slab.lb, slab.pos)]
    return [t.as_strided((B, H, n, D), (H * CAP * D, CAP * D, D, 1)) for t in (slab.k, slab.v)] + [t.as_strided((B, H, n), (H * CAP, CAP, 1)) for t in (slab.lb, slab.pos)]


def _same(got, want):
    for a, b in zip(got, want):
        assert type(a) is type(b) and a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype and a.data_ptr() == b.data_ptr()
        assert a._is_view() == b._is_view() and a._base is b._base and a.is_inference() == b.is_inference() and a.requires_grad == b.requires_grad and a.is_leaf == b.is_leaf
        if not a.is_inference():
            before = a._version
            b.add_(0)
            assert a._version == before + 1 == b._version


@pytest.mark.parametrize("n", [-1, 1, 7, CAP])
@pytest.mark.parametrize("mode", ["no_grad", "grad", "inference", "of inference"])
def test_views_are_those_of_torch(mode, n):
    with torch.inference_mode("inference" in mode and mode != "inference"):
        slab = _Slab()
    with {"no_grad": torch.no_grad, "grad": torch.enable_grad, "inference": torch.inference_mode, "of inference": torch.no_grad}[mode]():
        got, want = _lib.step().views(slab, n), _own(slab, n)
        _same(got, want)
    if mode == "no_grad":       # a view from where no gradients are recorded is not to be written where they are
        for t in (got[0], want[0]):
            with pytest.raises(RuntimeError):
                t.mul_(torch.ones(1, dtype=t.dtype, requires_grad=True))


def test_slabs_that_are_views_or_slices_and_rows_that_are_not_there():
    with torch.no_grad():
        big = torch.randn(2, B * H, CAP, D, dtype=torch.bfloat16)
        for k in (big[1], torch.nn.Parameter(big[0].clone(), requires_grad=True)):
            slab = _Slab(k=k)
            _same(_lib.step().views(slab, 5), _own(slab, 5))
        with pytest.raises(RuntimeError):
            _lib.step().views(_Slab(), B * H * CAP + 1)


def test_who_follows_operations_sees_the_views():
    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(str(func))
            return func(*args, **(kwargs or {}))

    names, slab = [], _Slab()
    with torch.no_grad(), Seen():
        _lib.step().views(slab, 5)
    assert names == ["aten.as_strided.default"] * 4
    with torch.no_grad(), torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        _lib.step().views(slab, 5)
    assert sum(e.count for e in prof.key_averages() if e.key == "aten::as_strided") == 4
