"""The native host side of decode steps (csrc/step.cpp): what it takes and what it leaves to the general way."""
import numpy as np
import pytest
import torch

from trimkv_amd import BatchedDynamicBudgetTrimKVCache, TrimKVCache, _lib, get_attention_interface

DEV = "cuda:0"
B, H, G, D, N = 2, 2, 2, 128, 700


class _Mod:
    training, num_key_value_groups, is_causal = False, G, True


def _rows(S, at, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    k, v = (torch.randn(B, H, S, D, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))
    return k, v, -torch.rand(B, H, S, generator=gen, device=DEV), torch.arange(at, at + S, device=DEV)


def _strided(t):
    """The same values with other strides over batch and head."""
    return torch.stack([t, t], dim=2).flatten(1, 2)[:, ::2]


class _Sub(torch.Tensor):
    pass


# how the new row arrives -> whether native code remembers it, whether it is deferred at all
ROWS = {"plain": (lambda k, v, lb, p: (k, v, lb, p), True, True),
        "strided": (lambda k, v, lb, p: (_strided(k), _strided(v), _strided(lb), p), True, True),
        "positions per head": (lambda k, v, lb, p: (k, v, lb, p.expand(B, H, 1)), True, True),
        "subclass": (lambda k, v, lb, p: (k.as_subclass(_Sub), v, lb, p), False, True),
        "strides differ": (lambda k, v, lb, p: (k, _strided(v), lb, p), False, False),
        "positions of 32 bits": (lambda k, v, lb, p: (k, v, lb, p.int()), False, False),
        "log beta of 16 bits": (lambda k, v, lb, p: (k, v, lb.to(torch.bfloat16), p), False, False)}


@pytest.mark.gpu
@pytest.mark.parametrize("how", list(ROWS))
@pytest.mark.parametrize("kind", [TrimKVCache, BatchedDynamicBudgetTrimKVCache])
def test_rows_that_native_code_remembers_and_rows_that_it_leaves(kind, how):
    change, native, deferred = ROWS[how]
    plain, fused = kind(), kind()
    fused.fuse_decode_append = True
    attend = get_attention_interface("trimkv_hip" if kind is TrimKVCache else "db_attn_flash_batched")
    for c in (plain, fused):
        c.update(*_rows(N, 0, 1), 0)
    slab = fused._slabs[0]
    q = torch.randn(B, H * G, 1, D, generator=torch.Generator(device=DEV).manual_seed(5), device=DEV).to(torch.bfloat16)
    row = change(*_rows(1, N, 2))
    assert (_lib.step().defer(slab, *row) is True) == native
    if native:
        assert slab.max_len == N + 1 and slab.total == B * H * (N + 1) and (slab.lens == N + 1).all()
        assert _lib.step().defer(slab, *row) is None       # a row is waiting
        slab.pending, slab.max_len, slab.total = None, N, B * H * N
        slab.lens -= 1
    assert slab.pending is None and slab.max_len == N and (slab.lens == N).all()
    got, want = fused.update(*row, 0), plain.update(*change(*_rows(1, N, 2)), 0)
    assert (slab.pending is not None) == deferred and slab.max_len == N + 1 and slab.total == B * H * (N + 1)
    outs = [attend(_Mod(), q, r[0], r[1], None, flash_attn_kwargs=r[-1])[0] for r in (got, want)]
    assert slab.pending is None and outs[0].shape == (B, 1, H * G, D) and torch.equal(*outs)
    for name in ("k", "v", "lb", "pos"):
        assert torch.equal(getattr(slab, name)[:, :N + 1], getattr(plain._slabs[0], name)[:, :N + 1])


@pytest.mark.gpu
def test_a_full_slab_grows_the_general_way():
    c = TrimKVCache()
    c.fuse_decode_append = True
    c.update(*_rows(N, 0, 1), 0)
    slab = c._slabs[0]
    slab.regrow(N)
    assert _lib.step().defer(slab, *_rows(1, N, 2)) is None and slab.max_len == N
    c.update(*_rows(1, N, 2), 0)
    assert slab.cap > N and slab.pending is not None and len(slab.step) == 31 * 8


@pytest.mark.gpu
def test_which_calls_are_the_usual_decode_step():
    c = TrimKVCache()
    c.fuse_decode_append = True
    c.update(*_rows(N, 0, 1), 0)
    k, v, _, _, kw = c.update(*_rows(1, N, 2), 0)
    slab, fits = c._slabs[0], _lib.step().fits
    q = torch.zeros(B, H * G, 1, D, dtype=torch.bfloat16, device=DEV)
    assert fits(q, k, slab) == G
    assert fits(q[:, :3], k, slab) == 0 and fits(q[:1], k, slab) == 0 and fits(q.expand(B, H * G, 2, D), k, slab) == 0 and fits(q[..., :64], k, slab) == 0
    assert fits(q.half(), k, slab) == 0 and fits(q.cpu(), k, slab) == 0 and fits(q, k.clone(), slab) == 0 and fits(q, k[:, :, :-1], slab) == 0 and fits(q[:, :0], k, slab) == 0
    assert fits(q.as_subclass(_Sub), k, slab) == 0 and fits(None, k, slab) == 0 and fits(q[0], k, slab) == 0
    c._flush_all()
    assert fits(q, k, slab) == 0
    r = BatchedDynamicBudgetTrimKVCache()
    r.fuse_decode_append = True
    r.update(*_rows(N, 0, 1), 0)
    k, v, _, _, kw = r.update(*_rows(1, N, 2), 0)
    assert fits(q, k, r._slabs[0]) == 0


def test_calls_that_make_no_sense_are_errors():
    step = _lib.step()
    for call in (lambda: step.defer(1, 2), lambda: step.views(1), lambda: step.fits(1), lambda: step.attend(1), lambda: step.attend(*range(11)), lambda: step.views(object(), "n")):
        with pytest.raises(TypeError):
            call()
    with pytest.raises(RuntimeError):
        step.views(object(), 1)
    assert step.fits(torch.zeros(1), torch.zeros(1), object()) == 0 and step.defer(object(), *[torch.zeros(1)] * 4) is None


def test_views_of_a_layer():
    from trimkv_amd.cache_utils import _Slab
    s = _Slab(2, 3, 64, 10, torch.bfloat16, torch.float32, "cpu", False)
    for t, base, tail in zip(s.rows(7), (s.k, s.v, s.lb, s.pos), ((64,), (64,), (), ())):
        assert t.shape == (2, 3, 7, *tail) and t.data_ptr() == base.data_ptr() and t.stride() == base.view(2, 3, 10, *tail).stride()
    for t, base, width in zip(s.flat(), (s.k, s.v, s.lb, s.pos), (64, 64, 1, 1)):
        assert t.shape == (60, width) and t.data_ptr() == base.data_ptr() and t.is_contiguous()
    assert np.frombuffer(s.step, dtype=np.int64)[6:10].tolist() == [6, 3, 10, 64]
