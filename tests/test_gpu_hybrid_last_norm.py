"""The norm behind the last layer in that layer's own launch: trimkv_last_norm against the launches it stands for.

Bound: both are fp32 expressions of the same sums in another order (at most 2^-20 of the value here), rounded once."""
import pytest
import torch

from .hybrid_util import attention, build, config, mlstm, weights
from trimkv_amd import hybrid_ops as ops
from trimkv_amd.hybrid_cache import HybridCache

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width,top", [(8, 1), (72, 1), (1023, 1), (1024, 3), (1028, 1), (2048, 1), (4096, 4), (8192, 1), (8200, 2), (16384, 1)])
def test_against_the_launches_it_stands_for(width, top, dtype):
    gen = torch.Generator(device=DEV).manual_seed(width)
    rnd = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    T, stride = 7, ops.padded(width)
    x, y, w, v = rnd(T, stride), rnd(T * top, width).to(dtype), 1 + 0.2 * rnd(width), 1 + 0.2 * rnd(width)
    yw = rnd(T, top).abs() if top > 1 else None
    cu, slots, seen = (torch.tensor(a, dtype=torch.int32, device=DEV) for a in ([0, 3, 4, 7], [4, 0, 2], [[5, 1], [9, 9], [0, 0], [7, 7], [3, 2]]))
    batch = ops.PackedBatch((3, 1, 3), (4, 0, 2), cu, slots, seen.clone(), 5)
    before = x.clone()
    got = ops.last_norm(x, y, w, 1e-5, yw, 0.7, v, batch)
    assert torch.equal(x, before)
    ops.residual_norm(x, None, y, w, 1e-5, yw, 0.7)
    want = ops.rms_rows(x, None, v, 1e-5, dtype)
    assert ((got.float() - want.float()).abs() <= (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -20) * want.float().abs() + 1e-30).all()
    if dtype == torch.bfloat16:
        assert (got != want).float().mean() < 0.01        # a rounding here and there
    other = ops.PackedBatch((3, 1, 3), (4, 0, 2), cu, slots, seen.clone(), 5)
    ops.advance(other)
    assert torch.equal(batch.seen_dev, other.seen_dev)


@pytest.mark.gpu
def test_who_looks_at_the_stream_sees_it():
    cfg = config([attention(), mlstm()])
    model = build(cfg, weights(cfg), torch.bfloat16).to(DEV).eval()
    ids = torch.randint(0, 97, (9,), device=DEV)
    run = lambda **kw: model(ids, past_key_values=model.new_cache(2), lengths=[5, 4], **kw).logits
    want, streams = run(), []
    copies = []
    assert torch.allclose(run(layers_out=copies), want, rtol=2 ** -6, atol=1e-2)
    for module, look in ((model.model, lambda m, i, o: streams.append(o.clone())), (model.model.layers[-1], lambda m, i, o: streams.append(i[0].clone()))):
        handle = module.register_forward_hook(look)
        assert torch.allclose(run(), want, rtol=2 ** -6, atol=1e-2)
        handle.remove()
    for s in streams:
        assert torch.equal(s[:, :copies[-1].shape[1]], copies[-1])


@pytest.mark.gpu
def test_caches_that_count_tokens_by_a_way_of_their_own():
    """A subclass or an instance with an ``advance`` of its own is asked once a step, and tokens count once."""
    class Own(HybridCache):
        def advance(self, batch):
            asked.append(batch.lengths)
            super().advance(batch)

    cfg = config([attention(), mlstm()])
    model = build(cfg, weights(cfg), torch.bfloat16).to(DEV).eval()
    ids = torch.randint(0, 97, (9,), device=DEV)

    def steps(cache):
        out = model(ids, past_key_values=cache, lengths=[5, 4]).logits, model(ids[:2], past_key_values=cache, lengths=[1, 1]).logits
        return *out, cache.seen.tolist(), list(cache.tokens_seen)
    want, asked = steps(model.new_cache(2)), []
    own, patched = model.new_cache(2), model.new_cache(2)
    own.__class__ = Own
    real = patched.advance
    patched.advance = lambda batch: (asked.append(batch.lengths), real(batch))
    for cache in (own, patched):
        got = steps(cache)
        assert asked == [(5, 4), (1, 1)] and got[2:] == want[2:]
        for a, b in zip(got[:2], want[:2]):
            assert torch.allclose(a, b, rtol=2 ** -6, atol=1e-2)
        asked.clear()
