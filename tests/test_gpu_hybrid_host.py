"""What the host tells a step of the hybrid decoders travels in launches' arguments: nothing waits for the stream."""
import ctypes

import pytest
import torch

from trimkv_amd import _lib, hybrid_ops as ops
from trimkv_amd.fusitar import FusitarConfig, FusitarForCausalLM

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 63, 65, 255, 256, 257, 512, 513, 1300])
def test_words_arrive_whole(count):
    values = [(i * 2654435761) % (1 << 31) for i in range(count)]
    assert ops.put(values, torch.int32, torch.device(DEV)).tolist() == values
    wide = [v * 5 - (1 << 33) for v in values]
    assert ops.put(wide, torch.int64, torch.device(DEV)).tolist() == wide
    seen = torch.ones(2 * count + 3, 2, dtype=torch.int32, device=DEV)
    slots = list(range(1, 2 * count, 2))
    ops.reset_slots(seen, slots)
    want = torch.ones_like(seen)
    want[torch.tensor(slots, device=DEV)] = 0
    assert torch.equal(seen, want)


@pytest.mark.gpu
def test_prompts_wait_for_nothing_and_are_not_recorded():
    cfg = {"architecture": "Fusitar", "vocab": 64, "width": 128, "norm": {"eps": 1e-6}, "embedding": {"scale": 1.0}, "layers": [
        {"type": "attention", "mlp": None, "mixer": {"heads": 2, "kv_heads": 1, "dim": 32, "vdim": 32, "scale": 0.2, "mask": {"size": 16, "keep_first": 4}}}]}
    with torch.device(DEV):
        model = FusitarForCausalLM(FusitarConfig.from_dict(cfg), torch.bfloat16).eval().randomize(1)
    ids = torch.randint(0, 64, (40,), device=DEV)
    cache = model.new_cache(4)
    model(ids, past_key_values=cache, lengths=[30, 10], slots=cache.allocate(2), rows=None)      # first use of libraries
    want = model(ids[:25], past_key_values=cache, lengths=[25], slots=cache.allocate(1), logits_to_keep=2).logits
    torch.cuda.synchronize()
    torch.cuda.set_sync_debug_mode("error")
    try:
        slots = cache.allocate(1)
        got = model(ids[:25], past_key_values=cache, lengths=[25], slots=slots, logits_to_keep=2).logits
    finally:
        torch.cuda.set_sync_debug_mode("default")
    assert torch.equal(got, want)
    s = torch.cuda.Stream()
    cache.release(slots)
    before = list(cache.active), cache._free[:]
    with torch.cuda.stream(s):
        g = torch.cuda.CUDAGraph()
        g.capture_begin()
        try:
            for call in (lambda: ops.put([1], torch.int32, torch.device(DEV)), lambda: cache.allocate(1)):
                with pytest.raises(RuntimeError):
                    call()
        finally:
            g.capture_end()
    assert (list(cache.active), cache._free) == before


def test_bad_calls_are_refused():
    lib = ctypes.CDLL(_lib.HYBRID_LIB_PATHS["hybrid"])
    for name in ("trimkv_put_words", "trimkv_reset_slots"):
        getattr(lib, name).argtypes = _lib.HYBRID_SIGNATURES["hybrid"][name][1]
    one, words = ctypes.c_void_p(16), (ctypes.c_int32 * 2)(3, -1)
    at = ctypes.addressof(words)
    assert lib.trimkv_put_words(None, at, 1, None) == -1 and lib.trimkv_put_words(one, None, 1, None) == -1 and lib.trimkv_put_words(one, at, 0, None) == -2
    assert lib.trimkv_reset_slots(None, at, 1, 4, None) == -1 and lib.trimkv_reset_slots(one, at, 1, 3, None) == -2 and lib.trimkv_reset_slots(one, at, 2, 4, None) == -2
