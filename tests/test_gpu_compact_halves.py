"""GPU tests of trimkv_compact_threshold_halves (keys and values of a segment moved by a workgroup each) against the compaction that
moves both, bit for bit."""
import numpy as np
import pytest
import torch

from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,lb_dtype", [(128, torch.float32), (96, torch.bfloat16), (64, torch.float32), (8, torch.float16)])
@pytest.mark.parametrize("lens", [[1, 0, 4097, 31], [2048, 2047, 2049, 300], [9000, 5, 1023, 1024]])
def test_halves_leave_what_the_whole_leaves(D, lb_dtype, lens):
    """Segments without rows, shorter than a tile and of several tiles; nothing, some and all of the rows below the cut, ties at it
    (log beta of few values); a segment whose length is corrupt stays as it is."""
    from trimkv_amd import _lib
    lib, L, nseg, cap = _lib.load(), 2, len(lens), max(lens) + 7
    gen = torch.Generator(device=DEV).manual_seed(D + sum(lens))
    # scores are log beta * age: ages around 40000, 16 values of log beta, the cut on one of them
    lb0 = [(-torch.randint(1, 17, (nseg, cap), generator=gen, device=DEV) / 16.0).to(lb_dtype) for _ in range(L)]
    pos0 = [torch.randint(0, 2, (nseg, cap), generator=gen, device=DEV) + torch.arange(cap, device=DEV) // 4096 for _ in range(L)]
    k0, v0 = ([torch.randn(nseg, cap, D, generator=gen, device=DEV, dtype=torch.bfloat16) for _ in range(L)] for _ in range(2))
    q = 40000
    score = (-0.5 * (q - 1.0)) if lb_dtype == torch.float32 else float((torch.tensor(q - 1.0).to(lb_dtype) * torch.tensor(-0.5).to(lb_dtype)))
    key = np.float32(score).view(np.uint32)
    key = int(~key & 0xffffffff) if key >> 31 else int(key | 0x80000000)
    thr = torch.tensor([[key, key], [0, 0xffffffff]], dtype=torch.int64, device=DEV).to(torch.int32)         # layer 0: the cut; layer 1: keep all, keep none
    take = torch.tensor([[50, 2 ** 31 - 1], [2 ** 31 - 1, 0]], dtype=torch.int32, device=DEV)
    base = torch.tensor([[0, 20, 0, 5], [0] * 4], dtype=torch.int32, device=DEV)
    dt = np.dtype([("k", "<u8"), ("v", "<u8"), ("lb", "<u8"), ("pos", "<u8"), ("len", "<u8"), ("q", "<i8"), ("cap", "<i4"), ("res", "<i4")])

    def run(name):
        slabs = [[t.clone() for t in s] for s in zip(k0, v0, lb0, pos0)]
        seg = [torch.tensor(lens, dtype=torch.int32, device=DEV), torch.tensor(lens[::-1], dtype=torch.int32, device=DEV)]
        seg[1][1] = cap + 1
        arr = np.zeros(L, dtype=dt)
        for i, s in enumerate(slabs):
            arr[i] = (*(t.data_ptr() for t in s), seg[i].data_ptr(), 0, cap, 0)
        table = torch.from_numpy(arr.view(np.uint8)).to(DEV)
        need = lib.trimkv_compact_halves_workspace(L, nseg, max(lens))
        ws = torch.full((need + 64,), 7, dtype=torch.uint8, device=DEV)
        _lib.check(getattr(lib, name)(table.data_ptr(), L, nseg, 2, D, _lib.BF16, _lib.dtype_code(lb_dtype), thr.data_ptr(), take.data_ptr(), 2, base.data_ptr(), q,
                                      _lib.SCORE_ALPHA, _lib.ROUND_NATIVE, max(lens), ws.data_ptr(), need, _lib.current_stream(torch.device(DEV))), name)
        assert (ws[need:] == 7).all()
        return slabs, seg

    (want, wlen), (got, glen) = run("trimkv_compact_threshold_layers"), run("trimkv_compact_threshold_halves")
    for l in range(L):
        assert torch.equal(wlen[l], glen[l])
        for w, g in zip(want[l], got[l]):
            for s in range(nseg):
                n = min(int(wlen[l][s]), cap)
                assert torch.equal(w[s, :n], g[s, :n]), (l, s)
    assert 0 < int(glen[0][lens.index(max(lens))]) < max(lens) and int(glen[1][1]) == cap + 1


def test_bad_arguments_are_refused():
    from trimkv_amd import _lib
    lib, x = _lib.load(), torch.zeros(4096, dtype=torch.uint8, device=DEV)
    p = x.data_ptr()
    call = lambda strategy=_lib.SCORE_ALPHA, max_len=64, ws=p, size=4096: lib.trimkv_compact_threshold_halves(p, 1, 2, 2, 8, _lib.BF16, _lib.F32, p, p, 0, p, 10, strategy, _lib.ROUND_NATIVE, max_len,
                                                                                                              ws, size, None)
    assert call(strategy=_lib.SCORE_KNORM_ALPHA) < 0 and call(max_len=32769, size=1 << 30) < 0 and call(ws=None) < 0 and call(size=100) < 0 and call(ws=p + 4) < 0


def test_a_cache_keeps_no_scratch_of_halves():
    from trimkv_amd import BatchedDynamicBudgetTrimKVCache
    from trimkv_amd.cache_utils import compact_halves
    L, B, H, S, D, keep = 2, 2, 4, 1500, 64, 500
    gen = torch.Generator(device=DEV).manual_seed(2)
    cache = BatchedDynamicBudgetTrimKVCache()
    for l in range(L):
        k, v = (torch.randn(B, H, S, D, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(2))
        cache.update(k, v, -torch.rand(B, H, S, generator=gen, device=DEV), torch.arange(S, device=DEV), l)
    assert compact_halves(L * B * H, S, L * B * H * S)
    cache.compress(strategy="alpha", memory_size=keep, buffer_size=0)
    assert cache.get_total_cached_tokens() == L * B * H * keep
    assert sum(t.numel() for t in cache._ws.values()) < 12 * L * B * H * S
