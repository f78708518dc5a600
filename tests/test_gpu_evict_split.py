"""Evictions whose rows are moved by several workgroups per segment (trimkv_evict_split) against a plain gather: patterns whose
shifts are the smallest and the largest, rows on both sides of a chunk's end, chunks that lose everything, work lists, segments
that lose more rows than the workspace was sized for, and every row size and log-beta type."""
import numpy as np
import pytest
import torch

from trimkv_amd import BatchedDynamicBudgetTrimKVCache, TrimKVCache, _lib
import trimkv_amd.cache_utils as cache_utils
from tests.gpu_util import DEV
from tests.test_gpu_evict_patterns import _patterns

pytestmark = pytest.mark.gpu


@pytest.fixture
def always_split(monkeypatch):
    calls = []
    monkeypatch.setattr(cache_utils, "split_evict", lambda *a: calls.append(a) or True)
    return calls


def _filled(cls, layers, B, H, n, D, kv_dtype, lb_dtype, keep):
    """A cache whose segments keep exactly the rows ``keep`` when cut to keep.size rows; returns it and its contents."""
    gen = torch.Generator().manual_seed(n + D)
    cache, held = cls(), []
    for l in range(layers):
        k, v = (torch.randn(B, H, n, D, generator=gen).to(kv_dtype) for _ in range(2))
        lb = torch.full((B, H, n), -5.0)
        lb[:, :, torch.from_numpy(keep)] = -1e-7 * (1.0 + torch.rand(B, H, keep.size, generator=gen))
        lb = lb.to(lb_dtype)
        cache.update(k.to(DEV), v.to(DEV), lb.to(DEV), torch.arange(n, device=DEV), l)
        held.append((k, v, lb))
    return cache, held


def _check(cache, held, rows, what):
    for l, (k, v, lb) in enumerate(held):
        s = cache._slabs[l]
        m = rows.size
        assert (s.seg_len.cpu() == m).all(), what
        for got, want in ((s.k, k), (s.v, v), (s.lb, lb)):
            want = want.flatten(0, 1)[:, torch.from_numpy(rows)]
            assert torch.equal(got[:, :m].cpu(), want), what
        assert torch.equal(s.pos[:, :m].cpu(), torch.from_numpy(rows).expand(s.nseg, m)), what


@pytest.mark.parametrize("D,kv_dtype,lb_dtype", [(128, torch.bfloat16, torch.float32), (96, torch.float16, torch.float32), (64, torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("n,M", [(4224, 4096), (5000, 4999), (3000, 1025), (2600, 1024), (2049, 1537), (9000, 3000), (2100, 1)])
def test_patterns(n, M, D, kv_dtype, lb_dtype, always_split):
    for name, keep in _patterns(n, M):
        keep = np.asarray(keep)
        if keep.size != M:
            continue
        cache, held = _filled(TrimKVCache, 2 if D == 128 else 1, 1, 3, n, D, kv_dtype, lb_dtype, keep)
        cache.compress("alpha", memory_size=M, buffer_size=n - M)
        _check(cache, held, keep, name)
    assert always_split


@pytest.mark.parametrize("spill", [4, 130, 512])
def test_segments_that_lose_more_than_the_workspace_was_sized_for(spill, always_split):
    n, M = 3300, 3100          # 200 rows lost: more than 4 and 130 (moved whole), less than 512
    keep = np.sort(np.random.default_rng(1).choice(n, size=M, replace=False))
    cache, held = _filled(TrimKVCache, 2, 2, 2, n, 128, torch.bfloat16, torch.float32, keep)
    cache._evict_layers([0, 1], M, None, 0, _lib.SCORE_ALPHA, _lib.ROUND_UPCAST, 0, n + 1, spill=spill)
    _check(cache, held, keep, f"spill {spill}")


def test_work_list_with_budgets_of_its_own_against_one_workgroup_per_segment(monkeypatch):
    """Budgets from one row to all but one, a few segments due: the listed split against trimkv_evict_listed."""
    B, H, n, L = 2, 4, 4000, 2
    budgets = np.array([[n, 3900, n, 1, n, n, 2000, n], [n, n, 1030, n, 3999, n, n, 520]])
    states = []
    for split in (False, True):
        monkeypatch.setattr(cache_utils, "split_evict", lambda *a, split=split: split)
        gen = torch.Generator().manual_seed(5)
        cache = BatchedDynamicBudgetTrimKVCache()
        for l in range(L):
            k, v = (torch.randn(B, H, n, 128, generator=gen).to(torch.bfloat16).to(DEV) for _ in range(2))
            cache.update(k, v, (-torch.rand(B, H, n, generator=gen) - 0.01).to(DEV), torch.arange(n, device=DEV), l)
        cache.set_budgets(budgets)
        cache.evict_to_budgets(buffer_size=0)
        states.append([(t.cpu() for t in (cache.key_cache[l], cache.value_cache[l], cache.retention_weights[l], cache.kv_positions[l], cache.head_lens[l], cache.cu_seqlens_k[l]))
                       for l in range(L)])
    for a, b in zip(*states):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
    assert [int(t) for t in cache.head_lens[0]] == budgets[0].tolist()


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("layers", [3, 48, 49])
def test_layers_in_the_arguments_and_in_a_device_table(layers, split, monkeypatch):
    """Up to 48 layers travel with the launch, more in a device table; one query index for all, or one per layer."""
    monkeypatch.setattr(cache_utils, "split_evict", lambda *a: split)
    n, M = 2200, 2000
    keep = np.sort(np.random.default_rng(layers).choice(n, size=M, replace=False))
    for qs in (n + 1, [n + 1 + l for l in range(layers)]):
        cache, held = _filled(TrimKVCache, layers, 1, 1, n, 64, torch.bfloat16, torch.float32, keep)
        every = list(range(layers))
        cache._evict_layers(every, M, None, 0, _lib.SCORE_ALPHA, _lib.ROUND_UPCAST, 0, qs)
        _check(cache, held, keep, f"{layers} layers")
        assert (("host", *every) in cache._table_cache) == (layers <= 48)


def _selected_both_ways(lens, cap, budget, lb_dtype, strategy):
    lib, gen = _lib.load(), torch.Generator().manual_seed(budget % 97)
    (L, nseg), B, H, D = lens.shape, 2, 4, 64
    lb = [(-torch.randint(1, 6, (nseg, cap), generator=gen) / 8.0).to(lb_dtype).to(DEV) for _ in range(L)]
    pos = [torch.arange(cap, device=DEV).div(3, rounding_mode="floor").repeat(nseg, 1).contiguous() for _ in range(L)]
    k = [torch.randn(nseg, cap, D, generator=gen).to(torch.bfloat16).to(DEV) for _ in range(L)]
    ln = [lens[l].clone().to(DEV) for l in range(L)]
    tables = [torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device=DEV) for ts in (lb, pos, k, ln)]
    stream, code = _lib.current_stream(torch.device(DEV)), _lib.SCORE_ALPHA if strategy == "alpha" else _lib.SCORE_KNORM_ALPHA
    results = []
    for wide in (False, True):
        out = [torch.full((L, B), -1, dtype=torch.int32, device=DEV) for _ in range(2)] + [torch.full((L, nseg), -1, dtype=torch.int32, device=DEV) for _ in range(3)]
        args = (*(t.data_ptr() for t in tables), L, nseg, H, cap, D, _lib.BF16, _lib.dtype_code(lb_dtype), budget, 0, 0.0, cap + 5, code, _lib.ROUND_NATIVE,
                *(t.data_ptr() for t in out))
        if wide:
            ws = torch.full((L * lib.trimkv_group_threshold_workspace(1, nseg, H),), 255, dtype=torch.uint8, device=DEV)
            _lib.check(lib.trimkv_group_threshold_wide_each_layer(*args, ws.data_ptr(), ws.numel(), stream), "wide")
        else:
            _lib.check(lib.trimkv_group_threshold_each_layer(*args, stream), "single")
        results.append([t.cpu() for t in out])
    for a, b in zip(*results):
        assert torch.equal(a, b)
    want = lens.view(L, B, H).sum(-1).clamp(max=budget)
    assert torch.equal(results[0][3].view(L, B, H).sum(-1).int(), want.int())


@pytest.mark.parametrize("lb_dtype,strategy", [(torch.float32, "alpha"), (torch.bfloat16, "alpha"), (torch.float32, "knorm")])
@pytest.mark.parametrize("budget", [0, 1, 700, 10 ** 6])
def test_budgets_of_a_layer_selected_by_one_workgroup_and_by_one_per_segment(budget, lb_dtype, strategy):
    """Ties by the hundred, empty segments, lengths around the rows of wavefronts (64) and of the 256 or 1024 threads that read at a time."""
    lens = torch.tensor([[0, 1, 255, 256, 257, 1023, 1024, 1025], [1300, 1300, 64, 65, 0, 0, 0, 0], [5, 900, 1281, 1279, 3, 1, 2, 700]], dtype=torch.int32)
    _selected_both_ways(lens, 1300, budget, lb_dtype, strategy)


@pytest.mark.parametrize("lb_dtype,strategy", [(torch.float32, "alpha"), (torch.bfloat16, "alpha"), (torch.float32, "knorm")])
@pytest.mark.parametrize("budget", [4096, 12000])
def test_segments_of_more_rows_than_a_workgroup_has_in_flight(budget, lb_dtype, strategy):
    """4096 rows are four for each of 1024 threads: one less, as many, one more, twice as many and some."""
    lens = torch.tensor([[4095, 4096, 4097, 8191, 8192, 8193, 8200, 0], [5119, 5120, 5121, 3, 8200, 8200, 4097, 4096]], dtype=torch.int32)
    _selected_both_ways(lens, 8200, budget, lb_dtype, strategy)


@pytest.mark.parametrize("lb_dtype,strategy", [(torch.float32, "alpha"), (torch.bfloat16, "knorm")])
@pytest.mark.parametrize("layers,cap", [(32, 1024), (32, 1025), (33, 1025), (3, 1024)])
def test_either_side_of_where_workgroups_are_large(layers, cap, lb_dtype, strategy):
    """256 segments and 264; room for 1024 rows and for one more."""
    lens = torch.from_numpy(np.random.default_rng(layers + cap).integers(0, cap + 1, size=(layers, 8)).astype(np.int32))
    lens[0, :4] = torch.tensor([cap, 1023, 1024, 0])
    _selected_both_ways(lens, cap, 900, lb_dtype, strategy)


def _uneven(split, monkeypatch):
    """192 segments with lognormal budgets of 1 to 7600 rows, filled, cut, and 700 tokens later due again."""
    monkeypatch.setattr(cache_utils, "split_evict", lambda *a: False)
    L, B, H, n = 6, 4, 8, 7600
    budgets = np.exp(np.random.default_rng(3).normal(np.log(800.0), 1.0, (L, B * H))).clip(1, n).astype(np.int64)
    budgets[0, 0] = n
    gen = torch.Generator(device=DEV).manual_seed(4)
    cache, seen = BatchedDynamicBudgetTrimKVCache(), 0
    for more in (n + 1, 700):
        for l in range(L):
            k, v = (torch.randn(B, H, more, 128, generator=gen, device=DEV, dtype=torch.bfloat16) for _ in range(2))
            lb = -torch.rand(B, H, more, generator=gen, device=DEV) - 0.01
            cache.update(k, v, lb, torch.arange(seen, seen + more, device=DEV), l)
        seen += more
        cache.set_budgets(budgets)
        if more == 700:
            monkeypatch.setattr(cache_utils, "split_evict", lambda *a: split)
            del k, v, lb
            torch.cuda.synchronize()
            before = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
        cache.evict_to_budgets(buffer_size=0)
    torch.cuda.synchronize()
    peak, after = torch.cuda.max_memory_allocated() - before, torch.cuda.memory_allocated() - before
    held = [tuple(t.cpu() for t in (s.seg_len, s.cu)) + tuple(torch.cat([t[i, :int(m)] for i, m in enumerate(s.lens)]).cpu() for t in (s.k, s.v, s.lb, s.pos))
            for s in cache._slabs]
    assert all((s.lens == budgets[l]).all() for l, s in enumerate(cache._slabs))
    return held, peak, after, cache.memory_bytes()


def test_scratch_is_sized_by_what_the_due_segments_keep_and_given_back(monkeypatch):
    """Segments of unlike budgets: the scratch follows the rows that they keep, not the longest of them times their number, and
    nothing but work lists (a few KB) outlives the launches."""
    want, _, _, _ = _uneven(False, monkeypatch)
    got, peak, after, cache_bytes = _uneven(True, monkeypatch)
    for a, b in zip(want, got):
        assert all(torch.equal(x, y) for x, y in zip(a, b))
    assert 1 << 20 < peak < cache_bytes / 6, (peak, cache_bytes)
    assert after < 1 << 20


@pytest.mark.parametrize("how", ["limit", "out of memory"])
def test_without_room_for_scratch_a_workgroup_moves_each_segment(how, monkeypatch, always_split):
    n, M = 4224, 4096
    keep = np.sort(np.random.default_rng(2).choice(n, size=M, replace=False))
    cache, held = _filled(TrimKVCache, 2, 1, 3, n, 128, torch.bfloat16, torch.float32, keep)
    if how == "limit":
        monkeypatch.setattr(cache_utils, "SPLIT_SCRATCH", 1 << 20)
    else:
        empty, refused = torch.empty, []

        def short(*a, **kw):
            if kw.get("dtype") == torch.uint8:
                refused.append(a)
                raise torch.OutOfMemoryError("no memory")
            return empty(*a, **kw)
        monkeypatch.setattr(torch, "empty", short)
    cache.compress("alpha", memory_size=M, buffer_size=n - M)
    monkeypatch.undo()
    assert how == "limit" or refused
    _check(cache, held, keep, how)


@pytest.mark.parametrize("on_host", [0, 1])
def test_pairs_with_chunks_of_their_own(on_host):
    """A pair with just enough chunks, one with one too few, one with none, and lists that name chunks past the workspace's: those
    that do not fit are moved by one workgroup, nothing is written behind the workspace."""
    lib, n, M = _lib.load(), 3300, 3100                       # seven chunks of 512 kept rows
    keep = np.sort(np.random.default_rng(6).choice(n, size=M, replace=False))
    for first in ([0, 7, 13, 13, 20], [0, 0, 7, 21, 28], [-1, 7, 14, 20, 27], [0, 7, 14, 10 ** 9, 10 ** 9 + 7]):
        cache, held = _filled(TrimKVCache, 2, 1, 2, n, 128, torch.bfloat16, torch.float32, keep)
        total = 28
        need = lib.trimkv_evict_split_rooms_workspace(4, total, 128, 200)
        ws = torch.full((need + 4096,), 9, dtype=torch.uint8, device=DEV)
        lists = torch.tensor([3, 0, 2, 1] + first, dtype=torch.int32, device=DEV)
        table = cache._host_table([0, 1])
        at = table.ctypes.data if on_host else cache._device_tables([0, 1])["slabs"].data_ptr()
        _lib.check(lib.trimkv_evict_split_rooms(at, on_host, 2, 2, 128, _lib.BF16, _lib.F32, M, None, 0, 0, n + 1, _lib.SCORE_ALPHA, _lib.ROUND_UPCAST, 0, n, 200,
                                                lists.data_ptr(), 4, lists.data_ptr() + 16, total, 7, ws.data_ptr(), need, _lib.current_stream(ws.device)), "rooms")
        assert (ws[need:] == 9).all()
        _check(cache, held, keep, str(first))


@pytest.mark.parametrize("moved", [639, 640, 641])
@pytest.mark.parametrize("first", [0, 100, 512, 700])
def test_fewest_rows_that_are_moved_by_several_workgroups(first, moved):
    """A kept prefix stays where it is; behind it 640 rows go to chunks, 639 do not, listed and not."""
    lib, M = _lib.load(), first + moved
    n, spill, per = M + 150, 200, -(-M // 512)
    keep = np.concatenate([np.arange(first), first + 1 + np.sort(np.random.default_rng(first + moved).choice(n - first - 1, size=moved, replace=False))])
    need = lib.trimkv_evict_split_rooms_workspace(4, 4 * per, 128, spill)
    lists = torch.tensor([3, 0, 2, 1] + [per * i for i in range(5)], dtype=torch.int32, device=DEV)
    for listed in (False, True):
        cache, held = _filled(TrimKVCache, 2, 1, 2, n, 128, torch.bfloat16, torch.float32, keep)
        ws = torch.full((need + 4096,), 9, dtype=torch.uint8, device=DEV)
        _lib.check(lib.trimkv_evict_split_rooms(cache._host_table([0, 1]).ctypes.data, 1, 2, 2, 128, _lib.BF16, _lib.F32, M, None, 0, 0, n + 1, _lib.SCORE_ALPHA, _lib.ROUND_UPCAST,
                                                0, n, spill, lists.data_ptr() if listed else None, 4, lists.data_ptr() + 16 if listed else None, 4 * per, per, ws.data_ptr(), need,
                                                _lib.current_stream(ws.device)), "rooms")
        assert (ws[need:] == 9).all()
        assert (int((ws[:need] != 9).sum()) > 4 * 16) == (moved >= cache_utils._SPLIT_FROM)       # more than a head for each pair: lists of rows
        _check(cache, held, keep, f"{first} {moved} {listed}")


@pytest.mark.parametrize("longest,segments,kept,spill,D,split", [
    (2176, 64, 2048, 128, 128, True), (2176, 64, 2048, 128, 96, True), (2176, 64, 2048, 128, 64, False), (2176, 66, 2048, 128, 128, True), (2176, 67, 2048, 128, 128, False),
    (4224, 64, 4096, 128, 64, True), (4224, 72, 4096, 511, 128, True), (4224, 73, 4096, 128, 128, False), (4224, 64, 4096, 512, 128, False),
    (8320, 64, 8192, 128, 128, True), (8320, 128, 8192, 128, 128, False), (12288, 32, 8192, 512, 64, True), (12288, 64, 8192, 512, 96, False),
    (4096, 8, 2048, 512, 128, True), (4096, 8, 2047, 512, 128, False), (4096, 8, 2048, 512, 96, True), (4096, 8, 2048, 512, 64, False),
    (2688, 8, 2559, 128, 64, False), (2688, 8, 2560, 128, 64, True), (32769, 8, 32000, 512, 128, False), (8320, 8, 8192, 128, 256, False)])
def test_where_rows_are_moved_by_several_workgroups(longest, segments, kept, spill, D, split):
    assert cache_utils.split_evict(longest, segments * longest, kept, spill, D) is split


@pytest.mark.parametrize("entry", ["split", "split_listed", "host_layers"])
@pytest.mark.parametrize("spill", [200, 512])
def test_entry_points_that_give_every_pair_room_for_the_longest_segment(entry, spill):
    lib, n, M = _lib.load(), 3300, 3100
    keep = np.sort(np.random.default_rng(7).choice(n, size=M, replace=False))
    cache, held = _filled(TrimKVCache, 2, 1, 2, n, 96, torch.float16, torch.float32, keep)
    need = lib.trimkv_evict_split_workspace(4, n, 96, spill)
    ws = torch.full((need + 4096,), 9, dtype=torch.uint8, device=DEV)
    work = torch.tensor([2, 0, 3, 1], dtype=torch.int32, device=DEV)
    shape = (2, 2, 96, _lib.F16, _lib.F32, M, None, 0, 0, n + 1, _lib.SCORE_ALPHA, _lib.ROUND_UPCAST, 0, n, spill)
    room = (ws.data_ptr(), need, _lib.current_stream(ws.device))
    if entry == "host_layers":
        _lib.check(lib.trimkv_evict_host_layers(cache._host_table([0, 1]).ctypes.data, *shape, *room), entry)
    else:
        listed = (work.data_ptr(), 4) if entry == "split_listed" else (None, 0)
        _lib.check(lib.trimkv_evict_split(cache._device_tables([0, 1])["slabs"].data_ptr(), *shape, *listed, *room), entry)
    assert (ws[need:] == 9).all()
    _check(cache, held, keep, entry)
