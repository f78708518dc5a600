"""GPU tests of trimkv_append where a segment's new rows are spread over several workgroups, against plain indexing."""
import pytest
import torch

from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,D,cap", [(127, 128, 400), (128, 128, 400), (129, 96, 400), (257, 64, 400), (300, 256, 1000), (147, 8, 1 << 20), (130945, 8, 131072)])
def test_rows_lengths_and_prefix_sums(S, D, cap):
    """Around the 128 rows of a workgroup; rows of more pieces than it has in flight; a slab of 2^20 rows and a chunk of 1024 workgroups, whose lengths a launch of its own
    advances; segments that are empty, end flush with the slab, or would not fit (untouched)."""
    from trimkv_amd import _lib
    lib, B, H = _lib.load(), 2, 2
    gen = torch.Generator().manual_seed(S)
    nseg = B * H
    lens = torch.tensor([0, cap - S, 7, cap - S + 1], dtype=torch.int32)
    k, v = (torch.randn(B, H, S, D, generator=gen).to(torch.bfloat16) for _ in range(2))
    lb, pos = torch.randn(B, H, S, generator=gen), torch.arange(5, 5 + S)
    slabs = [torch.zeros(nseg, cap, D, dtype=torch.bfloat16, device=DEV) for _ in range(2)] + [torch.zeros(nseg, cap, device=DEV), torch.zeros(nseg, cap, dtype=torch.int64, device=DEV)]
    want = [t.cpu() for t in slabs]
    for s in range(nseg - 1):
        n = int(lens[s])
        for t, new in zip(want, (k.view(nseg, S, D), v.view(nseg, S, D), lb.view(nseg, S), pos.expand(nseg, S))):
            t[s, n:n + S] = new[s]
    seg_len, cu = lens.to(DEV), torch.zeros(nseg + 1, dtype=torch.int32, device=DEV)
    kd, vd, lbd, pd = (t.to(DEV) for t in (k, v, lb, pos))
    _lib.check(lib.trimkv_append(*(t.data_ptr() for t in slabs), seg_len.data_ptr(), cu.data_ptr(), nseg, H, cap, D, _lib.BF16, _lib.F32,
                                 kd.data_ptr(), vd.data_ptr(), *kd.stride()[:3], lbd.data_ptr(), *lbd.stride(), pd.data_ptr(), 0, 0, 1,
                                 S, cap, _lib.current_stream(kd.device)), "trimkv_append")
    assert seg_len.tolist() == [S, cap, 7 + S, cap - S + 1]
    assert cu.tolist() == [0, S, 2 * S, 3 * S, 0]
    assert all(torch.equal(got.cpu(), w) for got, w in zip(slabs, want))


@pytest.mark.parametrize("S,length", [(100, (1 << 20) + 5), (100, 2 ** 31 - 100), (300, (3 << 20) + 5), (300, 2 ** 31 - 1), (300, -5)])
def test_lengths_that_cannot_be_are_left_alone(S, length):
    """One workgroup to a segment takes a length as it is; three leave a count of up to two in its upper bits."""
    from trimkv_amd import _lib
    lib, cap, D = _lib.load(), 400, 64
    k = torch.ones(1, 2, S, D, dtype=torch.bfloat16, device=DEV)
    slabs = [torch.zeros(2, cap, D, dtype=torch.bfloat16, device=DEV) for _ in range(2)] + [torch.zeros(2, cap, device=DEV), torch.zeros(2, cap, dtype=torch.int64, device=DEV)]
    seg_len, lb, pos = torch.tensor([length, 3], dtype=torch.int32, device=DEV), torch.ones(1, 2, S, device=DEV), torch.ones(S, dtype=torch.int64, device=DEV)
    _lib.check(lib.trimkv_append(*(t.data_ptr() for t in slabs), seg_len.data_ptr(), None, 2, 2, cap, D, _lib.BF16, _lib.F32, k.data_ptr(), k.data_ptr(), *k.stride()[:3],
                                 lb.data_ptr(), *lb.stride(), pos.data_ptr(), 0, 0, 1, S, cap, _lib.current_stream(k.device)), "trimkv_append")
    assert seg_len.tolist() == [length, 3 + S]
    assert all(not t[0].any() and t[1].float().sum() == t[1, 3:3 + S].numel() for t in slabs)
