"""GPU tests of the chunk-prefill attention with the keys of a query tile divided among workgroups
(trimkv_prefill_attn_split), against the undivided kernel and the fp32 oracle."""
import numpy as np
import pytest
import torch

from oracle.attn_ref import ragged_attention
from tests.gpu_util import DEV, attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,D,dtype,Q,lens,shares_of", [
    (1, 128, torch.bfloat16, 300, [300, 1025, 0, 30], (1, 2, 17, 40)),     # an empty segment and one shorter than the chunk
    (3, 96, torch.float16, 64, [64, 65, 127, 640], (1, 3)),                # the shortest chunk; padded rows of a query tile
    (5, 64, torch.bfloat16, 130, [191, 192, 193, 1500], (2, 8)),           # lengths around a tile of 64 keys
    (8, 128, torch.bfloat16, 77, [2000, 77, 1999, 400], (5, 32)),
    (1, 128, torch.bfloat16, 63, [63, 1025, 0, 30], (1, 3, 17)),           # short chunks
    (2, 96, torch.float16, 33, [64, 129, 500, 700], (1, 5)),
    (3, 64, torch.bfloat16, 2, [1, 64, 65, 900], (1, 2)),
    (8, 128, torch.bfloat16, 17, [800, 17, 16, 400], (4, 13)),
])
def test_divided_keys_match_the_whole_and_the_oracle(G, D, dtype, Q, lens, shares_of):
    """The two kernels round P to 16 bits against different references: u Sum p |v| on either side, the row sums the same
    again, and one rounding of each output -- together below 4 u max|v| + 2 u |out| <= 6 u max|v|, u = 2^-9 (bf16), 2^-12 (fp16)."""
    from trimkv_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(G * 100 + D)
    B, H, N, longest = 2, 2, sum(lens), max(lens)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    base = torch.randn(D, generator=gen)
    ramp = torch.cat([torch.linspace(-1.0, 1.0, n) * (-1) ** i for i, n in enumerate(lens)])[:, None]
    k = (torch.randn(N, D, generator=gen) + base * ramp).to(dtype)         # row maxima in the last shares, or in the first
    v = torch.randn(N, D, generator=gen).to(dtype)
    q = (torch.randn(B, H * G, Q, D, generator=gen) + 0.5 * base).to(dtype)
    want = ragged_attention(q, k, v, cu, H)
    qd, kd, vd, start = q.to(DEV), k.to(DEV), v.to(DEV), cu[:-1].contiguous().to(DEV)
    ln = torch.tensor(lens, dtype=torch.int32, device=DEV)
    stream = _lib.current_stream(qd.device)

    def call(name, *more):
        out = torch.full((B, Q, H * G, D), float("nan"), dtype=dtype, device=DEV)
        _lib.check(getattr(lib, name)(qd.data_ptr(), *qd.stride()[:3], out.data_ptr(), kd.data_ptr(), vd.data_ptr(), ln.data_ptr(), start.data_ptr(),
                                      B, H, G, Q, longest, D, _lib.dtype_code(dtype), D ** -0.5, longest, *more, stream), name)
        return out.cpu()

    whole = call("trimkv_prefill_attn")
    bound = 6 * float(v.abs().max()) * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12)
    for tiles in shares_of:
        need = lib.trimkv_prefill_split_workspace(B, H, G, Q, longest, tiles)
        work = torch.full((need // 4 + 64,), float("nan"), device=DEV)     # what it held counts for nothing, nothing past it is written
        work[need // 4:] = 7.0
        out = call("trimkv_prefill_attn_split", tiles, work.data_ptr(), need)
        assert (work[need // 4:] == 7.0).all()
        assert float((out.float() - whole.float()).abs().max()) <= bound, tiles
        ok, err = attn_close(out, want)
        assert ok, (tiles, err)


@pytest.mark.parametrize("B,H,G,Q,n", [(1, 2, 4, 300, 3000), (1, 1, 2, 128, 8200), (2, 8, 2, 640, 2100), (1, 8, 4, 50, 3000)])
def test_the_rule_divides_few_query_tiles_and_the_public_call_follows_it(B, H, G, Q, n):
    from trimkv_amd import _lib
    from trimkv_amd.attn.hip_attn import prefill_attention
    assert 0 < _lib.load().trimkv_prefill_split_tiles(B, H, G, Q, n, 0) < (n + 63) // 64
    gen = torch.Generator().manual_seed(n)
    q = torch.randn(B, Q, H * G, 128, generator=gen).to(torch.bfloat16).transpose(1, 2)
    k, v = (torch.randn(B * H * n, 128, generator=gen).to(torch.bfloat16) for _ in range(2))
    cu = torch.arange(B * H + 1, dtype=torch.int32) * n
    out = prefill_attention(q.to(DEV), k.to(DEV), v.to(DEV), B, H, G, None, None, n, n, 128 ** -0.5)
    ok, err = attn_close(out, ragged_attention(q, k, v, cu, H))
    assert ok, err


def test_the_rule_hears_how_uneven_the_segments_are(monkeypatch):
    """A ragged cache of equal lengths is no uneven one; after budgets have been applied the mean length says how uneven it is.
    Rows that come packed without their number count as alike."""
    from trimkv_amd import BatchedDynamicBudgetTrimKVCache, get_attention_interface
    from trimkv_amd.attn import hip_attn
    heard, plain = [], hip_attn._prefill_split
    monkeypatch.setattr(hip_attn, "_prefill_split", lambda *a: heard.append(a[-1]) or plain(*a))
    attend, gen = get_attention_interface("db_attn_flash_batched"), torch.Generator().manual_seed(0)
    B, H, Q, n = 1, 4, 70, 400
    cache = BatchedDynamicBudgetTrimKVCache()

    def chunk(S, at, **how):
        k, v = (torch.randn(B, H, S, 128, generator=gen).to(torch.bfloat16).to(DEV) for _ in range(2))
        keys, values, _, _, kw = cache.update(k, v, -torch.rand(B, H, S, generator=gen).to(DEV) - 0.01, torch.arange(at, at + S).to(DEV), 0, how)
        q = torch.randn(B, 2 * H, S, 128, generator=gen).to(torch.bfloat16).to(DEV)
        attend(None, q, keys, values, None, flash_attn_kwargs=kw)
        return q, keys, values, kw
    chunk(n, 0)
    cache.set_budgets(np.array([400, 100, 100, 200]))
    cache.evict_to_budgets()
    chunk(Q, n)                                       # 470, 170, 170, 270: 57 % of 470 in the mean
    q, keys, values, kw = chunk(Q, n + Q, packed=True)
    del kw["rows"]
    attend(None, q, keys, values, None, flash_attn_kwargs=kw)
    assert heard == [0, 57, 62, 0]
