"""GPU tests of the chunk-prefill attention whose keys are cut into equal runs over all query tiles (trimkv_prefill_attn_shares),
against the undivided kernel and the fp32 oracle."""
import numpy as np
import pytest
import torch

from oracle.attn_ref import ragged_attention
from tests.gpu_util import DEV, attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,D,dtype,Q,lens", [
    (1, 128, torch.bfloat16, 300, [300, 1025, 0, 30]),              # an empty segment, one shorter than the chunk; fewer units than workgroups
    (3, 96, torch.float16, 64, [64, 65, 127, 640]),                 # the shortest chunk; padded rows of a query tile
    (5, 64, torch.bfloat16, 130, [191, 192, 193, 9000]),            # one query tile over many workgroups
    (8, 128, torch.bfloat16, 333, [2000, 333, 0, 400]),             # runs that hold whole query tiles
    (2, 128, torch.bfloat16, 2100, [2100, 4000, 2163, 2500, 2101, 3000, 2164, 2600, 2100, 2200, 2300, 0, 2165, 5, 2400, 3500]),   # 272 query tiles, two and more to a run
])
def test_equal_shares_match_the_whole_and_the_oracle(G, D, dtype, Q, lens):
    """The bound of the divided kernel holds: the kernels round P to 16 bits against different references, u Sum p |v| on either
    side, the row sums the same again, and one rounding of each output -- below 6 u max|v|, u = 2^-9 (bf16), 2^-12 (fp16)."""
    from trimkv_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(G * 100 + D)
    H = 2
    B, N, longest = len(lens) // H, sum(lens), max(lens)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    base = torch.randn(D, generator=gen)
    ramp = torch.cat([torch.linspace(-1.0, 1.0, n) * (-1) ** i for i, n in enumerate(lens)])[:, None]
    k = (torch.randn(N, D, generator=gen) + base * ramp).to(dtype)         # row maxima in the last shares, or in the first
    v = torch.randn(N, D, generator=gen).to(dtype)
    q = (torch.randn(B, H * G, Q, D, generator=gen) + 0.5 * base).to(dtype)
    qd, kd, vd, start = q.to(DEV), k.to(DEV), v.to(DEV), cu[:-1].contiguous().to(DEV)
    ln = torch.tensor(lens, dtype=torch.int32, device=DEV)
    stream = _lib.current_stream(qd.device)

    def call(name, *more):
        out = torch.full((B, Q, H * G, D), float("nan"), dtype=dtype, device=DEV)
        _lib.check(getattr(lib, name)(qd.data_ptr(), *qd.stride()[:3], out.data_ptr(), kd.data_ptr(), vd.data_ptr(), ln.data_ptr(), start.data_ptr(),
                                      B, H, G, Q, longest, D, _lib.dtype_code(dtype), D ** -0.5, longest, *more, stream), name)
        return out.cpu()

    whole = call("trimkv_prefill_attn")
    need = lib.trimkv_prefill_shares_workspace(B, H, G, Q)
    work = torch.full((need // 4 + 64,), float("nan"), device=DEV)         # what it held counts for nothing, nothing past it is written
    work[need // 4:] = 7.0
    out = call("trimkv_prefill_attn_shares", work.data_ptr(), need)
    assert (work[need // 4:] == 7.0).all()
    bound = 6 * float(v.abs().max()) * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12)
    assert float((out.float() - whole.float()).abs().max()) <= bound
    if N < 20000:
        ok, err = attn_close(out, ragged_attention(q, k, v, cu, H))
        assert ok, err


@pytest.mark.parametrize("B,H,G,Q,n,pays", [(3, 8, 2, 777, 9000, True), (1, 8, 4, 2100, 4200, True), (1, 8, 4, 2040, 2100, False), (4, 8, 5, 2048, 7000, False)])
def test_the_public_call_follows_the_rule(B, H, G, Q, n, pays, monkeypatch):
    """168 and 264 query tiles of long caches in equal shares, 256 of short ones and 1312 of many segments whole: all as the whole kernel has it."""
    from trimkv_amd import _lib
    from trimkv_amd.attn import hip_attn
    lib = _lib.load()
    assert lib.trimkv_prefill_split_tiles(B, H, G, Q, n, 0) == 0 and bool(lib.trimkv_prefill_equal_shares(B, H, G, Q, n, 0)) == pays
    gen = torch.Generator(device=DEV).manual_seed(n)
    q = torch.randn(B, H * G, Q, 128, generator=gen, device=DEV, dtype=torch.bfloat16)
    k, v = (torch.randn(B * H * n, 128, generator=gen, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    out = hip_attn.prefill_attention(q, k, v, B, H, G, None, None, n, n, 128 ** -0.5)
    monkeypatch.setattr(hip_attn, "_prefill_shares", lambda *a: 0)
    whole = hip_attn.prefill_attention(q, k, v, B, H, G, None, None, n, n, 128 ** -0.5)
    assert float((out.float() - whole.float()).abs().max()) <= 6 * float(v.abs().max()) * 2.0 ** -9
    if not pays:
        assert torch.equal(out, whole)
