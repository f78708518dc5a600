"""GPU tests of the chunk-prefill attention where scores outgrow the exponent reference that a row began with: within what bf16's exponents take, up to the last
powers of two of a row sum, beyond them (the query tile is done again, with row maxima), gradually (the reference moves by the row sums) and in fp16, against
64-bit sums."""
import numpy as np
import pytest
import torch

from oracle.attn_ref import ragged_attention
from tests.gpu_util import DEV, attn_close

pytestmark = pytest.mark.gpu


def _heights(how, n):
    """Height of every key along the direction that all queries share; 1 is about 65 powers of two of a score."""
    at = torch.arange(n, dtype=torch.float32)
    return {"jump": (at >= 700).float() * 6, "small jump": (at >= 700).float() * 0.8, "climb": at * (6 / n), "steep": ((at - 300) / 400).clamp(0, 1) * 6, "fall": 6 - at * (6 / n),
            "peak": (at == 1000).float() * 6, "last": (at == n - 140).float() * 6, "steps": (at / 300).floor()}[how]


def _whole(q, k, v, lens, B, H, G, n, at_most):
    """Undivided query tiles; lengths and starts are there, so that a bound of the lengths beyond them only chooses the kernel."""
    from trimkv_amd import _lib
    D, Q = q.shape[-1], q.shape[2]
    start = torch.arange(B * H, dtype=torch.int32, device=DEV) * n
    out = torch.empty(B, Q, H * G, D, dtype=q.dtype, device=DEV)
    _lib.check(_lib.load().trimkv_prefill_attn(q.data_ptr(), *q.stride()[:3], out.data_ptr(), k.data_ptr(), v.data_ptr(), lens.data_ptr(), start.data_ptr(),
                                               B, H, G, Q, n, D, _lib.dtype_code(q.dtype), D ** -0.5, at_most, _lib.current_stream(q.device)), "trimkv_prefill_attn")
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("G,D,Q", [(1, 128, 300), (5, 64, 130)])
@pytest.mark.parametrize("how", ["jump", "small jump", "climb", "steep", "fall", "peak", "last", "steps"])
def test_scores_that_outgrow_their_reference(how, G, D, Q, dtype):
    from trimkv_amd import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(G + D)
    B, H, lens = 1, 2, [1500, 1100]
    N, longest = sum(lens), max(lens)
    base = torch.randn(D, generator=gen)
    base = base * (D ** 0.5 / base.norm())
    k = (torch.cat([_heights(how, n) for n in lens])[:, None] * base + 0.3 * torch.randn(N, D, generator=gen)).to(dtype)
    v = torch.randn(N, D, generator=gen).to(dtype)
    q = (45.0 / D ** 0.5 * base + 0.3 * torch.randn(B, H * G, Q, D, generator=gen)).to(dtype)      # 45 nats, 65 powers of two
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    # Q * scale is rounded once: the oracle takes it as the kernel does, so that large scores agree
    c = D ** -0.5 * 1.4426950408889634
    rounded = (q.float() * c).to(dtype).double() / c
    s = torch.einsum("bhgqd,bhnd->bhgqn", rounded.view(B, H, G, Q, D), torch.stack([torch.cat([x.double(), torch.zeros(longest - x.shape[0], D, dtype=torch.float64)]) for x in k.split(lens)])[None]) * D ** -0.5
    ln = torch.tensor(lens)
    seen = torch.arange(longest)[None, None, :] <= (ln[:, None, None] - Q + torch.arange(Q)[None, :, None])
    p = torch.softmax(s.masked_fill(~seen[None, :, None], -float("inf")), -1)
    want = torch.einsum("bhgqn,bhnd->bqhgd", p, torch.stack([torch.cat([x.double(), torch.zeros(longest - x.shape[0], D, dtype=torch.float64)]) for x in v.split(lens)])[None]).reshape(B, Q, H * G, D)
    qd, kd, vd, start, lend = q.to(DEV), k.to(DEV), v.to(DEV), cu[:-1].contiguous().to(DEV), ln.int().to(DEV)
    stream = _lib.current_stream(qd.device)
    # P and the row sums rounded to 16 bits, one rounding of the output, as in the divided launches' bound: 6 u max|v|
    bound = 6 * float(v.abs().max()) * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12)

    def call(name, *more, at_most=longest):
        out = torch.full((B, Q, H * G, D), float("nan"), dtype=dtype, device=DEV)
        _lib.check(getattr(lib, name)(qd.data_ptr(), *qd.stride()[:3], out.data_ptr(), kd.data_ptr(), vd.data_ptr(), lend.data_ptr(), start.data_ptr(),
                                      B, H, G, Q, longest, D, _lib.dtype_code(dtype), D ** -0.5, at_most, *more, stream), name)
        return out.cpu()

    # a bound of the lengths that says much work: the kernel of launches that fill the chip
    outs = {"whole": call("trimkv_prefill_attn"), "whole, in two parts": call("trimkv_prefill_attn", at_most=1 << 20)}
    for tiles in (1, 5):
        need = lib.trimkv_prefill_split_workspace(B, H, G, Q, longest, tiles)
        work = torch.full((need // 4,), float("nan"), device=DEV)
        outs[f"split {tiles}"] = call("trimkv_prefill_attn_split", tiles, work.data_ptr(), need)
    need = lib.trimkv_prefill_shares_workspace(B, H, G, Q)
    work = torch.full((need // 4,), float("nan"), device=DEV)
    outs["shares"] = call("trimkv_prefill_attn_shares", work.data_ptr(), need)
    for name, out in outs.items():
        assert out.isfinite().all(), name
        assert float((out.double() - want).abs().max()) <= bound, (name, float((out.double() - want).abs().max()), bound)


@pytest.mark.parametrize("keys", [1, 4])
@pytest.mark.parametrize("at", ["first turn", "middle", "end"])
def test_row_sums_up_to_the_last_powers_of_two(at, keys):
    """One row of a query tile outgrows its reference by 118 to 134 powers of two, segment by segment half a power more: sums that the reference is moved by,
    those whose inverse is no normal number any more, and those that overflow.  Values are small, so that it is the sums that do."""
    from trimkv_amd import _lib
    lib = _lib.load()
    H, Q, n, D = 33, 300, 1100, 128
    gen = torch.Generator().manual_seed(keys)
    q, k, v = 0.3 * torch.randn(1, H, Q, D, generator=gen), 0.3 * torch.randn(H, n, D, generator=gen), (torch.rand(H, n, D, generator=gen) - 0.5)
    first = {"first turn": 100, "middle": 600, "end": n - Q + 5 - keys + 1}[at]
    q[..., 0] = k[..., 0] = 0.0
    for t in (5, 256 + 7):                                         # a row of either query tile; the first one sees nothing behind the keys of "end"
        q[0, :, t, 0] = 4.0 * D ** 0.5 / 1.4426950408889634        # 4 powers of two per unit of a key, up to one rounding
    k[:, first:first + keys, 0] = (118 + 0.5 * torch.arange(H))[:, None] / 4
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    c = D ** -0.5 * 1.4426950408889634
    s = torch.einsum("hqd,hnd->hqn", (q[0].float() * c).to(torch.bfloat16).double(), k.double())       # powers of two, as the kernel rounds Q
    p = torch.exp2(s.masked_fill(torch.arange(n)[None, :] > n - Q + torch.arange(Q)[:, None], -float("inf")) - s.amax(-1, keepdim=True))
    want = ((p @ v.double()) / p.sum(-1, keepdim=True)).transpose(0, 1)[None]                          # [1, Q, H, D]
    qd, kd, vd, lens = q.to(DEV), k.to(DEV), v.to(DEV), torch.full((H,), n, dtype=torch.int32, device=DEV)
    bound = 6 * float(v.abs().max()) * 2.0 ** -9                    # as above
    outs = {"in two parts": _whole(qd, kd, vd, lens, 1, H, 1, n, 1 << 20), "in step": _whole(qd, kd, vd, lens, 1, H, 1, n, n)}
    shares = torch.full((1, Q, H, D), float("nan"), dtype=torch.bfloat16, device=DEV)
    need = lib.trimkv_prefill_shares_workspace(1, H, 1, Q)
    work = torch.full((need // 4,), float("nan"), device=DEV)
    _lib.check(lib.trimkv_prefill_attn_shares(qd.data_ptr(), *qd.stride()[:3], shares.data_ptr(), kd.data_ptr(), vd.data_ptr(), lens.data_ptr(), None, 1, H, 1, Q, n, D,
                                              _lib.BF16, D ** -0.5, n, work.data_ptr(), need, _lib.current_stream(qd.device)), "trimkv_prefill_attn_shares")
    outs["shares"] = shares
    for name, out in outs.items():
        far = (out.cpu().double() - want).abs().amax((0, 1, 3))     # of every segment
        assert far.max() <= bound, (name, [118 + 0.5 * i for i in range(H) if not far[i] <= bound], bound)


@pytest.mark.parametrize("at_most", [900, 1 << 20])
@pytest.mark.parametrize("what,value", [("k", float("nan")), ("v", float("inf")), ("q", float("inf"))])
def test_values_that_are_not_finite_stay_with_the_rows_that_see_them(what, value, at_most):
    gen = torch.Generator().manual_seed(1)
    H, G, Q, n = 2, 2, 200, 900
    q, k, v = (torch.randn(1, H * G, Q, 128, generator=gen).to(torch.bfloat16), *(torch.randn(H * n, 128, generator=gen).to(torch.bfloat16) for _ in range(2)))
    lens = torch.full((H,), n, dtype=torch.int32, device=DEV)
    clean = _whole(q.to(DEV), k.to(DEV), v.to(DEV), lens, 1, H, G, n, at_most).cpu()
    {"k": k, "v": v}.get(what, q.view(-1, 128))[5, 7] = value      # row 5 of the first segment, seen by all queries of its heads; or the sixth query of the first head
    out = _whole(q.to(DEV), k.to(DEV), v.to(DEV), lens, 1, H, G, n, at_most).cpu()
    assert torch.equal(out[:, :, G:], clean[:, :, G:])             # the second segment
    hit = out[0, 5, 0] if what == "q" else out[0, :, :G, 7] if what == "v" else out[0, :, :G]
    assert not hit.isfinite().any()
    if what == "v":
        rest = [d for d in range(128) if d != 7]
        assert out[0, :, :G][..., rest].isfinite().all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,G,D,Q,n", [(1, 1, 8, 128, 64, 64), (2, 3, 3, 96, 97, 200), (1, 8, 1, 64, 257, 321), (3, 8, 5, 128, 130, 1025), (1, 2, 4, 128, 400, 300)])
def test_both_kernels_of_whole_query_tiles(B, H, G, D, Q, n, dtype):
    """Little work and much of it, as the bound of the lengths says: the same up to the roundings of P and of the sums."""
    gen = torch.Generator().manual_seed(n)
    q = torch.randn(B, H * G, Q, D, generator=gen).to(dtype).to(DEV)
    k, v = (torch.randn(B * H * n, D, generator=gen).to(dtype).to(DEV) for _ in range(2))
    lens = torch.tensor([max(1, n - 17 * i) for i in range(B * H)], dtype=torch.int32, device=DEV)
    few, two = (_whole(q, k, v, lens, B, H, G, n, at_most).double() for at_most in (n, 1 << 20))
    assert float((few - two).abs().max()) <= 6 * float(v.abs().max()) * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12)


@pytest.mark.parametrize("dtype,n", [(torch.bfloat16, 4000), (torch.float16, 8000)])
def test_query_tiles_for_two_thirds_of_the_chip_are_attended_in_step(dtype, n):
    """160 query tiles of long keys go to the kernel that divided launches have, which is the faster one there: bit for bit what a single share gives."""
    from trimkv_amd import _lib
    H, G, Q, D = 8, 8, 640, 64
    gen = torch.Generator(device=DEV).manual_seed(n)
    q = torch.randn(1, H * G, Q, D, generator=gen, device=DEV).to(dtype)
    k, v = (torch.randn(H * n, D, generator=gen, device=DEV).to(dtype) for _ in range(2))
    lens = torch.full((H,), n, dtype=torch.int32, device=DEV)
    one, lib, share = torch.empty(1, Q, H * G, D, dtype=dtype, device=DEV), _lib.load(), (n + 63) // 64
    need = lib.trimkv_prefill_split_workspace(1, H, G, Q, n, share)
    work = torch.empty(need, dtype=torch.uint8, device=DEV)
    _lib.check(lib.trimkv_prefill_attn_split(q.data_ptr(), *q.stride()[:3], one.data_ptr(), k.data_ptr(), v.data_ptr(), lens.data_ptr(), None, 1, H, G, Q, n, D,
                                             _lib.dtype_code(dtype), D ** -0.5, n, share, work.data_ptr(), need, _lib.current_stream(q.device)), "trimkv_prefill_attn_split")
    assert torch.equal(_whole(q, k, v, lens, 1, H, G, n, n), one)
