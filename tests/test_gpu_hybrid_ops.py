"""The mechanisms of the hybrid decoders one by one against the plain oracle (oracle/hybrid_ref.py), on the GPU."""
import math

import pytest
import torch

from oracle import hybrid_ref as ref
from trimkv_amd import hybrid_ops as ops
from trimkv_amd.hybrid_cache import HybridCache

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def close(got, want, tol, what=""):
    got = got.detach().double().cpu()
    err = (got - want).abs().max().item() / max(want.abs().max().item(), 1e-30)
    assert err <= tol, f"{what}: error {err:.3e} of the largest value, tolerance {tol:.1e}"


def rnd(*shape, seed=0, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [40, 100, 192])
def test_embedding_scale_and_padding(dtype, width):
    table = rnd(50, width, dtype=dtype)
    ids = torch.tensor([3, 0, 49, 3])
    x, xh = ops.embed_scaled(ids.to(DEV), table.to(DEV), 2.75, ops.padded(width))
    close(x[:, :width], table[ids].double() * 2.75, 1e-7)
    assert not x[:, width:].any()
    if dtype == torch.bfloat16:
        assert torch.equal(xh, x.to(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,n,k", [(1, 3, 64), (17, 40, 352), (70, 16, 1024), (2100, 33, 192), (2050, 130, 128)])
def test_linear_keeps_fp32(dtype, rows, n, k):
    x, w = rnd(rows, k, seed=1) * 3.0, rnd(n, k, seed=2, dtype=dtype)
    out = ops.linear_f32(x.to(DEV), w.to(DEV))
    close(out, x.double() @ w.double().T, 2e-6)        # the fp32 input is not rounded to the weights' 16 bits on the way


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,top", [(72, 1), (101, 3), (1536, 1), (4096, 8)])
def test_residual_norm(dtype, width, top):
    T, eps, stride = 5, 1e-3, ops.padded(width)
    x = torch.zeros(T, stride)
    x[:, :width] = rnd(T, width, seed=1)
    y, w = (rnd(T * top, width, seed=2) * 0.05).to(dtype), rnd(width, seed=3)
    wt = torch.rand(T, top, generator=torch.Generator().manual_seed(4)) if top > 1 else None
    summed = y.double().view(T, top, width) * (1.0 if wt is None else wt.double()[:, :, None])
    want = x[:, :width].double() + ref.rms(summed.sum(1), eps) * w.double()
    xd = x.to(DEV)
    xh = torch.empty(T, stride, dtype=dtype, device=DEV) if dtype != torch.float32 else None
    ops.residual_norm(xd, xh, y.to(DEV), w.to(DEV), eps, None if wt is None else wt.to(DEV))
    close(xd[:, :width], want, 1e-6)
    if xh is not None:
        assert torch.equal(xh[:, :width], xd[:, :width].to(dtype))
    rows = torch.tensor([4, 0, 4])
    out = ops.rms_rows(xd, rows.to(DEV), w.to(DEV), eps, dtype)
    close(out, (ref.rms(want, eps) * w.double())[rows], 1e-6 if dtype == torch.float32 else 6e-3)


# ---- windowed attention ------------------------------------------------------------------------------
def run_window(spec, dtype, seqs, cuts, stand_out=()):
    """Projection rows of several sequences through the cache in portions (``cuts``: per sequence a list of portion lengths,
    all sequences advance together); compares everything with the oracle.  ``stand_out``: (sequence, query position, key
    position) whose q and k are made to point the same way, far above all other scores."""
    s, eps = spec, 1e-5
    H, G, D, Dv = s.heads, s.kv_heads, s.dim, s.vdim
    qw, kw = 1 + 0.3 * rnd(H * D, seed=11), 1 + 0.3 * rnd(G * D, seed=12)
    sizes = [H * D, G * D, G * Dv, H * Dv]
    offs = [0, sizes[0], sizes[0] + sizes[1], sum(sizes[:3])]
    rows = [rnd(n, sum(sizes), seed=20 + i) for i, n in enumerate(seqs)]
    for b, qi, kj in stand_out:
        u = rnd(G, D, seed=1000 + kj) * 6.0          # one direction per KV head, shared by its query heads
        rows[b][kj, offs[1]:offs[2]] = u.reshape(-1)
        rows[b][qi, :offs[1]] = u.repeat_interleave(H // G, dim=0).reshape(-1)
    rows = [r.to(dtype) for r in rows]
    want = []
    for r in rows:
        r = r.double()
        q = (ref.rms(r[:, :offs[1]], eps) * qw.double()).view(-1, H, D)
        k = (ref.rms(r[:, offs[1]:offs[2]], eps) * kw.double()).view(-1, G, D)
        if dtype == torch.bfloat16:
            q, k = q.to(dtype).double(), k.to(dtype).double()
        o = ref.window_attention(q, k, r[:, offs[2]:offs[3]].reshape(-1, G, Dv), s.scale, s.window, s.keep_first)
        want.append(o.reshape(-1, H * Dv) * torch.sigmoid(r[:, offs[3]:]))
    cache = HybridCache([spec], dtype, DEV, num_slots=len(seqs) + 1)
    for t in cache.layers_state[0].values():
        t.fill_(float("nan") if dtype == torch.float32 else 7.0)          # whatever a slot held before must not matter
    slots = cache.allocate(len(seqs) + 1)[1:]
    got = [[] for _ in seqs]
    at = [0] * len(seqs)
    for step in range(max(len(c) for c in cuts)):
        live = [b for b in range(len(seqs)) if step < len(cuts[b])]
        lens = [cuts[b][step] for b in live]
        proj = torch.cat([rows[b][at[b]:at[b] + n] for b, n in zip(live, lens)]).to(DEV)
        batch = cache.batch(lens, [slots[b] for b in live])
        out = ops.window_attention(proj, offs, qw.to(DEV), kw.to(DEV), eps, s, cache.layers_state[0], batch)
        cache.advance(batch)
        for b, part in zip(live, out.split(lens)):
            got[b].append(part)
            at[b] += part.shape[0]
    for b, n in enumerate(seqs):
        assert at[b] == n
        close(torch.cat(got[b]), want[b], 3e-6 if dtype == torch.float32 else 1.2e-2, f"sequence {b} of {seqs}, cut {cuts[b][:4]}")


SPECS = {
    "tiny": ops.WindowSpec(3, 1, 8, 16, 5, 2, 0.4),
    "odd": ops.WindowSpec(6, 2, 20, 36, 17, 0, 0.3),
    "one_head_each": ops.WindowSpec(2, 2, 64, 48, 1, 1, 0.125),
    "group_of_eight": ops.WindowSpec(8, 1, 128, 128, 70, 64, 0.09),
    "group_of_twelve": ops.WindowSpec(12, 1, 40, 8, 33, 65, 0.2),
    "wide": ops.WindowSpec(4, 2, 200, 96, 64, 4, 0.07),
    "long_window": ops.WindowSpec(4, 1, 64, 64, 300, 30, 0.15),
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(SPECS))
def test_window_prompts_and_decode(name, dtype):
    s = SPECS[name]
    edge = s.keep_first + s.window
    seqs = [1, edge + 1, 2 * edge + 150, 65]
    run_window(s, dtype, seqs, [[n] for n in seqs])                                        # whole prompts, unequal lengths
    run_window(s, dtype, [7, edge + 12], [[1] * 7, [1] * (edge + 12)])                     # decoding from the first token on
    n = 2 * edge + 40
    run_window(s, dtype, [n, n], [[n - 20] + [1] * 20, [n - 20] + [1] * 20])
    for cut in (2, 3, s.window, edge, 64, 65):
        if n // cut < 120:
            run_window(s, dtype, [n], [[cut] * (n // cut) + ([n % cut] if n % cut else [])])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["tiny", "group_of_eight", "group_of_twelve", "long_window"])
@pytest.mark.parametrize("how", ["prompt", "decode", "portions"])
def test_window_edges_stand_out(name, dtype, how):
    """One query points at one key: the last kept token and the first not kept, the oldest token inside the window and the one
    that has just left it.  A window or a kept prefix that is one token off changes the output completely."""
    s = SPECS[name]
    n = 2 * (s.window + s.keep_first) + 70
    qi = n - 3
    keys = [max(s.keep_first - 1, 0), s.keep_first, qi - s.window + 1, qi - s.window, qi - s.window - 1, qi, 0, 63, 64]
    for kj in sorted(set(k for k in keys if 0 <= k <= qi)):
        cuts = {"prompt": [n], "decode": [n - 6] + [1] * 6, "portions": [50] * ((n - 6) // 50) + [(n - 6) % 50 or 2] + ([6] if (n - 6) % 50 else [4])}[how]
        assert sum(cuts) == n
        run_window(s, dtype, [n], [cuts], stand_out=[(0, qi, kj)])


@pytest.mark.parametrize("spec,seqs,cuts", [
    ((48, 1, 32, 40, 40, 3, 0.2), [150, 33], [[90, 60], [33]]),                  # more heads to a KV head than 32 rows hold
    ((32, 1, 64, 64, 70, 0, 0.1), [131, 64], [[65, 66], [64]]),                  # one time to 32 rows
    ((5, 1, 128, 100, 64, 10, 0.1), [200, 1, 63], [[7, 193], [1], [31, 32]]),    # rows of a workgroup that are nobody's, part of a ring's only tile
    ((2, 2, 36, 128, 200, 64, 0.15), [700], [[300, 200, 200]]),                  # a ring that has gone round
    ((8, 8, 12, 8, 90, 5, 0.3), [577] + [200 - 9 * i for i in range(8)], [[300, 277]] + [[100, 100 - 9 * i] for i in range(8)]),    # 64 rows: many tiles
])
def test_window_fp32_rows_of_a_workgroup(spec, seqs, cuts):
    """32 rows to a workgroup with the keys in two halves, and 64 rows, over rings and portions that end within a tile."""
    run_window(ops.WindowSpec(*spec), torch.float32, seqs, cuts)


@pytest.mark.parametrize("H,G,T", [(4, 2, 200), (48, 1, 130)])
def test_window_fp32_values_that_are_not_finite(H, G, T):
    """An infinite value reaches the rows that see its key and no other, in either half of a tile."""
    s, D = ops.WindowSpec(H, G, 64, 64, 50, 3, 0.1), 64
    offs = [0, H * D, (H + G) * D, (H + 2 * G) * D]
    for at in (70, 110, T - 1):
        proj = rnd(T, offs[3] + H * D, seed=7)
        proj[at, offs[2]] = float("inf")
        cache = HybridCache([s], torch.float32, DEV, num_slots=1)
        batch = cache.batch([T], cache.allocate(1))
        w = torch.ones(H * D, device=DEV)
        out = ops.window_attention(proj.to(DEV), offs, w, w[:G * D], 1e-5, s, cache.layers_state[0], batch).cpu()
        seen = torch.zeros(T, H * D, dtype=torch.bool)
        seen[at:at + 50, [h * D for h in range(H // G)]] = True
        assert torch.equal(~out.isfinite(), seen)


def test_window_sensitivity_of_the_edge_test():
    """The inputs of the edge test tell windows apart: with the key just inside, a window one token shorter moves the output."""
    s = SPECS["tiny"]
    u = rnd(1, 8, seed=5) * 6
    q, k, v = rnd(30, 3, 8, seed=6), rnd(30, 1, 8, seed=7), rnd(30, 1, 16, seed=8)
    k[24 - s.window + 1] = u
    q[24] = u.repeat(3, 1)
    a, b = (ref.window_attention(q, k, v, s.scale, w, s.keep_first)[24] for w in (s.window, s.window - 1))
    assert (a - b).abs().max() > 0.5


# ---- mLSTM ---------------------------------------------------------------------------------------------
def run_mlstm(spec, dtype, seqs, cuts, gate_scale=1.0, f_shift=2.0, tol=None):
    s, eps = spec, 1e-5
    H, D, Dv = s.heads, s.dim, s.vdim
    sizes = [H * D, H * D, H * Dv, H * Dv]
    offs = [0, sizes[0], 2 * sizes[0], sum(sizes[:3])]
    rows = [rnd(n, sum(sizes), seed=30 + i).to(dtype) for i, n in enumerate(seqs)]
    raw = [rnd(n, 2 * H, seed=60 + i) * gate_scale for i, n in enumerate(seqs)]
    ib, fb, w = rnd(H, seed=90), f_shift + rnd(H, seed=91), 1 + 0.3 * rnd(H * Dv, seed=92)
    want = []
    for r, z in zip(rows, raw):
        r, z = r.double(), z.double()
        li = ref.soft_cap(z[:, :H] + ib.double(), s.gate_cap)
        lf = torch.nn.functional.logsigmoid(ref.soft_cap(z[:, H:] + fb.double(), s.gate_cap))
        o, _ = ref.mlstm_scan(r[:, :offs[1]].reshape(-1, H, D) * D ** -0.5, r[:, offs[1]:offs[2]].reshape(-1, H, D), r[:, offs[2]:offs[3]].reshape(-1, H, Dv), li, lf)
        want.append(ref.rms(o, eps).reshape(-1, H * Dv) * w.double() * torch.sigmoid(r[:, offs[3]:]))
    cache = HybridCache([spec], dtype, DEV, num_slots=len(seqs) + 1)
    for t in cache.layers_state[0].values():
        t.fill_(float("nan"))                                   # a fresh sequence starts from zero whatever the slot held
    slots = cache.allocate(len(seqs) + 1)[1:]
    got, at = [[] for _ in seqs], [0] * len(seqs)
    for step in range(max(len(c) for c in cuts)):
        live = [b for b in range(len(seqs)) if step < len(cuts[b])]
        lens = [cuts[b][step] for b in live]
        proj = torch.cat([rows[b][at[b]:at[b] + n] for b, n in zip(live, lens)]).to(DEV)
        gates = torch.cat([raw[b][at[b]:at[b] + n] for b, n in zip(live, lens)]).to(DEV)
        batch = cache.batch(lens, [slots[b] for b in live])
        out = ops.mlstm(proj, offs, gates, ib.to(DEV), fb.to(DEV), w.to(DEV), eps, s, cache.layers_state[0], batch)
        cache.advance(batch)
        for b, part in zip(live, out.split(lens)):
            got[b].append(part)
            at[b] += part.shape[0]
    for b, n in enumerate(seqs):
        assert at[b] == n
        close(torch.cat(got[b]), want[b], tol or (2e-5 if dtype == torch.float32 else 1e-2), f"sequence {b} of {seqs}, cut {cuts[b][:4]}")


MSPECS = {
    "tiny": ops.MlstmSpec(2, 8, 16, 5.0),
    "odd": ops.MlstmSpec(3, 20, 36, 3.0),
    "mid": ops.MlstmSpec(2, 48, 72, 9.0),
    "wide_values": ops.MlstmSpec(1, 64, 200, 12.0),
    "square": ops.MlstmSpec(2, 128, 128, 15.0),
    "large": ops.MlstmSpec(1, 256, 136, 15.0),
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(MSPECS))
def test_mlstm_prompts_portions_and_decode(name, dtype):
    s = MSPECS[name]
    run_mlstm(s, dtype, [1, 64, 65, 200], [[1], [64], [65], [200]])
    run_mlstm(s, dtype, [90, 90], [[70] + [1] * 20] * 2)
    run_mlstm(s, dtype, [40], [[1] * 40])
    for cut in (2, 3, 63, 64, 65):
        run_mlstm(s, dtype, [140, 131], [[cut] * (140 // cut) + ([140 % cut] if 140 % cut else []), [cut] * (131 // cut) + ([131 % cut] if 131 % cut else [])])


@pytest.mark.parametrize("dtype", DTYPES)
def test_mlstm_segments_side_by_side(dtype):
    """Long prompts are cut into segments that run in parallel: segment borders, a sequence that ends inside the first one, a
    state from earlier portions, and decoding behind it."""
    s = ops.MlstmSpec(2, 32, 24, 8.0)
    run_mlstm(s, dtype, [1100, 70, 513], [[1100], [70], [513]], f_shift=5.0)
    run_mlstm(s, dtype, [1400], [[30, 1300] + [1] * 70], f_shift=6.0)
    run_mlstm(s, dtype, [1100], [[512, 580, 8]], f_shift=6.0)


@pytest.mark.parametrize("dtype", DTYPES)
def test_mlstm_segments_of_unequal_sequences(dtype):
    """More sequences than a wavefront has lanes, long ones at either end and among the others, and segments that are shorter than the longest
    sequence by itself would have them."""
    seqs = [900] + [1 + i % 5 for i in range(66)] + [1301, 64, 65, 130]
    run_mlstm(ops.MlstmSpec(1, 32, 24, 8.0), dtype, seqs, [[n] for n in seqs], f_shift=5.0)
    run_mlstm(ops.MlstmSpec(2, 32, 24, 8.0), dtype, [64, 2000, 3, 700], [[60, 4], [1, 1999], [3], [699, 1]], f_shift=5.0)


@pytest.mark.parametrize("H,D,Dv,lens", [(2, 128, 64, [128, 7]), (2, 128, 64, [193, 449, 64]), (3, 20, 68, [700, 320]), (1, 256, 136, [129]), (8, 128, 256, [511, 300])])
def test_mlstm_fp32_segments_against_one_chain(H, D, Dv, lens):
    """fp32 portions of two chunks and from three on, segments of one chunk and of several, the last of them short or missing: the same as the
    one chain that runs without a workspace, also from a state that is there already and with a value that is not finite."""
    from trimkv_amd import _lib
    lib, B, T, width = _lib.load_hybrid("mlstm"), len(lens), sum(lens), 2 * H * D + H * Dv
    need = lib.trimkv_mlstm_workspace(B, max(lens), H, D, Dv, _lib.F32)
    assert (need > 0) == (max(lens) > 2 * (64 if D <= 128 else 32))
    proj, gates, ib, fb = rnd(T, width, seed=1).to(DEV), rnd(T, 2 * H, seed=2).to(DEV), rnd(H, seed=3).to(DEV), (4 + rnd(H, seed=4)).to(DEV)
    bad = lens[0] - 40                                          # of head 0 and sequence 0, in its last segment
    cu = torch.tensor([0] + lens).cumsum(0).int().to(DEV)
    slots = torch.arange(B, 0, -1, dtype=torch.int32, device=DEV)
    seen = torch.tensor([0, 0] + [9, 1] * B, dtype=torch.int32, device=DEV)
    seen[2 * B] = 0                                             # sequence 0 is fresh
    for value in (None, math.inf, math.nan):
        if value is not None:
            proj[bad, 2 * H * D + 3] = value
        got = []
        for floats in (0, need):
            S, nm, o = rnd(B + 1, H, D, Dv, seed=5).to(DEV), rnd(2, B + 1, H, D + 1, seed=6).to(DEV), torch.zeros(T, H, Dv, device=DEV)
            ws = torch.full((floats,), math.nan, device=DEV) if floats else None
            assert lib.trimkv_mlstm(proj.data_ptr(), width, 0, H * D, 2 * H * D, gates.data_ptr(), ib.data_ptr(), fb.data_ptr(), 9.0, S.data_ptr(), nm.data_ptr(),
                                    cu.data_ptr(), slots.data_ptr(), seen.data_ptr(), o.data_ptr(), B, max(lens), H, D, Dv, B + 1, D ** -0.5, _lib.ptr(ws), _lib.F32,
                                    _lib.current_stream(proj.device)) == 0
            got.append((o, S[1:], nm[:, 1:]))
        for one, cut in zip(*got):
            assert torch.equal(one.isfinite(), cut.isfinite())
            one, cut = one.nan_to_num(0, 0, 0).double(), cut.nan_to_num(0, 0, 0).double()
            assert (one - cut).norm() <= 4e-6 * one.norm()      # sums of 2^-24 terms whose order differs, over chunks of 64
        assert value is None or (not got[1][0][bad, 0, 3].isfinite() and got[1][0][:bad].isfinite().all())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lens", [[700, 1500], [3000], [40, 513, 9, 1200]])
def test_mlstm_sequences_longer_than_they_were_said_to_be(lens, dtype):
    """A max_len below the longest sequence costs time only: segments stay within the workspace that it asks for, and no token is left out."""
    from trimkv_amd import _lib
    lib, B, T, H, D, Dv, said = _lib.load_hybrid("mlstm"), len(lens), sum(lens), 2, 64, 128, 512
    width, code = 2 * H * D + H * Dv, _lib.dtype_code(dtype)
    proj, gates, ib, fb = rnd(T, width, seed=1).to(dtype).to(DEV), rnd(T, 2 * H, seed=2).to(DEV), rnd(H, seed=3).to(DEV), (4 + rnd(H, seed=4)).to(DEV)
    cu = torch.tensor([0] + lens).cumsum(0).int().to(DEV)
    slots = torch.arange(B, dtype=torch.int32, device=DEV)
    seen = torch.tensor([9, 1] * B, dtype=torch.int32, device=DEV)
    got = []
    for max_len in (max(lens), said):
        need = lib.trimkv_mlstm_workspace(B, max_len, H, D, Dv, code)
        assert need > 0
        ws = torch.full((4 * need + (1 << 20),), 7.0, device=DEV)
        S, nm, o = rnd(B, H, D, Dv, seed=5).to(DEV), rnd(2, B, H, D + 1, seed=6).to(DEV), torch.zeros(T, H, Dv, dtype=dtype, device=DEV)
        assert lib.trimkv_mlstm(proj.data_ptr(), width, 0, H * D, 2 * H * D, gates.data_ptr(), ib.data_ptr(), fb.data_ptr(), 9.0, S.data_ptr(), nm.data_ptr(),
                                cu.data_ptr(), slots.data_ptr(), seen.data_ptr(), o.data_ptr(), B, max_len, H, D, Dv, B, D ** -0.5, ws.data_ptr(), code,
                                _lib.current_stream(proj.device)) == 0
        assert (ws[need:] == 7.0).all()
        got.append((o, S, nm))
    for right, short in zip(*got):
        assert (right.double() - short.double()).norm() <= (4e-6 if dtype == torch.float32 else 1e-2) * right.double().norm()      # as for segments against one chain; bf16 as above


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["square", "odd", "mid"])
def test_mlstm_sequences_without_tokens_keep_their_state(name, dtype, monkeypatch):
    """A packed step may hold sequences that bring nothing: first, last, or not begun yet; the state they left goes on behind it,
    through chunks and token by token.  (The cache's own ``batch`` does not make such steps; the C entry point takes them.)"""
    def batch(self, lengths, slots):
        cu = torch.tensor([0] + list(lengths)).cumsum(0).int().to(DEV)
        return ops.PackedBatch(tuple(lengths), tuple(slots), cu, torch.tensor(slots, dtype=torch.int32, device=DEV), self.seen, self.num_slots)
    monkeypatch.setattr(HybridCache, "batch", batch)
    run_mlstm(MSPECS[name], dtype, [21, 31, 12, 40], [[9, 0, 1, 11], [0, 20, 0, 11], [12, 0, 0, 0], [30, 0, 0, 10]])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("gate_scale,f_shift", [(30.0, 0.0), (1.0, 12.0), (1.0, -12.0)])
def test_mlstm_extreme_gates(dtype, gate_scale, f_shift):
    """Gates at their caps in both directions, nothing forgotten, everything forgotten: the running maximum carries it."""
    s = ops.MlstmSpec(2, 32, 48, 10.0)
    run_mlstm(s, dtype, [330], [[300] + [1] * 30], gate_scale, f_shift, tol=1e-4 if dtype == torch.float32 else 1e-2)


# ---- routed experts --------------------------------------------------------------------------------------
@pytest.mark.parametrize("E,top,count,keep", [(14, 3, 2, 1), (8, 2, 1, 1), (6, 2, 6, 2), (64, 8, 8, 4), (130, 7, 10, 3), (4, 4, 2, 2), (5, 1, 1, 1)])
def test_router(E, top, count, keep):
    z = rnd(300, E, seed=E) * 2
    for shift in (0.0, -3.0):              # all choice scores negative: a closed group must not win with a zero
        corr = 0.5 * rnd(E, seed=E + 1) + shift
        ids, wt = ops.route(z.to(DEV), corr.to(DEV), ops.RouterSpec(E, top, count, keep))
        want_ids, want_w = ref.choose_experts(z.double(), corr.double(), top, count, keep)
        assert torch.equal(ids.cpu().long(), want_ids)
        close(wt, want_w, 1e-6)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,E,top,ff,width", [(1, 6, 2, 40, 72), (5, 3, 1, 64, 64), (37, 10, 3, 24, 100), (700, 8, 3, 136, 200), (130, 4, 4, 320, 256), (900, 5, 2, 64, 520)])
def test_experts(dtype, T, E, top, ff, width):
    wp, fp = ops.padded(width), ops.padded(ff)
    x = torch.zeros(T, wp)
    x[:, :width] = rnd(T, width, seed=1)
    up, down = torch.zeros(E, fp, wp), torch.zeros(E, wp, fp)
    up[:, :ff, :width] = rnd(E, ff, width, seed=2) * width ** -0.5
    down[:, :width, :ff] = rnd(E, width, ff, seed=3) * ff ** -0.5
    x, up, down = x.to(dtype), up.to(dtype), down.to(dtype)
    gen = torch.Generator().manual_seed(4)
    ids = torch.stack([torch.randperm(E, generator=gen)[:top] for _ in range(T)]).int()
    if E > 4:
        ids[ids == 2] = 0 if top == 1 else ids[ids == 2]          # an expert nobody asks for
    y = ops.experts(x.to(DEV), ids.to(DEV), ops.pack_matrix(up).contiguous().to(DEV), ops.pack_matrix(down).contiguous().to(DEV), width).view(T, top, width)
    want = torch.stack([torch.stack([ref.expert(x[t].double()[:width], up[e].double()[:ff, :width], down[e].double()[:width, :ff]) for e in ids[t].tolist()]) for t in range(T)])
    close(y, want, 2e-6 if dtype == torch.float32 else 1.2e-2)


def test_experts_with_row_counts_at_the_edges_of_tiles():
    """Prompt-sized products (row tiles of 256, blocks of 32 of which only those with rows are multiplied): experts with no row, one
    row, one short of a block or a tile, exactly one, one more, and both kinds of tiles at once."""
    counts = [0, 1, 31, 32, 33, 255, 256, 257, 512, 545]
    E, top, ff, width, T = len(counts), 1, 64, 64, sum(counts)
    assert T >= 96 * E
    x = rnd(T, width, seed=1, dtype=torch.bfloat16)
    up, down = (rnd(E, ff, width, seed=2) * width ** -0.5).to(torch.bfloat16), (rnd(E, width, ff, seed=3) * ff ** -0.5).to(torch.bfloat16)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=torch.Generator().manual_seed(4))]
    y = ops.experts(x.to(DEV), ids[:, None].int().to(DEV), ops.pack_matrix(up).contiguous().to(DEV), ops.pack_matrix(down).contiguous().to(DEV), width)
    want = torch.empty(T, width, dtype=torch.float64)
    for e in range(E):
        want[ids == e] = ref.expert(x[ids == e].double(), up[e].double(), down[e].double())
    close(y, want, 1.2e-2)      # hidden values and outputs rounded to bf16 once each: 2^-8 of the largest each, and slack for their spread


@pytest.mark.parametrize("ff,width", [(64, 64), (128, 192), (192, 320), (576, 256), (264, 520)])
def test_experts_of_either_tile_height(ff, width):
    """Products of one, two, three and more steps of 64 k, outputs that end in the first or the second half of a tile, and tiles of
    256 and of 128 rows on either side of the line between them."""
    counts = [300, 1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 384, 385, 640, 0, 17]
    E, T, wp, fp = len(counts), sum(counts), ops.padded(width), ops.padded(ff)
    assert T >= 12 * E and T >= 1200
    x, up, down = torch.zeros(T, wp), torch.zeros(E, fp, wp), torch.zeros(E, wp, fp)
    x[:, :width] = rnd(T, width, seed=1)
    up[:, :ff, :width] = rnd(E, ff, width, seed=2) * width ** -0.5
    down[:, :width, :ff] = rnd(E, width, ff, seed=3) * ff ** -0.5
    x, up, down = (t.to(torch.bfloat16) for t in (x, up, down))
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=torch.Generator().manual_seed(4))]
    y = ops.experts(x.to(DEV), ids[:, None].int().to(DEV), ops.pack_matrix(up).contiguous().to(DEV), ops.pack_matrix(down).contiguous().to(DEV), width)
    want = torch.empty(T, width, dtype=torch.float64)
    for e in range(E):
        want[ids == e] = ref.expert(x[ids == e].double()[:, :width], up[e].double()[:ff, :width], down[e].double()[:width, :ff])
    close(y[:, :width], want, 1.2e-2)      # hidden values and outputs rounded to bf16 once each, as above


@pytest.mark.parametrize("rows,E,tile", [(2048, 5, 32), (2049, 5, 32), (10007, 300, 256), (32767, 64, 256), (33001, 1, 256), (70001, 1024, 16)])
def test_plan_by_several_workgroups(rows, E, tile):
    """Rows just within and beyond a workgroup's, in chunks that end within a round of loads, and more chunks than workgroups."""
    from trimkv_amd import _lib
    ids = torch.randint(0, E, (rows,), generator=torch.Generator().manual_seed(rows)).int()
    ids[ids == E // 2] = 0                                  # an expert without rows, unless it is the only one
    most, dev_ids = (rows - E) // tile + E, ids.to(DEV)
    order, offsets, tiles = (torch.full((n,), -1, dtype=torch.int32, device=DEV) for n in (rows, E + 1, 1 + 2 * most))
    assert _lib.load_hybrid("moe").trimkv_moe_plan(dev_ids.data_ptr(), rows, E, tile, order.data_ptr(), offsets.data_ptr(), tiles.data_ptr(),
                                                   _lib.current_stream(dev_ids.device)) == 0
    counts = torch.bincount(ids.long(), minlength=E)
    order, offsets, tiles = order.cpu().long(), offsets.cpu().long(), tiles.cpu().tolist()
    assert torch.equal(order.sort().values, torch.arange(rows)) and torch.equal(offsets.diff(), counts) and offsets[0] == 0
    assert torch.equal(ids[order].long(), torch.repeat_interleave(torch.arange(E), counts))
    want = [v for e in range(E) for r in range(0, int(counts[e]), tile) for v in (e, int(offsets[e]) + r)]
    assert tiles[0] == len(want) // 2 and tiles[1:1 + len(want)] == want


@pytest.mark.parametrize("E,ff,width", [(1, 2560, 64), (64, 64, 576), (65, 320, 64), (150, 64, 320)])
def test_experts_cut_into_runs(E, ff, width):
    """As many experts as a wavefront has lanes, more of them and a single one, most of them with a few rows or none beside some with
    several tiles: runs of tiles that begin within an expert and between two, and more workgroups than tiles."""
    counts = [0 if e % 7 == 3 else 1 + (e * 37) % 40 if e % 11 else 1300 + 90 * (e % 5) for e in range(E)]
    T = sum(counts)
    assert T >= 12 * E and T >= 1200
    x = rnd(T, ops.padded(width), seed=1, dtype=torch.bfloat16)
    up, down = torch.zeros(E, ops.padded(ff), ops.padded(width)), torch.zeros(E, ops.padded(width), ops.padded(ff))
    up[:, :ff, :width] = rnd(E, ff, width, seed=2) * width ** -0.5
    down[:, :width, :ff] = rnd(E, width, ff, seed=3) * ff ** -0.5
    up, down = up.to(torch.bfloat16), down.to(torch.bfloat16)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=torch.Generator().manual_seed(4))]
    y = ops.experts(x.to(DEV), ids[:, None].int().to(DEV), ops.pack_matrix(up).contiguous().to(DEV), ops.pack_matrix(down).contiguous().to(DEV), width)
    want = torch.empty(T, width, dtype=torch.float64)
    for e in range(E):
        want[ids == e] = ref.expert(x[ids == e].double(), up[e].double(), down[e].double())[:, :width]
    close(y, want, 1.2e-2)      # hidden values and outputs rounded to bf16 once each, as above


@pytest.mark.parametrize("ff,width", [(352, 640), (704, 352)])
def test_experts_whose_steps_go_round_the_buffers(ff, width):
    """Prompt-sized products of 6, 10 and 11 steps of 64 k: the operand buffers, two of them for tiles of 256 and 192 rows and three for tiles of 128, are
    filled anew two to five times, with an even and an odd number of steps, in full tiles and in ones that hold any part of their rows."""
    counts = [0, 1, 33, 65, 97, 129, 161, 193, 225, 256, 257, 545]
    E, T, wp, fp = len(counts), sum(counts), ops.padded(width), ops.padded(ff)
    assert T >= 96 * E and {wp // 64, fp // 64} in ({10, 6}, {6, 11})
    x, up, down = torch.zeros(T, wp), torch.zeros(E, fp, wp), torch.zeros(E, wp, fp)
    x[:, :width] = rnd(T, width, seed=1)
    up[:, :ff, :width] = rnd(E, ff, width, seed=2) * width ** -0.5
    down[:, :width, :ff] = rnd(E, width, ff, seed=3) * ff ** -0.5
    x, up, down = (t.to(torch.bfloat16) for t in (x, up, down))
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=torch.Generator().manual_seed(4))]
    want = torch.empty(T, width, dtype=torch.float64)
    for e in range(E):
        want[ids == e] = ref.expert(x[ids == e].double()[:, :width], up[e].double()[:ff, :width], down[e].double()[:width, :ff])
    args = (x.to(DEV), ids[:, None].int().to(DEV), ops.pack_matrix(up).contiguous().to(DEV), ops.pack_matrix(down).contiguous().to(DEV), width)
    first = ops.experts(*args)
    close(first[:, :width], want, 1.2e-2)      # hidden values and outputs rounded to bf16 once each: 2^-8 of the largest each, and slack for their spread
    assert all(torch.equal(ops.experts(*args), first) for _ in range(3))     # a buffer read too early or too late does not repeat itself


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("at", [3, 37, 64, 129])
def test_values_that_are_not_finite_stay_out_of_rows_that_do_not_see_them(bad, at):
    """fp32 prompts take tiles of keys (and chunks of tokens) at a time: a value that is masked for a row is multiplied by zero
    there and must not turn the row into NaN.  Rows in front of the token are as if it were harmless; in the window's case
    those behind it, too."""
    n, s, m = 150, ops.WindowSpec(4, 2, 24, 40, 20, 3, 0.3), ops.MlstmSpec(2, 40, 72, 9.0)
    outs = []
    for value in (1.0, bad):
        sizes = [s.heads * s.dim, s.kv_heads * s.dim, s.kv_heads * s.vdim, s.heads * s.vdim]
        offs = [0, sizes[0], sum(sizes[:2]), sum(sizes[:3])]
        proj = rnd(n, sum(sizes), seed=1)
        proj[at, offs[2]] = value
        cache = HybridCache([s], torch.float32, DEV, num_slots=1)
        batch = cache.batch([n], cache.allocate(1))
        ones = [torch.ones(k, device=DEV) for k in sizes[:2]]
        a = ops.window_attention(proj.to(DEV), offs, *ones, 1e-5, s, cache.layers_state[0], batch)
        sizes = [m.heads * m.dim] * 2 + [m.heads * m.vdim] * 2
        offs = [0, sizes[0], sum(sizes[:2]), sum(sizes[:3])]
        proj = rnd(n, sum(sizes), seed=2)
        proj[at, offs[2]] = value
        cache = HybridCache([m], torch.float32, DEV, num_slots=1)
        batch = cache.batch([n], cache.allocate(1))
        gates, z = rnd(n, 2 * m.heads, seed=3).to(DEV), torch.zeros(m.heads, device=DEV)
        r = ops.mlstm(proj.to(DEV), offs, gates, z, z + 3, torch.ones(m.heads * m.vdim, device=DEV), 1e-5, m, cache.layers_state[0], batch)
        outs.append((a.cpu(), r.cpu()))
    (a, r), (ab, rb) = outs
    sees = torch.tensor([t >= at and (t - at < s.window or at < s.keep_first) for t in range(n)])
    assert (ab[~sees] - a[~sees]).abs().max() <= 1e-6        # the same sums in the same or another order of 64 keys at most
    assert not ab[sees][:, 0].isfinite().any()
    assert (rb[:at] - r[:at]).abs().max() <= 1e-5
    assert not rb[at:, 0].isfinite().any()


@pytest.mark.parametrize("heads,kv_heads,seqs", [
    (4, 2, [1, 130, 2, 16, 15, 17, 129, 3]),                                          # 32 rows to a workgroup, one tile and several
    (4, 1, [700, 5, 1, 699, 8, 9]),                                                   # more tiles than a wavefront has lanes
    (4, 2, [300] + [1 + i % 5 for i in range(62)] + [299, 64, 65, 1, 40, 33] * 2),    # more sequences than lanes; 64 rows
    (2, 2, [1] * 64), (2, 2, [33] * 65),
])
def test_window_fp32_prompts_of_unequal_lengths(heads, kv_heads, seqs):
    """Workgroups find their tile among those that are there, the last ones of all sequences first: every tile of every sequence is done, once."""
    run_window(ops.WindowSpec(heads, kv_heads, 24, 40, 50, 3, 0.3), torch.float32, seqs, [[n] for n in seqs])
    run_window(ops.WindowSpec(heads, kv_heads, 24, 40, 50, 3, 0.3), torch.float32, seqs, [[n // 3] * 2 + [n - 2 * (n // 3)] if n > 8 else [n] for n in seqs])


@pytest.mark.parametrize("dtype", DTYPES)
def test_decode_of_sequences_with_fewer_rows_than_the_batch_is_split_for(dtype):
    """A window of 1520 rows is split over twelve workgroups (127 rows each): sequences that fill one row, one share, one share and a
    row, some, and all of them, decoded side by side."""
    spec = ops.WindowSpec(2, 1, 64, 64, 1500, 20, 0.15)
    run_window(spec, dtype, [4, 128, 129, 400, 1600], [[1] * 4, [125, 1, 1, 1], [126, 1, 1, 1], [397, 1, 1, 1], [1597, 1, 1, 1]])


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(2, 1, 128, 128), (6, 2, 72, 100), (4, 1, 100, 128), (8, 2, 128, 72), (5, 1, 128, 128), (16, 2, 96, 96), (12, 1, 128, 120), (1, 1, 128, 128)])
def test_decode_rows_of_sixteen_lanes_shared_by_heads(heads, kv_heads, dim, vdim):
    """In bf16 a step's products of 2, 4 or 8 heads and 8, 4 or 2 rows for each four are summed together: fewer rows than a step has, one row more, several shares; heads
    that are not there; head sizes that leave lanes without features."""
    seqs = [3, 17, 34, 65, 131, 420]
    run_window(ops.WindowSpec(heads, kv_heads, dim, vdim, 290, 11, 0.13), torch.bfloat16, seqs, [[n - 3] + [1] * 3 if n > 3 else [1] * 3 for n in seqs])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,n,k", [(1, 1, 32), (3, 7, 4128), (64, 32, 4096), (64, 33, 2080), (512, 16, 64), (513, 16, 2048), (128, 16, 260), (129, 16, 4)])
def test_linear_f32_on_either_side_of_its_rules(dtype, rows, n, k):
    """Rows of a decode step and more: fp32 sums of k exact products (bf16 weights) or fp32 ones, in any order."""
    gen = torch.Generator(device=DEV).manual_seed(rows + n + k)
    ks = (k + 7) // 8 * 8
    x, w = torch.randn(rows, k + 4, generator=gen, device=DEV), torch.randn(n, ks, generator=gen, device=DEV).to(dtype)[:, :k]
    out = ops.linear_f32(x[:, :k], w)
    exact, size = x[:, :k].double() @ w.double().T, x[:, :k].double().abs() @ w.double().abs().T
    assert ((out.double() - exact).abs() <= (k + 2) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("rows,n,k", [(2047, 33, 64), (2048, 33, 96), (2049, 16, 288), (3071, 17, 96), (3072, 17, 128), (5000, 16, 32), (4097, 64, 160)])
def test_linear_f32_of_prompts(rows, n, k):
    """Either side of the rules between the two divisions of a prompt's rows."""
    test_linear_f32_on_either_side_of_its_rules(torch.bfloat16, rows, n, k)


@pytest.mark.parametrize("rows,n,k", [(4096, 16, 96), (4097, 16, 96), (4100, 5, 32), (2048, 32, 64), (2049, 32, 160), (2050, 17, 32)])
def test_linear_f32_of_more_workgroups_than_compute_units(rows, n, k):
    """Sixteen wavefronts to a workgroup up to 256 of them, four beyond."""
    test_linear_f32_on_either_side_of_its_rules(torch.bfloat16, rows, n, k)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [4, 30, 1028, 2048, 2052, 4096, 4100])
def test_rms_rows_of_every_width(dtype, width):
    gen = torch.Generator(device=DEV).manual_seed(width)
    x, w = torch.randn(9, (width + 67) // 4 * 4, generator=gen, device=DEV) * 3, torch.randn(width, generator=gen, device=DEV)
    rows = torch.tensor([8, 0, 3], device=DEV)
    for r in (None, rows):
        out = ops.rms_rows(x[:, :width] if r is None else x[:, :width], r, w, 1e-6, dtype)
        src = x[:, :width].double() if r is None else x[rows, :width].double()
        want = src * torch.rsqrt(src.square().mean(-1, keepdim=True) + 1e-6) * w.double()
        assert ((out.double() - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20) * want.abs() + 1e-30).all()
