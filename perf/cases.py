"""What the framework is timed on: the work its users have it do, through the entry points they call.

Kinds of work and what each stands for:

* ``decode``   one eviction cycle of token steps over a dense cache: per token and layer ``update`` (append deferred to the
               attention), attention, then ``compress``, which evicts once, at the cycle's last token
* ``ragged``   token steps over a cache with a budget of its own per head, whose heads are cut back as they come due
* ``chunk``    a portion of a long prompt against a dense cache: append, causal attention, eviction back to the budget
* ``shared``   the same against the flat cache whose heads (of one layer, or of all) share a budget
* ``qwen3``    one token step of the whole Qwen3 decoder with its retention gate, replayed from a HIP graph
* ``siterax``, ``fusitar``   prompts of unequal length, or one replayed token step, of the two hybrid decoders
* ``experts``  the routed feed-forward of the hybrid decoders, for prompts and for token steps

Sizes are those of ``bench.py`` and of the decoders' default configurations (Qwen3-1.7B/4B/8B/14B and Phi-3-mini layers, the
two hybrid sizes), with fewer layers where a layer is like the next.  Everything is synthetic and made on the GPU.
"""
import math
from types import SimpleNamespace

import torch

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# width, attention heads / KV heads (of 128 features), window, kept first tokens, mLSTM heads (128 x 256), expert size; 32 experts, 4 chosen
HYBRID = {"8b": dict(W=4096, Hq=32, Hkv=8, window=4032, keep=64, mh=16, ff=4608), "1.7b": dict(W=2048, Hq=16, Hkv=8, window=1984, keep=64, mh=8, ff=2304)}
QWEN3 = {"8b": dict(W=4096, ff=12288, Hq=32), "1.7b": dict(W=2048, ff=6144, Hq=16)}
VOCAB = 1024
EXPERTS, CHOSEN, GROUPS, OPEN = 32, 4, 4, 2


def listed():
    return [
        # one conversation on a small model (Phi-3-mini heads, fp16): the shortest launches there are, bound by latency
        {"name": "decode_phi3_b1", "kind": "decode", "layers": 4, "batch": 1, "kv_heads": 32, "group": 1, "dim": 96, "memory": 512, "buffer": 32, "dtype": "fp16"},
        # the headline: a served batch at the Qwen3-8B layer shape, four layers of it
        {"name": "decode_8b_b64", "kind": "decode", "layers": 4, "batch": 64, "kv_heads": 8, "group": 4, "dim": 128, "memory": 4096, "buffer": 128, "dtype": "bf16"},
        # lognormal budgets per head at the Qwen3-4B layer shape: heads of very different length in one launch, evicted one by one
        {"name": "ragged_4b_b32", "kind": "ragged", "layers": 6, "batch": 32, "kv_heads": 8, "group": 4, "dim": 128, "median": 1024, "most": 8192, "buffer": 128, "tokens": 32},
        # a served batch of the smallest Qwen3 with its gate, half of its layers, one replayed token step
        {"name": "qwen3_step_1.7b_b16", "kind": "qwen3", "size": "1.7b", "layers": 14, "batch": 16, "memory": 2048, "buffer": 128},
        # a long prompt read in portions at the Qwen3-14B layer shape: matrix-bound attention, then eviction of a third of the rows
        {"name": "chunk_14b", "kind": "chunk", "layers": 2, "batch": 2, "kv_heads": 8, "group": 5, "dim": 128, "memory": 8192, "buffer": 512, "chunk": 4096, "dtype": "bf16"},
        # three prompts read in odd portions, one budget over all heads and layers of a sequence
        {"name": "shared_1.7b_b3", "kind": "shared", "layers": 8, "batch": 3, "kv_heads": 8, "group": 2, "dim": 128, "memory": 2048, "buffer": 128, "chunk": 777, "strategy": "alpha"},
        # a long prompt through rotary windowed attention and dense feed-forwards, one layer passed twice
        {"name": "siterax_prompt_8b", "kind": "siterax", "size": "8b", "mode": "prompt", "layers": 2, "lengths": "8192", "dtype": "bf16"},
        # prompts of unequal length through recurrent and windowed layers
        {"name": "fusitar_prompts_1.7b", "kind": "fusitar", "size": "1.7b", "mode": "prompt", "layers": 2, "lengths": "701,3999,1536,2050", "dtype": "bf16"},
        # a served batch of conversations of unequal length, one replayed token step
        {"name": "fusitar_step_8b_b64", "kind": "fusitar", "size": "8b", "mode": "step", "layers": 2, "batch": 64, "longest": 4096, "dtype": "bf16"},
        # what a trace is checked with: everything in fp32, short prompts
        {"name": "fusitar_fp32_1.7b", "kind": "fusitar", "size": "1.7b", "mode": "prompt", "layers": 2, "lengths": "300,511", "dtype": "fp32"},
        # routed experts under a long prompt (matrix-bound) and under a token step (weights streamed once)
        {"name": "experts_prompt_8b", "kind": "experts", "size": "8b", "tokens": 8192},
        {"name": "experts_step_8b", "kind": "experts", "size": "8b", "tokens": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(["decode", "decode", "ragged", "chunk", "chunk", "shared", "qwen3", "siterax", "siterax", "fusitar", "fusitar", "experts", "experts"])
    if kind in ("decode", "chunk"):
        kv, g, d = rng.choice([(8, 2, 128), (8, 4, 128), (8, 5, 128), (8, 8, 128), (32, 1, 96), (8, 4, 64)])
        case = {"kind": kind, "layers": rng.randint(1, 4), "batch": _log(rng, 1, 64 if kind == "decode" else 4), "kv_heads": kv, "group": g, "dim": d,
                "memory": _log(rng, 256, 8192), "buffer": _log(rng, 16, 128), "dtype": rng.choice(["bf16", "bf16", "fp16"])}
        if kind == "chunk":
            case["chunk"] = case["buffer"] + _log(rng, 33, 4096)
        return case
    if kind == "ragged":
        return {"kind": kind, "layers": rng.randint(2, 6), "batch": _log(rng, 1, 32), "kv_heads": 8, "group": rng.choice([2, 4, 5, 8]), "dim": 128,
                "median": _log(rng, 200, 1024), "most": 8192, "buffer": _log(rng, 32, 128), "tokens": _log(rng, 8, 32)}
    if kind == "shared":
        buffer = _log(rng, 32, 128)
        return {"kind": kind, "layers": rng.randint(2, 8), "batch": rng.randint(1, 4), "kv_heads": 8, "group": rng.choice([2, 4]), "dim": 128, "memory": _log(rng, 256, 4096),
                "buffer": buffer, "chunk": buffer + _log(rng, 33, 2048), "strategy": rng.choice(["alpha", "layer_wise_alpha"])}
    if kind == "qwen3":
        return {"kind": kind, "size": rng.choice(["1.7b", "8b"]), "layers": rng.randint(4, 12), "batch": _log(rng, 1, 64), "memory": _log(rng, 256, 4096), "buffer": 128}
    if kind == "experts":
        return {"kind": kind, "size": rng.choice(["1.7b", "8b"]), "tokens": _log(rng, 1, 8192)}
    size = rng.choice(["1.7b", "8b"])
    if rng.random() < 0.4:
        return {"kind": kind, "size": size, "mode": "step", "layers": 2, "batch": _log(rng, 1, 64), "longest": _log(rng, 64, 4096), "dtype": "bf16"}
    if rng.random() < 0.2:
        return {"kind": kind, "size": "1.7b", "mode": "prompt", "layers": 2, "lengths": ",".join(str(_log(rng, 16, 600)) for _ in range(rng.randint(1, 3))), "dtype": "fp32"}
    return {"kind": kind, "size": size, "mode": "prompt", "layers": 2, "lengths": ",".join(str(_log(rng, 16, 6000)) for _ in range(rng.randint(1, 5))), "dtype": "bf16"}


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 6e12, w["flops"] / 1e15)


def draw(rng):
    most = max(_cost(c) for c in listed() if c["kind"] != "decode")
    while True:
        case = _draw_once(rng)
        if _cost(case) <= most:
            return case


def work(case):
    return KINDS[case["kind"]].work(case)


def prepare(case, seed):
    with torch.no_grad():
        return KINDS[case["kind"]].prepare(case, seed)


def run(state):
    with torch.no_grad():
        return state["run"](state)


def exact(case, seed):
    with torch.no_grad():
        return KINDS[case["kind"]].exact(case, seed)


def tolerance(case):
    return KINDS[case["kind"]].tolerance(case)


# ---- the caches ------------------------------------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + 17)


def _kv(case, gen, rows, dt):
    """Keys, values and log beta of ``rows`` tokens of one layer, as a decoder's projections and its gate give them."""
    shape = (case["batch"], case["kv_heads"], rows, case["dim"])
    k, v = (torch.randn(shape, generator=gen, device=DEV, dtype=dt) for _ in range(2))
    return k, v, torch.nn.functional.logsigmoid(torch.randn(shape[:3], generator=gen, device=DEV) * 1.5 + 3.0)


def _q(case, gen, rows, dt):
    return torch.randn(case["batch"], case["kv_heads"] * case["group"], rows, case["dim"], generator=gen, device=DEV, dtype=dt)


def _module(case):
    """What an attention interface looks at of the module that calls it."""
    return SimpleNamespace(training=False, num_key_value_groups=case["group"], is_causal=True)


def _scores(lb, pos, query):
    """Retention scores as the design defines them: the fp32 product of log beta and age."""
    return lb.float() * (query - pos)


def _best(score, keep):
    """Mask of the ``keep`` largest along the last axis (an int or one per row); among equals the earlier ones."""
    rank = torch.empty_like(score, dtype=torch.int64)
    rank.scatter_(-1, score.sort(dim=-1, descending=True, stable=True).indices, torch.arange(score.shape[-1], device=score.device).expand_as(rank))
    return rank < (keep if isinstance(keep, int) else keep.unsqueeze(-1))


def _attend64(q, k, v, visible):
    """q [N, G, R, D], k and v [N, M, D], visible broadcastable to [N, G, R, M] -> [N, G, R, D] in 64 bits, a few N at a time."""
    N, G, R, D = q.shape
    out = torch.empty(N, G, R, D, dtype=torch.float64, device=q.device)
    step = max(1, int(2e8 // (G * R * k.shape[1])))
    for n in range(0, N, step):
        s = slice(n, n + step)
        score = torch.matmul(q[s].double().reshape(-1, G * R, D), k[s].double().transpose(1, 2).contiguous()).view(-1, G, R, k.shape[1]) * D ** -0.5
        score.masked_fill_(~(visible[s] if visible.shape[0] == N else visible), -math.inf)
        out[s] = torch.matmul(torch.softmax(score, -1).view(-1, G * R, k.shape[1]), v[s].double()).view(-1, G, R, D)
    return out


def _dense_prompt_rows(case):
    return case["memory"] + case["memory"] // 4 + case["buffer"]


def _dense_inputs(case, seed, tokens, portions):
    """Per layer the rows a long prompt left and, for each of ``portions``, ``tokens`` new rows with their queries."""
    gen, dt = _gen(seed), DTYPES[case["dtype"]]
    for _ in range(case["layers"]):
        yield _kv(case, gen, _dense_prompt_rows(case), dt), [(*_kv(case, gen, tokens, dt), _q(case, gen, tokens, dt)) for _ in range(portions)]


def _dense_prepare(case, seed, tokens, portions):
    from trimkv_amd import TrimKVCache, get_attention_interface
    cache, P = TrimKVCache(), _dense_prompt_rows(case)
    cache.fuse_decode_append = True
    new = [[None] * case["layers"] for _ in range(portions)]
    for l, (prompt, parts) in enumerate(_dense_inputs(case, seed, tokens, portions)):
        cache.update(*prompt, torch.arange(P, device=DEV), l)
        for t, part in enumerate(parts):
            new[t][l] = part
    cache.compress("alpha", memory_size=case["memory"], buffer_size=case["buffer"])
    return {"cache": cache, "attend": get_attention_interface("trimkv_hip"), "module": _module(case), "new": new, "tokens": tokens, "memory": case["memory"], "buffer": case["buffer"],
            "layers": case["layers"], "scale": case["dim"] ** -0.5, "run": _dense_run}


def _dense_run(s):
    cache, outs = s["cache"], [[] for _ in range(s["layers"])]
    for portion in s["new"]:
        seen = cache.get_seq_length()
        positions = torch.arange(seen, seen + s["tokens"], device=DEV)
        for l, (k, v, lb, q) in enumerate(portion):
            keys, values, _, _, kw = cache.update(k, v, lb, positions, l)
            outs[l].append(s["attend"](s["module"], q, keys, values, None, scaling=s["scale"], flash_attn_kwargs=kw)[0])
        cache.compress("alpha", memory_size=s["memory"], buffer_size=s["buffer"])
    return {"out": [torch.cat(o, dim=1) for o in outs], "k": list(cache.key_cache), "v": list(cache.value_cache), "log_beta": list(cache.retention_weights),
            "pos": list(cache.kv_positions)}


def _dense_exact(case, seed, tokens, portions):
    """All portions of a pass at once: nothing is evicted before the last of them."""
    P, M, B, H, G, D, S = _dense_prompt_rows(case), case["memory"], case["batch"], case["kv_heads"], case["group"], case["dim"], tokens * portions
    res = {"out": [], "k": [], "v": [], "log_beta": [], "pos": []}
    for (k, v, lb), parts in _dense_inputs(case, seed, tokens, portions):
        pos = torch.arange(P, device=DEV).expand(B, H, P)
        kept = _best(_scores(lb, pos, P + 1), M).nonzero()[:, 2].view(B, H, M)
        pick = lambda t, at: torch.gather(t, 2, at) if t.dim() == 3 else torch.gather(t, 2, at.unsqueeze(-1).expand(*at.shape, D))
        k, v, lb = (torch.cat([pick(t, kept)] + [part[i] for part in parts], dim=2) for i, t in enumerate((k, v, lb)))
        pos = torch.cat([kept, torch.arange(P, P + S, device=DEV).expand(B, H, S)], dim=2)
        q = torch.cat([part[3] for part in parts], dim=2).view(B * H, G, S, D)
        visible = torch.arange(M + S, device=DEV)[None, :] <= (M + torch.arange(S, device=DEV))[:, None]
        out = _attend64(q, k.view(B * H, M + S, D), v.view(B * H, M + S, D), visible[None, None])
        res["out"].append(out.view(B, H * G, S, D).transpose(1, 2).contiguous())
        last = _best(_scores(lb, pos, P + S + 1), M).nonzero()[:, 2].view(B, H, M)
        for name, t in (("k", k), ("v", v), ("log_beta", lb), ("pos", pos)):
            res[name].append(pick(t, last))
    return res


def _evict_bytes(segments, rows, kept, dim):
    """An eviction reads the score inputs of the rows there are and moves the kept rows with their metadata."""
    return segments * (12.0 * rows + 2 * 12.0 * kept + 2 * 2.0 * kept * dim * 2)


def _attention_tolerance(case):
    """Four times what the rounding of probabilities and outputs leaves (measured: 2.2e-3 to 2.9e-3 in bf16, an eighth of it in fp16)."""
    return {"rel": 1.5e-3, "max": 1.5e-2} if case.get("dtype") == "fp16" else {"rel": 1.2e-2, "max": 0.12}


class Decode:
    @staticmethod
    def prepare(case, seed):
        return _dense_prepare(case, seed, 1, case["buffer"])

    @staticmethod
    def exact(case, seed):
        return _dense_exact(case, seed, 1, case["buffer"])

    @staticmethod
    def work(case):
        n, T, M, G, D = case["batch"] * case["kv_heads"], case["buffer"], case["memory"], case["group"], case["dim"]
        rows = T * M + T * (T + 1) / 2
        return {"bytes": case["layers"] * (n * (rows * 4.0 * D + T * (4.0 * G * D + 8.0 * D + 24)) + _evict_bytes(n, M + T, M, D)),
                "flops": case["layers"] * 4.0 * n * G * D * rows}

    @staticmethod
    def tolerance(case):
        return _attention_tolerance(case)


class Chunk:
    @staticmethod
    def prepare(case, seed):
        return _dense_prepare(case, seed, case["chunk"], 1)

    @staticmethod
    def exact(case, seed):
        return _dense_exact(case, seed, case["chunk"], 1)

    @staticmethod
    def work(case):
        n, S, M, G, D = case["batch"] * case["kv_heads"], case["chunk"], case["memory"], case["group"], case["dim"]
        return {"bytes": case["layers"] * (n * ((M + S) * 4.0 * D + S * (4.0 * G * D + 8.0 * D + 24)) + _evict_bytes(n, M + S, M, D)),
                "flops": case["layers"] * 4.0 * n * G * D * (S * M + S * (S + 1) / 2.0)}

    @staticmethod
    def tolerance(case):
        return _attention_tolerance(case)


class Ragged:
    """Token steps with a budget per head.  Every head starts somewhere in its own cycle, so a few come due at every step."""

    @staticmethod
    def _sizes(case):
        """Budgets and starting lengths [layers, heads of all sequences]: the same for every seed, as they decide the work."""
        gen = torch.Generator().manual_seed(case["layers"] * 101 + case["batch"])
        shape = (case["layers"], case["batch"] * case["kv_heads"])
        budgets = torch.exp(math.log(case["median"]) + torch.randn(shape, generator=gen)).round().clamp(64, case["most"]).long()
        return budgets, budgets + torch.randint(0, case["buffer"], shape, generator=gen)

    @staticmethod
    def _inputs(case, seed, rows):
        gen, dt = _gen(seed), torch.bfloat16
        for _ in range(case["layers"]):
            yield _kv(case, gen, rows, dt), [(*_kv(case, gen, 1, dt), _q(case, gen, 1, dt)) for _ in range(case["tokens"])]

    @classmethod
    def prepare(cls, case, seed):
        from trimkv_amd import BatchedDynamicBudgetTrimKVCache, get_attention_interface
        budgets, start = cls._sizes(case)
        cache, P = BatchedDynamicBudgetTrimKVCache(), int(start.max())
        cache.fuse_decode_append = True
        cache.set_budgets(start)
        new = [[None] * case["layers"] for _ in range(case["tokens"])]
        for l, (prompt, parts) in enumerate(cls._inputs(case, seed, P)):
            cache.update(*prompt, torch.arange(P, device=DEV), l)
            cache.evict_to_budgets(buffer_size=0, layers=[l])
            for t, part in enumerate(parts):
                new[t][l] = part
        cache.set_budgets(budgets)
        return {"cache": cache, "attend": get_attention_interface("db_attn_flash_batched"), "module": _module(case), "new": new, "buffer": case["buffer"], "layers": case["layers"],
                "run": cls._run}

    @staticmethod
    def _run(s):
        cache, outs = s["cache"], [[] for _ in range(s["layers"])]
        for portion in s["new"]:
            seen = cache.get_seq_length()
            positions = torch.arange(seen, seen + 1, device=DEV)
            for l, (k, v, lb, q) in enumerate(portion):
                keys, values, _, _, kw = cache.update(k, v, lb, positions, l)
                outs[l].append(s["attend"](s["module"], q, keys, values, None, flash_attn_kwargs=kw)[0])
            cache.evict_to_budgets(buffer_size=s["buffer"])
        return {"out": [torch.cat(o, dim=1) for o in outs], "lens": cache.head_lens, "cu": cache.cu_seqlens_k}

    @classmethod
    def exact(cls, case, seed):
        budgets, start = (t.to(DEV) for t in cls._sizes(case))
        B, H, G, D, T, P = case["batch"], case["kv_heads"], case["group"], case["dim"], case["tokens"], int(start.max())
        res, N = {"out": [], "lens": [], "cu": []}, P + T
        pos = torch.arange(N, device=DEV)
        for l, ((k, v, lb), parts) in enumerate(cls._inputs(case, seed, P)):
            k, v, lb = (torch.cat([t] + [part[i] for part in parts], dim=2) for i, t in enumerate((k, v, lb)))
            k, v, lb = k.view(B * H, N, D), v.view(B * H, N, D), lb.view(B * H, N)
            held = torch.zeros(B * H, N, dtype=torch.bool, device=DEV)
            held[:, :P] = _best(_scores(lb[:, :P], pos[:P], P + 1), start[l])
            seen = torch.empty(B * H, T, N, dtype=torch.bool, device=DEV)
            for t in range(T):
                held[:, P + t] = True
                seen[:, t] = held
                due = held.sum(1) >= budgets[l] + case["buffer"]
                if bool(due.any()):
                    held[due] = _best(_scores(lb[due], pos, P + t + 2).masked_fill(~held[due], -math.inf), budgets[l][due])
            q = torch.cat([part[3] for part in parts], dim=2).view(B * H, G, T, D)
            res["out"].append(_attend64(q, k, v, seen[:, None]).view(B, H * G, T, D).transpose(1, 2).contiguous())
            lens = held.sum(1).int()
            res["lens"].append(lens)
            res["cu"].append(torch.cat([lens.new_zeros(1), lens.cumsum(0).int()]))
        return res

    @classmethod
    def work(cls, case):
        budgets, start = cls._sizes(case)
        n, T, G, D, rows, moved = budgets.numel(), case["tokens"], case["group"], case["dim"], 0.0, 0.0
        held = start.clone()
        for _ in range(T):
            held += 1
            rows += float(held.sum())
            due = held >= budgets + case["buffer"]
            moved += _evict_bytes(1, float(held[due].sum()), float(budgets[due].sum()), D)
            held = torch.where(due, budgets, held)
        return {"bytes": rows * 4.0 * D + n * T * (4.0 * G * D + 8.0 * D + 24) + moved, "flops": 4.0 * G * D * rows}

    @staticmethod
    def tolerance(case):
        return _attention_tolerance(case)


class Shared:
    """A portion of a prompt against the flat cache: heads take what they need of a budget of ``memory`` rows per head."""

    @staticmethod
    def _rows(case):
        return case["memory"] + case["memory"] // 4 + case["buffer"]

    @classmethod
    def _inputs(cls, case, seed):
        gen, dt = _gen(seed), torch.bfloat16
        for _ in range(case["layers"]):
            # heads differ in how long they remember, so that they end up with different shares
            tilt = torch.randn(case["batch"], case["kv_heads"], 1, generator=gen, device=DEV)
            made = [_kv(case, gen, rows, dt) for rows in (cls._rows(case), case["chunk"])]
            made = [(k, v, torch.nn.functional.logsigmoid(torch.log(torch.expm1(-lb).reciprocal()) + tilt)) for k, v, lb in made]
            yield made[0], (*made[1], _q(case, gen, case["chunk"], dt))

    @classmethod
    def prepare(cls, case, seed):
        from trimkv_amd import BatchedDynamicBudgetTrimKVCache, get_attention_interface
        cache, P, new = BatchedDynamicBudgetTrimKVCache(), cls._rows(case), []
        for l, (prompt, part) in enumerate(cls._inputs(case, seed)):
            cache.update(*prompt, torch.arange(P, device=DEV), l)
            new.append(part)
        cache.compress(case["strategy"], memory_size=case["memory"], buffer_size=case["buffer"])
        return {"cache": cache, "attend": get_attention_interface("db_attn_flash_batched"), "module": _module(case), "new": new, "case": case, "run": cls._run}

    @staticmethod
    def _run(s):
        cache, case, outs = s["cache"], s["case"], []
        seen = cache.get_seq_length()
        positions = torch.arange(seen, seen + case["chunk"], device=DEV)
        for l, (k, v, lb, q) in enumerate(s["new"]):
            keys, values, _, _, kw = cache.update(k, v, lb, positions, l)
            outs.append(s["attend"](s["module"], q, keys, values, None, flash_attn_kwargs=kw)[0])
        cache.compress(case["strategy"], memory_size=case["memory"], buffer_size=case["buffer"])
        return {"out": outs, "lens": cache.head_lens, "cu": cache.cu_seqlens_k}

    @classmethod
    def exact(cls, case, seed):
        B, H, G, D, L, M, S, P = case["batch"], case["kv_heads"], case["group"], case["dim"], case["layers"], case["memory"], case["chunk"], cls._rows(case)
        layers = list(cls._inputs(case, seed))
        pos, N = torch.arange(P + S, device=DEV), P + S

        def cut(lb, held, query, n):
            """[L, B, H, n] rows held -> the ones the budget leaves."""
            score = _scores(lb, pos[:n], query).masked_fill(~held, -math.inf)
            if case["strategy"] == "alpha":     # one budget over all heads and layers of a sequence
                flat = score.permute(1, 0, 2, 3).reshape(B, L * H * n)
                return _best(flat, L * H * M).view(B, L, H, n).permute(1, 0, 2, 3)
            return _best(score.reshape(L, B, H * n), H * M).view(L, B, H, n)

        lb0 = torch.stack([p[2] for p, _ in layers])
        held = cut(lb0, torch.ones_like(lb0, dtype=torch.bool), P + 1, P)
        res = {"out": [], "lens": [], "cu": []}
        causal = torch.cat([torch.ones(S, P, dtype=torch.bool, device=DEV), torch.ones(S, S, dtype=torch.bool, device=DEV).tril()], dim=1)
        for l, ((k0, v0, _), (k, v, _, q)) in enumerate(layers):
            k, v = torch.cat([k0, k], dim=2).view(B * H, N, D), torch.cat([v0, v], dim=2).view(B * H, N, D)
            rows = torch.cat([held[l], held.new_ones(B, H, S)], dim=2).view(B * H, 1, 1, N)
            out = torch.cat([_attend64(q.view(B * H, G, S, D)[i:i + 1], k[i:i + 1], v[i:i + 1], rows[i:i + 1] & causal) for i in range(B * H)])
            res["out"].append(out.view(B, H * G, S, D).transpose(1, 2).contiguous())
        lb = torch.cat([lb0, torch.stack([part[2] for _, part in layers])], dim=3)
        held = cut(lb, torch.cat([held, held.new_ones(L, B, H, S)], dim=3), N + 1, N)
        for l in range(L):
            lens = held[l].sum(-1).int().reshape(-1)
            res["lens"].append(lens)
            res["cu"].append(torch.cat([lens.new_zeros(1), lens.cumsum(0).int()]))
        return res

    @staticmethod
    def work(case):
        n, S, M, G, D = case["batch"] * case["kv_heads"], case["chunk"], case["memory"], case["group"], case["dim"]
        return {"bytes": case["layers"] * (n * ((M + S) * 4.0 * D + S * (4.0 * G * D + 8.0 * D + 24)) + _evict_bytes(n, M + S, M, D)),
                "flops": case["layers"] * 4.0 * n * G * D * (S * M + S * (S + 1) / 2.0)}

    @staticmethod
    def tolerance(case):
        return _attention_tolerance(case)


# ---- the Qwen3 decoder -----------------------------------------------------------------------------------------------------
def _rms64(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


class Qwen3:
    GATE, EPS, THETA, WARM = 512, 1e-6, 1e6, 2

    @classmethod
    def _weights(cls, case, gen):
        z, D, H = QWEN3[case["size"]], 128, 8
        normal = lambda *shape: torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16) * 0.02
        out = {"model.embed_tokens.weight": normal(VOCAB, z["W"]) * 50, "lm_head.weight": normal(VOCAB, z["W"]), "model.norm.weight": None}
        for l in range(case["layers"]):
            p = f"model.layers.{l}."
            for name, n, k in (("self_attn.q_proj", z["Hq"] * D, z["W"]), ("self_attn.k_proj", H * D, z["W"]), ("self_attn.v_proj", H * D, z["W"]),
                               ("self_attn.o_proj", z["W"], z["Hq"] * D), ("mlp.gate_proj", z["ff"], z["W"]), ("mlp.up_proj", z["ff"], z["W"]), ("mlp.down_proj", z["W"], z["ff"]),
                               ("self_attn.retention_gate.linear1", cls.GATE, z["W"]), ("self_attn.retention_gate.linear2", H, cls.GATE)):
                out[p + name + ".weight"] = normal(n, k)
        return out

    @classmethod
    def _inputs(cls, case, seed):
        """Weights, per layer the rows of a prompt, and the tokens of the steps."""
        gen = _gen(seed)
        shape = {"batch": case["batch"], "kv_heads": 8, "dim": 128}
        weights, P = cls._weights(case, gen), _dense_prompt_rows(case)
        ids = torch.randint(0, VOCAB, (cls.WARM + 1, case["batch"], 1), generator=gen, device=DEV)
        prompts = (_kv(shape, gen, P, torch.bfloat16) for _ in range(case["layers"]))
        return weights, ids, P, ((k, v, lb.to(torch.bfloat16)) for k, v, lb in prompts)

    @classmethod
    def prepare(cls, case, seed):
        from trimkv_amd import TrimKVCache
        from trimkv_amd.graphed import GraphedDecoder
        from trimkv_amd.qwen3 import TrimKVQwen3Config, TrimKVQwen3ForCausalLM
        z = QWEN3[case["size"]]
        cfg = TrimKVQwen3Config(vocab_size=VOCAB, hidden_size=z["W"], intermediate_size=z["ff"], num_hidden_layers=case["layers"], num_attention_heads=z["Hq"], num_key_value_heads=8,
                                head_dim=128, retention_gate="rg", retention_gate_intermediate_size=cls.GATE, retention_gate_bias_init=3.0, rms_norm_eps=cls.EPS, rope_theta=cls.THETA,
                                memory_size=case["memory"], buffer_size=case["buffer"])
        before = torch.get_default_dtype()
        torch.set_default_dtype(torch.bfloat16)
        try:
            with torch.device(DEV):
                model = TrimKVQwen3ForCausalLM(cfg).eval()
        finally:
            torch.set_default_dtype(before)
        weights, ids, P, prompts = cls._inputs(case, seed)
        model.load_state_dict({k: w for k, w in weights.items() if w is not None}, strict=False)
        del weights
        cache = TrimKVCache()
        for l, prompt in enumerate(prompts):
            cache.update(*prompt, torch.arange(P, device=DEV), l)
        cache.compress("alpha", memory_size=case["memory"], buffer_size=case["buffer"])
        step = GraphedDecoder(model, cache, logits_to_keep=1)
        for t in range(cls.WARM):       # the first call runs eagerly, the second one captures
            step(input_ids=ids[t])
        return {"step": step, "ids": ids[cls.WARM], "run": lambda s: {"logits": s["step"](input_ids=s["ids"]).logits}}

    @classmethod
    def exact(cls, case, seed):
        z, M, B, H, D = QWEN3[case["size"]], case["memory"], case["batch"], 8, 128
        G = z["Hq"] // H
        W, ids, P, prompts = cls._inputs(case, seed)
        x = [W["model.embed_tokens.weight"].double()[ids[t, :, 0]] for t in range(cls.WARM + 1)]
        freq = cls.THETA ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)

        def turn(y, at):
            c, s = torch.cos(at * freq), torch.sin(at * freq)
            a, b = y[..., :D // 2], y[..., D // 2:]
            return torch.cat([a * c - b * s, b * c + a * s], -1)

        for l, (k, v, lb) in enumerate(prompts):
            w = lambda name: W[f"model.layers.{l}.{name}.weight"].double()
            kept = _best(_scores(lb, torch.arange(P, device=DEV), P + 1), M).nonzero()[:, 2].view(B, H, M, 1).expand(B, H, M, D)
            k, v = (torch.gather(t, 2, kept).double() for t in (k, v))
            for t in range(cls.WARM + 1):
                h = _rms64(x[t], cls.EPS)
                q, kn, vn = ((h @ w(f"self_attn.{n}_proj").T).view(B, -1, D) for n in "qkv")
                q, kn = turn(_rms64(q, cls.EPS), P + t), turn(_rms64(kn, cls.EPS), P + t)
                k, v = torch.cat([k, kn.unsqueeze(2)], 2), torch.cat([v, vn.unsqueeze(2)], 2)
                score = torch.matmul(q.view(B, H, G, D), k.transpose(2, 3).contiguous()) * D ** -0.5
                x[t] = x[t] + torch.matmul(torch.softmax(score, -1), v).view(B, -1) @ w("self_attn.o_proj").T
                h = _rms64(x[t], cls.EPS)
                x[t] = x[t] + (torch.nn.functional.silu(h @ w("mlp.gate_proj").T) * (h @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T
        return {"logits": (_rms64(x[-1], cls.EPS) @ W["lm_head.weight"].double().T).unsqueeze(1)}

    @classmethod
    def work(cls, case):
        z, B, D, H, L = QWEN3[case["size"]], case["batch"], 128, 8, case["layers"]
        matrices = L * (z["W"] * D * (2 * z["Hq"] + 2 * H) + 3 * z["W"] * z["ff"] + cls.GATE * (z["W"] + H)) + VOCAB * z["W"]
        rows = case["memory"] + cls.WARM + 1
        return {"bytes": 2.0 * matrices + L * B * H * rows * 4.0 * D + 4.0 * B * VOCAB, "flops": 2.0 * B * matrices + L * 4.0 * B * z["Hq"] * D * rows}

    @staticmethod
    def tolerance(case):
        return {"rel": 3e-2, "max": 0.3}      # a bf16 residual stream: measured 7e-3 to 2e-2 by the number of layers


# ---- the hybrid decoders ---------------------------------------------------------------------------------------------------
class Hybrid:
    """Siterax: rotary windowed attention with a softmax sink and head gates, dense feed-forwards, its last layer passed twice.
    Fusitar: mLSTM and windowed attention in turn (their routed feed-forwards are the ``experts`` cases)."""
    EPS, CAP, GATE_CAP, MULT, WARM = 1e-6, 30.0, 15.0, 0.7, 2

    @classmethod
    def _config(cls, case):
        z, D, L = HYBRID[case["size"]], 128, case["layers"]
        base = {"vocab": VOCAB, "width": z["W"], "norm": {"eps": cls.EPS}}
        mixer = {"heads": z["Hq"], "kv_heads": z["Hkv"], "dim": D, "vdim": D, "scale": D ** -0.5}
        if case["kind"] == "siterax":
            layer = {"type": "attention", "mlp": {"kind": "dense", "ff": 3 * z["W"]},
                     "mixer": dict(mixer, mask={"size": z["window"] + z["keep"]}, rot={"base": 1e6, "dims": D, "scaling": {"factor": 2.0}})}
            return dict(base, architecture="Siterax", residual_mult=cls.MULT, logit_softcap=cls.CAP, loop={"start": L - 1, "stop": L, "times": 2}, layers=[layer] * L)
        kinds = [{"type": "mlstm", "mlp": None, "mixer": {"heads": z["mh"], "dim": 128, "vdim": 256, "gate_cap": cls.GATE_CAP}},
                 {"type": "attention", "mlp": None, "mixer": dict(mixer, mask={"size": z["window"], "keep_first": z["keep"]})}]
        return dict(base, architecture="Fusitar", embedding={"scale": 1.0}, layers=[kinds[i % 2] for i in range(L)])

    @classmethod
    def _weights(cls, cfg, gen):
        """Checkpoint name -> tensor: matrices of unit gain, norms around one, forget gates mostly open."""
        rnd = lambda *shape: torch.randn(shape, generator=gen, device=DEV)
        W, siterax = cfg["width"], cfg["architecture"] == "Siterax"
        out = {"embed": rnd(cfg["vocab"], W), "final.norm": 1 + 0.2 * rnd(W)}
        if siterax:
            out["head"] = rnd(cfg["vocab"], W) * W ** -0.5
        for i, layer in enumerate(cfg["layers"]):
            m, p = layer["mixer"], f"l{i}.mix."
            H, G, D, V = m["heads"], m.get("kv_heads", m["heads"]), m["dim"], m["vdim"]
            mats = {p + "q": (H * D, W), p + "k": (G * D, W), p + "v": (G * V, W), p + "g": (H if siterax else H * V, W), p + "o": (W, H * V)}
            norms = ["norm1", "norm1b", "norm2", "norm2b"] if siterax else ["norm1"]
            if layer["type"] == "mlstm":
                mats.update({p + "i": (H, W), p + "f": (H, W)})
                out.update({p + "i.b": 0.5 * rnd(H), p + "f.b": 4 + rnd(H), p + "norm": 1 + 0.2 * rnd(H * V)})
            else:
                n = 1 if siterax else 0
                out.update({p + "q.norm": 1.2 + 0.2 * rnd(D if n else H * D), p + "k.norm": 1.2 + 0.2 * rnd(D if n else G * D)})
                if siterax:
                    out.update({p + "q.b": 0.3 * rnd(H * D), p + "k.b": 0.3 * rnd(G * D), p + "v.b": 0.3 * rnd(G * V)})
            if layer["mlp"] is not None:
                ff, r = layer["mlp"]["ff"], f"l{i}.mlp."
                mats.update({r + "gate": (ff, W), r + "up": (ff, W), r + "down": (W, ff)})
            out.update({f"l{i}.{n}": 1 + 0.2 * rnd(W) for n in norms})
            out.update({name: rnd(*shape) * shape[1] ** -0.5 for name, shape in mats.items()})
        return {k: v.to(torch.bfloat16) for k, v in out.items()}

    @staticmethod
    def _lengths(case):
        if case["mode"] == "prompt":
            return [int(n) for n in case["lengths"].split(",")]
        B, longest = case["batch"], case["longest"]       # spread evenly over their logarithm, the longest sixteen times the shortest
        return [max(1, int(longest * 16.0 ** (-b / max(1, B - 1)))) for b in range(B)]

    @classmethod
    def _inputs(cls, case, seed):
        gen, cfg, lengths = _gen(seed), cls._config(case), cls._lengths(case)
        weights = cls._weights(cfg, gen)
        ids = torch.randint(0, VOCAB, (sum(lengths),), generator=gen, device=DEV)
        return cfg, weights, lengths, ids, torch.randint(0, VOCAB, (cls.WARM + 1, len(lengths), 1), generator=gen, device=DEV)

    @classmethod
    def prepare(cls, case, seed):
        from trimkv_amd.fusitar import FusitarConfig, FusitarForCausalLM
        from trimkv_amd.graphed import GraphedDecoder
        from trimkv_amd.siterax import SiteraxConfig, SiteraxForCausalLM
        cfg, weights, lengths, ids, steps = cls._inputs(case, seed)
        config, model = (SiteraxConfig, SiteraxForCausalLM) if case["kind"] == "siterax" else (FusitarConfig, FusitarForCausalLM)
        with torch.device(DEV):
            model = model(config.from_dict(cfg), DTYPES[case["dtype"]]).eval()
        model.load_tensors(weights)
        del weights
        cache = model.new_cache(len(lengths))
        if case["mode"] == "prompt":
            return {"model": model, "cache": cache, "lengths": lengths, "ids": ids, "run": cls._run_prompt}
        slots, at = cache.allocate(len(lengths)), 0
        for b, n in enumerate(lengths):
            model(ids[at:at + n], past_key_values=cache, lengths=[n], slots=[slots[b]], logits_to_keep=1)
            at += n
        step = GraphedDecoder(model, cache, logits_to_keep=1)
        for t in range(cls.WARM):       # the first call runs eagerly, the second one captures
            step(input_ids=steps[t])
        return {"step": step, "ids": steps[cls.WARM], "run": lambda s: {"logits": s["step"](input_ids=s["ids"]).logits}}

    @staticmethod
    def _run_prompt(s):
        """Prompts into fresh slots of a server's cache, the logits of every token; the slots are given back."""
        cache = s["cache"]
        slots = cache.allocate(len(s["lengths"]))
        out = s["model"](s["ids"], past_key_values=cache, lengths=s["lengths"], slots=slots, rows=None)
        cache.release(slots)
        return {"logits": out.logits}

    # -- the same in 64 bits, one sequence at a time
    @staticmethod
    def _window64(q, k, v, scale, size, keep, sink):
        """q [T, H, D], k and v [T, G, .] -> [T, H, V]."""
        T, H, D = q.shape
        G = k.shape[1]
        kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
        out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
        for a in range(0, T, 512):
            b = min(T, a + 512)
            i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(b, device=q.device)[None, :]
            hidden = (j > i) | ((i - j >= size) & (j >= keep))
            qs = q[a:b].permute(1, 0, 2).reshape(G, (H // G) * (b - a), D)
            score = (torch.matmul(qs, kt[:, :, :b]) * scale).view(H, b - a, b).masked_fill_(hidden, -math.inf)
            top = score.amax(-1, keepdim=True)
            if sink:
                top = top.clamp(min=0.0)
            e = torch.exp(score - top)
            e = e / (e.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0))
            out[a:b] = torch.matmul(e.view(G, (H // G) * (b - a), b), vt[:, :b]).view(H, b - a, -1).permute(1, 0, 2)
        return out

    @staticmethod
    def _mlstm64(q, k, v, log_i, log_f):
        """The recurrence unrolled: with F the running sum of log_f, token t reads token s with weight exp(F_t - F_s + i_s - m_t)."""
        T, H, _ = q.shape
        F = log_f.cumsum(0)
        out = torch.empty_like(v)
        for h in range(H):
            for a in range(0, T, 1024):
                b = min(T, a + 1024)
                d = F[a:b, h, None] - F[None, :b, h] + log_i[None, :b, h]
                d.masked_fill_(torch.arange(b, device=q.device)[None, :] > torch.arange(a, b, device=q.device)[:, None], -math.inf)
                m = torch.maximum(d.amax(1), F[a:b, h])
                w = torch.exp(d - m[:, None]) * (q[a:b, h] @ k[:b, h].T)
                out[a:b, h] = (w @ v[:b, h]) / (torch.maximum(w.sum(1).abs(), torch.exp(-m)) + 1e-6)[:, None]
        return out

    @classmethod
    def _mix64(cls, h, w, m, kind):
        T, H, D, V = h.shape[0], m["heads"], m["dim"], m["vdim"]
        lin = lambda name: h @ w[name].T
        if kind == "mlstm":
            cap = lambda z: cls.GATE_CAP * torch.tanh(z / cls.GATE_CAP)
            log_i, log_f = cap(lin("i") + w["i.b"]), torch.nn.functional.logsigmoid(cap(lin("f") + w["f.b"]))
            o = cls._mlstm64(lin("q").view(T, H, D) * D ** -0.5, lin("k").view(T, H, D), lin("v").view(T, H, V), log_i, log_f)
            o = _rms64(o, cls.EPS).reshape(T, H * V) * w["norm"] * torch.sigmoid(lin("g"))
            return o @ w["o"].T
        if "q.b" in w:
            turned = []
            for name, b in (("q", "q.b"), ("k", "k.b")):
                y = _rms64((lin(name) + w[b]).view(T, -1, D), cls.EPS) * w[name + ".norm"]
                half = m["rot"]["dims"] // 2
                freq = m["rot"]["base"] ** (-torch.arange(half, device=h.device, dtype=torch.float64) / half) / m["rot"]["scaling"]["factor"]
                angle = torch.arange(T, device=h.device, dtype=torch.float64)[:, None, None] * freq
                u, x, c, s = y[..., :half], y[..., half:2 * half], torch.cos(angle), torch.sin(angle)
                turned.append(torch.cat([u * c - x * s, x * c + u * s, y[..., 2 * half:]], -1))
            o = cls._window64(*turned, (lin("v") + w["v.b"]).view(T, -1, V), m["scale"], m["mask"]["size"], 0, True)
            return (o * torch.sigmoid(lin("g"))[:, :, None]).reshape(T, H * V) @ w["o"].T
        q, k = ((_rms64(lin(n), cls.EPS) * w[n + ".norm"]).view(T, -1, D) for n in "qk")
        o = cls._window64(q, k, lin("v").view(T, -1, V), m["scale"], m["mask"]["size"], m["mask"]["keep_first"], False)
        return (o.reshape(T, H * V) * torch.sigmoid(lin("g"))) @ w["o"].T

    @classmethod
    def exact(cls, case, seed):
        cfg, W, lengths, ids, steps = cls._inputs(case, seed)
        W = {k: t.double() for k, t in W.items()}
        siterax, out, at = case["kind"] == "siterax", [], 0
        order = [(i, False) for i in range(case["layers"])] + ([(case["layers"] - 1, True)] if siterax else [])
        norm = lambda name, x: _rms64(x, cls.EPS) * W[name]
        for b, n in enumerate(lengths):
            tokens = ids[at:at + n] if case["mode"] == "prompt" else torch.cat([ids[at:at + n], steps[:, b, 0]])
            at += n
            first = x = W["embed"][tokens]
            for i, again in order:
                layer, p = cfg["layers"][i], f"l{i}."
                mix = {k[len(p) + 4:]: t for k, t in W.items() if k.startswith(p + "mix.")}
                if again:
                    x = x + first
                if not siterax:
                    x = x + norm(p + "norm1", cls._mix64(x, mix, layer["mixer"], layer["type"]))
                    continue
                x = x + cls.MULT * norm(p + "norm1b", cls._mix64(norm(p + "norm1", x), mix, layer["mixer"], layer["type"]))
                h = norm(p + "norm2", x)
                y = (torch.nn.functional.silu(h @ W[p + "mlp.gate"].T) * (h @ W[p + "mlp.up"].T)) @ W[p + "mlp.down"].T
                x = x + cls.MULT * norm(p + "norm2b", y)
            x = norm("final.norm", x if case["mode"] == "prompt" else x[-1:])
            out.append(cls.CAP * torch.tanh(x @ W["head"].T / cls.CAP) if siterax else x @ W["embed"].T)
        if case["mode"] == "step":
            return {"logits": torch.stack(out)}
        # equal lengths (a single prompt among them) come back as a batch
        return {"logits": torch.stack(out) if len(set(lengths)) == 1 else torch.cat(out)}

    @classmethod
    def work(cls, case):
        z, cfg, lengths, D = HYBRID[case["size"]], cls._config(case), cls._lengths(case), 128
        e, window, keep = (4.0 if case["dtype"] == "fp32" else 2.0), z["window"], z["keep"]
        step, T = case["mode"] == "step", sum(lengths) if case["mode"] == "prompt" else len(lengths)
        # rows that the tokens of this pass see
        if step:
            seen = sum(min(n + cls.WARM + 1, window + keep) for n in lengths)
        else:
            most = lambda n: n * (n + 1) / 2 - max(0, n - window - keep) * (n - window - keep + 1) / 2
            seen = sum(most(n) for n in lengths)
        matrices, state, flops = VOCAB * z["W"] * 1.0, 0.0, 0.0
        runs = cfg["layers"] + ([cfg["layers"][-1]] if case["kind"] == "siterax" else [])
        for layer in runs:
            m = layer["mixer"]
            H, G, V = m["heads"], m.get("kv_heads", m["heads"]), m["vdim"]
            matrices += z["W"] * (H * D + G * D + G * V + 2 * H * V) + (9 * z["W"] ** 2 if layer["mlp"] else 0)
            if layer["type"] == "attention":
                flops += 4.0 * D * H * seen
                state += G * (D + V) * e * (seen if step else sum(min(n, window + keep) for n in lengths))
            else:       # outer product and read-out per token
                flops += 4.0 * H * D * V * T
                state += 4.0 * H * D * V * len(lengths) * (2 if step else 1)
        # the weights, the caches, the stream in and out of every layer once and the logits
        return {"bytes": e * matrices + state + T * (len(runs) * 8.0 * z["W"] + 4.0 * VOCAB), "flops": flops + 2.0 * T * matrices}

    @staticmethod
    def tolerance(case):
        return {"rel": 1e-5, "max": 1e-4} if case["dtype"] == "fp32" else {"rel": 2e-2, "max": 0.2}      # measured: 1.5e-6 and 5e-3


class Experts:
    """Routed squared-ReLU experts over the rows of the residual stream: router, choice, both products."""

    @staticmethod
    def _inputs(case, seed):
        z, gen = HYBRID[case["size"]], _gen(seed)
        W, ff = z["W"], z["ff"]
        rnd = lambda *shape: torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16)
        x = torch.randn(case["tokens"], W, generator=gen, device=DEV) * 1.5
        router, correction = rnd(EXPERTS, W) * (2.0 * W ** -0.5), torch.randn(EXPERTS, generator=gen, device=DEV) * 0.05
        return x, router, correction, ((rnd(ff, W) * W ** -0.5, rnd(W, ff) * ff ** -0.5) for _ in range(EXPERTS))

    @classmethod
    def prepare(cls, case, seed):
        from trimkv_amd.hybrid import RoutedExperts
        z = HYBRID[case["size"]]
        with torch.device(DEV):
            block = RoutedExperts({"expert": {"ff": z["ff"]}, "router": {"experts": EXPERTS, "top": CHOSEN, "groups": {"count": GROUPS, "keep": OPEN}}}, z["W"], torch.bfloat16)
        x, router, correction, matrices = cls._inputs(case, seed)
        parts = block.tensors()
        parts["router"].copy_(router)
        parts["correction"].copy_(correction)
        for e, (up, down) in enumerate(matrices):
            parts[f"e{e}.up"].copy_(up)
            parts[f"e{e}.down"].copy_(down)
        return {"block": block, "x": x, "xh": x.to(torch.bfloat16), "run": cls._run}

    @staticmethod
    def _run(s):
        rows, weights = s["block"](s["x"], s["xh"])
        return {"rows": rows, "weights": weights}

    @classmethod
    def exact(cls, case, seed):
        x, router, correction, matrices = cls._inputs(case, seed)
        T, h = x.shape[0], x.to(torch.bfloat16).double()
        s = torch.sigmoid(x.double() @ router.double().T)
        choice = s + correction.double()
        best = choice.view(T, GROUPS, -1).topk(2, -1).values.sum(-1).topk(OPEN, -1).indices
        shut = torch.ones(T, GROUPS, dtype=torch.bool, device=DEV).scatter_(1, best, False)
        ids = choice.masked_fill(shut.repeat_interleave(EXPERTS // GROUPS, 1), -math.inf).topk(CHOSEN, -1).indices
        rows = torch.empty(T * CHOSEN, x.shape[1], dtype=torch.float64, device=DEV)
        for e, (up, down) in enumerate(matrices):
            at = (ids.reshape(-1) == e).nonzero()[:, 0]
            rows[at] = torch.relu(h[at // CHOSEN] @ up.double().T).square() @ down.double().T
        return {"rows": rows, "weights": torch.gather(s, 1, ids)}

    @staticmethod
    def work(case):
        z, T = HYBRID[case["size"]], case["tokens"]
        used = EXPERTS * (1 - (1 - CHOSEN / EXPERTS) ** T)       # experts that some token is expected to choose
        return {"bytes": used * 4.0 * z["W"] * z["ff"] + T * z["W"] * (6.0 + 2.0 * CHOSEN), "flops": 4.0 * T * CHOSEN * z["W"] * z["ff"]}

    @staticmethod
    def tolerance(case):
        return {"rel": 1e-2, "max": 0.1}      # measured: 2.3e-3


KINDS = {"decode": Decode, "ragged": Ragged, "chunk": Chunk, "shared": Shared, "qwen3": Qwen3, "siterax": Hybrid, "fusitar": Hybrid, "experts": Experts}
