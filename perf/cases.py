"""The work that users of this framework have it do, as timed cases.

A case is one call sequence of an engine that holds its KV cache in a
``PagedKVCache``.  Four kinds:

* ``decode``   the attention core of a decode step, over some layers: the plan
  of the step, then per layer the new K/V row's norm, RoPE and append with
  decode attention (``append_decode``), as the engine's decode loop calls it;
* ``layer``    whole full-attention layers from the normed hidden state to the
  residual stream: ``project_append``, ``decode`` (one new token per
  sequence) or ``prefill``, both gated, and ``out_project``;
* ``prefill``  the attention core of a prompt chunk (``append_prefill``);
* ``tree``     speculative verify of a draft tree: append, ``tree_verify``,
  then ``rollback`` to the accepted path.

Shapes are the model's (24 query and 4 KV heads of 256, hidden 5120) or its
shards over 2 and 4 GPUs (12/2 and 6/1 heads).  Rows past the cached ones are
written by the pass itself, at the same slots in every pass, so a state can
be run again.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mi50grad_amd.kv_cache import PagedKVCache
from mi50grad_amd.rope import rope_tables
from mi50grad_amd.tree import depths, root_to_node_path, tree_bits

D = 256
PAGE = 16
HALF_ROT = 32
THETA = 10000000.0
EPS = 1e-6


def _case(kind, seqs, ctx_lo, ctx_hi, new_lo=1, new_hi=1, layers=1, heads=24, kv_heads=4, hidden=5120, gate=True,
          ragged=0):
    return {"kind": kind, "seqs": seqs, "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "new_lo": new_lo, "new_hi": new_hi,
            "layers": layers, "heads": heads, "kv_heads": kv_heads, "hidden": hidden, "gate": gate, "ragged": ragged}


def listed():
    return [
        # One chat user near the start of a conversation: all 16 layers of a
        # step, launches and latency only.
        dict(_case("decode", 1, 255, 255, layers=16), name="decode_b1_256"),
        # One user deep in a long document.
        dict(_case("decode", 1, 20011, 20011, layers=4), name="decode_b1_20k"),
        # A batch of short chats at ragged lengths.
        dict(_case("decode", 32, 64, 1000, layers=4, ragged=1), name="decode_b32_short"),
        # The serving batch of the benchmark: 32 ragged contexts of 1k to 8k.
        dict(_case("decode", 32, 1024, 8192, layers=2, ragged=2), name="decode_b32_8k"),
        # A whole layer of a single-user decode step.
        dict(_case("layer", 1, 1500, 1500, layers=2), name="layer_b1"),
        # A whole layer of a larger decode batch.
        dict(_case("layer", 48, 100, 4000, layers=1, ragged=3), name="layer_b48"),
        # The shard of a GPU of four (6 query heads, 1 KV head), small batch.
        dict(_case("layer", 5, 300, 3000, layers=2, heads=6, kv_heads=1, ragged=4), name="layer_b5_tp4"),
        # A whole layer over a short prompt, empty cache.
        dict(_case("layer", 1, 0, 0, 181, 181, layers=2), name="layer_prompt181"),
        # A whole layer over the chunks of four prompts at several depths.
        dict(_case("layer", 4, 0, 2048, 512, 512, layers=1, ragged=5), name="layer_4x512"),
        # A chunk late in a long prompt: the attention alone.
        dict(_case("prefill", 1, 16400, 16400, 2048, 2048, layers=1), name="prefill_2k_at_16k"),
        # Draft trees of nine nodes verified for eight users.
        dict(_case("tree", 8, 300, 3000, 9, 9, layers=2, ragged=6), name="tree_b8"),
        # The same for 64 long contexts.
        dict(_case("tree", 64, 4096, 32768, 9, 9, layers=1, ragged=7), name="tree_b64_32k"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "layer", "layer", "layer", "layer", "prefill", "tree", "tree"])
    heads, kv_heads = rng.choice([(24, 4), (24, 4), (12, 2), (6, 1)])
    gate = rng.random() < 0.75
    ragged = rng.randrange(1, 1 << 20)

    def rows_left(total, seqs):  # longest context that keeps the case within the listed ones' cost
        return max(16, total // seqs)

    if kind == "decode":
        seqs = _log(rng, 1, 64)
        hi = _log(rng, 16, min(32768, rows_left(400000, seqs)))
        lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
        layers = max(1, min(rng.choice([1, 2, 4, 8, 16]), 400000 // (seqs * hi)))
        return _case(kind, seqs, lo, hi, layers=layers, heads=heads, kv_heads=kv_heads, gate=gate, ragged=ragged)
    if kind == "layer":
        if rng.random() < 0.5:
            seqs = _log(rng, 1, 64)
            hi = _log(rng, 16, min(16384, rows_left(200000, seqs)))
            return _case(kind, seqs, max(1, int(hi * rng.uniform(0.1, 1.0))), hi, layers=rng.choice([1, 2]),
                         heads=heads, kv_heads=kv_heads, ragged=ragged)
        seqs = rng.choice([1, 1, 2, 4])
        new = _log(rng, 9, 2048 // seqs)
        hi = rng.choice([0, _log(rng, 1, 4096)])
        return _case(kind, seqs, int(hi * rng.uniform(0.0, 1.0)), hi, max(2, int(new * rng.uniform(0.5, 1.0))), new,
                     layers=1, heads=heads, kv_heads=kv_heads, ragged=ragged)
    if kind == "prefill":
        seqs = rng.choice([1, 1, 2, 4])
        new = _log(rng, 17, 2048 // seqs)
        hi = rng.choice([0, _log(rng, 16, 16384)])
        return _case(kind, seqs, int(hi * rng.uniform(0.0, 1.0)), hi, max(2, int(new * rng.uniform(0.5, 1.0))), new,
                     layers=1, heads=heads, kv_heads=kv_heads, gate=gate, ragged=ragged)
    seqs = _log(rng, 1, 64)
    hi = _log(rng, 64, min(32768, rows_left(1000000, seqs)))
    nodes = rng.randrange(3, 33)
    return _case("tree", seqs, max(1, int(hi * rng.uniform(0.1, 1.0))), hi, nodes, nodes, layers=1, heads=heads,
                 kv_heads=kv_heads, gate=gate, ragged=ragged)


class _Plan:
    """What a case's sizes come to: lengths, new rows, pages."""

    def __init__(self, case):
        self.c = case
        self.L, self.H, self.KV, self.B = case["layers"], case["heads"], case["kv_heads"], case["seqs"]
        r = np.random.default_rng(case["ragged"])
        self.base = [int(x) for x in r.integers(case["ctx_lo"], case["ctx_hi"] + 1, self.B)]
        self.new = [int(x) for x in r.integers(case["new_lo"], case["new_hi"] + 1, self.B)]
        self.T = sum(self.new)
        self.parents = [(i - 1) // 3 for i in range(self.new[0])] if case["kind"] == "tree" else None
        if self.parents:
            self.parents[0] = -1
            self.kept = root_to_node_path(self.parents, len(self.parents) - 1)
        # The pages that a pass writes come first in the pool, so that they
        # can be returned whole; the pages before them lie anywhere.
        first = [b // PAGE for b in self.base]
        last = [(b + n + PAGE - 1) // PAGE for b, n in zip(self.base, self.new)]
        self.tail = sum(e - s for s, e in zip(first, last))
        self.pages = sum(last)
        self.first, self.last = first, last
        self.widest = max(last)
        self.rows = max(b + n for b, n in zip(self.base, self.new))

    def block_ids(self, seed):
        rest = np.random.default_rng(seed).permutation(self.pages - self.tail) + self.tail
        ids, t, o = [], 0, 0
        for s, e in zip(self.first, self.last):
            ids.append([int(x) for x in rest[o:o + s]] + list(range(t, t + e - s)))
            o += s
            t += e - s
        return ids

    def positions(self):
        """Per new token: its RoPE position."""
        d = depths(self.parents) if self.parents else None
        return [b + (d[i] if d else i) for b, n in zip(self.base, self.new) for i in range(n)]


def _half(gen, *shape, scale=1.0):
    x = torch.empty(shape, dtype=torch.float16, device="cuda").normal_(generator=gen)
    return x * scale if scale != 1.0 else x


def _inputs(case, seed, pools=None):
    """Every tensor of a case, from the seed; the K and V pools go into
    `pools` when given."""
    p = _Plan(case)
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = {}
    shape = (p.L, p.pages, PAGE, p.KV, D)
    if pools is None:
        pools = [torch.empty(shape, dtype=torch.float16, device="cuda") for _ in range(2)]
    for pool in pools:
        pool.normal_(generator=g)
    x["k_pool"], x["v_pool"] = pools
    x["q_norm"] = 1.0 + 0.02 * torch.empty(p.L, D, device="cuda").normal_(generator=g)
    x["k_norm"] = 1.0 + 0.02 * torch.empty(p.L, D, device="cuda").normal_(generator=g)
    x["q_norm"], x["k_norm"] = x["q_norm"].half(), x["k_norm"].half()
    if case["kind"] == "layer":
        hid = case["hidden"]
        x["x"] = _half(g, p.L, p.T, hid)
        x["residual"] = _half(g, p.L, p.T, hid)
        x["w_q"] = _half(g, p.L, 2 * p.H * D, hid, scale=hid ** -0.5)
        x["w_kv"] = _half(g, p.L, 2 * p.KV * D, hid, scale=hid ** -0.5)
        x["w_o"] = _half(g, p.L, hid, p.H * D, scale=(p.H * D) ** -0.5)
    else:
        x["q"] = _half(g, p.L, p.T, p.H, D)
        x["k"] = _half(g, p.L, p.T, p.KV, D)
        x["v"] = _half(g, p.L, p.T, p.KV, D)
        x["gate"] = _half(g, p.L, p.T, p.H, D) if case["gate"] else None
    return p, x


class _Memory:
    """The cache's pools as a tensor (the memory stays the cache's own)."""

    def __init__(self, ptr, shape, owner):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f2", "data": (ptr, False), "version": 2}
        self.owner = owner


class _State:
    pass


def prepare(case, seed):
    p = _Plan(case)
    s = _State()
    s.p = p
    s.cache = PagedKVCache(n_layers=p.L, max_seqs=p.B, max_blocks=p.pages, max_blocks_per_seq=p.widest,
                           max_step_tokens=max(16, p.T), num_heads=p.H, num_kv_heads=p.KV)
    kp, vp = s.cache.layer_pools(0)
    shape = (p.L, p.pages, PAGE, p.KV, D)
    pools = [torch.as_tensor(_Memory(ptr, shape, s.cache), device="cuda") for ptr in (kp, vp)]
    _, s.x = _inputs(case, seed, pools)
    for b, ids in enumerate(p.block_ids(seed)):
        s.cache.set_blocks(b, ids)
        s.cache.set_len(b, p.base[b])
    s.cache.sync_tables()
    cos, sin = rope_tables(p.rows + 1)
    s.cos, s.sin = torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()
    s.seqs, s.nothing = list(range(p.B)), [[] for _ in range(p.B)]
    s.q = torch.empty(p.L, p.T, p.H, D, dtype=torch.float16, device="cuda")
    s.out = torch.empty_like(s.q)
    if case["kind"] == "layer":
        s.gate = torch.empty_like(s.q)
        s.y = torch.empty(p.L, p.T, case["hidden"], dtype=torch.float16, device="cuda")
    if case["kind"] == "tree":
        s.k = torch.empty_like(s.x["k"])
        s.rope_pos = p.positions()
        s.bits = tree_bits(p.parents) * p.B
        s.keep = [list(p.kept)] * p.B
    s.tail_k, s.tail_v = pools[0][:, :p.tail], pools[1][:, :p.tail]
    torch.cuda.synchronize()
    return s


def _ptr(t, layer):
    return t.data_ptr() + layer * t.stride(0) * t.element_size()


def run(s):
    p, x, cache = s.p, s.x, s.cache
    kind = p.c["kind"]
    tables = (s.cos.data_ptr(), s.sin.data_ptr(), p.rows + 1)
    cache.rollback(s.seqs, p.base, s.nothing)  # the last pass's rows go: this pass writes them again
    if kind == "tree":
        cache.begin_step(s.seqs, p.new, rope_pos=s.rope_pos, tree_bits=s.bits)
    else:
        cache.begin_step(s.seqs, p.new)
    if kind == "layer":
        hid = p.c["hidden"]
        for i in range(p.L):
            q, gate, out = _ptr(s.q, i), _ptr(s.gate, i), _ptr(s.out, i)
            cache.project_append(i, _ptr(x["x"], i), hid, _ptr(x["w_q"], i), _ptr(x["w_kv"], i),
                                 _ptr(x["q_norm"], i), _ptr(x["k_norm"], i), *tables, q, q_gate_out=gate)
            (cache.decode if p.c["new_hi"] == 1 else cache.prefill)(i, q, out, gate=gate)
            cache.out_project(out, p.T, p.H * D, _ptr(x["w_o"], i), hid, _ptr(s.y, i),
                              residual=_ptr(x["residual"], i))
        return {"q": s.q, "gate": s.gate, "out": s.out, "y": s.y, "k": s.tail_k, "v": s.tail_v}
    s.q.copy_(x["q"])  # the calls rotate q in place: the projection's fresh rows
    if kind == "tree":
        s.k.copy_(x["k"])
    for i in range(p.L):
        q, out = _ptr(s.q, i), _ptr(s.out, i)
        gate = _ptr(x["gate"], i) if x["gate"] is not None else None
        norms = (_ptr(x["q_norm"], i), _ptr(x["k_norm"], i))
        if kind == "tree":
            cache.append(i, q, _ptr(s.k, i), _ptr(x["v"], i), *norms, *tables)
            cache.tree_verify(i, q, out, gate=gate)
        else:
            call = cache.append_decode if kind == "decode" else cache.append_prefill
            call(i, q, _ptr(x["k"], i), _ptr(x["v"], i), *norms, *tables, out, gate=gate)
    if kind == "tree":
        cache.rollback(s.seqs, p.base, s.keep)
    return {"q": s.q, "out": s.out, "k": s.tail_k, "v": s.tail_v}


def _seen(p):
    """Rows that each new token attends to, summed over all of them."""
    total = 0
    for b, n in zip(p.base, p.new):
        total += b * n + (sum(d + 1 for d in depths(p.parents)) if p.parents else n * (n + 1) // 2)
    return total


def work(case):
    p = _Plan(case)
    cached = sum(p.base)
    q_row, kv_row = p.H * D * 2, 2 * p.KV * D * 2
    flops = 4.0 * p.H * D * _seen(p)
    if case["kind"] == "layer":
        hid = case["hidden"]
        w_rows = 2 * p.H * D + 2 * p.KV * D
        moved = (w_rows + p.H * D) * hid * 2 + p.T * (3 * hid * 2 + 3 * q_row + kv_row) + cached * kv_row
        flops += 2.0 * p.T * hid * (w_rows + p.H * D)
    else:
        moved = cached * kv_row + p.T * (2 * q_row + 2 * kv_row + q_row + (q_row if case["gate"] else 0))
        if case["kind"] == "tree":
            moved += p.B * 2 * len(p.kept) * kv_row
    return {"bytes": float(p.L * moved), "flops": float(p.L * flops)}


def tolerance(case):
    # fp16 results of 32-bit sums; the attention also rounds its probabilities
    # to fp16.
    return {"rel": 2e-3, "max": 2e-2}


def _tables64(rows):
    freqs = 1.0 / (THETA ** (np.arange(0, HALF_ROT, dtype=np.float32) * 2.0 / (2 * HALF_ROT)))
    ang = np.outer(np.arange(rows, dtype=np.float32), freqs)
    return [torch.from_numpy(f(ang).astype(np.float16)).cuda().double() for f in (np.cos, np.sin)]


def _norm_rope64(x, w, cos, sin):
    """x [T, heads, D], cos/sin [T, HALF_ROT]: RMSNorm, then the rotation of
    the pairs (2i, 2i+1), i < HALF_ROT."""
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w
    a, b = y[..., 0:2 * HALF_ROT:2].clone(), y[..., 1:2 * HALF_ROT:2].clone()
    c, s = cos[:, None, :], sin[:, None, :]
    y[..., 0:2 * HALF_ROT:2] = a * c - b * s
    y[..., 1:2 * HALF_ROT:2] = a * s + b * c
    return y


def _attend64(p, q, k_rows, v_rows, n_old):
    """q [n, H, D] over k_rows, v_rows [n_old + n, KV, D]."""
    n, G = q.shape[0], p.H // p.KV
    seen = torch.ones(n, k_rows.shape[0], dtype=torch.bool, device="cuda")
    if p.parents:
        bits = tree_bits(p.parents)
        seen[:, n_old:] = torch.tensor([[bool(b >> j & 1) for j in range(n)] for b in bits], device="cuda")
    else:
        seen[:, n_old:] = torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
    out = torch.empty_like(q)
    for h in range(p.KV):
        kt = k_rows[:, h].t().contiguous()
        vh = v_rows[:, h].contiguous()
        for g in range(h * G, (h + 1) * G):
            sc = (q[:, g].contiguous() @ kt) / 16.0
            sc.masked_fill_(~seen, float("-inf"))
            out[:, g] = torch.softmax(sc, -1) @ vh
    return out


def exact(case, seed):
    p, x = _inputs(case, seed)
    ids = p.block_ids(seed)
    cos, sin = _tables64(p.rows + 1)
    at = torch.tensor(p.positions(), device="cuda")
    cos, sin = cos[at], sin[at]
    got = {"q": [], "out": [], "gate": [], "y": [], "k": [], "v": []}
    for i in range(p.L):
        if case["kind"] == "layer":
            xs = x["x"][i].double()
            qg = (xs @ x["w_q"][i].double().t()).view(p.T, 2, p.H, D)
            kv = (xs @ x["w_kv"][i].double().t()).view(p.T, 2, p.KV, D)
            q, gate, k, v = qg[:, 0], qg[:, 1].contiguous(), kv[:, 0], kv[:, 1].contiguous()
        else:
            q, k, v = (x[n][i].double() for n in ("q", "k", "v"))
            gate = x["gate"][i].double() if x["gate"] is not None else None
        q = _norm_rope64(q, x["q_norm"][i].double(), cos, sin)
        k = _norm_rope64(k, x["k_norm"][i].double(), cos, sin)
        out = torch.empty_like(q)
        tails = [x[n][i, :p.tail].double() for n in ("k_pool", "v_pool")]
        t = 0
        for b in range(p.B):
            n_old, n = p.base[b], p.new[b]
            blocks = torch.tensor(ids[b], device="cuda")
            new = slice(t, t + n)
            rows = [torch.cat([x[name][i, blocks].reshape(-1, p.KV, D)[:n_old].double(), fresh[new]])
                    for name, fresh in (("k_pool", k), ("v_pool", v))]
            out[new] = _attend64(p, q[new], rows[0], rows[1], n_old)
            slots = torch.arange(n_old, n_old + n, device="cuda")
            for pool, fresh in zip(tails, (k, v)):
                pool[blocks[slots // PAGE], slots % PAGE] = fresh[new]
                if p.parents:  # the accepted path's rows move up behind the cached ones
                    m = len(p.kept)
                    pool[blocks[slots[:m] // PAGE], slots[:m] % PAGE] = fresh[new][torch.tensor(p.kept, device="cuda")]
            t += n
        if gate is not None:
            out = out * torch.sigmoid(gate)
        got["q"].append(q)
        got["out"].append(out)
        got["k"].append(tails[0])
        got["v"].append(tails[1])
        if case["kind"] == "layer":
            got["gate"].append(gate)
            got["y"].append(out.view(p.T, -1) @ x["w_o"][i].double().t() + x["residual"][i].double())
    return {n: torch.stack(v) for n, v in got.items() if v}
