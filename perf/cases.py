"""Performance cases of the KV-cache decode path: what is timed, on which inputs.

A case is a dict of plain values.  listed() names the fixed ones, draw(rng)
gives another of the same ranges, prepare(case, seed) builds its inputs on the
GPU, run(state) makes one pass through the library's public Python entry
points, exact(case, seed) is the same result in 64-bit torch, work(case) the
bytes and operations a pass cannot do without, tolerance(case) the error that
another correct implementation at the same precision may show.

Kinds of case:
  step       one decode step of `layers` layers: append + seal, score + select,
             sparse attention (sa.decode_step), one HIP graph per step as a
             serving loop launches it
  layer      the same with the query producer before it and the o-projection
             and residual after it (sa.decode_step_qkv, sa.linear), chained
  mixed      a batch of very different contexts and budgets: append + seal,
             chunked selection, chunked attention
  seal       the bulk seal after a prefill (sa.seal)
  represent  the InfLLM representatives of a prefill
             (sa.local_causal_representatives)
  dense      attention over a contiguous KV buffer (sa.attention_contiguous)
"""
from __future__ import annotations

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "solidattention-repro_amd"))

import solidattention_amd as sa  # noqa: E402

PAGE = 32
RMS_EPS = 1e-6
THETA = 1e6


def _step(name, batch, query_heads, kv_heads, context, budget, init, local, layers, head_dim=128, ragged=True,
          shared=False, online=False, half_tokens=False, outliers=False):
    return {"name": name, "kind": "step", "batch": batch, "query_heads": query_heads, "kv_heads": kv_heads,
            "head_dim": head_dim, "context": context, "budget": budget, "init": init, "local": local,
            "layers": layers, "ragged": ragged, "shared": shared, "online": online, "half_tokens": half_tokens,
            "outliers": outliers}


def listed():
    return [
        # one user, a short context, the reference's shared selection (one block set over all heads), every
        # layer of a 28-layer model: launches and latency count
        _step("step-1x2k-shared", 1, 16, 8, 2048, 16, 1, 2, 28, ragged=False, shared=True),
        # a few users of an InfLLM-style decode: per-query-head representatives, built online; in this step the
        # blocks of two of the sequences seal
        _step("step-4x8k-online", 4, 16, 8, 8191, 64, 4, 8, 2, online=True),
        # the headline of bench.py: 64 sequences of 16K tokens, 16 query heads on 8 KV heads
        _step("step-64x16k", 64, 16, 8, 16384, 64, 4, 8, 2, ragged=False),
        # the larger model of bench.py: 32 query heads on 8 KV heads, 32K contexts, raw FP16 tokens appended,
        # a few large key channels
        _step("step-32x32k-gqa4", 32, 32, 8, 32768, 64, 4, 8, 2, half_tokens=True, outliers=True),
        # 64 query heads on 8 KV heads (the widest group), a ragged batch
        _step("step-16x16k-gqa8", 16, 64, 8, 16384, 64, 4, 8, 4),
        # a smaller head dimension, ragged contexts
        _step("step-32x10k-hd64", 32, 16, 8, 10000, 64, 4, 8, 4, head_dim=64),
        # few sequences of a very long context (the miss-correction shape): long lists, a large budget
        _step("step-8x128k-gqa4", 8, 32, 8, 131072, 128, 4, 8, 2),
        # a decode layer as a model runs it: norm, q/k/v, decode step, o-projection, residual
        {"name": "layer-16x8k", "kind": "layer", "batch": 16, "query_heads": 16, "kv_heads": 8, "head_dim": 128,
         "context": 8192, "budget": 64, "init": 4, "local": 8, "layers": 4, "ragged": True, "hidden": 1024},
        # serving with mixed contexts (1K to 64K) and mixed budgets (512 tokens, 2048 tokens, everything)
        {"name": "mixed-128x64k", "kind": "mixed", "batch": 128, "query_heads": 16, "kv_heads": 8, "head_dim": 128,
         "context": 65536, "init": 4, "local": 8, "chunk": 128, "layers": 1},
        # the representatives of every whole block once a prefill has filled the pages
        {"name": "seal-64x16k", "kind": "seal", "batch": 64, "query_heads": 16, "kv_heads": 8, "head_dim": 128,
         "context": 16384, "ragged": False},
        # the InfLLM representatives of one 16K-token prompt
        {"name": "represent-16k", "kind": "represent", "query_heads": 16, "kv_heads": 8, "head_dim": 128,
         "context": 16384, "window": 32, "topk": 4},
        # the accelerator backend's dense attention of one query over a whole context of odd length
        {"name": "dense-20001", "kind": "dense", "query_heads": 32, "kv_heads": 8, "head_dim": 128,
         "context": 20001},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, then its sizes over their ranges (log-uniform where they span more than a factor of ten)."""
    kind = rng.choice(["step"] * 6 + ["layer", "mixed", "seal", "represent", "dense"])
    kv_heads = rng.choice([4, 8])
    group = rng.choice([1, 2, 4, 8])
    if kind == "represent":
        head_dim = rng.choice([128, 128, 64])
        return {"kind": kind, "query_heads": kv_heads * min(group, 4 if head_dim == 128 else 2), "kv_heads": kv_heads,
                "head_dim": head_dim, "context": PAGE * _log(rng, 8, 512),
                "window": rng.choice([16, 32, 64]), "topk": rng.choice([1, 4, 8])}
    if kind == "dense":
        return {"kind": kind, "query_heads": kv_heads * group, "kv_heads": kv_heads,
                "head_dim": rng.choice([128, 128, 64, 256]), "context": _log(rng, 100, 60000)}
    batch = _log(rng, 1, 64)
    context = _log(rng, 600, min(131072, 2 ** 20 // batch))
    if kind == "seal":
        return {"kind": kind, "batch": batch, "query_heads": kv_heads * group, "kv_heads": kv_heads,
                "head_dim": rng.choice([128, 128, 64]), "context": context, "ragged": True}
    if kind == "mixed":
        return {"kind": kind, "batch": max(batch, 8), "query_heads": kv_heads * group, "kv_heads": kv_heads,
                "head_dim": 128, "context": min(_log(rng, 8000, 65536), 2 ** 21 // max(batch, 8)), "init": 4,
                "local": 8, "chunk": rng.choice([64, 128]), "layers": 1}
    budget, init, local = rng.choice([(16, 1, 2), (32, 4, 8), (64, 4, 8), (96, 4, 8), (128, 4, 8)])
    layers = max(1, min(8, 2 ** 19 // (batch * context)))
    if kind == "layer":
        return {"kind": kind, "batch": batch, "query_heads": kv_heads * group, "kv_heads": kv_heads, "head_dim": 128,
                "context": context, "budget": budget, "init": init, "local": local, "layers": min(layers, 4),
                "ragged": True, "hidden": rng.choice([1024, 2048])}
    online = rng.random() < 0.15
    shared = not online and rng.random() < 0.15
    head_dim = 128 if online else rng.choice([128, 128, 128, 64, 256])
    if shared:  # a selection group is at most 32 query heads
        group = min(group, 32 // kv_heads)
    c = _step("", batch, kv_heads * group, kv_heads, context, budget, init, local,
              min(layers, 2) if online else layers, head_dim=head_dim,
              shared=shared, online=online, half_tokens=not online and rng.random() < 0.3,
              outliers=rng.random() < 0.3)
    del c["name"]
    return c


# ---- inputs (plain torch, from the seed alone) ------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _spread(n, lo, hi):
    return [hi if n == 1 else int(lo + (hi - lo) * i / (n - 1)) for i in range(n)]


def _lengths(c):
    """The context lengths of a batch, as a multiset (prepare() deals them out by the seed)."""
    n, context = c["batch"], c["context"]
    if c["kind"] == "mixed":
        return _spread(n, min(1024, context // 4), context)
    return _spread(n, context // 2, context) if c["ragged"] else [context] * n


def _budgets(c):
    """mixed: a third of the sequences each take 16 blocks, 64 blocks and every block."""
    stride = (c["context"] + 1) // PAGE
    return [min(16, stride), min(64, stride), stride], stride


def _normal(g, shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=g)


def _paged_inputs(c, seed):
    """Page pools, tables, lengths and the step's queries and tokens.  Keys of 8 blocks per (sequence, KV head)
    lean towards the queries, as the blocks that a real selection finds do."""
    g = _gen(seed)
    L, B, hq, hkv, d = c.get("layers", 1), c["batch"], c["query_heads"], c["kv_heads"], c["head_dim"]
    longest = c["context"]
    stride = (longest + 1 + PAGE - 1) // PAGE + 1
    lengths = torch.tensor(_lengths(c), dtype=torch.int32, device="cuda")
    lengths = lengths[torch.randperm(B, generator=g, device="cuda")]
    need = (lengths + 1 + PAGE - 1) // PAGE
    total = int(need.sum()) + 8
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    first = torch.cumsum(need, 0) - need
    col = torch.arange(stride, device="cuda")
    index = (first[:, None] + col[None, :]).clamp(max=total - 1)
    table = torch.where(col[None, :] < need[:, None], perm[index], torch.zeros_like(perm[index])).to(torch.int32)
    pool = _normal(g, (L, total, PAGE, 2, hkv, d), torch.float16)
    x = {"g": g, "lengths": lengths, "table": table.contiguous(), "pool": pool, "stride": stride, "pages": total}
    x["q"] = _normal(g, (L, B, hq, d))
    x["k"], x["v"] = _normal(g, (L, B, hkv, d)), _normal(g, (L, B, hkv, d))
    planted = 8
    full = int(lengths.min()) // PAGE
    if c["kind"] in ("step", "mixed") and full >= planted:
        blocks = torch.rand((B, hkv, full), generator=g, device="cuda").argsort(dim=-1)[..., :planted]
        pages = torch.gather(table.to(torch.int64), 1, blocks.reshape(B, -1)).reshape(-1)
        heads = torch.arange(hkv, device="cuda").view(1, hkv, 1).expand(B, hkv, planted).reshape(-1)
        for l in range(L):
            mean = x["q"][l].view(B, hkv, hq // hkv, d).mean(dim=2)
            noise = _normal(g, (B, hkv, planted, PAGE, d))
            keys = (0.5 * mean[:, :, None, None, :] + 0.5 * noise).to(torch.float16)
            pool[l][pages, :, 0, heads, :] = keys.reshape(-1, PAGE, d)
    if c.get("outliers"):  # a few key channels of large magnitude, as post-RoPE keys have
        pool[:, :, :, 0, :, :4] *= 8.0
        x["k"][..., :4] *= 8.0
    if c.get("half_tokens"):
        x["k"], x["v"] = x["k"].to(torch.float16), x["v"].to(torch.float16)
    return x


def _layer_inputs(c, seed):
    x = _paged_inputs(c, seed)
    g, L, B, hq, hkv, d, hidden = x["g"], c["layers"], c["batch"], c["query_heads"], c["kv_heads"], 128, c["hidden"]
    x["h0"] = _normal(g, (B, hidden))
    x["w"] = [{"inorm": 1 + 0.1 * _normal(g, (hidden,)), "qn": 1 + 0.1 * _normal(g, (d,)),
               "kn": 1 + 0.1 * _normal(g, (d,)), "wq": _normal(g, (hq * d, hidden)) * hidden ** -0.5,
               "wk": _normal(g, (hkv * d, hidden)) * hidden ** -0.5,
               "wv": _normal(g, (hkv * d, hidden)) * hidden ** -0.5,
               "wo": _normal(g, (hidden, hq * d)) * (hq * d) ** -0.5} for _ in range(L)]
    return x


def _prompt_inputs(c, seed):
    g = _gen(seed)
    kv = _normal(g, (c["context"], 2, c["kv_heads"], c["head_dim"]), torch.float16)
    if c["kind"] == "dense":
        return {"kv": kv, "q": _normal(g, (c["query_heads"], c["head_dim"]))}
    return {"kv": kv, "q": _normal(g, (c["query_heads"], c["context"], c["head_dim"]))}


# ---- states and passes ------------------------------------------------------

def _scale(d):
    return float(torch.tensor(d, dtype=torch.float32).rsqrt())


class _Decode:
    """The device state of a decode loop, and one step of it as a HIP graph.  The step first sets the lengths and
    seal counters back, so that every pass decodes the same token."""

    def __init__(self, c, seed):
        x = _layer_inputs(c, seed) if c["kind"] == "layer" else _paged_inputs(c, seed)
        self.c, self.x = c, x
        L, B, hq, hkv, d = c.get("layers", 1), c["batch"], c["query_heads"], c["kv_heads"], c["head_dim"]
        self.layers = L
        rep_heads = hq if c.get("online") else hkv
        rep_stride = sa.default_rep_stride(x["stride"])
        # [layer][length, sealed, generation][sequence]
        self.base = torch.zeros((L, 3, B), dtype=torch.int32, device="cuda")
        self.base[:, 0] = x["lengths"]
        self.live = self.base.clone()
        self.reps = torch.zeros((L, B, rep_heads, d, rep_stride), dtype=torch.float32, device="cuda")
        self.kvs = []
        for l in range(L):
            kv = sa.PagedKV(B, hq, hkv, x["stride"], num_pages=x["pages"], rep_heads=rep_heads, rep_stride=rep_stride,
                            head_dim=d, pool=x["pool"][l].view(torch.uint16))
            kv.block_table, kv.reps = x["table"], self.reps[l]
            kv.seq_len, kv.sealed, kv.generation = self.live[l, 0], self.live[l, 1], self.live[l, 2]
            self.kvs.append(kv)
        self.status = torch.zeros(1, dtype=torch.int32, device="cuda")
        if c["kind"] == "seal":
            return
        for kv in self.kvs:  # the prefill's blocks
            sa.seal(kv, 0, status=self.status)
        self.base.copy_(self.live)
        groups = 1 if c.get("shared") else hkv
        self.groups = groups
        budget = _budgets(c)[1] if c["kind"] == "mixed" else c["budget"]
        self.selected = torch.full((L, B, groups, budget), -1, dtype=torch.int32, device="cuda")
        self.counts = torch.zeros((L, B, groups), dtype=torch.int32, device="cuda")
        self.out = torch.empty((L, B, hq, d), dtype=torch.float32, device="cuda")
        kv = self.kvs[0]
        if c["kind"] == "mixed":
            small, mid, every = _budgets(c)[0]
            classes = torch.arange(B, device="cuda")[torch.randperm(B, generator=x["g"], device="cuda")] % 3
            pick = torch.tensor([small, mid, every], dtype=torch.int32, device="cuda")
            self.budgets = pick[classes].contiguous()
            self.max_chunks = max(2, (budget + 1 + c["chunk"] - 1) // c["chunk"])
            self.select_ws = sa.score_select_chunked_workspace(kv, groups, budget, c["init"], c["local"], budget)[0]
            nbytes = sa.lib().sa_hip_attention_chunked_workspace_bytes(B, hq, hkv, d, self.max_chunks)
            self.ws = torch.zeros(nbytes // 4, dtype=torch.float32, device="cuda")
        else:
            self.splits = sa.select_attend_default_splits(kv, groups, budget)
            self.ws = sa.decode_step_workspace(kv, self.splits)[0]
        if c.get("online"):
            self.seals = [sa.OnlineSeal(kv) for kv in self.kvs]
            self.rings = _normal(x["g"], (L, *self.seals[0].ring.shape))
            for l, seal in enumerate(self.seals):
                seal.ring = self.rings[l]
        if c["kind"] == "layer":
            hidden = c["hidden"]
            self.h = torch.empty((L + 1, B, hidden), dtype=torch.float32, device="cuda")
            self.h[0].copy_(x["h0"])
            self.qkv_ws = torch.empty(sa.lib().sa_hip_qkv_workspace_bytes(B, hidden, hq, hkv) // 4,
                                      dtype=torch.float32, device="cuda")
            self.lin_ws = torch.empty(max(1, sa.lib().sa_hip_linear_workspace_bytes(B, hq * d, hidden) // 4),
                                      dtype=torch.float32, device="cuda")
        self.k = x["k"].view(torch.uint16) if c.get("half_tokens") else x["k"]
        self.v = x["v"].view(torch.uint16) if c.get("half_tokens") else x["v"]
        self.step()  # the first launches of a program are not captured
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.step()

    def step(self):
        c, x = self.c, self.x
        scale, st = _scale(c["head_dim"]), self.status
        torch.add(self.base, 0, out=self.live)
        for l, kv in enumerate(self.kvs):
            sel, cnt, out = self.selected[l], self.counts[l], self.out[l]
            if c["kind"] == "mixed":
                sa.append_seal(kv, self.k[l], self.v[l], 0, status=st)
                sa.score_select_chunked(kv, x["q"][l], self.groups, sel.shape[2], c["init"], c["local"],
                                        self.select_ws, selected=sel, counts=cnt, status=st, budgets=self.budgets)
                sa.sparse_decode_attention_chunked(kv, x["q"][l], sel, cnt, scale, c["chunk"], self.max_chunks,
                                                   out=out, workspace=self.ws, status=st)
            elif c["kind"] == "layer":
                w = x["w"][l]
                sa.decode_step_qkv(kv, self.h[l], w["wq"], w["wk"], w["wv"], w["qn"], w["kn"], kv.seq_len, x["q"][l],
                                   self.k[l], self.v[l], self.qkv_ws, 0, self.groups, c["budget"], c["init"],
                                   c["local"], scale, self.ws, input_norm=w["inorm"], input_eps=RMS_EPS, theta=THETA,
                                   eps=RMS_EPS, selected=sel, counts=cnt, out=out, splits=self.splits, status=st)
                sa.linear(out.view(c["batch"], -1), w["wo"], self.h[l], out=self.h[l + 1], workspace=self.lin_ws)
            elif c["online"]:
                sa.decode_step_online(kv, self.k[l], self.v[l], 0, x["q"][l], self.seals[l], self.groups, c["budget"],
                                      c["init"], c["local"], scale, self.ws, selected=sel, counts=cnt, out=out,
                                      splits=self.splits, status=st)
            else:
                sa.decode_step(kv, self.k[l], self.v[l], 0, x["q"][l], self.groups, c["budget"], c["init"],
                               c["local"], scale, self.ws, selected=sel, counts=cnt, out=out, splits=self.splits,
                               status=st)

    def outputs(self):
        # the pages as halves where the appended keys are themselves computed, else as whole values
        pool = self.x["pool"] if self.c["kind"] == "layer" else self.x["pool"].view(torch.int16)
        got = {"selected": self.selected, "counts": self.counts, "out": self.out, "pool": pool, "reps": self.reps,
               "state": self.live, "status": self.status}
        if self.c["kind"] == "layer":
            got.update(q=self.x["q"], k=self.k, v=self.v, hidden=self.h)
        if self.c.get("online"):
            got["ring"] = self.rings
        return got


def prepare(case, seed):
    kind = case["kind"]
    if kind not in ("represent", "dense"):
        return _Decode(case, seed)
    x = _prompt_inputs(case, seed)
    x["case"] = case
    if kind == "represent":
        hq, d = case["query_heads"], case["head_dim"]
        x["stride"] = sa.default_rep_stride(case["context"] // PAGE)
        x["reps"] = torch.zeros((hq, d, x["stride"]), dtype=torch.float32, device="cuda")
        nbytes = sa.lib().sa_hip_local_causal_workspace_bytes(case["context"], hq, case["window"])
        x["ws"] = torch.empty(max(nbytes // 4, 1), dtype=torch.float32, device="cuda")
    else:
        x["out"] = torch.empty((case["query_heads"], case["head_dim"]), dtype=torch.float32, device="cuda")
    return x


def run(state):
    if isinstance(state, _Decode):
        if state.c["kind"] == "seal":
            torch.add(state.base, 0, out=state.live)
            sa.seal(state.kvs[0], 0, status=state.status)
            return {"reps": state.reps, "state": state.live, "status": state.status}
        state.graph.replay()
        return state.outputs()
    c = state["case"]
    if c["kind"] == "represent":
        _, offsets = sa.local_causal_representatives(
            state["q"], state["kv"].view(torch.uint16), c["context"], c["query_heads"], c["kv_heads"], c["window"],
            c["topk"], values=False, reps=state["reps"], rep_stride=state["stride"], workspace=state["ws"],
            head_dim=c["head_dim"])
        return {"offsets": offsets, "reps": state["reps"]}
    return {"out": sa.attention_contiguous(state["kv"].view(torch.uint16), state["q"], c["context"],
                                           c["query_heads"], c["kv_heads"], _scale(c["head_dim"]), out=state["out"],
                                           head_dim=c["head_dim"])}


# ---- work and tolerance -----------------------------------------------------

def work(case):
    c = case
    hq, hkv, d, kind = c["query_heads"], c["kv_heads"], c["head_dim"], c["kind"]
    token = 2 * hkv * d * 2  # K and V of a token, FP16
    if kind == "dense":
        return {"bytes": c["context"] * token + 2 * hq * d * 4, "flops": 4 * c["context"] * hq * d}
    if kind == "represent":
        t, w, blocks = c["context"], c["window"], c["context"] // PAGE
        pairs = hq * (t * w - w * (w - 1) // 2)
        return {"bytes": hq * t * d * 4 + t * hkv * d * 2 + hq * blocks * (d * 4 + c["topk"] * 4),
                "flops": 2 * pairs * d}
    lengths = _lengths(c)
    if kind == "seal":
        blocks = sum(n // PAGE for n in lengths)
        return {"bytes": blocks * hkv * d * (PAGE * 2 + 4), "flops": blocks * PAGE * hkv * d}
    if kind == "mixed":
        three, _ = _budgets(c)
        budgets = [three[i % 3] for i in range(len(lengths))]
    else:
        budgets = [c["budget"]] * len(lengths)
    rep_heads = hq if c.get("online") else hkv
    bytes_, flops = 0.0, 0.0
    for i, n in enumerate(lengths):
        sealed, tail = (n + 1) // PAGE, (n + 1) % PAGE
        if kind == "mixed":  # budgets are dealt out by the seed: the mean over the three classes
            taken = sum(min(b, sealed) for b in three) / 3
        else:
            taken = min(budgets[i], sealed)
        scored = sealed if taken < sealed else 0
        attended = taken * PAGE + tail
        bytes_ += scored * rep_heads * d * 4 + attended * token + 2 * hq * d * 4 + 2 * hkv * d * 4 + token
        bytes_ += hkv * taken * 4
        flops += 2 * scored * hq * d + 4 * attended * hq * d
    if kind == "layer":
        heads, hidden, rows = hq + 2 * hkv, c["hidden"], c["batch"]
        bytes_ += (heads + hq) * d * hidden * 4 + rows * 4 * 2 * (2 * hidden + heads * d)
        flops += 2 * rows * hidden * (heads + hq) * d
    return {"bytes": bytes_ * c["layers"], "flops": flops * c["layers"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "seal":
        return "exact"  # sums of FP16 keys in a stated order
    if kind == "represent":
        return "exact"  # the reference's arithmetic, bit for bit
    if kind == "layer":
        # fp32 sums over the hidden width, then softmax sums; an appended key may round to the next FP16 value
        return {"rel": 4e-6, "max": 2e-3}
    # fp32 dot products, exponentials and sums over a few thousand tokens; ids, pages and counters are whole values
    # (measured against 64 bits: 2e-7 to 6.5e-7)
    return {"rel": 4e-6, "max": 2e-4}


# ---- 64-bit results ---------------------------------------------------------

def _softmax_attention(q, k, v, scale):
    """q [heads, G, d], k and v [heads, tokens, d], all float64."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    return torch.matmul(torch.softmax(s, dim=-1), v)


def _select(scores, budget, init, local):
    """Ids [lists][count], ascending: the first `init`, the last `local` and the best of the rest."""
    n = scores.shape[-1]
    if n <= budget:
        return torch.arange(n, device=scores.device).expand(scores.shape)
    s = scores.clone()
    s[:, :init] = math.inf
    s[:, n - local:] = math.inf
    order = torch.sort(s, dim=-1, descending=True, stable=True).indices[:, :budget]
    return order.sort(dim=-1).values


def _exact_step(c, x, l, q, k, v, budgets=None):
    """One layer's step on float64 copies: out and representatives; appends k, v ([B][kv heads][d]) to the pool."""
    B, hq, hkv, d = c["batch"], c["query_heads"], c["kv_heads"], c["head_dim"]
    pool, table, lengths = x["pool"][l], x["table"].long(), x["lengths"].tolist()
    out = torch.empty((B, hq, d), dtype=torch.float64, device="cuda")
    reps = torch.zeros((B, hkv, d, _rep_stride(x["stride"])), dtype=torch.float64, device="cuda")
    heads = torch.arange(hkv, device="cuda")
    for b, n in enumerate(lengths):
        page = table[b, n // PAGE]
        pool[page, n % PAGE, 0], pool[page, n % PAGE, 1] = k[b].to(torch.float16), v[b].to(torch.float16)
        n += 1
        sealed, tail = n // PAGE, n % PAGE
        pages = table[b, :sealed]
        means = torch.empty((sealed, hkv, d), dtype=torch.float64, device="cuda")
        for i in range(0, sealed, 512):
            means[i:i + 512] = pool[pages[i:i + 512], :, 0].double().mean(dim=1)
        reps[b, :, :, :sealed] = means.permute(1, 2, 0)
        qb = q[b].double().view(hkv, hq // hkv, d)
        scores = torch.matmul(qb, means.permute(1, 2, 0).contiguous())  # [hkv, G, sealed]
        scores = scores.mean(dim=(0, 1))[None] if c.get("shared") else scores.mean(dim=1)
        budget = c["budget"] if budgets is None else budgets[b]
        ids = _select(scores, budget, c["init"], c["local"]).expand(hkv, -1)
        where = pages[ids]
        kk = pool[where, :, 0, heads[:, None]].double().reshape(hkv, -1, d)
        vv = pool[where, :, 1, heads[:, None]].double().reshape(hkv, -1, d)
        if tail:
            last = pool[table[b, sealed], :tail].double()
            kk = torch.cat([kk, last[:, 0].transpose(0, 1)], dim=1)
            vv = torch.cat([vv, last[:, 1].transpose(0, 1)], dim=1)
        out[b] = _softmax_attention(qb, kk, vv, d ** -0.5).view(hq, d)
    return out, reps


def _rep_stride(blocks):
    return (blocks + 31) // 32 * 32


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + RMS_EPS) * w.double()


def _rope(x, positions):
    """NeoX pairs (i, i + 64) at fp32 angles position * frequency, frequencies rounded to fp32."""
    freq = torch.pow(torch.tensor(THETA, dtype=torch.float64), -torch.arange(0, 128, 2, dtype=torch.float64) / 128)
    angle = (positions.to(torch.float32)[:, None] * freq.to(torch.float32).cuda()[None]).double()[:, None, :]
    lo, hi = x[..., :64], x[..., 64:]
    return torch.cat([lo * angle.cos() - hi * angle.sin(), hi * angle.cos() + lo * angle.sin()], dim=-1)


def _exact_layer(c, seed):
    x = _layer_inputs(c, seed)
    B, hq, hkv = c["batch"], c["query_heads"], c["kv_heads"]
    h = x["h0"].double()
    got = {"out": [], "reps": [], "q": [], "k": [], "v": [], "hidden": [h]}
    for l in range(c["layers"]):
        w = x["w"][l]
        n = _rms(h, w["inorm"])
        q = _rope(_rms((n @ w["wq"].double().t()).view(B, hq, 128), w["qn"]), x["lengths"])
        k = _rope(_rms((n @ w["wk"].double().t()).view(B, hkv, 128), w["kn"]), x["lengths"])
        v = (n @ w["wv"].double().t()).view(B, hkv, 128)
        out, reps = _exact_step(c, x, l, q, k, v)
        h = h + out.view(B, -1) @ w["wo"].double().t()
        for name, t in (("out", out), ("reps", reps), ("q", q), ("k", k), ("v", v), ("hidden", h)):
            got[name].append(t)
    return {**{name: torch.stack(t) for name, t in got.items()}, "pool": None, "selected": None, "counts": None,
            "state": None, "status": None}


def _exact_represent(c, seed):
    x = _prompt_inputs(c, seed)
    hq, hkv, d, t, w = c["query_heads"], c["kv_heads"], c["head_dim"], c["context"], c["window"]
    blocks = t // PAGE
    reps = torch.zeros((hq, d, _rep_stride(blocks)), dtype=torch.float64, device="cuda")
    back = torch.arange(t, device="cuda")[:, None] - torch.arange(w - 1, -1, -1, device="cuda")[None]  # [t, w] keys
    for h in range(hq):
        k = x["kv"][:, 0, h // (hq // hkv)].double()
        s = torch.empty((t, w), dtype=torch.float64, device="cuda")
        for j in range(w):
            s[:, j] = (x["q"][h].double() * k[back[:, j].clamp(min=0)]).sum(dim=-1) * d ** -0.5
        p = torch.softmax(s.masked_fill(back < 0, -math.inf), dim=-1)
        mass = torch.zeros(t, dtype=torch.float64, device="cuda")
        for j in range(w):
            ok = back[:, j] >= 0
            mass[back[ok, j]] += p[ok, j]  # one query per key for a fixed distance
        best = torch.sort(mass.view(blocks, PAGE), dim=-1, descending=True, stable=True).indices[:, :c["topk"]]
        rows = torch.gather(k.view(blocks, PAGE, d), 1, best[..., None].expand(-1, -1, d))
        reps[h, :, :blocks] = rows.mean(dim=1).t()
    return {"offsets": None, "reps": reps}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "layer":
        return _exact_layer(c, seed)
    if kind == "represent":
        return _exact_represent(c, seed)
    if kind == "dense":
        x = _prompt_inputs(c, seed)
        hq, hkv, d = c["query_heads"], c["kv_heads"], c["head_dim"]
        k, v = (x["kv"][:, i].double().transpose(0, 1).contiguous() for i in (0, 1))
        return {"out": _softmax_attention(x["q"].double().view(hkv, hq // hkv, d), k, v, d ** -0.5).view(hq, d)}
    x = _paged_inputs(c, seed)
    if kind == "seal":
        reps = torch.zeros((1, c["batch"], c["kv_heads"], c["head_dim"], _rep_stride(x["stride"])),
                           dtype=torch.float64, device="cuda")
        for b, n in enumerate(x["lengths"].tolist()):
            pages = x["table"][b, :n // PAGE].long()
            for i in range(0, len(pages), 512):
                means = x["pool"][0][pages[i:i + 512], :, 0].double().mean(dim=1)
                reps[0, b, :, :, i:i + means.shape[0]] = means.permute(1, 2, 0)
        return {"reps": reps, "state": None, "status": None}
    budgets = None
    if kind == "mixed":
        three, _ = _budgets(c)
        B = c["batch"]
        classes = (torch.arange(B, device="cuda")[torch.randperm(B, generator=x["g"], device="cuda")] % 3).tolist()
        budgets = [three[i] for i in classes]
    got = [_exact_step(c, x, l, x["q"][l], x["k"][l], x["v"][l], budgets) for l in range(c["layers"])]
    res = {"out": torch.stack([o for o, _ in got]), "reps": torch.stack([r for _, r in got]), "selected": None,
           "counts": None, "pool": None, "state": None, "status": None}
    if c.get("online"):  # per query head, and a block sealed in the step by the local-causal builder
        res["reps"] = res["ring"] = None
    return res
