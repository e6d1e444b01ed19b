"""What this framework is timed on: the calls a D2SD decoding loop makes, from one
eager layer call to a batch of long fp8 prefixes.

Kinds of case
  verify  tree-verification attention through CascadeVerifyAttention.plan() / run():
          `layers` calls of one step, each with a KV cache of its own, replayed from
          one HipGraph as a decoding loop does (graph False: the calls are issued
          eagerly, as in a first step or a prompt-by-prompt script)
  step    one whole verify step in one HipGraph: tree build, dynamic-prefix attention
          of every layer, acceptance walk, commit into the paged cache
  dropin  the reference's own call site over the drop-ins (single_prefill_with_kv_cache,
          then CascadeGraphRunner.run, or per-row attention + merge_state_in_place)
  draft   the draft model's shared level: two-segment prefix, block-diagonal mask
  accept  the acceptance walk over the target's logits, greedy or sampled
  rope    QK norm + RoPE of the new tokens of every layer
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "d2-sd_amd"))

import d2sd  # noqa: E402
from d2sd import tree as dtree  # noqa: E402
from d2sd import workloads as wl  # noqa: E402

DEV = "cuda"


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _verify(name, hq, hkv, d, layers, reqs, lo, hi, tree, branches, row_len, page=16, fp8=False, window=0, sinks=False,
            graph=True, shape=0):
    """window > 0: every other layer (the even ones) sees the last `window` prefix keys only."""
    c = dict(kind="verify", hq=hq, hkv=hkv, d=d, layers=layers, reqs=reqs, lo=lo, hi=hi, tree=tree, branches=branches,
             row_len=row_len, page=page, fp8=fp8, window=window, sinks=sinks, graph=graph, shape=shape)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # the smallest call: one layer, one short conversation, issued eagerly (host work and two launches)
        _verify("verify_one_layer_1k", 32, 8, 128, 1, 1, 1024, 1024, "star", 4, 16, page=0, graph=False),
        # the ordinary step of one user: all 36 layers over a 4K cache, the tree that drafting makes (150 nodes)
        _verify("verify_36_layers_4k", 32, 8, 128, 36, 1, 4096, 4096, "d3", 5, 32),
        # a server's ordinary batch: ragged prefixes of a few hundred to 4K keys, small trees
        _verify("verify_batch16_ragged", 32, 8, 128, 4, 16, 300, 4000, "star", 4, 16, shape=5),
        # long contexts: 8 users at 8K to 32K keys (HBM bound)
        _verify("verify_batch8_8k_32k", 32, 8, 128, 1, 8, 8192, 32768, "star", 4, 16),
        # head size 64 with sinks, sliding (128) and full layers in turn, a wide tree
        _verify("verify_d64_sinks_sliding", 64, 8, 64, 24, 1, 8192, 8192, "random", 8, 32, window=128, sinks=True),
        # the largest: a full server batch over an fp8 cache
        _verify("verify_batch32_fp8_8k", 64, 8, 128, 1, 32, 8192, 8192, "random", 8, 32, fp8=True),
        # one whole step of a growing cache, nothing left to the host
        dict(name="whole_step", kind="step", layers=36, prefix=4096, reserve=512, vocab=151936, shape=0),
        # the reference's code with its import swapped: 5 rows of 32 tokens per layer, eager
        dict(name="dropin_call_site", kind="dropin", hq=32, hkv=8, d=128, rows=5, row_len=32, prefix=4096, layers=4,
             runner=True),
        # the draft model's layers: 4 rows of 16 tokens over its cache and the projected context
        dict(name="draft_two_segments", kind="draft", rows=4, row_len=16, cache=4096, ctx=17, layers=8),
        # acceptance over every node's logits, at temperature 0 and sampled
        dict(name="accept_greedy", kind="accept", vocab=151936, tree="d3", branches=5, row_len=32, f32=False, temp=0.0,
             shape=0),
        dict(name="accept_sampled", kind="accept", vocab=151936, tree="d3", branches=5, row_len=32, f32=False,
             temp=0.7, shape=0),
        # QK norm + RoPE of the step's new tokens, every layer
        dict(name="qk_norm_rope_36_layers", kind="rope", tokens=150, hq=32, hkv=8, d=128, layers=36, norm=True,
             half=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


MOST_FLOPS, MOST_BYTES = 6e11, 7e8  # below the largest listed case's


def draw(rng):
    kind = rng.choices(["verify", "dropin", "draft", "accept", "rope", "step"], [10, 1, 1, 2, 2, 1])[0]
    if kind == "verify":
        hq, hkv, d = rng.choice([(32, 8, 128), (32, 8, 128), (64, 8, 128), (64, 8, 64)])
        reqs = _log(rng, 1, 32)
        lo = _log(rng, 100, 24000)
        hi = min(32768, int(lo * rng.uniform(1.0, 4.0)))
        tree = rng.choice(["star", "star", "random", "d3"])
        branches, row_len = rng.randint(2, 8), rng.randint(6, 32)
        if tree == "d3":
            branches, row_len = 5, 32
        fp8 = rng.random() < 0.25
        sliding = d == 64 and rng.random() < 0.5
        c = _verify(None, hq, hkv, d, rng.choice([1, 2, 4, 12, 24, 36]), reqs, lo, hi, tree, branches, row_len,
                    page=rng.choice([0, 16, 16, 16, 32, 64]), fp8=fp8, window=128 if sliding else 0,
                    sinks=d == 64, graph=True, shape=rng.randrange(1 << 16))
        while True:
            w = work(c)
            if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
                return c
            if c["layers"] > 1:
                c["layers"] = max(1, c["layers"] // 2)
            elif c["reqs"] > 1:
                c["reqs"] = max(1, c["reqs"] * 3 // 4)
            else:
                c["lo"], c["hi"] = c["lo"] // 2 + 1, c["hi"] // 2 + 1
    if kind == "step":
        return dict(kind="step", layers=rng.randint(4, 36), prefix=_log(rng, 300, 4500), reserve=rng.randint(64, 700),
                    vocab=rng.choice([32000, 151936]), shape=rng.randrange(1 << 16))
    if kind == "dropin":
        return dict(kind="dropin", hq=32, hkv=8, d=128, rows=rng.randint(1, 8), row_len=rng.randint(8, 40),
                    prefix=_log(rng, 200, 8000), layers=rng.randint(1, 8), runner=rng.random() < 0.7)
    if kind == "draft":
        return dict(kind="draft", rows=rng.randint(1, 8), row_len=rng.randint(8, 32), cache=_log(rng, 100, 8000),
                    ctx=rng.randint(1, 40), layers=rng.randint(1, 12))
    if kind == "accept":
        tree = rng.choice(["d3", "star"])
        branches, row_len = (5, 32) if tree == "d3" else (rng.randint(2, 8), rng.randint(8, 32))
        return dict(kind="accept", vocab=rng.choice([32000, 151936, rng.randint(5000, 200000)]), tree=tree,
                    branches=branches, row_len=row_len, f32=rng.random() < 0.4, temp=rng.choice([0.0, 0.0, 0.6, 1.0]),
                    shape=rng.randrange(1 << 16))
    hq, hkv, d, norm = rng.choice([(32, 8, 128, True), (64, 8, 128, True), (64, 8, 64, False)])
    return dict(kind="rope", tokens=_log(rng, 16, 4600), hq=hq, hkv=hkv, d=d, layers=rng.randint(1, 6), norm=norm,
                half=d == 64)


# ---------------------------------------------------------------------------
# shapes of a case (the same for every seed) and its inputs
# ---------------------------------------------------------------------------
def _tree(case, rng):
    if case["tree"] == "d3":
        return dtree.d3_verify_tree(rng.uniform(0.0, 1.0, size=15), block_size=16, block_size_2=32, topk=4)
    return wl.random_branch_tree(rng, case["branches"], case["row_len"], chain_to_row0=case["tree"] == "star")


def _requests(case):
    rng = np.random.default_rng(case["shape"])
    return [(_tree(case, rng), int(rng.integers(case["lo"], case["hi"] + 1))) for _ in range(case["reqs"])]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.bfloat16)


def _fp8(x, head_axis):
    """Per-kv-head scale (absmax / 448) and the e4m3fn cache."""
    red = [a for a in range(x.dim()) if a not in (0, head_axis)]
    scale = x.float().abs().amax(dim=red).amax(dim=0) / 448.0
    shape = [1] * x.dim()
    shape[head_axis] = scale.numel()
    out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
    for l in range(x.shape[0]):
        out[l] = (x[l:l + 1].float() / scale.view(shape))[0].to(torch.float8_e4m3fn)
    return out, scale


class _Verify:
    """Inputs, plans and (graph) the captured step of a `verify` case."""

    def __init__(self, case, seed, launch=True):
        gen, rng = _gen(seed), np.random.default_rng(seed)
        self.case, self.reqs = case, _requests(case)
        hq, hkv, d, nl, P = case["hq"], case["hkv"], case["d"], case["layers"], case["page"]
        self.qo = [0]
        for t, _ in self.reqs:
            self.qo.append(self.qo[-1] + t.num_nodes)
        T, lens = self.qo[-1], [L for _, L in self.reqs]
        self.page_indptr = self.table = self.tok = None
        if P:
            self.page_indptr = [0]
            for L in lens:
                self.page_indptr.append(self.page_indptr[-1] + -(-L // P))
            n = self.page_indptr[-1]
            self.table = torch.from_numpy(rng.permutation(n).astype(np.int32)).to(DEV)
            shape = (nl, n, hkv, P, d)
        else:
            self.tok = [0]
            for L in lens:
                self.tok.append(self.tok[-1] + L)
            shape = (nl, hkv, self.tok[-1], d)
        self.q, self.ks, self.vs = _randn(gen, nl, T, hq, d), _randn(gen, nl, T, hkv, d), _randn(gen, nl, T, hkv, d)
        self.kp, self.vp = _randn(gen, *shape), _randn(gen, *shape)
        self.kscale = self.vscale = None
        if case["fp8"]:
            self.kp, self.kscale = _fp8(self.kp, 2 if P else 1)
            self.vp, self.vscale = _fp8(self.vp, 2 if P else 1)
        self.sinks = torch.randn(hq, generator=gen, device=DEV) if case["sinks"] else None
        self.masks = [dtree.ancestor_mask(t.parents) for t, _ in self.reqs]
        if not launch:
            return
        self.out = torch.zeros(nl, T, hq, d, dtype=torch.bfloat16, device=DEV)
        self.lse = torch.zeros(nl, T, hq, dtype=torch.float32, device=DEV)
        kw = dict(tree_masks=self.masks, page_size=P, page_indptr=self.page_indptr, page_table=self.table,
                  prefix_tok_indptr=self.tok[:-1] if self.tok else None, sinks=self.sinks,
                  kv_dtype=torch.float8_e4m3fn if case["fp8"] else torch.bfloat16, k_scale=self.kscale,
                  v_scale=self.vscale)
        self.plans = [d2sd.CascadeVerifyAttention(DEV).plan(self.qo, lens, hq, hkv, d, window_left=w, **kw)
                      for w in self.windows()]
        self.graph = None
        if case["graph"]:
            self.calls()
            torch.cuda.synchronize()
            self.graph = d2sd.HipGraph()
            with self.graph.capture():
                self.calls()

    def windows(self):
        return [self.case["window"], -1] if self.case["window"] else [-1]

    def calls(self):
        for l in range(self.case["layers"]):
            self.plans[l % len(self.plans)].run(self.q[l], self.ks[l], self.vs[l], self.kp[l], self.vp[l],
                                                out=self.out[l], lse=self.lse[l])

    def run(self):
        if self.graph is None:
            self.calls()
        else:
            self.graph.replay()
        return {"out": self.out, "lse": self.lse}


class _Step:
    """One captured verify step at a fixed cache length (every replay verifies and commits at the same place)."""

    def __init__(self, case, seed, launch=True):
        gen, rng = _gen(seed), np.random.default_rng(seed)
        hq, hkv, d, P, nl = 32, 8, 128, 16, case["layers"]
        self.case = case
        self.conf = torch.from_numpy(np.random.default_rng(case["shape"]).uniform(0.0, 1.0, size=15)).to(torch.bfloat16)
        self.builder = dtree.D3TreeBuilder(16, 32, 4, DEV)
        cap, rows, lb = self.builder.capacity, self.builder.rows_cap, self.builder.block_size_2
        longest = case["prefix"] + case["reserve"]
        npages = -(-longest // P)
        self.kp, self.vp = _randn(gen, nl, npages, hkv, P, d), _randn(gen, nl, npages, hkv, P, d)
        self.table = torch.from_numpy(rng.permutation(npages).astype(np.int32)).to(DEV)
        self.q, self.ks, self.vs = _randn(gen, nl, cap, hq, d), _randn(gen, nl, cap, hkv, d), _randn(gen, nl, cap, hkv, d)
        if not launch:
            return
        self.logits = _logits(gen, cap, case["vocab"], torch.bfloat16)
        self.builder.build(self.conf.to(DEV))
        self.drafts = _drafts(gen, self.logits, self.builder.node_index.long(), case["vocab"])
        self.out = torch.zeros(nl, cap, hq, d, dtype=torch.bfloat16, device=DEV)
        self.lse = torch.zeros(nl, cap, hq, dtype=torch.float32, device=DEV)
        self.attn = d2sd.CascadeVerifyAttention(DEV).plan(
            [0, cap], [longest], hq, hkv, d, tree_masks=[np.eye(cap, dtype=bool)], page_size=P, page_indptr=[0, npages],
            page_table=self.table, dynamic_prefix=True)
        self.attn.set_prefix_len([case["prefix"]])
        self.acc = d2sd.GreedyAccept(cap, case["vocab"], lb, DEV)
        self.commit = d2sd.PagedKVCommit(list(self.kp), list(self.vp), list(self.ks), list(self.vs))
        conf_dev = self.conf.to(DEV)

        def step():
            self.builder.build(conf_dev, tree_mask=self.attn.tree_mask_dev)
            for l in range(nl):
                self.attn.run(self.q[l], self.ks[l], self.vs[l], self.kp[l], self.vp[l], out=self.out[l], lse=self.lse[l])
            _, nodes, res = self.acc(self.logits, self.builder.node_index, self.drafts)
            self.commit.commit(self.table, self.attn.prefix_len_dev[0:1], nodes, num_accepted=lb, num_accepted_dev=res)

        torch.cuda.synchronize()
        self.graph = d2sd.HipGraph()
        with self.graph.capture():
            step()

    def run(self):
        self.graph.replay()
        return {"out": self.out, "lse": self.lse, "ids": self.acc.accept_ids, "nodes": self.acc.accept_nodes,
                "result": self.acc.result, "mask": self.attn.tree_mask_dev, "k_pool": self.kp, "v_pool": self.vp}


class _Dropin:
    """generation/verification.py:137-165 after `import d2sd as flashinfer`, for some layers of a model."""

    def __init__(self, case, seed):
        gen = _gen(seed)
        b, lb, hq, hkv, d, L, nl = (case[k] for k in ("rows", "row_len", "hq", "hkv", "d", "prefix", "layers"))
        self.case = case
        self.q, self.kn, self.vn = (_randn(gen, nl, b, h, lb, d) for h in (hq, hkv, hkv))
        self.k, self.v = _randn(gen, nl, hkv, L, d), _randn(gen, nl, hkv, L, d)
        self.scale = d ** -0.5
        self.runner = d2sd.CascadeGraphRunner(lb, hq, hkv, d, torch.bfloat16, torch.device(DEV), self.scale, causal=True)

    def run(self):
        c = self.case
        b, lb, hq, d = c["rows"], c["row_len"], c["hq"], c["d"]
        outs, lses = [], []
        for l in range(c["layers"]):
            k_fi, v_fi = self.k[l].transpose(0, 1).contiguous(), self.v[l].transpose(0, 1).contiguous()
            q_fi = self.q[l].transpose(1, 2).contiguous()
            k_new, v_new = self.kn[l].transpose(1, 2).contiguous(), self.vn[l].transpose(1, 2).contiguous()
            out, lse = d2sd.single_prefill_with_kv_cache(q_fi.view(b * lb, hq, d), k_fi, v_fi, causal=False,
                                                         return_lse=True, sm_scale=self.scale)
            out, lse = out.view(b, lb, hq, d), lse.view(b, lb, hq)
            if c["runner"]:
                self.runner.run(q_fi, k_new, v_new, out, lse)
            else:
                for r in range(b):
                    o, s = d2sd.single_prefill_with_kv_cache(q_fi[r], k_new[r], v_new[r], causal=True, return_lse=True,
                                                             sm_scale=self.scale)
                    d2sd.merge_state_in_place(out[r], lse[r], o, s)
            outs.append(out)
            lses.append(lse)
        return {"out": outs, "lse": lses}


class _Draft:
    """model/dflash.py:96-133 over plan() / run(): [draft cache | projected context] read in place."""

    def __init__(self, case, seed, launch=True):
        gen = _gen(seed)
        hq, hkv, d = 32, 8, 128
        b, lb, lc, ctx, nl = (case[k] for k in ("rows", "row_len", "cache", "ctx", "layers"))
        n = b * lb
        self.case = case
        self.q, self.ks, self.vs = _randn(gen, nl, n, hq, d), _randn(gen, nl, n, hkv, d), _randn(gen, nl, n, hkv, d)
        self.kc, self.vc = _randn(gen, nl, 1, hkv, lc + 256, d), _randn(gen, nl, 1, hkv, lc + 256, d)
        self.kx, self.vx = _randn(gen, nl, hkv, ctx + lb, d), _randn(gen, nl, hkv, ctx + lb, d)
        self.mask = np.kron(np.eye(b, dtype=bool), np.ones((lb, lb), dtype=bool))
        if not launch:
            return
        self.out = torch.zeros(nl, n, hq, d, dtype=torch.bfloat16, device=DEV)
        self.lse = torch.zeros(nl, n, hq, dtype=torch.float32, device=DEV)
        self.plan = d2sd.CascadeVerifyAttention(DEV).plan([0, n], [lc + ctx], hq, hkv, d, tree_masks=[self.mask],
                                                          page_size=0, prefix_split=[lc])

        def calls():
            for l in range(nl):
                self.plan.run(self.q[l], self.ks[l], self.vs[l], (self.kc[l], self.kx[l][:, :ctx]),
                              (self.vc[l], self.vx[l][:, :ctx]), out=self.out[l], lse=self.lse[l])

        calls()
        torch.cuda.synchronize()
        self.graph = d2sd.HipGraph()
        with self.graph.capture():
            calls()

    def run(self):
        self.graph.replay()
        return {"out": self.out, "lse": self.lse}


def _logits(gen, n, vocab, dtype):
    """A language model's logits: a broad bulk and, per node, a few dozen likely tokens above it."""
    x = torch.randn((n, vocab), generator=gen, device=DEV) * 2.5
    top = torch.randint(0, vocab, (n, min(48, vocab)), generator=gen, device=DEV)
    lift = 18.0 - 4.0 * torch.rand(top.shape, generator=gen, device=DEV) * torch.arange(
        1, top.shape[1] + 1, device=DEV).float().log()
    return x.scatter(1, top, lift).to(dtype)


def _drafts(gen, logits, node_index, vocab):
    """Draft tokens that follow the target for some positions of each row."""
    am = logits.argmax(-1)
    d = torch.randint(0, vocab, tuple(node_index.shape), generator=gen, device=DEV)
    d[:, 1:] = torch.where(torch.rand(d[:, 1:].shape, generator=gen, device=DEV) < 0.85, am[node_index[:, :-1]], d[:, 1:])
    return d


class _Accept:
    def __init__(self, case, seed):
        gen = _gen(seed)
        t = _tree(case, np.random.default_rng(case["shape"]))
        self.logits = _logits(gen, t.num_nodes, case["vocab"], torch.float32 if case["f32"] else torch.bfloat16)
        self.node_index = torch.from_numpy(np.ascontiguousarray(t.node_index, dtype=np.int32)).to(DEV)
        self.drafts = _drafts(gen, self.logits, self.node_index.long(), case["vocab"])
        self.acc = d2sd.TreeAccept(t.num_nodes, case["vocab"], t.row_len, DEV, temperature=case["temp"], seed=int(seed))

    def run(self):
        ids, nodes, res = self.acc(self.logits, self.node_index, self.drafts)
        return {"ids": ids, "nodes": nodes, "result": res, "node_tokens": self.acc.node_tokens}


class _Rope:
    """In place on the fused projection output [tokens, Hq + 2 Hkv, D] of every layer."""

    def __init__(self, case, seed, launch=True):
        gen = _gen(seed)
        n, hq, hkv, d, nl = (case[k] for k in ("tokens", "hq", "hkv", "d", "layers"))
        self.case = case
        self.qkv = _randn(gen, nl, n, hq + 2 * hkv, d)
        w = torch.rand((nl, 2, d), generator=gen, device=DEV) + 0.5
        self.w = w.to(torch.bfloat16) if case["norm"] else None
        inv = 1.0 / (1e6 ** (torch.arange(0, d, 2, device=DEV).float() / d))
        ang = (torch.arange(n, device=DEV) + 4096)[:, None].float() * inv[None]
        emb = ang if case["half"] else torch.cat([ang, ang], -1)
        self.cos, self.sin = emb.cos().to(torch.bfloat16), emb.sin().to(torch.bfloat16)
        if not launch:
            return
        stream_in = self.qkv.clone()

        def calls():
            for l in range(nl):
                d2sd.qk_norm_rope(self.qkv[l][:, :hq], self.qkv[l][:, hq:hq + hkv], self.w[l, 0] if case["norm"] else None,
                                  self.w[l, 1] if case["norm"] else None, self.cos, self.sin)

        calls()
        torch.cuda.synchronize()
        self.graph = d2sd.HipGraph()
        with self.graph.capture():
            calls()
        self.qkv.copy_(stream_in)

    def run(self):
        self.graph.replay()
        return {"qkv": self.qkv}


_KINDS = {"verify": _Verify, "step": _Step, "dropin": _Dropin, "draft": _Draft, "accept": _Accept, "rope": _Rope}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------------------
# work, tolerance, 64-bit results
# ---------------------------------------------------------------------------
def _attn_work(hq, hkv, d, pairs, prefix_keys, new_keys, queries, kv_bytes, extra=0):
    """Visible (query, key) pairs of one layer; each key and value, query, output and LSE once."""
    return {"bytes": 2 * hkv * d * (prefix_keys * kv_bytes + new_keys * 2) + queries * hq * (4 * d + 4) + extra,
            "flops": 4 * hq * d * pairs}


def work(case):
    k = case["kind"]
    if k == "verify":
        reqs = _requests(case)
        total = {"bytes": 0, "flops": 0}
        for l in range(case["layers"]):
            w = case["window"] if case["window"] and l % 2 == 0 else None
            pairs = keys = new = extra = 0
            for t, L in reqs:
                n, vis = t.num_nodes, L if w is None else min(L, w)
                anc = int(dtree.ancestor_mask(t.parents).sum()) if n <= 512 else n * 16
                pairs, keys, new = pairs + n * vis + anc, keys + vis, new + n
                extra += n * ((n + 63) // 64) * 8 + (4 * -(-vis // case["page"]) if case["page"] else 0)
            one = _attn_work(case["hq"], case["hkv"], case["d"], pairs, keys, new, new, 1 if case["fp8"] else 2, extra)
            total = {x: total[x] + one[x] for x in total}
            if not case["window"]:
                return {x: one[x] * case["layers"] for x in one}
        return total
    if k == "step":
        conf = np.random.default_rng(case["shape"]).uniform(0.0, 1.0, size=15)
        t = dtree.d3_verify_tree(conf, block_size=16, block_size_2=32, topk=4)
        n = t.num_nodes
        a = _attn_work(32, 8, 128, n * case["prefix"] + int(dtree.ancestor_mask(t.parents).sum()), case["prefix"], n, n, 2)
        return {"bytes": case["layers"] * a["bytes"] + n * case["vocab"] * 2, "flops": case["layers"] * a["flops"]}
    if k == "dropin":
        n = case["rows"] * case["row_len"]
        pairs = n * case["prefix"] + case["rows"] * case["row_len"] * (case["row_len"] + 1) // 2
        a = _attn_work(case["hq"], case["hkv"], case["d"], pairs, case["prefix"], n, n, 2)
        return {x: a[x] * case["layers"] for x in a}
    if k == "draft":
        n, L = case["rows"] * case["row_len"], case["cache"] + case["ctx"]
        a = _attn_work(32, 8, 128, n * L + case["rows"] * case["row_len"] ** 2, L, n, n, 2)
        return {x: a[x] * case["layers"] for x in a}
    if k == "accept":
        t = _tree(case, np.random.default_rng(case["shape"]))
        return {"bytes": t.num_nodes * case["vocab"] * (4 if case["f32"] else 2), "flops": 0}
    rows, d = case["tokens"] * (case["hq"] + case["hkv"]), case["d"]
    return {"bytes": case["layers"] * (4 * rows * d + 4 * case["tokens"] * d), "flops": case["layers"] * rows * d * 8}


def tolerance(case):
    if case["kind"] == "accept":
        return "exact"
    if case["kind"] == "rope":
        # bf16 rounding steps; another order of the 32-bit sum of squares turns a few of them
        return {"rel": 2e-3, "max": 3e-2}
    # bf16 outputs of 32-bit sums; probabilities and partial outputs rounded to bf16 in another order
    return {"rel": 1e-2, "max": 8e-2}


def _attend(q, k, v, scale, visible=None, sinks=None):
    """64-bit attention: q [n, Hq, D], k / v [L, Hkv, D]; visible [n, L] or None.  (out, lse)"""
    n, hq, d = q.shape
    g = hq // k.shape[1]
    out = torch.empty(n, hq, d, dtype=torch.float64, device=q.device)
    lse = torch.empty(n, hq, dtype=torch.float64, device=q.device)
    for h in range(k.shape[1]):
        kk, vv = k[:, h].double(), v[:, h].double()
        s = (q[:, h * g:(h + 1) * g].double().reshape(n * g, d) @ kk.T).view(n, g, -1) * scale
        if visible is not None:
            s = s.masked_fill(~visible[:, None, :], float("-inf"))
        m = s.amax(-1, keepdim=True)
        p = (s - m).exp()
        z = p.sum(-1, keepdim=True)
        out[:, h * g:(h + 1) * g] = ((p / z).reshape(n * g, -1) @ vv).view(n, g, d)
        lse[:, h * g:(h + 1) * g] = (m + z.log())[..., 0]
    if sinks is not None:
        out *= torch.sigmoid(lse - sinks.double()[None]).unsqueeze(-1)
    return out, lse


def _tree_attend(q, ks, vs, kp, vp, mask, scale, sinks=None):
    vis = torch.cat([torch.ones(q.shape[0], kp.shape[0], dtype=torch.bool, device=q.device),
                     torch.as_tensor(mask, device=q.device)], 1)
    return _attend(q, torch.cat([kp.double(), ks.double()]), torch.cat([vp.double(), vs.double()]), scale, vis, sinks)


def _exact_verify(case, seed):
    s = _Verify(case, seed, launch=False)
    hq, hkv, d, nl, P = case["hq"], case["hkv"], case["d"], case["layers"], case["page"]
    out = torch.empty(nl, s.qo[-1], hq, d, dtype=torch.float64, device=DEV)
    lse = torch.empty(nl, s.qo[-1], hq, dtype=torch.float64, device=DEV)
    for l in range(nl):
        w = case["window"] if case["window"] and l % 2 == 0 else None
        for r, (t, L) in enumerate(s.reqs):
            def prefix(pool, scale):
                if P:
                    pg = s.table[s.page_indptr[r]:s.page_indptr[r + 1]].long()
                    x = pool[l].view(torch.uint8)[pg].view(pool.dtype) if case["fp8"] else pool[l][pg]
                    x = x.double().permute(0, 2, 1, 3).reshape(-1, hkv, d)[:L]
                else:
                    x = pool[l][:, s.tok[r]:s.tok[r] + L].double().transpose(0, 1)
                x = x if scale is None else x * scale.double()[None, :, None]
                return x if w is None else x[max(0, L - w):]
            a, b = s.qo[r], s.qo[r + 1]
            out[l, a:b], lse[l, a:b] = _tree_attend(s.q[l, a:b], s.ks[l, a:b], s.vs[l, a:b], prefix(s.kp, s.kscale),
                                                    prefix(s.vp, s.vscale), s.masks[r], d ** -0.5, s.sinks)
    return {"out": out, "lse": lse}


def _exact_step(case, seed):
    s = _Step(case, seed, launch=False)
    t = dtree.d3_verify_tree(s.conf.float().numpy(), block_size=16, block_size_2=32, topk=4)
    cap = s.builder.capacity
    if t.num_nodes > cap:
        return None
    s.builder.build(s.conf.to(DEV))
    if int(s.builder.num_nodes[0]) != t.num_nodes or not np.array_equal(
            s.builder.parents[:t.num_nodes].cpu().numpy(), t.parents):
        return None  # rates that tie in bf16: the device's tree is another one
    mask = dtree.padded_ancestor_mask(t, cap)
    L, out, lse = case["prefix"], [], []
    for l in range(case["layers"]):
        kp, vp = (x[l][s.table.long()].permute(0, 2, 1, 3).reshape(-1, 8, 128)[:L] for x in (s.kp, s.vp))
        o, z = _tree_attend(s.q[l], s.ks[l], s.vs[l], kp, vp, mask, 128 ** -0.5)
        out.append(o)
        lse.append(z)
    return {"out": torch.stack(out), "lse": torch.stack(lse), "ids": None, "nodes": None, "result": None, "mask": None,
            "k_pool": None, "v_pool": None}


def _exact_dropin(case, seed):
    s = _Dropin(case, seed)
    lb = case["row_len"]
    causal = torch.ones(lb, lb, dtype=torch.bool).tril()
    outs, lses = [], []
    for l in range(case["layers"]):
        kp, vp = s.k[l].transpose(0, 1), s.v[l].transpose(0, 1)
        rows = [_tree_attend(s.q[l, r].transpose(0, 1), s.kn[l, r].transpose(0, 1), s.vn[l, r].transpose(0, 1), kp, vp,
                             causal, s.scale) for r in range(case["rows"])]
        outs.append(torch.stack([o for o, _ in rows]))
        lses.append(torch.stack([z for _, z in rows]))
    return {"out": outs, "lse": lses}


def _exact_draft(case, seed):
    s = _Draft(case, seed, launch=False)
    lc, ctx, out, lse = case["cache"], case["ctx"], [], []
    for l in range(case["layers"]):
        kp = torch.cat([s.kc[l, 0, :, :lc], s.kx[l][:, :ctx]], 1).transpose(0, 1)
        vp = torch.cat([s.vc[l, 0, :, :lc], s.vx[l][:, :ctx]], 1).transpose(0, 1)
        o, z = _tree_attend(s.q[l], s.ks[l], s.vs[l], kp, vp, s.mask, 128 ** -0.5)
        out.append(o)
        lse.append(z)
    return {"out": torch.stack(out), "lse": torch.stack(lse)}


def _exact_rope(case, seed):
    s = _Rope(case, seed, launch=False)
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    x = s.qkv.double()
    h = x[:, :, :hq + hkv]
    if case["norm"]:
        w = torch.cat([s.w[:, 0:1].expand(-1, hq, -1), s.w[:, 1:2].expand(-1, hkv, -1)], 1).double()
        h = h / torch.sqrt((h * h).mean(-1, keepdim=True) + 1e-6) * w[:, None]
    cos, sin = s.cos.double(), s.sin.double()
    if case["half"]:
        cos, sin = torch.cat([cos, cos], -1), torch.cat([sin, sin], -1)
    rot = torch.cat([-h[..., d // 2:], h[..., :d // 2]], -1)
    x[:, :, :hq + hkv] = h * cos[None, :, None] + rot * sin[None, :, None]
    return {"qkv": x}


def exact(case, seed):
    f = {"verify": _exact_verify, "step": _exact_step, "dropin": _exact_dropin, "draft": _exact_draft,
         "rope": _exact_rope}.get(case["kind"])
    return f(case, seed) if f else None
