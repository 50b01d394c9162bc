"""What is timed when the speed of this package is looked at: the calls a scoring or extraction service makes, through the public
entry points, from one small request to the fullest pass.

A case is a dict of plain values.  Its "kind" says which calls it stands for:

  attn   one layer's attention over a packed stream whose masks are in hand (all layers of a forward share them)
  pass   the attention of a new packed stream: its masks, then one period of a model that alternates five sliding layers and a
         global one (the global layers with one key / value head of 512 dims)
  gdn    one Gated DeltaNet layer between its two projections: path convolution and gates, tree scan, output gate
  head   the lm head's read-out: selected rows of the hidden states to log-probabilities of the option columns
  xdec   one layer of one step of the extraction decoder: the new tokens' keys and values into the cache, then the attention

The shape of the trees belongs to the case; the seed draws the tensors and the order of the contents and of the branches.
"""

from __future__ import annotations

import os
import sys
import zlib

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "spinf-serve_amd"))

import spinf_serve_amd as sa  # noqa: E402
from spinf_serve_amd import decode as xd  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # the headline pass of the benchmark: 24 contents with 56 questions each, one global layer
        _attn("attn_pass", contents=24, trunk=470, branches=56, lo=8, hi=16, hq=16, hkv=8, d=256),
        # a 16k-token stream of a hybrid model: six query heads per key / value head, tensors that hold the real tokens only
        _attn("attn_rows", contents=14, trunk=700, branches=32, lo=4, hi=24, hq=24, hkv=4, d=256, rows=True),
        # long documents with two levels of questions, 128-dim heads
        _attn("attn_long", tree="two", contents=4, trunk=8192, branches=208, lo=6, hi=10, hq=32, hkv=16, d=128),
        # one request of a user who waits for it: everything is latency
        _pass("pass_request", contents=1, trunk=301, branches=24, lo=4, hi=24),
        # a full pass of a busy server: trunks of very different lengths, 65,536 tokens
        _pass("pass_full", contents=64, cap=65536, trunk=800, spread=0.6, branches=36, lo=4, hi=24),
        # one request through a recurrent layer
        _gdn("gdn_request", contents=1, trunk=301, branches=24, lo=4, hi=24),
        # a 16k-token stream of option tries: thousands of short segments over six or seven levels
        _gdn("gdn_tries", tree="trie", contents=22, trunk=300, branches=96, lo=1, hi=9),
        # long contents with short questions (a quarter of the benchmark's stream)
        _gdn("gdn_long", contents=32, trunk=2048, branches=32, lo=12, hi=12),
        # the read rows of one request, and a whole chunk of read rows of a full pass
        _head("head_request", rows=24, stream=640, hidden=2560, vocab=262144, cols=8),
        _head("head_chunk", rows=1024, stream=65536, hidden=2560, vocab=262144, cols=8),
        # a decoding step for one request on a global layer, and one of the benchmark's size
        _xdec("xdec_request", groups=1, plo=301, phi=301, slots=4, H=16, h=1, d=512, step=9),
        _xdec("xdec_step", groups=24, plo=470, phi=470, slots=8, H=16, h=8, d=256, step=32),
    ]


def _attn(name, tree="star", contents=1, cap=0, trunk=470, spread=0.0, branches=8, lo=8, hi=16, hq=16, hkv=8, d=256, window=0, rows=False):
    return dict(name=name, kind="attn", tree=tree, contents=contents, cap=cap, trunk=trunk, spread=spread, branches=branches, lo=lo, hi=hi,
                hq=hq, hkv=hkv, d=d, window=window, rows=rows)


def _pass(name, tree="star", contents=1, cap=0, trunk=470, spread=0.0, branches=8, lo=8, hi=16):
    return dict(name=name, kind="pass", tree=tree, contents=contents, cap=cap, trunk=trunk, spread=spread, branches=branches, lo=lo, hi=hi,
                hq=16, hkv=8, d=256, window=1024, ghq=16, ghkv=1, gd=512, sliding=5)


def _gdn(name, tree="star", contents=1, cap=0, trunk=470, spread=0.0, branches=8, lo=8, hi=16, h=16, hv=32):
    return dict(name=name, kind="gdn", tree=tree, contents=contents, cap=cap, trunk=trunk, spread=spread, branches=branches, lo=lo, hi=hi,
                h=h, hv=hv, dk=128, dv=128)


def _head(name, rows, stream, hidden, vocab, cols, softcap=30.0):
    return dict(name=name, kind="head", rows=rows, stream=stream, hidden=hidden, vocab=vocab, cols=cols, softcap=softcap)


def _xdec(name, groups, plo, phi, slots, H, h, d, step, beam=6, S=33, window=0):
    return dict(name=name, kind="xdec", groups=groups, plo=plo, phi=phi, slots=slots, beam=beam, S=S, H=H, h=h, d=d, step=step, window=window)


def _log(rng, a, b):
    """a whole number, spread over the logarithm of a .. b"""
    return min(b, max(a, int(round(a * (b / a) ** rng.random()))))


def draw(rng):
    """One more case of the ranges above.  Streams hold at most 65,536 tokens in whole blocks (gdn: as many as listed)."""
    kind = rng.choice(["attn", "attn", "pass", "gdn", "head", "xdec"])
    if kind == "head":
        rows = _log(rng, 1, 1024)
        c = _head("", rows, max(rows, _log(rng, 128, 65536)), 64 * rng.randint(16, 60), _log(rng, 32000, 262144), _log(rng, 1, 64), rng.choice([30.0, 0.0]))
        if rng.random() < 0.25:   # the extraction rows: every column
            c.update(rows=_log(rng, 1, 128), cols=0)
    elif kind == "xdec":
        H, h, d = rng.choice([(16, 8, 256), (16, 1, 512), (24, 4, 256), (32, 16, 128)])
        hi = _log(rng, 64, 4096)
        groups = min(_log(rng, 1, 64), max(1, 65536 // hi))
        c = _xdec("", groups, max(16, int(hi * rng.uniform(0.3, 1))), hi, rng.randint(1, 8), H, h, d, rng.randint(0, 32), window=1024 if d == 256 and rng.random() < 0.4 else 0)
    else:
        tree = rng.choice(["star", "star", "trie"])
        shape = dict(tree=tree, contents=_log(rng, 1, 64), cap=65536, trunk=_log(rng, 48, 2048), spread=rng.choice([0.0, 0.6]),
                     branches=_log(rng, 2, 96), lo=(lo := rng.randint(1, 12)), hi=lo + rng.randint(0, 12))
        if kind == "pass":
            c = _pass("", **shape)
        elif kind == "gdn":
            h = rng.choice([8, 16])
            c = _gdn("", h=h, hv=2 * h, **shape)
        elif rng.random() < 0.2:   # long documents
            c = _attn("", tree="two", contents=rng.randint(1, 4), trunk=_log(rng, 2048, 8192), branches=13 * rng.randint(2, 16), lo=6, hi=10, hq=32, hkv=16, d=128)
        else:
            hq, hkv, d, rows = rng.choice([(16, 8, 256, False), (16, 1, 512, False), (24, 4, 256, True), (32, 16, 128, False), (16, 4, 64, False)])
            c = _attn("", hq=hq, hkv=hkv, d=d, rows=rows, window=1024 if d == 256 and not rows and rng.random() < 0.5 else 0, **shape)
    del c["name"]
    return c


# ------------------------------------------------------------------------------------------------ trees
def _shape(case):
    """per content (trunk length, branch lengths, parents), from the case alone"""
    g = np.random.default_rng(zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode()))
    out, total = [], 0
    for _ in range(case["contents"]):
        trunk = int(np.clip(case["trunk"] * np.exp(case["spread"] * g.standard_normal()), 16, 8192))
        nb = case["branches"]
        lens = g.integers(case["lo"], case["hi"] + 1, nb)
        parents = np.full(nb, -1)
        if case["tree"] == "two":      # questions of 32 tokens with twelve short ones below each
            parents = np.array([-1 if b % 13 == 0 else b - b % 13 for b in range(nb)])
            lens[parents < 0] = 32
        elif case["tree"] == "trie":   # options that share their first tokens: in pre-order, at most six levels below the trunk
            last, depth = [-1] * 8, 0
            for b in range(nb):
                depth = int(g.integers(1, min(depth + 1, 6) + 1))
                parents[b] = last[depth - 1]
                last[depth] = b
        size = -(-(trunk + int(lens.sum())) // 128) * 128
        if case["cap"] and total and total + size > case["cap"]:
            break
        total += size
        out.append((trunk, lens, parents))
    return out


def _stream(case, seed=0):
    """the packed stream; the seed orders the contents and, where they all hang on the trunk, the branches"""
    g = np.random.default_rng(seed)
    trees = []
    for i in g.permutation(len(shape := _shape(case))):
        trunk, lens, parents = shape[i]
        lens = g.permutation(lens) if (parents < 0).all() else lens
        trees.append(sa.TokenTree([1] * trunk, [[2] * int(n) for n in lens], [int(p) for p in parents]))
    return sa.pack_stream(trees)


def _normal(gen, *shape, std=1.0):
    out = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    step = max(1, (1 << 27) // max(1, out[0].numel()))
    for a in range(0, shape[0], step):
        part = out[a : a + step]
        part.copy_(torch.randn(part.shape, generator=gen, device=DEV) * std)
    return out


# ------------------------------------------------------------------------------------------------ what a program has before the call
def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return globals()["_prepare_" + case["kind"]](case, seed, gen)


def _qkv(gen, n, hq, hkv, d):
    """normalised queries and keys, values of unit scale, as the [1, heads, tokens, dim] views the model layers pass on"""
    return [_normal(gen, n, h, d).transpose(0, 1)[None] for h in (hq, hkv, hkv)]


def _prepare_attn(case, seed, gen):
    b = _stream(case, seed)
    mask = sa.block_masks(b, case["window"] or None, device=DEV)["sliding_attention" if case["window"] else "full_attention"]
    sidx = torch.from_numpy(np.flatnonzero(b.art >= 0)).to(DEV) if case["rows"] else None
    return dict(kind="attn", mask=mask, sidx=sidx, scale=case["d"] ** -0.5,
                qkv=_qkv(gen, b.n_tokens if case["rows"] else b.length, case["hq"], case["hkv"], case["d"]))


def _prepare_pass(case, seed, gen):
    b = _stream(case, seed)
    return dict(kind="pass", batch=b, window=case["window"], sliding=case["sliding"], scales=(case["d"] ** -0.5, case["gd"] ** -0.5),
                local=_qkv(gen, b.length, case["hq"], case["hkv"], case["d"]), wide=_qkv(gen, b.length, case["ghq"], case["ghkv"], case["gd"]))


def _prepare_gdn(case, seed, gen):
    b = _stream(case, seed)
    h, hv, dk, dv = case["h"], case["hv"], case["dk"], case["dv"]
    cd = 2 * h * dk + hv * dv
    return dict(kind="gdn", heads=(h, hv, dk, dv), plan=sa.tree_plan(b.prev, b.art >= 0, DEV, rows=b.n_tokens),
                y=_normal(gen, b.n_tokens, cd + hv * dv + 2 * hv), z=slice(cd, cd + hv * dv),
                conv_w=torch.randn((cd, 4), generator=gen, device=DEV) * 0.5,
                a_log=torch.rand(hv, generator=gen, device=DEV), dt_bias=torch.randn(hv, generator=gen, device=DEV),
                norm_w=(torch.rand(dv, generator=gen, device=DEV) + 0.5).to(torch.bfloat16))


def _prepare_head(case, seed, gen):
    pick = lambda n, m: torch.randint(0, n, (m,), generator=gen, device=DEV)  # noqa: E731
    return dict(kind="head", h=_normal(gen, case["stream"], case["hidden"]), w=_normal(gen, case["vocab"], case["hidden"], std=0.05),
                sel=pick(case["stream"], case["rows"]).sort().values, cols=pick(case["vocab"], case["cols"]) if case["cols"] else None,
                softcap=case["softcap"] or None)


def _lengths(case):
    """prefix length per group and template length per group and slot, from the case alone"""
    g = np.random.default_rng(zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode()))
    prefix = g.integers(case["plo"], case["phi"] + 1, case["groups"])
    return prefix, np.minimum(prefix, case["window"] - 1) if case["window"] else prefix, g.integers(8, 17, (case["groups"], case["slots"]))


def _prepare_xdec(case, seed, gen):
    prefix, stored, template = _lengths(case)
    order = np.random.default_rng(seed).permutation(case["groups"])
    prefix, stored, template = prefix[order], stored[order], template[order]
    G, Q, S, h, d = case["groups"], case["slots"] * case["beam"], case["S"], case["h"], case["d"]
    Lp, Tt = int(stored.max()), int(template.sum(1).max())
    pos_p, pos_t, own_t = (np.full((G, n), -1, np.int32) for n in (Lp, Tt, Tt))
    for g in range(G):
        pos_p[g, : stored[g]] = np.arange(prefix[g] - stored[g], prefix[g])
        own = np.repeat(np.arange(case["slots"]), template[g])
        own_t[g, : len(own)] = own
        pos_t[g, : len(own)] = np.concatenate([prefix[g] + np.arange(n) for n in template[g]])
    up = lambda x: torch.from_numpy(x).to(DEV)  # noqa: E731
    c = sa.XCaches(beam=case["beam"])
    c.kp[0], c.vp[0] = _normal(gen, G, h, Lp, d), _normal(gen, G, h, Lp, d)
    c.kt[0], c.vt[0] = _normal(gen, G, h, Tt, d), _normal(gen, G, h, Tt, d)
    c.gk[0], c.gv[0] = _normal(gen, G, h, Q, S, d), _normal(gen, G, h, Q, S, d)
    c.pos_p[0], c.pos_t, c.own_t = up(pos_p), up(pos_t), up(own_t)
    c.qpos = up(np.repeat(prefix[:, None] + template, case["beam"], 1).astype(np.int64) + case["step"])
    c.step_t = torch.full((1,), case["step"], dtype=torch.int64, device=DEV)
    c.set_lengths()
    return dict(kind="xdec", caches=c, kv=sa.GroupKV(c), scale=d**-0.5, window=case["window"] or None, q=_normal(gen, G, Q, case["H"], d).transpose(1, 2),
                new=(_normal(gen, G, Q, h, d).transpose(1, 2), _normal(gen, G, Q, h, d).transpose(1, 2)))


# ------------------------------------------------------------------------------------------------ the call
def run(s):
    if s["kind"] == "attn":
        if s["sidx"] is not None:
            return sa.tree_attention(*s["qkv"], s["mask"], s["scale"], s["sidx"])
        return sa.tree_flex_forward(None, *s["qkv"], s["mask"], s["scale"])[0]
    if s["kind"] == "pass":
        masks = sa.block_masks(s["batch"], s["window"], device=DEV)
        outs = [sa.tree_flex_forward(None, *s["local"], masks["sliding_attention"], s["scales"][0])[0] for _ in range(s["sliding"])]
        return outs + [sa.tree_flex_forward(None, *s["wide"], masks["full_attention"], s["scales"][1])[0]]
    if s["kind"] == "gdn":
        q, k, v, g, beta = sa.gdn_prologue(s["y"], s["plan"].conv, s["conv_w"], s["a_log"], s["dt_bias"], *s["heads"], True)
        o = sa.gdn_tree(q, k, v, g, beta, s["plan"])
        return sa.gdn_gate(o, s["y"][:, s["z"]], s["norm_w"], 1e-6)
    if s["kind"] == "head":
        return sa.lm_head_logprobs(s["h"], s["sel"], s["w"], s["cols"], s["softcap"])
    c = s["caches"]
    xd._CURRENT[0] = c
    k, v = s["kv"].update(*s["new"], 0)
    return sa.x_attention(None, s["q"], k, v, None, s["scale"], s["window"])[0], c.gk[0], c.gv[0]


# ------------------------------------------------------------------------------------------------ what one pass cannot do without
def work(case):
    if case["kind"] == "head":
        out = case["cols"] or case["vocab"]
        return {"bytes": 2 * case["hidden"] * (case["vocab"] + case["rows"]) + 4 * case["rows"] * out, "flops": 2 * case["hidden"] * case["rows"] * case["vocab"]}
    if case["kind"] == "xdec":
        prefix, stored, template = _lengths(case)
        G, Q, n, d = case["groups"], case["slots"] * case["beam"], case["step"] + 1, case["d"]
        pairs = sum(Q * (int(stored[g]) + n) + case["beam"] * int(template[g].sum()) for g in range(G))   # (of a sliding layer: at most)
        keys = int(stored.sum() + template.sum()) + G * Q * n
        return {"bytes": 4 * d * (keys * case["h"] + G * Q * case["H"]) + 4 * d * G * Q * case["h"], "flops": 4 * d * case["H"] * pairs}
    b = _stream(case)
    n = b.n_tokens
    if case["kind"] == "gdn":
        h, hv, dk, dv = case["h"], case["hv"], case["dk"], case["dv"]
        return {"bytes": n * (2 * (2 * h * dk + 3 * hv * dv + 2 * hv) + 32), "flops": n * hv * dk * dv * 6}
    seen = b.pos[b.art >= 0].astype(np.int64) + 1
    layers = [(1, case["hq"], case["hkv"], case["d"], case["window"])]
    if case["kind"] == "pass":
        layers = [(case["sliding"],) + layers[0][1:], (1, case["ghq"], case["ghkv"], case["gd"], 0)]
    return {"bytes": sum(4 * m * n * (hq + hkv) * d for m, hq, hkv, d, _ in layers),
            "flops": sum(4 * m * d * hq * int((np.minimum(seen, w) if w else seen).sum()) for m, hq, hkv, d, w in layers)}


def tolerance(case):
    # fp32 log-probabilities of bf16 products summed in fp32; everything else is bf16 with probabilities or states in bf16 on the way
    return {"rel": 1e-5} if case["kind"] == "head" else {"rel": 1e-2}
