"""The pieces around the kernels that the forward pass of the reference touches: the capture hooks of the attention and the
recurrent-layer interfaces (spinf_serve/models/gemma4.py:98-119, spinf_serve/models/qwen35/qwen.py:514-623), the registration
with transformers (gemma4.py:121-122), the plan compilers under threads, and the CPU baseline's fp32 arithmetic against the
float64 oracle."""

import contextlib
import copy
import gc
import pickle
import sys
import threading
import time
import types

import numpy as np
import pytest
import torch

import spinf_serve_amd as sa
from oracle import attention as oattn
from oracle import cpu_baseline
from oracle import gdn as ogdn
from oracle import mask as omask
from spinf_serve_amd import attention, masks, synth


# ----------------------------------------------------------------------------------------------------------------- CPU

def test_registration_with_transformers():
    from transformers import AttentionInterface

    sa.register_tree_attention("tree_flex_test")
    assert AttentionInterface()["tree_flex_test"] is sa.tree_flex_forward
    sa.register_tree_attention("tree_flex_test")   # a second call leaves it alone
    assert AttentionInterface()["tree_flex_test"] is sa.tree_flex_forward


def test_ops_are_registered_with_torch_library():
    """the kernels are opaque torch.library ops (inductor never traces into them); the scan mutates its output and state tensors"""
    for name in ("tree_attn", "gdn_scan", "lm_logprobs", "lm_head_logprobs"):
        assert hasattr(torch.ops.spinf, name), name
    schema = str(torch.ops.spinf.gdn_scan.default._schema)
    assert "Tensor(a" in schema and "o" in schema and "-> ()" in schema, schema
    with pytest.raises(RuntimeError):   # no CPU path
        sa.gdn.recurrent(torch.zeros(1, 4, 1, 128, dtype=torch.bfloat16), torch.zeros(1, 4, 1, 128, dtype=torch.bfloat16), torch.zeros(1, 4, 2, 128, dtype=torch.bfloat16),
                         torch.zeros(1, 4, 2), torch.zeros(1, 4, 2, dtype=torch.bfloat16), 1.0, torch.tensor([0, 4]), 1)


def _wrapped_calls():
    """the calls a compiled or traced program may hold: (name, function of plain tensors, tensors)"""
    bf = torch.bfloat16
    plan = sa.tree_plan(np.arange(-1, 7), np.ones(8, bool), "cpu")
    q, caches = synth.xdecode_case(G=1, H=2, h=1, d=64, slots=1, beam=2, S=2, prefix=(4, 4), template=(2, 2), device="cpu")
    return [
        ("lm_logprobs", lambda x: sa.lm_logprobs(x, None, 30.0), (torch.zeros(3, 64),)),
        ("lm_head_logprobs", lambda h, w: sa.lm_head_logprobs(h, None, w, None, 30.0), (torch.zeros(3, 64, dtype=bf), torch.zeros(16, 64, dtype=bf))),
        ("gdn_prologue", lambda y, c, w, a, b: sa.gdn_prologue(y, c, w, a, b, 2, 4, 128, 128), (torch.zeros(8, 1544, dtype=bf), plan.conv, torch.zeros(1024, 4), torch.zeros(4), torch.zeros(4))),
        ("gdn_gate", lambda o, z, n: sa.gdn_gate(o, z, n, 1e-6), (torch.zeros(8, 4, 128, dtype=bf), torch.zeros(8, 512, dtype=bf), torch.ones(128, dtype=bf))),
        ("xdecode_attn", lambda x: sa.xdecode_attn(x, caches, 0, nsplit=1), (q,)),
    ]


@pytest.mark.parametrize("which", range(5))
def test_a_compiled_program_holds_the_registered_operator(which):
    """torch.compile(fullgraph=True) over the public calls: one opaque node each (the graph is looked at, not run: there is no CPU path)"""
    name, call, args = _wrapped_calls()[which]
    seen = []

    def backend(gm, example):
        seen.extend(str(n.target) for n in gm.graph.nodes if n.op == "call_function")
        return lambda *a: (torch.zeros(()),) * 8

    torch._dynamo.reset()
    compiled = torch.compile(call, fullgraph=True, backend=backend)
    try:
        compiled(*args)
    finally:
        torch._dynamo.reset()
    assert any(f"spinf.{name}" in t for t in seen), seen


def test_what_watches_operators_is_seen():
    """vmap, jvp, forward-mode duals, jit.trace, function and dispatch modes get the registered operator, a default device does not"""
    import torch.autograd.forward_ad as fwd
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from spinf_serve_amd import _lib

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatches(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, seen = torch.ones(3), {}

    def look(name, y):
        seen[name] = _lib.watched()
        return y * 2

    look("plain", x)
    with torch.device("cpu"):
        look("device", x)
    with torch.inference_mode():
        look("inference", x)
    assert seen == {"plain": False, "device": False, "inference": False}
    torch.vmap(lambda y: look("vmap", y))(x)
    torch.func.jvp(lambda y: look("jvp", y), (x,), (x,))
    torch.func.grad(lambda y: look("grad", y).sum())(x)
    torch.func.functionalize(lambda y: look("functionalize", y))(x)
    torch.jit.trace(lambda y: look("trace", y), (x,), check_trace=False)
    with fwd.dual_level():
        look("dual", fwd.make_dual(x, x))
    for name, mode in (("functions", Functions()), ("dispatches", Dispatches())):
        with mode:
            look(name, x)
        with torch.device("cpu"), mode:
            look(name + " on a default device", x)
    assert all(seen[n] for n in seen if n not in ("plain", "device", "inference")) and len(seen) == 13, seen
    assert not _lib.watched()


def test_shapes_without_memory_go_through_the_operators():
    """meta tensors have no memory to read: the operators give the outputs' shapes, types and device"""
    for name, call, args in _wrapped_calls()[:4]:
        out = call(*(a.to("meta") for a in args))
        out = out if isinstance(out, tuple) else (out,)
        assert all(o.device.type == "meta" and o.shape[0] == len(args[0]) for o in out), name


def test_plan_compilers_from_two_threads():
    """tile plans, their schedules and recurrent-layer plans built at the same time on different streams equal the ones built
    one after the other"""
    cfgs = [synth.attention_config("C2", seed=s, contents=6 + s) for s in range(4)]

    def build(cfg, window):
        b = cfg.batches[0]
        p = sa.TilePlan.build(b.art, b.end, b.pos, window)
        items, ptr = p.schedule(8)
        sitems, sptr = p.schedule_static(8, 64)
        g = sa.qwen_plan._compile(np.ascontiguousarray(b.prev, np.int64), np.ascontiguousarray(b.art >= 0).view(np.uint8), "indexed", 64, 8192, 96, None, None)
        return [p.qt_ptr, p.kv_idx, p.kv_bits, p.order, items, ptr, sitems, sptr, g["idx"], g["h0_idx"], g["ht_idx"], g["conv"], g["seg_len"]]

    jobs = [(c, w) for c in cfgs for w in (None, 512)]
    serial = [build(c, w) for c, w in jobs]
    for _ in range(3):
        got = [None] * len(jobs)

        def run(i):
            got[i] = build(*jobs[i])

        threads = [threading.Thread(target=run, args=(i,)) for i in range(len(jobs))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for a, b in zip(serial, got):
            assert all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


def _fresh_mask(seed=0):
    b = synth.attention_config("C2", seed=seed, contents=3).batches[0]
    return sa.TreeMask.build(b.art, b.end, b.pos, device="cpu")


def _owns_what_it_points_to(layer):
    owned = [t for t in layer.owned if t is not None] + [t for x in layer.shared for t in x.tensors]
    spans = [(t.untyped_storage().data_ptr(), t.untyped_storage().nbytes()) for t in owned]
    return all(any(a <= getattr(layer.args, f) < a + n for a, n in spans) for f in ("art", "end", "pos", "items", "list_ptr", "kv_idx", "kv_bits"))


def test_first_calls_of_two_threads_on_one_mask_share_what_they_make(monkeypatch):
    """calls from different host threads may overlap, also the first ones on a mask: one upload, one prepared call, and the call holds
    every buffer its argument block names"""
    monkeypatch.setattr(masks, "_static_lists", lambda device: 256)
    cpu, before = torch.device("cpu"), sys.getswitchinterval()
    sys.setswitchinterval(1e-5)
    try:
        for r in range(20):
            mask, start, got = _fresh_mask(), threading.Barrier(3), [None] * 3

            def run(i):
                start.wait()
                got[i] = attention._Layer.of(mask, 16, 8, (256, 256, 512)[i], 0, i == 2, cpu)

            threads = [threading.Thread(target=run, args=(i,)) for i in range(3)]
            for t in threads:
                t.start()
            for t in threads:
                t.join()
            assert got[0] is got[1] and all(_owns_what_it_points_to(x) for x in got), r
            assert all(x in mask._layers.values() for x in got) and mask.for_head_dim(512) is mask.for_head_dim(512)
    finally:
        sys.setswitchinterval(before)


def test_a_prepared_call_outlives_the_mask_its_buffers_came_from(monkeypatch):
    """a call through the mask of the other key-tile size reads this one's buffers: it keeps them when this one goes"""
    monkeypatch.setattr(masks, "_static_lists", lambda device: 256)
    mask = _fresh_mask()
    wide = mask.for_head_dim(512)
    layer = attention._Layer.of(wide, 4, 2, 256, 0, False, torch.device("cpu"))
    want = mask.pointers(layer.head_groups, layer.n_lists)
    assert layer.args.items == want[0] and layer.args.kv_bits == want[3] and not layer.ring
    del mask, want
    gc.collect()
    assert attention._Layer.of(wide, 4, 2, 256, 0, False, torch.device("cpu")) is layer and _owns_what_it_points_to(layer)


@pytest.mark.parametrize("compact", [False, True])
def test_a_prepared_mask_leaves_nothing_to_its_first_calls(monkeypatch, compact):
    """TreeMask.prepare compiles, schedules and uploads for the layers it is told of; a layer it was not told of still comes"""
    monkeypatch.setattr(masks, "_static_lists", lambda device: 256)
    cpu, mask = torch.device("cpu"), _fresh_mask()
    sidx = torch.from_numpy(np.flatnonzero(mask.art.numpy() >= 0)) if compact else None
    heads = [(16, 8, 256), (4, 2, 128), (8, 1, 512)]
    assert mask.prepare(*heads, sidx=sidx) is mask

    def more(*a, **k):
        raise AssertionError("a prepared mask makes something at a call")

    with monkeypatch.context() as m:
        m.setattr(sa.TilePlan, "compile", more)
        m.setattr(sa.TreeMask, "_upload", more)
        m.setattr(masks, "_Shared", more)
        for hq, hkv, d in heads:
            layer = attention._Layer.of(mask, hq, hkv, d, 0, compact, cpu)
            assert _owns_what_it_points_to(layer)
            if compact:
                mask.for_head_dim(d, ring=layer.ring).rows(sidx)
        with pytest.raises(AssertionError):
            attention._Layer.of(mask, 6, 2, 64, 0, compact, cpu)
    with pytest.raises(ValueError, match="do not group"):
        mask.prepare((5, 2, 64))


@pytest.mark.parametrize("bidir_all", [False, True])
def test_every_buffer_of_a_mask_with_images_is_shared(monkeypatch, bidir_all):
    """what the allocator is told of when another stream reads a mask: the metadata of the mask it shares it with among them"""
    monkeypatch.setattr(masks, "_static_lists", lambda device: 256)
    b = synth.attention_config("C2", contents=2).batches[0]
    grp = np.where(np.arange(b.length) % 300 < 20, np.arange(b.length) // 300, -1)
    for mask in sa.block_masks(b, sliding_window=100, device="cpu", grp=grp, bidir_all=bidir_all).values():
        layer = attention._Layer.of(mask, 4, 2, 128, 0, False, torch.device("cpu"))
        layer.owned = ()   # (the shared ones alone)
        assert _owns_what_it_points_to(layer)
        spans = [(t.untyped_storage().data_ptr(), t.untyped_storage().nbytes()) for x in layer.shared for t in x.tensors]
        assert mask.grp is None or any(a <= layer.args.grp < a + n for a, n in spans)


@pytest.mark.parametrize("how", [copy.copy, copy.deepcopy, lambda m: pickle.loads(pickle.dumps(m))])
def test_masks_are_copied_and_saved(how):
    b = synth.attention_config("C2", contents=2).batches[0]
    grp = np.where(np.arange(b.length) % 300 < 20, np.arange(b.length) // 300, -1)
    for mask in sa.block_masks(b, sliding_window=100, device="cpu", grp=grp, bidir_all=False).values():
        for used in (False, True):
            for m in (mask, mask.for_head_dim(512)):
                if used:
                    m.kv_idx
                mine = how(m)
                assert (mine.window, mine.grp_mode, mine.n, mine._ktile) == (m.window, m.grp_mode, m.n, m._ktile) and torch.equal(mine.art, m.art)
                assert torch.equal(mine.kv_idx, m.kv_idx) and torch.equal(mine.kv_bits, m.kv_bits) and mine.kv_idx.data_ptr() != m.kv_idx.data_ptr()


def test_a_row_map_follows_its_row_list():
    """kept for the tensor it was built from, and built again when that tensor was changed in place"""
    mask = _fresh_mask()
    sidx = torch.from_numpy(np.flatnonzero(mask.art.numpy() >= 0).copy())
    one = mask.rows(sidx)
    assert mask.rows(sidx)[0] is one[0]
    sidx[:64] = sidx[:64].flip(0)
    two = mask.rows(sidx)
    assert two[0] is not one[0] and torch.equal(two[0][sidx], torch.arange(len(sidx), dtype=torch.int32))
    with torch.inference_mode():
        other = sidx + 0
    assert mask.rows(other)[0] is mask.rows(other)[0]


def test_a_stream_the_compiler_refuses_is_refused_at_the_build():
    long = np.broadcast_to(np.int32(0), ((1 << 30) + 1,))
    with pytest.raises(ValueError, match="too long"):
        sa.TreeMask.build(long, long, long, device="cpu")


def test_a_call_on_another_stream_waits_for_what_the_first_one_uploaded(monkeypatch):
    """a mask's schedules, entries and row maps are uploaded by whichever call comes first, on its stream: every other stream waits for
    the copy of each buffer it reads, once, and the allocator hears of it; the stream that copied does not wait"""
    now, log = ["a"], []

    def join(shared):
        log.append((now[0], shared))
        return now[0] != "capture"

    monkeypatch.setattr(masks, "_static_lists", lambda device: 256)
    monkeypatch.setattr(masks._lib, "raw_stream", lambda index: now[0])
    monkeypatch.setattr(masks, "_join", join)
    cpu, mask = torch.device("cpu"), _fresh_mask()

    def call(stream, hq, sidx=None):
        now[0] = stream
        del log[:]
        layer = attention._Layer.of(mask, hq, 2, 256, 0, sidx is not None, cpu)
        if stream not in layer.streams:
            layer.reach(stream)
        if sidx is not None:
            mask.rows(sidx)
        return layer, [(s, shared.home) for s, shared in log]

    # the metadata, built on "a", is the caller's to wait for, as any tensor: other streams are named to the allocator only
    meta, = mask._meta
    assert meta.home is None and meta.streams == {"a"} and meta.tensors[0].data_ptr() == mask.art.data_ptr()
    assert call("b", 4)[1] == [("b", None)]        # uploads entries and its schedule on b
    assert call("b", 4)[1] == []
    assert call("c", 8)[1] == [("c", "b"), ("c", None)]        # another geometry on c: its schedule on c, the entries are b's
    assert call("c", 8)[1] == [] and call("c", 4)[1] == []     # (what b made has been waited for)
    assert call("b", 8)[1] == [("b", "c")]
    layer, seen = call("a", 4)
    assert seen == [("a", "b")] and all(x.made is None for x in layer.shared)
    for _ in range(2):                             # nothing can be waited for under capture, and it is not taken for done
        layer, seen = call("capture", 4)
        assert [s for s, _ in seen] == ["capture"] * 3 and "capture" not in layer.streams
    sidx = torch.from_numpy(np.flatnonzero(mask.art.numpy() >= 0))
    assert call("b", 4, sidx)[1] == [] and mask._rows[3].home == "b"
    assert call("d", 4, sidx)[1] == [("d", "b"), ("d", None), ("d", "b")]


@pytest.mark.parametrize("home", [0, 0x70])
def test_the_wait_is_for_the_stream_that_uploaded_the_default_stream_too(home, monkeypatch):
    """the default stream's handle is 0, and torch.cuda.ExternalStream(0) is not that stream: torch takes a handle of 0 for none given and
    makes a new one (restated here, as on the GPU: its cuda_stream is not 0), which there is nothing to wait for on"""
    class Stream:
        def __init__(self, handle):
            self.cuda_stream, self.waits = handle, []

        def wait_stream(self, other):
            self.waits.append(other.cuda_stream)

    here = Stream(0x10)
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "stream", lambda stream: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: here)
    monkeypatch.setattr(torch.cuda, "default_stream", lambda: Stream(0))
    monkeypatch.setattr(torch.cuda, "ExternalStream", lambda handle: Stream(handle or 0x5000))
    assert masks._join(types.SimpleNamespace(device=None, made=None, home=home, tensors=()))
    assert here.waits == [home]


def test_c1_in_fp32_on_the_cpu_against_the_oracle():
    """the CPU baseline leg (fp32 scaled_dot_product_attention under a dense tree mask per content) and torch's eager
    flex_attention under the same rule agree with the float64 oracle to 1e-5 on C1"""
    from torch.nn.attention.flex_attention import create_block_mask, flex_attention

    cfg = synth.attention_config("C1")
    b = cfg.batches[0]
    q, k, v = synth.qkv(cfg, b, seed=0, device="cpu")
    q, k, v = q.float(), k.float(), v.float()
    want = oattn.tree_attention(q.numpy(), k.numpy(), v.numpy(), b.art, b.end, b.pos, scale=cfg.scale, spans=oattn.job_spans(b.art))
    _, done, _, _, outs = cpu_baseline.attention_tokens_per_s(q, k, v, b.art, b.end, b.pos, cfg.scale)
    assert done == len(cfg.trees)
    for (a, e), o in outs.items():
        real = b.art[a:e] >= 0
        assert np.abs(o.numpy()[real] - want[a:e][real]).max() <= 1e-5
    art, end = torch.from_numpy(b.art), torch.from_numpy(b.end)

    def rule(_b, _h, qi, ki):   # spinf_serve/scorer.py:173-177
        return ((art[qi] >= 0) & (art[qi] == art[ki]) & (ki <= qi) & (end[ki] > qi)) | (qi == ki)

    n = b.length
    bm = create_block_mask(rule, None, None, n, n, device="cpu", BLOCK_SIZE=128)
    dense = omask.dense_tree_mask(b.art, b.end, b.pos)
    blocks = dense.reshape(n // 128, 128, n // 128, 128).any(axis=(1, 3))   # the oracle's view of which 128 x 128 blocks are live
    assert np.array_equal(bm.to_dense()[0, 0].bool().numpy(), blocks)
    o = flex_attention(q.transpose(0, 1)[None], k.transpose(0, 1)[None], v.transpose(0, 1)[None], block_mask=bm, scale=cfg.scale, enable_gqa=True)
    real = b.art >= 0
    assert np.abs(o[0].transpose(0, 1).numpy()[real] - want[real]).max() <= 1e-5


# ----------------------------------------------------------------------------------------------------------------- GPU

def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.gpu
def test_attention_capture_keeps_the_named_ranges(dev):
    """gemma4.py:100-106: under CAPTURE a global layer keeps the keys / values of each range, a sliding layer their last window - 1"""
    cfg = synth.attention_config("C2", contents=2)
    b = cfg.batches[0]
    q, k, v = synth.qkv(cfg, b, seed=2, device=dev)
    masks = sa.block_masks(b, sliding_window=64, device=dev)
    config = types.SimpleNamespace(layer_types=["sliding_attention", "full_attention"])
    ranges = [(0, 470, "trunk0"), (b.jobs[1][0], 30, "head1"), (5, 10, "short")]
    args = [t.transpose(0, 1)[None] for t in (q, k, v)]
    plain = [sa.tree_flex_forward(types.SimpleNamespace(config=config, layer_idx=i), *args, masks[config.layer_types[i]], scaling=cfg.scale)[0] for i in range(2)]
    attention.CAPTURE[dev] = {"window": 64, "ranges": ranges, "kv": {}}
    try:
        hooked = [sa.tree_flex_forward(types.SimpleNamespace(config=config, layer_idx=i), *args, masks[config.layer_types[i]], scaling=cfg.scale)[0] for i in range(2)]
        kept = attention.CAPTURE[dev]["kv"]
    finally:
        del attention.CAPTURE[dev]
    assert all(torch.equal(a, c) for a, c in zip(plain, hooked)) and plain[0].shape == (1, b.length, cfg.hq, cfg.d)
    for start, n, name in ranges:
        assert sorted(kept[name]) == [0, 1]
        for layer, first in ((0, start + max(0, n - 63)), (1, start)):
            kk, vv = kept[name][layer]
            assert torch.equal(kk[0], k[first : start + n].transpose(0, 1)) and torch.equal(vv[0], v[first : start + n].transpose(0, 1))
    assert dev not in attention.CAPTURE


@pytest.mark.gpu
@pytest.mark.parametrize("compact", [False, True])
def test_qwen_attention_capture_and_compact_rows(dev, compact):
    """qwen.py:604-623: plan.cap keeps the keys / values of the named row ranges per layer; with sidx the tensors hold the real
    rows only and every real row's output has the stream call's bits"""
    cfg = synth.attention_config("C2", contents=2)
    b = cfg.batches[0]
    q, k, v = synth.qkv(cfg, b, seed=3, device=dev)
    mask = sa.TreeMask.build(b.art, b.end, b.pos, device=dev)
    stream = sa.tree_attn(q, k, v, mask, cfg.scale)
    sidx = torch.from_numpy(np.flatnonzero(b.art >= 0)).to(dev) if compact else None
    if compact:
        q, k, v = (t[sidx].contiguous() for t in (q, k, v))
    plan = types.SimpleNamespace(cap={"ranges": [(3, 40, "a"), (500, 7, "b")], "out": {"kv": {}}})
    o = sa.tree_attention(*(t.transpose(0, 1)[None] for t in (q, k, v)), mask, cfg.scale, sidx=sidx, plan=plan, mod=types.SimpleNamespace(li=5))
    want = stream[sidx] if compact else stream
    assert torch.equal(o[0].transpose(0, 1), want)
    for r0, n, name in plan.cap["ranges"]:
        kk, vv = plan.cap["out"]["kv"][name][5]
        assert torch.equal(kk[0], k[r0 : r0 + n].transpose(0, 1)) and torch.equal(vv[0], v[r0 : r0 + n].transpose(0, 1))


@pytest.mark.gpu
def test_gdn_capture_keeps_inputs_and_final_states(dev):
    """qwen.py:520-526,558-565: plan.cap keeps the scan inputs of row ranges and the final state of the segment that holds a
    named row; the state equals the oracle's state after that segment's last token"""
    cfg = synth.gdn_config("C5", contents=2)
    b = cfg.batch
    t = synth.gdn_inputs(cfg, seed=4, device=dev)
    trunk_last = [s0 + P - 1 for s0, _, P, _ in b.jobs]
    leaf_row = int(np.flatnonzero(b.seg == 3)[2])                     # a row inside branch 2 of the first content
    leaf_last = int(np.flatnonzero((b.seg == 3) & (b.art == 0))[-1])
    keep = [trunk_last[0], trunk_last[1], leaf_last]
    plan = cfg.plan(dev, keep=keep)
    plain = sa.gdn_tree(t["q"], t["k"], t["v"], t["g"], t["beta"], cfg.plan(dev))
    plan.cap = {"tok": [(10, 20, "rows")], "state": [(5, "trunk0"), (trunk_last[1], "trunk1"), (leaf_row, "leaf")], "out": {"gdn": {}, "state": {}}}
    o = sa.gdn_tree(t["q"], t["k"], t["v"], t["g"], t["beta"], plan, mod=types.SimpleNamespace(li=7))
    torch.cuda.synchronize()
    assert torch.equal(o, plain)
    got = plan.cap["out"]["gdn"]["rows"][7]
    assert all(torch.equal(x, t[n][10:30]) for x, n in zip(got, ("q", "k", "v", "g", "beta")))
    _, states = ogdn.tree_scan(*(_np(t[x]) for x in ("q", "k", "v", "g", "beta")), b.prev, b.art >= 0, keep=keep)
    for name, pos in (("trunk0", trunk_last[0]), ("trunk1", trunk_last[1]), ("leaf", leaf_last)):
        s = _np(plan.cap["out"]["state"][name][7])
        assert s.shape == (cfg.hv, cfg.dk, cfg.dv)
        assert np.abs(s - states[pos]).max() <= 2e-2, name
    plan.cap = {"tok": [], "state": [(int(np.flatnonzero(b.seg == 5)[0]), "unkept")], "out": {"gdn": {}, "state": {}}}
    with pytest.raises(RuntimeError):
        sa.gdn_tree(t["q"], t["k"], t["v"], t["g"], t["beta"], plan, mod=types.SimpleNamespace(li=7))


@pytest.mark.gpu
def test_every_c3_pass(dev):
    """all 13 passes of C3, sliding and global: pad rows come out as their own V row, and the smallest content of each pass
    matches the float64 oracle"""
    cfg = synth.attention_config("C3")
    assert len(cfg.batches) == 13
    for i, b in enumerate(cfg.batches):
        q, k, v = synth.qkv(cfg, b, seed=i, device=dev)
        masks = sa.block_masks(b, sliding_window=cfg.window, device=dev)
        s0, n, _, _ = min(b.jobs, key=lambda j: j[1])
        e0 = s0 + -(-n // 128) * 128
        sub = (q[s0:e0], k[s0:e0], v[s0:e0])
        pad = torch.from_numpy(np.flatnonzero(b.art < 0)).to(dev)
        for name, window in (("sliding_attention", cfg.window), ("full_attention", None)):
            print(f"case C3 pass {i} n={b.length} {name} content at {s0}+{n}", flush=True)
            out = sa.tree_attn(q, k, v, masks[name], cfg.scale)
            assert torch.equal(out[pad], v[pad].repeat_interleave(cfg.hq // cfg.hkv, dim=1))
            want = oattn.tree_attention(*(_np(x) for x in sub), b.art[s0:e0], b.end[s0:e0] - s0, b.pos[s0:e0], window=window, scale=cfg.scale)
            real = b.art[s0:e0] >= 0
            assert np.abs(_np(out[s0:e0])[real] - want[real]).max() <= 2e-2


@pytest.mark.gpu
@pytest.mark.parametrize("call", ["prologue", "gate", "logprobs", "head", "xdecode"])
def test_tensors_of_another_device_are_refused_before_any_launch(dev, call):
    """each tensor of a call in turn on the host: its address would go to the kernel"""
    bf = dict(dtype=torch.bfloat16, device=dev)
    if call == "prologue":
        plan = sa.tree_plan(np.arange(-1, 39), np.ones(40, bool), dev)
        args = [torch.zeros(40, 2 * 256 + 2 * 512 + 8, **bf), plan.conv, torch.zeros(1024, 4, device=dev), torch.zeros(4, device=dev), torch.zeros(4, device=dev)]
        run = lambda *t: sa.gdn_prologue(*t, 2, 4, 128, 128)  # noqa: E731
    elif call == "gate":
        args = [torch.zeros(40, 4, 128, **bf), torch.zeros(40, 512, **bf), torch.zeros(128, **bf)]
        run = lambda *t: sa.gdn_gate(*t, 1e-6)  # noqa: E731
    elif call == "logprobs":
        args = [torch.zeros(3, 64, device=dev), torch.tensor([1, 5], device=dev)]
        run = sa.lm_logprobs
    elif call == "head":
        args = [torch.zeros(9, 64, **bf), torch.tensor([0, 8], device=dev), torch.zeros(128, 64, **bf), torch.tensor([1, 5], device=dev)]
        run = sa.lm_head_logprobs
    else:
        q, c = synth.xdecode_case(G=1, H=2, h=1, d=64, slots=1, beam=2, S=2, prefix=(4, 4), template=(2, 2), device=dev)
        for name in ("kp", "vp", "pos_p", "kt", "vt", "gk", "gv", "pos_t", "own_t", "qpos", "step_t"):
            whole = getattr(c, name)
            setattr(c, name, {0: whole[0].cpu()} if isinstance(whole, dict) else whole.cpu())
            with pytest.raises((ValueError, RuntimeError), match="device|must be on"):
                sa.xdecode_attn(q, c, 0)
            setattr(c, name, whole)
        sa.xdecode_attn(q, c, 0)
        return
    for i in range(len(args)):
        with pytest.raises((ValueError, RuntimeError), match="device|must be on"):
            run(*args[:i], args[i].cpu(), *args[i + 1 :])
    run(*args)


@pytest.mark.gpu
@pytest.mark.parametrize("default", [False, True])
def test_layers_of_one_mask_on_two_streams(dev, default):
    """the first call's stream is busy, so its uploads are late; a call on another stream gives the bits of one that has waited for
    everything, and what it reads is not handed out again when the mask goes while it is still to run"""
    cfg = synth.attention_config("C2", contents=2)
    b = cfg.batches[0]
    q, k, v = synth.qkv(cfg, b, seed=5, device=dev)
    few = [t[:, :n].contiguous() for t, n in ((q, 8), (k, 4), (v, 4))]
    ref = sa.TreeMask.build(b.art, b.end, b.pos, device=dev)
    want = [sa.tree_attn(q, k, v, ref, cfg.scale), sa.tree_attn(*few, ref, cfg.scale)]
    streams = [torch.cuda.default_stream() if default else torch.cuda.Stream(), torch.cuda.Stream()]
    mask = sa.TreeMask.build(b.art, b.end, b.pos, device=dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(streams[0]):
        torch.cuda._sleep(20_000_000)
        one = sa.tree_attn(q, k, v, mask, cfg.scale)
    with torch.cuda.stream(streams[1]):
        two = [sa.tree_attn(*few, mask, cfg.scale)]
        behind = torch.cuda.Event()
        behind.record()
        time.sleep(2e-3)   # (longer than that call takes)
        ran = behind.query()
        assert not (ran and not streams[0].query()), "the call has run while the stream that uploads what it reads is still busy"
        two.append(sa.tree_attn(q, k, v, mask, cfg.scale))
        torch.cuda._sleep(20_000_000)
        two.append(sa.tree_attn(*few, mask, cfg.scale))
    buffers = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for x in (*mask._sched.values(), mask._kv) for t in x[-1].tensors}
    streams[0].synchronize()
    del mask
    with torch.cuda.stream(streams[0]):   # (the stream whose pool they came from)
        fresh = [torch.empty(n, dtype=torch.uint8, device=dev) for n in buffers.values() for _ in range(4)]
    assert not streams[1].query() and not any(t.data_ptr() in buffers for t in fresh)
    torch.cuda.synchronize()
    assert torch.equal(one, want[0]) and torch.equal(two[0], want[1]) and torch.equal(two[1], want[0]) and torch.equal(two[2], want[1])


@pytest.mark.gpu
def test_a_traced_program_holds_the_operator(dev):
    """torch.jit.trace records the operator: the trace gives the next input's result, not the first one's"""
    gen = torch.Generator(device=dev).manual_seed(0)
    a, b = (torch.randn(5, 128, generator=gen, device=dev) for _ in range(2))
    traced = torch.jit.trace(lambda x: sa.lm_logprobs(x, None, 30.0), (a,), check_trace=False)
    assert "spinf::lm_logprobs" in str(traced.graph)
    for x in (a, b):
        assert torch.equal(traced(x), sa.lm_logprobs(x, None, 30.0))


@pytest.mark.gpu
def test_masks_prepared_on_a_thread_and_stream_of_their_own(dev):
    """a producer thread builds and prepares a forward's masks on its stream; the layers run on another stream with no order between
    the two but what the calls see to"""
    cfg = synth.attention_config("C2", contents=2)
    b = cfg.batches[0]
    q, k, v = synth.qkv(cfg, b, seed=6, device=dev)
    ref = sa.block_masks(b, sliding_window=100, device=dev)
    want = {name: sa.tree_attn(q, k, v, m, cfg.scale) for name, m in ref.items()}
    stream, made = torch.cuda.Stream(), {}
    sidx = torch.from_numpy(np.flatnonzero(b.art >= 0)).to(dev)
    compact = [x[sidx].contiguous() for x in (q, k, v)]
    torch.cuda.synchronize()

    def produce():
        with torch.cuda.device(dev), torch.cuda.stream(stream):
            torch.cuda._sleep(20_000_000)
            made.update({name: m.prepare((cfg.hq, cfg.hkv, cfg.d)) for name, m in sa.block_masks(b, sliding_window=100, device=dev).items()})
            made["full_attention"].prepare((cfg.hq, cfg.hkv, cfg.d), sidx=sidx)

    t = threading.Thread(target=produce)
    t.start()
    t.join()
    got = {name: sa.tree_attn(q, k, v, m, cfg.scale) for name, m in made.items()}
    rows = sa.tree_attn(*compact, made["full_attention"], cfg.scale, sidx=sidx)
    assert all(x.made is not None for m in made.values() for x in (m.for_head_dim(cfg.d, ring=l.ring)._kv[2] for l in m._layers.values()))
    made.clear()
    assert torch.equal(rows, want["full_attention"][sidx])
    assert all(torch.equal(got[name], want[name]) for name in want)


@pytest.mark.gpu
def test_the_model_layers_layout_refuses_what_the_general_path_refuses(dev):
    """tree_flex_forward and tree_attention take plain calls past the general path's checks: every refused form still ends there, and
    every accepted stride gives its bits"""
    cfg = synth.attention_config("C2", contents=1)
    b = cfg.batches[0]
    n, mask = b.length, sa.TreeMask.build(b.art, b.end, b.pos, device=dev)
    q, k, v = (t.transpose(0, 1)[None] for t in synth.qkv(cfg, b, seed=1, device=dev))
    want = sa.tree_attn(*(t[0].transpose(0, 1) for t in (q, k, v)), mask, cfg.scale)
    wide = torch.zeros(1, cfg.hkv, n, 2 * cfg.d, dtype=torch.bfloat16, device=dev)
    wide[..., : cfg.d] = v
    for qq, kk, vv in ((q, k, v), (q.contiguous(), k.contiguous(), v.contiguous()), (q, k.contiguous(), wide[..., : cfg.d])):
        assert torch.equal(sa.tree_flex_forward(None, qq, kk, vv, mask, cfg.scale)[0][0], want)
        assert torch.equal(sa.tree_attention(qq, kk, vv, mask, cfg.scale)[0].transpose(0, 1), want)
    bad = [(q, k[:, :0], v[:, :0]), (q, k[:, :, :-1], v), (q, k, v[:, :1]), (q[..., :-1], k, v), (q[:, :3], k, v), (q.float(), k, v), (q, k, v.half()),
           (q[:, :, :-128], k[:, :, :-128], v[:, :, :-128]), (q[..., ::2], k[..., ::2], v[..., ::2]), (q, k.cpu(), v)]
    for i, args in enumerate(bad):
        for call in (lambda *a: sa.tree_flex_forward(None, *a, mask, cfg.scale), lambda *a: sa.tree_attention(*a, mask, cfg.scale)):
            with pytest.raises((ValueError, RuntimeError)):
                call(*args)
                pytest.fail(f"case {i} was taken")
