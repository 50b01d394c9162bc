"""The extraction decoder's attention step behind the reference's boundary (spinf_serve/decode.py:35-104).

  XCaches       the tensors of decode.Decoder that the attention reads (decode.py:129-171): prefix, template and generated K/V
                by layer, their positions and owners, the queries' positions, the current step
  GroupKV       the cache object transformers' layers write the new tokens' K/V into (decode.py:51-68)
  x_attention   the attention interface callable "x_decode" (decode.py:71-104): same signature, same result layout
  register      AttentionInterface.register("x_decode", x_attention) (decode.py:35-41)

A step is ONE launch of spinf_xdecode_attn_fwd in libspinf_tree.so (plus a small merge launch when the key stream is split
over workgroups): nothing is copied per slot or per beam, no mask tensor is built.  There is no CPU or PyTorch path.
"""

from __future__ import annotations

import ctypes as C
from dataclasses import dataclass, field
from typing import Optional

import torch

from . import _lib

_CURRENT: list = [None]  # the caches of the decoder whose step is running (the attention interface reads them)


@dataclass
class XCaches:
    """by layer index: kp, vp [G, h, Lp, d], pos_p [G, Lp] (-1 = padding), kt, vt [G, h, Tt, d], gk, gv [G, h, Q, S, d]; shared by
    the layers: pos_t, own_t [G, Tt] (position and owning slot of each template token, -1 = padding), qpos [G, Q] int64,
    step_t [1] int64 (device), beam (queries per slot).  Positions and owners are kept as int32 device tensors."""

    kp: dict = field(default_factory=dict)
    vp: dict = field(default_factory=dict)
    pos_p: dict = field(default_factory=dict)
    kt: dict = field(default_factory=dict)
    vt: dict = field(default_factory=dict)
    gk: dict = field(default_factory=dict)
    gv: dict = field(default_factory=dict)
    pos_t: Optional[torch.Tensor] = None
    own_t: Optional[torch.Tensor] = None
    qpos: Optional[torch.Tensor] = None
    step_t: Optional[torch.Tensor] = None
    beam: int = 6
    len_p: dict = field(default_factory=dict)   # by layer: [G] int32, entries of each group's prefix that can hold keys (set_lengths)
    len_t: Optional[torch.Tensor] = None        # [G] int32, the same for the template range
    _spaces: dict = field(default_factory=dict)   # workspaces of the split launches, by device, each twice the one before
    _host_len: dict = field(default_factory=dict)   # by layer: (len_p, len_t) as host tuples (set_lengths)
    _plans: dict = field(default_factory=dict)      # split plans by geometry and lengths (plan_ragged)
    _calls: dict = field(default_factory=dict)      # prepared calls by layer and query shape (xdecode_attn)

    def set_lengths(self) -> None:
        """once per decoder, after the caches are filled: how far each group's prefix (pos_p >= 0) and template range
        (own_t >= 0) reach; the kernel then neither reads nor schedules the padding behind (decode.py:136-150 pads every group
        to the longest)"""
        def reach(valid):   # [G, L] bool -> index of the last True + 1
            L = valid.shape[1]
            idx = torch.arange(1, L + 1, device=valid.device, dtype=torch.int32)
            return (valid * idx).amax(1).to(torch.int32).contiguous() if L else torch.zeros(valid.shape[0], dtype=torch.int32, device=valid.device)

        for li, pos in self.pos_p.items():
            self.len_p[li] = reach(pos >= 0)
        self.len_t = reach(self.own_t >= 0)
        lt = tuple(self.len_t.tolist())
        self._host_len = {li: (tuple(n.tolist()), lt) for li, n in self.len_p.items()}
        self._plans.clear()
        self._calls.clear()

    def __setstate__(self, state):
        """copied and saved without the workspaces: the next step makes its own, on its stream"""
        self.__dict__.update(state, _spaces={})

    def workspace(self, device, nbytes: int, stream=None) -> torch.Tensor:
        """for a launch on the current stream of `device` (its raw handle)"""
        kept = self._spaces.setdefault(device, [])
        if not kept or kept[-1].numel() < nbytes:   # (a smaller one stays: a step in a captured graph may still write to it)
            kept.append(torch.empty(max(nbytes, 2 * kept[-1].numel() if kept else 0), dtype=torch.uint8, device=device))
            kept[-1].home = stream
        space = kept[-1]
        if space.home != stream and not torch.cuda.is_current_stream_capturing():
            # (the caller cannot name a buffer it does not know: when the caches go it is not handed out while this stream still writes to it)
            space.record_stream(torch.cuda.current_stream(device))
        return space


class GroupKV:
    """stores the new tokens' K/V at the current step and hands the layer index to the attention (decode.py:51-68).  The step is a device
    scalar: one outside the caches' 0 .. S - 1 cannot be refused here without a synchronisation; it puts NaN into the entry nearest
    to it, and the step's outputs are NaN."""

    is_compileable = False

    def __init__(self, caches: XCaches):
        self.caches = caches

    def update(self, key_states, value_states, layer_idx, *args, **kwargs):
        c = self.caches  # key_states [G, h, Q, d] -> entry step of every query's generated K/V
        gk, gv = c.gk[layer_idx], c.gv[layer_idx]
        put = _put_args(key_states, value_states, gk, gv, c.step_t)
        if put is not None:   # one launch for both
            _lib.launch(_lib.load_library().spinf_xdecode_put, put, gk.device, "spinf_xdecode_put")
            return ("x", layer_idx), ("x", layer_idx)
        c.gk[layer_idx].index_copy_(3, c.step_t, key_states.unsqueeze(3))
        c.gv[layer_idx].index_copy_(3, c.step_t, value_states.unsqueeze(3))
        return ("x", layer_idx), ("x", layer_idx)

    def get_seq_length(self, layer_idx: int = 0) -> int:
        return 0


def _put_args(k, v, gk, gv, step):
    """the arguments of spinf_xdecode_put for these tensors, or None where it does not take them (it wants bf16, 16-byte rows, contiguous
    caches; anything else goes through index_copy_)"""
    bf16, dev = torch.bfloat16, gk.device
    if not (k.dtype is bf16 and v.dtype is bf16 and gk.dtype is bf16 and gv.dtype is bf16 and step.dtype is torch.int64 and step.numel() == 1
            and gk.dim() == 5 and _lib.eager(k, v, gk, gv, step) and dev.type == "cuda"):
        return None
    G, h, Q, S, d = shape = gk.shape
    ks, vs, ptrs = k.stride(), v.stride(), (k.data_ptr(), v.data_ptr(), gk.data_ptr(), gv.data_ptr())
    if (gv.shape != shape or k.shape != (G, h, Q, d) or v.shape != k.shape or d % 8 or ks[3] != 1 or vs[3] != 1 or (ks[0] | ks[1] | ks[2] | vs[0] | vs[1] | vs[2]) % 8
            or (ptrs[0] | ptrs[1] | ptrs[2] | ptrs[3]) % 16 or not (gk.is_contiguous() and gv.is_contiguous()) or k.device != dev or v.device != dev or gv.device != dev or step.device != dev):
        return None
    return (ptrs[0], *ks[:3], ptrs[1], *vs[:3], ptrs[2], ptrs[3], step.data_ptr(), G, h, Q, S, d)


def _i32(t: Optional[torch.Tensor], what: str) -> Optional[torch.Tensor]:
    if t is None:
        return None
    if t.dtype != torch.int32 or not t.is_contiguous():
        raise ValueError(f"{what} must be a contiguous int32 tensor")
    return t


def _xdecode(query: torch.Tensor, kp: torch.Tensor, vp: torch.Tensor, pos_p: torch.Tensor, kt: torch.Tensor, vt: torch.Tensor,
             pos_t: torch.Tensor, own_t: torch.Tensor, gk: torch.Tensor, gv: torch.Tensor, qpos: torch.Tensor, step_t: torch.Tensor,
             len_p: Optional[torch.Tensor], len_t: Optional[torch.Tensor], workspace: Optional[torch.Tensor], nsplit: int, tiles_per_split: int, beam: int, scale: float, window: int, softcap: float) -> torch.Tensor:
    if query.is_cuda and query.stride(3) != 1:
        query = query.contiguous()
    a = _xdecode_args(query, kp, vp, pos_p, kt, vt, pos_t, own_t, gk, gv, qpos, step_t, len_p, len_t, nsplit, tiles_per_split, beam)
    a.scale, a.window, a.softcap = scale, window, softcap
    return _xdecode_run(a, query, workspace)


def _xdecode_args(query, kp, vp, pos_p, kt, vt, pos_t, own_t, gk, gv, qpos, step_t, len_p, len_t, nsplit, tiles_per_split, beam):
    """the argument block of a step but for its queries' and outputs' memory, scale, window and soft cap; raises on tensors the kernel does not take"""
    if not query.is_cuda:
        raise RuntimeError("spinf::xdecode_attn runs on ROCm device tensors only (no CPU path)")
    G, H, Q, d = query.shape
    h, Lp, Tt, S = gk.shape[1], kp.shape[2], kt.shape[2], gk.shape[3]
    for name, t in (("query", query), ("kp", kp), ("vp", vp), ("kt", kt), ("vt", vt), ("gk", gk), ("gv", gv)):
        if t.dtype != torch.bfloat16:
            raise ValueError(f"{name} must be bf16")
    for name, t, shape in (("kp", kp, (G, h, Lp, d)), ("vp", vp, (G, h, Lp, d)), ("kt", kt, (G, h, Tt, d)), ("vt", vt, (G, h, Tt, d)),
                           ("gk", gk, (G, h, Q, S, d)), ("gv", gv, (G, h, Q, S, d))):
        if tuple(t.shape) != shape or not t.is_contiguous():
            raise ValueError(f"{name} must be contiguous {shape}, got {tuple(t.shape)}")
    if tuple(pos_p.shape) != (G, Lp) or tuple(pos_t.shape) != (G, Tt) or tuple(own_t.shape) != (G, Tt):
        raise ValueError("pos_p [G, Lp], pos_t and own_t [G, Tt] expected")
    if qpos.dtype != torch.int64 or tuple(qpos.shape) != (G, Q) or not qpos.is_contiguous() or step_t.dtype != torch.int64:
        raise ValueError("qpos [G, Q] and step_t [1] must be int64")
    _lib.same_device(query.device, kp, vp, pos_p, kt, vt, pos_t, own_t, gk, gv, qpos, step_t, len_p, len_t)
    a = _lib.XdecArgs()
    a.kp, a.vp, a.pos_p = kp.data_ptr(), vp.data_ptr(), _i32(pos_p, "pos_p").data_ptr()
    a.kt, a.vt, a.pos_t, a.own_t = kt.data_ptr(), vt.data_ptr(), _i32(pos_t, "pos_t").data_ptr(), _i32(own_t, "own_t").data_ptr()
    a.gk, a.gv, a.qpos, a.step = gk.data_ptr(), gv.data_ptr(), qpos.data_ptr(), step_t.data_ptr()
    for name, t in (("len_p", len_p), ("len_t", len_t)):
        if t is not None:
            if tuple(t.shape) != (G,):
                raise ValueError(f"{name} must hold one length per group")
            setattr(a, name, _i32(t, name).data_ptr())
    a.nsplit, a.tiles_per_split = nsplit, tiles_per_split
    a.G, a.H, a.h, a.Q, a.S, a.Lp, a.Tt, a.d, a.beam = G, H, h, Q, S, Lp, Tt, d, beam
    return a


def _xdecode_run(a, query, workspace, stream=None):
    G, H, Q, d = query.shape
    out = torch.empty((G, Q, H, d), dtype=torch.bfloat16, device=query.device)
    a.q, (a.q_g, a.q_h, a.q_q, _), a.out = query.data_ptr(), query.stride(), out.data_ptr()
    if workspace is not None:
        a.workspace, a.workspace_bytes = workspace.data_ptr(), workspace.numel() * workspace.element_size()
    _lib.launch(_lib.load_library().spinf_xdecode_attn_fwd, a, query.device, "spinf_xdecode_attn_fwd", stream)
    return out


_xdecode_op = torch.library.custom_op("spinf::xdecode_attn", _xdecode, mutates_args=("workspace",))


@_xdecode_op.register_fake
def _(query, kp, vp, pos_p, kt, vt, pos_t, own_t, gk, gv, qpos, step_t, len_p, len_t, workspace, nsplit, tiles_per_split, beam, scale, window, softcap):
    G, H, Q, d = query.shape
    return torch.empty((G, Q, H, d), dtype=torch.bfloat16, device=query.device)


def plan_splits(G: int, H: int, h: int, Q: int, S: int, Lp: int, Tt: int, d: int, beam: int) -> tuple[int, int]:
    """-> (nsplit, workspace bytes) the library suggests for these sizes"""
    a = _lib.XdecArgs()
    a.G, a.H, a.h, a.Q, a.S, a.Lp, a.Tt, a.d, a.beam = G, H, h, Q, S, Lp, Tt, d, beam
    ns, wb = C.c_int32(0), C.c_int64(0)
    _lib.check(_lib.load_library().spinf_xdecode_plan(C.byref(a), C.byref(ns), C.byref(wb)), "spinf_xdecode_plan")
    return ns.value, wb.value


_TILE = 32   # keys per tile (csrc/xdecode_attn.hip)


def _list_tiles(Lp: int, Tt: int, S: int, len_p: int, len_t: int, qlo: int, qhi: int) -> int:
    """tiles of the list of a workgroup that owns queries qlo .. qhi (TileList of csrc/xdecode_attn.hip)"""
    lk = Lp + Tt
    e0 = -(-len_p // _TILE)
    s1 = max(Lp // _TILE if len_t > 0 else e0, e0)
    e1 = max(-(-(Lp + len_t) // _TILE) if len_t > 0 else s1, s1)
    s2 = max((lk + qlo * S) // _TILE, e1)
    e2 = max(-(-(lk + (qhi + 1) * S) // _TILE), s2)
    return e0 + (e1 - s1) + (e2 - s2)


def plan_ragged(G: int, H: int, h: int, Q: int, S: int, Lp: int, Tt: int, d: int, beam: int, len_p, len_t) -> tuple[int, int]:
    """-> (nsplit, tiles per split) for groups whose prefix / template ranges reach len_p[g] / len_t[g] entries (spinf_xdecode_plan_ragged)"""
    a = _lib.XdecArgs()
    a.G, a.H, a.h, a.Q, a.S, a.Lp, a.Tt, a.d, a.beam = G, H, h, Q, S, Lp, Tt, d, beam
    lens = [(C.c_int32 * max(G, 1))(*x) for x in (len_p, len_t)]
    ns, per = C.c_int32(1), C.c_int32(0)
    _lib.check(_lib.load_library().spinf_xdecode_plan_ragged(C.byref(a), lens[0], lens[1], C.byref(ns), C.byref(per)), "spinf_xdecode_plan_ragged")
    return ns.value, per.value


def xdecode_attn(query, caches: XCaches, layer_idx: int, scale=None, window=None, softcap=None, nsplit=None):
    """query [G, H, Q, d] bf16 -> [G, Q, H, d] bf16: softmax over (the group's prefix | the slot's own template | the beam's own
    generated tokens up to caches.step_t), see x_attention"""
    c, li = caches, layer_idx
    G, H, Q, d = query.shape
    kp, gk = c.kp[li], c.gk[li]
    tensors = (kp, c.vp[li], c.pos_p[li], c.kt[li], c.vt[li], c.pos_t, c.own_t, gk, c.gv[li], c.qpos, c.step_t, c.len_p.get(li), c.len_t)
    scale, window, softcap = float(scale if scale is not None else d**-0.5), int(window or 0), float(softcap or 0.0)
    eager = _lib.eager(query, *tensors) and query.dtype == torch.bfloat16 and query.is_cuda and query.device == gk.device and query.stride(3) == 1
    key = (li, query.shape, nsplit, c.beam)
    if eager:   # a decoder's later steps: the same caches, another query tensor
        where = [t if t is None else (t.data_ptr(), t.shape, t.stride(), t.dtype) for t in tensors]
        got = c._calls.get(key)
        if got is not None and got[0] == where:
            a = _lib.XdecArgs.from_buffer_copy(got[1])   # (kept as bytes: the caches can be copied and saved)
            a.scale, a.window, a.softcap = scale, window, softcap
            device = query.device
            stream = _lib.raw_stream(device.index)
            return _xdecode_run(a, query, c.workspace(device, got[2], stream) if got[2] else None, stream)
    per = 0
    if nsplit is None and li in c._host_len:   # the groups' own lengths are known: split sizes that balance them
        geo = (G, H, gk.shape[1], Q, gk.shape[3], kp.shape[2], c.kt[li].shape[2], d, c.beam)
        plan = geo + c._host_len[li]
        if plan not in c._plans:
            c._plans[plan] = plan_ragged(*geo, *c._host_len[li])
        nsplit, per = c._plans[plan]
    elif nsplit is None:
        nsplit, _ = plan_splits(G, H, gk.shape[1], Q, gk.shape[3], kp.shape[2], c.kt[li].shape[2], d, c.beam)
    nbytes = G * H * Q * nsplit * (d + 2) * 4 if nsplit > 1 else 0
    work = c.workspace(query.device, nbytes, _lib.raw_stream(query.device.index)) if nbytes else None
    if eager:
        a = _xdecode_args(query, *tensors, int(nsplit), int(per), int(c.beam))
        c._calls[key] = (where, bytes(a), nbytes)
        a.scale, a.window, a.softcap = scale, window, softcap
        return _xdecode_run(a, query, work)
    return _xdecode_op(query, *tensors, work, int(nsplit), int(per), int(c.beam), scale, window, softcap)


@torch.compiler.disable
def x_attention(module, query, key, value, attention_mask, scaling=None, sliding_window=None, softcap=None, **kw):
    """the attention interface "x_decode" (decode.py:71-104): `key` is what GroupKV.update returned, ("x", layer index); the
    K/V live in the caches of the decoder whose step is running.  -> (attn_output [G, Q, H, d], None)"""
    caches = _CURRENT[0]
    if caches is None:
        raise RuntimeError("x_decode attention outside a decoding step (no caches set)")
    return xdecode_attn(query, caches, key[1], scaling, sliding_window, softcap), None


def register(name: str = "x_decode") -> None:
    from transformers import AttentionInterface

    if name not in AttentionInterface._global_mapping:
        AttentionInterface.register(name, x_attention)
