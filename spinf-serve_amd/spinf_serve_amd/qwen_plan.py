"""Recurrent-layer planning and the tree scan of the hybrid (Qwen) stack behind the reference's interface
(spinf_serve/models/qwen35/qwen.py: Call :125-135, TreePlan :137-155, tree_plan :158-276, gdn_tree / gdn_indexed :514-590).

The plan itself is compiled by the library's host C++ (spinf_gdn_plan_build, csrc/gdnplan.cpp): one pass over the stream gives
the segments and their depth, a counting sort the levels, and the calls are slices of flat arrays.  This module only wraps those
arrays into the reference's Call / TreePlan objects and drives the HIP kernels level by level, states read and written by index.
"""

from __future__ import annotations

import ctypes as C
from dataclasses import dataclass

import numpy as np
import torch

from . import _lib, gdn


@dataclass
class Call:
    idx: object            # [n] int64 rows of the call's segments, back to back (device)
    cu: object             # [segs + 1] int64 cumulative lengths (device)
    cu_cpu: object         # the same on the host
    parent: object | None  # levels path: [segs] rows of the previous level's kept states, or None (roots)
    keep: bool             # levels path: leave the final states (segments with children)
    kind: str = "chunked"  # indexed path: chunked | recurrent
    h0_idx: object | None = None   # [segs] slot in the previous level's states (-1 zero); None at level 0
    ht_idx: object | None = None   # [segs] slot in this level's states (-1 none); None when nothing is kept


@dataclass
class TreePlan:
    conv: object           # [T, 4] int64: path predecessors 3, 2, 1 back and the token itself; T = "none" (a zero row)
    levels: list
    n_segments: int
    path: str = "levels"
    n_keep: list | None = None
    rows: int | None = None
    sidx: object | None = None
    seg_of_row: object | None = None
    seg_level: object | None = None
    seg_slot: object | None = None
    cap: dict | None = None
    pad_rows: object | None = None   # [pads] int64 (device): rows of the tensors no segment covers; their outputs are zero
    launches: list | None = None     # indexed path: per level the kernel launches (mode, segments, longest, places of cu, idx, h0_idx, ht_idx in data, -1 none), neighbouring calls of one kind as one
    program: list | None = None      # the same with the small subtrees as forests of their own (mode 2, csrc/gdn_forest.hip); None without any
    data: object | None = None       # [*] int64 (device): what the launches read (places, not addresses: a copied or reloaded plan has its own)


_PATHS = {"indexed": 0, "levels": 1}


def _compile(prev, real, path, short, call_tokens, max_init, rows, keep):
    """-> the flat arrays of spinf_gdn_plan_export, as a dict of numpy arrays"""
    lib = _lib.load_library()
    keep = np.ascontiguousarray([] if keep is None else list(keep), np.int64)
    handle = C.c_void_p()
    _lib.check(lib.spinf_gdn_plan_build(prev.ctypes.data, real.ctypes.data, len(prev), _PATHS[path], int(short), int(call_tokens), int(max_init),
                                        -1 if rows is None else int(rows), keep.ctypes.data if len(keep) else None, len(keep), C.byref(handle)),
               "tree_plan")
    try:
        counts = (C.c_int64 * 6)()
        _lib.check(lib.spinf_gdn_plan_counts(handle, counts), "tree_plan")
        n_seg, n_lev, n_call, n_cseg, n_rows, n_conv = (int(c) for c in counts)
        shapes = dict(level_ptr=(n_lev + 1, np.int64), call_kind=(n_call, np.int32), call_keep=(n_call, np.int32), call_seg_ptr=(n_call + 1, np.int64),
                      call_row_ptr=(n_call + 1, np.int64), seg_len=(n_cseg, np.int64), h0_idx=(n_cseg, np.int64), ht_idx=(n_cseg, np.int64),
                      idx=(n_rows, np.int64), n_keep=(n_lev, np.int64), conv=(n_conv * 4, np.int64), seg_of_row=(n_conv, np.int64),
                      seg_level=(n_seg, np.int64), seg_slot=(n_seg, np.int64))
        out = {name: np.empty(max(size, 1), dtype) for name, (size, dtype) in shapes.items()}
        _lib.check(lib.spinf_gdn_plan_export(handle, *(out[name].ctypes.data for name in shapes)), "tree_plan")
        out = {name: out[name][: shapes[name][0]] for name in shapes}
        out["n_segments"] = n_seg
        counts = (C.c_int64 * 2)()
        _lib.check(lib.spinf_gdn_plan_program(handle, counts, None, None), "tree_plan")
        out["program"], out["program_data"] = np.empty((counts[0], 8), np.int64), np.empty(counts[1], np.int64)
        _lib.check(lib.spinf_gdn_plan_program(handle, counts, out["program"].ctypes.data, out["program_data"].ctypes.data), "tree_plan")
        return out
    finally:
        lib.spinf_gdn_plan_free(handle)


def tree_plan(prev, real, device, max_init: int = 96, path: str = "indexed", short: int = 64, rows: int | None = None,
              keep=None, call_tokens: int = 8192) -> TreePlan:
    """prev[i] = token before i on its path (-1 none), real[i] = not a pad.  Arguments as the reference's tree_plan
    (qwen.py:158-174): rows = plan over compact rows (real tokens first), keep = positions whose segment must leave its
    final state, short / call_tokens = the indexed path's kernel choice and call size."""
    if path not in _PATHS:
        raise ValueError(f"tree_plan: unknown path {path!r}")
    prev = np.ascontiguousarray(prev, np.int64)
    real = np.ascontiguousarray(real, bool).view(np.uint8)
    if len(real) != len(prev):
        raise ValueError("tree_plan: prev and real differ in length")
    a = _compile(prev, real, path, short, call_tokens, max_init, rows, keep)
    dev = torch.device(device)

    indexed = path == "indexed"
    seg_len, call_kind, call_keep = a["seg_len"], a["call_kind"], a["call_keep"]
    seg_ptr, row_ptr, level_ptr = a["call_seg_ptr"].tolist(), a["call_row_ptr"].tolist(), a["level_ptr"].tolist()
    # A call's cumulative lengths, and those of the run of neighbouring calls of one kind and level that it belongs to: the indexed
    # path cuts a level's long segments into calls of call_tokens tokens (which bounded the reference's per-chunk snapshots), but the
    # kernel keeps none and wants all the segments of a level at once: 8 calls of 4 segments x 32 heads fill half the GPU eight times.
    runs = []   # per level: (first call, one past the last)
    for d in range(len(level_ptr) - 1):
        cuts = [c for c in range(level_ptr[d], level_ptr[d + 1]) if c == level_ptr[d] or call_kind[c] != call_kind[c - 1]] + [level_ptr[d + 1]]
        runs.append(list(zip(cuts[:-1], cuts[1:])))
    total = np.concatenate([[0], np.cumsum(seg_len)]).astype(np.int64)
    spans = [(c, c + 1) for c in range(len(call_kind))] + [r for lv in runs for r in lv if indexed and r[1] - r[0] > 1]
    cu_host = torch.from_numpy(np.concatenate([total[seg_ptr[i] : seg_ptr[j] + 1] - total[seg_ptr[i]] for i, j in spans]) if spans else np.zeros(0, np.int64))
    cu_at = np.concatenate([[0], np.cumsum([seg_ptr[j] - seg_ptr[i] + 1 for i, j in spans])]).astype(np.int64).tolist()
    # everything the kernels read, in one copy
    sidx_host = np.flatnonzero(real) if rows is not None else np.zeros(0, np.int64)
    parts = [a["conv"], a["idx"], a["h0_idx"], a["ht_idx"], cu_host.numpy(), sidx_host, np.flatnonzero(a["seg_of_row"] < 0), a["program_data"]]
    at = np.concatenate([[0], np.cumsum([-(-len(x) // 2) * 2 for x in parts])]).tolist()   # (each part 16-byte aligned)
    stage = torch.empty(at[-1], dtype=torch.int64, pin_memory=dev.type == "cuda")
    host = stage.numpy()
    for x, o in zip(parts, at):
        host[o : o + len(x)] = x
    on_dev = stage.to(dev, non_blocking=True)
    conv, idx_all, h0_all, ht_all, cu_all, sidx, pad_rows, _ = (on_dev[o : o + len(x)] for x, o in zip(parts, at))
    cu_of = {span: k for k, span in enumerate(spans)}

    levels, launches = [], []
    for d, lv in enumerate(runs):
        calls = []
        for c in range(level_ptr[d], level_ptr[d + 1]):
            seg, k = slice(seg_ptr[c], seg_ptr[c + 1]), slice(cu_at[c], cu_at[c + 1])     # (the first spans are the calls)
            idx, cu, cu_cpu, ends = idx_all[row_ptr[c] : row_ptr[c + 1]], cu_all[k], cu_host[k], ht_all[seg]
            starts = None if d == 0 else h0_all[seg]
            if indexed:
                calls.append(Call(idx, cu, cu_cpu, None, False, "chunked" if call_kind[c] else "recurrent", starts, ends if call_keep[c] else None))
            else:
                calls.append(Call(idx, cu, cu_cpu, starts, bool(call_keep[c])))
        levels.append(calls)
        launches.append([(int(call_kind[i]), seg_ptr[j] - seg_ptr[i], int(seg_len[seg_ptr[i] : seg_ptr[j]].max()) if call_kind[i] else 0,
                          at[4] + cu_at[cu_of[(i, j)]], at[1] + row_ptr[i], at[2] + seg_ptr[i] if d else -1, at[3] + seg_ptr[i] if call_keep[i:j].any() else -1)
                         for i, j in (lv if indexed else ())])
    program = None
    if len(a["program"]):
        program = [[] for _ in levels]
        first = at[7]
        for d, mode, n, longest, *places in a["program"].tolist():
            program[d].append((mode, n, longest, *(first + o if o >= 0 else -1 for o in places)))
    seg_of_row = a["seg_of_row"]
    return TreePlan(conv.view(-1, 4), levels, a["n_segments"], path, a["n_keep"].tolist() if indexed else None, rows, sidx if rows is not None else None, seg_of_row,
                    a["seg_level"], a["seg_slot"], pad_rows=pad_rows, launches=launches if indexed else None, program=program, data=on_dev if indexed else None)


def _kept_state_requests(plan: TreePlan, cap):
    """cap["state"] = [(row, name)]: the final state of the segment that holds `row` -> {level: [(slot, name)]}"""
    by_level = {}
    for row, name in cap["state"]:
        sg = int(plan.seg_of_row[row])
        slot = int(plan.seg_slot[sg]) if sg >= 0 else -1
        if slot < 0:
            raise RuntimeError(f"gdn_tree: no kept state for row {row} (segment {sg}, slot {slot})")
        by_level.setdefault(int(plan.seg_level[sg]), []).append((slot, name))
    return by_level


@torch.compiler.disable
def gdn_tree(q, k, v, g, beta, plan: TreePlan, mod=None):
    """q, k [T, Hk, Dk] (l2-normalised), v [T, Hv, Dv], g, beta [T, Hv] -> o [T, Hv, Dv]: every segment starts from its
    parent's final state (spinf_serve/models/qwen35/qwen.py:514-590).  Both kernels index the stream rows themselves, so a level
    costs at most two launches and no gathers.

    Capture (extraction, qwen.py:520-526,558-565): with plan.cap = {"tok": [(first row, rows, name)], "state": [(row, name)],
    "out": {"gdn": {}, "state": {}}} the layer's scan inputs of the row ranges and the final states of the named rows' segments
    are kept under out[...][name][layer]."""
    cap = plan.cap
    layer = mod.li if mod is not None else -1
    wanted = {}
    if cap is not None:
        for first, count, name in cap["tok"]:
            rows = slice(first, first + count)
            cap["out"]["gdn"].setdefault(name, {})[layer] = (q[rows].clone(), k[rows].clone(), v[rows].clone(), g[rows].clone(), beta[rows].clone())
        wanted = _kept_state_requests(plan, cap)
    scale = q.shape[-1] ** -0.5
    if plan.pad_rows is not None and len(plan.seg_of_row) == v.shape[0]:
        o = torch.empty_like(v)      # every covered row is written by a kernel; only the pads need the zero fill
        if plan.pad_rows.numel():
            o.index_fill_(0, plan.pad_rows, 0)
    else:
        o = torch.zeros_like(v)
    g32 = g if g.dtype == torch.float32 else g.float()
    b16 = beta if beta.dtype == torch.bfloat16 else beta.to(torch.bfloat16)
    indexed = plan.path == "indexed"
    args = gdn.level_args(q, k, v, g32, b16, o, scale, plan.data) if indexed and plan.launches is not None else None
    # a forest's nodes leave no states (and its kernel is built for 128 value dims): a caller that asks for states gets every level's
    launches = plan.launches if wanted or plan.program is None or v.shape[-1] != 128 else plan.program
    base = plan.data.data_ptr() if args is not None else 0
    run, stream = _lib.load_library().spinf_gdn_fwd, _lib.raw_stream(q.device.index)
    above = None   # the states the level above left
    for d, calls in enumerate(plan.levels):
        if args is not None and launches is plan.program:
            n_slots = plan.n_keep[d] if any(launch[-1] >= 0 for launch in launches[d]) else 0
        else:
            n_slots = plan.n_keep[d] if indexed else sum(len(c.cu_cpu) - 1 for c in calls if c.keep)
        states = q.new_empty((n_slots, v.shape[1], q.shape[-1], v.shape[-1]), dtype=torch.float32) if n_slots else None
        next_slot = 0
        if args is not None:
            h0, ht = None if above is None else above.data_ptr(), None if states is None else states.data_ptr()
            for args.mode, args.n_seg, args.max_len, cu, idx, h0_idx, ht_idx in launches[d]:
                args.cu, args.idx = base + 8 * cu, base + 8 * idx
                args.h0, args.h0_idx = (h0, base + 8 * h0_idx) if h0_idx >= 0 else (None, None)
                args.ht, args.ht_idx = (ht, base + 8 * ht_idx) if ht_idx >= 0 else (None, None)
                _lib.launch(run, args, q.device, "spinf_gdn_fwd", stream)
            calls = ()
        for c in calls:
            n_seg = len(c.cu_cpu) - 1
            if indexed:
                h0_idx, ht_idx, kind = c.h0_idx, c.ht_idx, c.kind
            else:   # levels path: a keeping call's segments take the next slots in order
                h0_idx = c.parent
                ht_idx = torch.arange(next_slot, next_slot + n_seg, device=q.device) if c.keep else None
                next_slot += n_seg if c.keep else 0
                kind = "chunked" if int((c.cu_cpu[1:] - c.cu_cpu[:-1]).max()) > 64 else "recurrent"
            kw = dict(h0=above if h0_idx is not None else None, h0_idx=h0_idx, ht=states if ht_idx is not None else None, ht_idx=ht_idx, idx=c.idx, o=o[None])
            if kind == "recurrent":
                gdn.recurrent(q[None], k[None], v[None], g32[None], b16[None], scale, c.cu, n_seg, **kw)
            else:
                gdn.chunked(q[None], k[None], v[None], g32[None], b16[None], scale, c.cu, c.cu_cpu, **kw)
        for slot, name in wanted.get(d, ()):
            cap["out"]["state"].setdefault(name, {})[layer] = states[slot].clone()
        above = states
    return o
