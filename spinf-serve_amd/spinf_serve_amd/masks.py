"""The mask side of the attention boundary: what Scorer._init_flex / Scorer._block_masks build per forward
(spinf_serve/scorer.py:163-238), as an opaque handle the attention op understands.

A TreeMask holds the stream's art / end / pos on the device and, instead of FlexAttention's nb x nb block tables
(spinf_serve/packer.py:426-491), a compact per-query-tile list of visible key tiles compiled on the host by the
library's tile-plan compiler: for the window and the key-tile size the layers ask for, at the first layer that asks (a pass
whose global layers have 512-dim heads never compiles the 64-key plan of its global mask) or ahead of it (TreeMask.prepare).
No dense mask is built anywhere.
"""

from __future__ import annotations

import ctypes as C
import threading
import weakref

import numpy as np

from . import _lib


class TilePlan:
    """a compiled plan (see include/spinf_tree.h): the native handle, and on first use its host arrays qt_ptr, kv_idx, kv_bits, order"""

    def __init__(self, handle, counts, n, window, grp_mode=0, ktile=64):
        self._handle = handle
        self.ktile = ktile
        self.n_qtiles, self.n_entries, self.active_blocks, self.masked_blocks = (int(c) for c in counts[:4])
        self.n, self.window, self.grp_mode = n, window, grp_mode
        self._schedules = {}
        self._arrays = None

    def __del__(self):
        h, self._handle = getattr(self, "_handle", None), None
        if h:
            try:
                _lib.load_library().spinf_tileplan_free(h)
            except Exception:  # noqa: BLE001  (interpreter shutdown)
                pass

    @classmethod
    def build(cls, art, end, pos, window=None, grp=None, grp_windowed=False, ktile=64) -> "TilePlan":
        """grp (image groups, spinf_serve/scorer.py:184-198): [n] int32, -1 none; the tokens of a group also see each other both
        ways, past the window unless grp_windowed.  ktile: keys per entry, 64, or 32 for the head dim 512 kernel."""
        host = _host_arrays(art, end, pos, grp)
        return cls.compile([None if a is None else a.ctypes.data for a in host], len(host[0]), window, grp_windowed, ktile)

    @classmethod
    def compile(cls, at, n, window, grp_windowed, ktile) -> "TilePlan":
        """build from the addresses of art, end, pos and grp (None: no groups), int32 [n] each"""
        lib = _lib.load_library()
        w = int(window) if window else 0
        h = C.c_void_p()
        mode = 0 if at[3] is None else 2 if grp_windowed else 1
        _lib.check(lib.spinf_tileplan_build_ktile(*at, mode, n, w, int(ktile), C.byref(h)), "tileplan_build")
        counts = (C.c_int64 * 5)()
        _lib.check(lib.spinf_tileplan_counts(h, counts), "tileplan_counts")
        return cls(h, counts, n, w, mode, int(ktile))

    def export(self, qt_ptr, kv_idx, kv_bits, order) -> None:
        """the plan's arrays into host memory at these addresses (qt_ptr [n_qtiles + 1], kv_idx / kv_bits [entries], order [n_qtiles])"""
        _lib.check(_lib.load_library().spinf_tileplan_export(self._handle, qt_ptr, kv_idx, kv_bits, order), "tileplan_export")

    def _array(self, i):
        if self._arrays is None:
            out = [np.zeros(max(k, 1), t) for k, t in ((self.n_qtiles + 1, np.int32), (self.n_entries, np.int32), (self.n_entries, np.uint32), (self.n_qtiles, np.int32))]
            self.export(*(x.ctypes.data for x in out))
            self._arrays = [out[0], out[1][: self.n_entries], out[2][: self.n_entries], out[3][: self.n_qtiles]]
        return self._arrays[i]

    qt_ptr = property(lambda self: self._array(0))
    kv_idx = property(lambda self: self._array(1))
    kv_bits = property(lambda self: self._array(2))
    order = property(lambda self: self._array(3))

    def schedule_into(self, head_groups: int, n_lists: int, items, list_ptr) -> None:
        """the work lists into host memory at these addresses: items [4 n_qtiles head_groups], list_ptr [9] or, for a static schedule
        (n_lists > 0), [n_lists + 1]"""
        lib = _lib.load_library()
        if n_lists:
            _lib.check(lib.spinf_tileplan_schedule_static(self._handle, head_groups, n_lists, items, list_ptr), "tileplan_schedule_static")
        else:
            _lib.check(lib.spinf_tileplan_schedule(self._handle, head_groups, items, list_ptr), "tileplan_schedule")

    def _schedule(self, head_groups: int, n_lists: int):
        got = self._schedules.get((head_groups, n_lists))
        if got is None:
            items = np.zeros((max(self.n_qtiles * head_groups, 1), 4), np.int32)
            list_ptr = np.zeros((n_lists or 8) + 1, np.int32)
            self.schedule_into(head_groups, n_lists, items.ctypes.data, list_ptr.ctypes.data)
            got = self._schedules[(head_groups, n_lists)] = (items[: self.n_qtiles * head_groups], list_ptr)
        return got

    def schedule(self, head_groups: int):
        """-> (items [n_qtiles * head_groups, 4] int32, list_ptr [9] int32): the kernel's work lists"""
        return self._schedule(head_groups, 0)

    def schedule_static(self, head_groups: int, n_lists: int):
        """-> (items [n_qtiles * head_groups, 4] int32, list_ptr [n_lists + 1] int32): the items dealt out to n_lists workgroups
        ahead of the launch (the kernel with decoupled waves)"""
        return self._schedule(head_groups, n_lists)


def _host_arrays(art, end, pos, grp=None):
    art, end, pos = (np.ascontiguousarray(a, np.int32) for a in (art, end, pos))
    if len(end) != len(art) or len(pos) != len(art):
        raise ValueError("art, end and pos differ in length")
    if grp is not None:
        grp = np.ascontiguousarray(grp, np.int32)
        if len(grp) != len(art):
            raise ValueError("grp differs in length from art")
    return art, end, pos, grp


_CUS: dict = {}   # compute units by device index


def _static_lists(device) -> int:
    """workgroups of a static schedule on this device: one per compute unit"""
    import torch

    got = _CUS.get(device.index)
    if got is None:
        got = _CUS[device.index] = int(torch.cuda.get_device_properties(device).multi_processor_count)
    return got


def _staging(n: int, device):
    """-> host tensor of n int32, in pinned memory where it is to be copied to a GPU"""
    import torch

    return torch.empty(n, dtype=torch.int32, pin_memory=device.type == "cuda")


def _mark(device):
    """an event behind what the current stream of `device` has been given"""
    import torch

    with torch.cuda.device(device):
        event = torch.cuda.Event()
        event.record()
        return event


def _join(shared) -> bool:
    """the current stream waits for what made these tensors and is named to the allocator as a reader; False under capture, where neither
    can be done"""
    import torch

    with torch.cuda.device(shared.device):
        if torch.cuda.is_current_stream_capturing():
            return False
        stream = torch.cuda.current_stream()
        if shared.made is not None:
            stream.wait_event(shared.made)
        elif shared.home is not None:
            # (the default stream's handle is 0, and of a handle of 0 ExternalStream makes a new stream)
            home = torch.cuda.ExternalStream(shared.home) if shared.home else torch.cuda.default_stream()
            try:
                with torch.cuda.stream(home):
                    done = torch.cuda.is_current_stream_capturing()   # (torch waits for the device before a capture begins)
                if not done:
                    stream.wait_stream(home)
            except RuntimeError:   # a stream of the caller's own that is gone by now
                torch.cuda.synchronize()
        for t in shared.tensors:
            t.record_stream(stream)
        return True


class _Shared:
    """Device tensors that one stream made and calls on any stream may read.  Another stream's first call waits for what made them, and
    tells the allocator of its stream: a buffer that goes with the last reference is then not handed out while that stream
    still reads it.  The caller cannot do either, as the buffers are made behind its back by whichever call comes first.

    The wait is for the event `made` where there is one (TreeMask.prepare), else for all that the stream `home` has been given by then: an
    event behind every upload cost a new stream's two masks 54 us, on a path where hardly any program needs it."""

    __slots__ = ("tensors", "device", "home", "made", "streams")

    def __init__(self, *tensors, wait=True):
        self.tensors, self.made = tensors, None
        self.device = device = tensors[0].device
        on = _lib.raw_stream(device.index)
        self.home = on if wait else None
        self.streams = {on}

    def reach(self, stream) -> bool:
        """makes the tensors safe to read for the current stream (`stream`: its raw handle)"""
        if stream in self.streams:
            return True
        if not _join(self):
            return False
        self.streams.add(stream)
        return True


class TreeMask:
    """Device-side handle: the stream's metadata, and per key-tile size a plan compiled when the first call that takes it comes (a
    forward's layers share it).  ``seq_lengths`` mirrors BlockMask.seq_lengths (spinf_serve/models/qwen35/qwen.py:615 reads it).
    Host threads and streams may share a mask: what a first call makes (plan, uploads, prepared calls) is made once, under a lock, and a
    call on another stream waits for the copies.  (The metadata is copied at the build: as with any tensor, a stream that is to use
    the mask waits for the one it was built on.)"""

    def __init__(self, plan, meta, device, grp=None, host=None, window=None, ktile=64, lock=None):
        """plan: a compiled plan, or None: compiled from host = (art, end, pos, grp or None, grp_windowed, the four arrays' addresses) for
        this window and ktile"""
        self._lock = lock or threading.RLock()   # (one for both key-tile sizes: they refer to each other)
        self._host = host
        self._plan = plan
        self._ktile = plan.ktile if plan is not None else ktile
        self._other = None                  # the same mask with the other key-tile size
        self.grp = grp                      # device copy of the image groups, or None
        self.grp_mode = 0 if grp is None else plan.grp_mode if plan is not None else 2 if host[4] else 1
        self.n = plan.n if plan is not None else len(host[0])
        self.window = plan.window if plan is not None else int(window) if window else 0
        self.seq_lengths = (self.n, self.n)
        self.art, self.end, self.pos = meta
        self.device = self.art.device       # (of "cuda" the GPU that was current at the build, whatever is current at the first call)
        self._meta = ()                     # art, end, pos, grp as shared tensors, where a build copied them
        self._kv = None                     # the buffer with the device copies of the plan's kv_idx, kv_bits, and where they lie in it
        self._sched = {}
        self._layers = {}                   # prepared calls by head geometry (attention.py)
        self._rows = None

    def __reduce__(self):
        """copied and saved as what it is built from: plans and uploads belong to one object"""
        if self._host is None:
            raise TypeError("a mask around a compiled plan cannot be copied or saved")
        art, end, pos, grp, grp_windowed, _ = self._host
        return _built, (art, end, pos, self.window, str(self.device), grp, grp_windowed, self._ktile)

    @property
    def plan(self) -> TilePlan:
        if self._plan is None:
            with self._lock:
                if self._plan is None:
                    self._plan = TilePlan.compile(self._host[5], self.n, self.window, self._host[4], self._ktile)
        return self._plan

    @property
    def n_qtiles(self) -> int:
        return -(-self.n // 128)

    @property
    def kv_idx(self):
        return self._entries()[0]

    @property
    def kv_bits(self):
        return self._entries()[1]

    def _entries(self):
        if self._kv is None:
            self._schedule(1, 0)
        dev, at, shared = self._kv
        shared.reach(_lib.raw_stream(self.device.index))
        return dev[at[2] : at[3]], dev[at[3] : at[4]]

    def for_head_dim(self, d: int, ring: bool = False) -> "TreeMask":
        """the mask with the plan granularity the kernel takes: 32-key entries at head dim 512 and for the kernel with decoupled
        waves (ring), 64-key ones otherwise (each plan is compiled on first use; both share the device metadata)"""
        ktile = 32 if d == 512 or ring else 64
        if ktile == self._ktile:
            return self
        other = self._other
        other = other() if isinstance(other, weakref.ref) else other
        if other is None:
            if self._host is None:
                raise ValueError(f"this mask was built for key tiles of {self._ktile}; head dim {d} takes {ktile}")
            with self._lock:
                other = self._other() if isinstance(self._other, weakref.ref) else self._other
                if other is None:
                    other = TreeMask(None, (self.art, self.end, self.pos), self.device, self.grp, self._host, self.window, ktile, self._lock)
                    other._meta = self._meta
                    other._other = weakref.ref(self)   # (no cycle: a pass's masks go, and give their device memory back, with the last reference)
                    self._other = other
        return other

    def prepare(self, *heads, sidx=None) -> "TreeMask":
        """makes now, on the current stream, what the first calls of layers with these heads would make: heads = (query heads, key / value
        heads, head dim) per kind of layer, sidx as the calls will pass it.  For a program that builds its masks on a thread or a
        stream of its own: plans are compiled and uploaded there, what the compiler refuses is raised there, and a call on any
        stream waits for the uploads.  Without it the first call of a kind does it, on its thread and its stream."""
        import torch

        from . import attention

        shared = attention.prepare_calls(self, heads, sidx)
        if self.device.type == "cuda" and not torch.cuda.is_current_stream_capturing():
            event, here = _mark(self.device), _lib.raw_stream(self.device.index)
            for x in shared:
                if x.home == here:
                    x.made = event
        return self

    def rows(self, sidx):
        """compact rows (spinf_serve/models/qwen35/qwen.py:613-622): sidx [R] = stream position of each real row (a device
        tensor) -> (row_of [n], kv_row0 [entries]) int32 device tensors for the kernel: the row of each stream position (-1:
        pad) and, per plan entry, the row of its first key where its 64 keys are consecutive rows (else -1).  Kept for the
        sidx tensor it was built from, as it was then (one forward: every layer passes the same tensor)."""
        import torch

        version = 0 if sidx.is_inference() else sidx._version   # (counts changes in place; tensors of inference mode keep none)
        got = self._rows   # (read once: another thread's rows may replace them)
        if got is not None and got[0] is sidx and got[4] == version:
            got[3].reach(_lib.raw_stream(self.device.index))
            return got[1], got[2]
        n = self.n
        row_of = torch.full((n + 63,), -1, dtype=torch.int32, device=self.device)   # padded: every key tile is 64 long
        row_of[sidx.to(self.device, torch.long)] = torch.arange(sidx.shape[0], dtype=torch.int32, device=self.device)
        kt = self._ktile
        tiles = row_of[: (n + kt - 1) // kt * kt].view(-1, kt)
        run = (tiles - tiles[:, :1]) == torch.arange(kt, dtype=torch.int32, device=self.device)
        tile_row0 = torch.where((tiles[:, 0] >= 0) & run.all(1), tiles[:, 0], torch.full_like(tiles[:, 0], -1))
        kv_row0 = tile_row0[self.kv_idx.long()].contiguous()
        row_of = row_of[:n].contiguous()
        self._rows = (sidx, row_of, kv_row0, _Shared(row_of, kv_row0), version)
        return row_of, kv_row0

    def _upload(self, head_groups: int, n_lists: int):
        """one staging buffer, one copy: items | list_ptr and, with the plan's first schedule, kv_idx | kv_bits.  (A copy per array, each
        from pinned memory of its own, was 11 copies and 150 us of a new stream's two masks.)"""
        plan, first = self.plan, self._kv is None
        ni, nl, ne, nq = 4 * max(plan.n_qtiles * head_groups, 1), (n_lists or 8) + 1, max(plan.n_entries, 1), plan.n_qtiles
        at = (0, ni, ni + nl, ni + nl + ne, ni + nl + 2 * ne)   # items (16-byte aligned), list_ptr, kv_idx, kv_bits, host only: qt_ptr, order
        buf = _staging(at[4] + 2 * nq + 1 if first else at[2], self.device)
        p = buf.data_ptr()
        plan.schedule_into(head_groups, n_lists, p, p + 4 * at[1])
        if first:
            plan.export(p + 4 * at[4], p + 4 * at[2], p + 4 * at[3], p + 4 * (at[4] + nq + 1))
            buf = buf[: at[4]]
        dev = buf.to(self.device, non_blocking=True)
        shared = _Shared(dev)
        if first:
            self._kv = dev, at, shared
        got = self._sched[(head_groups, n_lists)] = dev, at, plan.n_qtiles * head_groups, shared
        return got

    def _schedule(self, head_groups: int, n_lists: int):
        got = self._sched.get((head_groups, n_lists))
        if got is None:
            with self._lock:   # (two first calls at a time: the second one's buffers would replace the ones the first is about to read)
                got = self._sched.get((head_groups, n_lists)) or self._upload(head_groups, n_lists)
        return got

    def schedule(self, head_groups: int, n_lists: int = 0):
        """device copy of the work lists for this many head groups (built on first use, then kept); n_lists > 0: the static
        schedule for that many workgroups"""
        dev, at, n_items, shared = self._schedule(head_groups, n_lists)
        shared.reach(_lib.raw_stream(self.device.index))
        return dev[: at[1]].view(-1, 4), dev[at[1] : at[2]], n_items

    def pointers(self, head_groups: int, n_lists: int):
        """-> device addresses of items, list_ptr, kv_idx, kv_bits, the number of items, and the shared tensors the addresses lie in
        (whoever keeps an address keeps its tensor, and a stream that reads it reaches it)"""
        dev, at, n_items, shared = self._schedule(head_groups, n_lists)
        kv, kv_at, kv_shared = self._kv
        items, entries = dev.data_ptr(), kv.data_ptr()
        return items, items + 4 * at[1], entries + 4 * kv_at[2], entries + 4 * kv_at[3], n_items, (shared, kv_shared)

    @classmethod
    def build(cls, art, end, pos, window=None, device="cuda", meta=None, grp=None, grp_windowed=False, grp_dev=None):
        """the handle of a stream: its metadata is copied to the device; ``meta``: device art / end / pos tensors to share with another
        mask; grp: image groups (see TilePlan.build), grp_dev: their device copy to share"""
        import torch

        device = torch.device(device)
        if len(art) > 1 << 30:   # (what the plan compiler, which comes later, would refuse)
            raise ValueError(f"a stream of {len(art)} tokens is too long")
        host = _host_arrays(art, end, pos, grp)
        n, at = len(host[0]), [None] * 4
        given = [i for i in range(4) if host[i] is not None and not (grp_dev is not None if i == 3 else meta is not None)]
        shared = ()
        if given:
            buf = _staging(len(given) * n, device).view(len(given), n)
            rows, base, host = buf.numpy(), buf.data_ptr(), list(host)
            for r, i in enumerate(given):
                rows[r] = host[i]
                host[i], at[i] = rows[r], base + 4 * n * r   # (the caller may reuse its arrays)
            dev = buf.to(device, non_blocking=True)
            shared = (_Shared(dev, wait=False),)
            if meta is None:
                meta = tuple(dev[:3])
            if 3 in given:
                grp_dev = dev[-1]
        for i, h in enumerate(host):
            if h is not None and at[i] is None:
                at[i] = h.ctypes.data
        mask = cls(None, meta, device, grp_dev if grp is not None else None, (*host, grp_windowed, at), window)
        mask._meta = shared
        return mask


def _built(art, end, pos, window, device, grp, grp_windowed, ktile):
    mask = TreeMask.build(art, end, pos, window, device, grp=grp, grp_windowed=grp_windowed)
    mask._ktile = ktile
    return mask


def block_masks(batch, sliding_window=None, device="cuda", grp=None, bidir_all=True):
    """-> {"full_attention": TreeMask, "sliding_attention": TreeMask}: the dict Scorer._block_masks returns
    (spinf_serve/scorer.py:207-238).  With a window the sliding plan is always built (the reference's always_window,
    spinf_serve/packer.py:448-450); without one both keys name the global mask.
    grp: image groups of the stream's tokens (-1 none).  bidir_all (the model's _vision_bidir_all, scorer.py:186-198): the
    tokens of an image see each other both ways on every layer and past the window; otherwise on the sliding layers only,
    within the window, and the global layers stay causal."""
    full = TreeMask.build(batch.art, batch.end, batch.pos, None, device, grp=grp if bidir_all else None)
    if not sliding_window:
        return {"full_attention": full, "sliding_attention": full}
    meta = (full.art, full.end, full.pos)
    if grp is None or bidir_all:
        slid = TreeMask(None, meta, full.device, full.grp, full._host, sliding_window)
        slid._meta = full._meta
    else:
        slid = TreeMask.build(*full._host[:3], sliding_window, device, meta=meta, grp=grp, grp_windowed=True)
        slid._meta += full._meta
    return {"full_attention": full, "sliding_attention": slid}
