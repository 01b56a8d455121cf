"""Input-embedding gradient by sorted scatter, and a row-sparse AdamW with dense results.

Mirror of `build_id_groups` and the `_embed_dw_scatter` launch (ancora/kernels/fused.py:387-424,
used at ancora/model/resident_moe_model.py:262-271, 333-334). `RowSparseAdamW` has no counterpart
in the reference, whose AdamW sweeps the whole embedding every step (ancora/optim/adamw.py:92-97):
it updates only the rows a step's tokens touch and replays the steps a row missed when the row is
next needed, so that every row it hands out is bit-identical to the dense optimizer's.
"""
import ctypes
import threading

import numpy as np

from . import _lib
from ._lib import api, AdamWHyper, FORM_DIV, FORM_IBC
from .adamw import sr_seed_base
from .devbuf import DevBuf
from .gradnorm import ctl_ptr


def _ids32(ids):
    """Ids of any type as a contiguous int32 vector: fractions are cut off, what 32 bits do not hold wraps (an
    unsigned -1 as padding), and a row outside the table is left out by the kernels."""
    ids = np.asarray(ids).reshape(-1)
    with np.errstate(invalid="ignore"):
        return np.ascontiguousarray(ids, dtype=np.int32)


def _id_groups(ids_flat):
    """((4, M) int32: srt, start, cnt, gid; number of groups)."""
    _lib.load()
    ids = _ids32(ids_flat)
    out = np.empty((4, ids.size), np.int32)
    n = ctypes.c_int64(0)
    p, step = out.ctypes.data, 4 * ids.size
    api.anc_id_groups(ids.ctypes.data, ids.size, p, p + step, p + 2 * step, p + 3 * step, ctypes.byref(n))
    return out, n.value


def build_id_groups(ids_flat):
    """Stable-sort token ids into groups (ancora/kernels/fused.py:411-424). Returns
    (srt, start, cnt, gid), each (M, 1) int32: srt the stable argsort; for group g (one per
    distinct id, ascending) start[g] its first position in srt, cnt[g] its size, gid[g] its id;
    groups beyond the last are padding with cnt = 0."""
    out, _ = _id_groups(ids_flat)
    return tuple(a.reshape(-1, 1) for a in out)


class _Blocks:
    """Device blocks of the group arrays, kept between steps: an allocation and a release per step cost more than
    the arrays' upload, and a release waits for the whole device. A block given back may still be read by work in
    flight on any stream, so it is handed out again only after a device synchronisation, one for every
    KEEP blocks. A device's blocks stay on that device; at most 2 * KEEP of each are kept, `trim` gives them back."""

    KEEP = 8

    def __init__(self):
        self._lock = threading.Lock()
        self._ready, self._waiting = {}, {}          # device -> blocks

    def get(self, nbytes):
        dev = _lib.current_device()
        with self._lock:
            idle = self._waiting.pop(dev) if len(self._waiting.get(dev, ())) >= self.KEEP else []
        if idle:
            api.anc_device_sync()                    # (outside the lock: other threads need not wait for this device)
        with self._lock:
            ready = self._ready.setdefault(dev, [])
            ready += idle
            ready.sort(key=lambda b: b.nbytes)
            spare, ready[:] = ready[:-self.KEEP], ready[-self.KEEP:]
            block = next((ready.pop(i) for i, b in enumerate(ready) if nbytes <= b.nbytes <= 4 * nbytes + 65536), None)
        for b in spare:
            b.free()
        if block is None:
            block = DevBuf.empty((max(nbytes, 4096),), np.uint8)
            block.device = dev
        return block

    def put(self, b):
        with self._lock:
            waiting = self._waiting.setdefault(b.device, [])
            if len(waiting) < self.KEEP:
                waiting.append(b)
                return
        b.free()

    def trim(self):
        with self._lock:
            blocks = [b for kept in (self._ready, self._waiting) for bs in kept.values() for b in bs]
            self._ready, self._waiting = {}, {}
        for b in blocks:
            b.free()


_blocks = _Blocks()
trim_pool = _blocks.trim


class _GroupArray(DevBuf):
    """One of the group arrays. Its address is the caller's to use on any stream, so asking for it waits until the
    arrays are in place; the library's own launches on the stream they were sent on need not wait."""

    def __init__(self, owner, row):
        self.owner, self.row = owner, row
        self.shape, self.dtype, self.nbytes, self._owner = (owner.M, 1), np.dtype(np.int32), 4 * owner.M, False

    @property
    def ptr(self):
        return self.owner.settled() + self.row * self.nbytes

    def ptr_on(self, si):
        return self.owner.base_on(si) + self.row * self.nbytes

    def free(self):
        pass


class IdGroups:
    """The four group arrays, plus the number of distinct ids. They travel to the device with the first
    launch that uses them, in its stream's order; if that stream is being captured into a graph they are in place
    before it, once, and the graph's replays read them there."""

    def __init__(self, ids_flat):
        _lib.init()
        self._arrays, self.n_groups = _id_groups(ids_flat)
        self.M = self._arrays.shape[1]
        if self.M == 0:
            raise ValueError("IdGroups: no ids")
        self._block = _blocks.get(self._arrays.nbytes)         # (here: a capture may not allocate)
        self._si, self._settled = None, False
        self.srt, self.start, self.cnt, self.gid = (_GroupArray(self, i) for i in range(4))

    @property
    def host(self):
        """The arrays as `build_id_groups` returns them."""
        return tuple(a.reshape(-1, 1) for a in self._arrays)

    def base_on(self, si):
        """Device address of the arrays for work queued on stream `si`."""
        if self._block is None:
            raise _lib.AncoraError("IdGroups: freed")
        if self._si is None and not self._settled and not _lib.stream_is_capturing(si):
            api.anc_upload_async(self._block.ptr, self._arrays.ctypes.data, self._arrays.nbytes, int(si))
            self._si = si
        elif self._si != si:
            return self.settled()
        return self._block.ptr

    def settled(self):
        """Device address of the arrays, in place for any stream."""
        if self._block is None:
            raise _lib.AncoraError("IdGroups: freed")
        if not self._settled:
            if self._si is None:
                api.anc_upload_now(self._block.ptr, self._arrays.ctypes.data, self._arrays.nbytes)
            else:
                _lib.stream_sync(self._si)
            self._settled = True
        return self._block.ptr

    def free(self):
        if self._block is not None:
            _blocks.put(self._block)
            self._block = None


def embed_dw_scatter(groups, dy, si, out=None, compact=None, V=None):
    """dy: (M, H) bf16 DevBuf. out: (V, H) fp32 DevBuf, added onto in place (the reference's
    launch); or compact: (M, H) fp32 DevBuf that receives one summed row per group."""
    M, H = dy.shape
    if out is not None:
        V = out.shape[0] if V is None else V
    base, step = groups.base_on(si), 4 * groups.M          # srt, start, cnt, gid
    api.anc_embed_dw_scatter(base + 2 * step, base + step, base + 3 * step, base, dy.ptr,
                             0 if out is None else out.ptr, 0 if compact is None else compact.ptr,
                             M, 0 if V is None else V, H, int(si))


class RowSparseAdamW:
    """AdamW over one (V, H) fp32 tensor that steps only the rows named per step.

        opt = RowSparseAdamW(W, lr=3e-4, ...)
        opt.catch_up(row_ids, si)          # before the forward gathers these rows: p32/p16 current
        opt.step(groups.gid, n_groups, compact_grads, si, guard)   # after the backward
        opt.flush(si)                      # every row current (before a checkpoint / evaluation)

    State after `flush` equals the dense `AdamW` run on gradients that are zero outside the touched
    rows, bit for bit (stochastic rounding included). `lr` may change between steps."""

    def __init__(self, W, lr=3e-4, betas=(0.9, 0.95), eps=1e-8, wd=0.01, form="div", sr=False, seed=0,
                 tensor_seed=0, max_steps=1 << 16):
        _lib.init()
        W = np.ascontiguousarray(W, dtype=np.float32)
        if W.ndim != 2 or W.shape[1] % 64:
            raise ValueError(f"RowSparseAdamW: (V, H) tensor with H % 64 == 0 expected, got {W.shape}")
        self.V, self.H = W.shape
        self.lr, (self.b1, self.b2), self.eps, self.wd = lr, betas, eps, wd
        self.form, self.sr, self.seed, self.tensor_seed = form, bool(sr), int(seed), int(tensor_seed)
        self.t = 0
        self.p32 = DevBuf(W)
        self.p16 = DevBuf.zeros(W.shape, np.uint16)
        self.m = DevBuf.zeros(W.shape, np.float32)
        self.v = DevBuf.zeros(W.shape, np.float32)
        self.last = DevBuf.zeros((self.V,), np.int32)
        self._cap = int(max_steps)
        self.table = DevBuf.zeros((self._cap + 1, 4), np.uint32)
        self._rows_buf, self._rows_si = None, 0
        self.last_skipped = False
        self._filled_to = 0          # table entries 1 .. _filled_to hold the scalars of their steps
        self._filled_lr = None       # ... computed with this learning rate

    def _hyper(self):
        return AdamWHyper(beta1=self.b1, beta2=self.b2, omb1=1 - self.b1, omb2=1 - self.b2, eps=self.eps,
                          lr=0.0, bc1=1.0, bc2=1.0, form=FORM_DIV if self.form == "div" else FORM_IBC,
                          sr=int(self.sr), seed_base=0)

    FILL_AHEAD = 256

    def _step_record(self, t, lr):
        bc1, bc2 = 1 - self.b1 ** t, 1 - self.b2 ** t
        if self.form != "div":
            bc1, bc2 = 1.0 / bc1, 1.0 / bc2
        rec = np.zeros(4, np.uint32)
        rec[:3] = np.array([bc1, bc2, lr], np.float32).view(np.uint32)
        rec[3] = sr_seed_base(self.seed, t) if self.sr else 0
        return rec

    def _ensure_step(self, t, si):
        """Table entry t holds step t's scalars at the current learning rate. Entries are written
        FILL_AHEAD steps at a time, so a run at a constant learning rate uploads (and synchronises)
        once per FILL_AHEAD steps instead of at every step; a changed learning rate rewrites from t
        on (earlier entries keep the rate their steps ran with: the replay needs it)."""
        if t <= self._filled_to and self._filled_lr == self.lr:
            return
        hi = min(self._cap, t + self.FILL_AHEAD - 1)
        block = np.stack([self._step_record(s, self.lr) for s in range(t, hi + 1)])
        DevBuf(shape=block.shape, dtype=np.uint32, ptr=self.table.ptr + 16 * t).upload(block, si)
        self._filled_to, self._filled_lr = hi, self.lr

    def _rows(self, rows, si):
        if self._rows_buf is None or self._rows_buf.size < rows.size:
            if self._rows_buf is not None:
                _lib.stream_sync(self._rows_si)
                self._rows_buf.free()
            self._rows_buf = DevBuf.empty((max(rows.size, 1024),), np.int32)
        elif self._rows_si != si:
            _lib.stream_sync(self._rows_si)        # the buffer's last reader ran on another stream
        self._rows_si = si
        api.anc_upload_async(self._rows_buf.ptr, rows.ctypes.data, rows.nbytes, int(si))
        return self._rows_buf, rows.size

    def _launch(self, rows_ptr, n_rows, grads_ptr, t_now, ctl, si):
        h = self._hyper()
        api.anc_adamw_rows(rows_ptr, n_rows, grads_ptr, self.m.ptr, self.v.ptr, self.p32.ptr, self.p16.ptr,
                           self.last.ptr, self.V, self.H, self.table.ptr, int(t_now), ctypes.byref(h),
                           float(self.wd), self.tensor_seed, int(ctl), int(si))

    def catch_up(self, row_ids, si):
        """Replay, on the distinct rows in `row_ids` (host integers), the steps they missed."""
        if self.t == 0:
            return
        ids = _ids32(row_ids)
        rows, n = np.empty(ids.size, np.int32), ctypes.c_int64(0)
        api.anc_unique_ids(ids.ctypes.data, ids.size, rows.ctypes.data, ctypes.byref(n))
        buf, n = self._rows(rows[:n.value], si)
        self._launch(buf.ptr, n, 0, self.t, 0, si)

    def step(self, gid, n_groups, grads, si, guard=None):
        """gid: device int32 array of distinct row ids (e.g. `IdGroups.gid`), the first n_groups
        valid; grads: (>= n_groups, H) fp32 DevBuf, row i the gradient of gid[i]."""
        if self.t + 1 > self._cap:             # before the counter moves: t always matches the table
            raise RuntimeError(f"RowSparseAdamW: step table holds {self._cap} steps; raise max_steps")
        self._ensure_step(self.t + 1, si)
        self.t += 1
        if n_groups > 0:
            rows = gid.ptr_on(si) if isinstance(gid, _GroupArray) else gid.ptr
            self._launch(rows, int(n_groups), grads.ptr, self.t, ctl_ptr(guard), si)
        self.last_skipped = False
        if guard is not None:
            if guard.read(si)["skip"]:             # (synchronises)
                self.t -= 1
                self.last_skipped = True

    def flush(self, si):
        """Bring every row up to date."""
        if self.t:
            self._launch(0, self.V, 0, self.t, 0, si)

    def master(self):
        return self.p32.to_numpy()

    def free(self):
        for b in (self.p32, self.p16, self.m, self.v, self.last, self.table, self._rows_buf):
            if b is not None:
                b.free()
