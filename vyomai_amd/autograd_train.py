"""torch.autograd.Function wrappers whose forward AND backward are HIP kernel launches.

PyTorch supplies the tape only.  Parameters stay fp32 (master weights); activations and the
weights the kernels read are bf16 copies (``_shadow``), refreshed by the fused AdamW kernel when
the FlatTrainer owns the parameters.

Gradient delivery has two modes per parameter:
  * direct   -- ``param.grad`` is a preallocated fp32 view into the trainer's flat gradient arena
               (``param._vy_direct``): wgrad kernels accumulate straight into it (no temporaries,
               contiguous buckets for the RCCL reducer) and autograd receives ``None``;
  * returned -- otherwise a fresh fp32 gradient is computed and handed back to autograd.
"""
from __future__ import annotations

import ctypes
import functools
import itertools
import os
import weakref
from typing import Optional

import torch

from . import _lib, ops
from ._lib import ACT_GELU_ERF, ACT_NONE, VyomHipError
from .layers.attention import _shadow
from .layers.mask import AttnMask
from .layers.positional_embeddings import resolve_freqs

BF16 = torch.bfloat16
_ref = ctypes.addressof


_EPOCHS = itertools.count()


class _WtRegistry:
    """Every W^T the dgrad GEMMs read, of the parameters of one trainer (and one registry for parameters without).  The first backward
    transposes each matrix as it meets it; from then on ONE vy_transpose_batched launch per weight epoch refreshes all that were used
    in the previous epoch (the per-matrix launches are latency-bound: ~8 us each, 50 per step).  An epoch ends with a step of
    the trainer, whose AdamW kernel rewrites weights without touching tensor versions; its number is used once in a process.  Models that
    are trained in turn have an epoch each: one for all had the other models' matrices transposed at every step, and this one's
    one by one.  Owners are held weakly: a model that is dropped, or no longer trained, falls out of the batch."""

    def __init__(self) -> None:
        self.entries = []      # [weakref(owner), key_fn, src_fn, dst_view, last_used_epoch, number of the registry]
        self.batches = {}
        self.number = self.epoch = next(_EPOCHS)
        self.before = self.epoch_done = -1

    def bump(self) -> None:
        self.before, self.epoch = self.epoch, next(_EPOCHS)

    def register(self, owner, key_fn, src_fn, dst):
        e = [weakref.ref(owner), key_fn, src_fn, dst, self.epoch, self.number]
        self.entries.append(e)
        return e

    def refresh(self) -> None:
        """Re-transpose the recently used matrices for the current epoch (once per epoch)."""
        ep = self.epoch
        if self.epoch_done == ep:
            return
        self.epoch_done = ep
        entries, live = [], {}
        for e in self.entries:
            owner = e[0]()
            if owner is None or owner._vy_wt_entry is not e:
                continue
            entries.append(e)
            if e[4] == ep or e[4] == self.before:
                key, members = e[1](owner)
                if owner._vy_wt_key != key:
                    src = e[2](owner, members)
                    live.setdefault(src.dtype, []).append((owner, key, src, e[3]))
        self.entries = entries
        # one launch per dtype (a bf16 model and an fp32 one that no trainer owns share a registry)
        for dt, sub in live.items():
            keys = [(src.data_ptr(), dst.data_ptr()) for _, _, src, dst in sub]
            batch = self.batches.get(dt)
            if batch is None or batch.keys != keys:
                batch = self.batches[dt] = ops.TransposeBatch([(src, dst) for _, _, src, dst in sub])
            batch.run()
            for owner, key, *_ in sub:
                owner._vy_wt_key = key


_WT = _WtRegistry()


def _wt_cached(owner, reg: _WtRegistry, key, key_fn, src_fn, members=None) -> torch.Tensor:
    """Shared body of _wt / _wt_packed: owner carries _vy_wt_key / _vy_wt_view / _vy_wt_entry.
    key_fn / src_fn take the owner as their argument (the registry must not keep it alive); key, members: what key_fn returns now."""
    view = getattr(owner, "_vy_wt_view", None)
    if view is not None:
        entry = owner._vy_wt_entry
        if entry[5] != reg.number or entry[0]() is not owner:      # (the parameter has gone over to another trainer; a copy of a module)
            entry = owner._vy_wt_entry = reg.register(owner, key_fn, src_fn, view)
        entry[4] = reg.epoch
        if owner._vy_wt_key == key:
            return view
    src = src_fn(owner, members)
    if view is not None and view.dtype == src.dtype and view.device == src.device:
        reg.refresh()   # weights changed: all recently used matrices in one launch
        if owner._vy_wt_key != key:
            ops.transpose(src, view)   # not in the batch (first use after a pause, or an in-place edit)
            owner._vy_wt_key = key
        return view
    N, K = src.shape
    ld = _row_stride(N)
    view = torch.zeros((K, ld), dtype=src.dtype, device=src.device)[:, :N]  # pad columns stay zero
    ops.transpose(src, view)
    owner._vy_wt_view, owner._vy_wt_key = view, key
    owner._vy_wt_entry = reg.register(owner, key_fn, src_fn, view)
    return view


_ROW_GRANULE = int(os.environ.get("VY_ROW_GRANULE", "64"))   # (8: rows on 16 bytes, for A/B runs)


def _row_stride(n: int) -> int:
    """Row stride (elements) of a matrix with n columns that a GEMM reads as an operand: whole 128-byte lines per row
    (64 bf16), so that no row starts in the middle of a line.  With rows on 16 bytes the 50265-wide logits had a
    100,544-byte stride: every second row of the dgrad / wgrad operand began 64 bytes into a line and each 128-byte piece an
    LDS-DMA instruction fetches came from two lines."""
    g = _ROW_GRANULE
    return (n + g - 1) // g * g


def _wt(param: torch.Tensor, dtype) -> torch.Tensor:
    """W^T ([K, N], row stride padded to 8) of a 2-D parameter in `dtype`, cached per version."""
    reg = getattr(param, "_vy_weights", _WT)
    return _wt_cached(param, reg, (param._version, reg.epoch, dtype), lambda p: ((p._version, getattr(p, "_vy_weights", _WT).epoch, dtype), None),
                      lambda p, _: _shadow(p, dtype))


def _direct(p: Optional[torch.Tensor]) -> bool:
    return p is not None and getattr(p, "_vy_direct", False) and p.grad is not None


def _notify(*params) -> None:
    for p in params:
        if p is not None:
            cb = getattr(p, "_vy_ready", None)
            if cb is not None:
                cb(p)


_graph_task = torch._C._current_graph_task_id


class _Waiting:
    """What waits of one backward pass on one device, in one group.  The pass's callback alone holds it, so it goes with its pass, whether that ends
    or raises."""

    __slots__ = ("at", "number", "items", "tiles", "armed", "key", "stream", "__weakref__")
    numbers = itertools.count(1)

    def __init__(self, at=None):
        self.at, self.number = at, next(self.numbers)     # (backward pass, device), None: of none; what its parameters are marked with
        self.items, self.tiles, self.armed, self.key, self.stream = [], 0, False, None, None

    def unmark(self, items) -> None:
        for *_, members in items:
            for p in members:
                if getattr(p, "_vy_deferred", False) == self.number:     # (not of a later pass)
                    p._vy_deferred = False

    def __del__(self):
        self.unmark(self.items)


class _WgradGroup:
    """Weight gradients that accumulate straight into the gradient arena do not have to be launched where
    autograd reaches them: the projections of a layer are small wgrad problems (9-36 tiles of 256 x 256),
    and one at a time each needs M-splits -- fp32 atomic traffic -- to fill the chip.  They are collected
    here and go out as ONE launch per chip of tiles, ~2 layers (ops.linear_wgrad_grouped); the parameters are reported ready
    (per-bucket AdamW) when that launch has been enqueued, and its operands live until then (0.4 GB a layer at 16384 rows of
    768).  Parameters whose gradients are exchanged between ranks (training.BucketReducer) go out layer by layer: their buckets
    wait for the launch, and the exchange is what has to begin early.  Whatever is still pending when the backward pass ends is
    flushed by an autograd-engine callback.

    Every backward pass has its own (_Waiting): two threads' passes end at different times, one that raises launches nothing and leaves
    nothing to the next, and the engine calls a pass's backward functions in a thread for each device."""

    TILES = int(os.environ.get("VY_WGRAD_GROUP_TILES", "256"))   # most 256 x 256 output tiles of a launch: a CU each (a post-LN layer of 768: 108)
    MOST = 12                                                    # gradients of a launch
    EXCHANGED, EXCHANGED_MOST = 100, 8                           # exchanged gradients: as many tiles or gradients end a launch

    def __init__(self):
        self.passes = weakref.WeakValueDictionary()   # (backward pass, device) -> _Waiting
        self.outside = _Waiting()                     # of no pass (nothing flushes it)

    def _now(self, device) -> _Waiting:
        task = _graph_task()
        if task < 0:
            return self.outside
        w = self.passes.get((task, device))
        if w is None:
            w = self.passes[(task, device)] = _Waiting((task, device))
            torch.autograd.Variable._execution_engine.queue_callback(functools.partial(self._end_of_backward, w))
            w.armed = True
        return w

    def _here(self) -> list:
        """Of the backward pass that asks, on every device."""
        task = _graph_task()
        if task < 0:
            return [self.outside]
        return [w for w in [ref() for ref in self.passes.valuerefs()] if w is not None and w.at[0] == task]

    @property
    def items(self) -> list:
        return [item for w in self._here() for item in w.items]

    @property
    def tiles(self) -> int:
        return sum(w.tiles for w in self._here())

    @property
    def armed(self) -> bool:
        return any(w.armed for w in self._here())

    @armed.setter
    def armed(self, value: bool) -> None:
        for w in self._here():
            w.armed = value

    def wants(self, dy, w, alpha) -> bool:
        if alpha is not None or not _GROUP_WGRADS:
            return False
        N, K = w.shape
        return dy.numel() // N >= _GROUP_MIN_ROWS and N < 8192 and N * K >= 512 * 512 and K % 8 == 0

    def add(self, dy, x, w, b) -> None:
        self.add_tensors(dy, x, w.grad, None if b is None else b.grad, [p for p in (w, b) if p is not None])

    def add_tensors(self, dy, x, dw, db, members) -> None:
        """dw / db: the fp32 gradient tensors the launch accumulates into (views of the arena); members: the
        parameters to report ready once it has been enqueued (a packed projection has several).  A gradient of another type or
        on another stream than those that are waiting, or of a backward function called by hand, goes out by itself."""
        key = dy is not None and (dy.dtype, ops._raw_stream())
        w = self._now(dw.device)
        if not w.armed or (w.items and key != w.key):
            ops.linear_wgrad(dy, x, dw, db, accumulate=True)
            _notify(*members)
            return
        tiles = -(-dw.shape[0] // 256) * -(-dw.shape[1] // 256)
        exchanged = any(getattr(p, "_vy_exchanged", False) for p in members)
        if w.tiles + tiles > self.TILES and not exchanged:
            self._flush(w)
        self._hold(w, (dy, x, dw, db, members), tiles, key, exchanged)

    def _hold(self, w, item, tiles, key, exchanged) -> None:
        members = item[4]
        if not w.items:
            w.key, w.stream = key, torch.cuda.current_stream() if item[0] is not None and item[0].is_cuda else None
        w.items.append(item)
        # autograd's own post-accumulate hook fires for these parameters as soon as this backward function
        # returns -- the reducer must not take that for "gradient written" (training.BucketReducer._hook)
        for p in members:
            p._vy_deferred = w.number
        w.tiles += tiles
        if exchanged:
            full = w.tiles >= min(self.TILES, self.EXCHANGED) or len(w.items) >= self.EXCHANGED_MOST
        else:
            full = w.tiles >= self.TILES or len(w.items) >= self.MOST
        if full:
            self._flush(w)

    def flush(self) -> None:
        for w in self._here():
            self._flush(w)

    def _flush(self, w) -> None:
        items, w.items, w.tiles = w.items, [], 0
        if not items:
            return
        try:
            self._launch([item[:4] for item in items])
        finally:
            w.unmark(items)
        sums = _norm_sums.outside if w.at is None else _norm_sums.passes.get(w.at)
        if sums is not None and sums.items and sums.key[1] == ops._raw_stream():   # (so that whole buckets of parameters are ready)
            _norm_sums._flush(sums)
        for *_, members in items:
            _notify(*members)

    def _launch(self, items) -> None:
        ops.linear_wgrad_grouped(items)

    def _end_of_backward(self, w=None) -> None:
        """On the stream that the backward pass was called on.  What waits may be of another one, the forward pass's, or of another device: it goes
        out there, where its operands were made, and the caller's stream waits for it."""
        w = self.outside if w is None else w
        w.armed = False
        if not w.items or w.stream is None or (w.key[1] == ops._raw_stream() and (w.at is None or w.at[1].index == torch.cuda.current_device())):
            self._flush(w)
            return
        here, there = torch.cuda.current_stream(), w.stream
        with torch.cuda.stream(there):
            self._flush(w)
        here.wait_stream(there)


class _WgradRows(_WgradGroup):
    """The same for gradients over fewer rows than those: four layers' in a launch that sums each up in the slices of rows of a launch of its own
    (ops.wgrad_rows), in one of the orders in which their sums may arrive there: the same bits up to 256 rows, and up to 512 into a gradient
    of zeros; beyond, and where one is left alone in a launch, they differ as two runs of one by one do.  Exchanged gradients go out one by one."""

    MOST, FULL = 20, 16     # gradients of a launch; four layers' (with the language model head's dense layer before them: 17) fill it

    def gathers(self, dy, shape, members, alpha=None) -> bool:
        if alpha is not None or dy.dtype != torch.bfloat16 or any(getattr(p, "_vy_exchanged", False) for p in members):
            return False
        return _few_rows(dy.numel() // shape[0], *shape)

    def add_tensors(self, dy, x, dw, db, members) -> None:
        desc, operands = ops.wgrad_desc(dy, x, dw, db)
        self.add_descs([(desc, members)], (dy, dw, db, *operands))

    def add_descs(self, products, keep) -> None:
        """products: (vy_wgrad_desc, members) each; keep: every tensor they point into, the first one a bf16 operand."""
        key = (keep[0].dtype, ops._raw_stream())
        w = self._now(keep[0].device)
        if not w.armed or (w.items and key != w.key):
            ops.wgrad_rows([desc for desc, _ in products])
            for _, members in products:
                _notify(*members)
            return
        if len(w.items) + len(products) > self.MOST:
            self._flush(w)
        for desc, members in products:
            self._hold(w, (keep[0], desc, keep, None, members), 0, key, False)
        if len(w.items) >= self.FULL:
            self._flush(w)

    def _launch(self, items) -> None:
        ops.wgrad_rows([item[1] for item in items])


def _aligned(dy, x) -> bool:
    """Does a launch take these operands, as rows on 16 bytes (or as copies)?  One that does not would take others with it: it is launched, and
    refused, where its layer is reached."""
    return all(t.dtype != BF16 or t.stride(-1) != 1 or (t.data_ptr() % 16 == 0 and t.stride(-2) % 8 == 0 and t.stride(-2) >= t.shape[-1]) for t in (dy, x))


def _few_rows(M, N, K) -> bool:
    """Does a weight gradient N x K over M rows wait for those of other layers with few rows?"""
    return _GROUP_WGRADS and M < _GROUP_MIN_ROWS and N < 8192 and N * K >= 512 * 512 and K % 8 == 0


class _NormSums(_WgradGroup):
    """Column sums of the gradients of norms, whose partials lie in buffers of their own: they go out with the weight gradients of their
    layers, up to sixteen in a launch (ops.layernorm_sums); exchanged ones, and those on another stream than others that wait, at once."""

    MOST = 16

    def add_norms(self, items) -> None:
        """items: (ws, rows, gradients of weight and bias, (weight, bias)) each."""
        key = (torch.float32, ops._raw_stream())
        w = self._now(items[0][2].device)
        if not w.armed or (w.items and key != w.key) or any(getattr(p, "_vy_exchanged", False) for item in items for p in item[4]):
            self._launch([item[:4] for item in items])
            for item in items:
                _notify(*item[4])
            return
        for item in items:
            self._hold(w, item, 0, key, False)

    def _launch(self, items) -> None:
        ops.layernorm_sums(items)


_GROUP_WGRADS = os.environ.get("VY_WGRAD_GROUP", "1") != "0"
_DEFER_RESIDUALS = os.environ.get("VY_DEFER_RESIDUALS", "1") != "0"
_GROUP_MIN_ROWS = int(os.environ.get("VY_WGRAD_GROUP_ROWS", "2048"))   # 2112 rows of width 768, a layer's four gradients: 121 us one by one,
# 58 of a launch with its neighbours'.  Below, tiles of 128 x 128 that sum the rows up as launches one by one do are faster (2047 rows 50,
# 1665 rows 45 / 52 / 113 one by one) and keep the slices: other sums change gradients by 2e-7, and a step's weights in enough places that the
# next one's gradients, whose noise is the rounding of bf16, differ by 1 % from what they were (single values by more than the tensor's mean).
_GROUP_QKV = os.environ.get("VY_WGRAD_GROUP_QKV", "1") != "0"              # the packed QKV gradient joins the group
_wgrad_group = _WgradGroup()
_wgrad_rows = _WgradRows()
_norm_sums = _NormSums()


def _wgrad(dy, x, w: torch.Tensor, b: Optional[torch.Tensor], alpha: Optional[torch.Tensor] = None):
    """-> (dw, db) to return to autograd (None when accumulated in place)."""
    if _direct(w) and (b is None or _direct(b)):
        group = None
        if _wgrad_group.wants(dy, w, alpha):
            group = _wgrad_group
        elif _wgrad_rows.gathers(dy, w.shape, [p for p in (w, b) if p is not None], alpha):
            group = _wgrad_rows
        if group is not None and _aligned(dy, x):
            group.add(dy, x, w, b)
            return None, None
        ops.linear_wgrad(dy, x, w.grad, None if b is None else b.grad, accumulate=True, alpha=alpha)
        _notify(w, b)
        return None, None
    dw = torch.empty(w.shape, dtype=torch.float32, device=w.device)
    db = torch.empty(b.shape, dtype=torch.float32, device=w.device) if b is not None else None
    ops.linear_wgrad(dy, x, dw, db, accumulate=False, alpha=alpha)
    return dw.to(w.dtype), (db.to(b.dtype) if b is not None else None)


def _ln_bwd(dy, x, ln_w, ln_b, mean, rstd):
    dt = x.dtype
    if _direct(ln_w) and _direct(ln_b):
        dx = ops.layernorm_bwd(dy, x, _shadow(ln_w, dt), mean, rstd, ln_w.grad, ln_b.grad, accumulate=True)
        _notify(ln_w, ln_b)
        return dx, None, None
    dg = torch.empty(ln_w.shape, dtype=torch.float32, device=x.device)
    db = torch.empty(ln_b.shape, dtype=torch.float32, device=x.device)
    dx = ops.layernorm_bwd(dy, x, _shadow(ln_w, dt), mean, rstd, dg, db, accumulate=False)
    return dx, dg.to(ln_w.dtype), db.to(ln_b.dtype)


def _defer_list(t: torch.Tensor):
    """The list a layer attached to its input tensor (`_vy_defer`): backward functions that produce a
    residual-path gradient for that tensor append it there instead of returning it, and the
    self-attention backward -- which autograd necessarily runs after them -- adds them in its dgrad
    epilogue.  None when the layer did not opt in."""
    return getattr(t, "_vy_defer", None) if t is not None else None


def defer_residual_grads(x: torch.Tensor) -> None:
    """Called by a post-LN transformer layer on its input (training only): see _defer_list."""
    if torch.is_grad_enabled() and x.requires_grad and _DEFER_RESIDUALS:
        x._vy_defer = []


def _require_bf16(x: torch.Tensor) -> None:
    """The training kernels run in bf16 (the measured path: MFMA GEMMs, flash attention) and in fp32 (the parity
    path: plain-FMA kernels, gradients checked against the reference's autograd at 1e-4)."""
    if x.dtype != BF16 and x.dtype != torch.float32:
        raise VyomHipError("training kernels take bf16 or fp32 activations (fp32 master weights), not %s" % x.dtype)


class EmbeddingFn(torch.autograd.Function):
    """hidden = table[ids] read from the compute-dtype shadow of the fp32 table; the gradient rows are
    accumulated straight into the flat fp32 gradient arena (nn.Embedding: models/decoder.py:287)."""

    @staticmethod
    def forward(ctx, ids, weight, padding_idx, dtype):
        ctx.save_for_backward(ids)
        ctx.weight, ctx.padding_idx = weight, padding_idx
        return ops.embedding(_shadow(weight, dtype), ids)

    @staticmethod
    def backward(ctx, dout):
        (ids,) = ctx.saved_tensors
        w = ctx.weight
        if _direct(w):
            ops.embedding_bwd_(dout.contiguous(), ids, w.grad, ctx.padding_idx)
            _notify(w)
            return None, None, None, None
        dw = torch.zeros(w.shape, dtype=torch.float32, device=w.device)
        ops.embedding_bwd_(dout.contiguous(), ids, dw, ctx.padding_idx)
        return None, dw.to(w.dtype), None, None


class PatchifyFn(torch.autograd.Function):
    """tokens = patches W^T + b with W the stride == kernel Conv2d weight (d, C, p, p) viewed (d, C*p*p): the
    ViT patch embedding (reference models/vision_encoder.py:83-88, 114).  Backward is the weight / bias
    gradient only -- the pixels are data."""

    @staticmethod
    def forward(ctx, patches, w, b):
        _require_bf16(patches)
        dt = patches.dtype
        ctx.save_for_backward(patches)
        ctx.params = (w, b)
        return ops.linear(patches, _shadow(w, dt).reshape(w.shape[0], -1), _shadow(b, dt))

    @staticmethod
    def backward(ctx, dy):
        (patches,) = ctx.saved_tensors
        w, b = ctx.params
        dy = dy.contiguous()
        N = w.shape[0]
        if _direct(w) and (b is None or _direct(b)):
            ops.linear_wgrad(dy, patches, w.grad.view(N, -1), None if b is None else b.grad, accumulate=True)
            _notify(w, b)
            return None, None, None
        dw = torch.empty((N, w.numel() // N), dtype=torch.float32, device=w.device)
        db = torch.empty(b.shape, dtype=torch.float32, device=w.device) if b is not None else None
        ops.linear_wgrad(dy, patches, dw, db, accumulate=False)
        return None, dw.view(w.shape).to(w.dtype), (db.to(b.dtype) if b is not None else None)


class LinearResidualLayerNormFn(torch.autograd.Function):
    """y = LN(x W^T + b + residual).  AttentionSelfOutput (reference layers/attention.py:69-72)."""

    @staticmethod
    def forward(ctx, x, residual, w, b, ln_w, ln_b, eps, drop=None):
        _require_bf16(x)
        dt = x.dtype
        s = ops.linear(x, _shadow(w, dt), _shadow(b, dt), residual=residual, dropout=drop)
        y, mean, rstd = ops.layernorm(s, _shadow(ln_w, dt), _shadow(ln_b, dt), eps, save_stats=True)
        ctx.save_for_backward(x, s, mean, rstd)
        ctx.params = (w, b, ln_w, ln_b)
        ctx.defer = _defer_list(residual)
        ctx.drop = drop
        return y

    @staticmethod
    def backward(ctx, dy):
        x, s, mean, rstd = ctx.saved_tensors
        w, b, ln_w, ln_b = ctx.params
        dy = dy.contiguous()
        ds, dg, dbt = _ln_bwd(dy, s, ln_w, ln_b, mean, rstd)
        # dropout sits between the projection and the residual add: the projection's gradient is ds under
        # the forward's mask (regenerated from (seed, offset)), the residual's is ds itself
        dz = ops.dropout(ds, *ctx.drop) if ctx.drop is not None else ds
        dx = ops.linear_dgrad(dz, _wt(w, x.dtype))
        dw, db = _wgrad(dz, x, w, b)
        if ctx.defer is not None:      # the residual gradient rides to the QKV dgrad epilogue
            ctx.defer.append(ds)
            ds = None
        return dx, ds, dw, db, dg, dbt, None, None


class FfnBlockFn(torch.autograd.Function):
    """y = LN(act(x W1^T + b1) W2^T + b2 + residual).  FeedForward (reference layers/ffn.py:32-40)."""

    @staticmethod
    def forward(ctx, x, residual, w1, b1, w2, b2, ln_w, ln_b, eps, act, drop=None):
        _require_bf16(x)
        dt = x.dtype
        pre = torch.empty((*x.shape[:-1], w1.shape[0]), dtype=dt, device=x.device)
        hmid = torch.empty_like(pre)
        # `pre` holds act'(x W1^T + b1), not the pre-activation: the backward multiplies by it directly
        ops.linear(x, _shadow(w1, dt), _shadow(b1, dt), act=act | _lib.ACT_SAVE_DERIV, pre_out=pre, out=hmid)
        s = ops.linear(hmid, _shadow(w2, dt), _shadow(b2, dt), residual=residual, dropout=drop)
        ctx.drop = drop
        y, mean, rstd = ops.layernorm(s, _shadow(ln_w, dt), _shadow(ln_b, dt), eps, save_stats=True)
        ctx.save_for_backward(x, pre, hmid, s, mean, rstd)
        ctx.params = (w1, b1, w2, b2, ln_w, ln_b)
        ctx.act = act
        ctx.defer = _defer_list(residual) if residual is not x else None
        return y

    @staticmethod
    def backward(ctx, dy):
        x, pre, hmid, s, mean, rstd = ctx.saved_tensors
        w1, b1, w2, b2, ln_w, ln_b = ctx.params
        dt = x.dtype
        dy = dy.contiguous()
        ds, dg, dbt = _ln_bwd(dy, s, ln_w, ln_b, mean, rstd)
        dz = ops.dropout(ds, *ctx.drop) if ctx.drop is not None else ds   # the forward's mask (see above)
        dpre = ops.linear_dgrad(dz, _wt(w2, dt), pre=pre, act=ctx.act | _lib.ACT_SAVE_DERIV)  # (dz W2) * act'(pre), act' saved
        dw2, db2 = _wgrad(dz, hmid, w2, b2)
        dx = ops.linear_dgrad(dpre, _wt(w1, dt))
        dw1, db1 = _wgrad(dpre, x, w1, b1)
        if ctx.defer is not None:
            ctx.defer.append(ds)
            ds = None
        return dx, ds, dw1, db1, dw2, db2, dg, dbt, None, None, None


class SelfAttentionFn(torch.autograd.Function):
    """o = merge_heads(softmax(rope(q) rope(k)^T / sqrt(dh) + mask) v) with q,k,v = x W^T + b.
    Inputs after `mod` are the projection parameters in module order (q,k,v weights then biases,
    or the fused qkv weight and bias)."""

    @staticmethod
    def forward(ctx, x, mod, attention_mask, freqs, start_pos, *params):
        _require_bf16(x)
        B, L, _ = x.shape
        h, hk, dh = mod.num_attention_heads, mod.num_key_value_heads, mod.head_dim
        dt, dev = x.dtype, x.device
        w, b = mod._packed()
        if attention_mask is not None and not isinstance(attention_mask, AttnMask):
            raise VyomHipError("training needs a mask descriptor (AttnMask): dense additive masks have no "
                               "backward kernel")
        cos, sin, pos0 = resolve_freqs(freqs, dev)
        q = torch.empty((B, h, L, dh), dtype=dt, device=dev)
        k = torch.empty((B, hk, L, dh), dtype=dt, device=dev)
        v = torch.empty_like(k)
        sw, sb = mod._packed_shadow(dt)
        ops.qkv_rope(x, sw, sb, h, hk, dh, cos, sin, pos0, q, k, v)
        lse = torch.empty((B, h, L), dtype=torch.float32, device=dev)
        causal, kp, sp = False, None, 0
        if attention_mask is not None:
            causal, kp, sp = attention_mask.causal, attention_mask.keypad, attention_mask.start_pos
            if kp is not None:
                kp = kp[:, :L].contiguous() if kp.shape[1] != L else kp
        o = ops.attention(q, k, v, causal=causal, start_pos=sp, keypad=kp, lse=lse)
        ctx.save_for_backward(x, q, k, v, o, lse)
        ctx.meta = (mod, causal, kp, sp, cos, sin, pos0, params)
        ctx.defer = _defer_list(x)
        return o

    @staticmethod
    def backward(ctx, do):
        x, q, k, v, o, lse = ctx.saved_tensors
        mod, causal, kp, sp, cos, sin, pos0, params = ctx.meta
        B, L, _ = x.shape
        h, hk, dh = mod.num_attention_heads, mod.num_key_value_heads, mod.head_dim
        dt = x.dtype
        do = do.contiguous()
        W = (h + 2 * hk) * dh
        packed = torch.empty((B, L, W), dtype=dt, device=x.device)  # [dq | dk | dv], 'b l (h d)'
        dq = packed[:, :, : h * dh].view(B, L, h, dh).permute(0, 2, 1, 3)
        dk = packed[:, :, h * dh:(h + hk) * dh].view(B, L, hk, dh).permute(0, 2, 1, 3)
        dv = packed[:, :, (h + hk) * dh:].view(B, L, hk, dh).permute(0, 2, 1, 3)
        # RoPE is orthogonal: its backward (the inverse rotation of dq, dk) runs in the epilogues
        ops.attention_bwd(q, k, v, o, do, lse, dq, dk, dv, causal=causal, start_pos=sp, keypad=kp,
                          cos=cos, sin=sin, rope_pos0=pos0)
        w, b = mod._packed()
        # the layer input's other gradient contributions (residual paths of this layer's out-projection
        # and feed-forward, deferred by their backward) are added in this GEMM's epilogue
        adds = ctx.defer if ctx.defer is not None else []
        extra = None
        for t in adds[2:]:
            extra = t if extra is None else extra + t
        a1 = adds[0] if len(adds) > 0 else None
        a2 = adds[1] if len(adds) > 1 else None
        if extra is not None:
            a2 = a2 + extra
        dx = ops.linear_dgrad(packed, _wt_packed(mod, dt), add_to=a1, add_to2=a2)
        if ctx.defer is not None:
            ctx.defer.clear()
        grads = _packed_wgrad(mod, packed, x, w, b, params)
        return (dx, None, None, None, None, *grads)


def _segments(*sizes):
    """Where segments of so many elements begin in one buffer, each on a line of 128 bytes, and how long it is."""
    at, out = 0, []
    for n in sizes:
        out.append(at)
        at += (n + 63) // 64 * 64
    return out, at


@functools.lru_cache(maxsize=256)
def _kept_segments(B, L, d, hk_dh, inner, h):
    """Offsets of what the weight gradients of a layer multiply with, [o | a | inner], of the rest, [q | s1 | deriv | s2 | k | v], and of the
    statistics: waiting weight gradients hold their operands' buffer, so the rest has one of its own."""
    M = B * L
    return _segments(M * d, M * d, M * inner), _segments(M * d, M * d, M * inner, M * d, M * hk_dh, M * hk_dh), _segments(B * h * L, M, M, M, M)


@functools.lru_cache(maxsize=256)
def _work_segments(B, L, d, W, inner, h, slabs):
    """Of the weight gradients' other operands, [ds2 | dpre | ds1 | dqkv], of [da | dheads], and of the scratch [delta | ln_ws]."""
    M = B * L
    return _segments(M * d, M * inner, M * d, M * W), _segments(M * d, M * d), _segments(B * h * L, 2 * slabs * d)


class TextLayerFn(torch.autograd.Function):
    """A whole post-LN layer (autograd.layer_train): the launches of SelfAttentionFn, LinearResidualLayerNormFn and FfnBlockFn in their order,
    behind one native call each way; the gradients of the layer input's residual paths meet in the QKV dgrad's epilogue.  Every parameter's
    gradient goes into the arena.  keep: [Wqkv, bqkv, Wo, bo, .., both norms, W1, b1, W2, b2] in the compute type.

    Steps of a few hundred tokens are the host's, so it does here what they need and no more: 12 layers, 186 tokens, 4.9 -> 4.4 ms a step,
    captions of 3 images, 24 layers, 8.8 -> 6.6."""

    @staticmethod
    def _layer(att, ff, x, kp, causal, start, rope, keep, inner, kv):
        """The descriptor; kv: where the keys and the values are."""
        L = x.shape[1]
        hk, dh = att.num_key_value_heads, att.head_dim
        cos, sin, pos0 = rope
        kind = (_lib.MASK_CAUSAL if causal else 0) | (_lib.MASK_KEYPAD if kp is not None else 0)
        st = (hk * L * dh, L * dh, dh)
        return _lib.VyTextLayer(att.num_attention_heads, hk, dh, inner, ff.act, kind, _lib.dtype_code(x.dtype),
                                att._modules["out"]._modules["layernorm"].eps, ff._modules["layernorm"].eps,
                                *[None if t is None else t.data_ptr() for t in keep], None if cos is None else cos.data_ptr(),
                                None if sin is None else sin.data_ptr(), pos0, *kv, *st, *st, *kv, *st, *st, L, start,
                                None if kp is None else kp.data_ptr(), 0 if kp is None else kp.stride(0))

    @staticmethod
    def _places(x, rows, rest, stats, operands, others, numbers):
        """-> vy_text_layer_kept, and where the keys and the values are."""
        e, r0, t0, s0 = x.element_size(), rows.data_ptr(), rest.data_ptr(), stats.data_ptr()
        o, a, inner = [r0 + n * e for n in operands]
        q, s1, deriv, s2, k, v = [t0 + n * e for n in others]
        return _lib.VyTextLayerKept(q, o, s1, a, deriv, inner, s2, *[s0 + 4 * n for n in numbers]), (k, v)

    @staticmethod
    def forward(ctx, x, kp, att, ff, keep, causal, start, rope, *params):
        B, L, d = x.shape
        inner, dt, dev = keep[6].shape[0], x.dtype, x.device
        (operands, n), (others, m), (numbers, sn) = _kept_segments(B, L, d, att.num_key_value_heads * att.head_dim, inner, att.num_attention_heads)
        rows = torch.empty(n, dtype=dt, device=dev)
        rest = torch.empty(m, dtype=dt, device=dev)
        stats = torch.empty(sn, dtype=torch.float32, device=dev)
        y = torch.empty_like(x)
        kept, kv = TextLayerFn._places(x, rows, rest, stats, operands, others, numbers)
        desc = TextLayerFn._layer(att, ff, x, kp, causal, start, rope, keep, inner, kv)
        ops._mid_ws(B * L)
        _lib.call("vy_text_layer_train_fwd", _ref(desc), _ref(kept), x.data_ptr(), y.data_ptr(), B, L, ops._stream())
        ctx.save_for_backward(x, rows, rest, stats, kp)
        ctx.meta = (att, ff, causal, start, rope, params)
        return y

    @staticmethod
    def _waiting(M, d, W, inner, dt, params, nw):
        """The gradients of the parameters, [Wo, bo, first norm, W1, b1, W2, b2, second norm, projections], if every weight gradient of the
        layer waits for those of other layers with few rows (_WgradRows) and the projections' lie one behind the other."""
        if dt is not torch.bfloat16 or not _GROUP_QKV or not (_few_rows(M, d, d) and _few_rows(M, W, d) and _few_rows(M, inner, d) and _few_rows(M, d, inner)):
            return None
        grads = []
        for p in params:
            g = p.grad if getattr(p, "_vy_direct", False) else None
            if g is None or g.dtype is not torch.float32 or not g.is_contiguous() or getattr(p, "_vy_exchanged", False):
                return None
            grads.append(g)
        for group in (grads[10:10 + nw], grads[10 + nw:]):
            at = group[0].data_ptr() if group else 0
            for g in group:
                if g.data_ptr() != at:
                    return None
                at += 4 * g.numel()
        return grads

    @staticmethod
    def backward(ctx, dy):
        x, rows, rest, stats, kp = ctx.saved_tensors
        att, ff, causal, start, rope, params = ctx.meta
        B, L, d = x.shape
        dt, dev, M = x.dtype, x.device, B * L
        dy, rows, rest, stats = dy.contiguous(), rows.contiguous(), rest.contiguous(), stats.contiguous()
        wo, bo, g1, b1, w1, c1, w2, c2, g2, b2 = params[:10]
        members = att._params()
        h, hk_dh, inner = att.num_attention_heads, att.num_key_value_heads * att.head_dim, w1.shape[0]
        W = d + 2 * hk_dh
        (operands, _), (others, _), (numbers, _) = _kept_segments(B, L, d, hk_dh, inner, h)
        kept, kv = TextLayerFn._places(x, rows, rest, stats, operands, others, numbers)
        # (of the weights only the norms' are read here, the others transposed)
        keep = (None, None, None, None, _shadow(g1, dt), None, None, None, None, None, _shadow(g2, dt), None)
        desc = TextLayerFn._layer(att, ff, x, kp, causal, start, rope, keep, inner, kv)
        wt = (_wt_packed(att, dt, members), _wt(wo, dt), _wt(w1, dt), _wt(w2, dt))
        slabs = _lib.load().vy_layernorm_bwd_ws_rows(M)
        (to, n), (oo, on), (fo, fn) = _work_segments(B, L, d, W, inner, h, slabs)
        work = torch.empty(n, dtype=dt, device=dev)
        own = torch.empty(on, dtype=dt, device=dev)
        dx = torch.empty_like(x)
        nw = 1 if att._fused_qkv else 3
        waiting = TextLayerFn._waiting(M, d, W, inner, dt, (*params[:10], *members), nw) if x.is_contiguous() and x.data_ptr() % 16 == 0 else None
        wait = waiting is not None or (_GROUP_WGRADS and all(_direct(p) for p in (g1, b1, g2, b2)))    # the norms' column sums go out with other layers'
        scratch = torch.empty(fo[1] if wait else fn, dtype=torch.float32, device=dev)
        sums = torch.empty((2, 2 * slabs * d), dtype=torch.float32, device=dev) if wait else None
        e, f0, w0, o0 = x.element_size(), scratch.data_ptr(), work.data_ptr(), own.data_ptr()
        ds2, dpre, ds1, dqkv = [w0 + o * e for o in to]
        # (a gradient that has left the arena since the forward pass is returned)
        dln = [] if wait else [p.grad if _direct(p) else torch.zeros(d, dtype=torch.float32, device=dev) for p in (g1, b1, g2, b2)]
        at = sums.data_ptr() if wait else f0 + 4 * fo[1]
        grads = _lib.VyTextLayerGrads(*[t.data_ptr() for t in wt], *[t.stride(0) for t in wt], *((None,) * 4 if wait else [t.data_ptr() for t in dln]),
                                      ds2, dpre, o0 + oo[0] * e, ds1, o0 + oo[1] * e, dqkv, at, f0, at + 8 * slabs * d if wait else None)
        ops._mid_ws(M)
        _lib.call("vy_text_layer_bwd", _ref(desc), _ref(kept), _ref(grads), dy.data_ptr(), dx.data_ptr(), B, L, ops._stream())
        if waiting is not None:
            _norm_sums.add_norms([(sums[0], slabs, waiting[8], waiting[9], (g2, b2)), (sums[1], slabs, waiting[2], waiting[3], (g1, b1))])
            gwo, gbo, _, _, gw1, gc1, gw2, gc2, _, _, gq = [g.data_ptr() for g in waiting[:11]]
            gbq = waiting[10 + nw].data_ptr() if len(members) > nw else None
            D, kept_o, kept_a, kept_inner = _lib.VyWgradDesc, kept.o, kept.a, kept.inner
            _wgrad_rows.add_descs([(D(ds2, d, kept_inner, inner, gw2, inner, gc2, M, d, inner), (w2, c2)),
                                   (D(dpre, inner, kept_a, d, gw1, d, gc1, M, inner, d), (w1, c1)),
                                   (D(ds1, d, kept_o, d, gwo, d, gbo, M, d, d), (wo, bo)),
                                   (D(dqkv, W, x.data_ptr(), d, gq, d, gbq, M, W, d), members)], (work, rows, x, *waiting))
            return (dx, *[None] * (7 + len(params)))
        if wait:
            dg1 = db1 = dg2 = db2 = None
            _norm_sums.add_norms([(sums[0], slabs, g2.grad, b2.grad, (g2, b2)), (sums[1], slabs, g1.grad, b1.grad, (g1, b1))])
        else:
            dg1, db1, dg2, db2 = (None if _direct(p) else t.to(p.dtype) for p, t in zip((g1, b1, g2, b2), dln))
            _notify(*(p for p in (g2, b2, g1, b1) if _direct(p)))

        def of(t, o, cols):
            return t.as_strided((M, cols), (cols, 1), t.storage_offset() + o)
        dw2 = _wgrad(of(work, to[0], d), of(rows, operands[2], inner), w2, c2)
        dw1 = _wgrad(of(work, to[1], inner), of(rows, operands[1], d), w1, c1)
        dwo = _wgrad(of(work, to[2], d), of(rows, operands[0], d), wo, bo)
        dqkv_w = _packed_wgrad(att, of(work, to[3], W), x, *att._packed(members), params[10:], members)
        return (dx, *[None] * 7, *dwo, dg1, db1, *dw1, *dw2, dg2, db2, *dqkv_w)


class CrossAttentionFn(torch.autograd.Function):
    """o = merge_heads(softmax(q k^T / sqrt(dh) + key-padding mask) v), q = x Wq^T + bq,
    k/v = enc Wk/v^T + b: the encoder-decoder attention of the seq2seq decoder layer
    (reference layers/attention.py:410-474, 512-573).  Gradients flow to the decoder state, to the
    ENCODER output and to the three projections."""

    @staticmethod
    def forward(ctx, x, enc, mod, enc_mask, wq, bq, wk, bk, wv, bv):
        _require_bf16(x)
        B, L, _ = x.shape
        S = enc.shape[1]
        h, hk, dh = mod.num_attention_heads, mod.num_key_value_heads, mod.head_dim
        dt, dev = x.dtype, x.device
        if enc_mask is not None and not isinstance(enc_mask, AttnMask):
            raise VyomHipError("training needs a mask descriptor (AttnMask): dense additive masks have no "
                               "backward kernel")
        q2 = ops.linear(x, _shadow(wq, dt), _shadow(bq, dt))
        k2 = ops.linear(enc, _shadow(wk, dt), _shadow(bk, dt))
        v2 = ops.linear(enc, _shadow(wv, dt), _shadow(bv, dt))
        kp = None
        if enc_mask is not None:
            if enc_mask.causal:
                raise VyomHipError("cross-attention takes a key-padding mask, not a causal one")
            kp = enc_mask.keypad
            if kp is not None:
                kp = kp[:, :S].contiguous() if kp.shape[1] != S else kp
        lse = torch.empty((B, h, L), dtype=torch.float32, device=dev)
        o = ops.attention(_heads(q2, h, dh), _heads(k2, hk, dh), _heads(v2, hk, dh), causal=False, keypad=kp, lse=lse)
        ctx.save_for_backward(x, enc, q2, k2, v2, o, lse)
        ctx.meta = (mod, kp, (wq, bq, wk, bk, wv, bv))
        return o

    @staticmethod
    def backward(ctx, do):
        x, enc, q2, k2, v2, o, lse = ctx.saved_tensors
        mod, kp, (wq, bq, wk, bk, wv, bv) = ctx.meta
        h, hk, dh = mod.num_attention_heads, mod.num_key_value_heads, mod.head_dim
        dt = x.dtype
        do = do.contiguous()
        dq2, dk2, dv2 = torch.empty_like(q2), torch.empty_like(k2), torch.empty_like(v2)
        ops.attention_bwd(_heads(q2, h, dh), _heads(k2, hk, dh), _heads(v2, hk, dh), o, do, lse,
                          _heads(dq2, h, dh), _heads(dk2, hk, dh), _heads(dv2, hk, dh), causal=False, keypad=kp)
        dx = ops.linear_dgrad(dq2, _wt(wq, dt))
        denc = ops.linear_dgrad(dk2, _wt(wk, dt))
        denc = ops.linear_dgrad(dv2, _wt(wv, dt), add_to=denc)
        dwq, dbq = _wgrad(dq2, x, wq, bq)
        dwk, dbk = _wgrad(dk2, enc, wk, bk)
        dwv, dbv = _wgrad(dv2, enc, wv, bv)
        return dx, denc, None, None, dwq, dbq, dwk, dbk, dwv, dbv


def _heads(x2: torch.Tensor, heads: int, dh: int) -> torch.Tensor:
    B, L, _ = x2.shape
    return x2.view(B, L, heads, dh).permute(0, 2, 1, 3)


def _wt_packed(mod, dtype, members=None):
    """W^T of the packed projection: keyed on the versions of the member parameters.  (members: what mod._params() has just returned)"""
    def key(members):
        return (*[p._version for p in members], getattr(members[0], "_vy_weights", _WT).epoch, dtype)

    def key_of(m):
        members = m._params()
        return key(members), members
    if members is None:
        members = mod._params()
    return _wt_cached(mod, getattr(members[0], "_vy_weights", _WT), key(members), key_of, lambda m, members: m._packed_shadow(dtype, None, members)[0],
                      members)


def _packed_wgrad(mod, dy, x, w, b, params, members=None):
    if members is None:
        members = mod._params()
    nw = 1 if mod._fused_qkv else 3
    ws, bs = members[:nw], members[nw:]
    if all(_direct(p) for p in members):
        # the trainer lays the member gradients out adjacently, mirroring the packed weights
        g0 = ws[0].grad
        N = sum(p.shape[0] for p in ws)
        dw = torch.as_strided(g0, (N, g0.shape[1]), (g0.stride(0), 1))
        ok = all(p.grad.data_ptr() == g0.data_ptr() + off * g0.shape[1] * 4
                 for p, off in zip(ws, _offsets(ws)))
        db = None
        if bs:
            db0 = bs[0].grad
            db = torch.as_strided(db0, (N,), (1,))
            ok = ok and all(p.grad.data_ptr() == db0.data_ptr() + off * 4 for p, off in zip(bs, _offsets(bs)))
        if ok:
            dy2 = dy.view(-1, dy.shape[-1])
            may = _GROUP_QKV and _aligned(dy2, x)
            if _GROUP_WGRADS and may and dy2.shape[0] >= _GROUP_MIN_ROWS and N * dw.shape[1] >= 512 * 512 and dw.shape[1] % 8 == 0:
                # with the layer's other weight gradients in one grouped launch (27 of its 108 tiles: on its own
                # this launch ran at 670 TFLOP/s, the group at 850)
                _wgrad_group.add_tensors(dy2, x, dw, db, list(members))
            elif may and _wgrad_rows.gathers(dy2, dw.shape, members):
                _wgrad_rows.add_tensors(dy2, x, dw, db, list(members))
            else:
                ops.linear_wgrad(dy, x, dw, db, accumulate=True)
                _notify(*members)
            return [None] * len(params)
    N, K = w.shape
    dw = torch.empty((N, K), dtype=torch.float32, device=w.device)
    db = torch.empty((N,), dtype=torch.float32, device=w.device) if b is not None else None
    ops.linear_wgrad(dy, x, dw, db, accumulate=False)
    out, off = [], 0
    for p in ws:
        out.append(dw[off:off + p.shape[0]].to(p.dtype))
        off += p.shape[0]
    off = 0
    for p in bs:
        out.append(db[off:off + p.shape[0]].to(p.dtype))
        off += p.shape[0]
    return out


def _offsets(ps):
    offs, o = [], 0
    for p in ps:
        offs.append(o)
        o += p.shape[0]
    return offs


class LMHeadFn(torch.autograd.Function):
    """logits = LN(gelu(h Wd^T + bd)) Wv^T + bias (reference models/decoder.py:267-275).  The logits
    row stride is padded to 8 and the pad columns are zero, so the backward GEMMs can contract
    over the padded width."""

    @staticmethod
    def forward(ctx, hidden, wd, bd, ln_w, ln_b, wv, bias, eps):
        _require_bf16(hidden)
        dt = hidden.dtype
        pre = torch.empty_like(hidden)
        g = torch.empty_like(hidden)
        ops.linear(hidden, _shadow(wd, dt), _shadow(bd, dt), act=ACT_GELU_ERF, pre_out=pre, out=g)
        n, mean, rstd = ops.layernorm(g, _shadow(ln_w, dt), _shadow(ln_b, dt), eps, save_stats=True)
        V = wv.shape[0]
        ld = _row_stride(V)
        buf = torch.zeros((*hidden.shape[:-1], ld), dtype=dt, device=hidden.device)
        logits = buf[..., :V]
        ops.linear(n, _shadow(wv, dt), _shadow(bias, dt), out=logits)
        ctx.save_for_backward(hidden, pre, g, n, mean, rstd)
        ctx.params = (wd, bd, ln_w, ln_b, wv, bias)
        ctx.ld = ld
        return logits

    @staticmethod
    def backward(ctx, dlogits):
        hidden, pre, g, n, mean, rstd = ctx.saved_tensors
        wd, bd, ln_w, ln_b, wv, bias = ctx.params
        dt = hidden.dtype
        V, ld = wv.shape[0], ctx.ld
        # the contraction of the dgrad GEMM runs over the PADDED vocabulary width (multiple of 8, pad
        # columns of both operands zero): re-home the gradient unless it already sits in such a buffer
        if dlogits.stride(-1) != 1 or dlogits.stride(-2) != ld or dlogits.dtype != dt:
            buf = torch.zeros((*dlogits.shape[:-1], ld), dtype=dt, device=dlogits.device)
            buf[..., :V] = dlogits
        else:
            buf = torch.as_strided(dlogits, (*dlogits.shape[:-1], ld), dlogits.stride())
            if ld != V:
                buf[..., V:].zero_()
        dlogits = buf[..., :V]
        dn = ops.linear_dgrad(buf, _wt_padded(wv, dt, ld))
        dwv, dbias = _wgrad(dlogits, n, wv, bias)
        dg, dgam, dbet = _ln_bwd(dn, g, ln_w, ln_b, mean, rstd)
        dpre = _gelu_bwd(dg, pre)
        dh = ops.linear_dgrad(dpre, _wt(wd, dt))
        dwd, dbd = _wgrad(dpre, hidden, wd, bd)
        return dh, dwd, dbd, dgam, dbet, dwv, dbias, None


def _gelu_bwd(dy, pre):
    return ops.act_bwd(dy, pre, ACT_GELU_ERF)


class LMHeadLossFn(torch.autograd.Function):
    """Shifted causal-LM loss fused with the LM head: mean cross-entropy of logits[:, :-1] against
    labels[:, 1:] with ignore_index (Examples/vyom-ai-decoder_clm.ipynb cell 29).  The logits
    ([M, V] bf16, padded row stride) are produced by the vocabulary GEMM, then reduced AND
    overwritten IN PLACE by their unit gradient in one pass (vy_xent_fused; vy_xent_fwd + vy_xent_bwd
    beyond 65536 columns) -- they are never copied, up-cast or re-materialised.  Backward multiplies by the upstream gradient through the GEMMs (a device scalar)."""

    @staticmethod
    def forward(ctx, hidden, labels, ignore_index, wd, bd, ln_w, ln_b, wv, bias, eps, err_flag=None):
        _require_bf16(hidden)
        dt, dev = hidden.dtype, hidden.device
        B, L, _ = hidden.shape
        pre = torch.empty_like(hidden)
        g = torch.empty_like(hidden)
        ops.linear(hidden, _shadow(wd, dt), _shadow(bd, dt), act=ACT_GELU_ERF, pre_out=pre, out=g)
        n, mean, rstd = ops.layernorm(g, _shadow(ln_w, dt), _shadow(ln_b, dt), eps, save_stats=True)
        V = wv.shape[0]
        ld = _row_stride(V)
        buf = torch.empty((B * L, ld), dtype=dt, device=dev)
        logits = buf[:, :V]
        fused = V <= 65536 and dt == BF16   # (vy_xent_fused is a bf16 kernel; fp32 takes the two-pass pair)
        together = fused and labels.dtype == torch.long and labels.device == dev and labels.shape == (B, L)
        if not together and ld != V:
            buf[:, V:].zero_()  # only the pad columns: the GEMM writes the rest
        ops.linear(n.view(B * L, -1), _shadow(wv, dt), _shadow(bias, dt), out=logits)
        # acc: [loss_sum, count]
        if together:
            shifted, acc = ops.shift_labels(labels, ignore_index, logits, ld)
        else:
            shifted = torch.full((B, L), ignore_index, dtype=torch.long, device=dev)
            shifted[:, :-1] = labels[:, 1:]
            shifted = shifted.view(-1)
            acc = torch.zeros(2, dtype=torch.float32, device=dev)
        lse = torch.empty(B * L, dtype=torch.float32, device=dev)
        if fused:
            # one pass: loss AND the unit gradient (d loss / d logits for an upstream gradient of 1),
            # written over the logits; backward scales by the actual upstream gradient (linearity)
            # (rows with an out-of-range label contribute neither loss nor gradient -- the kernel raises err_flag for
            # them -- so they must not count in the mean either, exactly as on the two-pass path)
            if not together:
                acc[1] = ((shifted != ignore_index) & (shifted >= 0) & (shifted < V)).sum()
            ops.xent_fused_(logits, shifted, ignore_index, lse, acc[0:1], acc[1:2], _one(dev), err_flag)
        else:
            ops.xent_fwd(logits, shifted, ignore_index, lse, acc[0:1], acc[1:2], err_flag)
        ctx.save_for_backward(hidden, pre, g, n, mean, rstd, buf, shifted, lse, acc)
        ctx.params = (wd, bd, ln_w, ln_b, wv, bias)
        ctx.ignore = ignore_index
        ctx.fused = fused
        return acc[0] / acc[1].clamp_min(1.0)

    @staticmethod
    def backward(ctx, gout):
        hidden, pre, g, n, mean, rstd, buf, shifted, lse, acc = ctx.saved_tensors
        wd, bd, ln_w, ln_b, wv, bias = ctx.params
        dt = hidden.dtype
        V = wv.shape[0]
        logits = buf[:, :V]
        gs = gout.detach().to(torch.float32).reshape(1).contiguous()
        alpha = None
        if ctx.fused:
            alpha = gs          # logits already hold the unit gradient
        else:
            ops.xent_bwd_(logits, shifted, ctx.ignore, lse, gs, acc[1:2])   # logits <- dlogits
        # contract over the padded vocabulary width (pad columns of both operands are zero)
        dn = ops.linear_dgrad(buf, _wt_padded(wv, dt, buf.shape[1]))
        if alpha is not None:
            dn = dn * alpha.to(dt)
        dwv, dbias = _wgrad(logits, n.view(buf.shape[0], -1), wv, bias, alpha=alpha)
        dg, dgam, dbet = _ln_bwd(dn.view(g.shape), g, ln_w, ln_b, mean, rstd)
        dpre = _gelu_bwd(dg, pre)
        dh = ops.linear_dgrad(dpre, _wt(wd, dt))
        dwd, dbd = _wgrad(dpre, hidden, wd, bd)
        return dh, None, None, dwd, dbd, dgam, dbet, dwv, dbias, None, None


_ONES = {}


def _one(dev) -> torch.Tensor:
    t = _ONES.get(dev)
    if t is None:
        t = _ONES[dev] = torch.ones(1, dtype=torch.float32, device=dev)
    return t


def _wt_padded(param, dtype, ld):
    """[K, ld] zero-padded W^T (full padded width, for contractions over the padded vocabulary)."""
    wt = _wt(param, dtype)
    full = torch.as_strided(wt, (wt.shape[0], ld), (wt.stride(0), 1))
    assert wt.stride(0) == ld
    return full
