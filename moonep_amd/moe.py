"""Autograd glue and the expert-side consumer contract around ``Buffer``.

How a training framework wires MoonEP into an MoE layer (reference
README.md:43-156): dispatch forward pairs with combine as its backward, combine
forward pairs with a plan-reusing dispatch as its backward, ``prefetch_weight``
pairs with ``reduce_grad``, and the expert FFN consumes the dispatched rows as
``2*epn`` groups (``epn`` local experts, then ``epn`` prefetch slots) delimited
by ``cu_seqlens``.

One GPU stands in for all R ranks here, so the functions below act on the
whole emulated group at once (``[R, ...]`` tensors, one ``Buffer`` per rank on a
shared ``EmulatedWorld``): every rank dispatches before any rank's experts
run, every rank's experts finish before any rank combines -- the ordering the
reference gets from its cross-rank barriers.

``group_expert_ffn_hip`` is the expert stage of the layer on the matrix cores,
forward and backward: the compute views of every rank (its local experts, then
its prefetch slots pulled from their owners), the grouped SwiGLU FFN of every rank's
groups, and in backward the grouped input / weight gradient GEMMs followed by
``reduce_grad`` in fp32 -- no PyTorch GEMM on either pass.
"""

from __future__ import annotations

import ctypes as C

import torch

from . import _lib, ffn
from .api import Buffer, EmulatedWorld
from .grad_reduce import launch_grad_reduce
from .planning import MoonEPCommPlan, launch_planning_all_ranks
from .prefetch import launch_prefetch_pull


class EmulatedGroup:
    """R Buffers (one per rank) on one shared set of shards."""

    def __init__(self, S, H, K, E, R, token_padding=128):
        self.S, self.H, self.K, self.E, self.R = S, H, K, E, R
        self.epn = E // R
        self.world = EmulatedWorld(S, H, K, E, R, token_padding)
        self.buffers = [Buffer(S, H, K, E, R, token_padding=token_padding, rank=r,
                               world=self.world) for r in range(R)]
        self.NvS = self.world.NvS
        lay = self.world.layout
        self._mcp = lay["meta_chunk_padded"]
        # what the last whole-group operator dispatched or combined, until somebody asks for it in
        # the world's shards: rows [R,NvS,H]; slots [R,NvS], or 0.0 after a dispatch without weights
        self._rows = self._slots = None

    def _note(self, rows, slots=None):
        self._rows = rows.detach()     # its own tensor: a reference to the caller's would keep the graph alive
        if slots is not None:
            self._slots = slots.detach() if isinstance(slots, torch.Tensor) else slots

    def shards(self) -> torch.Tensor:
        """Every rank's shard ``[R, NvS, H]`` as the last whole-group operator saw it: the rows that
        ``group_dispatch`` wrote, or those that ``group_combine`` (or the backward pass of either)
        read or wrote.  It is the memory that the group's Buffers work on; the operators work on
        tensors of their own, and the rows are copied here by this call."""
        view = self.world.hidden_buf.view(self.R, self.NvS, self.H)
        if self._rows is not None:
            self._rows.record_stream(torch.cuda.current_stream())   # may be another than the operator's
            view.copy_(self._rows)
            self._rows = None
        return view

    def weight_slots(self) -> torch.Tensor:
        """Every rank's route-weight slots ``[R, NvS]``, likewise; zeros after a dispatch without weights."""
        view = self.world.meta_buf.view(self.R, self._mcp)[:, :self.NvS].view(torch.float32)
        if self._slots is not None:
            if isinstance(self._slots, torch.Tensor):
                self._slots.record_stream(torch.cuda.current_stream())
                view.copy_(self._slots)
            else:
                view.zero_()
            self._slots = None
        return view

    def destroy(self):
        self._rows = self._slots = None
        for b in self.buffers:
            b.destroy()


# Every operator below is one launch for the whole group (csrc: the *_ranks entry points).  The rows
# go straight into the tensor that the experts (or autograd) own and come straight out of it: on one
# GPU that tensor can be the destination of a dispatch and the source of a combine itself, so
# neither the shards of the world nor a copy into or out of them is needed.

def _group_ctx(group):
    return group.buffers[0]._require_ctx()


def _dispatch_all(group, x_all, w_all, dst_all, zero_fill, cu):
    """Rows ``[R,NvS,H]`` (+ slots ``[R,NvS]``) of every rank; every row is written."""
    ctx, R = _group_ctx(group), group.R
    group._rows = None     # its memory is free for the new rows
    # without the groups' ends (plans of another origin) the rows behind them are cleared first
    make = torch.empty if cu is not None else torch.zeros
    rows = make(R, group.NvS, group.H, dtype=torch.bfloat16, device=x_all.device)
    slots = None if w_all is None else make(R, group.NvS, dtype=torch.float32, device=x_all.device)
    rc = _lib.lib().mep_dispatch_ranks(
        x_all.data_ptr(), _lib.ptr(w_all), dst_all.data_ptr(), zero_fill.data_ptr(), _lib.ptr(cu), rows.data_ptr(),
        group.NvS, _lib.ptr(slots), group.NvS, 0, R, group.S, group.H, group.K, R, group.epn, group.NvS,
        int(ctx["token_padding"]), _lib.DISPATCH_WRITE_DUPS, _lib.current_stream())
    _lib.check(rc, "mep_dispatch_ranks")
    return rows, slots


def _combine_all(group, rows, slots, dst_all):
    """Token-major sums ``[R,S,H]`` (+ slots gathered back to ``[R,S,K]``) of every rank."""
    _group_ctx(group)
    R, S, K = group.R, group.S, group.K
    out = torch.empty(R, S, group.H, dtype=torch.bfloat16, device=rows.device)
    w = None if slots is None else torch.empty(R, S, K, dtype=torch.float32, device=rows.device)
    rc = _lib.lib().mep_combine_ranks(
        rows.data_ptr(), group.NvS, _lib.ptr(slots), group.NvS, dst_all.data_ptr(), out.data_ptr(), _lib.ptr(w), R,
        S, group.H, K, R, group.NvS, _lib.COMBINE_TWO_LEVEL, _lib.current_stream())
    _lib.check(rc, "mep_combine_ranks")
    return out, w


def _group_plans(group, topk_all, tpe):
    """Plans of every rank from one planner launch and one duplicate-group build: tensors with a
    leading rank dimension and the per-rank plans as views of them."""
    ctx, R, NvS, epn = _group_ctx(group), group.R, group.NvS, group.epn
    dst, cu, etc, zfr, stats = launch_planning_all_ranks(ctx, topk_all, tpe)
    i32 = dict(dtype=torch.int32, device=dst.device)
    groups, loffs, counts = torch.empty(R, NvS, 3, **i32), torch.empty(R, NvS, **i32), torch.empty(R, 2, **i32)
    n = R * _lib.lib().mep_dedup_scratch_bytes(group.S, R)
    work = torch.empty(n, dtype=torch.uint8, device=dst.device)
    rc = _lib.lib().mep_build_dedup_ranks(dst.data_ptr(), 0, R, group.S, group.K, R, NvS, groups.data_ptr(),
                                          loffs.data_ptr(), counts.data_ptr(), work.data_ptr(), n, _lib.current_stream())
    _lib.check(rc, "mep_build_dedup_ranks")
    t = _PlanTensors(dst, zfr, cu)
    # unbind makes a tensor's views in one call: 0.7 of the time of indexing each (8 ranks: 82 us against 124)
    views = zip(*(v.unbind(0) for v in (dst, zfr, stats, groups, loffs, counts)))
    plans = [MoonEPCommPlan(dst=d, experts_to_copy=etc, zero_fill_ranges=z, remote_stats=st, dup_groups=dg,
                            dup_loffs=dl, dup_counts=dc, N=group.S * group.K, R=R, E=group.E, NvS=NvS, K=group.K)
             for d, z, st, dg, dl, dc in views]
    for p in plans:
        p.dst._group_tensors = t
    return plans, t


class _PlanTensors:
    """A group's plans with a leading rank dimension: dst [R,N], zero_fill [R,2*epn,2], cu [R,2*epn]."""

    def __init__(self, dst, zero_fill, cu):
        self.dst, self.zero_fill, self.cu = dst, zero_fill, cu


def _rank_addresses(t):
    """Where each rank's part of a tensor with a leading rank dimension starts."""
    first, step = t.data_ptr(), t.stride(0) * t.element_size()
    return list(range(first, first + step * t.shape[0], step))


def _plan_tensors(group, plans):
    """The stacked tensors of ``plans``: those they are views of, where a whole-group dispatch made
    them (any of those in flight: the plans carry them), else stacked here; the groups' ends are
    known to the former only."""
    # the kernels read and write where the plans say, for as many ranks as the group has
    R, sizes = group.R, (group.S * group.K, group.R, group.E, group.NvS, group.K)
    assert len(plans) == R, f"a group of {R} ranks takes {R} plans, got {len(plans)}"
    for r, p in enumerate(plans):
        got = (p.N, p.R, p.E, p.NvS, p.K)
        assert got == sizes, f"plan {r} must be of N, R, E, NvS, K = {sizes}, got {got}"
    own = getattr(plans[0].dst, "_group_tensors", None)
    # `own` holds its memory, so an equal address is the same memory
    if own is None or [p.dst.data_ptr() for p in plans] != _rank_addresses(own.dst):
        return _PlanTensors(torch.stack([p.dst for p in plans]), torch.stack([p.zero_fill_ranges for p in plans]), None)
    if [p.zero_fill_ranges.data_ptr() for p in plans] == _rank_addresses(own.zero_fill):
        return own
    return _PlanTensors(own.dst, torch.stack([p.zero_fill_ranges for p in plans]), own.cu)


def _check_group_tokens(group, x_all, w_all):
    R, S, H, K = group.R, group.S, group.H, group.K
    assert x_all.dtype == torch.bfloat16 and x_all.is_cuda and tuple(x_all.shape) == (R, S, H), (
        f"tokens must be bf16 [R={R}, S={S}, H={H}] on the GPU, got {tuple(x_all.shape)} {x_all.dtype}")
    if w_all is not None:
        assert w_all.dtype == torch.float32 and tuple(w_all.shape) == (R, S, K) and w_all.device == x_all.device, (
            f"route weights must be fp32 [R={R}, S={S}, K={K}], got {tuple(w_all.shape)} {w_all.dtype}")


class _GroupDispatch(torch.autograd.Function):
    """tokens [R,S,H] (+ weights [R,S,K]) -> rows [R,NvS,H] (+ slots [R,NvS])."""

    @staticmethod
    def forward(ctx, group, x_all, w_all, topk_all, tpe):
        _check_group_tokens(group, x_all, w_all)
        plans, t = _group_plans(group, topk_all, tpe)
        rows, slots = _dispatch_all(group, x_all.contiguous(), None if w_all is None else w_all.contiguous(),
                                    t.dst, t.zero_fill, t.cu)
        ctx.group, ctx.t, ctx.has_w = group, t, w_all is not None
        group._note(rows, 0.0 if slots is None else slots)
        group.last_plans, group.last_cu_seqlens = plans, t.cu
        ctx.mark_non_differentiable(t.cu)
        ctx.set_materialize_grads(False)   # `cu` has none: a zero tensor for it is an allocation and a launch
        return rows, slots, t.cu

    @staticmethod
    def backward(ctx, g_rows, g_slots, _g_cu):
        if g_rows is None:     # only the weight slots were used
            g_rows = torch.zeros(ctx.group.R, ctx.group.NvS, ctx.group.H, dtype=torch.bfloat16, device=ctx.t.dst.device)
        slots = None
        if ctx.has_w:
            slots = (torch.zeros(g_rows.shape[:2], dtype=torch.float32, device=g_rows.device) if g_slots is None
                     else g_slots.float().contiguous())
        rows = g_rows.to(torch.bfloat16).contiguous()
        ctx.group._note(rows, slots)
        gx, gw = _combine_all(ctx.group, rows, slots, ctx.t.dst)
        return None, gx, gw, None, None


class _GroupCombine(torch.autograd.Function):
    """expert outputs [R,NvS,H] -> token-major [R,S,H] (unweighted K-sum)."""

    @staticmethod
    def forward(ctx, group, plans, y_all):
        ctx.group, ctx.t = group, _plan_tensors(group, plans)
        assert tuple(y_all.shape) == (group.R, group.NvS, group.H)
        rows = y_all.to(torch.bfloat16).contiguous()
        group._note(rows)
        return _combine_all(group, rows, None, ctx.t.dst)[0]

    @staticmethod
    def backward(ctx, g_out):
        t, g = ctx.t, g_out.to(torch.bfloat16).contiguous()
        rows = _dispatch_all(ctx.group, g, None, t.dst, t.zero_fill, t.cu)[0]
        ctx.group._note(rows)
        return None, None, rows


class _GroupPrefetch(torch.autograd.Function):
    """fp32 master weights [R,epn,H,H'] -> bf16 compute views [R,2*epn,H,H']:
    each rank's local experts followed by its prefetch slots.  Backward is
    ``reduce_grad``: the slots' grads are summed into their owners' grads in
    fp32."""

    @staticmethod
    def forward(ctx, group, experts_to_copy, master):
        R, epn = group.R, group.epn
        local = master.to(torch.bfloat16).contiguous()
        pool = torch.zeros_like(local)
        for r in range(R):     # a rank's slots filled from all owners in one launch
            launch_prefetch_pull((local,) * 3, (pool,) * 3, experts_to_copy, rank=r)
        ctx.group, ctx.etc = group, experts_to_copy
        return torch.cat([local, pool], dim=1)

    @staticmethod
    def backward(ctx, g_views):
        group = ctx.group
        R, epn = group.R, group.epn
        grad = g_views[:, :epn].float().contiguous()
        slots = g_views[:, epn:].float().contiguous()
        for r in range(R):
            # every rank reads before any rank clears (a barrier in the reference): only
            # the summing half runs here, the slot grads are temporaries nobody reads again
            launch_grad_reduce(grad[r], slots, ctx.etc, rank=r, phase="reduce")
        return None, None, grad


class _GroupExpertFFN(torch.autograd.Function):
    """Rows of every rank through its experts on the matrix cores.

    fp32 master weights in the orientation the kernels read: gate / up
    [R, epn, H', H], down [R, epn, H, H'].  Forward: bf16 compute views (local
    experts, then the prefetch slots), then the fused gate/up GEMM and the down
    GEMM with the route weight applied, each one launch over the groups of all
    ranks (a rank's own have too few tiles to fill the GPU).  Backward: the
    grouped gradient GEMMs, then every slot's fp32 weight gradient is summed
    into its owner's."""

    @staticmethod
    def forward(ctx, group, experts_to_copy, cu_all, rows_all, slots_all, gate_m, up_m, down_m):
        tp = group.world.token_padding
        views = _fill_views(group, experts_to_copy, (gate_m, up_m, down_m))              # [R, 2*epn, ...]
        args = (rows_all.contiguous(), None if slots_all is None else slots_all.contiguous(), cu_all.contiguous(), *views)
        res = _lib.host().ffn_forward(*args, tp, True)
        ctx.native = res is not None
        if not ctx.native:     # sizes that only the single products take: rank by rank
            each = [ffn.grouped_ffn_hip_forward(*_of_rank(args, r), token_padding=tp) for r in range(group.R)]
            res = torch.stack([y for y, _ in each]), [keep for _, keep in each]
        ctx.group, ctx.etc, ctx.args, ctx.saved = group, experts_to_copy, args, res[1]
        return res[0]

    @staticmethod
    def backward(ctx, g_out):
        group, args = ctx.group, ctx.args
        R, epn, tp = group.R, group.epn, group.world.token_padding
        g_out = g_out.to(torch.bfloat16).contiguous()
        # every rank's weight gradients in fp32: its local experts' and its slots' (the latter are
        # read for occupied slots only, so those of unused ones are left unwritten)
        own, slots = (tuple(torch.empty(R, epn, *v.shape[2:], dtype=torch.float32, device=v.device) for v in args[3:])
                      for _ in range(2))
        res = _lib.host().ffn_backward(*args, tp, g_out, *ctx.saved, True, own, slots) if ctx.native else None
        if res is not None:
            drows, dslots = res[:2]
        else:
            drows, dslots = [], []
            for r in range(R):
                keep = [t[r] for t in ctx.saved] if ctx.native else ctx.saved[r]
                g = ffn.grouped_ffn_hip_backward(g_out[r], *_of_rank(args, r), keep, token_padding=tp,
                                                 skip_unused_slots=True)
                drows.append(g[0])
                dslots.append(g[1])
                for o, s, full in zip(own, slots, g[2:]):
                    o[r].copy_(full[:epn])
                    s[r].copy_(full[epn:])
            drows = torch.stack(drows)
            dslots = None if args[1] is None else torch.stack(dslots)
        # every rank reads before any rank would clear: summing half only
        arr_p, arr_i = C.c_void_p * 3, C.c_int64 * 3
        elems = [int(v.shape[2]) * int(v.shape[3]) for v in args[3:]]
        rc = _lib.lib().mep_grad_reduce_batch(
            3, arr_p(*[t.data_ptr() for t in own]), arr_p(*[t.data_ptr() for t in slots]),
            arr_i(*[epn * n for n in elems]), arr_i(*elems), ctx.etc.data_ptr(), 0, R, epn, R, _lib.REDUCE_NO_CLEAR,
            _lib.current_stream())
        _lib.check(rc, "mep_grad_reduce_batch")
        return (None, None, None, drows, dslots, *own)


def _of_rank(args, r):
    return [None if t is None else t[r] for t in args]


def _fill_views(group, experts_to_copy, masters):
    """bf16 compute views ``[R, 2*epn, ...]`` of the three projections: every rank's local experts
    rounded from the masters, its occupied slots copied from their owners (one launch each).  Slots
    that hold no expert are left as they are: no row goes there."""
    R, epn = group.R, group.epn
    assert experts_to_copy.dtype == torch.int32 and experts_to_copy.is_contiguous() and \
        tuple(experts_to_copy.shape) == (R, epn), f"experts_to_copy must be int32 [R={R}, epn={epn}]"
    for m in masters:
        assert m.dim() == 4 and tuple(m.shape[:2]) == (R, epn), f"masters must be [R={R}, epn={epn}, ., .]"
    views = [torch.empty(R, 2 * epn, *m.shape[2:], dtype=torch.bfloat16, device=m.device) for m in masters]
    per = [int(m.shape[2]) * int(m.shape[3]) for m in masters]
    assert all(n % 8 == 0 for n in per)
    arr_p, arr_i = C.c_void_p * 3, C.c_int64 * 3
    lib, st = _lib.lib(), _lib.current_stream()
    dense = [m.detach().float().contiguous() for m in masters]
    rc = lib.mep_cast_bf16(3, arr_p(*[m.data_ptr() for m in dense]), arr_p(*[v.data_ptr() for v in views]),
                           arr_i(*[epn * n for n in per]), arr_i(*[2 * epn * n for n in per]), R, st)
    _lib.check(rc, "mep_cast_bf16")
    rank_bytes = arr_i(*[4 * epn * n for n in per])
    rc = lib.mep_prefetch_pull_ranks(
        3, arr_p(*[v.data_ptr() for v in views]), rank_bytes,
        arr_p(*[v.data_ptr() + 2 * epn * n for v, n in zip(views, per)]), rank_bytes, arr_i(*[2 * n for n in per]),
        experts_to_copy.data_ptr(), 0, R, epn, R, st)
    _lib.check(rc, "mep_prefetch_pull_ranks")
    return views


def group_expert_ffn_hip(group, experts_to_copy, cu_all, rows_all, slots_all, gate_m, up_m, down_m):
    """rows [R,NvS,H] bf16, slots [R,NvS] fp32 | None, cu_all [R,2*epn]; fp32 masters gate / up
    [R,epn,H',H], down [R,epn,H,H'] -> expert outputs [R,NvS,H] bf16.  Differentiable in rows,
    slots and the three masters; needs token_padding % 128 == 0 and H, H' multiples of 256."""
    return _GroupExpertFFN.apply(group, experts_to_copy, cu_all, rows_all, slots_all, gate_m, up_m, down_m)


def group_dispatch(group, x_all, w_all, topk_all, tpe):
    """-> (rows [R,NvS,H], weight slots [R,NvS] | None, cu_seqlens [R,2*epn], plans)"""
    hidden, slots, cu = _GroupDispatch.apply(group, x_all, w_all, topk_all, tpe)
    return hidden, slots, cu, group.last_plans


def group_combine(group, plans, y_all):
    return _GroupCombine.apply(group, plans, y_all)


def group_compute_views(group, experts_to_copy, master_weights):
    return _GroupPrefetch.apply(group, experts_to_copy, master_weights)
