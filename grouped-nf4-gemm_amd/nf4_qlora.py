"""Differentiable grouped 4-bit expert projection for QLoRA training.

The frozen base weight stays packed. Forward runs the grouped forward kernel;
backward needs only the input gradient ``grad_out @ W`` (the base weight is
not trained), which the grouped dgrad kernel computes from the same packed
bytes in one launch. No decoded weight is kept between forward and backward.

LoRA composes pre-activation: ``fused_grouped_lora`` returns
``W x + scaling * B (A x)`` per group, so a caller applies SwiGLU after it.

Interface and semantics follow the reference's kernel/nf4_qlora.py:32-305
(``FusedGroupedNf4``, ``gemm_4bit_grouped_train``, ``lora_delta_grouped``,
``_lora_delta_grouped_loop``, ``fused_grouped_lora``, ``_PAD_WASTE_LIMIT``).
"""
from __future__ import annotations

import numpy as np
import torch

import _hiplib
import mxfp4_grouped
import nf4_grouped

# Padded-bmm cutoff for lora_delta_grouped: above this many padded rows per
# real row the per-expert loop is used instead (reference nf4_qlora.py:26-30).
_PAD_WASTE_LIMIT = 4.0


def _host_ints(x):
    """A host list of ints from a list, tuple or tensor (one transfer)."""
    if isinstance(x, (list, tuple)):
        return [int(v) for v in x]
    return [int(v) for v in x.tolist()]


def _exact_dgrad_loop(grad_out, packed, scales, sizes, expert_ids, decode):
    """grad_a = grad_out @ decode(W[e]) one group at a time, each decoded
    expert dropped before the next (the reference's exact backward,
    nf4_qlora.py:137-166). Runs where grad_out lives; the weights of one
    expert are moved there if they are stored elsewhere."""
    _E, N, half = packed.shape
    K = half * 2
    grad_a = torch.empty(grad_out.shape[0], K, dtype=grad_out.dtype, device=grad_out.device)
    sizes_h, eids_h = _host_ints(sizes), _host_ints(expert_ids)
    row = 0
    for g, e in enumerate(eids_h):
        m = sizes_h[g]
        if m == 0:
            continue
        pe = packed[e].to(grad_out.device, non_blocking=True)
        se = scales[e].to(grad_out.device, non_blocking=True)
        w = decode(pe, se, N, K).to(grad_out.dtype)
        grad_a[row:row + m] = grad_out[row:row + m] @ w
        del pe, se, w
        row += m
    return grad_a


class FusedGroupedNf4(torch.autograd.Function):
    """Grouped NF4 forward through the kernel; input gradient through the
    grouped dgrad kernel (or, with ``dgrad_kernel=False``, through the exact
    per-expert decode). ``packed`` / ``absmax`` are constants: they are kept
    on ctx (or re-fetched from ``weights_fn`` at backward time, so offloaded
    storage is not pinned by a reference here), never saved for gradient."""

    @staticmethod
    def forward(ctx, a_cat, packed, absmax, sizes, expert_ids, weights_fn=None,
                dgrad_kernel=True):
        out = nf4_grouped.gemm_4bit_grouped(a_cat, packed, absmax, sizes, expert_ids)
        ctx.weights_fn = weights_fn
        ctx.packed, ctx.absmax = (packed, absmax) if weights_fn is None else (None, None)
        ctx.sizes, ctx.expert_ids = sizes, expert_ids   # as given: no device reads here
        ctx.dgrad_kernel = dgrad_kernel
        return out

    @staticmethod
    def backward(ctx, grad_out):
        if not ctx.needs_input_grad[0]:
            return (None,) * 7
        packed, absmax = ((ctx.packed, ctx.absmax) if ctx.weights_fn is None
                          else ctx.weights_fn())
        grad_out = grad_out.contiguous()
        if (ctx.dgrad_kernel and packed.device == grad_out.device
                and nf4_grouped.dgrad_eligible(grad_out, packed, absmax) is None):
            grad_a = nf4_grouped.dgrad_4bit_grouped(grad_out, packed, absmax,
                                                    ctx.sizes, ctx.expert_ids)
        else:
            grad_a = _exact_dgrad_loop(grad_out, packed, absmax, ctx.sizes, ctx.expert_ids,
                                       nf4_grouped.dequant_ref)
        return (grad_a,) + (None,) * 6


def gemm_4bit_grouped_train(a_cat, packed, absmax, sizes, expert_ids, weights_fn=None,
                            dgrad_kernel=True):
    """``gemm_4bit_grouped`` with a gradient for ``a_cat`` (reference
    nf4_qlora.py:168-178). ``weights_fn``: zero-argument callable returning
    ``(packed, absmax)`` at backward time, for offload-staged storage."""
    return FusedGroupedNf4.apply(a_cat, packed, absmax, sizes, expert_ids, weights_fn,
                                 dgrad_kernel)


class FusedGroupedMxfp4(torch.autograd.Function):
    """The MXFP4 counterpart: forward and input gradient both through the
    kernels (the reference's GPU backward is a per-expert decode loop,
    kernel/mxfp4_qlora.py:106-122; ``dgrad_kernel=False`` keeps that)."""

    @staticmethod
    def forward(ctx, a_cat, blocks, scales, sizes, expert_ids, weights_fn=None,
                dgrad_kernel=True):
        out = mxfp4_grouped.gemm_mxfp4_grouped(a_cat, blocks, scales, sizes, expert_ids)
        ctx.weights_fn = weights_fn
        ctx.blocks, ctx.scales = (blocks, scales) if weights_fn is None else (None, None)
        ctx.sizes, ctx.expert_ids = sizes, expert_ids
        ctx.dgrad_kernel = dgrad_kernel
        return out

    @staticmethod
    def backward(ctx, grad_out):
        if not ctx.needs_input_grad[0]:
            return (None,) * 7
        blocks, scales = ((ctx.blocks, ctx.scales) if ctx.weights_fn is None
                          else ctx.weights_fn())
        grad_out = grad_out.contiguous()
        flat = mxfp4_grouped._flat_blocks(blocks)
        if ctx.dgrad_kernel and flat.device == grad_out.device:
            grad_a = mxfp4_grouped.dgrad_mxfp4_grouped(grad_out, flat, scales, ctx.sizes,
                                                       ctx.expert_ids)
        else:
            from mxfp4_pack_ref import dequant_mxfp4

            def decode(pe, se, n, k):
                return dequant_mxfp4(pe.reshape(n, k // 32, 16), se.reshape(n, k // 32))

            grad_a = _exact_dgrad_loop(grad_out, flat, scales, ctx.sizes, ctx.expert_ids,
                                       decode)
        return (grad_a,) + (None,) * 6


def gemm_mxfp4_grouped_train(a_cat, blocks, scales, sizes, expert_ids, weights_fn=None,
                             dgrad_kernel=True):
    """``gemm_mxfp4_grouped`` with a gradient for ``a_cat``."""
    return FusedGroupedMxfp4.apply(a_cat, blocks, scales, sizes, expert_ids, weights_fn,
                                   dgrad_kernel)


def lora_delta_grouped(a_cat, lora_A, lora_B, sizes, expert_ids, scaling=1.0):
    """Per-group low-rank delta ``scaling * (x @ A[e].T) @ B[e].T`` over a
    group-sorted block (reference nf4_qlora.py:181-254). ``lora_A`` is
    ``[E, r, K]``, ``lora_B`` ``[E, N, r]``; returns ``[T, N]`` or ``None``
    when no group has rows. Groups are padded to the widest and run as two
    batched matmuls; when padding would exceed ``_PAD_WASTE_LIMIT`` times the
    real rows, the per-group loop runs instead. ``expert_ids`` on the device
    is never read on the host."""
    nz = [g for g in range(len(sizes)) if int(sizes[g]) > 0]
    if not nz:
        return None
    rows = [int(sizes[g]) for g in nz]
    total, widest = sum(rows), max(rows)
    if len(rows) * widest > _PAD_WASTE_LIMIT * total:
        return _lora_delta_grouped_loop(a_cat, lora_A, lora_B, sizes, expert_ids, scaling)
    dev = a_cat.device
    if torch.is_tensor(expert_ids) and expert_ids.device.type != "cpu":
        sz_d, nz_d = nf4_grouped.to_device_i32((rows, nz), dev)
        eid = expert_ids.to(dev)[nz_d.to(torch.int64)].to(torch.int64)
    else:
        ids = _host_ints(expert_ids)
        ids = [ids[g] for g in nz]
        E = min(lora_A.shape[0], lora_B.shape[0])
        if max(ids) >= E:   # (on the device, indexing would abort the process)
            raise IndexError(f"expert id {max(ids)} is out of range for adapters of {E} experts")
        sz_d, eid_d = nf4_grouped.to_device_i32((rows, ids), dev)
        eid = eid_d.to(torch.int64)
    sz = sz_d.to(torch.int64)
    # row -> (group, position in group), built on the device; output_size
    # keeps repeat_interleave from reading sz on the host
    grp = torch.repeat_interleave(torch.arange(len(rows), device=dev), sz, output_size=total)
    start = torch.cumsum(sz, 0) - sz
    pos = torch.arange(total, device=dev) - start[grp]
    A, B = lora_A[eid], lora_B[eid]                        # [G, r, K], [G, N, r]
    x = a_cat.new_zeros(len(rows), widest, a_cat.shape[1], dtype=A.dtype)
    x[grp, pos] = a_cat[:total].to(A.dtype)
    d = scaling * torch.bmm(torch.bmm(x, A.transpose(1, 2)), B.transpose(1, 2))
    out = torch.zeros(a_cat.shape[0], B.shape[1], dtype=d.dtype, device=dev)
    out[:total] = d[grp, pos]
    return out


def _lora_delta_grouped_loop(a_cat, lora_A, lora_B, sizes, expert_ids, scaling=1.0):
    """Per-group reference for ``lora_delta_grouped`` (reference
    nf4_qlora.py:257-283); the fallback for heavily skewed groups."""
    out = None
    row = 0
    for g, e in enumerate(_host_ints(expert_ids)):
        m = int(sizes[g])
        if m == 0:
            continue
        A, B = lora_A[e], lora_B[e]
        d = scaling * ((a_cat[row:row + m].to(A.dtype) @ A.T) @ B.T)
        if out is None:
            out = torch.zeros(a_cat.shape[0], B.shape[0], dtype=d.dtype, device=a_cat.device)
        out[row:row + m] = d
        row += m
    return out


# ------------------------------------------------- the fused low-rank kernels --

def _watched() -> bool:
    """Whether functorch, a dispatch or function mode or a tracer watches the
    torch calls of this thread."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing()
            or torch._C._functorch.peek_interpreter_stack() is not None
            or torch._C._len_torch_dispatch_stack() > 0
            or torch._C._len_torch_function_stack() > 0)


def _transforming() -> bool:
    """Whether something other than plain eager autograd watches the forward's
    torch calls (also forward-mode and autocast): then the torch composition
    runs, which they all see."""
    from torch.autograd import forward_ad
    return _watched() or forward_ad._current_level >= 0 or torch.is_autocast_enabled()


def _kernels_take(out, a_cat, lora_A, lora_B, sizes, scaling, expert_ids, n_packed) -> bool:
    """Whether the HIP kernels take this low-rank delta: bf16 rows and fp32
    adapters on one GPU, plain contiguous tensors, r % 4 == 0 and r <= 64,
    widths that are multiples of 8, every row in a group, a plain number as
    ``scaling`` (a tensor may be learnable, live on the device or have one
    value per column: the torch composition multiplies by it), and adapters
    for every expert of the packed stack or for every id known on the host
    (the kernels add nothing for others; the composition's indexing raises)."""
    if not isinstance(scaling, (int, float)):
        return False
    ts = (out, a_cat, lora_A, lora_B)
    if not all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda
               and t.device == out.device for t in ts):
        return False
    if (out.dtype, a_cat.dtype) != (torch.bfloat16, torch.bfloat16) or lora_A.dim() != 3:
        return False
    if (lora_A.dtype, lora_B.dtype) != (torch.float32, torch.float32) or lora_B.dim() != 3:
        return False
    (T, N), K = out.shape, a_cat.shape[1]
    E, r, _ = lora_A.shape
    return (tuple(lora_A.shape) == (E, r, K) and tuple(lora_B.shape) == (E, N, r)
            and 0 < E <= 65535 and 4 <= r <= 64 and r % 4 == 0 and K % 8 == 0 and N % 8 == 0
            and lora_A.is_contiguous() and lora_B.is_contiguous()
            and lora_A.data_ptr() % 16 == 0 and lora_B.data_ptr() % 16 == 0
            and T > 0 and sum(sizes) == T and not _transforming()
            and (E >= n_packed or not (torch.is_tensor(expert_ids) and expert_ids.is_cuda)
                 and all(e < E for e, m in zip(_host_ints(expert_ids), sizes) if m > 0)))


# Rows of a chunk of gnf4_hip_lora_wgrad_split
_WGRAD_CHUNK = 256


class _LoraTables:
    """Device tables of one routing: tile and row offsets, expert ids. Nothing
    of the caller's is kept: it may write the next layer's routing into the
    same tensor or list before backward."""

    def __init__(self, sizes, expert_ids, dev, E):
        self.sizes, self.G = sizes, len(sizes)   # (a list of ints of its own)
        on_dev = torch.is_tensor(expert_ids) and expert_ids.is_cuda
        ids = [] if on_dev else [nf4_grouped._np_ids(expert_ids).copy()]
        m = np.asarray(sizes, dtype=np.int32)
        most = max(sizes)   # rows of the largest expert (device ids: group)
        if not on_dev and len(set(ids[0].tolist())) < self.G:
            most = int(np.bincount(ids[0], m).max())
        # Whether the adapter gradients take the kernel that splits an
        # expert's rows over waves: where one wave per expert would run long
        # (from 384 rows) while other waves idle (fewer than 32 such experts'
        # worth of rows). Direct and split, MI355X, K = 2048, r = 16, even
        # groups: 8 experts of 320 / 384 / 512 / 4096 rows 25 / 29 / 38 / 328
        # and 23 / 23 / 24 / 46 us; 32 experts of 320 / 384 / 1024 31 / 36 / 88
        # and 31 / 32 / 44 us; 64 experts of 384 / 512 / 1024 39 / 50 / 101 and
        # 45 / 45 / 75 us, at r = 64 90 / 113 / 211 and 132 / 133 / 275 us.
        # More device ids than experts: some are repeated, so it splits.
        self.split = most >= 384 and 32 * most >= sum(sizes) or self.G > E
        off = np.zeros((3 if self.split else 2, self.G + 1), dtype=np.int32)
        np.cumsum((m + 15) // 16, out=off[0, 1:])
        np.cumsum(m, out=off[1, 1:])
        if self.split:
            np.cumsum((m + _WGRAD_CHUNK - 1) // _WGRAD_CHUNK, out=off[2, 1:])
            self.n_chunks = int(off[2, -1])
        views = nf4_grouped.to_device_i32([*off, *ids], dev)
        self.n = int(off[0, -1])
        self.tile_off, self.row_off = views[:2]
        self.chunk_off = views[2] if self.split else None
        self.ids = (torch.empty(self.G, dtype=torch.int32, device=dev).copy_(expert_ids)
                    if on_dev else views[-1])
        self.expert_ids = self.ids if on_dev else ids[0]   # for the composition
        self.args = (self.tile_off.data_ptr(), self.row_off.data_ptr(), self.ids.data_ptr(),
                     self.G, self.n)


def _rows(t):
    """``t [T, C]`` as the kernels read it: 16-byte aligned rows of unit stride
    that do not overlap. Anything else is copied: a gradient may come
    broadcast (row stride 0, from ``out.sum(0)``), transposed or at any
    offset."""
    if (t.stride(1) != 1 or t.stride(0) % 8 or t.stride(0) < t.shape[1]
            or t.data_ptr() % 16):
        return t.clone(memory_format=torch.contiguous_format)
    return t


class _Launches:
    """The LoRA launches of one direction: the library and the current stream
    of a device, looked up once."""

    def __init__(self, dev):
        self.lib = _hiplib.load()
        self.stream = nf4_grouped._stream_ptr(dev)

    def __call__(self, name, *args):
        _hiplib.check(getattr(self.lib, name)(*args, self.stream), "fused_grouped_lora")


def _lora_down(call, x, w, transposed, tb, scale, r):
    E, C = w.shape[0], x.shape[1]
    y = torch.empty(x.shape[0], r, dtype=torch.float32, device=x.device)
    call("gnf4_hip_lora_down", x.data_ptr(), x.stride(0), w.data_ptr(), transposed, E, C, r,
         *tb.args, scale, y.data_ptr())
    return y


def _lora_up(call, u, w, transposed, C, tb, scale, base=None):
    T, r = u.shape
    out = torch.empty(T, C, dtype=torch.bfloat16, device=u.device)
    call("gnf4_hip_lora_up", u.data_ptr(), w.data_ptr(), transposed, w.shape[0], C, r, *tb.args,
         scale, base.data_ptr() if base is not None else None,
         base.stride(0) if base is not None else 0, out.data_ptr(), out.stride(0))
    return out


def _lora_wgrad(call, p, q, like, transposed, tb, scale):
    dw = torch.empty_like(like)
    E, C, r = like.shape[0], p.shape[1], q.shape[1]
    if tb.split:
        part = torch.empty(tb.n_chunks, C * r, dtype=torch.float32, device=p.device)
        call("gnf4_hip_lora_wgrad_split", p.data_ptr(), p.stride(0), q.data_ptr(), transposed, E,
             C, r, tb.chunk_off.data_ptr(), tb.row_off.data_ptr(), tb.ids.data_ptr(), tb.G,
             tb.n_chunks, scale, part.data_ptr(), dw.data_ptr())
        return dw
    call("gnf4_hip_lora_wgrad", p.data_ptr(), p.stride(0), q.data_ptr(), transposed, E, C, r,
         tb.ids.data_ptr(), tb.row_off.data_ptr(), tb.G, scale, dw.data_ptr())
    return dw


class _LoraAdd(torch.autograd.Function):
    """``base + bf16(scaling * (a A[e]^T) B[e]^T)`` through the kernels of
    csrc/gnf4_lora.hip (two forward, four backward launches, fp32 sums): the
    values and gradients of adding ``lora_delta_grouped``. A backward that is
    itself differentiated, batched (``is_grads_batched``) or watched runs that
    torch composition instead.

    Backward reads copies of the activations and adapters, as the
    composition's gathered ones are: a program may update the adapters, or
    refill its activation buffer, before it. They are outputs of this function
    as well, so that a second differentiation reaches the inputs through them
    (MI355X, 8192 rows, 128 experts, K = 2048, N = 1536, r = 16: 26 of the
    352 us of kernels of a training pass)."""

    @staticmethod
    def forward(ctx, base, a_cat, lora_A, lora_B, sizes, expert_ids, scaling, recording):
        need = ctx.needs_input_grad[1:4]   # by requires_grad, also under no_grad
        recording = recording and any(need)
        if recording:
            a_cat, lora_A, lora_B = a_cat.clone(), lora_A.clone(), lora_B.clone()
        a = _rows(a_cat.detach())
        tb = _LoraTables(sizes, expert_ids, a.device, lora_A.shape[0])
        with nf4_grouped._device_ctx(a.device):
            call = _Launches(a.device)
            u = _lora_down(call, a, lora_A, 0, tb, 1.0, lora_A.shape[1])
            out = _lora_up(call, u, lora_B, 0, lora_B.shape[1], tb, float(scaling), _rows(base))
        if not recording:
            return out
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(a_cat, lora_A, lora_B, u)
        ctx.tables, ctx.scaling = tb, scaling
        copies = (a_cat, lora_A, lora_B)
        ctx.mark_non_differentiable(*(t for t, n in zip(copies, need) if not n))
        return (out, *copies)

    @staticmethod
    def backward(ctx, g, *g_copies):
        if g is None or not g_copies:
            return (g, *(g_copies or (None,) * 3), None, None, None, None)
        a_cat, A, B, u = ctx.saved_tensors
        tb, scaling, need = ctx.tables, ctx.scaling, ctx.needs_input_grad
        twice = torch.is_grad_enabled()
        if (twice or _watched() or type(g) is not torch.Tensor
                or torch._C._functorch.is_legacy_batchedtensor(g)):
            with torch.enable_grad():
                ins = [t for t, n in zip((a_cat, A, B), need[1:4]) if n]
                d = lora_delta_grouped(a_cat, A, B, tb.sizes, tb.expert_ids,
                                       scaling).to(g.dtype)
                got = iter(torch.autograd.grad(d, ins, g, create_graph=twice))
            grads = [next(got) if n else None for n in need[1:4]]
        else:
            s = float(scaling)
            ga = gA = gB = gu = None
            with nf4_grouped._device_ctx(g.device):
                call, gv = _Launches(g.device), _rows(g)
                if need[1] or need[2]:
                    gu = _lora_down(call, gv, B, 1, tb, s, A.shape[1])
                if need[1]:
                    ga = _lora_up(call, gu, A, 1, a_cat.shape[1], tb, 1.0)
                if need[2]:
                    gA = _lora_wgrad(call, _rows(a_cat), gu, A, 1, tb, 1.0)
                if need[3]:
                    gB = _lora_wgrad(call, gv, u, B, 0, tb, s)
            grads = [ga, gA, gB]
        grads = [x if y is None else y if x is None else x + y for x, y in zip(grads, g_copies)]
        return (g, *grads, None, None, None, None)


def fused_grouped_lora(a_cat, packed, absmax, sizes, expert_ids, lora_A=None, lora_B=None,
                       weights_fn=None, scaling=1.0, dgrad_kernel=True):
    """Frozen NF4 projection plus the trainable delta, pre-activation
    (reference nf4_qlora.py:286-305): differentiable in ``a_cat``, ``lora_A``
    and ``lora_B``."""
    out = gemm_4bit_grouped_train(a_cat, packed, absmax, sizes, expert_ids,
                                  weights_fn=weights_fn, dgrad_kernel=dgrad_kernel)
    if lora_A is None or lora_B is None:
        return out
    rows = [int(m) for m in sizes]
    if _kernels_take(out, a_cat, lora_A, lora_B, rows, scaling, expert_ids, packed.shape[0]):
        out = _LoraAdd.apply(out, a_cat, lora_A, lora_B, rows, expert_ids, scaling,
                             torch.is_grad_enabled())
        return out[0] if isinstance(out, tuple) else out
    delta = lora_delta_grouped(a_cat, lora_A, lora_B, sizes, expert_ids, scaling)
    return out if delta is None else out + delta.to(out.dtype)
