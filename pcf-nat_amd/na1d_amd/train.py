"""An encoder layer in training as one autograd node (``na1d_train_layer_*`` of the C ABI).

:func:`layer` runs norm -> attention -> residual -> norm -> MLP -> residual of ``models.NATFLayer`` and its backward
through the kernels of ``csrc/na1d_train.hip``, all launched from native code: the parameters, buffers, random draws and
results are those of the modules, which stay what runs wherever something here does not fit.
"""
from __future__ import annotations

import ctypes

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd.function import once_differentiable
from torch.autograd.graph import increment_version

from . import _lib

_P, _I, _F = ctypes.c_void_p, ctypes.c_int32, ctypes.c_float


class _Norm(ctypes.Structure):                     # na1d_train_norm
    _fields_ = [(n, _P) for n in "weight bias batch_mean batch_var batches dweight dbias".split()] + [("eps", _F)]


class _Layer(ctypes.Structure):                    # na1d_train_layer
    _fields_ = ([(n, _I) for n in "dtype dim hidden heads window left dilation groups ordered".split()] + [("scale", _F)]
                + [("late", _I), ("norm", _Norm * 2)] + [(n, _P * 5) for n in "w b dw db".split()]
                + [(n, _P) for n in "rpb drpb pos scale_attn scale_mlp".split()])


def _aligned(t):
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


class _ByCtypes:
    """``train_forward`` and ``train_backward`` of ``csrc/na1d_torch.cpp``, which belongs to the library beside it, for one that
    NA1D_LIB names."""

    @staticmethod
    def _ptr(t):
        return None if t is None else t.data_ptr()

    @classmethod
    def _ptrs(cls, ts):
        return (_P * 5)(*map(cls._ptr, ts))

    @classmethod
    def train_forward(cls, x, by_channel, geom, state, numbers, scale_attn, scale_mlp, pos, params):
        lib, c, (n, t, dim) = _lib.load(), _Layer(*geom), x.shape
        dense, norms = pos is not None, params[1:5]
        c.w, c.b = cls._ptrs([*params[5::2], params[0] if dense else None]), cls._ptrs(params[6::2])
        for i, to in enumerate(c.norm):
            to.weight, to.bias, to.eps, to.batches = norms[2 * i].data_ptr(), norms[2 * i + 1].data_ptr(), numbers[2 * i + 1], state[3 * i + 2].data_ptr()
        c.rpb, c.pos, c.scale_attn, c.scale_mlp = None if dense else params[0].data_ptr(), cls._ptr(pos), cls._ptr(scale_attn), cls._ptr(scale_mlp)
        ref, out = ctypes.byref(c), torch.empty_like(x)
        with torch.cuda.device(x.device):
            stream = torch.cuda.current_stream().cuda_stream
            sizes = lib.na1d_train_layer_saved_bytes(ref, n, t), lib.na1d_train_layer_workspace_bytes(ref, n, t, 0)
            _lib.check(min(*sizes, 0), "na1d_train_layer_saved_bytes")
            saved, ws = (torch.empty(s, dtype=torch.uint8, device=x.device) for s in sizes)
            if by_channel is None:
                by_channel = x.new_empty((n, dim, t))
                _lib.check(lib.na1d_train_to_channels(ref, by_channel.data_ptr(), x.data_ptr(), n, t, stream), "na1d_train_to_channels")
            x1 = x.new_empty((n, dim, t))
            for part, (of, to) in enumerate(((by_channel, x1), (x1, out))):
                stats = torch.batch_norm_update_stats(of, state[3 * part], state[3 * part + 1], numbers[2 * part])
                c.norm[part].batch_mean, c.norm[part].batch_var = map(cls._ptr, stats)
                _lib.check(lib.na1d_train_layer_forward(ref, part, to.data_ptr(), x.data_ptr(), saved.data_ptr(), sizes[0], ws.data_ptr(),
                                                        sizes[1], n, t, stream), "na1d_train_layer_forward")
        increment_version(state)
        return out, saved

    @classmethod
    def train_backward(cls, dout, x, saved, geom, rpb, n1w, n2w, scale_attn, scale_mlp, pos, shapes):
        lib, c, (n, t, _) = _lib.load(), _Layer(*geom), x.shape
        dout, dx = _aligned(dout), torch.empty_like(x)
        grads = [torch.zeros(shapes[0], dtype=torch.float32, device=x.device)]       # the bias of the scores is added to
        grads += [torch.empty(s, dtype=torch.float32, device=x.device) for s in shapes[1:]]
        c.dw, c.db = cls._ptrs(grads[5::2] + ([] if pos is None else grads[:1])), cls._ptrs(grads[6::2])
        for to, w, dw, db in zip(c.norm, (n1w, n2w), grads[1:5:2], grads[2:5:2]):
            to.weight, to.dweight, to.dbias = w.data_ptr(), dw.data_ptr(), db.data_ptr()
        c.rpb, c.drpb, c.pos, c.scale_attn, c.scale_mlp = cls._ptr(rpb), grads[0].data_ptr(), cls._ptr(pos), cls._ptr(scale_attn), cls._ptr(scale_mlp)
        ref = ctypes.byref(c)
        with torch.cuda.device(x.device):
            nbytes = lib.na1d_train_layer_workspace_bytes(ref, n, t, 1)
            _lib.check(min(nbytes, 0), "na1d_train_layer_workspace_bytes")
            ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
            _lib.check(lib.na1d_train_layer_backward(ref, dx.data_ptr(), dout.data_ptr(), x.data_ptr(), saved.data_ptr(), saved.numel(),
                                                     ws.data_ptr(), nbytes, n, t, torch.cuda.current_stream().cuda_stream),
                       "na1d_train_layer_backward")
        return [dx, *grads]


class _TrainLayer(torch.autograd.Function):
    """The node's bookkeeping; allocations and launches are ``train_forward`` and ``train_backward`` of ``csrc/na1d_torch.cpp``."""

    @staticmethod
    def forward(ctx, x, by_channel, geom, nodes, norms, scales, pos, *params):
        state = [bn._buffers[name] for bn in norms for name in ("running_mean", "running_var", "num_batches_tracked")]
        out, saved = nodes.train_forward(x, by_channel, geom, state, [v for bn in norms for v in (bn.momentum, bn.eps)], *scales, pos, params)
        ctx.save_for_backward(x, saved, pos, params[0] if pos is None else None, params[1], params[3], *scales)
        ctx.late, ctx.geom, ctx.nodes = geom[-1], geom, nodes
        ctx.shapes = [p.shape for p in params]
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, dout):
        x, saved, pos, rpb, n1w, n2w, *scales = ctx.saved_tensors
        dx, *grads = ctx.nodes.train_backward(dout, x, saved, ctx.geom, rpb, n1w, n2w, *scales, pos, ctx.shapes)
        return (dx, None, None, None, None, None, None, *(g if need else None for g, need in zip(grads, ctx.needs_input_grad[7:])))


def plain(m, *classes):
    """Whether calling module ``m`` runs the forward of its class and nothing else."""
    if type(m) not in classes:
        return False
    d = m.__dict__
    return not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"] or "forward" in d)


def plain_call(x):
    """Whether nothing but autograd looks at the operations on ``x``: no tracer, transform, subclass or dispatch mode."""
    return (type(x) in (torch.Tensor, nn.Parameter) and not torch.compiler.is_compiling() and not torch.jit.is_tracing()
            and not torch.nn.modules.module._has_any_global_hook() and torch._C._functorch.peek_interpreter_stack() is None
            and torch.autograd.forward_ad._current_level < 0 and torch._C._len_torch_dispatch_stack() == 0
            and not torch._C._functorch.is_legacy_batchedtensor(x))       # of is_grads_batched


def _norm_fits(bn, dim, device):
    mean, var, batches = (bn._buffers.get(name) for name in ("running_mean", "running_var", "num_batches_tracked"))
    return (bn.training and bn.track_running_stats and bn.affine and bn.momentum is not None and bn.num_features == dim
            and all(s is not None and s.dtype == torch.float32 and s.device == device and s.shape == (dim,) for s in (mean, var))
            and batches is not None and batches.dtype == torch.int64 and batches.device == device)


def _drop_path_scale(m, x):
    """Stochastic depth's factor of each sample, drawn as ``models.DropPath`` draws it."""
    if not getattr(m, "drop_prob", 0.0) or not m.training:
        return None
    keep = 1 - m.drop_prob
    mask = (keep + torch.rand((x.shape[0], 1, 1), dtype=x.dtype, device=x.device)).floor_()
    return mask.float().view(-1).div_(keep)


def layer(m, x, pos_emb=None, attn_mask_global=None):
    """``models.NATFLayer`` ``m`` in training on ``x`` ([N, T, C], or [N, C, T] for channels-first models), or ``None`` where
    the kernels or their one autograd node would not be the same as the modules."""
    from . import models as M
    if not (x.is_cuda and m.training and torch.is_grad_enabled() and torch.is_autocast_enabled("cuda")
            and x.dim() == 3 and x.dtype in (torch.bfloat16, torch.float16) and x.dtype == torch.get_autocast_dtype("cuda")):
        return None
    # Sixteen layers a step, some forty lookups each: by the modules' own dictionaries, past nn.Module.__getattr__.
    parts = m._modules
    a, mlp, norms = parts.get("attn"), parts.get("mlp"), (parts.get("norm1"), parts.get("norm2"))
    cf = getattr(a, "channels_first", False)
    linear, norm = (M.Conv1x1, M.BatchNorm1d) if cf else (M.TokenLinear, M.TokenBatchNorm)
    if not (plain_call(x) and plain(a, M.NAttention if m.local else M.GlobalAttention) and plain(mlp, M.Mlp) and plain(norms[0], norm) and plain(norms[1], norm)
            and plain(parts.get("drop_path"), nn.Identity, M.DropPath)):
        return None
    in_a, in_mlp = a._modules, mlp._modules
    act, drops, projections = in_mlp.get("act"), (in_mlp.get("drop"), in_a.get("proj_drop")), [in_a.get("qkv"), in_a.get("proj"), in_mlp.get("fc1"), in_mlp.get("fc2")]
    if not (plain(act, nn.GELU) and act.approximate == "none" and plain(drops[0], nn.Dropout) and plain(drops[1], nn.Dropout)
            and all(plain(p, linear) for p in projections)):
        return None
    if not cf:
        norms = [b._modules.get("norm") for b in norms]
    if (a.na != "fused_qkv" if m.local else a.dense != "native") or a.attn_drop or not a.training or drops[0].p or drops[1].p or (not cf and not all(plain(b, M.BatchNorm1d) for b in norms)):
        return None
    xt = x.transpose(1, 2) if cf else x
    if xt.is_contiguous() and xt.data_ptr() % 16:
        return None
    n, t, dim = xt.shape
    if (t != a.attn_mask.shape[-2] if m.local else attn_mask_global is not None) or not all(_norm_fits(b, dim, x.device) for b in norms):
        return None
    pos = None
    if not m.local:
        linear_pos = in_a.get("linear_pos")
        if (pos_emb is None or type(pos_emb) is not torch.Tensor or pos_emb.requires_grad or pos_emb.device != x.device
                or pos_emb.shape != ((1, dim, t) if cf else (1, t, dim)) or not plain(linear_pos, linear) or linear_pos.bias is not None):
            return None
        projections.append(linear_pos)
    groups = {getattr(p, "groups", 1) for p in projections}
    params = [a.relative_position_bias if m.local else linear_pos.weight]
    for p in (*norms, *projections[:4]):
        params += p._parameters.get("weight"), p._parameters.get("bias")
    device = x.device
    if len(groups) != 1 or any(p is None or type(p) is not nn.Parameter or p.dtype != torch.float32 or p.device != device
                               or not p.is_contiguous() or p.data_ptr() % 16 for p in params):
        return None
    hidden, groups = params[9].shape[0], groups.pop()
    sizes = (3 * dim, dim, dim, dim, hidden, dim, dim, hidden)
    if any(p.numel() != o * i // groups for p, o, i in zip(params[5::2], sizes[::2], sizes[1::2])):
        return None
    if params[0].numel() != (a.num_heads * a.win_size if m.local else dim * dim // groups):
        return None
    window = (a.win_size, a.left, a.dilation) if m.local else (0, 0, 1)
    # The modules' products of a stream that lies channels first in memory (a model's, from the patch embedding on) round
    # before the bias is added, those of a tokens-first tensor after.  The node's own output lies tokens first either way.
    late = cf or not x.is_contiguous() or getattr(x.grad_fn, "late", 0)
    geom = (_lib.dtype_tag(x.dtype), dim, hidden, a.num_heads, *window, groups, int(cf), a.scale, int(late))
    probe = _Layer(*geom)
    if _lib.load().na1d_train_layer_saved_bytes(ctypes.byref(probe), n, t) < 0:
        return None
    by_channel = xt.detach().transpose(1, 2)
    by_channel = by_channel if by_channel.is_contiguous() else None       # [N, C, T], the layout of the statistics, is there already
    xt = xt.contiguous()
    if not m.local:
        pos = _aligned((pos_emb.transpose(1, 2) if cf else pos_emb).to(x.dtype))
    scales = (_drop_path_scale(parts.get("drop_path"), xt), _drop_path_scale(parts.get("drop_path"), xt))
    out = _TrainLayer.apply(xt, by_channel, geom, _lib.nodes() or _ByCtypes, norms, scales, pos, *params)
    return out.transpose(1, 2) if cf else out


# ---------------------------------------------------------------------------------------------- attentive pooling
def context_of(x, eps):
    """``[x, mean, std]`` over the last axis along the channels (Pooling.py:30-45), and the variance and deviation in it."""
    mean, var, std = _statistics(x, eps)
    return torch.cat([x, mean.expand_as(x), std.expand_as(x)], dim=1), var, std


def _statistics(x, eps):
    mean, var = x.mean(-1, keepdim=True), x.var(-1, keepdim=True)
    return mean, var, torch.sqrt(var.clamp(eps))


def pooled_of(logits, x, eps):
    """Mean and standard deviation over the last axis, weighted by the logits' softmax (Pooling.py:47-59)."""
    w = F.softmax(logits, dim=-1)
    mean = (w * x).sum(-1, keepdim=True)
    std = torch.sqrt((w * (x - mean).pow(2)).sum(-1, keepdim=True).clamp(eps))
    return torch.cat((mean, std), dim=1).squeeze(-1)


class _Pooling(torch.autograd.Function):
    """Torch's forward - training amplifies any difference in it - and a backward of one launch instead of some thirty."""

    @staticmethod
    def again(ctx, grad, f, *inputs):
        """The same backward by torch, for a caller that differentiates it again, whose gradient is no plain tensor, or whose
        hooks hand saved tensors back in another form.  It is taken by views of the inputs, each a node of its own: an input
        that was made from another one (the logits from x) would hand that its gradient here too, and so twice."""
        create_graph = torch.is_grad_enabled()
        with torch.enable_grad(), torch.autocast("cuda", dtype=ctx.dtype):
            views = [t.view_as(t) for t in inputs]
            leaves = [t for t, need in zip(views, ctx.needs_input_grad) if need]
            grads = iter(torch.autograd.grad(f(*views), leaves, grad, create_graph=create_graph))
        return tuple(next(grads) if need else None for need in ctx.needs_input_grad)


class _Context(_Pooling):
    @staticmethod
    def forward(ctx, x, eps):
        n, c, t = x.shape
        mean, var, std = _statistics(x, eps)
        if x.is_cuda and t >= 8 and c * t * t < 1 << 32 and _lie(x, x.dtype, (n, c, 1), mean, std):
            out = torch.empty((n, 3 * c, t), dtype=x.dtype, device=x.device)
            with torch.cuda.device(x.device):
                _lib.check(_lib.load().na1d_train_context(out.data_ptr(), x.data_ptr(), mean.data_ptr(), std.data_ptr(), n, c, t,
                                                          torch.cuda.current_stream().cuda_stream), "na1d_train_context")
        else:
            out = torch.cat([x, mean.expand_as(x), std.expand_as(x)], dim=1)
        ctx.save_for_backward(x, var, std)
        ctx.eps, ctx.dtype = eps, x.dtype
        return out

    @staticmethod
    def backward(ctx, dctx):
        x, var, std = ctx.saved_tensors
        n, c, t = x.shape
        if torch.is_grad_enabled() or not (plain_call(dctx) and dctx.shape == (n, 3 * c, t) and _rows_fit(ctx.dtype, x)
                                           and _lie(x, x.dtype, (n, c, 1), var, std)):
            return _Pooling.again(ctx, dctx, lambda x: context_of(x, ctx.eps)[0], x)
        dctx, dx = _aligned(dctx), torch.empty_like(x)
        with torch.cuda.device(x.device):
            _lib.check(_lib.load().na1d_train_context_backward(
                dx.data_ptr(), dctx.data_ptr(), x.data_ptr(), var.data_ptr(), std.data_ptr(), n, c, t,
                torch.tensor(ctx.eps, dtype=x.dtype).item(), _lib.dtype_tag(x.dtype), torch.cuda.current_stream().cuda_stream),
                "na1d_train_context_backward")
        return dx, None


class _Pooled(_Pooling):
    @staticmethod
    def forward(ctx, logits, x, eps):
        out = pooled_of(logits, x, eps)
        ctx.save_for_backward(logits, x, out)
        ctx.eps, ctx.dtype = eps, x.dtype
        return out.clone()                          # the caller may write to its own

    @staticmethod
    def backward(ctx, dout):
        logits, x, out = ctx.saved_tensors
        n, c, t = x.shape
        if torch.is_grad_enabled() or not (plain_call(dout) and dout.shape == (n, 2 * c) and _rows_fit(ctx.dtype, logits, x)
                                           and _lie(x, torch.float32, (n, 2 * c), out)):
            return _Pooling.again(ctx, dout, lambda z, x: pooled_of(z, x, ctx.eps), logits, x)
        dout, dz, dx = dout.contiguous(), torch.empty_like(logits), torch.empty_like(x)
        with torch.cuda.device(x.device):
            _lib.check(_lib.load().na1d_train_pool_backward(
                dz.data_ptr(), dx.data_ptr(), logits.data_ptr(), x.data_ptr(), out.data_ptr(), dout.data_ptr(), n, c, t, ctx.eps,
                _lib.dtype_tag(x.dtype), torch.cuda.current_stream().cuda_stream), "na1d_train_pool_backward")
        return dz, dx, None


def _lie(x, dtype, shape, *tensors):
    return all(t.device == x.device and t.dtype == dtype and t.shape == shape and t.is_contiguous() for t in tensors)


def _rows_fit(dtype, *tensors):
    """Whether the kernels take these [N, C, T] tensors."""
    x = tensors[-1]
    return (x.is_cuda and x.dim() == 3 and dtype in (torch.bfloat16, torch.float16)
            and _lie(x, dtype, x.shape, *tensors) and all(plain_call(t) and t.data_ptr() % 16 == 0 for t in tensors)
            and 0 < x.shape[0] <= 65535 and x.shape[1] % 8 == 0 and 8 <= x.shape[1] <= 1 << 16 and 2 <= x.shape[2] <= 2048
            and x.shape[0] * x.shape[1] < 1 << 31)


def _pooling_fits(eps, *tensors):
    return (isinstance(eps, (int, float)) and torch.is_grad_enabled() and any(t.requires_grad for t in tensors) and torch.is_autocast_enabled("cuda")
            and _rows_fit(torch.get_autocast_dtype("cuda"), *tensors))


def pooling_context(x, eps):
    """:func:`context_of` as one autograd node where the kernels take ``x``."""
    return _Context.apply(x, eps) if _pooling_fits(eps, x) else context_of(x, eps)[0]


def pooled(logits, x, eps):
    """:func:`pooled_of` as one autograd node where the kernels take its inputs."""
    return _Pooled.apply(logits, x, eps) if _pooling_fits(eps, logits, x) else pooled_of(logits, x, eps)
