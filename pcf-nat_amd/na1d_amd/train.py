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


def _ptr(t):
    return None if t is None else t.data_ptr()


def _ptrs(ts):
    return (_P * 5)(*map(_ptr, ts))


def _aligned(t):
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


class _TrainLayer(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, by_channel, geom, norms, scales, pos, extra, n1w, n1b, n2w, n2b, wq, bq, wp, bp, w1, b1, w2, b2):
        lib = _lib.load()
        n, t, dim = x.shape
        dense = pos is not None                     # extra: linear_pos' weight, or the bias of a window's scores
        weights, biases = (wq, wp, w1, w2, extra if dense else None), (bq, bp, b1, b2)
        c = _Layer(*geom)
        c.w, c.b = _ptrs(weights), _ptrs(biases)
        for to, bn, w, b in zip(c.norm, norms, (n1w, n2w), (n1b, n2b)):
            to.weight, to.bias, to.eps, to.batches = w.data_ptr(), b.data_ptr(), bn.eps, bn.num_batches_tracked.data_ptr()
        c.rpb, c.pos, c.scale_attn, c.scale_mlp = None if dense else extra.data_ptr(), _ptr(pos), _ptr(scales[0]), _ptr(scales[1])
        ref = ctypes.byref(c)
        out = torch.empty_like(x)
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
                stats = torch.batch_norm_update_stats(of, norms[part].running_mean, norms[part].running_var, norms[part].momentum)
                c.norm[part].batch_mean, c.norm[part].batch_var = map(_ptr, stats)
                _lib.check(lib.na1d_train_layer_forward(ref, part, to.data_ptr(), x.data_ptr(), saved.data_ptr(), sizes[0], ws.data_ptr(),
                                                        sizes[1], n, t, stream), "na1d_train_layer_forward")
        increment_version([b for bn in norms for b in (bn.running_mean, bn.running_var, bn.num_batches_tracked)])
        ctx.save_for_backward(x, saved, pos, None if dense else extra, n1w, n2w, *scales)
        ctx.late = c.late
        ctx.geom, ctx.shapes = geom, [p.shape for p in (extra, n1w, n1b, n2w, n2b, wq, bq, wp, bp, w1, b1, w2, b2)]
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, dout):
        lib = _lib.load()
        x, saved, pos, rpb, n1w, n2w, *scales = ctx.saved_tensors
        n, t, dim = x.shape
        dout = _aligned(dout)
        dx = torch.empty_like(x)
        grads = [torch.zeros(ctx.shapes[0], dtype=torch.float32, device=x.device)]       # the bias of the scores is added to
        grads += [torch.empty(s, dtype=torch.float32, device=x.device) for s in ctx.shapes[1:]]
        c = _Layer(*ctx.geom)
        c.dw, c.db = _ptrs(grads[5::2] + ([] if pos is None else grads[:1])), _ptrs(grads[6::2])
        for to, w, dw, db in zip(c.norm, (n1w, n2w), grads[1:5:2], grads[2:5:2]):
            to.weight, to.dweight, to.dbias = w.data_ptr(), dw.data_ptr(), db.data_ptr()
        c.rpb, c.drpb, c.pos, c.scale_attn, c.scale_mlp = _ptr(rpb), grads[0].data_ptr(), _ptr(pos), _ptr(scales[0]), _ptr(scales[1])
        ref = ctypes.byref(c)
        with torch.cuda.device(x.device):
            nbytes = lib.na1d_train_layer_workspace_bytes(ref, n, t, 1)
            _lib.check(min(nbytes, 0), "na1d_train_layer_workspace_bytes")
            ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
            _lib.check(lib.na1d_train_layer_backward(ref, dx.data_ptr(), dout.data_ptr(), x.data_ptr(), saved.data_ptr(), saved.numel(),
                                                     ws.data_ptr(), nbytes, n, t, torch.cuda.current_stream().cuda_stream),
                       "na1d_train_layer_backward")
        return (dx, None, None, None, None, None, *(g if need else None for g, need in zip(grads, ctx.needs_input_grad[6:])))


def plain(m, *classes):
    """Whether calling module ``m`` runs the forward of its class and nothing else."""
    return (type(m) in classes and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks)
            and "forward" not in m.__dict__)


def plain_call(x):
    """Whether nothing but autograd looks at the operations on ``x``: no tracer, transform, subclass or dispatch mode."""
    return (type(x) in (torch.Tensor, nn.Parameter) and not torch.compiler.is_compiling() and not torch.jit.is_tracing()
            and not torch.nn.modules.module._has_any_global_hook() and torch._C._functorch.peek_interpreter_stack() is None
            and torch.autograd.forward_ad._current_level < 0 and torch._C._len_torch_dispatch_stack() == 0
            and not torch._C._functorch.is_legacy_batchedtensor(x))       # of is_grads_batched


def _norm_fits(bn, dim, device):
    return (bn.training and bn.track_running_stats and bn.affine and bn.momentum is not None and bn.num_features == dim
            and all(s is not None and s.dtype == torch.float32 and s.device == device and s.shape == (dim,) for s in (bn.running_mean, bn.running_var))
            and bn.num_batches_tracked is not None and bn.num_batches_tracked.dtype == torch.int64 and bn.num_batches_tracked.device == device)


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
    a, mlp = m.attn, m.mlp
    cf = getattr(a, "channels_first", False)
    linear, norm = (M.Conv1x1, M.BatchNorm1d) if cf else (M.TokenLinear, M.TokenBatchNorm)
    if not (plain_call(x) and plain(a, M.NAttention if m.local else M.GlobalAttention) and plain(mlp, M.Mlp) and plain(m.norm1, norm) and plain(m.norm2, norm)
            and plain(m.drop_path, nn.Identity, M.DropPath) and plain(mlp.act, nn.GELU) and mlp.act.approximate == "none"
            and plain(mlp.drop, nn.Dropout) and plain(a.proj_drop, nn.Dropout)
            and all(plain(p, linear) for p in (a.qkv, a.proj, mlp.fc1, mlp.fc2))):
        return None
    norms = (m.norm1, m.norm2) if cf else (m.norm1.norm, m.norm2.norm)
    if (a.na != "fused_qkv" if m.local else a.dense != "native") or a.attn_drop or not a.training or a.proj_drop.p or mlp.drop.p or (not cf and not all(plain(b, M.BatchNorm1d) for b in norms)):
        return None
    xt = x.transpose(1, 2) if cf else x
    if xt.is_contiguous() and xt.data_ptr() % 16:
        return None
    n, t, dim = xt.shape
    if (t != a.attn_mask.shape[-2] if m.local else attn_mask_global is not None) or not all(_norm_fits(b, dim, x.device) for b in norms):
        return None
    projections = [a.qkv, a.proj, mlp.fc1, mlp.fc2]
    pos = None
    if not m.local:
        if (pos_emb is None or type(pos_emb) is not torch.Tensor or pos_emb.requires_grad or pos_emb.device != x.device
                or pos_emb.shape != ((1, dim, t) if cf else (1, t, dim)) or not plain(a.linear_pos, linear) or a.linear_pos.bias is not None):
            return None
        projections.append(a.linear_pos)
    groups = {getattr(p, "groups", 1) for p in projections}
    params = (a.relative_position_bias if m.local else a.linear_pos.weight, norms[0].weight, norms[0].bias, norms[1].weight, norms[1].bias, a.qkv.weight, a.qkv.bias,
              a.proj.weight, a.proj.bias, mlp.fc1.weight, mlp.fc1.bias, mlp.fc2.weight, mlp.fc2.bias)
    hidden = mlp.fc1.weight.shape[0]
    sizes = (3 * dim, dim, dim, dim, hidden, dim, dim, hidden)
    if len(groups) != 1 or any(p is None or type(p) is not nn.Parameter or p.dtype != torch.float32 or p.device != x.device
                               or not p.is_contiguous() or p.data_ptr() % 16 for p in params):
        return None
    groups = groups.pop()
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
    scales = (_drop_path_scale(m.drop_path, xt), _drop_path_scale(m.drop_path, xt))
    out = _TrainLayer.apply(xt, by_channel, geom, norms, scales, pos, *params)
    return out.transpose(1, 2) if cf else out


# ---------------------------------------------------------------------------------------------- attentive pooling
def context_of(x, eps):
    """``[x, mean, std]`` over the last axis along the channels (Pooling.py:30-45), and the variance and deviation in it."""
    mean, var = x.mean(-1, keepdim=True), x.var(-1, keepdim=True)
    std = torch.sqrt(var.clamp(eps))
    return torch.cat([x, mean.expand_as(x), std.expand_as(x)], dim=1), var, std


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
        out, var, std = context_of(x, eps)
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
