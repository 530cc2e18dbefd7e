"""A whole embedding model in inference as one library call (``na1d_encode`` of the C ABI).

:func:`embed` runs the models of ``models.py`` through the token-local kernels of ``csrc/na1d_encoder.hip`` and the
attention kernels, launched back to back from native code.  Its plan holds the weights in the kernels' order with the
batch norms folded into them; it is rebuilt when a parameter or a running statistic changes.
"""
from __future__ import annotations

import ctypes
import weakref

import torch
import torch.nn as nn

from . import _lib
from .train import plain, plain_call

_P, _I, _F = ctypes.c_void_p, ctypes.c_int32, ctypes.c_float
DIM, HIDDEN, POOL_HIDDEN = 256, 1024, 128          # channels the kernels are built for


class _Layer(ctypes.Structure):                    # na1d_encoder_layer
    _fields_ = ([(n, _I) for n in "heads window left dilation groups embeds block_end".split()] + [("scale", _F)]
                + [(n, _P) for n in ("w_qkv w_proj w_fc1 w_fc2 b_qkv b_proj b_fc1 b_fc2 rpb w_embed b_embed w_pos gain "
                                     "shift").split()])


class _Encoder(ctypes.Structure):                  # na1d_encoder
    _fields_ = ([(n, _I) for n in "dtype layers blocks in_chans patch wide emb".split()]
                + [("layer", ctypes.POINTER(_Layer)), ("pos", _P), ("pos_rows", ctypes.c_int64)]
                + [(n, _P) for n in ("w_wide b_wide a_wide c_wide w_att w_ctx w_logit b_att a_att c_att a_pool c_pool w_fc "
                                     "b_fc").split()])


def fragment_order(w, dtype):
    """``[outputs, inputs]`` -> the kernels' order: blocks of 16 outputs x 32 inputs, lane by lane (na1d.h)."""
    o, i = w.shape
    return w.to(dtype).view(o // 16, 16, i // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()


class _Plan:
    """The C structures of one model in one dtype, and the tensors they point into."""

    def __init__(self, model, dtype):
        from . import models as M
        self.keep = []
        self.dtype = dtype

        def matrix(w):
            return self._hold(fragment_order(w.detach(), dtype))

        def vector(v):
            return self._hold(v.detach().float().contiguous())

        flat = [(block, i, layer) for block in model.blocks for i, layer in enumerate(block.blocks)]
        self.layers = (_Layer * len(flat))()
        for at, (l, (block, i, layer)) in enumerate(zip(self.layers, flat)):
            attn, dim, cf = layer.attn, DIM, layer.attn.channels_first
            bn = [n.norm if isinstance(n, M.TokenBatchNorm) else n for n in (layer.norm1, layer.norm2)]
            order = M._qkv_channel_order(dim, attn.groups, bn[0].weight.device) if cf else None
            projections = (attn.qkv, attn.proj, layer.mlp.fc1, layer.mlp.fc2)
            groups = {getattr(p, "groups", 1) for p in projections}
            l.groups = groups.pop() if len(groups) == 1 else 1
            l.heads, l.scale = attn.num_heads, attn.scale
            l.block_end = i == len(block.blocks) - 1
            if layer.local:
                l.window, l.left, l.dilation = attn.win_size, attn.left, attn.dilation
                l.rpb = vector(attn.relative_position_bias.reshape(attn.num_heads, attn.win_size))
                wq, bq = M._fold_norm(bn[0], attn.qkv, order)
            else:
                l.dilation = 1
                wq, bq = M._dense_weight(attn.qkv), attn.qkv.bias
                if order is not None:
                    wq, bq = wq.index_select(0, order), bq.index_select(0, order)
                gain, shift = M._bn_affine(bn[0])
                l.gain, l.shift, l.w_pos = vector(gain), vector(shift), matrix(M._dense_weight(attn.linear_pos))
            l.w_qkv, l.b_qkv = matrix(wq), vector(bq)
            l.w_proj, l.b_proj = matrix(M._dense_weight(attn.proj)), vector(attn.proj.bias)
            w1, b1 = M._fold_norm(bn[1], layer.mlp.fc1)
            l.w_fc1, l.b_fc1 = matrix(w1), vector(b1)
            l.w_fc2, l.b_fc2 = matrix(M._dense_weight(layer.mlp.fc2)), vector(layer.mlp.fc2.bias)
            if i == 0 and (model.channels_first or at == 0):
                embed = model.patch_embeds[list(model.blocks).index(block)] if model.channels_first else model.patch_embed
                conv = embed.proj
                w = conv.weight.reshape(conv.out_channels, -1).float()
                if conv.groups > 1:
                    w = torch.block_diag(*w.view(conv.groups, conv.out_channels // conv.groups, -1))
                a, b = M._bn_affine(embed.norm)
                l.embeds, l.w_embed, l.b_embed = 1, matrix(w * a.unsqueeze(1)), vector(conv.bias.float() * a + b)
        e = self.encoder = _Encoder()
        conv = (model.patch_embeds[0] if model.channels_first else model.patch_embed).proj
        wide = model.proj.conv.out_channels
        e.dtype, e.layers, e.blocks, e.layer = _lib.dtype_tag(dtype), len(flat), len(model.blocks), self.layers
        e.in_chans, e.patch, e.wide, e.emb = conv.in_channels, model.patch_size, wide, model.fc.out_features
        if model.attn_global:
            pos = M.sinusoid_table(DIM, 40000, False)[0].to(conv.weight.device)
            e.pos, e.pos_rows = self._hold(pos.to(dtype).contiguous()), pos.shape[0]
        w, b = M._fold_norm(model.norm, model.proj.conv)
        a, c = M._bn_affine(model.proj.norm)
        e.w_wide, e.b_wide, e.a_wide, e.c_wide = matrix(w), vector(b), vector(a), vector(c)
        tdnn = model.pool.tdnn
        w, (a, c) = M._dense_weight(tdnn.conv), M._bn_affine(tdnn.norm)
        e.w_att, e.w_ctx, e.b_att = matrix(w[:, :wide]), matrix(w[:, wide:]), vector(tdnn.conv.bias)
        e.a_att, e.c_att, e.w_logit = vector(a), vector(c), matrix(M._dense_weight(model.pool.conv))
        if isinstance(model.pool_norm, nn.Identity):
            a, c = torch.ones(2 * wide, device=w.device), torch.zeros(2 * wide, device=w.device)
        else:
            a, c = M._bn_affine(model.pool_norm)
        e.a_pool, e.c_pool, e.w_fc, e.b_fc = vector(a), vector(c), matrix(model.fc.weight), vector(model.fc.bias)

    def _hold(self, t):
        self.keep.append(t)
        return t.data_ptr()


class _Entry:
    """What is kept for a model: where its tensors are found, and the plans made of their present values."""

    def __init__(self, model):
        mods = list(model.modules())
        self.children = [(m._modules, list(m._modules.values())) for m in mods if m._modules]
        self.tensors = [d for m in mods for d in (m._parameters, m._buffers) if d]
        self.attn = [layer.attn for block in model.blocks for layer in block.blocks] if hasattr(model, "blocks") else []
        self.plans = {}                             # dtype -> (state of the tensors, plan or None)

    def same_modules(self):
        return all(len(d) == len(c) and all(a is b for a, b in zip(d.values(), c)) for d, c in self.children)

    def plan(self, model, dtype):
        state = [(t, t._version, t.data_ptr()) for d in self.tensors for t in d.values() if t is not None]
        have = self.plans.get(dtype)
        if have is not None and len(have[0]) == len(state) and all(
                a[0] is b[0] and a[1] == b[1] and a[2] == b[2] for a, b in zip(have[0], state)):
            return have[1]
        if torch.cuda.is_current_stream_capturing():          # it would record the preparation, not do it
            return None
        plan = _Plan(model, dtype) if _fits(model) else None
        torch.cuda.current_stream().synchronize()             # the next call may come on another stream
        self.plans[dtype] = (state, plan)
        return plan


_entries = weakref.WeakKeyDictionary()              # model -> _Entry


def _fits(model):
    """Whether the kernels cover the model's sizes (they are built for the sizes of the published models)."""
    from . import models as M
    layers = [layer for block in model.blocks for layer in block.blocks]
    conv = (model.patch_embeds[0] if model.channels_first else model.patch_embed).proj
    return (model.embed_dim == DIM and type(model.pool) is M.AttentiveStatisticsPooling
            and type(model.fc) is nn.Linear and model.fc.bias is not None and model.fc.in_features == 2 * model.proj.conv.out_channels
            and (type(model.pool_norm) is nn.Identity or type(model.pool_norm) is M.BatchNorm1d and model.pool_norm.affine
                 and model.pool_norm.running_mean is not None)
            and all(layer.mlp.fc1.weight.shape[0] == HIDDEN for layer in layers)
            and model.pool.tdnn.conv.out_channels == POOL_HIDDEN and model.proj.conv.out_channels % 256 == 0
            and model.fc.out_features % 16 == 0 and conv.in_channels * model.patch_size % 32 == 0
            and conv.in_channels * model.patch_size <= DIM
            and all(layer.attn.num_heads and DIM % (8 * layer.attn.num_heads) == 0 and DIM // layer.attn.num_heads <= 128
                    for layer in layers)
            and all(p.dtype == torch.float32 for p in model.parameters()))


def plans_of(model):
    """The plans a captured graph of this model reads from (whoever keeps such a graph keeps them too)."""
    entry = _entries.get(model)
    return [] if entry is None else [plan for _, plan in entry.plans.values() if plan is not None]


def embed(model, x, lens=None):
    """``[N, emb]`` embeddings of ``x [N, in_chans, frames]`` under autocast without gradients, or ``None`` where the
    kernels do not cover the model, its inputs or the mode: the caller then takes another path."""
    if model.training or not x.is_cuda or torch.is_grad_enabled() or not torch.is_autocast_enabled("cuda") or not plain_call(x):
        return None
    if getattr(model, "_is_replica", False):        # of DataParallel: lives for one call and holds plain tensors, no parameters
        return None
    if not all(plain(m, type(m)) for m in (model.pool_norm, model.fc)):
        return None                                 # called as modules otherwise: whatever hangs on them has to see the call
    dtype = torch.get_autocast_dtype("cuda")
    if dtype not in (torch.bfloat16, torch.float16) or x.dim() != 3 or x.dtype not in (torch.float32, torch.bfloat16, torch.float16):
        return None
    if lens is not None and (lens.dtype != torch.float32 or lens.device != x.device or lens.shape != (x.shape[0],)):
        return None
    if next(model.parameters()).device != x.device:
        return None
    if torch.cuda.current_device() != x.device.index:      # plans are made, and launches go, where the tensors are
        with torch.cuda.device(x.device):
            return embed(model, x, lens)
    entry = _entries.get(model)
    if entry is None or not entry.same_modules():
        entry = _entries[model] = _Entry(model)
    if any((a.na != "fused_qkv") if hasattr(a, "na") else (a.dense != "native") for a in entry.attn):
        return None
    plan = entry.plan(model, dtype)
    n, chans, frames = x.shape
    if plan is None or chans != plan.encoder.in_chans or plan.keep[0].device != x.device:
        return None
    lib = _lib.load()
    ref = ctypes.byref(plan.encoder)
    nbytes = lib.na1d_encode_workspace_bytes(ref, n, frames)
    if nbytes == _lib.UNSUPPORTED:
        return None
    _lib.check(min(nbytes, 0), "na1d_encode_workspace_bytes")
    x = x.float().contiguous()
    out = torch.empty((n, plan.encoder.emb), dtype=dtype, device=x.device)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    st = lib.na1d_encode(ref, out.data_ptr(), x.data_ptr(), None if lens is None else lens.contiguous().data_ptr(), n, frames,
                         ws.data_ptr(), nbytes, torch.cuda.current_stream(x.device).cuda_stream)
    if st == _lib.UNSUPPORTED:
        return None
    _lib.check(st, "na1d_encode")
    return out
