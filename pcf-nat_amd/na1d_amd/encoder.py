"""A whole embedding model in inference as one library call (``na1d_encode`` of the C ABI).

:func:`embed` runs the models of ``models.py`` through the token-local kernels of ``csrc/na1d_encoder.hip`` and the
attention kernels, launched back to back from native code.  Its plan holds the weights in the kernels' order with the
batch norms folded into them; what is made of a parameter or running statistic is made again when it changes (torch counts
the versions of a tensor; writes through ``.data`` are seen in the last layer, the pooled norm, dense layers' first norms and
the biases of scores and outputs, which the kernels read from the modules).
"""
from __future__ import annotations

import ctypes
import weakref
from operator import is_

import torch
import torch.nn as nn

from . import _lib
from .train import plain, plain_call

_P, _I, _F = ctypes.c_void_p, ctypes.c_int32, ctypes.c_float
DIM, HIDDEN, POOL_HIDDEN = 256, 1024, 128          # channels the kernels are built for


class _Norm(ctypes.Structure):                     # na1d_encoder_norm
    _fields_ = [(n, _P) for n in "weight bias mean var".split()] + [("eps", _F)]


class _Layer(ctypes.Structure):                    # na1d_encoder_layer
    _fields_ = ([(n, _I) for n in "heads window left dilation groups embeds block_end".split()] + [("scale", _F)]
                + [(n, _P) for n in ("w_qkv w_proj w_fc1 w_fc2 b_qkv b_proj b_fc1 b_fc2 rpb w_embed b_embed "
                                     "w_pos").split()] + [("norm", _Norm)])


class _Encoder(ctypes.Structure):                  # na1d_encoder
    _fields_ = ([(n, _I) for n in "dtype layers blocks in_chans patch wide emb".split()]
                + [("layer", ctypes.POINTER(_Layer)), ("pos", _P), ("pos_rows", ctypes.c_int64)]
                + [(n, _P) for n in ("w_wide b_wide a_wide c_wide w_att w_ctx w_logit b_att a_att c_att").split()]
                + [("pool_norm", _Norm), ("w_fc", _P), ("b_fc", _P)])


def fragment_order(w, dtype):
    """``[outputs, inputs]`` -> the kernels' order: blocks of 16 outputs x 32 inputs, lane by lane (na1d.h)."""
    o, i = w.shape
    return w.to(dtype).view(o // 16, 16, i // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()


def _stamps(tensors):
    return [(t, t._version, t.data_ptr()) for t in tensors if t is not None]


def _same(a, b):
    return len(a) == len(b) and all(x[0] is y[0] and x[1] == y[1] and x[2] == y[2] for x, y in zip(a, b))


class _Plan:
    """The C structures of one model in one dtype, and the tensors they point into.  What is derived from tensors that are
    as they were for the plan `before` is taken over from there: a changed tensor costs what was made of it."""

    def __init__(self, model, dtype, before=None):
        from . import models as M
        self.dtype, self.keep = dtype, []
        self.made = {}                              # name -> (stamps of its sources, tensors made of them)
        self.streams = set()                        # that have been told to the tensors' allocator
        known = {} if before is None else before.made

        def derive(name, sources, build):
            now = _stamps(sources)
            have = known.get(name)
            if have is None or not _same(have[0], now):
                have = (now, build())
            self.made[name] = have
            return (t.data_ptr() for t in have[1])

        def matrices(name, sources, build):         # build() -> weights [outputs, inputs]
            return derive(name, sources, lambda: [fragment_order(w.detach(), dtype) for w in build()])

        def product(name, sources, build):          # build() -> a weight and its bias
            def both():
                w, b = build()
                return fragment_order(w.detach(), dtype), b.detach().float().contiguous()
            return derive(name, sources, both)

        def affine(name, bn):
            return derive(name, M._bn_tensors(bn), lambda: [v.detach().contiguous() for v in M._bn_affine(bn)])

        def own(p):                                 # a parameter itself
            self.keep.append(p.detach())
            return p.data_ptr()

        def norm(bn):                               # a norm's own tensors
            return _Norm(*map(own, M._bn_tensors(bn)), bn.eps)

        flat = [(block, i, layer) for block in model.blocks for i, layer in enumerate(block.blocks)]
        self.layers = (_Layer * len(flat))()
        for at, (l, (block, i, layer)) in enumerate(zip(self.layers, flat)):
            attn, mlp, cf = layer.attn, layer.mlp, layer.attn.channels_first
            bn = [n.norm if isinstance(n, M.TokenBatchNorm) else n for n in (layer.norm1, layer.norm2)]
            order = (lambda: M._qkv_channel_order(DIM, attn.groups, attn.qkv.weight.device)) if cf else lambda: None
            groups = {getattr(p, "groups", 1) for p in (attn.qkv, attn.proj, mlp.fc1, mlp.fc2)}
            l.groups = groups.pop() if len(groups) == 1 else 1
            l.heads, l.scale = attn.num_heads, attn.scale
            l.block_end = i == len(block.blocks) - 1
            qkv = [attn.qkv.weight, attn.qkv.bias]
            if layer.local:
                l.window, l.left, l.dilation = attn.win_size, attn.left, attn.dilation
                l.rpb = own(attn.relative_position_bias)
                l.w_qkv, l.b_qkv = product((at, "qkv"), qkv + M._bn_tensors(bn[0]), lambda: M._fold_norm(bn[0], attn.qkv, order()))
            else:
                l.dilation = 1
                l.norm, (l.w_pos,) = norm(bn[0]), matrices((at, "pos"), [attn.linear_pos.weight], lambda: [M._dense_weight(attn.linear_pos)])
                def reordered():
                    w, b = M._dense_weight(attn.qkv), attn.qkv.bias
                    return (w.index_select(0, order()), b.index_select(0, order())) if cf else (w, b)
                l.w_qkv, l.b_qkv = product((at, "qkv"), qkv, reordered)
            (l.w_proj,), l.b_proj = matrices((at, "proj"), [attn.proj.weight], lambda: [M._dense_weight(attn.proj)]), own(attn.proj.bias)
            l.w_fc1, l.b_fc1 = product((at, "fc1"), [mlp.fc1.weight, mlp.fc1.bias] + M._bn_tensors(bn[1]), lambda: M._fold_norm(bn[1], mlp.fc1))
            (l.w_fc2,), l.b_fc2 = matrices((at, "fc2"), [mlp.fc2.weight], lambda: [M._dense_weight(mlp.fc2)]), own(mlp.fc2.bias)
            if i == 0 and (model.channels_first or at == 0):
                embed = model.patch_embeds[list(model.blocks).index(block)] if model.channels_first else model.patch_embed
                conv = embed.proj
                def patches():
                    w = conv.weight.reshape(conv.out_channels, -1).float()
                    if conv.groups > 1:
                        w = torch.block_diag(*w.view(conv.groups, conv.out_channels // conv.groups, -1))
                    a, b = M._bn_affine(embed.norm)
                    return w * a.unsqueeze(1), conv.bias.float() * a + b
                l.embeds = 1
                l.w_embed, l.b_embed = product((at, "embed"), [conv.weight, conv.bias] + M._bn_tensors(embed.norm), patches)
        e = self.encoder = _Encoder()
        conv, device = (model.patch_embeds[0] if model.channels_first else model.patch_embed).proj, model.fc.weight.device
        wide = model.proj.conv.out_channels
        e.dtype, e.layers, e.blocks, e.layer = _lib.dtype_tag(dtype), len(flat), len(model.blocks), self.layers
        e.in_chans, e.patch, e.wide, e.emb = conv.in_channels, model.patch_size, wide, model.fc.out_features
        if model.attn_global:
            table = model.eval_positions(device)
            (e.pos,) = derive("positions", [] if table.is_inference() else [table], lambda: [(table[0].t() if model.channels_first else table[0]).to(dtype).contiguous()])
            e.pos_rows = table.shape[2 if model.channels_first else 1]
        w = model.proj.conv
        e.w_wide, e.b_wide = product("wide", [w.weight, w.bias] + M._bn_tensors(model.norm), lambda: M._fold_norm(model.norm, w))
        e.a_wide, e.c_wide = affine("wide norm", model.proj.norm)
        tdnn, logit = model.pool.tdnn, model.pool.conv
        e.w_att, e.w_ctx = matrices("pooling", [tdnn.conv.weight], lambda: M._dense_weight(tdnn.conv).split([wide, 2 * wide], 1))
        e.b_att, (e.a_att, e.c_att) = own(tdnn.conv.bias), affine("pooling norm", tdnn.norm)
        (e.w_logit,) = matrices("logits", [logit.weight], lambda: [M._dense_weight(logit)])
        if not isinstance(model.pool_norm, nn.Identity):
            e.pool_norm = norm(model.pool_norm)
        e.w_fc, e.b_fc = own(model.fc.weight), own(model.fc.bias)


    def use_on(self, stream):
        """A plan that is replaced gives its memory back, also while another stream than the one that made it still reads."""
        if stream.cuda_stream not in self.streams:
            for _, tensors in self.made.values():
                for t in tensors:
                    t.record_stream(stream)
            self.streams.add(stream.cuda_stream)


# The modules' numbers that a plan is made of.
_NUMBERS = ("channels_first", "embed_dim", "patch_size", "attn_global", "local", "num_heads", "scale", "groups", "win_size", "left", "dilation",
            "eps")


class _Entry:
    """What is kept for a model: where its tensors are found, and the plans made of their present values."""

    def __init__(self, model):
        mods = [m for m in model.modules() if m is not model]             # nothing here may keep the model itself
        self.mods, self.kinds = mods, list(map(type, mods))
        self.children = [m._modules for m in [model] + mods]
        self.present = [list(d.values()) for d in self.children]
        self.methods = [m.__dict__ for m in mods if hasattr(m, "forward_tokens")]
        self.parameters = [m._parameters for m in mods if m._parameters]
        self.statistics = [m._buffers for m in mods if "running_mean" in m._buffers]
        self.numbers = [(m.__dict__, n) for m in [model] + mods if not isinstance(m, nn.Conv1d)
                        for n in _NUMBERS if n in m.__dict__]
        self.attn = [layer.attn for block in model.blocks for layer in block.blocks] if hasattr(model, "blocks") else []
        self.plans = {}                             # (dtype, device) -> (state, plan or None)

    def same_modules(self):
        return ([list(d.values()) for d in self.children] == self.present and list(map(type, self.mods)) == self.kinds
                and not any("forward_tokens" in d for d in self.methods))

    def state(self):
        """Everything that a plan is made of, as it is now."""
        tensors = [t for d in self.parameters for t in d.values()]
        tensors += [d.get(n) for d in self.statistics for n in ("running_mean", "running_var")]
        tensors = [t for t in tensors if t is not None]
        return tensors, [t._version for t in tensors], [t.data_ptr() for t in tensors], [d.get(n) for d, n in self.numbers]

    def plan(self, model, dtype, device):
        now = self.state()
        before, plan = self.plans.get((dtype, device), (None, None))
        if before is not None and now[1:] == before[1:] and len(now[0]) == len(before[0]) and all(map(is_, now[0], before[0])):
            return plan
        if torch.cuda.is_current_stream_capturing():          # it would record the preparation, not do it
            return None
        plan = _Plan(model, dtype, plan if before is not None and now[3] == before[3] else None) if _fits(model, device) else None
        torch.cuda.current_stream().synchronize()             # the next call may come on another stream
        self.plans[dtype, device] = (now, plan)
        return plan


_entries = weakref.WeakKeyDictionary()              # model -> _Entry


def _own(m, *classes):
    """Whether module ``m`` is of these classes, with their way through tokens and no other."""
    return type(m) in classes and "forward_tokens" not in m.__dict__


def _as_built(model):
    """Whether the model's pass over tokens is the one that the kernels compute."""
    from .models import _NATransformer as base
    return all(getattr(type(model), n) is getattr(base, n) and n not in model.__dict__ for n in ("_forward_tokens", "_tokens_path"))


def _fits(model, device):
    """Whether the kernels compute what the modules would: their own classes, at the sizes of the published models (those
    the kernels are built for), with parameters of their own in fp32 on the input's device."""
    from . import models as M
    def held(t, *shape):
        return t is not None and t.dtype == torch.float32 and t.device == device and t.shape == shape and t.is_contiguous()

    def norm(bn, channels):
        return (_own(bn, M.BatchNorm1d) and all(held(bn._parameters.get(n), channels) for n in ("weight", "bias"))
                and all(held(bn._buffers.get(n), channels) for n in ("running_mean", "running_var")))

    def projection(p, outputs, inputs, kernel=(), bias=True):
        """`kernel`: () for a linear layer, else the length of a convolution's."""
        if not _own(p, *((M.PatchConv, M.Conv1x1) if kernel else (M.TokenLinear, nn.Linear))):
            return False
        groups = p.groups if kernel else 1
        return (outputs % groups == 0 and inputs % groups == 0 and held(p._parameters.get("weight"), outputs, inputs // groups, *kernel)
                and (held(p._parameters.get("bias"), outputs) if bias else p._parameters.get("bias") is None))

    cf = model.channels_first
    token = (1,) if cf else ()
    if model.embed_dim != DIM or not all(_own(block, M.NATFBlock) for block in model.blocks):
        return False
    for layer in (layer for block in model.blocks for layer in block.blocks):
        if not (_own(layer, M.NATFLayer) and _own(layer.attn, M.NAttention if layer.local else M.GlobalAttention) and _own(layer.mlp, M.Mlp)):
            return False
        a, mlp, norms = layer.attn, layer.mlp, (layer.norm1, layer.norm2)
        if not cf:
            if not all(_own(n, M.TokenBatchNorm) for n in norms):
                return False
            norms = tuple(n.norm for n in norms)
        if not (a.channels_first == cf and a.num_heads >= 1 and DIM % (8 * a.num_heads) == 0 and DIM // a.num_heads <= 128
                and all(norm(n, DIM) for n in norms) and projection(a.qkv, 3 * DIM, DIM, token) and projection(a.proj, DIM, DIM, token)
                and projection(mlp.fc1, HIDDEN, DIM, token) and projection(mlp.fc2, DIM, HIDDEN, token)):
            return False
        if not (held(a._parameters.get("relative_position_bias"), 1, a.num_heads, 1, a.win_size) if layer.local
                else projection(a.linear_pos, DIM, DIM, token, bias=False)):
            return False
    embeds = list(model.patch_embeds) if cf else [model.patch_embed]
    if len(embeds) != (len(model.blocks) if cf else 1) or not all(_own(e, M.PatchEmbed) and norm(e.norm, DIM) for e in embeds):
        return False
    chans, patch = embeds[0].proj.in_channels, model.patch_size
    if chans * patch % 32 or chans * patch > DIM or not all(projection(e.proj, DIM, chans, (patch,)) for e in embeds):
        return False
    pool, wide = model.pool, model.proj.conv.out_channels
    if not (wide % 256 == 0 and norm(model.norm, DIM * len(model.blocks)) and _own(model.proj, M.TDNNBlock)
            and projection(model.proj.conv, wide, DIM * len(model.blocks), (1,)) and norm(model.proj.norm, wide)):
        return False
    if not (_own(pool, M.AttentiveStatisticsPooling) and pool.eps == 1e-12 and _own(pool.tdnn, M.TDNNBlock)
            and projection(pool.tdnn.conv, POOL_HIDDEN, 3 * wide, (1,)) and norm(pool.tdnn.norm, POOL_HIDDEN)
            and projection(pool.conv, wide, POOL_HIDDEN, (1,))):
        return False
    if not (type(model.pool_norm) is nn.Identity or norm(model.pool_norm, 2 * wide)):
        return False
    return type(model.fc) is nn.Linear and model.fc.out_features % 16 == 0 and projection(model.fc, model.fc.out_features, 2 * wide)


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
    if not _as_built(model) or model.pool_norm.training:
        return None
    dtype = torch.get_autocast_dtype("cuda")
    if dtype not in (torch.bfloat16, torch.float16) or x.dim() != 3 or x.dtype not in (torch.float32, torch.bfloat16, torch.float16):
        return None
    if lens is not None and (lens.dtype != torch.float32 or lens.device != x.device or lens.shape != (x.shape[0],)):
        return None
    if torch.cuda.current_device() != x.device.index:      # plans are made, and launches go, where the tensors are
        with torch.cuda.device(x.device):
            return embed(model, x, lens)
    entry = _entries.get(model)
    if entry is None or not entry.same_modules():
        entry = _entries[model] = _Entry(model)
    if any((a.na != "fused_qkv") if hasattr(a, "na") else (a.dense != "native") for a in entry.attn):
        return None
    plan = entry.plan(model, dtype, x.device)
    n, chans, frames = x.shape
    if plan is None or chans != plan.encoder.in_chans:
        return None
    lib = _lib.load()
    ref = ctypes.byref(plan.encoder)
    nbytes = lib.na1d_encode_workspace_bytes(ref, n, frames)
    if nbytes == _lib.UNSUPPORTED:
        return None
    _lib.check(min(nbytes, 0), "na1d_encode_workspace_bytes")
    stream = torch.cuda.current_stream(x.device)
    plan.use_on(stream)
    x, lens = x.float().contiguous(), None if lens is None else lens.contiguous()
    out = torch.empty((n, plan.encoder.emb), dtype=dtype, device=x.device)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    st = lib.na1d_encode(ref, out.data_ptr(), x.data_ptr(), None if lens is None else lens.data_ptr(), n, frames,
                         ws.data_ptr(), nbytes, stream.cuda_stream)
    if st == _lib.UNSUPPORTED:
        return None
    _lib.check(st, "na1d_encode")
    return out
