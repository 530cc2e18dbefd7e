"""Which models the native embedding call takes: decided on the host, so checked without a GPU."""
import copy
import ctypes
import gc
import os
import re
import types
import weakref

import pytest
import torch
import torch.nn as nn
import torch.nn.utils.parametrize  # noqa: F401

from na1d_amd import _lib, encoder, models

CPU = torch.device("cpu")
SMALL = dict(depths=(1, 1), num_heads=[[16], [4]], win_size=[[27], [0]], na="fused_qkv")


def _model(family="pcf", **kw):
    torch.manual_seed(0)
    kw = dict(SMALL, **kw)
    return (models.PCF_NATransformer(groups=(8, 4), **kw) if family == "pcf" else models.MFA_NATransformer(**kw)).eval()


def _subclass(cls, **methods):
    return type("Sub" + cls.__name__, (cls,), methods)


def _reclass(m, **methods):
    m.__class__ = _subclass(type(m), **methods)


def _weight_norm(m):
    """What torch.nn.utils.weight_norm leaves: the weight is a plain attribute that a hook works out."""
    w = m.weight.detach()
    del m._parameters["weight"]
    m.weight = w


CHANGES = {
    "layer of another class": lambda m: _reclass(m.blocks[0].blocks[0], forward_tokens=lambda self, x, *a: x),
    "block of another class": lambda m: _reclass(m.blocks[1], forward_tokens=lambda self, x, *a: x),
    "attention of another class": lambda m: _reclass(m.blocks[1].blocks[0].attn),
    "MLP of another class": lambda m: _reclass(m.blocks[0].blocks[0].mlp),
    "patch embedding of another class": lambda m: _reclass((m.patch_embeds[0] if m.channels_first else m.patch_embed)),
    "a layer's own method": lambda m: setattr(m.blocks[0].blocks[0], "forward_tokens", lambda x, *a: x),
    "a model's own method": lambda m: setattr(m, "_forward_tokens", types.MethodType(lambda self, *a: None, m)),
    "model of another class": lambda m: _reclass(m, _forward_tokens=lambda self, *a: None),
    "projection of another kind": lambda m: setattr(m.blocks[0].blocks[0].mlp, "fc1", nn.Sequential(m.blocks[0].blocks[0].mlp.fc1)),
    "projection without a bias": lambda m: setattr(m.blocks[0].blocks[0].mlp.fc2, "bias", None),
    "attention's projection without a bias": lambda m: setattr(m.blocks[1].blocks[0].attn.proj, "bias", None),
    "pooling without a bias": lambda m: setattr(m.pool.tdnn.conv, "bias", None),
    "head without a bias": lambda m: setattr(m.fc, "bias", None),
    "projection of another size": lambda m: setattr(m.blocks[0].blocks[0].mlp, "fc2", type(m.blocks[0].blocks[0].mlp.fc2)(512, 256)),
    "norm without statistics": lambda m: setattr(m.norm, "running_mean", None),
    "norm without weights": lambda m: setattr(m.proj.norm, "weight", None),
    "pooled norm of another kind": lambda m: setattr(m, "pool_norm", nn.LayerNorm(m.fc.in_features)),
    "pooling of another class": lambda m: _reclass(m.pool),
    "pooling's threshold": lambda m: setattr(m.pool, "eps", 1e-6),
    "window without its bias": lambda m: setattr(m.blocks[0].blocks[0].attn, "win_size", 25),
    "weight that is no parameter": lambda m: _weight_norm(m.blocks[0].blocks[0].attn.qkv),
    "16-bit parameters": lambda m: m.blocks[0].blocks[0].attn.qkv.to(torch.bfloat16),
    "double statistics": lambda m: m.pool_norm.double(),
    "a layer on another device": lambda m: m.fc.to("meta"),
    "statistics on another device": lambda m: m.norm._buffers.update(running_var=m.norm.running_var.to("meta")),
}


@pytest.mark.parametrize("family", ["pcf", "mfa"])
def test_models_as_constructed_fit(family):
    model = _model(family)
    assert encoder._as_built(model) and encoder._fits(model, CPU) and not encoder._fits(model, torch.device("cuda", 0))
    assert encoder._fits(_model(family, poolnorm=False), CPU) and not encoder._fits(_model(family, asp=False), CPU)
    assert not encoder._fits(_model(family, embed_dim=128), CPU) and not encoder._fits(_model(family, patch_size=5), CPU)
    assert encoder._fits(copy.deepcopy(model), CPU)


@pytest.mark.parametrize("family", ["pcf", "mfa"])
@pytest.mark.parametrize("change", sorted(CHANGES))
def test_what_the_kernels_do_not_know_stays_with_the_modules(change, family):
    model = _model(family)
    CHANGES[change](model)
    assert not (encoder._as_built(model) and encoder._fits(model, CPU))


@pytest.mark.parametrize("change", ["layer of another class", "a layer's own method", "projection of another kind", "parametrized weight"])
def test_changes_after_the_first_call_are_seen(change):
    model = _model()
    entry = encoder._Entry(model)
    assert entry.same_modules()
    if change in CHANGES:
        CHANGES[change](model)
    else:
        nn.utils.parametrize.register_parametrization(model.blocks[0].blocks[0].attn.qkv, "weight", nn.Identity())
    assert not entry.same_modules()


def test_what_is_kept_for_a_model_does_not_keep_the_model():
    model = _model()
    encoder._entries[model] = encoder._Entry(model)
    gone, held = weakref.ref(model), len(encoder._entries)
    del model
    gc.collect()
    assert gone() is None and len(encoder._entries) == held - 1


@pytest.mark.parametrize("family", ["pcf", "mfa"])
def test_a_changed_tensor_costs_what_was_made_of_it(family, monkeypatch):
    """A plan takes over what the plan before made of unchanged tensors, the table of positions among it; what it holds of
    the others is what a plan made from nothing holds."""
    model = _model(family)
    calls = []
    table = models.sinusoid_table
    monkeypatch.setattr(models, "sinusoid_table", lambda *a: calls.append(a) or table(*a))
    plan = encoder._Plan(model, torch.bfloat16)
    for change, renewed in ((lambda: model.blocks[0].blocks[0].mlp.fc1.weight.mul_(2), {(0, "fc1")}),
                            (lambda: model.blocks[0].blocks[0].norm2.load_state_dict(model.blocks[0].blocks[0].norm2.state_dict()), {(0, "fc1")}),
                            (lambda: model.norm.running_var.mul_(2), {"wide"}),
                            (lambda: model.blocks[1].blocks[0].attn.linear_pos.weight.mul_(2), {(1, "pos")}),
                            (lambda: model.fc.weight.mul_(2), set()),
                            (lambda: setattr(model.pool.conv, "weight", nn.Parameter(2 * model.pool.conv.weight)), {"logits"})):
        with torch.no_grad():
            change()
        after, fresh = encoder._Plan(model, torch.bfloat16, plan), encoder._Plan(model, torch.bfloat16)
        assert {n for n in after.made if after.made[n] is not plan.made[n]} == renewed
        assert all(torch.equal(a, b) for n in fresh.made for a, b in zip(after.made[n][1], fresh.made[n][1]))
        plan = after
    assert len(calls) == 1
    assert len(plan.made) == len(encoder._Plan(model, torch.float16, None).made)


@pytest.mark.parametrize("wide,emb,blocks,taken", [(1536, 192, 2, True), (65536, 8176, 2, True), (65536, 8192, 2, False), (65536, 65536, 2, False),
                                                   (65536, 16, 63, True), (65536, 16, 64, False)])
def test_weights_beyond_31_bits_are_refused(wide, emb, blocks, taken):
    plan = encoder._Plan(_model(), torch.bfloat16)
    e = plan.encoder
    e.wide, e.emb, e.blocks = wide, emb, blocks
    layers = (encoder._Layer * blocks)(*[plan.layers[0]] * blocks)
    for l in layers:
        l.block_end = 1
    e.layers, e.layer = blocks, layers
    assert (_lib.load().na1d_encode_workspace_bytes(ctypes.byref(e), 4, 100) > 0) == taken


_POINTERS = [n for n, t in encoder._Layer._fields_ if t is ctypes.c_void_p and n not in ("rpb", "w_pos")]


@pytest.mark.parametrize("name", _POINTERS + [n for n, t in encoder._Encoder._fields_ if t is ctypes.c_void_p and n != "pos"] + ["out", "x", "workspace"])
def test_missing_pointers_are_refused(name):
    """Before anything is launched: every argument but one is in order."""
    plan = encoder._Plan(_model(), torch.bfloat16)
    lib, e, args = _lib.load(), plan.encoder, {"out": 4096, "x": 4096, "workspace": 4096}
    need = lib.na1d_encode_workspace_bytes(ctypes.byref(e), 2, 64)
    assert need > 0
    if name in args:
        args[name] = None
    else:
        setattr(plan.layers[0] if name in _POINTERS else e, name, None)
    st = lib.na1d_encode(ctypes.byref(e), args["out"], args["x"], None, 2, 64, args["workspace"], need, None)
    assert st in (-1, _lib.UNSUPPORTED)                     # a weight's absence already says that nothing covers the call


def _gelu_errors(gelu):
    """Of an fp32 GELU against 64 bits: largest, largest relative one below 0.1, and rms for arguments of some deviations."""
    exact = lambda x: 0.5 * x.double() * torch.special.erfc(-x.double() * 0.5 ** 0.5)
    x = torch.linspace(-14, 14, 2000001)
    x = x[x != 0]
    error, small = (gelu(x).double() - exact(x)).abs(), x.abs() < 0.1
    draws = torch.randn(400000, generator=torch.Generator().manual_seed(0))
    rms = [(gelu(s * draws).double() - exact(s * draws)).square().mean().sqrt().item() for s in (0.02, 0.1, 0.3, 0.58, 1.0, 2.0, 4.0)]
    return [error.max().item(), (error / exact(x).abs())[small].max().item(), error[x < -3].max().item()] + rms


def test_gelu_is_no_worse_than_by_the_handbook():
    """The polynomial in inference's GELU, with fp32 roundings behind 64-bit multiply-adds, against formula 7.1.26 of Abramowitz
    and Stegun's handbook in the same arithmetic, by every measure: small arguments above all, where a constant term that is not
    -1 to the last bit costs all values the same share."""
    with open(os.path.join(os.path.dirname(_lib.__file__), "..", "csrc", "na1d_encoder.h")) as f:
        terms = [float(v.rstrip("f")) for v in re.search(r"kGelu\[\] = \{([^}]*)\}", f.read()).group(1).replace(" ", "").split(",")]
    fp32 = lambda v: v.float().double()

    def polynomial(x):
        a = x.double().abs()
        p = torch.full_like(a, terms[-1]).float().double()
        for t in terms[-2::-1]:
            p = fp32(p * a + torch.tensor(t).double())
        return fp32(x.double().clamp(min=0) - a * fp32(torch.exp2(p)))

    def handbook(x):
        a = x.double().abs()
        t = fp32(1 / fp32(a * torch.tensor(0.3275911 * 0.5 ** 0.5).double() + 1))
        e = torch.full_like(a, 0.5 * 1.061405429).float().double()
        for k in (-1.453152027, 1.421413741, -0.284496736, 0.254829592):
            e = fp32(e * t + torch.tensor(0.5 * k).double())
        e = fp32(e * fp32(torch.exp2(fp32(fp32(x.double() ** 2) * torch.tensor(-0.72134752).double()))))
        return fp32(x.double().clamp(min=0) - fp32(a * t) * e)

    assert terms[-1] < 0                                                       # the tail vanishes
    assert all(p <= h for p, h in zip(_gelu_errors(polynomial), _gelu_errors(handbook)))
    assert polynomial(torch.tensor([1e3, -1e3, 3e4, -3e4])).tolist() == [1e3, 0.0, 3e4, 0.0]
