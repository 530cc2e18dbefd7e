"""Embedding models in one native call: what it shares with the modules beyond ordinary inputs."""
import copy

import pytest
import torch

from na1d_amd import models
from oracle import na1d_oracle as O

pytestmark = pytest.mark.gpu
SMALL = dict(depths=(1, 1), num_heads=[[16], [4]], win_size=[[27], [0]], groups=(8, 4))


def _model(family="pcf", dtype=torch.bfloat16, seed=0, **kw):
    torch.manual_seed(seed)
    kw = dict(SMALL, **kw)
    if family == "mfa":
        kw.pop("groups")
    model = (models.PCF_NATransformer if family == "pcf" else models.MFA_NATransformer)(na="fused_qkv", dtype=dtype, **kw).cuda().eval()
    gen = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for m in model.modules():
            if isinstance(m, torch.nn.BatchNorm1d):                                     # statistics as training leaves them
                m.running_mean.copy_(0.1 * torch.randn(m.num_features, generator=gen))
                m.running_var.copy_(0.75 + 0.5 * torch.rand(m.num_features, generator=gen))
    return model


def _input(batch, frames, seed=1, chans=80):
    return torch.randn(batch, chans, frames, generator=torch.Generator().manual_seed(seed)).cuda()


def _both(model, x, lens=None, dtype=torch.bfloat16):
    """The native call's embeddings (None where it leaves the model to the modules), and the modules'."""
    with torch.no_grad(), torch.autocast("cuda", dtype=dtype):
        native = models.embed_natively(model, x, lens)
        handle = model.fc.register_forward_hook(lambda *a: None)                        # a hook keeps the modules in use
        try:
            modules = model(x, lens)
        finally:
            handle.remove()
    return native, modules


def _near(a, b, dtype=torch.bfloat16):
    """Two 16-bit evaluations of a few layers: each is within a few units of eps of the exact value."""
    return O.rel_l2(a.float(), b.float()) < (2e-2 if dtype == torch.bfloat16 else 2.5e-3)


@pytest.mark.parametrize("groups", [16, 32])
@pytest.mark.parametrize("batch,frames", [(3, 111), (16, 128), (17, 122), (80, 128)])
def test_group_counts_without_kernels_of_their_own(groups, batch, frames):
    """Weights in blocks of any number of groups but 2, 4 and 8 are multiplied as the dense matrices they are, in the split
    launches of up to 1024 tokens as in the larger ones."""
    model = _model(groups=(groups, 8), in_chans=64)
    native, modules = _both(model, _input(batch, frames, chans=64))
    assert native is not None and _near(native, modules)


@pytest.mark.parametrize("groups", [(8, 4), (2, 1)])
@pytest.mark.parametrize("batch,frames", [(53, 32), (81, 100), (86, 96), (163, 100), (164, 100), (293, 112), (331, 100)])
def test_tiles_of_every_size(groups, batch, frames):
    """Each side of the token counts at which the tiles grow (1024 is the split's; 4096, 8192, 16384), the last tile not full."""
    model = _model(groups=groups)
    native, modules = _both(model, _input(batch, frames))
    assert native is not None and _near(native, modules)


@pytest.mark.parametrize("groups", [(8, 4), (2, 1)])
@pytest.mark.parametrize("batch,frames", [(328, 100), (427, 96), (491, 100), (512, 96), (513, 96)])
def test_row_tiles_dealt_out_evenly(groups, batch, frames):
    """16385 to 24576 tokens: the first, the middle and the last numbers of workgroups with three row tiles, the last tile full and
    not, and the first size behind."""
    model = _model(groups=groups)
    native, modules = _both(model, _input(batch, frames))
    assert native is not None and _near(native, modules)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,frames", [(31, 100), (32, 256), (33, 258), (85, 260), (86, 260), (31, 400), (32, 400), (32, 402),
                                          (53, 402), (54, 402), (65, 1000), (65, 1002), (68, 1002), (69, 1002), (86, 1002)])
def test_pooling_with_one_wave_or_four_to_an_utterance(batch, frames, dtype):
    """Each side of the sizes at which the waves of a pooling workgroup part by channels alone; lengths from one token on."""
    model = _model(dtype=dtype)
    lens = torch.rand(batch, generator=torch.Generator().manual_seed(batch))
    lens[0], lens[1], lens[2] = 1.0, 2.0 / frames, 34.0 / frames
    lens = lens.clamp(2.0 / frames, 1.0).cuda()
    x = _input(batch, frames)
    x *= (torch.arange(frames).cuda() < (lens * frames).round().unsqueeze(1)).unsqueeze(1)
    native, modules = _both(model, x, lens, dtype)
    assert native is not None and _near(native, modules, dtype)


@pytest.mark.parametrize("groups", [0, 3, 16])
@pytest.mark.parametrize("batch,frames", [(3, 111), (80, 128)])
def test_layers_of_the_c_interface_are_dense_unless_2_4_or_8(groups, batch, frames):
    """na1d_encoder_layer.groups: any other number says nothing about the weights.  (The models' own 16 or 32 groups have
    zeros where the quarters of the hidden layer do not meet; dense weights do not.)"""
    from na1d_amd import encoder
    model = _model("mfa")
    x = _input(batch, frames)
    want, _ = _both(model, x)
    for l in encoder.plans_of(model)[0].layers:
        l.groups = groups
    got, _ = _both(model, x)
    assert torch.equal(got, want)


@pytest.mark.parametrize("batch,frames", [(3, 64), (40, 128), (180, 100)])
@pytest.mark.parametrize("family", ["pcf", "mfa"])
def test_nan_stays_in_its_utterance_and_is_not_lost(family, batch, frames):
    """A frame without a number makes its utterance's embedding so, as in the modules; the others' stay what they were."""
    model = _model(family, dtype=torch.float16)
    x = _input(batch, frames)
    clean, _ = _both(model, x, dtype=torch.float16)
    broken = x.clone()
    broken[1, 5, 7] = float("nan")
    native, modules = _both(model, broken, dtype=torch.float16)
    assert torch.isnan(modules[1]).all() and torch.isnan(native[1]).all()
    rest = [i for i in range(batch) if i != 1]
    assert torch.equal(native[rest], clean[rest])


def test_overflow_is_not_lost():
    """Values beyond fp16 become infinities, and what is made of them not a number, exactly where the modules' do."""
    model = _model("mfa", dtype=torch.float16)
    x = _input(4, 64)
    x[2] *= 1e9
    native, modules = _both(model, x, dtype=torch.float16)
    assert not torch.isfinite(modules[2]).all()
    assert torch.equal(torch.isfinite(native), torch.isfinite(modules))


def test_replicas_run():
    """What DataParallel makes of a model for each call: copies whose weights are plain tensors."""
    model = _model()
    x = _input(3, 64)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        replica = torch.nn.parallel.replicate(model, [0])[0]
        assert not list(replica.parameters())
        assert _near(replica(x), model(x))


def test_models_that_do_not_fit_run_as_they_did():
    """A layer of a class of its own is called, a projection without a bias runs, tensors on two devices are refused."""
    x = _input(3, 64)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        model = _model()
        before = model(x)
        layer = model.blocks[1].blocks[0]
        layer.__class__ = type("Skipped", (models.NATFLayer,), {"forward_tokens": lambda self, x, *a: 0.5 * x})
        assert models.embed_natively(model, x) is None and not _near(model(x), before)
        model = _model()
        model.blocks[0].blocks[0].mlp.fc2.bias = None
        assert models.embed_natively(model, x) is None
        a = model(x)
        model.blocks[0].blocks[0].mlp.fc2.bias = torch.nn.Parameter(torch.zeros(256, device="cuda"))
        assert models.embed_natively(model, x) is not None and _near(model(x), a)
        model.fc.cpu()
        assert models.embed_natively(model, x) is None
        with pytest.raises(RuntimeError):
            model(x)
        model.fc.cuda()
        assert _near(model(x), a)
        model.pool_norm.train()
        assert models.embed_natively(model, x) is None and not _near(model(x), a)      # statistics of the batch


def _dilation(m):
    m.blocks[0].blocks[0].attn.dilation = 2


def _scale(m):
    m.blocks[0].blocks[0].attn.scale *= 1.5


def _dense_scale(m):
    m.blocks[1].blocks[0].attn.scale *= 3.0


def _left(m):
    m.blocks[0].blocks[0].attn.left = 3


def _heads(m):
    m.blocks[1].blocks[0].attn.num_heads = 16


def _eps(m):
    m.norm.eps = 0.5


def _head_eps(m):
    m.pool_norm.eps = 0.5


@pytest.mark.parametrize("change", [_dilation, _scale, _dense_scale, _left, _heads, _eps, _head_eps])
def test_numbers_are_read_at_each_call(change):
    """Scales, windows, dilations, heads and a norm's eps are attributes that a program may set between two calls; the copy is a
    model made with them."""
    model, x = _model(), _input(5, 90)
    with torch.no_grad():                                                               # attentions that tell their keys apart
        for block in model.blocks:
            block.blocks[0].attn.qkv.weight.mul_(4.0)
    before, _ = _both(model, x)
    change(model)
    fresh = copy.deepcopy(model)
    native, _ = _both(model, x)
    again, modules = _both(fresh, x)
    assert _near(native, modules) and torch.equal(native, again) and not torch.equal(native, before)


@pytest.mark.parametrize("name", ["fc.weight", "fc.bias", "pool_norm.weight", "pool_norm.bias", "pool_norm.running_mean", "pool_norm.running_var",
                                  "blocks.1.blocks.0.norm1.weight", "blocks.1.blocks.0.norm1.bias", "blocks.1.blocks.0.norm1.running_mean",
                                  "blocks.1.blocks.0.norm1.running_var", "blocks.0.blocks.0.attn.relative_position_bias"])
@pytest.mark.parametrize("batch,frames", [(3, 64), (40, 128), (600, 16)])
def test_what_the_modules_read_at_each_call_is_read_at_each_call(name, batch, frames):
    """The head, the pooled norm, a dense layer's first norm and a window's bias are never copied: a write that torch counts
    no version for (through .data) shows in the next call, and in the next replay of a graph."""
    model, x = _model(), _input(batch, frames)
    before, _ = _both(model, x)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16), torch.cuda.graph(graph):
        captured = models.embed_natively(model, x)
    t = model.get_parameter(name) if not name.rpartition(".")[2].startswith("running") else model.get_buffer(name)
    version = t._version
    t.data.mul_(1.5).add_(0.5 * torch.randn(t.shape, generator=torch.Generator().manual_seed(2)).cuda().abs())
    assert t._version == version
    native, modules = _both(model, x)
    assert _near(native, modules) and not torch.equal(native, before)
    for _ in range(2):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, native)


@pytest.mark.parametrize("emb", [16, 64, 208, 256])
@pytest.mark.parametrize("batch", [1, 17, 513])
def test_embedding_sizes(emb, batch):
    """The last layer at every remainder of its tiles of 16 rows and of the rounds of inputs."""
    for poolnorm in (True, False):
        model = _model("mfa", dtype=torch.float16, output_emb_size=emb, proj_channel=256 * (1 + emb % 3), poolnorm=poolnorm)
        native, modules = _both(model, _input(batch, 16), dtype=torch.float16)
        assert native.shape == (batch, emb) and _near(native, modules, torch.float16)


def test_first_calls_and_changes_in_inference_mode():
    """Plans and the table of positions may be made while torch tracks no versions of new tensors."""
    model, x = _model(), _input(3, 64)
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.bfloat16):
        first = models.embed_natively(model, x)
    native, _ = _both(model, x)
    assert torch.equal(first, native)
    with torch.no_grad():
        model.blocks[0].blocks[0].mlp.fc1.weight.mul_(2.0)
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.bfloat16):
        second = models.embed_natively(model, x)
    native, modules = _both(model, x)
    assert torch.equal(second, native) and _near(native, modules) and not torch.equal(first, second)


def test_a_plan_outlives_its_use_on_other_streams():
    """Weights change, and another stream makes the new plan, while a queue of passes still reads the old one: the memory of
    the old one is not handed out before they are done."""
    model, x = _model("mfa"), _input(64, 600)
    want, _ = _both(model, x)
    side, outs = torch.cuda.Stream(), []
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
                outs.append(models.embed_natively(model, x))
    with torch.no_grad():
        for block in model.blocks:
            for m in (block.blocks[0].attn.proj, block.blocks[0].mlp.fc1, block.blocks[0].mlp.fc2):
                m.weight = torch.nn.Parameter(torch.zeros_like(m.weight))              # the passes read biases, not these
    after, _ = _both(model, x[:1])
    filled = [torch.full((n,), float("nan"), dtype=torch.bfloat16, device="cuda") for n in (256 * 256, 256 * 1024) * 40]
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs) and not _near(after, want[:1])
    del filled


@pytest.mark.parametrize("batch,frames", [(3, 64), (40, 128), (86, 96), (331, 100)])
@pytest.mark.parametrize("groups", [(8, 4), (2, 1)])
def test_parameters_on_any_float(groups, batch, frames):
    """Biases that are views of a flat buffer, on 4, 8 and 12 bytes: to the bit what they are on their own."""
    model = _model(groups=groups)
    x = _input(batch, frames)
    want, _ = _both(model, x)
    moved = copy.deepcopy(model)
    for at, layer in enumerate(l for b in moved.blocks for l in b.blocks):
        for k, m in enumerate((layer.attn.proj, layer.mlp.fc2)):
            flat = torch.zeros(264, device="cuda")
            at_float = 1 + (2 * at + k) % 3
            flat[at_float:at_float + 256] = m.bias.detach()
            m.bias = torch.nn.Parameter(flat[at_float:at_float + 256])
            assert m.bias.data_ptr() % 16
    got, _ = _both(moved, x)
    assert got is not None and torch.equal(got, want)
