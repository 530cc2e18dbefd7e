"""A windowed encoder layer in training as one native node (na1d_train_layer_*) against the fp32 module on the CPU."""
import contextlib
import copy

import pytest
import torch

from na1d_amd import _lib, models, train
from oracle import na1d_oracle as O

pytestmark = pytest.mark.gpu
DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _cpu_attention(q, k, v, W, left, rpb=None, t_valid=None, num_heads=1, dilation=1):
    """The operator in plain torch, differentiable: the keys of every window slot gathered by row."""
    B, T, C = q.shape
    t, j = torch.arange(T).unsqueeze(1), torch.arange(W)
    key = t + (j - left) * dilation
    inside = (key >= 0) & (key < T)
    kk, vv = (z[:, key.clamp(0, T - 1)] for z in (k, v))                          # [B, T, W, C]
    s = (q.unsqueeze(2) * kk).sum(-1) * inside
    s = (s.view(-1, num_heads, T, W) + rpb.view(1, num_heads, 1, W)).view(B, T, W) + (~inside) * models.MASK_VALUE
    p = torch.softmax(s, -1) * inside
    return (p.unsqueeze(-1) * vv).sum(2)


def _layers(family, groups, heads, window, dilation, frames, drop_path, seed, dim=256):
    torch.manual_seed(seed)
    layer = models.NATFLayer(frames, dim, heads, window, groups, drop_path, family == "pcf", torch.bfloat16, _cpu_attention,
                             dilation=dilation)
    with torch.no_grad():
        for p in layer.parameters():
            p.mul_(2.0)                                                              # far from the initial near-identity
        for bn in (m for m in layer.modules() if isinstance(m, torch.nn.BatchNorm1d)):
            bn.weight.uniform_(0.5, 1.5)
            bn.bias.normal_(0, 0.3)
    gpu = copy.deepcopy(layer).cuda()
    if window:
        gpu.attn.na = "fused_qkv"
    return layer.train(), gpu.train()


def _errors(cpu, gpu, x, g, dtype, pos=None):
    """Relative errors of the native layer's output, gradients and running statistics against the fp32 module."""
    xg = x.cuda().to(dtype).requires_grad_(True)
    torch.manual_seed(5)
    with torch.autocast("cuda", dtype=dtype):
        out = models.train_layer(gpu, xg, None if pos is None else pos.cuda())
    assert out is not None, "not the native path"
    gd = g.cuda().to(dtype)
    out.backward(gd)
    torch.manual_seed(5)
    xc = x.to(dtype).float().requires_grad_(True)
    want = cpu(xc, pos_emb=None if pos is None else pos.to(dtype).float())
    want.backward(gd.float().cpu())
    err = {"out": O.rel_l2(out.float(), want), "dx": O.rel_l2(xg.grad.float(), xc.grad)}
    for (name, p), q in zip(cpu.named_parameters(), gpu.parameters()):
        if name.endswith("proj.bias") or name.endswith("fc2.bias") or p.grad.norm() > 1e-3 * p.grad.numel() ** 0.5:
            err["d " + name] = O.rel_l2(q.grad, p.grad)
    for (name, p), q in zip(cpu.named_buffers(), gpu.buffers()):
        if "running" in name:
            err[name] = O.rel_l2(q, p)
        elif name.endswith("batches_tracked"):
            assert q.item() == p.item() == 1
    return err


# tokens: fewer than a tile (of two rows a norm makes +-1 whatever they hold: nothing to compare), one chunk of rows, remainders of every tile, the launch sizes of both product tiles
@pytest.mark.parametrize("batch,T", [(2, 5), (1, 33), (3, 50), (7, 101), (37, 100), (64, 260)])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("family,groups,heads,window,dilation", [
    ("mfa", 1, 16, 27, 1), ("mfa", 1, 4, 65, 1), ("pcf", 8, 16, 27, 1), ("pcf", 4, 8, 9, 2), ("pcf", 2, 16, 27, 1), ("pcf", 1, 32, 5, 3),
    ("mfa", 1, 4, 0, 1), ("mfa", 1, 16, 0, 1), ("pcf", 8, 4, 0, 1), ("pcf", 1, 2, 0, 1)])
def test_native_training_layer(family, groups, heads, window, dilation, dtype, batch, T):
    """16-bit rounding of weights, activations and gradients passes through six products and two norms: single results
    are within a few units of eps (2^-9, 2^-12) in norm; a few rows leave the statistics of the gradients little to
    average over, and what is left of sums that cancel (qkv's gradients behind the softmax) carries the most."""
    if batch * T > 5000 and (dtype, family) not in (("fp16", "mfa"), ("bf16", "pcf")):
        pytest.skip("the large batch once per family")
    cpu, gpu = _layers(family, groups, heads, window, dilation, T, 0.0, seed=T)
    gen = torch.Generator().manual_seed(batch)
    shape = (batch, 256, T) if family == "pcf" else (batch, T, 256)
    x = torch.randn(shape, generator=gen) + 0.5 * torch.randn((1,) + tuple(256 if s == 256 else 1 for s in shape[1:]), generator=gen)
    pos = None if window else models.sinusoid_table(256, T, family == "pcf")
    err = _errors(cpu, gpu, x, torch.randn(shape, generator=gen), DT[dtype], pos)
    print("errors", {k: "%.1e" % v for k, v in err.items()})
    eps = 2.0 ** -9 if dtype == "bf16" else 2.0 ** -12
    for name, e in err.items():
        # running statistics: norm1's come of exact inputs; norm2's are means of the attention half's outputs, and of few
        # rows no better than a single one
        bound = 1e-5 if "norm1" in name and "running" in name else 4 * eps if "running" in name or name == "out" else 32 * eps
        assert e < bound, (name, e)


# The product in front of a norm's backward: it sums for the norm in blocks of 32 rows up to 8128 tokens and of 64 rows up to 16384;
# beyond, a kernel of its own does.  Last blocks of 4, 6, 64, 44 and 16 rows.
@pytest.mark.parametrize("batch,T", [(81, 100), (83, 98), (128, 100), (163, 100), (164, 100)])
@pytest.mark.parametrize("family,groups,heads,window,dtype", [("mfa", 1, 16, 27, "fp16"), ("pcf", 8, 16, 27, "bf16"), ("mfa", 1, 4, 0, "fp16")])
def test_gradients_behind_every_form_of_the_norms_sums(family, groups, heads, window, dtype, batch, T):
    """Bounds as in test_native_training_layer."""
    cpu, gpu = _layers(family, groups, heads, window, 1, T, 0.0, seed=T)
    gen = torch.Generator().manual_seed(batch)
    shape = (batch, 256, T) if family == "pcf" else (batch, T, 256)
    x = torch.randn(shape, generator=gen) + 0.5 * torch.randn((1,) + tuple(256 if s == 256 else 1 for s in shape[1:]), generator=gen)
    err = _errors(cpu, gpu, x, torch.randn(shape, generator=gen), DT[dtype], None if window else models.sinusoid_table(256, T, False))
    eps = 2.0 ** -9 if dtype == "bf16" else 2.0 ** -12
    assert {"dx", "d norm1.norm.weight", "d norm2.norm.bias"} <= set(err) or {"dx", "d norm1.weight", "d norm2.bias"} <= set(err)
    for name, e in err.items():
        assert e < (1e-5 if "norm1" in name and "running" in name else 4 * eps if "running" in name or name == "out" else 32 * eps), (name, e)


def test_stochastic_depth_draws_like_the_modules():
    cpu, gpu = _layers("mfa", 1, 16, 27, 1, 64, 0.4, seed=1)
    gen = torch.Generator().manual_seed(0)
    x, g = torch.randn(9, 64, 256, generator=gen).half().cuda(), torch.randn(9, 64, 256, generator=gen).half().cuda()
    results = []
    for native in (True, False):
        layer = copy.deepcopy(gpu)
        xg = x.clone().requires_grad_(True)
        handle = None if native else layer.mlp.fc2.register_forward_hook(lambda *a: None)    # a hook keeps the modules in use
        torch.manual_seed(3)
        with torch.autocast("cuda", dtype=torch.float16):
            assert (models.train_layer(layer, xg) is not None) == native
            torch.manual_seed(3)
            out = layer(xg)
        out.backward(g)
        results.append((out.detach(), xg.grad, layer.mlp.fc2.weight.grad, layer.attn.qkv.weight.grad))
    for a, b in zip(*results):
        assert O.rel_l2(a.float(), b.float()) < 32 * 2.0 ** -12


def test_what_the_node_does_not_cover_stays_with_the_modules():
    _, gpu = _layers("mfa", 1, 16, 27, 1, 40, 0.0, seed=1)
    x = torch.randn(4, 40, 256).half().cuda().requires_grad_(True)

    def native(layer=gpu, x=x):
        return models.train_layer(layer, x) is not None
    assert not native()                                                              # no autocast
    with torch.autocast("cuda", dtype=torch.float16):
        assert native()
        assert not native(x=x.float())
        assert not native(x=x[:, :39])                                              # the layer itself refuses this length
        with pytest.raises(AssertionError):
            gpu(x[:, :39])
        with torch.no_grad():
            assert not native()
        for change in (lambda m: setattr(m.norm1.norm, "momentum", None), lambda m: m.norm2.norm.eval(),
                       lambda m: setattr(m.mlp.drop, "p", 0.1), lambda m: setattr(m.attn, "attn_drop", 0.1),
                       lambda m: setattr(m.mlp, "act", torch.nn.ReLU()), lambda m: m.attn.register_forward_hook(lambda *a: None),
                       lambda m: setattr(m.mlp, "fc1", torch.nn.Sequential(m.mlp.fc1)), lambda m: m.half()):
            layer = copy.deepcopy(gpu)
            change(layer)
            assert not native(layer)
        layer = copy.deepcopy(gpu)
        layer.mlp.fc1.weight.requires_grad_(False)
        before = layer.norm1.norm.running_mean._version
        layer(x).sum().backward()
        assert layer.mlp.fc1.weight.grad is None and layer.mlp.fc2.weight.grad is not None
        assert layer.norm1.norm.running_mean._version > before


@pytest.mark.parametrize("family,groups,heads,window,drop_path", [("mfa", 1, 16, 27, 0.3), ("pcf", 8, 16, 27, 0.0), ("mfa", 1, 4, 0, 0.0), ("pcf", 1, 4, 0, 0.3)])
def test_a_library_that_is_named_serves_training_layers_too(family, groups, heads, window, drop_path, monkeypatch):
    """Without the extension beside the package's own library the launches go through ctypes: the same bits and version counts."""
    _, gpu = _layers(family, groups, heads, window, 1, 40, drop_path, seed=2)
    gen = torch.Generator().manual_seed(1)
    shape = (6, 256, 40) if family == "pcf" else (6, 40, 256)
    x, g = (torch.randn(shape, generator=gen).half().cuda() for _ in range(2))
    pos = None if window else models.sinusoid_table(256, 40, family == "pcf").cuda()
    results = []
    for named in (False, True):
        monkeypatch.setattr(_lib, "_other_build", named)
        layer, leaf = copy.deepcopy(gpu), x.clone().requires_grad_(True)
        torch.manual_seed(4)
        with torch.autocast("cuda", dtype=torch.float16):
            out = models.train_layer(layer, leaf, pos)
        assert out is not None
        out.backward(g)
        results.append(([out.detach(), leaf.grad, *(b for b in layer.buffers())], [p.grad for p in layer.parameters()], [b._version for b in layer.buffers()]))
    for a, b in zip(results[0][0], results[1][0]):
        assert torch.equal(a, b)
    for (name, _), a, b in zip(gpu.named_parameters(), results[0][1], results[1][1]):
        assert torch.equal(a, b) if "relative" not in name else O.rel_l2(a, b) < 1e-5, name       # the scores' bias: float atomics
    assert results[0][2] == results[1][2]


def _off_alignment(t):
    return torch.empty(t.numel() + 8, dtype=t.dtype, device=t.device)[1:t.numel() + 1].view(t.shape).copy_(t)


@pytest.mark.parametrize("window", [27, 0])
def test_tensors_off_their_alignment(window):
    """An input that starts anywhere goes to the modules, a gradient and positions that do are copied."""
    _, gpu = _layers("mfa", 1, 16, window, 1, 40, 0.0, seed=1)
    gen = torch.Generator().manual_seed(2)
    x, g = (torch.randn(4, 40, 256, generator=gen).half().cuda() for _ in range(2))
    pos = None if window else models.sinusoid_table(256, 40, False).half().cuda()
    results = []
    for move in (lambda t: t, _off_alignment):
        layer = copy.deepcopy(gpu)
        xg = x.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.float16):
            out = layer(xg, pos_emb=None if pos is None else move(pos))
        assert type(out.grad_fn).__name__ == "_TrainLayerBackward"
        out.backward(move(g))
        results.append((out.detach(), xg.grad, layer.mlp.fc1.weight.grad, layer.attn.qkv.weight.grad))
    assert all(torch.equal(a, b) for a, b in zip(*results))
    off = _off_alignment(x).requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.float16):
        assert models.train_layer(copy.deepcopy(gpu), off, pos) is None
        out = copy.deepcopy(gpu)(off, pos_emb=pos)
    out.backward(g)
    assert O.rel_l2(off.grad.float(), results[0][1].float()) < 32 * 2.0 ** -12


# both product tiles (64 rows from 128 blocks of 64 rows x 256 outputs on, else 32), remainders of either, one sample
@pytest.mark.parametrize("batch,T", [(1, 33), (7, 101), (37, 100), (128, 100), (64, 260)])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("family,groups,heads,window,dilation", [
    ("mfa", 1, 16, 27, 1), ("mfa", 1, 4, 65, 1), ("pcf", 8, 16, 27, 1), ("pcf", 4, 8, 9, 2), ("pcf", 2, 16, 27, 1), ("pcf", 1, 32, 5, 3),
    ("mfa", 1, 4, 0, 1), ("mfa", 1, 16, 0, 1), ("pcf", 8, 4, 0, 1), ("pcf", 1, 2, 0, 1)])
def test_forward_is_the_modules_to_the_bit(family, groups, heads, window, dilation, dtype, batch, T):
    """Output and running statistics, at these sizes: training amplifies a difference in the last bit of a forward over its
    layers.  The residual stream lies in memory as it does in the models, channels first in both families (torch sums
    statistics and adds biases in another way for the other layout)."""
    _, gpu = _layers(family, groups, heads, window, dilation, T, 0.3, seed=T)
    gen = torch.Generator().manual_seed(batch)
    x = torch.randn(batch, 256, T, generator=gen).cuda().to(DT[dtype])
    x = x if family == "pcf" else x.transpose(1, 2)
    pos = None if window else models.sinusoid_table(256, T, family == "pcf").cuda()
    results = []
    for native in (True, False):
        layer = copy.deepcopy(gpu)
        if not native:
            layer.mlp.fc2.register_forward_hook(lambda *a: None)
        torch.manual_seed(3)
        with torch.autocast("cuda", dtype=DT[dtype]):
            out = layer(x.clone().requires_grad_(True), pos_emb=pos)
        assert ("_TrainLayer" in repr(out.grad_fn) or "_TrainLayer" in repr(out.grad_fn.next_functions)) == native
        results.append([out.detach()] + [b for n, b in layer.named_buffers() if "running" in n or "batches" in n])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_layers_behind_each_other_are_the_modules_to_the_bit(dtype):
    """The tokens-first model's stream: channels first in the modules' memory, tokens first between two native layers."""
    stack = torch.nn.ModuleList(_layers("mfa", 1, heads, window, 1, 100, 0.2, seed=i)[1] for i, (heads, window) in enumerate(((16, 27), (4, 0), (16, 27))))
    x = torch.randn(24, 256, 100, generator=torch.Generator().manual_seed(0)).cuda().to(DT[dtype]).transpose(1, 2)
    pos = models.sinusoid_table(256, 100, False).cuda()
    results = []
    for native in (True, False):
        layers = copy.deepcopy(stack)
        torch.manual_seed(3)
        y = x.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=DT[dtype]):
            for layer in layers:
                if not native:
                    layer.mlp.fc2.register_forward_hook(lambda *a: None)
                y = layer(y, pos_emb=pos)
        results.append([y.detach()] + [b for n, b in layers.named_buffers() if "running" in n])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("heads,window", [(16, 27), (4, 0)])
def test_tokens_first_inputs_lose_nothing(heads, window, dtype):
    """A layer called by itself on tokens that lie one behind the other is as near to 64 bits as the modules are."""
    cpu, gpu = _layers("mfa", 1, heads, window, 1, 100, 0.0, seed=2)
    gen = torch.Generator().manual_seed(0)
    x, g = (torch.randn(24, 100, 256, generator=gen).to(DT[dtype]) for _ in range(2))
    pos = None if window else models.sinusoid_table(256, 100, False)
    exact, xc = copy.deepcopy(cpu).double(), x.double().requires_grad_(True)
    want = exact(xc, pos_emb=None if pos is None else pos.to(DT[dtype]).double())
    want.backward(g.double())
    errors = []
    for native in (True, False):
        layer, xg = copy.deepcopy(gpu), x.cuda().requires_grad_(True)
        if not native:
            layer.mlp.fc2.register_forward_hook(lambda *a: None)
        with torch.autocast("cuda", dtype=DT[dtype]):
            out = layer(xg, pos_emb=None if pos is None else pos.cuda())
        assert (type(out.grad_fn).__name__ == "_TrainLayerBackward") == native
        out.backward(g.cuda())
        errors.append([O.rel_l2(out.float(), want.float()), O.rel_l2(xg.grad.float(), xc.grad.float())])
    print(errors)
    assert all(a < 1.02 * b for a, b in zip(*errors))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,c,t", [(2, 8, 2), (3, 16, 100), (2, 24, 131), (1, 8, 2048), (5, 136, 33), (2, 1536, 100)])
def test_pooling_nodes_against_64_bits(n, c, t, dtype):
    """Rows of every remainder, blocks that span samples: the forward is torch's to the bit, the gradients are what the type
    gives (a rounding or two of 2^-9 or 2^-12; the context's deviations are rounded too), and a second derivative is torch's."""
    gen = torch.Generator().manual_seed(n * c + t)
    make = lambda *s: torch.randn(s, generator=gen).to("cuda", dtype).requires_grad_(True)
    tol = 1e-2 if dtype == torch.bfloat16 else 1.5e-3
    rel = lambda a, b: float((a.double() - b).norm() / b.norm())
    x, z, d1 = make(n, c, t), make(n, c, t), torch.randn(n, 3 * c, t, generator=gen).to("cuda", dtype)
    d2 = torch.randn(n, 2 * c, generator=gen).cuda()
    with torch.autocast("cuda", dtype=dtype):
        got, want = train.pooling_context(x, 1e-12), train.context_of(x, 1e-12)[0]
        assert "Context" in type(got.grad_fn).__name__ and torch.equal(got, want)
        out, same = train.pooled(z, x, 1e-12), train.pooled_of(z, x, 1e-12)
        assert "Pooled" in type(out.grad_fn).__name__ and torch.equal(out, same)
    exact = [v.detach().double().requires_grad_(True) for v in (x, z)]
    (dx,), (ex,) = torch.autograd.grad(got, (x,), d1), torch.autograd.grad(train.context_of(exact[0], 1e-12)[0], exact[:1], d1.double())
    assert rel(dx, ex) < tol
    grads = torch.autograd.grad(out, (x, z), d2, retain_graph=True)
    for g, e in zip(grads, torch.autograd.grad(train.pooled_of(exact[1], exact[0], 1e-12), exact, d2.double())):
        assert rel(g, e) < tol
    twice = [torch.autograd.grad(torch.autograd.grad(o, x, d2, create_graph=True)[0].float().square().sum(), x)[0] for o in (out, same)]
    assert torch.allclose(*[v.float() for v in twice], rtol=5e-2, atol=1e-3 * float(twice[1].float().abs().max()))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_pooling_gradients_that_are_differentiated_again(dtype):
    """The module's gradients with create_graph and without, and a second derivative, against its operations in 64 bits.  Every
    tensor on the way is rounded to the type some ten times (2^-9 or 2^-12 each: the operations' own gradients are 9.4e-3 and
    6.6e-4 off, the second ones 3.9e-2 and, in fp16, no numbers); a path counted twice is 40 % and more."""
    torch.manual_seed(0)
    tol = 2e-2 if dtype == torch.bfloat16 else 2e-3
    pool = models.AttentiveStatisticsPooling(64, 32).cuda()
    exact = copy.deepcopy(pool).double()
    x, d = torch.randn(3, 64, 50).to("cuda", dtype).requires_grad_(True), torch.randn(3, 128).cuda()
    xe, de = x.detach().double().requires_grad_(True), d.double()
    with torch.autocast("cuda", dtype=dtype):
        out = pool(x)
    assert "Pooled" in type(out.grad_fn).__name__
    (want,) = torch.autograd.grad(exact(xe), xe, de, create_graph=True)
    (plain,) = torch.autograd.grad(out, x, d, retain_graph=True)
    (dx,) = torch.autograd.grad(out, x, d, create_graph=True)
    twice, wanted = (torch.autograd.grad(g.to(w.dtype).square().sum(), v)[0] for g, w, v in ((dx, d, x), (want, de, xe)))
    assert O.rel_l2(plain.float(), want.float()) < tol and O.rel_l2(dx.float(), want.float()) < tol
    assert dtype == torch.float16 or O.rel_l2(twice.float(), wanted.float()) < 4 * tol


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_pooling_gradients_in_batches(dtype):
    """Each of several gradients taken at once is what it is by itself; by the kernels there, which round in other places."""
    torch.manual_seed(1)
    pool = models.AttentiveStatisticsPooling(64, 32).cuda()
    x, d = torch.randn(3, 64, 50).to("cuda", dtype).requires_grad_(True), torch.randn(4, 3, 128).cuda()
    with torch.autocast("cuda", dtype=dtype):
        out = pool(x)
    assert "Pooled" in type(out.grad_fn).__name__
    (batch,) = torch.autograd.grad(out, x, d, retain_graph=True, is_grads_batched=True)
    for got, one in zip(batch, d):
        (want,) = torch.autograd.grad(out, x, one, retain_graph=True)
        assert O.rel_l2(got.float(), want.float()) < (2e-2 if dtype == torch.bfloat16 else 2e-3)


def test_pooling_output_can_be_written_to():
    torch.manual_seed(2)
    pool = models.AttentiveStatisticsPooling(64, 32).cuda()
    x, d = torch.randn(3, 64, 50).to("cuda", torch.bfloat16).requires_grad_(True), torch.randn(3, 128).cuda()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = pool(x)
        twice = pool(x).mul_(2)                     # a factor of two rounds nothing
    assert "Pooled" in type(out.grad_fn).__name__ and torch.equal(twice, 2 * out)
    assert torch.equal(*(torch.autograd.grad(o, x, d)[0] for o in (twice, 2 * out)))


@pytest.mark.parametrize("pack,unpack", [(lambda t: t.mT.contiguous() if t.dim() > 1 else t, lambda t: t.mT if t.dim() > 1 else t),
                                         (lambda t: t.double(), lambda t: t)], ids=["other strides", "another type"])
def test_pooling_under_hooks_on_saved_tensors(pack, unpack):
    """Hooks may hand saved tensors back in another form; what torch's operations make of it is what counts."""
    torch.manual_seed(3)
    pool, d, grads = models.AttentiveStatisticsPooling(64, 32).cuda(), torch.randn(3, 128).cuda(), []
    x = torch.randn(3, 64, 50).to("cuda", torch.bfloat16).requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        hidden = pool.tanh(pool.tdnn(train.context_of(x, pool.eps)[0])).detach()       # the nodes alone under the hooks
        logits = pool.conv(hidden).detach().requires_grad_(True)
        for hooked in (False, True):
            with torch.autograd.graph.saved_tensors_hooks(pack, unpack) if hooked else contextlib.nullcontext():
                out, ctx = train.pooled(logits, x, pool.eps), train.pooling_context(x, pool.eps)
            assert "Pooled" in type(out.grad_fn).__name__ and "Context" in type(ctx.grad_fn).__name__
            grads.append(torch.autograd.grad((out, ctx), (logits, x), (d, torch.ones_like(ctx) * d[:, :1, None].bfloat16())))
    for got, want in zip(*grads):
        assert got.dtype == want.dtype and O.rel_l2(got.float(), want.float()) < 2e-2        # bfloat16, see above


def test_pooling_with_a_tensor_for_eps():
    """clamp() takes a tensor too; such a bound is left to torch."""
    torch.manual_seed(4)
    pool = models.AttentiveStatisticsPooling(64, 32).cuda()
    x, d, results = torch.randn(3, 64, 50).to("cuda", torch.bfloat16).requires_grad_(True), torch.randn(3, 128).cuda(), []
    for eps in (1e-3, torch.tensor(1e-3, device="cuda")):
        pool.eps = eps
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = pool(x)
        results.append((out, torch.autograd.grad(out, x, d)[0]))
    for got, want in zip(*results):
        assert O.rel_l2(got.float(), want.float()) < 2e-2


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,c,t", [(2, 16, 9), (3, 72, 100)])
def test_pooling_nodes_where_the_variance_is_bounded(n, c, t, dtype):
    """Rows that are constant over T, as a dead channel's, and rows whose variance lies on either side of a bound that 16 bits can
    hold: no gradient comes through a bounded deviation.  Against 64 bits; rows whose variance is within the rounding of the
    bound are none here."""
    gen, eps = torch.Generator().manual_seed(n * c), 2.0 ** -6
    size = torch.tensor([0.0, 0.03, 1.0, 0.5])[torch.arange(c) % 4].view(1, c, 1)             # variances 0, 2^-10, 1, 2^-2
    x = (torch.randn(n, c, 1, generator=gen) + size * torch.randn(n, c, t, generator=gen)).to("cuda", dtype).requires_grad_(True)
    z = (0.1 * torch.randn(n, c, t, generator=gen)).to("cuda", dtype).requires_grad_(True)
    d1, d2 = torch.randn(n, 3 * c, t, generator=gen).to("cuda", dtype), torch.randn(n, 2 * c, generator=gen).cuda()
    with torch.autocast("cuda", dtype=dtype):
        got, out = train.pooling_context(x, eps), train.pooled(z, x, eps)
    assert "Context" in type(got.grad_fn).__name__ and "Pooled" in type(out.grad_fn).__name__
    xe, ze = (v.detach().double().requires_grad_(True) for v in (x, z))
    bounded = (train.context_of(xe, eps)[1] < eps).view(n, c)
    assert torch.equal(bounded, (torch.arange(c, device="cuda") % 4 < 2).expand(n, c))
    grads = torch.autograd.grad(got, x, d1) + torch.autograd.grad(out, (x, z), d2)
    exact = torch.autograd.grad(train.context_of(xe, eps)[0], xe, d1.double()) + torch.autograd.grad(train.pooled_of(ze, xe, eps), (xe, ze), d2.double())
    for g, e in zip(grads, exact):
        for rows in (bounded, ~bounded):
            assert O.rel_l2(g[rows].float(), e[rows].float()) < (1e-2 if dtype == torch.bfloat16 else 1.5e-3)
