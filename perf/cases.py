"""The work that users of na1d_amd give it, as cases for timing: attention layers called by themselves (inference and
training, through each of the public entry points) and the two speaker-embedding models around them.

A case is a dict of plain values with a "kind":

  fused    na1d_fused on split heads [batch * heads, T, head_dim]
  qkv      na1d_fused_qkv on a projection's output [batch, T, 3, heads, head_dim]
  twocall  the reference's own chain, QK -> + bias -> + mask -> softmax -> AV, through getNA1dFunction
  dense    global_attention, the models' layers without a window
  infer    a model's forward pass under autocast; with "graph" replayed by GraphedInference
  train    a model's training step in fp16: forward, margin loss, backward, scaled and applied by SGD

"train" of an attention case says that the pass runs its backward too and returns the gradients.  "lens" says that the
sequences of a batch have lengths of their own, uniform over 15 to 100 % of the longest.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("pcf-nat_amd"))

from na1d_amd import models, na1d_fused, na1d_fused_qkv  # noqa: E402
from na1d_amd.dense import global_attention  # noqa: E402
from na1d_amd.graphs import GraphedInference  # noqa: E402
from na1d_amd.nattn import getNA1dFunction  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
CLASSES = 5994          # speakers of the training set (VoxCeleb2)
MOST_ELEMENTS = 14_000_000       # batch * heads * T * head_dim of a drawn attention case
MOST_TOKENS = 26_000             # batch * T of a drawn model pass
MOST_TRAIN_TOKENS = 12_800


def _attention(name, kind, dtype, batch, heads, T, head_dim, window, train, lens=False, dilation=1, dropout=0.0):
    return {"name": name, "kind": kind, "dtype": dtype, "batch": batch, "heads": heads, "T": T, "head_dim": head_dim,
            "window": window, "train": train, "lens": lens, "dilation": dilation, "dropout": dropout}


def _model(name, kind, model, dtype, batch, frames, lens=False, graph=False):
    return {"name": name, "kind": kind, "model": model, "dtype": dtype, "batch": batch, "frames": frames, "lens": lens,
            "graph": graph}


def listed():
    return [
        # one windowed layer for one 2 s utterance, as an online service calls it: nothing but latency
        _attention("layer_one_utterance", "qkv", "bf16", 1, 16, 100, 16, 27, False),
        # a short-window layer of wide heads in inference, on heads that the caller has split
        _attention("layer_split_heads", "fused", "bf16", 32, 4, 200, 64, 7, False),
        # forward and backward of a windowed layer at a training batch: the operator's headline size
        _attention("layer_train", "fused", "fp16", 128, 8, 300, 32, 15, True),
        # the same on the projection's layout at the models' training size: 128 crops of 2 s, 16 heads
        _attention("layer_train_in_place", "qkv", "fp16", 128, 16, 100, 16, 27, True),
        # code written for the reference's two-call operator, unchanged: scores in memory, softmax by torch
        _attention("layer_train_two_calls", "twocall", "bf16", 64, 16, 100, 16, 27, True),
        # a wide window over 3 s crops
        _attention("layer_train_wide", "fused", "bf16", 128, 8, 300, 32, 65, True),
        # everything odd at once: heads of 48 channels, an even window, dilation, dropout, lengths
        _attention("layer_train_ragged", "fused", "fp16", 37, 6, 333, 48, 20, True, lens=True, dilation=2, dropout=0.1),
        # training through a layer without a window over 20 s utterances of different lengths
        _attention("dense_train_long", "dense", "bf16", 64, 4, 1000, 64, 0, True, lens=True),
        # one 3 s utterance through the whole model, replayed from a graph: enrolment and verification online
        _model("embed_one_utterance", "infer", "pcf4x4", "bf16", 1, 300, graph=True),
        # bulk extraction of embeddings from 2 s crops
        _model("embed_batch", "infer", "pcf4x4", "bf16", 256, 200),
        # evaluation over whole utterances of 3 to 20 s, padded to the longest, with the deeper model
        _model("embed_long_utterances", "infer", "pcf6x4", "bf16", 64, 2000, lens=True),
        # a training step of the tokens-first model at its batch size
        _model("train_step", "train", "mfa4x4", "fp16", 128, 200),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fused", "fused", "qkv", "qkv", "twocall", "dense", "infer", "infer", "train"])
    dtype = rng.choice(["bf16", "fp16"]) if kind != "train" else "fp16"
    if kind == "infer":
        graph = rng.random() < 0.4
        model = rng.choice(["pcf4x4", "pcf6x4", "mfa4x4"])
        frames = _log(rng, 150, 2000)
        most = max(1, MOST_TOKENS // (frames // 2))
        batch = _log(rng, 1, min(8, most)) if graph else _log(rng, 2, min(256, most))
        case = _model("", kind, model, dtype, batch, frames, lens=rng.random() < 0.5, graph=graph)
    elif kind == "train":
        frames = rng.choice([200, 200, 300])
        case = _model("", kind, rng.choice(["pcf4x4", "mfa4x4"]), dtype, _log(rng, 16, MOST_TRAIN_TOKENS // (frames // 2)), frames)
    elif kind == "dense":
        head_dim, heads = 8 * rng.randint(4, 16), rng.randint(1, 8)
        T = _log(rng, 40, 1500)
        batch = _log(rng, 1, max(1, min(256, MOST_ELEMENTS // (heads * T * head_dim), int(2.6e8 // (heads * T * T)))))
        case = _attention("", kind, dtype, batch, heads, T, head_dim, 0, rng.random() < 0.6, lens=rng.random() < 0.5)
    else:
        head_dim, heads = 8 * rng.randint(1, 16) if rng.random() < 0.5 else rng.choice([16, 32, 64]), rng.randint(1, 16)
        T = _log(rng, 20, 2000)
        batch = _log(rng, 1, max(1, min(512, MOST_ELEMENTS // (heads * T * head_dim))))
        window = rng.randint(3, 32) if rng.random() < 0.75 else rng.randint(33, 80)
        train = rng.random() < 0.6
        fused = kind != "twocall"
        case = _attention("", kind, dtype, batch, heads, T, head_dim, window, train, lens=fused and rng.random() < 0.4,
                          dilation=rng.choice([1, 1, 1, 2, 3]) if fused else 1,
                          dropout=0.1 if fused and train and rng.random() < 0.3 else 0.0)
    del case["name"]
    return case


# ------------------------------------------------------------------------------------------------ preparation
def _lengths(n, longest, gen):
    """n lengths, uniform over 15 to 100 % of the longest, which is among them."""
    lens = (longest * (0.15 + 0.85 * torch.rand(n, generator=gen))).round().long().clamp(1, longest)
    lens[0] = longest
    return lens


def _prepare_attention(case, gen, dev):
    N, H, T, C, W = case["batch"], case["heads"], case["T"], case["head_dim"], case["window"]
    dtype, kind = DTYPES[case["dtype"]], case["kind"]
    host = torch.Generator().manual_seed(gen.initial_seed())

    def rows(*shape):
        return torch.randn(shape, generator=gen, device=dev).to(dtype)

    s = {"kind": kind, "case": case, "t_valid": _lengths(N, T, host).to(dev, torch.int32) if case["lens"] else None}
    if kind != "dense":
        s["rpb"] = 0.1 * torch.randn(H, W, generator=gen, device=dev)
        s["left"] = W - 1 - W // 2
    s["dropout_seed"] = int(torch.randint(0, 2 ** 62, (1,), generator=host))
    s["scale"] = C ** -0.5
    if kind == "qkv":
        s["qkv"] = rows(N, T, 3, H, C)
        s["dout"] = rows(N, T, H * C) if case["train"] else None
        leaves = ["qkv", "rpb"]
    else:
        s["q"], s["k"], s["v"] = (rows(N * H, T, C) for _ in range(3))
        if kind != "dense":
            s["q"] *= s["scale"]                       # as the models hand it over
        s["dout"] = rows(N * H, T, C) if case["train"] else None
        leaves = ["q", "k", "v"] + (["rpb"] if kind != "dense" else [])
    if kind == "twocall":
        s["QK"], s["AV"] = getNA1dFunction(C, 1, dtype)
        t, j = torch.arange(T, device=dev).unsqueeze(1), torch.arange(W, device=dev)
        key = t + j - s["left"]
        s["mask"] = torch.zeros(T, W, device=dev).masked_fill((key < 0) | (key >= T), models.MASK_VALUE)
    if case["train"]:
        for name in leaves:
            s[name].requires_grad_(True)
    s["leaves"] = leaves
    return s


def _flat_weights(modules, dev):
    """The modules' weights and running statistics moved into one buffer, each on a 256-byte boundary: what is
    written to a checkpoint in one piece."""
    kept = [t for m in modules for t in m.parameters()]
    kept += [t for m in modules for name, t in m.named_buffers() if "running_" in name]
    flat = torch.zeros(sum(-(-t.numel() // 64) * 64 for t in kept), device=dev)
    at = 0
    for t in kept:
        t.data = flat[at:at + t.numel()].view(t.shape).copy_(t.data)
        at += -(-t.numel() // 64) * 64
    return flat


def _prepare_model(case, gen, dev):
    dtype, frames, batch = DTYPES[case["dtype"]], case["frames"], case["batch"]
    factory = {"pcf4x4": models.PCF_NATransformer, "pcf6x4": models.pcf_nat_6x4, "mfa4x4": models.MFA_NATransformer}[case["model"]]
    host = torch.Generator().manual_seed(gen.initial_seed())
    torch.manual_seed(gen.initial_seed())
    with torch.device(dev):
        model = factory(na="fused_qkv", dtype=dtype, frames=frames if case["kind"] == "train" else 300)
    model = model.to(dev)
    s = {"kind": case["kind"], "dtype": dtype, "model": model, "lens": None}
    x = torch.randn(batch, 80, frames, generator=gen, device=dev)          # log mel energies, mean taken off over time
    x -= x.mean(-1, keepdim=True)
    if case["kind"] == "train":
        with torch.device(dev):
            s["head"] = models.ArcMarginSubCenters(192, CLASSES, m=0.2, s=32.0, subcenters=3)
        model.train()
        s["labels"] = torch.randint(0, CLASSES, (batch,), generator=gen, device=dev)
        s["weights"] = _flat_weights([model, s["head"]], dev)
        s["optimizer"] = torch.optim.SGD([*model.parameters(), *s["head"].parameters()], lr=0.01, momentum=0.9, nesterov=True)
        s["scaler"] = torch.amp.GradScaler("cuda", init_scale=1024.0)
    else:
        with torch.no_grad():                                              # statistics as training leaves them
            for name, t in model.state_dict().items():
                if name.endswith("running_mean"):
                    t.copy_(0.1 * torch.randn(t.shape, generator=gen, device=dev))
                if name.endswith("running_var"):
                    t.copy_(0.75 + 0.5 * torch.rand(t.shape, generator=gen, device=dev))
        model.eval()
        if case["lens"]:
            lens = _lengths(batch, frames, host)
            x *= (torch.arange(frames).unsqueeze(0) < lens.unsqueeze(1)).to(dev).unsqueeze(1)
            s["lens"] = (lens.float() / frames).to(dev)
    s["x"] = x
    if case.get("graph"):
        s["graph"] = GraphedInference(model, x, s["lens"], autocast=dtype)
    return s


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    return (_prepare_model if case["kind"] in ("infer", "train") else _prepare_attention)(case, gen, dev)


# ------------------------------------------------------------------------------------------------ one pass
def _run_attention(s):
    case, kind = s["case"], s["kind"]
    W = case["window"]
    with torch.set_grad_enabled(case["train"]):
        if kind == "qkv":
            out = na1d_fused_qkv(s["qkv"], W, s["left"], rpb=s["rpb"], t_valid=s["t_valid"], scale=s["scale"],
                                 dilation=case["dilation"], dropout_p=case["dropout"], seed=s["dropout_seed"])
        elif kind == "fused":
            out = na1d_fused(s["q"], s["k"], s["v"], W, s["left"], rpb=s["rpb"], t_valid=s["t_valid"],
                             num_heads=case["heads"], dilation=case["dilation"], dropout_p=case["dropout"],
                             seed=s["dropout_seed"])
        elif kind == "dense":
            out = global_attention(s["q"], s["k"], s["v"], case["heads"], t_valid=s["t_valid"], scale=s["scale"])
        else:
            N, H, T = case["batch"], case["heads"], case["T"]
            attn = s["QK"].apply(s["q"], s["k"], W, s["left"], 1).view(N, H, T, W)
            attn = attn + s["rpb"].view(1, H, 1, W) + s["mask"]
            out = s["AV"].apply(torch.softmax(attn.view(N * H, T, W), dim=-1), s["v"], W, s["left"], 1)
    if not case["train"]:
        return out
    return [out.detach(), *torch.autograd.grad(out, [s[name] for name in s["leaves"]], s["dout"])]


def _run_train(s):
    s["optimizer"].zero_grad()
    with torch.autocast("cuda", dtype=s["dtype"]):
        emb = s["model"](s["x"])
    loss, _ = s["head"](emb.float(), s["labels"])
    s["scaler"].scale(loss).backward()
    s["scaler"].step(s["optimizer"])
    s["scaler"].update()
    return {"loss": loss.detach(), "embeddings": emb.detach(), "weights": s["weights"]}


def run(state):
    if state["kind"] == "train":
        return _run_train(state)
    if state["kind"] != "infer":
        return _run_attention(state)
    if "graph" in state:
        return state["graph"](state["x"], state["lens"])
    with torch.no_grad(), torch.autocast("cuda", dtype=state["dtype"]):
        return state["model"](state["x"]) if state["lens"] is None else state["model"](state["x"], state["lens"])


# ------------------------------------------------------------------------------------------------ bounds and tolerances
GROUPED = (1 / 8 + 1 / 4 + 1 / 2 + 1) / 4      # of a dense projection's weights: PCF-NAT's blocks have 8, 4, 2, 1 groups
MODELS = {"pcf4x4": (14, 2, 4, GROUPED), "pcf6x4": (22, 2, 4, GROUPED), "mfa4x4": (14, 2, 1, 1.0)}   # layers with and without a window, patch embeddings, share


def work(case):
    if case["kind"] in ("infer", "train"):
        windowed, dense, embeds, share = MODELS[case["model"]]
        n, T, dim, blocks, wide, pool, emb = case["batch"], case["frames"] // 2, 256, 4, 1536, 128, 192
        layers = windowed + dense
        grouped = share * ((layers * 12 + dense) * dim * dim + embeds * 160 * dim)
        per_token = grouped + windowed * 2 * 27 * dim + dense * 2 * T * dim + blocks * dim * wide + 2 * wide * pool
        weights = grouped + blocks * dim * wide + 4 * wide * pool + 2 * wide * emb
        flops = 2.0 * (n * T * per_token + n * (2 * wide * pool + 2 * wide * emb))
        nbytes = 4.0 * n * 80 * case["frames"] + 4.0 * weights + 4.0 * n * emb
        if case["kind"] == "train":
            head = CLASSES * 3 * emb
            flops = 3 * (flops + 2.0 * n * head)
            nbytes += 4.0 * (2 * head + weights)                  # the loss head's weights, and every gradient written
        return {"bytes": nbytes, "flops": flops}
    rows = case["batch"] * case["heads"] * case["T"]
    C, keys = case["head_dim"], case["window"] or case["T"]
    tensors = 8 if case["train"] else 4                              # q k v -> out; with dout -> dq dk dv too
    nbytes, flops = 2.0 * tensors * rows * C, 4.0 * rows * keys * C
    if case["train"]:
        flops *= 3
    if case["kind"] == "twocall":                                    # the scores between the two calls are the caller's
        nbytes += 4.0 * rows * keys * (8 if case["train"] else 2)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what each path measures against itself in 64 bits (attention) or 32 (models), over seeds and
    sizes: attention 2.5e-3 / 3e-4 in norm and 2e-2 / 5e-3 at worst (bf16 / fp16), embeddings 5e-3 / 6e-4 and
    2e-2 / 2e-3; a training step's embeddings 2e-3 and 1e-2, its weights 3e-4 and 7e-2 (batch statistics amplify the rounding of 16
    layers, and single gradients are what is left of large sums that cancel)."""
    bf16 = case["dtype"] == "bf16"
    if case["kind"] == "train":
        return {"rel": 1e-2, "max": 0.3}
    if case["kind"] == "infer":
        return {"rel": 2e-2, "max": 0.1} if bf16 else {"rel": 2.5e-3, "max": 0.012}
    return {"rel": 1e-2, "max": 0.1} if bf16 else {"rel": 1.2e-3, "max": 0.02}
