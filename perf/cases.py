"""The work that a user of this framework has it do, as cases that can be timed.

What a program calls, once per training iteration or once per matrix:

  train  `clip_grad_norm_` over the model's parameters, then `Muon.step()`: the 2-D weights of the layers in a Muon
         group, embedding, head and norm vectors in an AdamW group
  adam   `Muon.step()` of an AdamW group alone (embedding, head, norm vectors)
  ns     `fast_newtonschulz` of one matrix, or of a stack of same-shape matrices
  mmt    `matmul_transpose` of one matrix

`listed()` holds one case for each thing such programs are, from a toy model to the layers of a large one; `draw()` gives
more of the same ranges.  Gradients carry a per-row scale on top of normal noise, and momentum and Adam moments are those
of a run under way.  Tensors of one shape lie in one buffer (each at a 512-byte boundary, as an allocator puts them), so
that `run` can return every updated tensor whole.
"""
import math

import torch

from lmms_engine_amd.clip_grad import clip_grad_norm_
from lmms_engine_amd.muon_utils import Muon, fast_newtonschulz, matmul_transpose

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
SIZES = {"f32": 4, "bf16": 2}
TRAIN = dict(kind="train", attn=0, kv=0, inter=0, experts=0, expert_inter=0, rank=0, vocab=0, tied=False, max_norm=1.0,
             grad_norm=2.0, rms_scale=False, nesterov=True, lr=0.02)


def listed():
    return [
        # a toy model: what a unit test or a first script steps; launches and host time are all of it
        dict(TRAIN, name="train_toy", layers=2, hidden=128, attn=128, kv=64, inter=384, vocab=512, dtype="f32", momentum="f32"),
        # a small language model in bf16 that trains all of its parameters, the reference constructor's rms_scale default
        dict(TRAIN, name="train_small", layers=8, hidden=512, attn=512, kv=256, inter=1408, vocab=32000, tied=True, dtype="bf16",
             momentum="f32", rms_scale=True, lr=2e-3, grad_norm=0.5),
        # sizes that are no whole number of anything, bf16 momentum (the reference's own layout), plain momentum
        dict(TRAIN, name="train_ragged", layers=6, hidden=1000, attn=1000, kv=200, inter=2731, vocab=10007, dtype="bf16",
             momentum="bf16", rms_scale=True, nesterov=False, lr=2e-3, grad_norm=5.0),
        # low-rank adapters beside frozen weights: every matrix has a short side of 16
        dict(TRAIN, name="train_adapters", layers=28, hidden=2048, attn=2048, kv=512, inter=5632, rank=16, dtype="f32",
             momentum="f32", grad_norm=0.3),
        # all 24 layers of the Qwen2.5-0.5B-shaped set in fp32, with its tied embedding
        dict(TRAIN, name="train_qwen2.5_0.5b", layers=24, hidden=896, attn=896, kv=128, inter=4864, vocab=151936, tied=True,
             dtype="f32", momentum="f32", grad_norm=0.8),
        # a third of the layers of the Qwen3-8B-shaped set: bf16 parameters and gradients, fp32 momentum
        dict(TRAIN, name="train_qwen3_8b", layers=12, hidden=4096, attn=4096, kv=1024, inter=12288, dtype="bf16", momentum="f32",
             grad_norm=2.0),
        # layers of the Qwen3-MoE-30B-A3B-shaped set: 128 experts each, thousands of small matrices
        dict(TRAIN, name="train_qwen3_moe", layers=4, hidden=2048, attn=4096, kv=512, experts=128, expert_inter=768, dtype="bf16",
             momentum="f32", grad_norm=0.6),
        # embedding, head and 73 norm vectors of a Qwen3-8B-shaped model in the AdamW group
        dict(kind="adam", name="adam_embeddings", vocab=151936, hidden=4096, tied=False, vectors=73, dtype="bf16"),
        # one MLP matrix of a small model, orthogonalised on its own
        dict(kind="ns", name="ns_896x4864", rows=896, cols=4864, batch=0, dtype="f32"),
        # a large square matrix on its own
        dict(kind="ns", name="ns_8192x8192", rows=8192, cols=8192, batch=0, dtype="bf16"),
        # a stack of small matrices, taller than wide
        dict(kind="ns", name="ns_stack_48x1024x256", rows=1024, cols=256, batch=48, dtype="bf16"),
        # the symmetric product on its own
        dict(kind="mmt", name="mmt_2048x5632", rows=2048, cols=5632, dtype="bf16"),
    ]


# What a drawn case may cost, below the largest listed one whatever rate its shapes run at.
MOST_FLOPS, MOST_ELEMENTS = 4e13, 6e8


def draw(rng):
    def size(lo, hi):
        """Log-uniform; half of the sizes are whole multiples of what hardware likes, the others are what they are."""
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        step = rng.choice([1, 1, 1, 16, 64, 128])
        return max(lo, int(round(v / step)) * step)

    while True:
        kind = rng.choice(["train", "train", "train", "train", "ns", "ns", "adam", "mmt"])
        dtype = rng.choice(["f32", "bf16"])
        if kind == "train":
            hidden = size(64, 4096)
            case = dict(TRAIN, layers=int(math.exp(rng.uniform(0.0, math.log(28.5)))), hidden=hidden, attn=hidden,
                        kv=max(16, hidden // rng.choice([1, 2, 4, 8])), inter=size(hidden, 4 * hidden),
                        vocab=rng.choice([0, size(256, 50000)]), tied=rng.random() < 0.5, dtype=dtype,
                        momentum="f32" if dtype == "f32" else rng.choice(["f32", "bf16"]), rms_scale=rng.random() < 0.5,
                        nesterov=rng.random() < 0.8, grad_norm=round(math.exp(rng.uniform(math.log(0.1), math.log(10.0))), 3))
            case["lr"] = 2e-3 if case["rms_scale"] else 0.02
            flavour = rng.choice(["dense", "dense", "dense", "experts", "adapters"])
            if flavour == "experts":
                case.update(inter=0, experts=rng.choice([8, 16, 32, 64, 128]), expert_inter=size(64, 2 * hidden))
            elif flavour == "adapters":
                case.update(rank=rng.choice([4, 8, 16, 24, 32, 64]))
        elif kind == "ns":
            batch = rng.choice([0, 0, int(math.exp(rng.uniform(math.log(2), math.log(200))))])
            case = dict(kind="ns", rows=size(16, 8192), cols=size(16, 8192), batch=batch, dtype=dtype)
        elif kind == "adam":
            case = dict(kind="adam", vocab=size(512, 160000), hidden=size(64, 4096), tied=rng.random() < 0.5,
                        vectors=rng.randint(1, 120), dtype=dtype)
        else:
            case = dict(kind="mmt", rows=size(64, 8192), cols=size(64, 16384), dtype="bf16")
        elements = sum(n * math.prod(s) for n, s in muon_shapes(case) + adam_shapes(case))
        if elements <= MOST_ELEMENTS and work(case)["flops"] <= MOST_FLOPS:
            return case


def muon_shapes(case):
    """[(count, (rows, cols))] of the matrices a case orthogonalises (or multiplies), equal shapes together."""
    if case["kind"] in ("ns", "mmt"):
        return [(case.get("batch") or 1, (case["rows"], case["cols"]))]
    if case["kind"] == "adam":
        return []
    h, L = case["hidden"], case["layers"]
    linears = [(case["attn"], h, 1), (case["kv"], h, 2), (h, case["attn"], 1)]  # q, k and v, o as (out, in, how many)
    if case["inter"]:
        linears += [(case["inter"], h, 2), (h, case["inter"], 1)]  # gate and up, down
    if case["experts"]:
        linears += [(case["expert_inter"], h, 2 * case["experts"]), (h, case["expert_inter"], case["experts"])]
    counts = {}
    for out, inp, n in linears:
        r = case["rank"]
        for s in [(r, inp), (out, r)] if r else [(out, inp)]:
            counts[s] = counts.get(s, 0) + n * L
    return [(n, s) for s, n in counts.items()]


def adam_shapes(case):
    if case["kind"] == "adam":
        return [(1 if case["tied"] else 2, (case["vocab"], case["hidden"])), (case["vectors"], (case["hidden"],))]
    if case["kind"] == "train" and case["vocab"]:
        return [(1 if case["tied"] else 2, (case["vocab"], case["hidden"])), (2 * case["layers"] + 1, (case["hidden"],))]
    return []


class Tensors:
    """`n` tensors of one shape in one buffer, each at a multiple of 512 bytes."""

    def __init__(self, n, shape, dtype, fill):
        numel = math.prod(shape)
        self.buf = torch.zeros(n, -(-numel // 256) * 256, dtype=dtype, device="cuda")
        self.each = [self.buf[i, :numel].view(shape) for i in range(n)]
        for t in self.each:
            t.copy_(fill(shape))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(scale):
        return lambda shape: torch.randn(shape, device="cuda", generator=gen) * scale

    def gradient(scale):
        def fill(shape):
            rows = torch.exp(0.5 * torch.randn(shape[0], *([1] * (len(shape) - 1)), device="cuda", generator=gen) - 0.25)
            return torch.randn(shape, device="cuda", generator=gen) * rows * scale
        return fill

    dt = DTYPES[case["dtype"]]
    if case["kind"] in ("ns", "mmt"):
        shape = (case["rows"], case["cols"])
        g = gradient(1e-3)(shape) if not case.get("batch") else torch.stack([gradient(1e-3)(shape) for _ in range(case["batch"])])
        return {"case": case, "g": g.to(dt)}
    muon, adam = muon_shapes(case), adam_shapes(case)
    total = sum(n * math.prod(s) for n, s in muon + adam)
    g_scale = case.get("grad_norm", 1.0) / math.sqrt(total)  # the rows' scales have mean square 1
    groups, out, params, state = [], {}, [], {}
    if muon:
        md = DTYPES[case["momentum"]]
        mats = []
        for n, s in muon:
            key = "%dx%d" % s
            w, g = Tensors(n, s, dt, normal(0.02)), Tensors(n, s, dt, gradient(g_scale))
            m = Tensors(n, s, md, gradient(0.5 * g_scale))
            out["p" + key], out["g" + key], out["m" + key] = w.buf, g.buf, m.buf
            for wi, gi, mi in zip(w.each, g.each, m.each):
                p = torch.nn.Parameter(wi)
                p.grad = gi
                state[p] = {"momentum_buffer": mi}
                mats.append(p)
        groups.append(dict(params=mats, use_muon=True, lr=case["lr"], momentum=0.95, weight_decay=0.01, rms_scale=case["rms_scale"],
                           nesterov=case["nesterov"], ns_steps=5))
        params += mats
    if adam:
        rest = []
        for n, s in adam:
            key = "x".join(str(d) for d in s)
            w, g = Tensors(n, s, dt, normal(0.02)), Tensors(n, s, dt, gradient(g_scale))
            e1, e2 = Tensors(n, s, dt, normal(0.3 * g_scale)), Tensors(n, s, dt, lambda shape: normal(g_scale)(shape).square())
            out["ap" + key], out["ag" + key], out["ae" + key], out["as" + key] = w.buf, g.buf, e1.buf, e2.buf
            for wi, gi, ai, bi in zip(w.each, g.each, e1.each, e2.each):
                p = torch.nn.Parameter(wi)
                p.grad = gi
                state[p] = {"exp_avg": ai, "exp_avg_sq": bi, "step": 100}
                rest.append(p)
        groups.append(dict(params=rest, use_muon=False, lr=3e-4, betas=(0.9, 0.95), eps=1e-8, weight_decay=0.01))
        params += rest
    opt = Muon(groups, momentum_dtype=DTYPES[case["momentum"]] if muon else None)
    opt.state.update(state)
    return {"case": case, "opt": opt, "params": params, "out": out}


def run(state):
    case = state["case"]
    if case["kind"] == "ns":
        return fast_newtonschulz(state["g"], 5)
    if case["kind"] == "mmt":
        return matmul_transpose(state["g"])
    if case["kind"] == "adam":
        state["opt"].step()
        return state["out"]
    total = clip_grad_norm_(state["params"], case["max_norm"])
    state["opt"].step()
    return {"total_norm": total, **state["out"]}


def work(case):
    e = SIZES[case["dtype"]]
    muon, adam = muon_shapes(case), adam_shapes(case)
    n_muon, n_adam = (sum(n * math.prod(s) for n, s in shapes) for shapes in (muon, adam))
    if case["kind"] == "mmt":
        M, K = case["rows"], case["cols"]
        return {"bytes": (M * K + M * M) * e, "flops": float(M) * M * K}  # a symmetric result: half of the dense product
    flops = sum(n * 5 * (3.0 * min(s) ** 2 * max(s) + float(min(s)) ** 3) for n, s in muon)
    if case["kind"] == "ns":
        return {"bytes": n_muon * (e + 2), "flops": flops}
    # gradients in (and out, where they are clipped), parameters, momentum or both Adam moments in and out
    clipped = case["kind"] == "train" and case["grad_norm"] > case["max_norm"]
    bytes_ = (n_muon + n_adam) * e * (2 if clipped else 1) + n_muon * 2 * (e + (SIZES[case["momentum"]] if muon else 0)) + n_adam * 6 * e
    return {"bytes": bytes_, "flops": flops + 12.0 * n_adam}


def tolerance(case):
    """About four times what the path differs from itself by when its fp32 sums run in another order (and from fp64, for the
    single product).  A sum that falls on the other side of a bf16 rounding point moves through five iterations: 0.7 to 1.1 %
    of an orthogonalised matrix, 0.02 to 0.1 % of the parameter it updates; a bf16 gradient norm that falls on the neighbouring
    value moves every clipped gradient by 0.4 %."""
    bf16 = case["dtype"] == "bf16"
    if case["kind"] == "mmt":
        return {"rel": 4e-3, "max": 0.016}
    if case["kind"] == "ns":
        return {"rel": 3e-2, "max": 0.6}
    if case["kind"] == "adam":
        return {"rel": 2e-3, "max": 0.016} if bf16 else {"rel": 1e-5, "max": 1e-4}
    return {"rel": 5e-3, "max": 0.05} if bf16 else {"rel": 3e-3, "max": 0.08}
