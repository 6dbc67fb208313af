"""Performance cases of the llama-zero training framework on one MI355X.

listed() names the calls that stand for the framework's use: single layers of
the model presets (model/config.py) as its training and inference programs
call them, one whole forward + backward, one whole forward and one optimizer
step.  draw() gives more of the same ranges.  prepare() builds what a program
holds before the call (module, inputs, output gradient), run() makes one call
through the public modules and engines, exact() restates it in float64.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "cs244c-llama-zero_amd")
if os.path.abspath(_PKG) not in [os.path.abspath(p) for p in sys.path]:
    sys.path.insert(0, os.path.abspath(_PKG))

from lzhip import functional as LF  # noqa: E402
from model import LlamaForCausalLM, build_config  # noqa: E402
from model.llama import GroupedQueryAttention, HipLMHead, RMSNorm, SwiGLU  # noqa: E402
from zero import ZeROStage1Optimizer  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = ("plumbing", "tiny", "125m", "small", "medium", "1b", "7b")
DEV = "cuda"


def listed():
    return [
        # the smallest layer of a step: the pre-norm of train.py's default
        # model (tiny, batch 2 x 512, bf16), forward and backward
        {"name": "norm_tiny", "kind": "norm", "size": "tiny", "dtype": "bf16", "batch": 2, "seq": 512},
        # train.py's defaults: tiny, batch 2, seq 512, bf16
        {"name": "attn_tiny", "kind": "attn", "size": "tiny", "dtype": "bf16", "batch": 2, "seq": 512,
         "train": True, "mask": ""},
        # train_zero.py's defaults: the same model and batch in float32
        {"name": "attn_tiny_fp32", "kind": "attn", "size": "tiny", "dtype": "fp32", "batch": 2, "seq": 512,
         "train": True, "mask": ""},
        # the headline benchmark's attention layer (1B, batch 8 x 2048)
        {"name": "attn_1b", "kind": "attn", "size": "1b", "dtype": "bf16", "batch": 8, "seq": 2048,
         "train": True, "mask": ""},
        # training on a padded batch: attention_mask given, 125M model
        {"name": "attn_125m_padded", "kind": "attn", "size": "125m", "dtype": "bf16", "batch": 4, "seq": 500,
         "train": True, "mask": "padding"},
        # one generate() step's attention layer: a prompt of odd length, no gradients
        {"name": "attn_1b_prompt", "kind": "attn", "size": "1b", "dtype": "bf16", "batch": 1, "seq": 777,
         "train": False, "mask": ""},
        # the headline benchmark's MLP
        {"name": "mlp_1b", "kind": "mlp", "size": "1b", "dtype": "bf16", "batch": 8, "seq": 2048, "train": True},
        # train.py --dtype float16 on a ragged batch of the small preset
        {"name": "mlp_small_fp16", "kind": "mlp", "size": "small", "dtype": "fp16", "batch": 3, "seq": 341,
         "train": True},
        # the 125M benchmark's LM head and loss (batch 16 x 1024, vocab 32000)
        {"name": "head_125m", "kind": "head", "size": "125m", "dtype": "bf16", "batch": 16, "seq": 1024,
         "vocab": 32000},
        # train_zero.py's default model, whole: forward, loss and every gradient
        {"name": "model_tiny_fp32", "kind": "model", "size": "tiny", "dtype": "fp32", "batch": 2, "seq": 512,
         "vocab": 8192, "train": True},
        # one generate() step of the 125M model: logits of a prompt of odd length
        {"name": "model_125m_prompt", "kind": "model", "size": "125m", "dtype": "bf16", "batch": 1, "seq": 333,
         "vocab": 32000, "train": False},
        # the optimizer step of the 125M ZeRO-1 benchmark, with clipping
        {"name": "step_125m", "kind": "step", "size": "125m", "dtype": "bf16", "vocab": 32000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# Work limits of a drawn case: below the largest listed one, and for the
# precisions and options whose arithmetic runs slower, below that by as much.
_MOST_FLOPS = {"bf16": 2.0e12, "fp16": 1.0e12, "fp32": 1.5e11}


def draw(rng):
    while True:
        kind = rng.choice(["norm", "attn", "attn", "attn", "mlp", "mlp", "head", "model", "step"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32", "fp16"])
        case = {"kind": kind, "size": rng.choice(SIZES[:-1]), "dtype": dtype}
        case["batch"] = _log_int(rng, 1, 16)
        # half of the sequence lengths are whole blocks, half are what a text gives
        case["seq"] = _log_int(rng, 24, 2048)
        if rng.random() < 0.5:
            case["seq"] = max(64, case["seq"] // 64 * 64)
        if kind in ("norm", "attn", "mlp") and rng.random() < 0.15:
            case["size"] = "7b"
        if kind == "attn":
            case["train"] = rng.random() < 0.7
            case["mask"] = rng.choice(["", "", "padding", "additive"])
            if case["mask"] and (case["seq"] > 1024 or case["batch"] * case["seq"] > 4096):
                continue
        elif kind == "mlp":
            case["train"] = rng.random() < 0.7
        elif kind == "head":
            case["vocab"] = rng.choice([8192, 32000, 128256, _log_int(rng, 1000, 60000)])
            if case["dtype"] == "fp16":  # fp16 models return their logits; see "model"
                case["dtype"] = "bf16"
        elif kind == "model":
            case["size"] = rng.choice(["plumbing", "tiny", "125m"])
            case["train"] = case["size"] != "125m" and rng.random() < 0.6
            case["vocab"] = rng.choice([8192, 32000])
            case["batch"] = min(case["batch"], 4)
        elif kind == "step":
            case = {"kind": kind, "size": rng.choice(["plumbing", "tiny", "125m", "small"]),
                    "dtype": rng.choice(["bf16", "fp32"]), "vocab": rng.choice([8192, 32000, _log_int(rng, 1000, 60000)])}
        if work(case)["flops"] <= _MOST_FLOPS[case["dtype"]]:
            return case


def _config(case):
    return build_config(case["size"], vocab_size=case.get("vocab", 32000), max_seq_len=max(case.get("seq", 0), 2048))


def _randn(gen, *shape, dtype, std=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV) * std).to(dtype)


def _mask(case, gen):
    """[B, 1, S, S] causal mask that also hides the padding at each
    sequence's end (the first token is always kept)."""
    B, S = case["batch"], case["seq"]
    keep = torch.randint(max(1, S // 2), S + 1, (B,), generator=gen, device=DEV)
    if case["seq"] > 1:
        keep[0] = S
    pos = torch.arange(S, device=DEV)
    m = (pos[None, None, :] <= pos[None, :, None]) & (pos[None, None, :] < keep[:, None, None])
    m = m[:, None]
    if case["mask"] == "additive":
        low = torch.finfo(DTYPES[case["dtype"]]).min
        return torch.zeros(m.shape, dtype=DTYPES[case["dtype"]], device=DEV).masked_fill(~m, low)
    return m


def _init(module, gen, std=0.02):
    """The presets' initial weights (normal, 0.02; norms near one)."""
    for p in module.parameters():
        with torch.no_grad():
            if p.dim() == 1:
                p.copy_(1.0 + 0.1 * torch.randn(p.shape, generator=gen, device=DEV))
            else:
                p.copy_(torch.randn(p.shape, generator=gen, device=DEV) * std)
    return module


def prepare(case, seed):
    kind, dtype, cfg = case["kind"], DTYPES[case["dtype"]], _config(case)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    B, S, d = case.get("batch"), case.get("seq"), cfg.dim
    state = {"case": dict(case)}
    with torch.device(DEV):
        if kind == "norm":
            module = RMSNorm(d, cfg.rms_norm_eps)
        elif kind == "attn":
            module = GroupedQueryAttention(cfg)
        elif kind == "mlp":
            module = SwiGLU(cfg)
        elif kind == "head":
            module = HipLMHead(d, cfg.vocab_size, bias=False)
        else:
            module = LlamaForCausalLM(cfg)
    module = _init(module, gen).to(dtype)
    LF.pack_parameters_(module)  # as train.py does; the ZeRO engines lay parameters out alike
    state["module"] = module
    state["params"] = list(module.parameters())
    if kind == "step":
        engine = ZeROStage1Optimizer(module, lr=3e-4)
        for p in module.parameters():
            p.grad = _randn(gen, *p.shape, dtype=dtype, std=1e-3)
        state["engine"] = engine
        # the engine keeps every parameter in one flat buffer, in this order
        state["flat"] = state["params"][0].detach().as_strided((sum(p.numel() for p in state["params"]),), (1,))
        return state
    if kind == "model":
        module.set_loss_chunk_size(128)
        state["ids"] = torch.randint(0, cfg.vocab_size, (B, S), generator=gen, device=DEV)
        module.train(case["train"])
        return state
    train = case.get("train", True)
    module.train(train)
    state["x"] = _randn(gen, B, S, d, dtype=dtype).requires_grad_(train)
    if kind == "attn":
        state["mask"] = _mask(case, gen) if case["mask"] else None
    if kind == "head":
        state["labels"] = torch.randint(0, cfg.vocab_size, (B, S), generator=gen, device=DEV)
    elif train:
        state["dy"] = _randn(gen, B, S, d, dtype=dtype, std=0.01)
    if kind == "norm":
        state["dres"] = _randn(gen, B, S, d, dtype=dtype, std=0.01)
    return state


def run(state):
    case = state["case"]
    kind, module = case["kind"], state["module"]
    if kind == "step":
        engine = state["engine"]
        norm = engine.step_with_stats(max_grad_norm=1.0)["grad_norm"]
        return {"norm": norm, "master": engine.local_master_param_shard, "exp_avg": engine.exp_avg,
                "exp_avg_sq": engine.exp_avg_sq, "params": state["flat"]}
    if kind == "model":
        if not case["train"]:
            with torch.no_grad():
                return module(state["ids"]).logits
        loss = module(input_ids=state["ids"], labels=state["ids"], return_logits=False).loss
        return [loss, torch.autograd.grad(loss, state["params"])]
    x = state["x"]
    if kind == "head":
        loss = module(x, state["labels"])
        return [loss, torch.autograd.grad(loss, [x] + state["params"])]
    if kind == "norm":
        # as the pre-norm block calls it: the norm and the residual branch
        y, res = module.forward_with_residual(x)
        return [y, torch.autograd.grad([y, res], [x] + state["params"], [state["dy"], state["dres"]])]
    args = (state["mask"],) if kind == "attn" else ()
    if not case["train"]:
        with torch.no_grad():
            return module(x, *args)
    y = module(x, *args)
    return [y, torch.autograd.grad(y, [x] + state["params"], state["dy"])]


def _block_weights(cfg):
    kv = cfg.n_kv_heads * cfg.head_dim
    return 2 * cfg.dim * cfg.dim + 2 * cfg.dim * kv, 3 * cfg.dim * cfg.ffn_dim


def work(case):
    """Each input read once, each output written once; products and attention
    pairs forward, and twice that backward."""
    cfg, e = _config(case), {"bf16": 2, "fp16": 2, "fp32": 4}[case["dtype"]]
    kind, B, S, d = case["kind"], case.get("batch", 0), case.get("seq", 0), cfg.dim
    T, V = B * S, cfg.vocab_size
    attn_w, mlp_w = _block_weights(cfg)
    pairs = B * cfg.n_heads * (S * S if case.get("mask") else S * (S + 1) // 2)
    if kind == "norm":
        return {"bytes": 5 * T * d * e, "flops": 12 * T * d}
    if kind == "step":
        n = V * d + cfg.n_layers * (attn_w + mlp_w + 2 * d) + d
        # gradient; master and both moments read and written; parameters written
        return {"bytes": n * (e + 6 * 4 + e), "flops": 20 * n}
    if kind == "attn":
        fl, w, io = 2 * T * attn_w + 4 * pairs * cfg.head_dim, attn_w, 2 * T * d
        io_mask = B * S * S * (1 if case["mask"] == "padding" else e) if case["mask"] else 0
    elif kind == "mlp":
        fl, w, io, io_mask = 2 * T * mlp_w, mlp_w, 2 * T * d, 0
    elif kind == "head":
        return {"bytes": (2 * T * d + 2 * V * d) * e, "flops": 6 * T * V * d}
    else:
        fl = cfg.n_layers * (2 * T * (attn_w + mlp_w) + 4 * pairs * cfg.head_dim) + 2 * T * V * d
        w, io, io_mask = V * d + cfg.n_layers * (attn_w + mlp_w), 0, 0
        if not case["train"]:
            io = T * V
    if case["train"]:
        return {"bytes": (2 * w + 2 * io) * e + io_mask, "flops": 3 * fl}
    return {"bytes": (w + io) * e + io_mask, "flops": fl}


def tolerance(case):
    kind, dtype = case["kind"], case["dtype"]
    if kind == "step":
        return {"rel": 1e-5} if dtype == "fp32" else {"rel": 1e-3}
    if kind == "model":
        return {"rel": {"bf16": 3e-2, "fp16": 8e-3, "fp32": 2e-5}[dtype]}
    return {"rel": {"bf16": 1.5e-2, "fp16": 2e-3, "fp32": 1e-5}[dtype]}


# ---------------------------------------------------------------------------
# the same calls in float64
# ---------------------------------------------------------------------------

def _rms_norm(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _rope_tables(cfg, S, dtype):
    """The model's cos/sin tables: positions and angles are formed in the
    parameter dtype (the inverse frequencies are a buffer of the module)."""
    hd = cfg.head_dim
    inv = (1.0 / (cfg.rope_theta ** (torch.arange(0, hd, 2).float() / hd))).to(dtype)
    ang = torch.outer(torch.arange(S, dtype=dtype), inv)
    ang = torch.cat((ang, ang), dim=-1)
    return ang.cos().to(DEV).double(), ang.sin().to(DEV).double()


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return x * cos + torch.cat((-b, a), dim=-1) * sin


def _attention(x, wq, wk, wv, wo, cfg, tables, mask):
    B, S, _ = x.shape
    hd, rep = cfg.head_dim, cfg.n_heads // cfg.n_kv_heads
    q = (x @ wq.T).view(B, S, cfg.n_heads, hd).transpose(1, 2)
    k = (x @ wk.T).view(B, S, cfg.n_kv_heads, hd).transpose(1, 2)
    v = (x @ wv.T).view(B, S, cfg.n_kv_heads, hd).transpose(1, 2)
    q, k = _rotate(q, *tables), _rotate(k, *tables)
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    s = (q @ k.transpose(-1, -2)) * hd**-0.5
    if mask is None:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=x.device).triu(1), -math.inf)
    elif mask.dtype == torch.bool:
        s = s.masked_fill(~mask, -math.inf)
    else:
        s = s + mask.double()
    y = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(B, S, -1)
    return y @ wo.T


def _mlp(x, wg, wu, wd):
    g = x @ wg.T
    return (g * torch.sigmoid(g) * (x @ wu.T)) @ wd.T


def _shifted_loss(logits, labels):
    return torch.nn.functional.cross_entropy(logits[:, :-1].reshape(-1, logits.shape[-1]), labels[:, 1:].reshape(-1))


def exact(case, seed):
    state, cfg, kind = prepare(case, seed), _config(case), case["kind"]
    if kind == "step":
        return _exact_step(state)
    P = [p.detach().double().requires_grad_() for p in state["params"]]
    S = case.get("seq")
    if kind == "model":
        by_name = dict(zip([n for n, _ in state["module"].named_parameters()], P))
        tables = _rope_tables(cfg, S, DTYPES[case["dtype"]])
        h = by_name["tok_embeddings.weight"][state["ids"]]
        for i in range(cfg.n_layers):
            W = {k: by_name[f"layers.{i}.{k}.weight"] for k in (
                "input_norm", "attn.q_proj", "attn.k_proj", "attn.v_proj", "attn.o_proj", "post_attn_norm",
                "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj")}
            n = _rms_norm(h, W["input_norm"], cfg.rms_norm_eps)
            h = h + _attention(n, W["attn.q_proj"], W["attn.k_proj"], W["attn.v_proj"], W["attn.o_proj"], cfg, tables,
                               None)
            n = _rms_norm(h, W["post_attn_norm"], cfg.rms_norm_eps)
            h = h + _mlp(n, W["mlp.gate_proj"], W["mlp.up_proj"], W["mlp.down_proj"])
        logits = _rms_norm(h, by_name["norm.weight"], cfg.rms_norm_eps) @ by_name["tok_embeddings.weight"].T
        if not case["train"]:
            return logits.detach()
        loss = _shifted_loss(logits, state["ids"])
        return [loss.detach(), torch.autograd.grad(loss, P)]
    x = state["x"].detach().double().requires_grad_()
    if kind == "head":
        loss = _shifted_loss(x @ P[0].T, state["labels"])
        return [loss.detach(), torch.autograd.grad(loss, [x] + P)]
    if kind == "norm":
        y = _rms_norm(x, P[0], cfg.rms_norm_eps)
        dx, dw = torch.autograd.grad(y, [x] + P, state["dy"].double())
        return [y.detach(), [dx + state["dres"].double(), dw]]
    if kind == "attn":
        y = _attention(x, *P, cfg, _rope_tables(cfg, S, DTYPES[case["dtype"]]), state["mask"])
    else:
        y = _mlp(x, *P)
    if not case["train"]:
        return y.detach()
    return [y.detach(), torch.autograd.grad(y, [x] + P, state["dy"].double())]


def _exact_step(state):
    """AdamW (betas 0.9, 0.95, eps 1e-8, weight decay 0.1) after clipping the
    global norm to 1, first step, on the float32 master."""
    lr, b1, b2, eps, wd = 3e-4, 0.9, 0.95, 1e-8, 0.1
    p = torch.cat([q.detach().double().reshape(-1) for q in state["params"]])
    g = torch.cat([q.grad.double().reshape(-1) for q in state["params"]])
    norm = float(g.norm())
    if norm > 1.0:
        g = g * (1.0 / (norm + 1e-6))
    m, v = (1 - b1) * g, (1 - b2) * g * g
    p = p * (1 - lr * wd) - lr * (m / (1 - b1)) / ((v / (1 - b2)).sqrt() + eps)
    return {"norm": norm, "master": p, "exp_avg": m, "exp_avg_sq": v, "params": p}
