"""The work that programs have this framework do, as cases that can be timed and checked.

Five kinds of call, each through the public entry points and over the sizes that the framework's
configurations, tests and benchmark use:

  forward   rh_forward_dev: tokens in HBM -> logits, per-token losses, per-sequence mean losses
  prompt    rh_prefill: host prompts into the KV cache -> the logits that choose the first new token
  generate  rh_prefill, then one rh_decode_step per new token with its logits on the host (a sampler's loop)
  grads     rh_zero_grads, rh_forward_backward over several micro-batches, rh_read_grads_f32
  step      rh_train_step (accumulation, clipping, AdamW) on a token file, rh_read_weights_f32

Weights are the synthetic N(0, 0.02^2) ones of rh_init_weights_normal and unit norm gains, as in the benchmark;
token ids are drawn log-uniformly over the vocabulary, so that few ids are frequent and most are rare, as in text.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch  # before the framework: the process then has one HIP runtime

from rustane_amd import hip_bridge as hb
from rustane_amd.engine import ModelConfig

STD = 0.02
EPS = 1e-5
ROPE_BASE = 1e4
LOSS_SCALE = 256.0  # TrainConfig's default
# Per layer, RSTK order: wq wk wv wo w1 w3 w2 gamma1 gamma2
TENSORS = ("wq", "wk", "wv", "wo", "w1", "w3", "w2", "gamma1", "gamma2")

# width: (dim, hidden, heads, head_dim), the shapes of the framework's presets and measured configurations
WIDTHS = {
    "512": (512, 1408, 8, 64),
    "768": (768, 2048, 6, 128),
    "1024": (1024, 2816, 8, 128),
    "1536": (1536, 4096, 12, 128),
    "2048": (2048, 5632, 16, 128),
    "2304": (2304, 6144, 18, 128),
    "2560": (2560, 6912, 20, 128),
    "4096": (4096, 11008, 32, 128),
}


def _case(kind, width, layers, vocab, batch, seq, softcap=0.0, steps=0, micro=0, name=None):
    c = {"kind": kind, "width": width, "layers": layers, "vocab": vocab, "batch": batch, "seq": seq,
         "softcap": softcap, "steps": steps, "micro": micro}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest model's forward (evaluation of one window): launches and latency count
        _case("forward", "512", 8, 8192, 1, 256, name="forward_tiny_b1"),
        # a small whole model, one window
        _case("forward", "1536", 20, 32000, 1, 512, name="forward_600m_b1"),
        # the benchmark's headline: the whole 7B model, one 512-token window
        _case("forward", "4096", 32, 32000, 1, 512, name="forward_7b_b1"),
        # validation and scoring in full batches at 7B width (four of its layers and its head)
        _case("forward", "4096", 4, 32000, 16, 512, name="forward_7b_4l_b16"),
        # long documents of an odd length with capped logits, where attention counts
        _case("forward", "2560", 4, 8192, 2, 3001, softcap=30.0, name="forward_5b_4l_long"),
        # the first token after a short chat turn: the whole 7B model over a few dozen tokens
        _case("prompt", "4096", 32, 32000, 1, 45, name="prompt_7b_short"),
        # several medium prompts at once on a small model
        _case("prompt", "1536", 20, 32000, 8, 131, name="prompt_600m_b8"),
        # one user, long context: a 2048-token prompt and 32 new tokens
        _case("generate", "4096", 32, 32000, 1, 2048, steps=32, name="generate_7b_b1_ctx2048"),
        # a full serving batch: 16 short prompts, 24 new tokens each
        _case("generate", "4096", 32, 32000, 16, 128, steps=24, name="generate_7b_b16"),
        # a small model serving a few users
        _case("generate", "1536", 20, 32000, 4, 100, steps=40, name="generate_600m_b4"),
        # gradients at 7B width (one layer and the tied head), accumulated over eight micro-batches
        _case("grads", "4096", 1, 8192, 8, 512, micro=8, name="grads_7b_1l"),
        # whole optimizer steps of a small preset: 40 sequences accumulated in batches of 8
        _case("step", "1024", 8, 8192, 8, 512, micro=40, name="step_1024"),
    ]


# The most that a drawn case may cost: the listed ones' largest product of work and, per kind, their passes.
_CAP = {"forward": 17e12, "prompt": 17e12, "generate": 40e12, "grads": 46e12, "step": 15e12}


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """A case of the same ranges: any width and depth of the family, odd lengths among them."""
    while True:
        kind = rng.choice(["forward", "forward", "forward", "prompt", "generate", "generate", "grads", "step"])
        train = kind in ("grads", "step")
        # the train kinds read every gradient or weight back: widths whose passes are not mostly that copy
        width = rng.choice(["768", "1024", "1536"] if kind == "step" else list(WIDTHS))
        layers = _log_int(rng, 1, 4 if train else 24)
        vocab = rng.choice([8192, 8192, 8200] if train else [8192, 32000, 32000])
        batch, seq, softcap, steps, micro = 1, 1, 0.0, 0, 0
        if kind == "forward":
            batch, seq, softcap = _log_int(rng, 1, 16), _log_int(rng, 32, 4096), rng.choice([0.0, 0.0, 30.0])
        elif kind == "prompt":
            batch, seq = _log_int(rng, 1, 16), _log_int(rng, 8, 2048)
        elif kind == "generate":
            batch, seq, steps = _log_int(rng, 1, 16), _log_int(rng, 16, 2048), rng.randint(16, 40)
        elif kind == "grads":
            batch, seq, micro = _log_int(rng, 1, 8), _log_int(rng, 64, 1024), rng.randint(4, 8)
        else:
            batch, seq, micro = _log_int(rng, 2, 8), _log_int(rng, 128, 512), rng.randint(16, 40)
        c = _case(kind, width, layers, vocab, batch, seq, softcap, steps, micro)
        if batch * seq <= 8192 and work(c)["flops"] <= _CAP[kind] and _params(c) <= 3.2e9:
            return c


# ------------------------------------------------------------------ sizes
def _shape(case):
    D, F, H, hd = WIDTHS[case["width"]]
    return D, F, H, hd, case["layers"], case["vocab"]


def _params(case):
    D, F, _, _, L, V = _shape(case)
    return L * (4 * D * D + 3 * D * F) + V * D


def _config(case):
    D, F, H, hd, L, V = _shape(case)
    return ModelConfig(D, F, H, H, hd, case["seq"], L, V).to_rh(case["softcap"])


def work(case):
    """Products and causal attention; weights once per pass over them, results once."""
    D, F, _, _, L, V = _shape(case)
    B, S, P = case["batch"], case["seq"], _params(case)
    layer_p = L * (4 * D * D + 3 * D * F)

    def causal(n0, n):  # scores and weighted values of queries n0 .. n0 + n - 1
        return 4 * D * L * sum(range(n0 + 1, n0 + n + 1))

    if case["kind"] == "forward":
        return {"flops": B * (S * 2 * P + causal(0, S)), "bytes": 2 * P + 4 * B * S * V}
    if case["kind"] == "prompt":
        return {"flops": B * (S * 2 * layer_p + causal(0, S) + 2 * D * V), "bytes": 2 * P + B * (4 * S * D * L + 4 * V)}
    if case["kind"] == "generate":
        n = case["steps"]
        kv = sum(4 * D * L * (S + i + 1) for i in range(n))
        return {"flops": B * (S * 2 * layer_p + causal(0, S + n) + n * 2 * P + 2 * D * V),
                "bytes": 2 * P * (n + 1) + B * (kv + 4 * S * D * L + 4 * V * (n + 1))}
    seqs = case["micro"] * B if case["kind"] == "grads" else case["micro"]
    flops = 3 * seqs * (S * 2 * P + causal(0, S))
    # grads: fp16 weights in, fp32 gradients out and to the host; step: AdamW's 30 bytes a parameter, weights to the host
    return {"flops": flops, "bytes": (2 + 4 + 4 if case["kind"] == "grads" else 30 + 4) * P}


# ------------------------------------------------------------------ inputs
def _tokens(case, seed):
    """Every sequence's ids: [sequences, seq + 1 (+ the new tokens' ids)], log-uniform over the vocabulary."""
    n = {"grads": case["micro"] * case["batch"]}.get(case["kind"], case["batch"])
    rng = np.random.default_rng(seed)
    u = rng.random((n, case["seq"] + 1 + case["steps"]))
    t = np.minimum(np.exp(u * math.log(case["vocab"])) - 1.0, case["vocab"] - 1).astype(np.int64)
    return rng.permutation(case["vocab"])[t].astype(np.uint32)


def _stream(case, seed):
    """A token file's ids for the optimizer step."""
    rng = np.random.default_rng(seed)
    u = rng.random(200_003)
    t = np.minimum(np.exp(u * math.log(case["vocab"])) - 1.0, case["vocab"] - 1).astype(np.int64)
    return rng.permutation(case["vocab"])[t].astype("<u2")


class _HostTensors:
    """Page-locked fp32 arrays in the weights' shapes, one [layers, ...] array a kind, and their pointers in RSTK
    order: what a training program keeps to read gradients or weights into."""

    def __init__(self, case):
        D, F, _, _, L, V = _shape(case)
        shapes = [(D, D)] * 4 + [(D, F)] * 3 + [(D,)] * 2
        self.embed = torch.empty((V, D), pin_memory=True)
        self.gamma_final = torch.empty((D,), pin_memory=True)
        self.layers = [torch.empty((L,) + s, pin_memory=True) for s in shapes]
        fp = ctypes.POINTER(ctypes.c_float)
        self.pe, self.pg = (ctypes.cast(t.data_ptr(), fp) for t in (self.embed, self.gamma_final))
        self.pl = (fp * (9 * L))(*[ctypes.cast(self.layers[j][i].data_ptr(), fp) for i in range(L) for j in range(9)])

    def named(self):
        return dict(zip(TENSORS, self.layers), embed=self.embed, gamma_final=self.gamma_final)


def prepare(case, seed):
    kind, B, S = case["kind"], case["batch"], case["seq"]
    ctx = hb.Context(_config(case), 0, B, S + case["steps"] if kind in ("prompt", "generate") else 0)
    ctx.init_normal(seed, STD)
    st = {"case": case, "ctx": ctx}
    if kind == "forward":
        t = _tokens(case, seed).astype(np.int32)
        st["tokens"] = torch.from_numpy(np.ascontiguousarray(t[:, :S])).cuda()
        st["targets"] = torch.from_numpy(np.ascontiguousarray(t[:, 1:])).cuda()
        st["logits"] = torch.empty((B, S, case["vocab"]), device="cuda")
        st["losses"] = torch.empty((B, S), device="cuda")
        st["mean"] = torch.empty((B,), device="cuda")
    elif kind in ("prompt", "generate"):
        t = _tokens(case, seed)
        st["prompt"] = np.ascontiguousarray(t[:, :S])
        # the ids that the sampler chose, fixed here so that every pass decodes the same text
        st["next"] = [np.ascontiguousarray(t[:, S + i]) for i in range(case["steps"])]
    elif kind == "grads":
        t = _tokens(case, seed).reshape(case["micro"], B, S + 1)
        st["micro"] = [(np.ascontiguousarray(m[:, :S]), np.ascontiguousarray(m[:, 1:])) for m in t]
        st["host"] = _HostTensors(case)
    else:
        fd, path = tempfile.mkstemp(suffix=".bin")
        with os.fdopen(fd, "wb") as f:
            f.write(_stream(case, seed).tobytes())
        st["data"] = hb.TokenData(path)
        os.unlink(path)  # the mapping stays
        st["config"] = hb.train_config(accum_steps=case["micro"], warmup_steps=0)
        st["step"] = 0
        st["host"] = _HostTensors(case)
    return st


# ------------------------------------------------------------------ one pass
def run(st):
    ctx, kind, case = st["ctx"], st["case"]["kind"], st["case"]
    if kind == "forward":
        ctx.forward_dev(st["tokens"].data_ptr(), st["targets"].data_ptr(), case["batch"], case["seq"],
                        st["logits"].data_ptr(), st["losses"].data_ptr(), st["mean"].data_ptr())
        return {"logits": st["logits"], "losses": st["losses"], "mean": st["mean"]}
    if kind == "prompt":
        return {"logits": ctx.prefill(st["prompt"], want_logits=True)[1]}
    if kind == "generate":
        out = {"prompt": ctx.prefill(st["prompt"], want_logits=True)[1]}
        out["steps"] = [ctx.decode_step(t, want_logits=True)[1] for t in st["next"]]
        return out
    h = st["host"]
    if kind == "grads":
        ctx.zero_grads()
        losses = [ctx.forward_backward(tok, tgt, LOSS_SCALE) for tok, tgt in st["micro"]]
        ctx._ck(hb.lib().rh_read_grads_f32(ctx.h, h.pe, h.pg, h.pl), "rh_read_grads_f32")
        return dict(h.named(), losses=np.stack(losses))
    loss, norm = ctx.train_step(st["data"], st["step"], st["config"])
    st["step"] += 1
    ctx._ck(hb.lib().rh_read_weights_f32(ctx.h, h.pe, h.pg, h.pl), "rh_read_weights_f32")
    return dict(h.named(), loss=loss, norm=norm)


def tolerance(case):
    """Four times what the start of a series of changes showed against 64 bits. The products take fp16 operands (11
    bits) and sum in fp32, so every layer adds rounding: a forward's logits are off by 6e-4 of their norm after one or
    two layers, and later by 1.9e-4 (512 wide) to 8e-4 (4096 wide) per square root of a layer; a gradient's tensors by
    up to 1e-3 (2e-3 after several layers); an updated embedding by 1.1e-3, since AdamW's first steps move every value
    by the learning rate and where a gradient is near zero rounding chooses the direction."""
    if case["kind"] == "grads":
        return {"rel": 8e-3, "max": 0.3}
    if case["kind"] == "step":
        return {"rel": 5e-3, "max": 0.3}
    D, L = WIDTHS[case["width"]][0], case["layers"]
    return {"rel": min(0.03, 4.0 * max(6e-4, math.sqrt(L) * (1e-4 + 1.7e-7 * D)))}


# ------------------------------------------------------------------ the same in 64 bits
def _normal(n, seed, tensor):
    """rh_init_weights_normal's values: Philox4x32-10 (Salmon et al., SC'11) keyed by the seed, counter (pair, tensor),
    Box-Muller pairs, rounded to the fp16 that the framework keeps; as float64."""
    m32 = 0xFFFFFFFF
    p = torch.arange((n + 1) // 2, dtype=torch.int64, device="cuda")
    c = [p & m32, p >> 32, torch.full_like(p, tensor), torch.full_like(p, 0x52485354)]
    k0, k1 = seed & m32, (seed >> 32) & m32
    for _ in range(10):
        a, b = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57  # wraps; the shift below takes the unsigned high half
        c = [((b >> 32) & m32) ^ c[1] ^ k0, b & m32, ((a >> 32) & m32) ^ c[3] ^ k1, a & m32]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    u1 = ((c[0] >> 8).float() + 1.0) * (1.0 / 16777216.0)
    u2 = (c[1] >> 8).float() * (1.0 / 16777216.0)
    r, th = STD * torch.sqrt(-2.0 * torch.log(u1)), 6.283185307179586 * u2
    x = torch.stack([r * torch.cos(th), r * torch.sin(th)], dim=1).reshape(-1)[:n]
    return x.half().double()


def _matrix(case, seed, layer, j):
    D, F = WIDTHS[case["width"]][:2]
    shape = (D, D) if j < 4 else (D, F)
    return _normal(shape[0] * shape[1], seed, 1 + 9 * layer + j).reshape(shape)


def _rms(x, g):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * g


def _rope(x):  # [heads, n, hd], interleaved pairs
    n, hd = x.shape[1:]
    i = torch.arange(hd // 2, device=x.device, dtype=torch.float64)
    th = torch.arange(n, device=x.device, dtype=torch.float64)[:, None] / ROPE_BASE ** (2.0 * i / hd)
    c, s = th.cos(), th.sin()
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], dim=-1).reshape(x.shape)


def _attention(q, k, v):
    """Causal attention of one sequence [n, D] by heads, a stretch of queries at a time."""
    H, n, hd = q.shape
    kt, out = k.transpose(1, 2).contiguous(), []
    for a in range(0, n, 1024):
        b = min(n, a + 1024)
        s = torch.matmul(q[:, a:b], kt) / math.sqrt(hd)
        past = torch.arange(n, device=q.device)[None, :] > torch.arange(a, b, device=q.device)[:, None]
        out.append(torch.matmul(torch.softmax(s.masked_fill(past, float("-inf")), -1), v))
    return torch.cat(out, 1)


def _layer(x, w, B, case):
    """x [B * n, D] through one layer; w its nine tensors."""
    D, _, H, hd, L, _ = _shape(case)
    alpha, n = 1.0 / math.sqrt(2.0 * L), x.shape[0] // B
    xn = _rms(x, w[7])
    heads = [(xn @ w[j]).reshape(B, n, H, hd).transpose(1, 2) for j in range(3)]
    o = [_attention(_rope(heads[0][b]).contiguous(), _rope(heads[1][b]).contiguous(), heads[2][b].contiguous()) for b in range(B)]
    x = x + alpha * (torch.stack(o).transpose(1, 2).reshape(B * n, D) @ w[3])
    xn = _rms(x, w[8])
    return x + alpha * ((torch.nn.functional.silu(xn @ w[4]) * (xn @ w[5])) @ w[6].t())


def _head(x, embed, g, softcap):
    z = _rms(x, g) @ embed.t()
    return softcap * torch.tanh(z / softcap) if softcap else z


def _weights(case, seed):
    D, _, _, _, L, V = _shape(case)
    one = torch.ones(D, dtype=torch.float64, device="cuda")
    return (_normal(V * D, seed, 0).reshape(V, D), one.clone(),
            [[_matrix(case, seed, l, j) for j in range(7)] + [one.clone(), one.clone()] for l in range(L)])


def _gradients(case, w, seqs, scale):
    """Mean losses [sequences] and scale times the summed gradients of w = (embed, gamma_final, layers)."""
    flat = [w[0], w[1]] + [t for lw in w[2] for t in lw]
    for t in flat:
        t.requires_grad_(True)
    losses = []
    for s in torch.from_numpy(seqs.astype(np.int64)).cuda():
        x = w[0][s[:-1]]
        for lw in w[2]:
            x = _layer(x, lw, 1, case)
        loss = torch.nn.functional.cross_entropy(_head(x, w[0], w[1], case["softcap"]), s[1:])
        (scale * loss).backward()
        losses.append(loss.detach())
    for t in flat:
        t.requires_grad_(False)
    return torch.stack(losses)


def _named(w, f):
    return dict({t: torch.stack([f(lw[j]) for lw in w[2]]) for j, t in enumerate(TENSORS)}, embed=f(w[0]), gamma_final=f(w[1]))


def exact(case, seed):
    kind, B, S = case["kind"], case["batch"], case["seq"]
    D, _, _, _, L, V = _shape(case)
    if kind in ("forward", "prompt", "generate"):
        t = torch.from_numpy(_tokens(case, seed).astype(np.int64)).cuda()
        n = S + case["steps"]
        embed = _normal(V * D, seed, 0).reshape(V, D)
        one = torch.ones(D, dtype=torch.float64, device="cuda")
        x = embed[t[:, :n]].reshape(B * n, D)
        for l in range(L):
            x = _layer(x, [_matrix(case, seed, l, j) for j in range(7)] + [one, one], B, case)
        if kind != "forward":
            x = x.reshape(B, n, D)[:, S - 1:]
            z = _head(x, embed, one, case["softcap"])
            if kind == "prompt":
                return {"logits": z[:, 0]}
            return {"prompt": z[:, 0], "steps": [z[:, i + 1].contiguous() for i in range(case["steps"])]}
        z = _head(x, embed, one, case["softcap"]).reshape(B, S, V)
        ce = torch.nn.functional.cross_entropy(z.reshape(B * S, V), t[:, 1:].reshape(-1), reduction="none").reshape(B, S)
        return {"logits": z, "losses": ce, "mean": ce.mean(1)}
    w = _weights(case, seed)
    if kind == "grads":
        losses = _gradients(case, w, _tokens(case, seed), LOSS_SCALE)
        return dict(_named(w, lambda t: t.grad), losses=losses.reshape(case["micro"], B))
    # one optimizer step from zero moments: the accumulated mean gradient, clipped to norm 1, then AdamW at t = 1
    ids, micro = _stream(case, seed), case["micro"]
    at = [(i * 104729) % (len(ids) - S - 1) for i in range(micro)]
    losses = _gradients(case, w, np.stack([ids[p:p + S + 1] for p in at]), 1.0 / micro)
    flat = [w[0], w[1]] + [t for lw in w[2] for t in lw]
    norm = torch.sqrt(sum((t.grad ** 2).sum() for t in flat))
    tc = {"lr": 3e-4, "b1": 0.9, "b2": 0.95, "eps": 1e-8, "decay": 0.1, "matrix": 0.05, "embed": 5.0}

    def updated(t, lr, decay):
        g = t.grad / max(1.0, float(norm))
        m, v = (1 - tc["b1"]) * g, (1 - tc["b2"]) * g * g
        return t - lr * (m / (1 - tc["b1"]) / (torch.sqrt(v / (1 - tc["b2"])) + tc["eps"]) + decay * t)

    out = {t: torch.stack([updated(lw[j], tc["lr"] * (tc["matrix"] if j < 7 else 1.0), tc["decay"] if j < 7 else 0.0)
                           for lw in w[2]]) for j, t in enumerate(TENSORS)}
    return dict(out, embed=updated(w[0], tc["lr"] * tc["embed"], 0.0), gamma_final=updated(w[1], tc["lr"], 0.0),
                loss=losses.mean(), norm=norm)
