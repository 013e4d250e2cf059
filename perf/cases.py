"""What this framework's users have it do, as cases that can be timed and compared.

Two families, each in both directions of serving:

  DeepSeek engine   one token of decode (dsk_forward) and one prompt (dsk_hydrate): V2-Lite's shapes at full depth, where the bytes
                    of a launch take a microsecond and latency counts; V3's shapes at full width on a slice of 1 dense + 4 MoE
                    blocks (a block is what repeats; 61 of them fill the card by themselves).  Q2_K is what the engine is for;
                    Q3_K, F8E5M2 and F16 checkpoints run too.  MHA is the default attention, MLA the compact-cache one.
  layered designs   prompts (alone and several at once), steps of single tokens (alone and batched): Timerax and Ranutar at the
                    `lite` and `wide` layer sizes, bf16; and Ranutar in 32 bits, the precision of parity runs.

Weights are random and made in HBM from the seed (the engine's own synthesis: no checkpoint of these sizes is at hand), tokens
are uniform over the vocabulary.  A layered step appends a token to its sequences, as decoding does: the next pass is the next
position."""
import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "deepseek.cpp_amd"))
import dsk  # noqa: E402

V3_LAYERS = 5  # 1 dense + 4 MoE blocks
DEVICE = "cuda"


# ---- models -----------------------------------------------------------------------------------------------------------
def deepseek(case):
    """the engine's configuration of a case"""
    q, mla = case["quant"], case["mla"]
    kq = q in ("q2_k", "q3_k")
    c = dict(rope_theta=10000.0, norm_eps=1e-6, act="silu", use_mla=mla, quant=q, block_size=(128, 128) if q == "f8e5m2" else (0, 0),
             rs_original_max_position_embeddings=4096, max_seq_len=4096, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
             v_head_dim=128, first_k_dense_replace=1)
    if case["model"] == "v3":
        c.update(dim=7168, hidden_dim=18432, n_layers=V3_LAYERS, n_heads=128, vocab_size=129280, n_shared_experts=1, n_routed_experts=256,
                 n_active_routed=8, moe_intermediate_size=2048, routed_scaling_factor=2.5, n_group=8, topk_group=4,
                 topk_method="group_limited_greedy", scoring_func="sigmoid", norm_topk_prob=True, has_moegate_bias=True, q_lora_rank=1536)
    else:  # V2-Lite; K-quants need rows of a multiple of 256, so these checkpoints are padded
        c.update(dim=2048, hidden_dim=11008 if kq else 10944, n_layers=27, n_heads=16, vocab_size=102400, n_shared_experts=2,
                 n_routed_experts=64, n_active_routed=6, moe_intermediate_size=1536 if kq else 1408, routed_scaling_factor=1.0, n_group=1,
                 topk_group=1, topk_method="greedy", scoring_func="softmax", norm_topk_prob=False, has_moegate_bias=False, q_lora_rank=0,
                 max_seq_len=1024)
    return SimpleNamespace(**c)


def layered(case):
    """config.json of a layered design"""
    wide = case["size"] == "wide"
    D, H = (7168, 64) if wide else (2048, 16)
    delta = {"conv": 4, "dim": 128, "heads": H, "kv_heads": H, "vdim": 128}
    if case["design"] == "timerax":
        moe = {"kind": "moe", "router": {"experts": 256 if wide else 64, "top": 8 if wide else 6},
               "expert": {"ff": 2048 if wide else 1408, "limit": 7.0}, "shared": {"ff": 2048 if wide else 2816, "limit": 7.0}}
        attn = {"heads": H, "kv_heads": H // 4, "dim": 128, "vdim": 128, "mask": {"size": 4096}, "scale": 0.0883883,
                "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
        mlstm = {"heads": H, "dim": 64, "vdim": 128, "gate_cap": 15.0}
        kinds = [{"type": "channel_delta", "mixer": delta, "mlp": moe}] * 2 + [{"type": "parallel", "mixer": {"left": attn, "right": mlstm}, "mlp": moe}]
        more = {"architecture": "Timerax", "logit_softcap": 30.0}
    else:
        mlp = {"kind": "dense", "ff": 27648 if wide else 16896}
        lat = {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 1536, "kv_rank": 512, "mask": {"size": 4096}, "scale": 0.0721688,
               "rot": {"base": 500000.0, "dims": 64}}
        kinds = [{"type": "wkv", "mixer": {"heads": D // 64, "dim": 64}, "mlp": mlp}, {"type": "delta", "mixer": delta, "mlp": mlp},
                 {"type": "latent_attention", "mixer": lat, "mlp": mlp}]
        more = {"architecture": "Ranutar", "canon": {"taps": 4}, "logit_scale": 0.5}
    return dict(more, width=D, vocab=129280 if wide else 102400, norm={"eps": 1e-6}, layers=kinds * (case["layers"] // 3))


# ---- the cases --------------------------------------------------------------------------------------------------------
def token(model, quant, mla, pos):
    return {"kind": "token", "model": model, "quant": quant, "mla": mla, "pos": pos}


def prompt(mla, tokens):
    return {"kind": "prompt", "model": "v3", "quant": "q2_k", "mla": mla, "tokens": tokens}


def prompts(design, size, lengths, dtype="bfloat16", want=1):
    return {"kind": "prompts", "design": design, "size": size, "layers": 3 if size == "wide" else 9, "dtype": dtype,
            "lengths": ",".join(str(n) for n in lengths), "want": want}


def step(design, size, batch, context):
    return {"kind": "step", "design": design, "size": size, "layers": 3 if size == "wide" else 27, "dtype": "bfloat16", "batch": batch,
            "context": context}


def listed():
    return [
        # one chat user on the small model: the smallest calls, bound by launches and latency
        dict(token("v2lite", "q2_k", False, 61), name="lite_token_q2k"),
        # the same model from an F8E5M2 checkpoint
        dict(token("v2lite", "f8e5m2", False, 24), name="lite_token_f8"),
        # the flagship: V3 Q2_K decode, the reference's default attention, a chat's context
        dict(token("v3", "q2_k", False, 199), name="v3_token_mha"),
        # ... with the compact cache deep in a long document
        dict(token("v3", "q2_k", True, 3001), name="v3_token_mla_long"),
        # a full prompt chunk of the flagship
        dict(prompt(False, 512), name="v3_prompt_512"),
        # a short question (an odd number of tokens), MLA
        dict(prompt(True, 77), name="v3_prompt_mla_77"),
        # a document into the layered MoE design: the largest amount of arithmetic
        dict(prompts("timerax", "lite", [2048]), name="timerax_prompt_2048"),
        # a server's batch of decoding sequences, wide layers
        dict(step("timerax", "wide", 16, 300), name="timerax_step_16"),
        # several users' prompts of different lengths arriving together, dense design
        dict(prompts("ranutar", "lite", [331, 700, 64, 901]), name="ranutar_prompts_4"),
        # one user decoding
        dict(step("ranutar", "lite", 1, 512), name="ranutar_step_1"),
        # a few users at the wide layer sizes: bound by the weights' bytes
        dict(step("ranutar", "wide", 4, 200), name="ranutar_step_4"),
        # a parity run in 32 bits, the logits of the last tokens
        dict(prompts("ranutar", "lite", [301], "float32", want=8), name="ranutar_scores_f32"),
    ]


def draw(rng):
    """a case of the same ranges; sizes spread over their logarithm, odd ones among them"""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["token", "token", "prompt", "prompts", "prompts", "step", "step"])
    if kind == "token":
        if rng.random() < 0.5:
            return token("v2lite", rng.choice(["q2_k", "q3_k", "f8e5m2", "fp16"]), False, log(5, 200))
        return token("v3", "q2_k", rng.random() < 0.5, log(5, 3500))
    if kind == "prompt":
        return prompt(rng.random() < 0.5, log(5, 512))
    design, size = rng.choice(["timerax", "ranutar"]), rng.choice(["lite", "wide"])
    if kind == "step":
        return step(design, size, log(1, 16), log(20, 1500))
    if rng.random() < 0.2:
        return prompts("ranutar", "lite", [log(20, 400)], "float32", want=rng.randint(1, 8))
    n, left, lengths = rng.randint(1, 4), 2048 if size == "lite" else 1536, []
    for _ in range(n):
        lengths.append(log(20, max(24, left - 24 * n)))
        left -= lengths[-1]
    return prompts(design, size, [m for m in lengths if m > 0])


# ---- state and passes -------------------------------------------------------------------------------------------------
_ctx = None


def context():
    global _ctx
    if _ctx is None:
        _ctx = dsk.Ctx(0)
    return _ctx


def tokens_of(case, seed):
    """what the case's sequences are made of, in the order they are used"""
    rng = np.random.default_rng(seed)
    if case["kind"] == "token":
        return rng.integers(0, deepseek(case).vocab_size, case["pos"] + 1).astype(np.int32)
    if case["kind"] == "prompt":
        return rng.integers(0, deepseek(case).vocab_size, case["tokens"]).astype(np.int32)
    vocab = layered(case)["vocab"]
    if case["kind"] == "prompts":
        return [rng.integers(0, vocab, int(n)).astype(np.int32) for n in case["lengths"].split(",")]
    return rng.integers(0, vocab, (case["batch"], case["context"] + 1)).astype(np.int32)


def prepare(case, seed):
    toks = tokens_of(case, seed)
    if case["kind"] in ("token", "prompt"):
        m = dsk.Model(context(), deepseek(case), None, synth_seed=seed)
        if case["kind"] == "token":
            if case["pos"]:  # the context; its last token by itself, so that the model has decoded before
                if case["pos"] > 1:
                    m.hydrate(toks[:case["pos"] - 1], 0)
                m.forward_nocopy(int(toks[case["pos"] - 1]), case["pos"] - 1)
        else:  # a server has taken prompts before (the first one makes the batched path's copies of some matrices)
            m.hydrate(toks[:16], 0)
        return {"case": case, "model": m, "tokens": toks}
    c = layered(case)
    m = dsk.LM(context(), dtype=case["dtype"], config=c, seed=seed)
    if case["kind"] == "prompts":
        return {"case": case, "model": m, "tokens": toks}
    seqs = [m.seq_open() for _ in toks]
    for i in range(0, len(seqs), 4):
        m.step([(s, t[:-2], []) for s, t in zip(seqs[i:i + 4], toks[i:i + 4])])
    m.step([(s, t[-2:-1], [0]) for s, t in zip(seqs, toks)])  # (a step of single tokens: the model has decoded before)
    return {"case": case, "model": m, "seqs": seqs, "tokens": toks}


class Logits(np.ndarray):
    """the engine's own buffer of logits; keeps its model alive"""
    model = None


def run(state):
    case, m, toks = state["case"], state["model"], state["tokens"]
    if case["kind"] == "token":
        out = m.forward_nocopy(int(toks[-1]), case["pos"]).view(Logits)
        out.model = m
        return out
    if case["kind"] == "prompt":
        return m.hydrate(toks, 0, dsk.MODE_OUTPUT_LOGITS)
    if case["kind"] == "step":
        return m.step([(s, t[-1:], [0]) for s, t in zip(state["seqs"], toks)])
    seqs = [m.seq_open() for _ in toks]
    out = m.step([(s, t, range(len(t) - min(case["want"], len(t)), len(t))) for s, t in zip(seqs, toks)])
    for s in seqs:
        m.seq_close(s)
    return out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def distinct(n, top, rows):
    """experts that `rows` tokens reach, if each takes `top` of `n` at random"""
    return n * (1 - (1 - top / n) ** rows)


def work(case):
    if case["kind"] in ("token", "prompt"):
        c = deepseek(case)
        rows = 1 if case["kind"] == "token" else case["tokens"]
        last = case["pos"] + 1 if case["kind"] == "token" else case["tokens"]
        bpw = {"q2_k": 84 / 256, "q3_k": 110 / 256, "f8e5m2": 1 + 4 / 128 ** 2, "fp16": 2}[c.quant]
        H, hd = c.n_heads, c.qk_nope_head_dim + c.qk_rope_head_dim
        attn = c.dim * (c.kv_lora_rank + c.qk_rope_head_dim) + c.dim * H * c.v_head_dim
        if c.use_mla:
            attn += c.dim * c.q_lora_rank + c.q_lora_rank * H * (c.kv_lora_rank + c.qk_rope_head_dim) + H * c.v_head_dim * c.kv_lora_rank
            kv_row, kv_flop = c.kv_lora_rank + c.qk_rope_head_dim, H * (2 * c.kv_lora_rank + c.qk_rope_head_dim)
        else:
            attn += (c.dim * c.q_lora_rank + c.q_lora_rank * H * hd if c.q_lora_rank else c.dim * H * hd)
            attn += c.kv_lora_rank * H * (c.qk_nope_head_dim + c.v_head_dim)
            kv_row, kv_flop = H * (hd + c.v_head_dim), H * (hd + c.v_head_dim)
        expert, shared = 3 * c.dim * c.moe_intermediate_size, 3 * c.dim * c.moe_intermediate_size * c.n_shared_experts
        dense, n_moe = 3 * c.dim * c.hidden_dim, c.n_layers - c.first_k_dense_replace
        read = c.n_layers * attn + dense + n_moe * (shared + distinct(c.n_routed_experts, c.n_active_routed, rows) * expert) + c.vocab_size * c.dim
        used = c.n_layers * attn + dense + n_moe * (shared + c.n_active_routed * expert)
        router = n_moe * c.n_routed_experts * c.dim
        pairs = last if rows == 1 else rows * (rows + 1) / 2
        return {"bytes": read * bpw + router * 4 + c.n_layers * last * kv_row * 2 + c.vocab_size * 4,
                "flops": 2.0 * rows * (used + router) + 2.0 * c.vocab_size * c.dim + 2.0 * c.n_layers * pairs * kv_flop}
    c = layered(case)
    D, flops, weights, state = c["width"], 0.0, 0.0, 0.0
    es = 4 if case["dtype"] == "float32" else 2
    lens = [int(n) for n in case["lengths"].split(",")] if case["kind"] == "prompts" else [1] * case["batch"]
    before = 0 if case["kind"] == "prompts" else case["context"]
    rows, pairs, seen = sum(lens), sum(n * before + n * (n + 1) / 2 for n in lens), sum(before + n for n in lens)
    for layer in c["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        if layer["type"] == "parallel":
            a, b = m["left"], m["right"]
            w = D * (2 * a["heads"] * a["dim"] + 2 * a["kv_heads"] * a["dim"] + b["heads"] * (2 * b["dim"] + 3 * b["vdim"]))
            flops += 2 * pairs * a["heads"] * (a["dim"] + a["vdim"]) + 4.0 * rows * b["heads"] * b["dim"] * b["vdim"]
            state += seen * a["kv_heads"] * (a["dim"] + a["vdim"]) * es + len(lens) * 8 * b["heads"] * b["dim"] * b["vdim"]
        elif layer["type"] in ("channel_delta", "delta"):
            w = D * m["dim"] * (2 * m["kv_heads"] + 2 * m["heads"]) + (D * m["heads"] * m["vdim"] if layer["type"] == "delta" else 2 * m["dim"] * (D + m["heads"] * m["dim"]))
            flops += 6.0 * rows * m["heads"] * m["dim"] * m["vdim"]
            state += len(lens) * 8 * m["heads"] * m["dim"] * m["vdim"]
        elif layer["type"] == "wkv":
            w = 5 * D * m["heads"] * m["dim"] + 64 * (D + m["heads"] * m["dim"])
            flops += 4.0 * rows * m["heads"] * m["dim"] ** 2
            state += len(lens) * 8 * m["heads"] * m["dim"] ** 2
        else:
            hd = m["dim"] + m["rot_dim"]
            w = D * (m["q_rank"] + m["kv_rank"] + m["rot_dim"]) + m["heads"] * (m["q_rank"] * hd + m["kv_rank"] * (m["dim"] + m["vdim"]) + m["vdim"] * D)
            flops += 2 * pairs * m["heads"] * (hd + m["vdim"])
            state += seen * (m["kv_rank"] + m["rot_dim"]) * es
        used = w
        if f["kind"] == "moe":
            e, s, n = 3 * D * f["expert"]["ff"], 3 * D * f["shared"]["ff"], f["router"]["experts"]
            w += n * D + s + distinct(n, f["router"]["top"], rows) * e
            used += n * D + s + f["router"]["top"] * e
        else:
            w += 2 * D * f["ff"]
            used += 2 * D * f["ff"]
        weights += w
        flops += 2.0 * rows * used
    want = sum(min(case.get("want", 1), n) for n in lens)
    return {"bytes": 2 * (weights + c["vocab"] * D + rows * D) + state + 4 * want * c["vocab"], "flops": flops + 2.0 * want * c["vocab"] * D}


def tolerance(case):
    if case["kind"] in ("token", "prompt"):
        if case["quant"] in ("q2_k", "q3_k"):
            # every activation vector becomes 8-bit codes: another order of a sum moves codes over their rounding edges, and the
            # next layers carry that on (0.011 - 0.018 between the engine's own layouts of V3's weights, 0.3 - 0.5 over 27 layers)
            return {"rel": 0.03, "max": 0.3}
        return {"rel": 5e-3, "max": 0.05}  # (0.0017 from 64 bits: keys and values are cached in half precision)
    if case["dtype"] == "float32":
        return {"rel": 3e-5, "max": 2e-4}  # (4e-6 between recurrences by chunks and by tokens)
    # bf16: 0.004 - 0.008 between recurrences by chunks and by tokens, 0.016 - 0.034 from 64 bits; Timerax's router may decide a
    # close call the other way
    return {"rel": 0.03, "max": 0.3}


# ---- the same passes in 64 bits ---------------------------------------------------------------------------------------
# The weights are drawn again from the seed (counter-based generators, stated here by themselves); the designs are plain torch.
# Models with K-quant weights have no such value - their results are defined through 8-bit codes of every activation vector - and
# neither has a mixture of experts in bf16, whose routing follows bf16 rounding.
U64 = 1 << 64


def i64(v):
    v %= U64
    return v - U64 if v >= U64 // 2 else v


def shr(z, s):
    return (z >> s) & ((1 << (64 - s)) - 1)


def splitmix(z):
    z = (z ^ shr(z, 30)) * i64(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * i64(0x94D049BB133111EB)
    return z ^ shr(z, 31)


def count(n):
    return torch.arange(n, dtype=torch.int64, device=DEVICE)


class DeepSeekWeights:
    """matrices and vectors of a synthesised float model, by role and layer"""
    ROLE = dict(embed=0, final_norm=1, output=2, attn_norm=10, kv_a_norm=12, ffn_norm=13, wq=14, wkv_a=17, wkv_b=18, wo=19, w1=23, w2=24, w3=25,
                shared_w1=26, shared_w2=27, shared_w3=28, moegate=29)

    def __init__(self, c, seed):
        self.c, self.seed = c, seed

    def key(self, role, layer, expert=0):
        return self.seed * 0x9E3779B97F4A7C15 + (layer + 1) * 1000003 + self.ROLE[role] * 7919 + expert * 0x100000001B3

    @staticmethod
    def mix(key, n, mult):
        return splitmix((i64(key) ^ (count(n) * i64(mult))) + i64(0x9E3779B97F4A7C15))

    @staticmethod
    def u01(r):
        return ((shr(r, 40) + 1).float() * np.float32(1.0 / 16777217.0).item()).double()

    def gauss(self, key, n):
        r = self.mix(key, n, 0xD1342543DE82EF95)
        u2 = self.u01(splitmix(r + i64(0x9E3779B97F4A7C15)))
        return torch.sqrt(-2 * torch.log(self.u01(r))) * torch.cos(6.28318530718 * u2)

    def vector(self, role, layer, n):
        return (1 + 0.1 * self.gauss(self.key(role, layer), n)).float().double()

    def matrix(self, role, layer, rows, n, expert=0, std=None):
        std, key = 1 / math.sqrt(n) if std is None else std, self.key(role, layer, expert)
        if role == "moegate":
            return (std * self.gauss(key, rows * n)).float().double().view(rows, n)
        if self.c.quant == "fp16":
            return (std * self.gauss(key, rows * n)).half().double().view(rows, n)
        w = (self.gauss(key, rows * n).half().view(torch.int16) & -256).view(torch.half).double().view(rows, n)
        sr, sn = -(-rows // 128), -(-n // 128)
        s = (0.5 + self.u01(self.mix(i64(key) ^ 0x5CA1E, sr * sn, 0x9E3779B97F4A7C15))) * std
        return w * s.float().double().view(sr, sn).repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :n]


def rmsnorm(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def deepseek_exact(case, seed):
    """logits behind the last token; every token of the context at once"""
    c, toks = deepseek(case), torch.from_numpy(tokens_of(case, seed)).long().to(DEVICE)
    W, T, H = DeepSeekWeights(c, seed), len(toks), c.n_heads
    nope, rope, vd, lora, hid = c.qk_nope_head_dim, c.qk_rope_head_dim, c.v_head_dim, c.kv_lora_rank, c.moe_intermediate_size
    x = W.matrix("embed", -1, c.vocab_size, c.dim, std=1.0)[toks]
    ang = torch.arange(T, device=DEVICE).double()[:, None] * c.rope_theta ** (-torch.arange(0, rope, 2, device=DEVICE).double() / rope)

    def turn(v):  # [T, ..., rope], pairs of neighbours; (the order of a key's values does not matter to a product with a query)
        a = ang.view(T, *[1] * (v.dim() - 2), rope // 2)
        u, w = v[..., 0::2], v[..., 1::2]
        return torch.cat([u * torch.cos(a) - w * torch.sin(a), u * torch.sin(a) + w * torch.cos(a)], -1)

    def glu(h, names, layer, n, expert=0):
        w1, w3, w2 = (W.matrix(r, layer, *((n, c.dim) if r[-1] != "2" else (c.dim, n)), expert) for r in names)
        return (torch.nn.functional.silu(h @ w1.T) * (h @ w3.T)) @ w2.T

    for layer in range(c.n_layers):
        h = rmsnorm(x, c.norm_eps) * W.vector("attn_norm", layer, c.dim)
        q = (h @ W.matrix("wq", layer, H * (nope + rope), c.dim).T).view(T, H, nope + rope)
        kv = h @ W.matrix("wkv_a", layer, lora + rope, c.dim).T
        kb = (rmsnorm(kv[:, :lora], c.norm_eps) * W.vector("kv_a_norm", layer, lora)) @ W.matrix("wkv_b", layer, H * (nope + vd), lora).T
        kb = kb.view(T, H, nope + vd)
        q = torch.cat([q[..., :nope], turn(q[..., nope:])], -1)
        k = torch.cat([kb[..., :nope], turn(kv[:, lora:])[:, None].expand(T, H, rope)], -1)
        s = torch.bmm(q.transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous()) / math.sqrt(nope + rope)
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=DEVICE).triu(1), -math.inf)
        o = torch.bmm(s.softmax(-1), kb[..., nope:].transpose(0, 1).contiguous()).transpose(0, 1).reshape(T, H * vd)
        x = x + o @ W.matrix("wo", layer, c.dim, H * vd).T
        h = rmsnorm(x, c.norm_eps) * W.vector("ffn_norm", layer, c.dim)
        if layer < c.first_k_dense_replace:
            x = x + glu(h, ("w1", "w3", "w2"), layer, c.hidden_dim)
            continue
        w, e = (h @ W.matrix("moegate", layer, c.n_routed_experts, c.dim).T).softmax(-1).topk(c.n_active_routed, -1)
        y = glu(h, ("shared_w1", "shared_w3", "shared_w2"), layer, c.n_shared_experts * hid)
        for i in e.unique().tolist():
            at, k = (e == i).nonzero(as_tuple=True)
            y[at] += w[at, k][:, None] * glu(h[at], ("w1", "w3", "w2"), layer, hid, i)
        x = x + y
    h = rmsnorm(x[-1:], c.norm_eps) * W.vector("final_norm", -1, c.dim)
    return (h @ W.matrix("output", -1, c.vocab_size, c.dim).T)[0].cpu().numpy()


class LayeredWeights:
    """the tensors of a random layered model, in the order in which they are drawn"""

    def __init__(self, seed):
        self.seed = seed + 1

    def get(self, rows, cols):
        n, scale = max(rows, 1) * cols, np.sqrt(np.float32(3.0) / np.float32(cols)) if rows else np.float32(0.1)
        z = splitmix((count(n) + 1) * i64(0x9E3779B97F4A7C15) + i64(self.seed))
        self.seed += 1
        v = shr(z, 40).float() * (2.0 / 16777216.0) - 1.0
        v = (float(scale) * v).bfloat16().double()
        return v.view(rows, cols) if rows else v


def one_plus(x, w, eps):
    return rmsnorm(x, eps) * (1 + w)


def input_conv(h, w, spans):
    taps, out = w.shape[1], h.clone()
    for a, b in spans:
        full = torch.cat([torch.zeros(taps - 1, h.shape[1], dtype=h.dtype, device=h.device), h[a:b]])
        for j in range(taps):
            out[a:b] += full[j:j + b - a] * w[:, j]
    return out


def halves(x, pos, rot):
    n = rot["dims"] // 2
    a = pos.double().view(-1, *[1] * (x.dim() - 1)) * float(rot["base"]) ** (-2 * torch.arange(n, device=DEVICE).double() / rot["dims"])
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * torch.cos(a) - v * torch.sin(a), v * torch.cos(a) + u * torch.sin(a), x[..., 2 * n:]], -1)


def ranutar_exact(case, seed):
    """logits of the wanted tokens; all sequences' tokens behind each other, each recurrence token by token"""
    c, W, step_case = layered(case), LayeredWeights(seed), case["kind"] == "step"
    seqs = [torch.from_numpy(np.asarray(t)).long().to(DEVICE) for t in tokens_of(case, seed)]
    ends = np.cumsum([len(t) for t in seqs]).tolist()
    spans = [(e - len(t), e) for e, t in zip(ends, seqs)]
    pos, toks = torch.cat([torch.arange(len(t), device=DEVICE) for t in seqs]), torch.cat(seqs)
    D, T, eps, V = c["width"], len(toks), c["norm"]["eps"], c["vocab"]
    x, final, head = W.get(V, D)[toks], W.get(0, D), W.get(V, D)
    longest = max(b - a for a, b in spans)
    slot = torch.full((len(spans), longest), T, dtype=torch.long, device=DEVICE)  # rows by sequence and place; T: none
    for i, (a, b) in enumerate(spans):
        slot[i, :b - a] = torch.arange(a, b, device=DEVICE)

    def by_seq(v):  # [T, ...] -> [place, sequence, ...]
        return torch.cat([v, torch.zeros_like(v[:1])])[slot.T]

    def behind(v, o):  # ... and back
        out = torch.zeros_like(torch.cat([o.reshape(-1, *o.shape[2:])[:1]] * (T + 1)))
        out[slot.T.reshape(-1)] = o.reshape(-1, *o.shape[2:])
        return out[:T]

    def sigmoid(v):
        return torch.sigmoid(v)

    for layer in c["layers"]:
        m, f, kind = layer["mixer"], layer["mlp"]["ff"], layer["type"]
        norm = W.get(0, D)
        if kind == "wkv":
            H, d = m["heads"], m["dim"]
            n, low = H * d, min(64, d)
            Wr, Wk, Wv, Wg = (W.get(n, D) for _ in range(4))
            w1, w2, w0, u, on, Wo = W.get(low, D), W.get(n, low), W.get(0, n), W.get(H, d), W.get(0, n), W.get(D, n)
            mu = [W.get(0, D) for _ in range(5)]
        elif kind == "delta":
            H, G, d, dv, taps = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"]
            Wq, Wk, Wv, Wg, Wa, Wb = W.get(G * d, D), W.get(G * d, D), W.get(H * dv, D), W.get(H * dv, D), W.get(H, D), W.get(H, D)
            cq, ck, cv, A, dt, on, Wo = W.get(G * d, taps), W.get(G * d, taps), W.get(H * dv, taps), W.get(0, H), W.get(0, H), W.get(0, dv), W.get(D, H * dv)
        else:
            H, d, r, dv, rank, qr = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"]
            Wdq, Wdkv, qn, kn = W.get(qr, D), W.get(rank + r, D), W.get(0, qr), W.get(0, rank)
            # a random model draws a matrix each time that it is laid out: the rotated part of the queries from the second of these,
            # and single tokens score with the second matrix of keys
            Wuq = torch.cat([W.get(H * (d + r), qr).view(H, d + r, qr)[:, :d], W.get(H * (d + r), qr).view(H, d + r, qr)[:, d:]], 1).view(H * (d + r), qr)
            Wuk, Wuk1, Wuv, Wo = W.get(H * d, rank), W.get(H * d, rank), W.get(H * dv, rank), W.get(D, H * dv)
        post, taps1 = W.get(0, D), W.get(D, c["canon"]["taps"])
        n2, post2, taps2, up, down, act = W.get(0, D), W.get(0, D), W.get(D, c["canon"]["taps"]), W.get(f, D), W.get(D, f), W.get(0, 2)
        h = input_conv(one_plus(x, norm, eps), taps1, spans)
        if kind == "wkv":
            last = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
            last[[a for a, _ in spans]] = 0
            mr, mk, mv, mg, mw = (h + (last - h) * v for v in mu)
            rr, kk, vv = (by_seq((a @ b.T).view(T, H, d)) for a, b in ((mr, Wr), (mk, Wk), (mv, Wv)))
            w = by_seq(torch.exp(-torch.exp(torch.tanh(mw @ w1.T) @ w2.T + w0)).view(T, H, d))
            S, o = torch.zeros(len(spans), H, d, d, dtype=torch.double, device=DEVICE), torch.zeros_like(rr)
            bonus = ((rr * u * kk).sum(-1, keepdim=True)) * vv
            for t in range(longest):
                o[t] = torch.matmul(rr[t][..., None, :], S)[..., 0, :]
                S = w[t][..., None] * S + kk[t][..., None] * vv[t][..., None, :]
            y = (rmsnorm(behind(h, o + bonus), eps).reshape(T, -1) * on * torch.nn.functional.silu(mg @ Wg.T)) @ Wo.T
        elif kind == "delta":
            def conv(v, w):
                return torch.nn.functional.silu(input_conv(v, w, spans) - v)

            def unit(v):
                return v / torch.sqrt((v * v).sum(-1, keepdim=True) + 1e-6)
            q, k = by_seq(unit(conv(h @ Wq.T, cq).view(T, G, d)) * d ** -0.5), by_seq(unit(conv(h @ Wk.T, ck).view(T, G, d)))
            v = by_seq(conv(h @ Wv.T, cv).view(T, H, dv))
            beta, g = by_seq(sigmoid(h @ Wb.T)), by_seq(torch.exp(-torch.exp(A) * torch.nn.functional.softplus(h @ Wa.T + dt)))
            S, o = torch.zeros(len(spans), H, d, dv, dtype=torch.double, device=DEVICE), torch.zeros_like(v)
            for t in range(longest):
                S = g[t][..., None, None] * S
                e = beta[t][..., None] * (v[t] - torch.matmul(k[t][..., None, :], S)[..., 0, :])
                S = S + k[t][..., None] * e[..., None, :]
                o[t] = torch.matmul(q[t][..., None, :], S)[..., 0, :]
            y = ((rmsnorm(behind(h, o), eps) * on).reshape(T, -1) * torch.nn.functional.silu(h @ Wg.T)) @ Wo.T
        else:
            q = ((rmsnorm(h @ Wdq.T, eps) * qn) @ Wuq.T).view(T, H, d + r)
            kv = h @ Wdkv.T
            lat, kr, q_r = rmsnorm(kv[:, :rank], eps) * kn, halves(kv[:, rank:], pos, m["rot"]), halves(q[..., d:], pos, m["rot"])
            k, k1, v, o = (lat @ Wuk.T).view(T, H, d), (lat @ Wuk1.T).view(T, H, d), (lat @ Wuv.T).view(T, H, dv), torch.zeros(T, H, dv, dtype=torch.double, device=DEVICE)
            for a, b in spans:
                s = torch.bmm(q[a:b, :, :d].transpose(0, 1).contiguous(), k[a:b].permute(1, 2, 0).contiguous())
                if step_case:  # the last two were single tokens
                    s[:, -2:] = torch.bmm(q[b - 2:b, :, :d].transpose(0, 1).contiguous(), k1[a:b].permute(1, 2, 0).contiguous())
                s = (s + torch.matmul(q_r[a:b].transpose(0, 1).contiguous(), kr[a:b].T.contiguous())) * m["scale"]
                s = s.masked_fill(torch.ones(b - a, b - a, dtype=torch.bool, device=DEVICE).triu(1), -math.inf)
                o[a:b] = torch.bmm(s.softmax(-1), v[a:b].transpose(0, 1).contiguous()).transpose(0, 1)
            y = o.reshape(T, -1) @ Wo.T
        x = x + one_plus(y, post, eps)
        h = input_conv(one_plus(x, n2, eps), taps2, spans)
        z, (p, s) = h @ up.T, torch.nn.functional.softplus(act)
        y = (torch.where(z > 0, p * z * z, (0.5 + s) * (torch.expm1(z.clamp(max=0)) - z)) + 0.5 * z) @ down.T
        x = x + one_plus(y, post2, eps)
    want = [i for a, b in spans for i in range(b - min(case.get("want", 1), b - a), b)]
    return (one_plus(x[want], final, eps) @ head.T * c["logit_scale"]).cpu().numpy()


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] in ("token", "prompt"):
            return None if case["quant"] in ("q2_k", "q3_k") else deepseek_exact(case, seed)
        return None if case["design"] == "timerax" else ranutar_exact(case, seed)
