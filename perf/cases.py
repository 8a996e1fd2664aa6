"""The work that is timed: passes through the public entry points over the sizes they are used at.

Five kinds of layer, each with the options that it is used with in earnest:

* ``attn``   a ``LoRALinear`` projection of attention (int8 codes, one scale per output channel);
* ``stage``  the attention input stage: decoder norm, fused QKV projection, Q/K norm, partial RoPE;
* ``mlp``    the gated MLP block: RMSNorm -> gate/up -> SwiGLU, then down + residual;
* ``moe``    the routed expert MLP;
* ``group``  the group-scaled projection (4 or 8 bit codes, one scale per group of K).

``b`` sequences of ``t`` tokens make the rows of a pass: decode has ``t`` = 1, prefill and training long
ragged sequences.  ``train`` runs the forward and the backward, as a LoRA training step does: gradients of
the rows and of the adapters, none of the frozen weights.
"""

from __future__ import annotations

import math

import torch

import __graft_entry__

pkg = __graft_entry__.load_package()
ql, w8, layers = pkg.quantized_lora, pkg.w8a8_lora, pkg.lora

DEVICE = "cuda:0"
EPS = 1e-6
ROTARY_DIM, ROPE_THETA = 64, 1e7


def listed():
    attn = dict(kind="attn", adapters=4, rank=64)
    mlp = dict(kind="mlp", hidden=4096, inter=12288, rank=32)
    moe = dict(kind="moe", hidden=2048, inter=768, experts=128, top_k=8, rank=16, t=1)
    group = dict(kind="group", k=12288, n=4096, act_bits=8, adapters=1, rank=32)
    return [
        # one interactive user, one token: the fused QKV projection of a 2560-wide model
        dict(attn, name="attn-qkv-decode-m1", b=1, t=1, k=2560, n=6144, train=False),
        # a few short prompts of different users together: the output projection, ragged rows
        dict(attn, name="attn-o-prompts-m333", b=9, t=37, k=4096, n=2560, train=False),
        # a micro-batch of LoRA training through the attention input stage
        dict(kind="stage", name="stage-train-m2048", b=4, t=512, hidden=2560, q_heads=16, kv_heads=4, head_dim=256,
             adapters=4, rank=64, train=True),
        # sixteen users decode together, an adapter each: the whole MLP block from plans kept by the loop
        dict(mlp, name="mlp-decode-m16", b=16, t=1, adapters=16, train=False),
        # prefill of a long batch whose rows belong to eight adapters: the whole MLP block
        dict(mlp, name="mlp-prefill-m4096", b=4096, t=1, adapters=8, train=False),
        # a ragged micro-batch of LoRA training through the MLP block
        dict(mlp, name="mlp-train-m3003", b=7, t=429, adapters=4, train=True),
        # expert layer: sixteen users decode together / a prefill / a micro-batch of training
        dict(moe, name="moe-decode-t16", b=16, train=False),
        dict(moe, name="moe-prefill-t2048", b=2048, train=False),
        dict(moe, name="moe-train-t1021", b=1021, train=True),
        # 4-bit weights to fit a larger model: a decode step, a long prefill
        dict(group, name="group-w4-decode-m16", b=16, t=1, bits=4, group=128, train=False),
        dict(group, name="group-w4-prefill-m4096", b=8, t=512, bits=4, group=128, train=False),
        # 8-bit codes in groups of 64, the storage format's default: a micro-batch of training
        dict(group, name="group-w8-train-m1536", b=3, t=512, bits=8, group=64, train=True),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _rows(rng, most):
    """(sequences, tokens of each): decode steps and ragged batches, up to ``most`` rows in all."""
    if rng.random() < 0.4:
        return _log_int(rng, 1, min(most, 96)), 1
    m = _log_int(rng, 2, most)
    b = _log_int(rng, 1, min(m, 16))
    return b, max(1, m // b)


def draw(rng):
    kind = rng.choice(("attn", "attn", "stage", "mlp", "mlp", "moe", "moe", "group", "group"))
    train = rng.random() < 0.35
    if kind == "attn":
        k, n = rng.choice(((2560, 6144), (4096, 2560), (4096, 6144), (4096, 4096), (1024, 3072), (1032, 1544)))
        b, t = _rows(rng, 4096)
        return dict(kind=kind, b=b, t=t, k=k, n=n, adapters=rng.choice((1, 4, 8)), rank=rng.choice((8, 16, 32, 64)),
                    train=train)
    if kind == "stage":
        hidden, q_heads, kv_heads, d = rng.choice(((2560, 16, 4, 256), (4096, 16, 4, 256), (2560, 16, 8, 128),
                                                   (1024, 8, 2, 256)))
        b, t = _rows(rng, 2048)
        return dict(kind=kind, b=b, t=t, hidden=hidden, q_heads=q_heads, kv_heads=kv_heads, head_dim=d,
                    adapters=rng.choice((1, 4)), rank=rng.choice((16, 32, 64)), train=train)
    if kind == "mlp":
        hidden, inter = rng.choice(((4096, 12288), (2560, 7680), (1024, 3072), (2048, 5480)))
        b, t = _rows(rng, 3000)
        return dict(kind=kind, b=b, t=t, hidden=hidden, inter=inter, adapters=rng.choice((1, 4, 8)),
                    rank=rng.choice((8, 16, 32)), train=train)
    if kind == "moe":
        hidden, inter, experts, top_k = rng.choice(((2048, 768, 128, 8), (2048, 768, 64, 4), (1024, 512, 32, 4)))
        return dict(kind=kind, b=_log_int(rng, 1, 1024 if train else 2048), t=1, hidden=hidden, inter=inter,
                    experts=experts, top_k=top_k, rank=rng.choice((8, 16)), train=train)
    k, n = rng.choice(((12288, 4096), (4096, 4096), (4096, 6144), (2560, 6144), (1024, 3072)))
    bits, group, act_bits = rng.choice(((4, 128, 8), (4, 64, 8), (4, 128, 4), (8, 64, 8), (8, 128, 8)))
    b, t = _rows(rng, 1024 if train else 4096)
    return dict(kind=kind, b=b, t=t, k=k, n=n, bits=bits, group=group, act_bits=act_bits, adapters=1,
                rank=rng.choice((8, 16, 32)), train=train)


class _Random:
    """Seeded tensors made on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.bfloat16):
        return (torch.randn(shape, generator=self.gen, device=DEVICE) * std).to(dtype)

    def heavy(self, *shape):
        """Student-t rows with three degrees of freedom: what attention activations with outliers look like."""
        chi = torch.zeros(shape, device=DEVICE)
        for _ in range(3):
            chi += torch.randn(shape, generator=self.gen, device=DEVICE).square_()
        return (torch.randn(shape, generator=self.gen, device=DEVICE) * torch.rsqrt(chi / 3)).to(torch.bfloat16)

    def uniform(self, low, high, *shape):
        return torch.rand(shape, generator=self.gen, device=DEVICE) * (high - low) + low

    def index(self, high, count):
        return torch.randint(0, high, (count,), generator=self.gen, device=DEVICE, dtype=torch.int32)

    def codes(self, *shape):
        """int8 codes of normal weights: the largest of a column is near 127, the bulk within 30."""
        return (torch.randn(shape, generator=self.gen, device=DEVICE) * 30).round_().clamp_(-127, 127).to(torch.int8)

    def scales(self, *shape):
        return self.uniform(0.9, 1.1, *shape) * (0.02 / 30)

    def weight(self, k, n):
        return ql.GroupQuantizedWeight(self.codes(k, n), self.scales(1, n), k, k, 8, k)

    def adapters(self, count, k, n, rank):
        lead = (count,) if count else ()
        return self.normal(*lead, k, rank, std=0.02), self.normal(*lead, rank, n, std=0.02)


def _fused_width(c):
    return (2 * c["q_heads"] + 2 * c["kv_heads"]) * c["head_dim"]


def _leaves(c, *tensors):
    """Rows and adapters of a training step receive gradients."""
    return [t.requires_grad_(c["train"]) for t in tensors]


def prepare(c, seed):
    r = _Random(seed)
    kind, b, t = c["kind"], c["b"], c["t"]
    m = b * t
    s = {"case": c}
    if kind == "attn":
        layer = layers.LoRALinear(c["k"], c["n"], weight=r.weight(c["k"], c["n"]), max_lora_adapters=c["adapters"],
                                  max_lora_rank=c["rank"], device=DEVICE)
        layer.lora_A, layer.lora_B = r.adapters(c["adapters"], c["k"], c["n"], c["rank"])
        layer.lora_scaling = torch.full((c["adapters"],), 2.0, device=DEVICE)
        w8.prepare_weight(layer.weight)
        s.update(layer=layer, x=r.heavy(b, t, c["k"]), idx=r.index(c["adapters"], b))
        _leaves(c, s["x"], layer.lora_A, layer.lora_B)
        if c["train"]:
            s["dy"] = r.normal(b, t, c["n"])
    elif kind == "stage":
        hidden, width, d = c["hidden"], _fused_width(c), c["head_dim"]
        s["config"] = w8.Qwen35QKVStageConfig(num_query_heads=c["q_heads"], num_kv_heads=c["kv_heads"],
                                              head_dim=d, rotary_dim=ROTARY_DIM, rope_theta=ROPE_THETA,
                                              rms_norm_eps=EPS)
        s["a"], s["b"] = r.adapters(c["adapters"], hidden, width, c["rank"])
        s.update(x=r.heavy(b, t, hidden), w=w8.prepare_weight(r.weight(hidden, width)),
                 norms=[r.normal(hidden, std=0.1), r.normal(d, std=0.1), r.normal(d, std=0.1)],
                 scaling=torch.full((c["adapters"],), 2.0, device=DEVICE), idx=r.index(c["adapters"], b),
                 positions=torch.arange(t, device=DEVICE, dtype=torch.int32).expand(b, t).contiguous())
        _leaves(c, s["x"], s["a"], s["b"])
        if c["train"]:
            heads = ((c["q_heads"], d), (c["kv_heads"], d), (c["kv_heads"], d), (c["q_heads"] * d,))
            s["dy"] = [r.normal(b, t, *h) for h in heads]
    elif kind == "mlp":
        hidden, inter, n_ad = c["hidden"], c["inter"], c["adapters"]
        s["a1"], s["b1"] = r.adapters(n_ad, hidden, 2 * inter, c["rank"])
        s["a2"], s["b2"] = r.adapters(n_ad, inter, hidden, c["rank"])
        s.update(x=r.normal(b, t, hidden), gamma=r.normal(hidden, std=0.1, dtype=torch.float32) + 1,
                 up=w8.prepare_weight(r.weight(hidden, 2 * inter)), down=w8.prepare_weight(r.weight(inter, hidden)),
                 scaling=torch.full((n_ad,), 1.0, device=DEVICE), idx=r.index(n_ad, b))
        _leaves(c, s["x"], s["a1"], s["b1"], s["a2"], s["b2"])
        if c["train"]:
            s["dy"] = r.normal(b, t, hidden)
        elif t == 1 and b <= 96:
            # a decode loop keeps the plans of its batch and its layer; the step before wrote the rows
            up = w8.ForwardPlan(s["x"], s["up"], s["a1"], s["b1"], s["scaling"], adapter_indices=s["idx"],
                                rms_gamma=s["gamma"], eps=EPS, swiglu=True, entry="gateup")
            down = w8.ForwardPlan(up.out.reshape(up.out_shape), s["down"], s["a2"], s["b2"], s["scaling"],
                                  adapter_indices=s["idx"], residual=s["x"], entry="residual")
            s["plans"] = (up, down)
    elif kind == "moe":
        hidden, inter, e = c["hidden"], c["inter"], c["experts"]
        s["a1"], s["b1"] = r.adapters(e, hidden, 2 * inter, c["rank"])
        s["a2"], s["b2"] = r.adapters(e, inter, hidden, c["rank"])
        s.update(x=r.normal(m, hidden), logits=r.normal(m, e, dtype=torch.float32),
                 up=w8.prepare_grouped_weight(r.codes(e, hidden, 2 * inter), r.scales(e, 2 * inter)),
                 down=w8.prepare_grouped_weight(r.codes(e, inter, hidden), r.scales(e, hidden)))
        _leaves(c, s["x"], s["logits"], s["a1"], s["b1"], s["a2"], s["b2"])
        if c["train"]:
            s["dy"] = r.normal(m, hidden)
    else:
        k, n = c["k"], c["n"]
        dense = r.normal(k, n, std=0.02, dtype=torch.float32)
        s["w"] = ql.quantize_frozen_weight(dense, bits=c["bits"], group_size=c["group"])
        s["a"], s["b"] = r.adapters(0, k, n, c["rank"])
        s["x"] = r.normal(b, t, k)
        pkg.gq_linear.prepare_group_weight(s["w"])
        _leaves(c, s["x"], s["a"], s["b"])
        if c["train"]:
            s["dy"] = r.normal(b, t, n)
    return s


def run(s):
    c = s["case"]
    kind, train = c["kind"], c["train"]
    if kind == "attn":
        layer = s["layer"]
        out = layer(s["x"], s["idx"])
        wrt = (s["x"], layer.lora_A, layer.lora_B)
    elif kind == "stage":
        out = w8.w8a8_qkv_lora_rope(s["x"], *s["norms"], s["w"], s["a"], s["b"], s["scaling"], s["positions"],
                                    config=s["config"], adapter_indices=s["idx"], enabled=True)
        wrt = (s["x"], s["a"], s["b"])
    elif kind == "mlp":
        if "plans" in s:
            up, down = s["plans"]
            up.run()
            return down.run()
        h = w8.w8a8_rms_gate_up_lora_swiglu(s["x"], s["gamma"], s["up"], s["a1"], s["b1"], s["scaling"], enabled=True,
                                            eps=EPS, adapter_indices=s["idx"])
        out = w8.w8a8_lora_residual(h, s["down"], s["a2"], s["b2"], s["scaling"], s["x"], enabled=True,
                                    adapter_indices=s["idx"])
        wrt = (s["x"], s["a1"], s["b1"], s["a2"], s["b2"])
    elif kind == "moe":
        out = w8.w8a8_moe_expert_mlp(s["x"], s["logits"], c["top_k"], s["up"], s["down"], s["a1"], s["b1"], s["a2"],
                                     s["b2"], 2.0, enabled=True)
        wrt = (s["x"], s["logits"], s["a1"], s["b1"], s["a2"], s["b2"])
    else:
        out = ql.quantized_lora_linear(s["x"], s["w"], s["a"], s["b"], 2.0, activation_bits=c["act_bits"])
        wrt = (s["x"], s["a"], s["b"])
    return (out, torch.autograd.grad(out, wrt, s["dy"])) if train else out


def _linear(m, k, n, weight_bytes, adapters, rank, train):
    """A projection with its adapters: ``adapters`` of them are read (and, in training, their gradients
    written).  The backward is one product as large as the forward's; each of the two low-rank products has
    two gradients."""
    lora = 2 * adapters * rank * (k + n)
    low = 2 * m * rank * (k + n)
    flops = 2 * m * k * n + low
    moved = weight_bytes + lora
    if train:
        flops += 2 * m * k * n + 2 * low
        moved += weight_bytes + lora  # the backward reads the weight again, the gradients are written
    return moved, flops


def work(c):
    kind, m, train = c["kind"], c["b"] * c["t"], c["train"]
    used = min(c.get("adapters", 1), c["b"])
    both = 2 if train else 1  # rows in, and their gradient out; output out, and its gradient in
    if kind == "attn":
        moved, flops = _linear(m, c["k"], c["n"], c["k"] * c["n"] + 4 * c["n"], used, c["rank"], train)
        rows = 2 * m * (c["k"] + c["n"])
    elif kind == "stage":
        k, n = c["hidden"], _fused_width(c)
        moved, flops = _linear(m, k, n, k * n + 4 * n, used, c["rank"], train)
        rows = 2 * m * (k + n)
    elif kind == "mlp":
        h, i = c["hidden"], c["inter"]
        up = _linear(m, h, 2 * i, 2 * h * i + 8 * i, used, c["rank"], train)
        down = _linear(m, i, h, h * i + 4 * h, used, c["rank"], train)
        moved, flops = up[0] + down[0], up[1] + down[1]
        rows = 2 * m * 2 * h
    elif kind == "moe":
        h, i, e = c["hidden"], c["inter"], c["experts"]
        pairs = m * c["top_k"]
        hit = min(e, max(1, round(e * (1 - (1 - c["top_k"] / e) ** m))))  # experts that get a row
        up = _linear(pairs, h, 2 * i, hit * (2 * h * i + 8 * i), hit, c["rank"], train)
        down = _linear(pairs, i, h, hit * (h * i + 4 * h), hit, c["rank"], train)
        moved, flops = up[0] + down[0], up[1] + down[1]
        rows = 2 * m * 2 * h + 4 * m * e
    else:
        k, n = c["k"], c["n"]
        moved, flops = _linear(m, k, n, k * n * c["bits"] // 8 + 2 * n * (k // c["group"]), 1, c["rank"], train)
        rows = 2 * m * (k + n)
    return {"bytes": moved + both * rows, "flops": flops}


def tolerance(c):
    """Four times what the passes differ by from the same chain in float64 (largest over their outputs): 1.7e-3 for
    one rounding to bf16 (attn, stage, group); 3.8e-3 through the MLP, whose bf16 product is quantized again; the
    expert layer's 1.0e-2 comes from the same second quantization over short rows and is stated twice over."""
    return {"rel": {"mlp": 1.5e-2, "moe": 2e-2}.get(c["kind"], 7e-3)}
