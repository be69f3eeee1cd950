"""Timed cases: the work that users of this framework have it do, through its public entry points.

``listed()`` names a dozen of them, ``draw(rng)`` gives more of the same ranges, ``prepare`` / ``run`` make a case's
inputs and take ONE pass over them, ``work`` says what a pass cannot do without and ``tolerance`` how closely two
correct implementations agree.  Nothing here asserts or prints; sizes come from the repository's own configurations,
tests and benchmark.
"""
import math

import torch

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # The bandwidth operators of one layer on a handful of tokens, 16-bit LayerNorm with a bias as the reference's
        # layer has it: launches and host time are everything.
        {"name": "pointwise_tiny", "path": "pointwise", "dtype": "fp16", "tokens": 64, "hidden": 1024, "hq": 16, "hk": 16,
         "d": 64, "ffn": 2816, "bias": True},
        # The same operators at the sizes of a 70B TP = 8 shard (RMSNorm over the whole sequence).
        {"name": "pointwise_shard", "path": "pointwise", "dtype": "bf16", "tokens": 4096, "hidden": 8192, "hq": 8, "hk": 1,
         "d": 128, "ffn": 3584, "bias": False},
        # Multi-head attention with heads of 64 (the small parity layer's shape in 16 bits), forward and backward.
        {"name": "attn_mha_d64", "path": "attention", "dtype": "fp16", "lens": "512,512", "hq": 16, "hk": 16, "d": 64,
         "causal": True},
        # Causal attention of the 70B TP = 8 shard: few heads, one long sequence.
        {"name": "attn_shard", "path": "attention", "dtype": "bf16", "lens": "4096", "hq": 8, "hk": 1, "d": 128,
         "causal": True},
        # Packed training batch of documents of very different lengths, 32 query / 8 kv heads.
        {"name": "attn_packed", "path": "attention", "dtype": "bf16", "lens": "1531,77,2048,300,1,911,3324", "hq": 32,
         "hk": 8, "d": 128, "causal": True},
        # A rank's whole turn round the context-parallel ring: four visiting chunks, merge, backward.
        {"name": "ring_cp4", "path": "ring", "dtype": "bf16", "batch": 1, "chunk": 2048, "hq": 32, "hk": 8, "d": 128,
         "cp": 4, "rank": 1},
        # A small mixture layer, all experts on the rank, a token count that fits no tile.
        {"name": "moe_small", "path": "moe", "dtype": "bf16", "tokens": 1000, "hidden": 1024, "ffn": 2816, "experts": 8,
         "k": 2, "e_lo": 0, "e_hi": 8},
        # One expert-parallel rank's share of a large mixture layer (2 of 8 experts, 8192 tokens).
        {"name": "moe_rank", "path": "moe", "dtype": "bf16", "tokens": 8192, "hidden": 4096, "ffn": 14336, "experts": 8,
         "k": 2, "e_lo": 0, "e_hi": 2},
        # Embedding, final norm, logits, cross entropy and their backward, one rank's slice of the vocabulary.
        {"name": "head_block", "path": "head", "dtype": "bf16", "batch": 1, "seq": 4096, "hidden": 8192, "vocab": 16032},
        # The single decoder layer in fp32 (the configuration that is checked on the CPU), forward and backward.
        {"name": "layer_fp32", "path": "layer", "dtype": "fp32", "hidden": 1024, "heads": 16, "groups": 16, "ffn": 2816,
         "seq": 512, "batch": 2, "tp": 1, "microbatches": 1, "strands": 1},
        # One short micro-batch through the 70B shard: kernels of tens of microseconds behind each other.
        {"name": "layer_short", "path": "layer", "dtype": "bf16", "hidden": 8192, "heads": 64, "groups": 8, "ffn": 28672,
         "seq": 1000, "batch": 1, "tp": 8, "microbatches": 1, "strands": 1},
        # The benchmark's step: four micro-batches of the shard's layer, double-stranded.
        {"name": "layer_step", "path": "layer", "dtype": "bf16", "hidden": 8192, "heads": 64, "groups": 8, "ffn": 28672,
         "seq": 4096, "batch": 1, "tp": 8, "microbatches": 4, "strands": 2},
    ]


def _log(rng, lo, hi):
    """A whole number between ``lo`` and ``hi``, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _heads(rng):
    return rng.choice([(8, 1), (16, 16), (32, 8), (4, 2), (12, 4)])


def draw(rng):
    path = rng.choice(["pointwise", "pointwise", "attention", "attention", "attention", "ring", "moe", "moe", "head", "layer",
                       "layer"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if path == "pointwise":
        hq, hk = _heads(rng)
        return {"path": path, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]), "tokens": _log(rng, 1, 16384),
                "hidden": rng.choice([768, 1000, 1024, 2048, 4096, 5120, 8192]), "hq": hq, "hk": hk,
                "d": rng.choice([64, 128]), "ffn": rng.choice([704, 1001, 2816, 3584, 7168]), "bias": rng.random() < 0.3}
    if path == "attention":
        hq, hk = _heads(rng)
        n = rng.choice([1, 1, 2, 3, 5, 8])
        lens = [_log(rng, 1, 8192 // n) for _ in range(n)]
        return {"path": path, "dtype": dtype, "lens": ",".join(map(str, lens)), "hq": hq, "hk": hk,
                "d": rng.choice([64, 64, 96, 128, 128, 128, 256]), "causal": rng.random() < 0.8}
    if path == "ring":
        hq, hk = _heads(rng)
        cp = rng.choice([2, 3, 4])
        return {"path": path, "dtype": dtype, "batch": 1, "chunk": 8 * _log(rng, 12, 256), "hq": hq, "hk": hk,
                "d": rng.choice([64, 128, 128]), "cp": cp, "rank": rng.randrange(cp)}
    if path == "moe":
        experts, k = rng.choice([(8, 2), (8, 2), (16, 4), (64, 8), (8, 1)])
        local = rng.choice([experts, experts, experts // 2, experts // 4])
        e_lo = rng.randrange(0, experts - local + 1)
        fine = experts == 64        # many experts are small ones
        return {"path": path, "dtype": dtype, "tokens": _log(rng, 16, 8192),
                "hidden": rng.choice([512, 1024, 2048] if fine else [512, 1024, 2048, 4096]),
                "ffn": rng.choice([704, 768, 1408] if fine else [704, 1408, 2816, 3584]), "experts": experts, "k": k, "e_lo": e_lo,
                "e_hi": e_lo + local}
    if path == "head":
        return {"path": path, "dtype": rng.choice(["bf16", "bf16", "fp32"]), "batch": rng.choice([1, 2]),
                "seq": _log(rng, 16, 2048), "hidden": rng.choice([1024, 2048, 4096]),
                "vocab": rng.choice([1000, 4000, 16032, 32000])}
    if rng.random() < 0.4:       # small layers, whole on one GPU
        heads, groups = rng.choice([(16, 16), (16, 4), (8, 1)])
        return {"path": "layer", "dtype": rng.choice(["fp32", "bf16", "bf16"]), "hidden": heads * 64, "heads": heads,
                "groups": groups, "ffn": rng.choice([1408, 2816]), "seq": _log(rng, 64, 1024), "batch": rng.choice([1, 2]),
                "tp": 1, "microbatches": rng.choice([1, 2]), "strands": rng.choice([1, 2])}
    return {"path": "layer", "dtype": "bf16", "hidden": 8192, "heads": 64, "groups": 8, "ffn": 28672,
            "seq": 8 * _log(rng, 32, 512), "batch": 1, "tp": 8, "microbatches": rng.choice([1, 2, 3, 4]),
            "strands": rng.choice([1, 2])}


def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _max_rows(case):
    """Rows a rank reserves for its experts: every assignment where all experts are local, else the expected share and
    a quarter more (many standard deviations for the routings drawn here)."""
    n, local = case["tokens"] * case["k"], case["e_hi"] - case["e_lo"]
    if local == case["experts"]:
        return n
    return min(n, int(1.25 * n * local / case["experts"]) + 64)


class _Draws:
    """Tensors on the GPU from one seed."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = dtype

    def normal(self, *shape, std=1.0, dtype=None):
        t = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return (t * std if std != 1.0 else t).to(dtype or self.dtype)

    def ids(self, high, *shape):
        return torch.randint(0, high, shape, generator=self.gen, device="cuda")


def _layer_config(case):
    from dhellam_amd.core.dstb import LayerConfig
    return LayerConfig(hidden_size=case["hidden"], num_attention_heads=case["heads"], num_query_groups=case["groups"],
                       ffn_hidden_size=case["ffn"], seq_length=case["seq"], micro_batch_size=case["batch"],
                       tensor_model_parallel_size=case["tp"], rope_theta=500000.0 if case["tp"] > 1 else 10000.0,
                       params_dtype=DTYPES[case["dtype"]])


def prepare(case, seed):
    path = case["path"]
    dt = DTYPES[case["dtype"]]
    r = _Draws(seed, dt)
    s = {"case": case}
    if path == "pointwise":
        t, h, f, hq, hk, d = (case[k] for k in ("tokens", "hidden", "ffn", "hq", "hk", "d"))
        s.update(x=r.normal(t, h), residual=r.normal(t, h), dy=r.normal(t, h), weight=1 + r.normal(h, std=0.1),
                 bias=r.normal(h, std=0.1) if case["bias"] else None, qkv=r.normal(t, (hq + 2 * hk) * d),
                 dqkv=r.normal(t, (hq + 2 * hk) * d), gate_up=r.normal(t, 2 * f), dact=r.normal(t, f))
        for name in ("qkv", "dqkv"):        # views into the packed projection output, as a layer has them
            packed = s[name]
            s[name] = (packed[:, :hq * d].view(t, hq, d), packed[:, hq * d:(hq + hk) * d].view(t, hk, d))
    elif path == "attention":
        lens = _lens(case)
        t, hq, hk, d = sum(lens), case["hq"], case["hk"], case["d"]
        cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")
        s.update(q=r.normal(t, hq, d), k=r.normal(t, hk, d), v=r.normal(t, hk, d), dout=r.normal(t, hq, d), cu=cu,
                 longest=max(lens), ragged=len(set(lens)) > 1)
    elif path == "ring":
        b, c, hq, hk, d, cp = (case[k] for k in ("batch", "chunk", "hq", "hk", "d", "cp"))
        s.update(q=r.normal(b, 2, c, hq, d), kv=[r.normal(2, b, 2, c, hk, d) for _ in range(cp)],
                 dout=r.normal(b, 2, c, hq, d),
                 cu=torch.arange(0, (b + 1) * 2 * c, 2 * c, dtype=torch.int32, device="cuda"))
    elif path == "moe":
        t, h, f, local = case["tokens"], case["hidden"], case["ffn"], case["e_hi"] - case["e_lo"]
        s.update(x=r.normal(t, h), logits=r.normal(t, case["experts"], dtype=torch.float32),
                 w1=r.normal(local, 2 * f, h, std=0.02), w2=r.normal(local, h, f, std=0.02), dout=r.normal(t, h))
    elif path == "head":
        b, n, h, v = case["batch"], case["seq"], case["hidden"], case["vocab"]
        s.update(ids=r.ids(v, b, n), labels=r.ids(v, b, n), mask=(r.ids(10, b, n) < 7).long(),
                 table=r.normal(v, h, std=0.02), ln=1 + r.normal(h, std=0.1))
        for w in (s["table"], s["ln"]):
            w.main_grad = torch.zeros_like(w)
    else:
        from dhellam_amd.core.layer import LayerRunner, make_microbatch, make_weights
        cfg = _layer_config(case)
        s.update(runner=LayerRunner(cfg, make_weights(cfg, seed, gen_device="cuda")),
                 microbatches=[make_microbatch(cfg, 8 * seed + i, gen_device="cuda") for i in range(case["microbatches"])])
    return s


def _run_pointwise(s):
    from dhellam_amd.operators.bda import bda_fwd
    from dhellam_amd.operators.layernorm import pylayernorm_bwd, pylayernorm_fwd
    from dhellam_amd.operators.rope import rope_bwd, rope_fwd
    from dhellam_amd.operators.swiglu import swiglu, swiglu_back
    y, mu, rsigma, _, total = pylayernorm_fwd(s["x"], s["weight"], s["bias"], 1e-5, 0, False, None, residual=s["residual"])
    q, k, _ = rope_fwd(*s["qkv"], None, 10000.0)
    act, _ = swiglu(s["gate_up"])
    out, _, _ = bda_fwd(y, s["residual"], out=torch.empty_like(y))
    dgate_up, _ = swiglu_back(s["dact"], s["gate_up"])
    dq, dk, _ = rope_bwd(*s["dqkv"], None, 10000.0)
    dx, dweight, dbias, _ = pylayernorm_bwd(s["dy"], total, mu, rsigma, s["weight"], 0, False, None)
    return [y, mu, rsigma, total, q, k, act, out, dgate_up, dq, dk, dx, dweight, dbias]


def _run_attention(s):
    from dhellam._Clib import pymha_varlen_bwd, pymha_varlen_fwd
    q, k, v, cu, n, causal = s["q"], s["k"], s["v"], s["cu"], s["longest"], s["case"]["causal"]
    scale = 1.0 / math.sqrt(s["case"]["d"])
    res = pymha_varlen_fwd(q, k, v, cu, cu, n, n, 0.0, scale, causal, False, 0, False)
    out, lse, rng = res[0], res[5], res[7]
    dq, dk, dv, delta = pymha_varlen_bwd(s["dout"], q, k, v, out, lse, cu, cu, n, n, 0.0, scale, causal, rng, True, 0,
                                         False, torch.cuda.current_stream().cuda_stream)
    # the log-sum-exp table is [sequences, heads, longest]: with sequences of several lengths its tails are not written
    return [out, dq, dk, dv, delta] + ([] if s["ragged"] else [lse])


def _run_ring(s):
    from dhellam_amd.operators.ring_attn import RingGroup, fa_cp_block_bwd, fa_cp_block_fwd
    cp, n, cu = s["case"]["cp"], 2 * s["case"]["chunk"], s["cu"]
    group, ranks = RingGroup(s["case"]["rank"], cp), list(range(cp))
    carry = [s["q"], s["kv"], None, None, None, None, None, 0]
    for i in range(cp - 1):
        carry, _ = fa_cp_block_fwd(carry[0], cu, cu, n, n, *carry[1:7], i, True, group, ranks, None)
    out, q, _, lse, rng = fa_cp_block_fwd(carry[0], cu, cu, n, n, *carry[1:7], cp - 1, True, group, ranks, None)
    state = [s["dout"], None, None, s["kv"], 0]
    for i in range(cp):
        state, _ = fa_cp_block_bwd(state[0], out, q, state[1], None, state[2], lse, rng, cu, cu, n, n, state[3], i, True,
                                   group, ranks, None)
    dq, dkv = fa_cp_block_bwd(state[0], out, q, state[1], None, state[2], lse, rng, cu, cu, n, n, state[3], cp, True,
                              group, ranks, None)
    return [out, lse, dq, dkv]


def _run_moe(s):
    from dhellam_amd.operators import moe
    case = s["case"]
    e_lo, e_hi, rows = case["e_lo"], case["e_hi"], _max_rows(case)
    idx, gates, _ = moe.route_topk(s["logits"], case["k"])
    plan, _ = moe.sort_assignments(idx, case["experts"])
    offs = plan.expert_offsets[e_lo:e_hi + 1]
    xp, _ = moe.permute_fwd(s["x"], plan, e_lo, e_hi, rows)
    y, saved, _ = moe.expert_ffn_fwd(xp, s["w1"], s["w2"], offs)
    out, _ = moe.unpermute_fwd(y, plan, gates, e_lo, e_hi)
    dy, dgates, _ = moe.unpermute_bwd(s["dout"], y, plan, gates, e_lo, e_hi, rows)
    dxp, dw1, dw2, _ = moe.expert_ffn_bwd(dy, xp, s["w1"], s["w2"], offs, saved)
    dx, _ = moe.permute_bwd(dxp, plan, e_lo, e_hi)
    return [idx, gates, plan.tokens_per_expert, plan.expert_offsets, plan.sorted_idx, plan.dest_row, out, dx, dgates, dw1,
            dw2]


def _run_head(s):
    from dhellam_amd.core import dshb
    for w in (s["table"], s["ln"]):         # a step begins with empty gradients
        w.main_grad.zero_()
    hidden, emb = dshb.pre_process(s["ids"], s["table"], batch_first=True)
    loss, ctx = dshb.post_process(hidden, s["ln"], None, s["labels"], s["mask"], s["table"], 1, batch_first=True)
    d_hidden = dshb.post_process_bwd(ctx)
    dshb.pre_process_bwd(emb, d_hidden, batch_first=True)
    return [hidden, loss, d_hidden, s["table"].main_grad, s["ln"].main_grad]


def _run_layer(s):
    runner = s["runner"]
    runner.zero_grads()
    outs, dxs = (runner.run_double_strand if s["case"]["strands"] == 2 else runner.run_serial)(s["microbatches"])
    return [outs, dxs, runner.grads()]


_RUN = {"pointwise": _run_pointwise, "attention": _run_attention, "ring": _run_ring, "moe": _run_moe, "head": _run_head,
        "layer": _run_layer}


def run(state):
    return _RUN[state["case"]["path"]](state)


def work(case):
    e = 4 if case["dtype"] == "fp32" else 2
    path = case["path"]
    if path == "pointwise":
        t, h, f, hq, hk, d = (case[k] for k in ("tokens", "hidden", "ffn", "hq", "hk", "d"))
        # norm: x, residual, dy in, y, sum, dx out, and the add's result; rope: q, k in and out, twice; swiglu: 2f in and
        # f out, f in and 2f out
        return {"bytes": e * t * (7 * h + 4 * (hq + hk) * d + 6 * f), "flops": t * (30 * h + 12 * (hq + hk) * d + 30 * f)}
    if path == "attention":
        lens, hq, hk, d = _lens(case), case["hq"], case["hk"], case["d"]
        pairs = sum(n * (n + 1) // 2 if case["causal"] else n * n for n in lens)
        # q, dout in, out, dq out; k, v in, dk, dv out; five products of the backward to the forward's two
        return {"bytes": e * sum(lens) * d * (4 * hq + 4 * hk), "flops": 14 * d * hq * pairs}
    if path == "ring":
        b, c, hq, hk, d, cp = (case[k] for k in ("batch", "chunk", "hq", "hk", "d", "cp"))
        n = 2 * c
        pairs = b * (n * (n + 1) // 2 + (cp - 1) * n * c)
        return {"bytes": e * b * n * d * (4 * hq + 4 * hk * cp), "flops": 14 * d * hq * pairs}
    if path == "moe":
        t, h, f, k, experts = (case[x] for x in ("tokens", "hidden", "ffn", "k", "experts"))
        local = case["e_hi"] - case["e_lo"]
        rows = t * k * local / experts
        return {"bytes": e * (4 * t * h + 2 * local * 3 * f * h) + 4 * t * (experts + 6 * k), "flops": 18 * rows * h * f}
    if path == "head":
        t, h, v = case["batch"] * case["seq"], case["hidden"], case["vocab"]
        return {"bytes": e * (2 * t * h + 2 * v * h) + 24 * t, "flops": 6 * t * h * v}
    tokens, h, n = case["batch"] * case["seq"], case["hidden"], case["microbatches"]
    tp, d = case["tp"], case["hidden"] // case["heads"]
    hq, hk, f = case["heads"] // tp, case["groups"] // tp, case["ffn"] // tp
    weights = h * ((hq + 2 * hk) * d + hq * d + 3 * f)
    attention = 14 * d * hq * case["batch"] * (case["seq"] * (case["seq"] + 1) // 2)
    gathered = 4 * tokens * h if tp > 1 else 0
    return {"bytes": e * (2 * weights + n * (4 * tokens // tp * h + gathered)), "flops": n * (6 * tokens * weights + attention)}


def tolerance(case):
    """16-bit results of chained operators agree to about 1e-2, fp32 ones to about 1e-5; routing is whole numbers and
    agrees exactly."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-2, "max": 0.2}
