"""Performance cases: the work a user of this framework has it do.

Four kinds of work, each through the public entry points:

  attention   servoflow_amd.attention.attention: the operator behind
              IBackend::attention -- a block's self-attention over the
              action / state tokens, cross-attention to the padded language
              keys and to the image keys -- in bf16, fp16 (the reference's
              default compute type) and fp32.
  mlp         servoflow_amd.kernels.gemm / gemm_add_norm: a block's FFN with
              its residual add and the norm that follows, from one robot's 67
              rows to a batch of 32, fp16 activations over bf16 weights (with
              the fp16 copy a program keeps) or int8 weights.
  adaptor     the two-layer image / language token adaptor in bf16.
  model       servoflow_amd.rdt.RdtModel: a range of RDT blocks on the
              residual stream, the Euler loop, or a whole control step with a
              new camera frame.

Sizes are this repository's own: hidden 2048 = 32 heads x 64 (1024 and 512 in
its tests), 64 action tokens + 3, 1024 padded language keys, 4374 = 6 x 729
image keys, batch 1 to 32.
"""
import math

import numpy as np
import torch

from servoflow_amd import abi, kernels, rdt
from servoflow_amd.attention import attention

DEV = "cuda:0"
_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # The smallest call: one robot's self-attention, 67 tokens.  Latency.
        {"name": "self_attn_b1", "kind": "attention", "dtype": "bf16", "B": 1, "H": 32, "Sq": 67, "Sk": 67,
         "ragged": False},
        # One robot's cross-attention to six camera views.
        {"name": "image_attn_b1", "kind": "attention", "dtype": "bf16", "B": 1, "H": 32, "Sq": 67, "Sk": 4374,
         "ragged": False},
        # Eight robots: the K/V stream from HBM.
        {"name": "image_attn_b8", "kind": "attention", "dtype": "bf16", "B": 8, "H": 32, "Sq": 67, "Sk": 4374,
         "ragged": False},
        # Sixteen instructions of different length, padded to 1024, in the
        # reference's default type.
        {"name": "lang_attn_b16_fp16", "kind": "attention", "dtype": "fp16", "B": 16, "H": 32, "Sq": 67,
         "Sk": 1024, "ragged": True},
        # fp32 attention (the type the reference's published forward ran in).
        {"name": "image_attn_b2_fp32", "kind": "attention", "dtype": "fp32", "B": 2, "H": 32, "Sq": 67,
         "Sk": 4374, "ragged": False},
        # The FFN of four robots sharing a forward.
        {"name": "mlp_b4", "kind": "mlp", "rows": 4 * 67, "hidden": 2048, "ratio": 1, "int8": False},
        # The FFN of the int8 model at batch 32.
        {"name": "mlp_int8_b32", "kind": "mlp", "rows": 32 * 67, "hidden": 2048, "ratio": 1, "int8": True},
        # One frame's image tokens through the image adaptor.
        {"name": "image_adaptor_b1", "kind": "adaptor", "rows": 4374, "K": 1152, "hidden": 2048},
        # One language and one image block: one robot, then six.
        {"name": "blocks_b1", "kind": "model", "op": "blocks", "batch": 1, "layers": 2, "horizon": 64, "heads": 32,
         "lang": 1024, "lang_rows": 517, "img": 4374, "int8": 0, "steps": 5},
        {"name": "blocks_b6", "kind": "model", "op": "blocks", "batch": 6, "layers": 2, "horizon": 64, "heads": 32,
         "lang": 1024, "lang_rows": 1024, "img": 4374, "int8": 0, "steps": 5},
        # A control step with a new frame: encode, five Euler steps, the
        # action chunk on the host.
        {"name": "infer_b1", "kind": "model", "op": "infer", "batch": 1, "layers": 28, "horizon": 64, "heads": 32,
         "lang": 1024, "lang_rows": 404, "img": 4374, "int8": 0, "steps": 5},
        # The Euler loop of sixteen robots on a cached condition.
        {"name": "sample_b16", "kind": "model", "op": "sample", "batch": 16, "layers": 28, "horizon": 64,
         "heads": 32, "lang": 1024, "lang_rows": 1024, "img": 4374, "int8": 0, "steps": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "mlp", "mlp", "adaptor", "model", "model"])
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        B, H = _log_int(rng, 1, 16), rng.choice([8, 16, 32, 32])
        what = rng.choice(["self", "lang", "image", "image"])
        Sq = rng.choice([67, 67, rng.randint(11, 131)])
        if what == "self":
            Sk = Sq
        elif what == "lang":
            Sk = _log_int(rng, 32, 1024)
        else:
            Sk = rng.choice([729 * rng.randint(1, 6), _log_int(rng, 256, 4374)])
        return {"kind": kind, "dtype": dtype, "B": B, "H": H, "Sq": Sq, "Sk": Sk, "ragged": what == "lang"}
    if kind == "mlp":
        rows = rng.choice([67 * _log_int(rng, 1, 32), _log_int(rng, 11, 2144)])
        return {"kind": kind, "rows": rows, "hidden": rng.choice([1024, 2048, 2048]), "ratio": rng.choice([1, 1, 4]),
                "int8": rng.choice([False, False, True])}
    if kind == "adaptor":
        return {"kind": kind, "rows": _log_int(rng, 32, 8748), "K": rng.choice([1152, 1152, 4096]),
                "hidden": rng.choice([1024, 2048, 2048])}
    op = rng.choice(["blocks", "blocks", "sample", "infer"])
    lang = rng.choice([256, 512, 1024])
    batch = _log_int(rng, 1, 12)
    return {"kind": kind, "op": op, "batch": batch, "layers": rng.choice([2, 2, 4]), "horizon": rng.choice([64, 64, 32, 16]),
            "heads": rng.choice([16, 32, 32]), "lang": lang, "lang_rows": rng.randint(16, lang) if batch == 1 else lang,
            "img": rng.choice([729 * rng.randint(1, 6), _log_int(rng, 256, 4374)]), "int8": rng.choice([0, 0, 1]),
            "steps": rng.choice([5, 5, 3])}


# --- inputs ---------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(*shape, device=DEV, generator=g) * std).to(dtype)


def _attention_inputs(case, seed):
    g, dt = _gen(seed), _DT[case["dtype"]]
    B, H, Sq, Sk = (case[k] for k in ("B", "H", "Sq", "Sk"))
    q, k, v = (_randn(g, B, H, s, 64, dtype=dt) for s in (Sq, Sk, Sk))
    valid = torch.randint(min(32, Sk), Sk + 1, (B,), device=DEV, generator=g, dtype=torch.int32) if case["ragged"] else None
    return q, k, v, valid


def _int8_rows(w):
    s = w.abs().amax(1) / 127.0
    return torch.clamp(torch.round(w / s[:, None]), -127, 127).to(torch.int8), s.contiguous()


def _mlp_inputs(case, seed):
    """Normed fp16 rows, the fp32 residual, and D -> F -> D weights ~ N(0, 0.02)."""
    g, M, D = _gen(seed), case["rows"], case["hidden"]
    F = D * case["ratio"]
    t = {"n": _randn(g, M, D, dtype=torch.float16), "x": _randn(g, M, D), "gamma": 1 + _randn(g, D, std=0.1),
         "b1": _randn(g, F, std=0.02), "b2": _randn(g, D, std=0.02)}
    for nm, (N, K) in (("w1", (F, D)), ("w2", (D, F))):
        w = _randn(g, N, K, std=0.02)
        if case["int8"]:
            t[nm], t["s" + nm] = _int8_rows(w)
        else:
            t[nm], t["s" + nm] = w.to(torch.bfloat16), None
    return t


def _adaptor_inputs(case, seed):
    g, M, K, D = _gen(seed), case["rows"], case["K"], case["hidden"]
    bf = torch.bfloat16
    return {"t": _randn(g, M, K, dtype=bf), "w1": _randn(g, D, K, dtype=bf, std=0.02), "b1": _randn(g, D, std=0.02),
            "w2": _randn(g, D, D, dtype=bf, std=0.02), "b2": _randn(g, D, std=0.02)}


def _model_dims(case):
    return case["batch"], case["horizon"] + 3, 64 * case["heads"], case["lang"], case["img"]


def _block_weights(case, seed):
    """Parameters of the blocks and the condition's position embeddings, by
    checkpoint name, in the type the model holds them in."""
    _, _, D, L, I = _model_dims(case)
    g, p = _gen(seed + 101), {}
    p["lang_cond_pos_embed"] = _randn(g, 1, L, D, std=0.02)
    p["img_cond_pos_embed"] = _randn(g, 1, I, D, std=0.02)
    for i in range(case["layers"]):
        b = "blocks.%d." % i
        for nm in ("norm1", "norm2", "norm3"):
            p[b + nm + ".weight"] = 1 + _randn(g, D, std=0.1)
        for nm in ("attn.q_norm", "attn.k_norm", "cross_attn.q_norm", "cross_attn.k_norm"):
            p[b + nm + ".weight"] = 1 + _randn(g, 64, std=0.1)
        for nm, N in (("attn.qkv", 3 * D), ("attn.proj", D), ("cross_attn.q", D), ("cross_attn.kv", 2 * D),
                      ("cross_attn.proj", D), ("ffn.fc1", D), ("ffn.fc2", D)):
            p[b + nm + ".weight"] = _randn(g, N, D, dtype=torch.bfloat16, std=0.02)
            p[b + nm + ".bias"] = _randn(g, N, std=0.02)
    return p


def _condition(case, seed):
    """Adaptor outputs for a condition set directly, and the residual rows."""
    B, S, D, L, I = _model_dims(case)
    g, bf = _gen(seed + 202), torch.bfloat16
    hi = case["lang_rows"]
    valid = torch.randint(max(1, hi // 2), hi + 1, (B,), device=DEV, generator=g, dtype=torch.int32)
    return {"lang": _randn(g, B, L, D, dtype=bf), "valid": valid, "img": _randn(g, B, I, D, dtype=bf),
            "state": _randn(g, B, D, dtype=bf), "x": _randn(g, B, S, D)}


def _write_params(model, p):
    at = {nm: i for i, (nm, _, _) in enumerate(model.params())}
    for nm, t in p.items():
        t = t.view(torch.int16) if t.dtype == torch.bfloat16 else t
        model.param_write(at[nm], t.cpu().numpy().reshape(-1))
    model.params_changed()


def _prepare_model(case, seed):
    cfg = rdt.default_config(hidden=64 * case["heads"], heads=case["heads"], layers=case["layers"],
                             horizon=case["horizon"], lang_max=case["lang"], img_len=case["img"],
                             batch=case["batch"], int8_weights=case["int8"], num_steps=case["steps"])
    m = rdt.RdtModel(cfg)
    m.init_random(1000 + seed, 0.02)
    if case["batch"] == 1 and case["lang_rows"] != case["lang"]:
        m.set_lang_rows(case["lang_rows"])
    if case["op"] == "blocks":
        if not case["int8"]:
            _write_params(m, _block_weights(case, seed))
        c = _condition(case, seed)
        m.set_condition(c["lang"], c["valid"], c["img"], c["state"])
        torch.cuda.synchronize()
        return {"model": m, "x": c["x"]}
    B, g, bf = case["batch"], _gen(seed + 303), torch.bfloat16
    st = {"model": m, "frame": 1,
          "lang": _randn(g, B, case["lang"], cfg.lang_token_dim, dtype=bf),
          "valid": torch.randint(max(1, case["lang_rows"] // 2), case["lang_rows"] + 1, (B,), device=DEV, generator=g,
                                 dtype=torch.int32),
          "img": _randn(g, B, case["img"], cfg.img_token_dim, dtype=bf),
          "state": _randn(g, B, cfg.state_dim, dtype=bf),
          "noise": _randn(g, B, case["horizon"], cfg.action_dim), "noise_seed": 5 + seed}
    torch.cuda.synchronize()
    if case["op"] == "sample":
        m.encode_condition(st["lang"], st["valid"], st["img"], st["state"])
        m.sample(st["noise"].clone())   # a program warms its loop up before it serves
    else:
        m.infer(0, st["lang"], st["valid"], st["img"], st["state"], st["noise_seed"])
    torch.cuda.synchronize()
    return st


def _plan_gemm(M, w, a_dtype, w16):
    """The one-time set-up of a projection's shape."""
    d = abi.GemmDesc()
    d.M, d.N, d.K = M, w.shape[0], w.shape[1]
    d.lda = d.ldw = w.shape[1]
    d.a_dtype, d.w_dtype = a_dtype, abi.SF_I8 if w.dtype == torch.int8 else abi.SF_BF16
    d.w16_f16 = 1 if w16 else 0
    abi.check(abi.lib().sf_gemm_prepare(d), "sf_gemm_prepare")


def prepare(case, seed):
    seed = int(seed) % (1 << 30)
    if case["kind"] == "attention":
        q, k, v, valid = _attention_inputs(case, seed)
        return {"case": case, "q": q, "k": k, "v": v, "valid": valid}
    if case["kind"] == "mlp":
        t = _mlp_inputs(case, seed)
        if case["int8"]:
            t["c1"] = t["c2"] = None
        else:
            t["c1"], t["c2"] = kernels.weights_to_f16([t["w1"], t["w2"]])
        for nm in ("w1", "w2"):
            _plan_gemm(case["rows"], t[nm], abi.SF_F16, not case["int8"])
        return {"case": case, **t}
    if case["kind"] == "adaptor":
        t = _adaptor_inputs(case, seed)
        for nm in ("w1", "w2"):
            _plan_gemm(case["rows"], t[nm], abi.SF_BF16, False)
        return {"case": case, **t}
    return {"case": case, **_prepare_model(case, seed)}


def run(s):
    c = s["case"]
    if c["kind"] == "attention":
        return attention(s["q"], s["k"], s["v"], valid_len=s["valid"])
    if c["kind"] == "mlp":
        # the residual stream is the pass's own: the FFN adds into it
        x = s["x"].clone()
        h = kernels.gemm(s["n"], s["w1"], s["b1"], act=abi.SF_ACT_GELU_TANH, out_dtype=torch.float16,
                         w_scale=s["sw1"], w16=s["c1"])
        n = kernels.gemm_add_norm(h, s["w2"], s["b2"], x, s["gamma"], w_scale=s["sw2"], norm_dtype=torch.float16,
                                  round_product=True, w16=s["c2"])
        return {"x": x, "n": n}
    if c["kind"] == "adaptor":
        h = kernels.gemm(s["t"], s["w1"], s["b1"], act=abi.SF_ACT_GELU_TANH)
        return kernels.gemm(h, s["w2"], s["b2"])
    m = s["model"]
    if c["op"] == "blocks":
        return m.run_blocks(s["x"].clone())
    if c["op"] == "sample":
        return m.sample(s["noise"].clone())
    s["frame"] += 1   # a new camera frame: the condition is encoded
    return m.infer(s["frame"], s["lang"], s["valid"], s["img"], s["state"], s["noise_seed"])[0]


# --- what a pass cannot do without ----------------------------------------


def _block_work(case):
    """(bytes, flops) of one language and one image block."""
    B, S, D, L, I = _model_dims(case)
    M, wb = B * S, 1 if case["int8"] else 2
    out = []
    for keys in (0.75 * case["lang_rows"], I):   # valid lengths are uniform in [rows / 2, rows]
        by = 8 * D * D * wb + 2 * B * keys * D * 2 + 2 * M * D * 4
        fl = 2 * M * 8 * D * D + 4 * B * S * S * D + 4 * B * S * keys * D
        out.append((by, fl))
    return out


def work(case):
    if case["kind"] == "attention":
        B, H, Sq, Sk, e = case["B"], case["H"], case["Sq"], case["Sk"], _BYTES[case["dtype"]]
        keys = (min(32, Sk) + Sk) / 2 if case["ragged"] else Sk
        return {"bytes": 2 * B * H * 64 * (Sq + keys) * e, "flops": 4 * B * H * Sq * keys * 64}
    if case["kind"] == "mlp":
        M, D, F = case["rows"], case["hidden"], case["hidden"] * case["ratio"]
        return {"bytes": 2 * D * F * (1 if case["int8"] else 2) + M * D * (2 + 8 + 2), "flops": 4 * M * D * F}
    if case["kind"] == "adaptor":
        M, K, D = case["rows"], case["K"], case["hidden"]
        return {"bytes": 2 * (M * K + D * K + D * D + M * D), "flops": 2 * M * D * (K + D)}
    B, S, D, L, I = _model_dims(case)
    blocks = _block_work(case)
    by = sum(blocks[i % 2][0] for i in range(case["layers"]))
    fl = sum(blocks[i % 2][1] for i in range(case["layers"]))
    if case["op"] == "blocks":
        return {"bytes": by, "flops": fl}
    by, fl = by * case["steps"], fl * case["steps"]
    if case["op"] == "infer":   # the adaptors and every block's K/V projection
        lr, half = B * case["lang_rows"], case["layers"] / 2
        fl += 2 * lr * D * (4096 + D) + 2 * B * I * D * (1152 + D) + half * 2 * (lr + B * I) * 2 * D * D
        by += 2 * (lr * 4096 + B * I * 1152) + 2 * D * (4096 + 1152 + 2 * D)
        by += case["layers"] * 2 * D * D * (1 if case["int8"] else 2) + half * 2 * 2 * (lr + B * I) * D
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """About four times what two correct implementations at the same
    precision (another summation order) show on these inputs."""
    if case["kind"] == "attention":
        return {"bf16": {"rel": 6e-3}, "fp16": {"rel": 1.1e-3}, "fp32": {"rel": 4e-6}}[case["dtype"]]
    if case["kind"] == "mlp":
        return {"rel": 1e-3}
    if case["kind"] == "adaptor":
        return {"rel": 8e-3}
    if case["op"] == "blocks":
        return {"rel": 4e-3}
    return {"rel": 1e-2}


# --- the same in 64 bits ---------------------------------------------------


def _attend(q, k, v, valid=None):
    """softmax(q k^T / 8) v per (batch, head) in float64; [B, H, S, 64]."""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b in range(q.shape[0]):
        n = k.shape[2] if valid is None else int(valid[b])
        kb, vb = k[b, :, :n].double(), v[b, :, :n].double()
        p = torch.softmax(torch.matmul(q[b].double(), kb.transpose(1, 2).contiguous()) / 8.0, -1)
        out[b] = torch.matmul(p, vb)
    return out


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _rms(x, gamma, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * gamma.double()


def _exact_blocks(case, seed):
    B, S, D, L, I = _model_dims(case)
    p, c, H = _block_weights(case, seed), _condition(case, seed), case["heads"]
    lin = lambda a, nm: torch.matmul(a, p[nm + ".weight"].double().t()) + p[nm + ".bias"].double()  # noqa: E731
    heads = lambda a: a.reshape(a.shape[0], a.shape[1], H, 64).transpose(1, 2)  # noqa: E731
    rows = lambda a: a.transpose(1, 2).reshape(B, S, D)  # noqa: E731
    conds = [c["lang"].double() + p["lang_cond_pos_embed"].double(), c["img"].double() + p["img_cond_pos_embed"].double()]
    x = c["x"].double()
    for i in range(case["layers"]):
        b = "blocks.%d." % i
        q, k, v = lin(_rms(x, p[b + "norm1.weight"]), b + "attn.qkv").split(D, -1)
        q, k = _rms(heads(q), p[b + "attn.q_norm.weight"]), _rms(heads(k), p[b + "attn.k_norm.weight"])
        x = x + lin(rows(_attend(q, k, heads(v))), b + "attn.proj")
        q = _rms(heads(lin(_rms(x, p[b + "norm2.weight"]), b + "cross_attn.q")), p[b + "cross_attn.q_norm.weight"])
        a = torch.empty(B, S, D, dtype=torch.float64, device=DEV)
        for j in range(B):   # one batch element's keys at a time
            k, v = lin(conds[i % 2][j:j + 1], b + "cross_attn.kv").split(D, -1)
            k = _rms(heads(k), p[b + "cross_attn.k_norm.weight"])
            o = _attend(q[j:j + 1], k, heads(v), c["valid"][j:j + 1] if i % 2 == 0 else None)
            a[j] = o.transpose(1, 2).reshape(S, D)
        x = x + lin(a, b + "cross_attn.proj")
        x = x + lin(_gelu(lin(_rms(x, p[b + "norm3.weight"]), b + "ffn.fc1")), b + "ffn.fc2")
    return x


def exact(case, seed):
    seed = int(seed) % (1 << 30)
    if case["kind"] == "attention":
        return _attend(*_attention_inputs(case, seed))
    if case["kind"] == "mlp":
        t = _mlp_inputs(case, seed)
        w = [t[nm].double() * (t["s" + nm].double()[:, None] if case["int8"] else 1) for nm in ("w1", "w2")]
        h = _gelu(torch.matmul(t["n"].double(), w[0].t()) + t["b1"].double())
        x = t["x"].double() + torch.matmul(h, w[1].t()) + t["b2"].double()
        return {"x": x, "n": _rms(x, t["gamma"])}
    if case["kind"] == "adaptor":
        t = {k: v.double() for k, v in _adaptor_inputs(case, seed).items()}
        return torch.matmul(_gelu(torch.matmul(t["t"], t["w1"].t()) + t["b1"]), t["w2"].t()) + t["b2"]
    if case["op"] == "blocks" and not case["int8"]:
        return _exact_blocks(case, seed)
    return None   # whole loops and in-library int8 weights: no value without the model's own arithmetic
