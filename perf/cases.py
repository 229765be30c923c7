"""The work that a user of this library has it do, as cases that can be timed.

The library runs one job: a search over edits of a quantised language model.
Its trial edits the output projections of every layer, runs the batched
prompt forward for residuals and last-token logits, and scores the logits
against the unedited model's; between trials it decodes answers token by
token. The cases are the parts of that job, from one matrix product on one
token to a whole 24-layer forward:

  product  one registered weight times n activation rows, with a bias in
           half of the drawn ones (every projection is one of these);
  head     the lm_head product, its log-softmax, and the KL divergence from
           a baseline (the scorer of a trial);
  prefill  the batched prompt forward with the residual window captured at
           every layer entry and the last-token logits (dense, routed
           experts, latent attention);
  decode   one token per prompt through the persistent KV cache (generation);
  trial    the edit of every output projection, then the forward.

Shapes are those of the benchmark's configurations (`SHAPES`). Where a case
is about a layer, the model has one or a few layers and a vocabulary of 8192,
so that the head, which has a case of its own, stays small.

Inputs are made from the seed: weights N(0, 0.02) quantised to the case's
format, norms around 1, random tokens. `exact` computes the same numbers in
64-bit torch from the decoded weights.
"""
import ctypes
import math

import numpy as np
import torch

from ditch_amd import abi, synth
from ditch_amd.hip import Device, Model
from ditch_amd.spec import ModelSpec
from ditch_amd.weights import HostWeight

# The decoder layers of the benchmark's configurations: a small dense model
# with q/k/v biases and tied embeddings, a dense 4096-wide one, one of 128
# routed experts (softmax router, q/k head norm), and one with latent
# attention, a shared expert and group-limited sigmoid routing (16 experts of
# its 256, top 4 of its top 8: a layer that is quick to make).
SHAPES = {
    "d896": dict(hidden=896, heads=14, kv_heads=2, head_dim=64, inter=4864, rope_theta=1e6, qkv_bias=1,
                 tie_embeddings=1),
    "d4096": dict(hidden=4096, heads=32, kv_heads=8, head_dim=128, inter=14336, rope_theta=5e5),
    "moe2048": dict(hidden=2048, heads=32, kv_heads=4, head_dim=128, inter=8192, rope_theta=1e6, qk_norm=1,
                    n_experts=128, top_k=8, moe_inter=768, norm_topk_prob=1, scoring=abi.SCORING_SOFTMAX),
    "mla7168": dict(hidden=7168, heads=128, kv_heads=128, head_dim=192, v_head_dim=128, inter=18432,
                    rope_theta=1e4, rope_style=abi.ROPE_GPTJ, mla=1, q_lora_rank=1536, kv_lora_rank=512,
                    qk_nope_dim=128, qk_rope_dim=64, n_experts=16, top_k=4, moe_inter=2048, shared_inter=2048,
                    norm_topk_prob=1, scoring=abi.SCORING_SIGMOID, group_limited=1, n_group=4, topk_group=2,
                    routed_scaling=2.5),
}
FORMATS = ("f32", "f16", "bf16", "q8_0", "fp8", "mxfp4", "int4")
# stored bytes of a weight: codes and their share of the scales
WEIGHT_BYTES = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q8_0": 34 / 32, "fp8": 1 + 4 / 16384, "mxfp4": 17 / 32,
                "int4": 0.5 + 2.5 / 128}
WINDOW = 4  # last positions of a prompt whose residuals a trial captures
DISTINCT = 2  # different random layers of a deeper model; the others repeat them


# ---------------------------------------------------------------------------
# the cases

def listed():
    return [
        # decode of one prompt: a projection on a single token
        dict(name="product_q8_0_1", kind="product", fmt="q8_0", n=1, rows=14336, cols=4096, bias=False),
        # a few short prompts, or a decode batch over 16, on an attention projection
        dict(name="product_int4_24", kind="product", fmt="int4", n=24, rows=4096, cols=2048, bias=False),
        # one long prompt on a down projection, its length of no particular multiple
        dict(name="product_fp8_300", kind="product", fmt="fp8", n=300, rows=4096, cols=14336, bias=False),
        # scoring of 64 prompts' last tokens over a full vocabulary
        dict(name="head_bf16_64", kind="head", fmt="bf16", n=64, rows=128256, cols=4096),
        # the whole small model in f32 on one batch of prompts
        dict(name="prefill_f32_16x64", kind="prefill", shape="d896", fmt="f32", layers=24, vocab=151936, prompts=16,
             tokens=64, ragged=False),
        # a layer of the headline workload: 64 prompts of 128 tokens
        dict(name="prefill_mxfp4_64x128", kind="prefill", shape="d4096", fmt="mxfp4", layers=1, vocab=8192,
             prompts=64, tokens=128, ragged=False),
        # real prompts: few, of different lengths
        dict(name="prefill_fp8_12x90", kind="prefill", shape="d4096", fmt="fp8", layers=2, vocab=8192, prompts=12,
             tokens=90, ragged=True),
        # a routed layer on a full batch
        dict(name="prefill_moe_int4_32x128", kind="prefill", shape="moe2048", fmt="int4", layers=1, vocab=8192,
             prompts=32, tokens=128, ragged=False),
        # a latent-attention layer with routed and shared experts on longer prompts
        dict(name="prefill_mla_fp8_16x256", kind="prefill", shape="mla7168", fmt="fp8", layers=1, vocab=8192,
             prompts=16, tokens=256, ragged=False),
        # generation with the whole small model: a token for each of 16 prompts
        dict(name="decode_bf16_16", kind="decode", shape="d896", fmt="bf16", layers=24, vocab=151936, prompts=16,
             tokens=96, ragged=True),
        # generation for one prompt with a long context, 4-bit weights
        dict(name="decode_mxfp4_1", kind="decode", shape="d4096", fmt="mxfp4", layers=4, vocab=8192, prompts=1,
             tokens=500, ragged=False),
        # a search trial on the small model: the default edit, then the prompts
        dict(name="trial_full_bf16_16x32", kind="trial", shape="d896", fmt="bf16", layers=2, vocab=8192, prompts=16,
             tokens=32, ragged=True, mode="full"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["product", "product", "head", "prefill", "prefill", "decode", "decode", "trial"])
    if kind == "product":
        fmt = rng.choice(FORMATS)
        rows, cols = _log(rng, 256, 16384), _log(rng, 2, 112) * 128
        # up to the work of the large listed prompts
        n = _log(rng, 1, 2048)
        while n * rows * cols > 3e11:
            n = max(1, n // 2)
        return dict(kind=kind, fmt=fmt, n=n, rows=rows, cols=cols, bias=rng.random() < 0.5)
    if kind == "head":
        return dict(kind=kind, fmt=rng.choice(["bf16", "f16", "q8_0", "fp8"]), n=_log(rng, 1, 64),
                    rows=_log(rng, 8192, 128256), cols=rng.choice([896, 2048, 4096]))
    if kind == "prefill":
        shape = rng.choice(["d896", "d4096", "d4096", "moe2048", "mla7168"])
        fmt = rng.choice({"d896": ["f32", "bf16", "q8_0"], "d4096": ["mxfp4", "fp8", "int4", "q8_0", "bf16"],
                          "moe2048": ["int4", "fp8", "mxfp4"], "mla7168": ["fp8"]}[shape])
        rows = _log(rng, 32, {"d896": 4096, "d4096": 4096, "moe2048": 4096, "mla7168": 2048}[shape])
        tokens = min(rows, _log(rng, 16, 512))
        return dict(kind=kind, shape=shape, fmt=fmt, layers=rng.choice([1, 2]) if shape != "mla7168" else 1,
                    vocab=8192, prompts=max(1, rows // tokens), tokens=tokens, ragged=rng.random() < 0.6)
    if kind == "decode":
        shape = rng.choice(["d896", "d4096", "d4096", "moe2048"])
        fmt = rng.choice({"d896": ["f32", "bf16", "q8_0"], "d4096": ["mxfp4", "fp8", "int4", "q8_0", "bf16"],
                          "moe2048": ["int4", "fp8", "mxfp4"]}[shape])
        return dict(kind=kind, shape=shape, fmt=fmt, layers=rng.choice([2, 3, 4] if shape != "moe2048" else [1, 2]),
                    vocab=8192, prompts=_log(rng, 1, 48), tokens=_log(rng, 16, 900), ragged=rng.random() < 0.7)
    mode = rng.choice(["none", "pre", "full"])
    shape = rng.choice(["d896", "d4096"] + (["moe2048"] if mode == "none" else []))
    fmt = rng.choice({"d896": ["f32", "bf16", "q8_0"], "d4096": ["mxfp4", "fp8", "int4", "bf16"],
                      "moe2048": ["int4"]}[shape])
    return dict(kind=kind, shape=shape, fmt=fmt, layers=rng.choice([1, 2]) if shape != "d4096" else 1, vocab=8192,
                prompts=_log(rng, 2, 32), tokens=_log(rng, 8, 100), ragged=True, mode=mode)


# ---------------------------------------------------------------------------
# inputs

_dev = None


def _device():
    global _dev
    if _dev is None:
        _dev = Device(0)
    return _dev


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _weight(fmt, rows, cols, gen):
    w = torch.randn(rows, cols, generator=gen, device="cuda") * 0.02
    if fmt == "f16":
        return HostWeight.f16(w.half().cpu().numpy())
    return synth.QUANTIZERS[fmt](w)


def _vec(n, gen, around):
    return (around + torch.randn(n, generator=gen, device="cuda") * 0.02).cpu().numpy()


def _lengths(case):
    """Prompt lengths: all `tokens`, or between a third of it and all of it."""
    n, lo = case["tokens"], max(1, case["tokens"] // 3)
    if not case["ragged"]:
        return [n] * case["prompts"]
    return [n] + [lo + b * 7919 % (n - lo + 1) for b in range(1, case["prompts"])]


def _spec(case, gen):
    c = dict(SHAPES[case["shape"]], layers=case["layers"], vocab=case["vocab"], rms_eps=1e-6, rope_len=1024)
    routed = "n_experts" in c
    spec = ModelSpec(**c, moe_layers=[1 if routed else 0] * case["layers"])
    fmt, h, nh, hd = case["fmt"], c["hidden"], c["heads"], c["head_dim"]
    kvd, od = c["kv_heads"] * hd, nh * c.get("v_head_dim", hd)
    plain = fmt if fmt in ("f32", "f16") else "bf16"
    spec.set("EMBED", _weight(plain, c["vocab"], h, gen))
    if not c.get("tie_embeddings"):
        spec.set("LM_HEAD", _weight(plain, c["vocab"], h, gen))
    spec.set("FINAL_NORM", _vec(h, gen, 1))
    pool = []
    for _ in range(min(DISTINCT, case["layers"])):
        lw = {("ATTN_NORM", -1): _vec(h, gen, 1), ("FFN_NORM", -1): _vec(h, gen, 1)}
        mats = []
        if c.get("mla"):
            ql, kl, nope, rd = c["q_lora_rank"], c["kv_lora_rank"], c["qk_nope_dim"], c["qk_rope_dim"]
            mats += [("MLA_Q_A", ql, h), ("MLA_Q_B", nh * hd, ql), ("MLA_KV_A", kl + rd, h),
                     ("MLA_KV_B", nh * (nope + c["v_head_dim"]), kl)]
            lw[("MLA_Q_A_NORM", -1)], lw[("MLA_KV_A_NORM", -1)] = _vec(ql, gen, 1), _vec(kl, gen, 1)
        else:
            mats += [("Q", nh * hd, h), ("K", kvd, h), ("V", kvd, h)]
            for name, n, on in (("Q_BIAS", nh * hd, "qkv_bias"), ("K_BIAS", kvd, "qkv_bias"),
                                ("V_BIAS", kvd, "qkv_bias"), ("Q_NORM", hd, "qk_norm"), ("K_NORM", hd, "qk_norm")):
                if c.get(on):
                    lw[(name, -1)] = _vec(n, gen, 1 if on == "qk_norm" else 0)
        mats.append(("O", h, od))
        if routed:
            lw[("ROUTER", -1)] = _weight("bf16", c["n_experts"], h, gen)
            if c.get("group_limited"):
                lw[("ROUTER_CORRECTION", -1)] = _vec(c["n_experts"], gen, 0)
            for e in range(c["n_experts"]):
                lw[("EXPERT_GATE", e)] = _weight(fmt, c["moe_inter"], h, gen)
                lw[("EXPERT_UP", e)] = _weight(fmt, c["moe_inter"], h, gen)
                lw[("EXPERT_DOWN", e)] = _weight(fmt, h, c["moe_inter"], gen)
            if c.get("shared_inter"):
                mats += [("SHARED_GATE", c["shared_inter"], h), ("SHARED_UP", c["shared_inter"], h),
                         ("SHARED_DOWN", h, c["shared_inter"])]
        else:
            mats += [("GATE", c["inter"], h), ("UP", c["inter"], h), ("DOWN", h, c["inter"])]
        for name, r, k in mats:
            lw[(name, -1)] = _weight(fmt, r, k, gen)
        pool.append(lw)
    for li in range(case["layers"]):
        for (name, e), w in pool[li % len(pool)].items():
            spec.set(name, w, li, e)
    return spec


def _tokens(case, lens, gen, extra):
    """The prompts' token ids, each with `extra` more than its length."""
    n = sum(lens) + extra * len(lens)
    return torch.randint(0, case["vocab"], (n,), generator=gen, device="cuda", dtype=torch.int32)


def _edit(case, gen):
    """One unit direction a layer and the matrices that a trial edits with it."""
    h, targets = SHAPES[case["shape"]]["hidden"], []
    for li in range(case["layers"]):
        v = torch.randn(1, h, generator=gen, device="cuda")
        v = (v / v.norm()).cpu().numpy()
        targets.append((li, abi.SLOT["O"], -1, v, 1.0))
        if "n_experts" in SHAPES[case["shape"]]:
            targets += [(li, abi.SLOT["EXPERT_DOWN"], e, v, 0.8) for e in range(SHAPES[case["shape"]]["n_experts"])]
        else:
            targets.append((li, abi.SLOT["DOWN"], -1, v, 0.8))
    return targets


class _State:
    """What a user's program holds; the library's handles go with it."""

    def __init__(self, case):
        self.case, self.model, self.cache, self.tensor = case, None, None, None

    def __del__(self):
        try:
            torch.cuda.synchronize()
            if self.cache:
                self.model.kv_cache_free(self.cache)
            if self.model:
                self.model.free()
            if self.tensor:
                self.tensor.free()
        except Exception:
            pass


def _i64(values):
    return torch.tensor(values, dtype=torch.int64, device="cuda")


def _f32(*shape):
    return torch.zeros(shape, dtype=torch.float32, device="cuda")


def _product_inputs(case, seed):
    gen = _gen(seed)
    w = _weight(case["fmt"], case["rows"], case["cols"], gen)
    x = torch.randn(case["n"], case["cols"], generator=gen, device="cuda")
    extra = None
    if case["kind"] == "head":
        # the baseline's log-probabilities: those of an unedited model's activations
        extra = x + 0.3 * torch.randn(x.shape, generator=gen, device="cuda")
    elif case["bias"]:
        extra = 0.02 * torch.randn(case["rows"], generator=gen, device="cuda")
    return w, x, extra


def _prompt_inputs(case, seed):
    gen = _gen(seed)
    spec = _spec(case, gen)
    lens = _lengths(case)
    toks = _tokens(case, lens, gen, 1 if case["kind"] == "decode" else 0)
    targets = _edit(case, gen) if case["kind"] == "trial" else None
    return spec, lens, toks, targets


def prepare(case, seed):
    s = _State(case)
    dev = s.dev = _device()
    if case["kind"] in ("product", "head"):
        w, s.x, extra = _product_inputs(case, seed)
        s.tensor = dev.upload(w)
        s.out = _f32(case["n"], case["rows"])
        s.bias = extra if case["kind"] == "product" else None
        if case["kind"] == "head":
            s.lp, s.base, s.kl = _f32(case["n"], case["rows"]), _f32(case["n"], case["rows"]), \
                torch.zeros(case["n"], dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            s.tensor.matmul_device(s.out.data_ptr(), extra.data_ptr(), case["n"])
            dev.logSoftmaxRows_device(s.base.data_ptr(), s.out.data_ptr(), case["n"], case["rows"])
        torch.cuda.synchronize()
        return s
    spec, lens, toks, targets = _prompt_inputs(case, seed)
    s.model = Model(dev, spec)
    nb = len(lens)
    if case["kind"] == "decode":
        # the prompts in the cache, then the row of each prompt's next token
        s.cache = s.model.kv_cache(nb, max(lens) + 1)
        pre, nxt, rows, at = [], [], [], 0
        for b, n in enumerate(lens):
            pre += range(at, at + n)
            nxt.append(at + n)
            rows += [(b, p) for p in range(n)]
            at += n + 1
        p_tok, p_rows = toks[_i64(pre)], torch.tensor(rows, dtype=torch.int32, device="cuda")
        s.tok = toks[_i64(nxt)]
        s.rows = torch.tensor([(b, n) for b, n in enumerate(lens)], dtype=torch.int32, device="cuda")
        s.last, s.logits = _i64(range(nb)), _f32(nb, case["vocab"])
        torch.cuda.synchronize()
        _cached(s, p_tok, p_rows, len(pre), s.last, 0, s.logits)
        torch.cuda.synchronize()
        return s
    s.n, s.nb, s.max_len = sum(lens), nb, max(lens)
    rows, cap, last = [], [], []
    for b, n in enumerate(lens):
        rows += [(b, p) for p in range(n)]
        last.append(len(rows) - 1)
        cap += range(len(rows) - min(n, WINDOW), len(rows))
    s.tok, s.rows = toks, torch.tensor(rows, dtype=torch.int32, device="cuda")
    s.cap, s.last = _i64(cap), _i64(last)
    s.res = _f32(case["layers"] + 1, len(cap), spec.config["hidden"])
    s.logits = _f32(nb, case["vocab"])
    if targets:
        s.targets = Model.edit_targets(targets, 1) if case["mode"] == "none" else targets
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# one pass

def _cached(s, tok, rows, n, last, n_logit, logits):
    m = s.model
    m.dev.check(m.dev.lib.ditch_hip_forward_cached(
        m.h, s.cache, ctypes.c_void_p(tok.data_ptr()), ctypes.c_void_p(rows.data_ptr()), n,
        ctypes.c_void_p(last.data_ptr()), n_logit, ctypes.c_void_p(logits.data_ptr()), logits.numel() * 4))


def run(s):
    case, dev = s.case, s.dev
    if case["kind"] in ("product", "head"):
        n, rows = case["n"], case["rows"]
        s.tensor.matmul_device(s.out.data_ptr(), s.x.data_ptr(), n, None if s.bias is None else s.bias.data_ptr())
        if case["kind"] == "product":
            return s.out
        dev.logSoftmaxRows_device(s.lp.data_ptr(), s.out.data_ptr(), n, rows)
        dev.klRows_device(s.kl.data_ptr(), s.base.data_ptr(), s.out.data_ptr(), n, rows)
        return {"logits": s.out, "logprobs": s.lp, "kl": s.kl}
    if case["kind"] == "decode":
        _cached(s, s.tok, s.rows, len(s.tok), s.last, len(s.last), s.logits)
        return s.logits
    m = s.model
    if case["kind"] == "trial":
        m.reset_deltas()
        if case["mode"] == "none":
            m.edit_batch(s.targets)
        else:
            for layer, slot, expert, v, weight in s.targets:
                m.edit_ex(layer, slot, expert, v, weight, mode=case["mode"])
    m.forward_device(s.tok.data_ptr(), s.rows.data_ptr(), s.n, s.nb, s.max_len, s.cap.data_ptr(), len(s.cap),
                     s.res.data_ptr(), s.last.data_ptr(), len(s.last), s.logits.data_ptr())
    return {"residuals": s.res, "logits": s.logits}


# ---------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    if case["kind"] in ("product", "head"):
        n, rows, cols = case["n"], case["rows"], case["cols"]
        nbytes = rows * cols * WEIGHT_BYTES[case["fmt"]] + n * cols * 4 + n * rows * 4
        if case["kind"] == "head":  # the baseline in, the log-probabilities out
            nbytes += 2 * n * rows * 4
        return {"bytes": nbytes, "flops": 2.0 * n * rows * cols}
    c, lens, L = SHAPES[case["shape"]], _lengths(case), case["layers"]
    h, nh, hd = c["hidden"], c["heads"], c["head_dim"]
    vd, kvd = c.get("v_head_dim", hd), c["kv_heads"] * hd
    decode = case["kind"] == "decode"
    n = len(lens) if decode else sum(lens)
    if c.get("mla"):
        attn = c["q_lora_rank"] * (h + nh * hd) + (c["kv_lora_rank"] + c["qk_rope_dim"]) * h + \
            nh * (c["qk_nope_dim"] + vd) * c["kv_lora_rank"] + h * nh * vd
    else:
        attn = h * (nh * hd + 2 * kvd) + h * nh * hd
    if "n_experts" in c:
        e, sh = 3 * h * c["moe_inter"], 3 * h * c.get("shared_inter", 0)
        ffn, ffn_read = c["top_k"] * e + sh, min(c["n_experts"], n * c["top_k"]) * e + sh
    else:
        ffn = ffn_read = 3 * h * c["inter"]
    keys = sum(x + 1 for x in lens) if decode else sum(x * (x + 1) // 2 for x in lens)
    flops = L * (2.0 * n * (attn + ffn) + 2.0 * keys * nh * (hd + vd)) + 2.0 * len(lens) * h * case["vocab"]
    wb = WEIGHT_BYTES[case["fmt"]]
    plain = 4.0 if case["fmt"] == "f32" else 2.0
    nbytes = L * wb * (attn + ffn_read) + plain * h * case["vocab"] + plain * n * h + len(lens) * case["vocab"] * 4
    if decode:
        nbytes += L * keys * 2 * kvd * 4
    else:
        nbytes += (L + 1) * sum(min(x, WINDOW) for x in lens) * h * 4
    if case["kind"] == "trial":
        # one reading of each edited matrix (two and a product each way for the row-normalised modes)
        edited = L * (h * nh * vd + h * (c["n_experts"] * c["moe_inter"] if "n_experts" in c else c["inter"]))
        nbytes += edited * wb * {"none": 1, "pre": 2, "full": 3}[case["mode"]]
        flops += 2.0 * edited
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times the error against `exact`: a product's activations
    # enter as two bf16 terms (2.5e-6 over the product), the KL divergence is
    # a difference of the logits' distributions (8e-6), a forward's residuals
    # and logits are 1e-5 to 2.2e-5 off
    return {"rel": {"product": 1e-5, "head": 4e-5}.get(case["kind"], 1e-4)}


# ---------------------------------------------------------------------------
# the same numbers in 64 bits

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _bf16(w):
    return w.to(torch.bfloat16).double()


def _dense(w):
    """The values of a host weight, from its stored bytes."""
    data, scale, zero, _ = (None if a is None else torch.from_numpy(a).cuda() for a in w.arrays)
    rows, cols = w.rows, w.cols
    if w.dtype == abi.F32:
        return data.reshape(rows, cols).double()
    if w.dtype == abi.F16:
        return data.view(torch.float16).reshape(rows, cols).double()
    if w.dtype == abi.BF16:
        return data.view(torch.bfloat16).reshape(rows, cols).double()
    if w.dtype == abi.Q8_0:
        b = data.reshape(rows, cols // 32, 34)
        d = b[..., :2].contiguous().view(torch.float16).double()
        return (b[..., 2:].contiguous().view(torch.int8).double() * d).reshape(rows, cols)
    if w.dtype == abi.FP8:
        s = scale.repeat_interleave(128, 0)[:rows].repeat_interleave(128, 1)[:, :cols]
        return _bf16(data.view(torch.float8_e4m3fn).float() * s)
    if w.dtype == abi.MXFP4:
        table = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device="cuda")
        codes = torch.stack([data & 15, data >> 4], 2).reshape(rows, cols).long()
        s = torch.exp2(scale.double() - 127).repeat_interleave(32, 1)
        return table[codes] * s
    shifts = 4 * torch.arange(8, device="cuda", dtype=torch.int32)
    q = ((data.reshape(rows, cols // 8, 1) >> shifts) & 15).reshape(rows, cols)
    z = ((zero.reshape(-1, 1, zero.shape[-1]) >> shifts.reshape(1, 8, 1)) & 15).reshape(-1, zero.shape[-1])[:rows]
    group = cols // z.shape[1]
    s = scale.view(torch.float16).reshape(rows, -1).float()
    return _bf16((q - z.repeat_interleave(group, 1)).float() * s.repeat_interleave(group, 1))


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w


def _delta(w, v, weight, mode):
    """The edited matrix for one direction over its rows; `full` is the best
    approximation of the lora rank (3) to the row-normalised edit."""
    if mode == "none":
        return w - weight * v[:, None] * (v @ w)[None]
    n = w.norm(dim=1)
    a = (v / n) @ w
    if mode == "pre":
        return w - weight * (n * v)[:, None] * a[None]
    new = w / n[:, None] - weight * v[:, None] * a[None]
    d = new * (n / new.norm(dim=1))[:, None] - w
    q = torch.linalg.qr(d @ torch.randn(d.shape[1], 48, generator=_gen(1), device="cuda", dtype=torch.float64))[0]
    for _ in range(60):
        q = torch.linalg.qr(d @ (d.T @ q))[0]
    u, s, vt = torch.linalg.svd(q.T @ d, full_matrices=False)
    return w + (q @ u[:, :3] * s[:3]) @ vt[:3]


def _reference(spec, lens, toks, targets, mode):
    """Residuals at every layer entry [layers + 1][rows][hidden] and the
    final-norm'd rows' logits weight, of prompts laid out one after another."""
    c = spec.config
    nb, T = len(lens), max(lens)
    at = torch.cumsum(_i64([0] + lens[:-1]), 0)
    pos = torch.arange(T, device="cuda")
    valid = pos[None] < _i64(lens)[:, None]
    idx = (at[:, None] + torch.minimum(pos[None], _i64(lens)[:, None] - 1)).reshape(-1)
    vec = {}

    def get(name, li=-1, e=-1):
        w = spec.get(name, li, e)
        if w is None:
            return None
        if id(w) not in vec or abi.SLOT[name] not in abi.VECTOR_SLOTS:
            d = _dense(w)
            if abi.SLOT[name] not in abi.VECTOR_SLOTS:
                for layer, slot, expert, v, weight in targets or ():
                    if (layer, slot, expert) == (li, abi.SLOT[name], e):
                        d = _delta(d, torch.from_numpy(v[0]).cuda().double(), weight, mode)
                return d
            vec[id(w)] = d.reshape(-1)
        return vec[id(w)]

    nh, hd, nkv = c["heads"], c["head_dim"], c["kv_heads"]
    vd, half = c["v_head_dim"], c["rotary_dim"] // 2
    ang = pos.double()[:, None] * c["rope_theta"] ** (-torch.arange(half, device="cuda").double() / half)[None]
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]

    def rope(x):  # [nb][T][heads][2 half]
        if c["rope_style"] == abi.ROPE_GPTJ:
            a, b = x[..., 0::2], x[..., 1::2]
            return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2)
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def ffn(x, gate, up, down):
        g = x @ gate.T
        return (g * torch.sigmoid(g) * (x @ up.T)) @ down.T

    emb = get("EMBED")
    x = emb[toks.long()[idx]].reshape(nb, T, -1)
    keep = valid.reshape(-1)
    res = [x.reshape(nb * T, -1)[keep]]
    mask = (pos[None] > pos[:, None])[None, None]
    for li in range(c["layers"]):
        h = _norm(x, get("ATTN_NORM", li))
        if c["mla"]:
            nope, rd, kl = c["qk_nope_dim"], c["qk_rope_dim"], c["kv_lora_rank"]
            q = _norm(h @ get("MLA_Q_A", li).T, get("MLA_Q_A_NORM", li)) @ get("MLA_Q_B", li).T
            q = q.reshape(nb, T, nh, hd)
            kva = h @ get("MLA_KV_A", li).T
            kvb = (_norm(kva[..., :kl], get("MLA_KV_A_NORM", li)) @ get("MLA_KV_B", li).T).reshape(nb, T, nh, nope + vd)
            q = torch.cat([q[..., :nope], rope(q[..., nope:])], -1)
            pe = rope(kva[..., None, kl:]).expand(nb, T, nh, rd)
            k, v = torch.cat([kvb[..., :nope], pe], -1), kvb[..., nope:]
        else:
            def proj(name, n):
                y, b = h @ get(name, li).T, get(name + "_BIAS", li)
                return (y if b is None else y + b).reshape(nb, T, n, hd)
            q, k, v = proj("Q", nh), proj("K", nkv), proj("V", nkv)
            if c["qk_norm"]:
                q, k = _norm(q, get("Q_NORM", li)), _norm(k, get("K_NORM", li))
            q, k = rope(q), rope(k)
            k, v = k.repeat_interleave(nh // nkv, 2), v.repeat_interleave(nh // nkv, 2)
        out = torch.empty(nb, T, nh, vd, dtype=torch.float64, device="cuda")
        for b in range(nb):
            s = q[b].transpose(0, 1) @ k[b].permute(1, 2, 0).contiguous() * c["attn_scale"]
            s = s.masked_fill(mask[0], -math.inf).softmax(-1)
            out[b] = (s @ v[b].transpose(0, 1).contiguous()).transpose(0, 1)
        x = x + out.reshape(nb, T, nh * vd) @ get("O", li).T
        h = _norm(x, get("FFN_NORM", li))
        if c["n_experts"]:
            hf, k = h.reshape(nb * T, -1), c["top_k"]
            logit = hf @ get("ROUTER", li).T
            p = torch.sigmoid(logit) if c["scoring"] == abi.SCORING_SIGMOID else logit.softmax(-1)
            corr = get("ROUTER_CORRECTION", li)
            choice = p if corr is None else p + corr
            if c["group_limited"]:
                per = choice.reshape(len(p), c["n_group"], -1)
                score = per.topk(1 if corr is None else 2, -1)[0].sum(-1)
                on = torch.zeros_like(score).scatter(1, score.topk(c["topk_group"], -1)[1], 1.0)
                choice = per.masked_fill(on[..., None] == 0, -math.inf).reshape(len(p), -1)
            sel = choice.topk(k, -1)[1]
            w = p.gather(1, sel)
            w = w / w.sum(-1, keepdim=True) * c["routed_scaling"]
            y = torch.zeros_like(hf)
            for e in range(c["n_experts"]):
                t, j = (sel == e).nonzero(as_tuple=True)
                if len(t):
                    y[t] += w[t, j, None] * ffn(hf[t], *(get("EXPERT_" + m, li, e) for m in ("GATE", "UP", "DOWN")))
            if c["shared_inter"]:
                y = y + ffn(hf, *(get("SHARED_" + m, li) for m in ("GATE", "UP", "DOWN")))
            x = x + y.reshape(x.shape)
        else:
            x = x + ffn(h, get("GATE", li), get("UP", li), get("DOWN", li))
        res.append(x.reshape(nb * T, -1)[keep])
    head = emb if c["tie_embeddings"] else get("LM_HEAD")
    return res, get("FINAL_NORM"), head


def exact(case, seed):
    if case["kind"] in ("product", "head"):
        w, x, extra = _product_inputs(case, seed)
        w = _dense(w)
        y = x.double() @ w.T
        if case["kind"] == "product":
            return y if extra is None else y + extra.double()
        lp, base = y.log_softmax(-1), (extra.double() @ w.T).log_softmax(-1)
        return {"logits": y, "logprobs": lp, "kl": (base.exp() * (base - lp)).sum(-1)}
    spec, lens, toks, targets = _prompt_inputs(case, seed)
    if case["kind"] == "decode":
        lens = [n + 1 for n in lens]
    res, norm, head = _reference(spec, lens, toks, targets, case.get("mode"))
    end = np.cumsum(lens)
    last = _i64([int(e) - 1 for e in end])
    logits = _norm(res[-1][last], norm) @ head.T
    if case["kind"] == "decode":
        return logits
    cap = _i64([r for e, n in zip(end, lens) for r in range(int(e) - min(n, WINDOW), int(e))])
    return {"residuals": torch.stack([r[cap] for r in res]), "logits": logits}
