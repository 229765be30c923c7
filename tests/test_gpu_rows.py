"""Row kernels and the few-token forward at the edges of their ranges, against
the oracle (needs an MI355X)."""
import ctypes

import numpy as np
import pytest

import model_gen as mg
import weights_gen as wg
from ditch_amd import abi, hipmem
from ditch_amd.hip import Model
from oracle.ref import RefModel

pytestmark = pytest.mark.gpu


# one 8-column piece, a wave's edge, more columns than a workgroup of 512, the
# longest row of the row kernel; then the general kernel (longer, not of 8)
@pytest.mark.parametrize("length", [8, 512, 520, 7168, 8192, 8200, 1020])
@pytest.mark.parametrize("n", [1, 129])
def test_rmsnorm_row_lengths(dev, ref, n, length):
    rng = np.random.default_rng(length + n)
    x = (rng.standard_normal((n, length)) * 3).astype(np.float32)
    w = rng.standard_normal(length).astype(np.float32)
    # sums of squares and products in f32, at most a few roundings a value
    for weight, gemma in ((w, False), (w, True), (None, False)):
        want = ref.rmsnorm_rows(x, weight, 1e-6, gemma=gemma)
        got = dev.rmsnormRows(x, weight, 1e-6, gemma_style=gemma)
        assert np.abs(got - want).max() <= 4e-6 * np.abs(want).max()


def _check(gm, cm, lens, vocab, seed):
    tokens, rows, last = mg.batch(len(lens), lens, vocab, seed=seed)
    rg, lg = gm.forward(tokens, rows, capture_rows=last, logit_rows=last)
    rc, lc = cm.forward(tokens, rows, capture_rows=last, logit_rows=last)
    # two-term products (2^-18 an activation) and other summation orders
    # through two layers: 1e-5 of the largest value, ten times that allowed
    assert np.abs(lg - lc).max() <= 1e-4 * np.abs(lc).max()
    assert np.abs(rg - rc).max() <= 1e-4 * np.abs(rc).max()


# f32 rows up to 8 tokens, fragments above; one and two token blocks; the last
# count of the few-token path and the first two of the tiled one
LENS = [[1], [5, 3], [9], [7, 9], [17], [33], [63, 64], [128], [100, 30]]


# (gate and up in one launch: above 8 tokens where their rows are a multiple of 128; int4 rows are whole 128-column groups)
@pytest.mark.parametrize("fmt,inter", [(f, i) for f in ("bf16", "fp8", "mxfp4", "int4", "q8_0", "f32") for i in (640, 672)
                                       if f != "int4" or i == 640])
def test_forward_token_counts_match_oracle(dev, ref, fmt, inter):
    """Plain layers, then with deltas on o and down (whose inputs stay f32)."""
    spec = mg.dense(fmt, hidden=384, inter=inter, heads=6, kv_heads=2, head_dim=64, layers=2, vocab=640, seed=4)
    gm, cm = Model(dev, spec), RefModel(spec)
    rng = np.random.default_rng(5)
    try:
        for i, lens in enumerate(LENS):
            _check(gm, cm, lens, 640, i)
        for slot, k, rank, li in ((abi.SLOT["O"], 384, 3, 0), (abi.SLOT["DOWN"], inter, 2, 1)):
            a = (rng.standard_normal((rank, k)) * 0.05).astype(np.float32)
            b = (rng.standard_normal((384, rank)) * 0.05).astype(np.float32)
            for m in (gm, cm):
                m.set_delta(li, slot, -1, a, b)
        for i, lens in enumerate(LENS):
            _check(gm, cm, lens, 640, 20 + i)
    finally:
        gm.free()
        cm.free()


# Gate and up in one launch (launch_glu): a layer on each side of its lines, by the 16-row groups of both matrices (rows
# / 8), the 128-column steps and, from fragments, the 16-token blocks. The waves K is split over, from f32 rows and
# from fragments, and the token blocks x row groups of a matrix a workgroup has there
GLU_SHAPES = {
    "8_waves_rows_and_fragments": (2176, 256, [[3], [9], [16]]),  # 32 groups, 17 steps, one block: 8; 8, 1 x 1
    "8_waves_rows_last_step_half": (1088, 640, [[1], [2], [4], [5, 3], [13]]),  # 80 groups, 9 steps: 8; 4, 1 x 1
    "4_waves_wide_rows": (1152, 4096, [[1], [6], [11]]),  # 512 groups, 9 steps: 4; 4, 1 x 1
    "two_blocks": (128, 4096, [[17], [20, 12]]),  # 512 groups x 2 blocks: 4, 2 x 1
    "two_blocks_of_two_groups": (128, 12288, [[17], [20, 12]]),  # 1536 groups x 2 blocks: 4, 2 x 2 (FP8: 2 x 1)
}


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "mxfp4", "int4", "q8_0"])
@pytest.mark.parametrize("shape", list(GLU_SHAPES))
def test_gate_up_of_few_tokens_matches_oracle(dev, ref, fmt, shape):
    hidden, inter, lens = GLU_SHAPES[shape]
    if fmt == "int4":
        hidden = -(-hidden // 128) * 128  # (whole 128-column groups)
    spec = mg.dense(fmt, hidden=hidden, inter=inter, heads=2, kv_heads=1, head_dim=64, layers=1, vocab=256, seed=3)
    gm, cm = Model(dev, spec), RefModel(spec)
    try:
        for i, prompts in enumerate(lens):
            _check(gm, cm, prompts, 256, 40 + i)
    finally:
        gm.free()
        cm.free()


# 33 to 127 tokens where the few-token kernel takes a part of a layer: from 65 on all but o and down (16384 rows: two
# rounds each), which read the fragments of the attention and the gate/up product, or with a delta its f32 rows; all
# but gate and up (32768 rows: eight rounds). On 48 all of both
@pytest.mark.parametrize("fmt,hidden,inter", [("bf16", 16384, 256), ("bf16", 256, 32768), ("q8_0", 256, 32768)])
def test_layers_partly_of_few_token_products_match_oracle(dev, ref, fmt, hidden, inter):
    spec = mg.dense(fmt, hidden=hidden, inter=inter, heads=2, kv_heads=1, head_dim=128, layers=1, vocab=256, seed=8)
    gm, cm = Model(dev, spec), RefModel(spec)
    rng = np.random.default_rng(7)
    try:
        for i, lens in enumerate([[48], [65], [60, 51]]):
            _check(gm, cm, lens, 256, 60 + i)
        for slot, k in ((abi.SLOT["O"], 256), (abi.SLOT["DOWN"], inter)):
            a = (rng.standard_normal((2, k)) * 0.05).astype(np.float32)
            b = (rng.standard_normal((hidden, 2)) * 0.05).astype(np.float32)
            for m in (gm, cm):
                m.set_delta(0, slot, -1, a, b)
        _check(gm, cm, [60, 51], 256, 63)
    finally:
        gm.free()
        cm.free()


# one element, the edges of a 2048-element chunk, of the lanes that add 64
# chunks, and rows that are not whole float4s
@pytest.mark.parametrize("V", [1, 2047, 2048, 2052, 133120, 131073])
def test_log_softmax_and_kl_row_lengths(dev, ref, V):
    rng = np.random.default_rng(V)
    x = (rng.standard_normal((3, V)) * 5).astype(np.float32)
    x[1, : V // 2] = -np.inf  # whole chunks of masked logits
    x[2, 0] = 80.0
    lp = dev.logSoftmaxRows(x)
    want = ref.log_softmax_rows(x)
    fin = np.isfinite(want)
    # one f32 rounding of lse and one of the difference, at most 100 large
    assert np.array_equal(fin, np.isfinite(lp)) and np.abs(lp[fin] - want[fin]).max() <= 4 * 2.0**-24 * 128
    # a row against its own log-probs; masked logits on both sides are NaN (0 * inf)
    kl = dev.klRows(lp, x)
    assert kl[0] == 0 and kl[2] == 0
    if V > 1:
        assert np.isnan(kl[1]) and np.isnan(ref.kl_rows(want, x)[1])


# one buffer off 16-byte alignment (read element by element), rows of whole float4s or not
@pytest.mark.parametrize("V", [5000, 4099])
@pytest.mark.parametrize("off", [(0, 0, 4), (0, 4, 0), (4, 0, 0), (4, 4, 4)])
def test_kl_against_own_log_probs_is_zero_at_any_alignment(dev, V, off):
    x = (np.random.default_rng(V).standard_normal((3, V)) * 5).astype(np.float32)
    bufs = [hipmem.Buffer(x.nbytes + 16) for _ in range(3)]  # the logits, their log-softmax, the logits for KL
    at = [ctypes.c_void_p(b.ptr.value + o) for b, o in zip(bufs, off)]
    for i in (0, 2):
        bufs[i].upload(np.concatenate([np.zeros(off[i] // 4, np.float32), x.reshape(-1)]))
    kl = hipmem.Buffer(3 * 8)
    dev.logSoftmaxRows_device(at[1], at[0], 3, V)
    dev.klRows_device(kl.ptr, at[1], at[2], 3, V)
    dev.sync()
    assert (kl.download(np.float64, (3,)) == 0).all()


# one to eight rows an expert (instances of 2, 4 and 8 rows), nine (two chunks
# each: the GEMV), chunks of unequal experts, with and without deltas on the experts' down projections
@pytest.mark.parametrize("fmt,experts", [("bf16", 4), ("fp8", 4), ("mxfp4", 4), ("int4", 4), ("q8_0", 4), ("int4", 12)])
def test_few_rows_an_expert_match_oracle(dev, ref, fmt, experts):
    spec = mg.moe(fmt, layers=1, experts=experts, top_k=4, seed=13)
    c = spec.config
    gm, cm = Model(dev, spec), RefModel(spec)
    rng = np.random.default_rng(6)
    try:
        for i in range(2):
            for j, lens in enumerate([[1], [2], [3], [5], [3, 5], [9], [13, 6]]):  # (4 experts: every row at each)
                _check(gm, cm, lens, c["vocab"], 10 * i + j)
            for e in (0, 3):
                a = (rng.standard_normal((e + 1, c["moe_inter"])) * 0.05).astype(np.float32)
                b = (rng.standard_normal((c["hidden"], e + 1)) * 0.05).astype(np.float32)
                for m in (gm, cm):
                    m.set_delta(0, abi.SLOT["EXPERT_DOWN"], e, a, b)
    finally:
        gm.free()
        cm.free()


# an expert's gate and up need not share their scale layout: other group widths, scale types and block widths,
# in every expert or in one that is not the first
LAYOUTS = {
    "int4_groups": ("int4", dict(group=64), dict(group=128)),
    "int4_groups_up_finer": ("int4", dict(group=128), dict(group=64)),
    "int4_scale_types": ("int4", dict(scale_kind="f16"), dict(scale_kind="bf16")),
    "fp8_blocks": ("fp8", dict(block=(128, 64)), dict(block=(128, 128))),
}


def _mixed_experts(layout, which, seed):
    fmt, gate, up = LAYOUTS[layout]
    make = wg.int_random if fmt == "int4" else wg.fp8_random
    spec = mg.moe(fmt, layers=1, experts=4, top_k=4, seed=seed)
    c, rng = spec.config, np.random.default_rng(seed)
    for e in range(4):
        spec.set("EXPERT_GATE", make(c["moe_inter"], c["hidden"], rng, **gate), 0, e)
        spec.set("EXPERT_UP", make(c["moe_inter"], c["hidden"], rng, **(up if which in ("all", e) else gate)), 0, e)
    return spec


@pytest.mark.parametrize("which", ["all", 2])
@pytest.mark.parametrize("layout", list(LAYOUTS))
def test_experts_of_unequal_scale_layouts_match_oracle(dev, ref, layout, which):
    spec = _mixed_experts(layout, which, 21)
    gm, cm = Model(dev, spec), RefModel(spec)
    try:
        # (every row at each expert; 40 rows take the tiled products)
        for j, lens in enumerate([[1], [5], [9], [40]]):
            _check(gm, cm, lens, spec.config["vocab"], 30 + j)
    finally:
        gm.free()
        cm.free()
