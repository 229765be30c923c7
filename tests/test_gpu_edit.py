"""The edit in every row-normalisation mode on the device
(ditch_hip_edit_delta_ex / ditch_hip_model_edit_ex) against the oracle and
against the reference's own invariants (abliterate.zig:554-707) checked on
the device's deltas: the direction vanishes for none/pre, the rank-5 `full`
delta reproduces the exact renormalised 6 x 5 matrix, the input-side
ablation removes the read pattern; at realistic sizes the `full` delta's
error is within 10 % of the best rank-r error and its product B A matches
the oracle's (same test matrix, same algorithm). Then a forward after the
device edits against the oracle model carrying the oracle's deltas."""
import numpy as np
import pytest
import torch

import model_gen as mg
from ditch_amd import abi, synth
from ditch_amd.hip import Model
from ditch_amd.weights import HostWeight
from oracle.ref import RefModel
from test_gpu_forward import check_parity
from test_oracle_edit import MODES, exact_full, materialize, orthonormal_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [0, 9, (1 << 63) + 5])
def test_edit_gaussian_is_the_oracle_stream(dev, ref, seed):
    """The full edit's test matrix: Zig's floatNorm(f32) stream of
    DefaultPrng.init(seed), bit for bit the oracle's."""
    n = 200000
    out = np.empty(n, dtype=np.float32)
    dev.lib.ditch_hip_edit_gaussian(out.ctypes.data, n, seed)
    np.testing.assert_array_equal(out, ref.edit_gaussian(n, seed))


@pytest.mark.parametrize("k", [1, 2])
@pytest.mark.parametrize("mode", ["none", "pre", "full"])
def test_device_edit_reference_invariants_6x5(dev, k, mode):
    rng = np.random.default_rng(7)
    w = rng.standard_normal((6, 5)).astype(np.float32)
    v = orthonormal_rows(rng, 2, 6)[:k]
    a, b = dev.edit_delta_ex(HostWeight.f32(w), v, 1.0, mode, lora_rank=5, seed=1)
    assert a.shape[0] == (5 if mode == "full" else k)
    wp = materialize(w, a, b)
    n = np.ones(6) if mode == "none" else np.linalg.norm(w.astype(np.float64), axis=1)
    if mode != "full":
        assert np.abs((v / n) @ wp).max() < 1e-4
    else:
        np.testing.assert_allclose(wp, exact_full(w, v), atol=1e-3)


def test_device_input_side_ablation(dev):
    rng = np.random.default_rng(3)
    w = rng.standard_normal((6, 5)).astype(np.float32)
    v = orthonormal_rows(rng, 1, 6)
    u = (v.astype(np.float64) @ w)[0]
    u /= np.linalg.norm(u)
    for mode in ("none", "pre"):
        a, b = dev.edit_delta_ex(HostWeight.f32(w), v, 1.0, mode, ablate=True)
        wp = materialize(w, a, b)
        assert a.shape[0] == 2 and np.abs(wp @ u).max() < 1e-4
    a, b = dev.edit_delta_ex(HostWeight.f32(w), v, 1.0, "full", lora_rank=5, ablate=True)
    assert a.shape[0] == 6 and np.abs(materialize(w, a, b) @ u).max() < 1e-3


def _weight(fmt, rows, cols, seed):
    gen = torch.Generator().manual_seed(seed)
    return synth.QUANTIZERS[fmt](torch.randn(rows, cols, generator=gen) * 0.02)


CASES = [("bf16", 256, 512, 2, "none", False), ("fp8", 384, 1024, 2, "pre", False),
         ("mxfp4", 512, 768, 1, "full", False), ("int4", 384, 512, 2, "full", True),
         ("f32", 200, 150, 2, "full", False), ("q8_0", 256, 1024, 3, "pre", True)]


@pytest.mark.parametrize("fmt,rows,cols,k,mode,ablate", CASES, ids=[f"{c[0]}-{c[4]}-{c[5]}" for c in CASES])
def test_device_edit_matches_oracle(dev, ref, fmt, rows, cols, k, mode, ablate):
    w = _weight(fmt, rows, cols, rows + k)
    rng = np.random.default_rng(rows)
    v = orthonormal_rows(rng, k, rows)
    ga, gb = dev.edit_delta_ex(w, v, 1.0, mode, lora_rank=3, seed=9, ablate=ablate)
    ca, cb = ref.edit_delta_ex(w, v, 1.0, MODES[mode], lora_rank=3, seed=9, ablate=ablate)
    assert ga.shape == ca.shape and gb.shape == cb.shape
    gd = gb.astype(np.float64) @ ga.astype(np.float64)
    cd = cb.astype(np.float64) @ ca.astype(np.float64)
    scale = np.linalg.norm(cd)
    assert np.linalg.norm(gd - cd) <= (1e-2 if mode == "full" else 1e-4) * scale, np.linalg.norm(gd - cd) / scale
    if mode == "full" and not ablate:
        dense = ref.dequant(w)
        dense = ((dense.astype(np.uint32) << 16).view(np.float32) if dense.dtype == np.uint16 else dense)
        dstar = exact_full(dense, v) - dense.astype(np.float64)
        s = np.linalg.svd(dstar, compute_uv=False)
        best = np.sqrt((s[3:] ** 2).sum())
        assert np.linalg.norm(dstar - gd) <= 1.10 * best + 1e-6 * np.linalg.norm(dstar)


# the input side's U = orth(W^T V): one workgroup of 1, 4 and 8 columns a thread (up to 4, 4 and 2 vectors), three
# launches past them
@pytest.mark.parametrize("cols,k", [(30, 1), (1024, 4), (1026, 2), (4096, 4), (4096, 5), (4100, 1), (4100, 3), (8192, 2),
                                    (8194, 2)])
def test_input_side_directions_are_orthonormal(dev, ref, cols, k):
    rng = np.random.default_rng(cols + k)
    w = HostWeight.f32((rng.standard_normal((96, cols)) * 0.02).astype(np.float32))
    v = orthonormal_rows(rng, k, 96)
    a, _ = dev.edit_delta_ex(w, v, 1.0, "none", ablate=True)
    u = a[k:].astype(np.float64)
    want = v.astype(np.float64) @ ref.dequant(w).astype(np.float64)
    for i in range(k):
        for j in range(i):
            want[i] -= (want[i] @ want[j]) * want[j]
        want[i] /= np.linalg.norm(want[i])
    # one rounding an element; f32 sums over 96 rows (at most 96 * 2^-24 of the norm, nearly orthogonal vectors)
    assert np.abs(u @ u.T - np.eye(k)).max() <= 2.0**-22
    assert np.linalg.norm(u - want, axis=1).max() <= 96 * 2.0**-24 * 2


def test_input_side_direction_that_repeats_is_zero(dev):
    rng = np.random.default_rng(3)
    w = HostWeight.f32((rng.standard_normal((64, 700)) * 0.02).astype(np.float32))
    v = orthonormal_rows(rng, 3, 64)
    v[1] = v[0]
    a, b = dev.edit_delta_ex(w, v, 1.0, "none", ablate=True)
    u = a[3:].astype(np.float64)
    assert (u[1] == 0).all() and np.abs(u[[0, 2]] @ u[[0, 2]].T - np.eye(2)).max() <= 2.0**-22
    assert np.isfinite(a).all() and np.isfinite(b).all()


WIDE = [("f32", 300, 400, 2, "full", 40), ("bf16", 320, 400, 3, "full", 70), ("int4", 384, 512, 20, "pre", 3),
        ("fp8", 384, 1024, 24, "none", 3)]


@pytest.mark.parametrize("fmt,rows,cols,k,mode,lora", WIDE, ids=[f"{c[0]}-{c[4]}-k{c[3]}-r{c[5]}" for c in WIDE])
def test_device_edit_wide_ranks_match_oracle(dev, ref, fmt, rows, cols, k, mode, lora):
    """Ranks and direction counts the reference allows without a cap: the
    full edit at lora rank 40 (SVD width 84, Jacobi in LDS) and 70 (width
    144, Jacobi in global memory, delta rank above 64), and 20 / 24
    directions."""
    w = _weight(fmt, rows, cols, rows + k)
    rng = np.random.default_rng(rows + k)
    v = orthonormal_rows(rng, k, rows)
    ga, gb = dev.edit_delta_ex(w, v, 1.0, mode, lora_rank=lora, seed=3)
    ca, cb = ref.edit_delta_ex(w, v, 1.0, MODES[mode], lora_rank=lora, seed=3)
    assert ga.shape == ca.shape and gb.shape == cb.shape
    gd = gb.astype(np.float64) @ ga.astype(np.float64)
    cd = cb.astype(np.float64) @ ca.astype(np.float64)
    scale = np.linalg.norm(cd)
    assert np.linalg.norm(gd - cd) <= (1e-2 if mode == "full" else 1e-4) * scale, np.linalg.norm(gd - cd) / scale
    if mode == "full":
        dense = ref.dequant(w)
        dense = ((dense.astype(np.uint32) << 16).view(np.float32) if dense.dtype == np.uint16 else dense)
        dstar = exact_full(dense, v) - dense.astype(np.float64)
        s = np.linalg.svd(dstar, compute_uv=False)
        best = np.sqrt((s[lora:] ** 2).sum())
        assert np.linalg.norm(dstar - gd) <= 1.10 * best + 1e-6 * np.linalg.norm(dstar)


@pytest.mark.parametrize("mode", ["pre", "full"])
def test_model_edit_ex_then_forward(dev, ref, mode):
    """Edits of every o_proj, dense down_proj and routed expert down_proj
    (resident and streamed through a quarter-size cache), then the forward,
    against the oracle model carrying the oracle's deltas."""
    spec = mg.moe("int4", layers=3, dense_first=1, experts=8, top_k=2, seed=31)
    c = spec.config
    rng = np.random.default_rng(4)
    v = orthonormal_rows(rng, 2, c["hidden"])
    tokens, rows, last = mg.batch(3, [20, 33, 7], c["vocab"], seed=5)
    targets = []
    for li in range(c["layers"]):
        targets.append((li, abi.SLOT["O"], -1))
        if spec.moe_layers[li]:
            targets += [(li, abi.SLOT["EXPERT_DOWN"], e) for e in range(c["n_experts"])]
        else:
            targets.append((li, abi.SLOT["DOWN"], -1))
    cm = RefModel(spec)
    try:
        for li, slot, e in targets:
            ca, cb = ref.edit_delta_ex(spec.get(slot, li, e), v, 0.8, MODES[mode], lora_rank=3, seed=li * 100 + e + 1)
            cm.set_delta(li, slot, e, ca, cb)
        rc, lc = cm.forward(tokens, rows, capture_rows=last, logit_rows=last)
        for cache in (0, 1):
            gm = Model(dev, spec, expert_cache_bytes=(1 << 40) if cache else 0)
            try:
                if cache:  # a cache of a quarter of the experts
                    gm.forward(tokens, rows, logit_rows=last)
                    slot_bytes = gm.expert_cache_stats()["slot_bytes"]
                    gm.free()
                    gm = Model(dev, spec, expert_cache_bytes=2 * c["n_experts"] * slot_bytes // 4)
                for li, slot, e in targets:
                    gm.edit_ex(li, slot, e, v, 0.8, mode, lora_rank=3, seed=li * 100 + e + 1)
                rg, lg = gm.forward(tokens, rows, capture_rows=last, logit_rows=last)
            finally:
                gm.free()
            check_parity(ref, rg, lg, rc, lc, f"edit_ex {mode} cache={cache}")
    finally:
        cm.free()


# SVD widths q = 2 lora + 4 at the edges of the chunked orthonormalisation's
# instances (12 | 14, 24 | 26), more directions than it takes beside it, and
# widths around a chunk of 64 columns
@pytest.mark.parametrize("rows,cols,k,lora", [(256, 320, 1, 4), (193, 4160, 2, 5), (129, 65, 1, 10), (128, 64, 1, 11),
                                              (200, 300, 8, 8), (200, 300, 9, 9), (31, 40, 3, 1)])
def test_full_edit_svd_widths_match_oracle(dev, ref, rows, cols, k, lora):
    w = _weight("f32", rows, cols, rows + k)
    rng = np.random.default_rng(rows + k)
    v = orthonormal_rows(rng, k, rows)
    ga, gb = dev.edit_delta_ex(w, v, 1.0, "full", lora_rank=lora, seed=5, ablate=lora == 4)
    ca, cb = ref.edit_delta_ex(w, v, 1.0, MODES["full"], lora_rank=lora, seed=5, ablate=lora == 4)
    assert ga.shape == ca.shape and gb.shape == cb.shape
    gd = gb.astype(np.float64) @ ga.astype(np.float64)
    cd = cb.astype(np.float64) @ ca.astype(np.float64)
    # the randomised SVD's tail, as in the tests above
    assert np.linalg.norm(gd - cd) <= 1e-2 * np.linalg.norm(cd)


@pytest.mark.parametrize("rank", [0, 1, 3])
def test_full_edit_of_a_rank_deficient_weight(dev, ref, rank):
    """Fewer independent columns than SVD vectors: the dependent ones vanish
    and the factors stay finite."""
    rng = np.random.default_rng(rank)
    rows, cols = 96, 130
    w = (rng.standard_normal((rows, rank)) @ rng.standard_normal((rank, cols))).astype(np.float32) * 0.1
    v = orthonormal_rows(rng, 1, rows)
    ga, gb = dev.edit_delta_ex(HostWeight.f32(w), v, 1.0, "full", lora_rank=3, seed=2)
    assert np.isfinite(ga).all() and np.isfinite(gb).all()
    ca, cb = ref.edit_delta_ex(HostWeight.f32(w), v, 1.0, MODES["full"], lora_rank=3, seed=2)
    gd = gb.astype(np.float64) @ ga.astype(np.float64)
    cd = cb.astype(np.float64) @ ca.astype(np.float64)
    # directions of rounding noise differ; they carry at most its 1e-6
    assert np.linalg.norm(gd - cd) <= 1e-2 * np.linalg.norm(cd) + 1e-6 * np.linalg.norm(w)


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "mxfp4", "int4", "q8_0", "f32"])
@pytest.mark.parametrize("k", [1, 2, 3, 9])
def test_directions_of_one_launch_match_oracle(dev, ref, fmt, k):
    """A = V^T W with one, two and four directions a workgroup; the last
    workgroup's beyond k."""
    w = _weight(fmt, 272, 640, k)
    v = orthonormal_rows(np.random.default_rng(k), k, 272)
    ga, gb = dev.edit_delta_ex(w, v, 1.0, "none")
    ca, cb = ref.edit_delta_ex(w, v, 1.0, MODES["none"])
    # f32 sums of 272 products in another order: 272 * 2^-24 of the largest
    assert np.abs(ga - ca).max() <= 2e-5 * np.abs(ca).max() and np.array_equal(gb, cb)


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "q8_0"])
@pytest.mark.parametrize("k", [1, 5])
def test_a_delta_has_the_same_bits_alone_and_in_a_batch(dev, fmt, k):
    """Batches of more than 512 column units, each matrix of far fewer: the
    forward after them is that after an edit per matrix, bit for bit."""
    inter = {"bf16": 4096, "fp8": 8192, "q8_0": 8192}[fmt]
    spec = mg.dense(fmt, hidden=128, inter=inter, layers=5, heads=2, kv_heads=2, head_dim=64, vocab=256, seed=k)
    rng = np.random.default_rng(k)
    targets = [(li, abi.SLOT["DOWN"], -1, orthonormal_rows(rng, k, 128), 0.7) for li in range(5)]
    tokens, rows, last = mg.batch(2, [3, 9], 256, seed=2)
    gm = Model(dev, spec)
    try:
        gm.edit_batch(targets, k)
        want = gm.forward(tokens, rows, capture_rows=last, logit_rows=last)
        gm.reset_deltas()
        for t in targets:
            gm.edit(*t)
        got = gm.forward(tokens, rows, capture_rows=last, logit_rows=last)
    finally:
        gm.free()
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
