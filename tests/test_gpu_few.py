"""The few-token product (csrc/gemm_few.hip) against the oracle at the edges of
its dispatch and tiles: every format, up to 8 tokens from f32 rows and more
from fragments, K of less than one 128-column step, of partial units and steps
and of K slices of unequal length, rows that leave a row group and a row block
part empty, the grids on both sides of each tile choice, and the last token
count it takes."""
import ctypes

import numpy as np
import pytest

import weights_gen as wg
from ditch_amd import hipmem
from test_gpu_kernels import TOL_MATMUL, dequant_f32, split_bound

pytestmark = pytest.mark.gpu

# kind, n, rows, cols
CASES = [
    ("bf16", 1, 17, 36), ("bf16", 3, 33, 132), ("bf16", 4, 40, 30), ("bf16", 8, 8208, 160),
    ("bf16", 9, 50, 96), ("bf16", 16, 64, 4128), ("bf16", 49, 4096, 288), ("bf16", 255, 100, 160),
    ("fp8", 1, 520, 4160), ("fp8", 2, 31, 64), ("fp8", 7, 130, 1216), ("fp8", 12, 48, 4160),
    ("fp8", 33, 3000, 320), ("fp8", 200, 1100, 128),
    ("mxfp4", 1, 48, 160), ("mxfp4", 5, 130, 4256), ("mxfp4", 8, 8200, 128), ("mxfp4", 17, 24, 4096),
    ("mxfp4", 31, 700, 544), ("mxfp4", 100, 4096, 256), ("mxfp4", 200, 72, 640),
    ("int4", 1, 130, 192), ("int4", 4, 72, 4224), ("int4", 8, 16, 128), ("int4", 10, 260, 2240),
    ("int4", 48, 4000, 256), ("int4", 130, 72, 1024),
    ("q8_0", 2, 8208, 96), ("q8_0", 6, 70, 4128), ("q8_0", 15, 33, 1056), ("q8_0", 64, 3080, 64), ("q8_0", 129, 40, 416),
    # 17 to 31 tokens: chunks of rows up to 2^22 weights, fragments above
    ("fp8", 31, 4096, 1024), ("bf16", 24, 4100, 1028), ("mxfp4", 31, 2080, 2080), ("int4", 17, 4112, 1152),
    # odd rows of up to 8 tokens on both sides of the GEMV's line
    ("bf16", 5, 40, 4094), ("bf16", 5, 40, 4098), ("fp8", 3, 40, 30),
    # the tallest weights from 17 tokens on: the products that ran before
    ("bf16", 24, 65540, 64), ("bf16", 32, 65540, 96), ("bf16", 17, 65540, 516), ("q8_0", 20, 65540, 64),
    ("q8_0", 32, 65540, 64), ("int4", 31, 65540, 128),
]


@pytest.mark.parametrize("kind,n,rows,cols", CASES)
def test_few_token_product(dev, ref, kind, n, rows, cols):
    """Two-term products with bias and accumulate on a resident tensor."""
    rng = np.random.default_rng(n * 7919 + rows + cols)
    w = wg.make(kind, rows, cols, rng)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    bias = rng.standard_normal(rows).astype(np.float32)
    prior = rng.standard_normal((n, rows)).astype(np.float32)
    t = dev.upload(w)
    try:
        bx, bb, bo = (hipmem.Buffer.from_array(a) for a in (x, bias, prior))
        t.matmul_device(bo.ptr, bx.ptr, n, d_bias=bb.ptr, accumulate=True)
        dev.sync()
        got = bo.download(np.float32, (n, rows))
    finally:
        t.free()
    want = prior.astype(np.float64) + ref.matmulT(x, w).astype(np.float64) + bias
    # the activations' two terms: 2^-18 of each (split_bound's bf16 form, four times it)
    bound = split_bound("bf16", x, dequant_f32(ref, w))
    bad = np.abs(got - want) > TOL_MATMUL["atol"] + TOL_MATMUL["rtol"] * np.abs(want) + bound
    assert not bad.any(), f"{bad.sum()} of {bad.size} outside the bound"


@pytest.mark.parametrize("kind", ["bf16", "fp8", "mxfp4", "int4", "q8_0"])
@pytest.mark.parametrize("n", [1, 6, 16, 32])
def test_few_token_exact_product(dev, ref, kind, n):
    """Three-term products (the VTable entry) at the reference's tolerance."""
    rng = np.random.default_rng(n)
    w = wg.make(kind, 600, 1216, rng)
    x = rng.standard_normal((n, 1216)).astype(np.float32)
    got, want = dev.matmulT(x, w), ref.matmulT(x, w)
    bad = np.abs(got - want) > TOL_MATMUL["atol"] + TOL_MATMUL["rtol"] * np.abs(want)
    assert not bad.any()


@pytest.mark.parametrize("n", [6, 20])
def test_non_finite_activations_stay_in_their_token(dev, ref, n):
    rng = np.random.default_rng(3)
    w = wg.make("fp8", 96, 320, rng)
    x = rng.standard_normal((n, 320)).astype(np.float32)
    clean = dev.matmulT(x, w)
    x[2, 5], x[4, 300] = np.inf, np.nan
    got = dev.matmulT(x, w)
    others = [i for i in range(n) if i not in (2, 4)]
    assert not np.isfinite(got[[2, 4]]).any()
    np.testing.assert_array_equal(got[others], clean[others])


@pytest.mark.parametrize("n,rows,cols", [(128, 72, 640), (255, 40, 4096)])
def test_mxfp4_from_128_tokens_keeps_the_scaled_product_s_precision(dev, ref, n, rows, cols):
    """Three terms, as the fp6 terms of the scaled MFMA hold 18 bits: the error
    against 64 bits is that of f32 sums (two terms: 2.5e-6)."""
    rng = np.random.default_rng(n)
    w = wg.make("mxfp4", rows, cols, rng)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    t = dev.upload(w)
    try:
        bx, bo = hipmem.Buffer.from_array(x), hipmem.Buffer(n * rows * 4)
        t.matmul_device(bo.ptr, bx.ptr, n)
        dev.sync()
        got = bo.download(np.float32, (n, rows)).astype(np.float64)
    finally:
        t.free()
    want = x.astype(np.float64) @ dequant_f32(ref, w).astype(np.float64).T
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


def _stream(lib):
    s = ctypes.c_void_p()
    assert lib.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0  # non-blocking, default priority
    return s


@pytest.mark.parametrize("kind,n,rows,cols", [("bf16", 17, 50, 132), ("fp8", 24, 8208, 320), ("mxfp4", 25, 4096, 256),
                                              ("int4", 31, 130, 2240), ("q8_0", 20, 33, 1056), ("bf16", 18, 40, 30),
                                              ("fp8", 5, 50, 131), ("bf16", 8, 33, 4099),
                                              ("bf16", 20, 65540, 64), ("q8_0", 31, 98304, 64), ("bf16", 17, 65540, 1028)])
def test_chunks_of_rows_on_another_stream(dev, ref, kind, n, rows, cols):
    """17 to 31 tokens without scratch: chunks of 8 rows (the last one of any
    size), or the register-staged product where rows are not whole float4s or the
    weights are the tallest.
    Up to 8 tokens of such rows: the GEMV."""
    rng = np.random.default_rng(n + rows + cols)
    w = wg.make(kind, rows, cols, rng)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    bias = rng.standard_normal(rows).astype(np.float32)
    prior = rng.standard_normal((n, rows)).astype(np.float32)
    lib = hipmem.hip()
    s, t = _stream(lib), dev.upload(w)
    try:
        bx, bb, bo = (hipmem.Buffer.from_array(a) for a in (x, bias, prior))
        t.matmul_device(bo.ptr, bx.ptr, n, d_bias=bb.ptr, accumulate=True, stream=s.value)
        assert lib.hipStreamSynchronize(s) == 0
        got = bo.download(np.float32, (n, rows))
    finally:
        t.free()
        lib.hipStreamDestroy(s)
    want = prior.astype(np.float64) + ref.matmulT(x, w).astype(np.float64) + bias
    bound = split_bound("bf16", x, dequant_f32(ref, w))
    assert (np.abs(got - want) <= TOL_MATMUL["atol"] + TOL_MATMUL["rtol"] * np.abs(want) + bound).all()


@pytest.mark.parametrize("counts,kinds", [((17, 24, 31), (("fp8", 2048, 1024), ("int4", 1024, 4096))),
                                          ((1, 5, 8), (("fp8", 2048, 1026), ("bf16", 512, 4102)))])
def test_products_without_shared_scratch_on_two_streams(dev, ref, counts, kinds):
    """17 to 31 tokens, and up to 8 whose rows are not whole float4s. No order
    between the streams and the context's own: every output is that of the
    call alone."""
    rng = np.random.default_rng(8)
    lib = hipmem.hip()
    streams = [_stream(lib).value, _stream(lib).value, None]
    t = [dev.upload(wg.make(*kind, rng)) for kind in kinds]
    try:
        jobs = []
        for i in range(24):
            w, n = t[i % 2], counts[i // 2 % 3]
            bx = hipmem.Buffer.from_array(rng.standard_normal((n, w.cols)).astype(np.float32))
            outs = [hipmem.Buffer(n * w.rows * 4) for _ in range(2)]
            jobs.append((w, n, bx, outs, streams[i % 3]))
        for alone in (False, True):
            for w, n, bx, outs, s in jobs:
                w.matmul_device(outs[alone].ptr, bx.ptr, n, stream=s)
                if alone:
                    hipmem.synchronize()
            hipmem.synchronize()
        for w, n, bx, outs, s in jobs:
            a, b = (o.download(np.float32, (n, w.rows)) for o in outs)
            np.testing.assert_array_equal(a, b)
    finally:
        for w in t:
            w.free()
        for s in streams[:2]:
            lib.hipStreamDestroy(s)


@pytest.mark.parametrize("n,cols", [(24, 2048), (6, 2050)])
@pytest.mark.parametrize("own", [False, True])
def test_product_captured_without_a_warm_up(dev, own, n, cols):
    """On another stream and on the context's own: nothing is allocated under
    the capture, and a larger product afterwards leaves the graph's replays."""
    lib = hipmem.hip()
    P = ctypes.c_void_p
    for name, args in {"hipStreamBeginCapture": [P, ctypes.c_int], "hipStreamEndCapture": [P, ctypes.POINTER(P)],
                       "hipGraphInstantiate": [ctypes.POINTER(P), P, P, P, ctypes.c_size_t],
                       "hipGraphLaunch": [P, P], "hipGraphExecDestroy": [P], "hipGraphDestroy": [P]}.items():
        getattr(lib, name).argtypes = args
        getattr(lib, name).restype = ctypes.c_int
    rng = np.random.default_rng(9)
    rows = 512
    t, big = dev.upload(wg.make("fp8", rows, cols, rng)), dev.upload(wg.make("fp8", 64, 16384, rng))
    made = None if own else _stream(lib)
    stream = P(dev.stream) if own else made
    graph, ge = P(), P()
    try:
        bx, bo, want = hipmem.Buffer(n * cols * 4), hipmem.Buffer(n * rows * 4), hipmem.Buffer(n * rows * 4)
        bb, ob = hipmem.Buffer.from_array(np.ones((31, 16384), np.float32)), hipmem.Buffer(31 * 64 * 4)
        assert lib.hipStreamBeginCapture(stream, 0) == 0  # hipStreamCaptureModeGlobal
        t.matmul_device(bo.ptr, bx.ptr, n, stream=stream.value)
        assert lib.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert lib.hipGraphInstantiate(ctypes.byref(ge), graph, None, None, 0) == 0
        for _ in range(3):
            bx.upload(rng.standard_normal((n, cols)).astype(np.float32))
            big.matmul_device(ob.ptr, bb.ptr, 31)
            t.matmul_device(want.ptr, bx.ptr, n)
            hipmem.synchronize()
            assert lib.hipGraphLaunch(ge, stream) == 0
            hipmem.synchronize()
            a, b = bo.download(np.float32, (n, rows)), want.download(np.float32, (n, rows))
            # the same products, summed in another order: f32 rounding only
            assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()
    finally:
        if ge.value:
            lib.hipGraphExecDestroy(ge)
        if graph.value:
            lib.hipGraphDestroy(graph)
        if made:
            lib.hipStreamDestroy(made)
        t.free()
        big.free()
