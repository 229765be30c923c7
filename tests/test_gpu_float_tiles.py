"""Products on f32 / f16 weights above 16 tokens (csrc/gemm_f32.hip) at the
edges of the staged tiles: each tile and slice count of the dispatch and each
span of its sums, ragged rows and tokens, K of one unit (slices without any),
of slices of unequal length and of whole spans with a remainder, rows that are
not whole units, and a gathered non-finite activation that must stay in its
token."""
import os
import re

import numpy as np
import pytest

import weights_gen as wg
from ditch_amd import hipmem
from test_gpu_kernels import TOL_MATMUL, close, dequant_f32

pytestmark = pytest.mark.gpu


# The kernel that each case runs, as <waves a side, K slices, units a sum>
# (None: rows that are not whole units, the register-staged kernel)
CASES = {
    (17, 33, 32): (1, 4, 16), (40, 130, 160): (1, 4, 16), (100, 1000, 96): (1, 4, 16),
    (1100, 950, 96): (1, 4, 16), (1090, 1030, 32): (1, 4, 16),
    (40, 130, 2208): (1, 4, 16),  # 69 units: slices of 17 and 18, a whole sum and a remainder
    (1024, 896, 160): (2, 2, 2), (1000, 885, 32): (2, 2, 2),  # (one unit: a slice without any)
    (1000, 885, 1056): (2, 2, 4), (1000, 885, 2144): (2, 2, 16),  # 33 units: 16 and 17; 67: 33 and 34
    (1030, 1310, 32): (2, 1, 2), (1030, 1310, 288): (2, 1, 2), (1030, 1310, 544): (2, 1, 4),
    (1030, 1310, 2144): (2, 1, 16),
    (50, 70, 72): None,
}


def _instance(n, rows, cols):
    """launch_staged's choice, with the constants that its source has."""
    path = os.path.join(os.path.dirname(__file__), "..", "ditch_amd", "csrc", "gemm_f32.hip")
    with open(path) as f:
        src = f.read()
    one, two, small = map(float, re.search(r"\* 4 / ([\d.]+) : 4 / ([\d.]+);\n.*?/ 256\) / ([\d.]+);", src).groups())
    whole, quarter = map(int, re.search(r"units_k < (\d+)\) \{\n +if \(p\.w\.units_k < (\d+)\)", src).groups())
    if cols % 32:
        return None

    def tiles(side):
        return -(-n // side) * -(-rows // side)

    big = -(-tiles(64) // 256) * 4 / one if tiles(64) > 256 else 4 / two
    wg, ks = (1, 4) if -(-tiles(32) // 256) / small < big else (2, 1) if tiles(64) > 256 else (2, 2)
    units = cols // 32
    return wg, ks, 16 if ks == 4 or units >= whole else 4 if units >= quarter else 2


@pytest.mark.parametrize("kind", ["f32", "f16"])
@pytest.mark.parametrize("n,rows,cols", list(CASES))
def test_float_tiles(dev, ref, kind, n, rows, cols):
    assert _instance(n, rows, cols) == CASES[n, rows, cols]
    rng = np.random.default_rng(n + rows + cols)
    w = wg.float_random(kind, rows, cols, rng)
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
    close(got, prior.astype(np.float64) + ref.matmulT(x, w).astype(np.float64) + bias, **TOL_MATMUL)


def test_infinite_activation_keeps_its_sign(dev, ref):
    """Exact products: an infinite activation gives infinities in its own
    token's outputs, as f32 multiply-adds do, and nothing elsewhere."""
    rng = np.random.default_rng(1)
    w = wg.float_random("f32", 100, 96, rng)
    x = rng.standard_normal((40, 96)).astype(np.float32)
    x[7, 5] = np.inf
    got, want = dev.matmulT(x, w), ref.matmulT(x, w)
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    assert np.isinf(want[7]).all() and (np.sign(got[7]) == np.sign(want[7])).all()
    close(np.delete(got, 7, 0), np.delete(want, 7, 0), **TOL_MATMUL)


# The error against 64 bits, N(0, 1) activations and N(0, 0.02) weights: at most that of the register-staged kernel
# that these products had before (four K slices, measured: 1.6e-7 at 288 columns, 2.7e-7 at 896), 3 % for other inputs
@pytest.mark.parametrize("kind", ["f32", "f16"])
@pytest.mark.parametrize("n,rows,cols,bound", [(64, 256, 256, 1.53e-7), (200, 256, 288, 1.61e-7), (64, 896, 512, 2.08e-7),
                                               (200, 896, 896, 2.73e-7), (1024, 896, 896, 2.73e-7), (64, 512, 2048, 4.1e-7)])
def test_error_against_64_bits(dev, ref, kind, n, rows, cols, bound):
    rng = np.random.default_rng(n + cols)
    w = wg.float_random(kind, rows, cols, rng, scale=0.02)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    got = dev.matmulT(x, w).astype(np.float64)
    want = x.astype(np.float64) @ dequant_f32(ref, w).astype(np.float64).T
    assert np.linalg.norm(got - want) <= 1.03 * bound * np.linalg.norm(want)
