"""The matrix-core GEMM at the edges of its tiles and of its K loop, bit-exact on integer-valued
operands (every partial sum is an exact f32 integer times a power of two): rows around 16- and
32-row tiles and a workgroup's 64 and 128, tokens around 32, 64 and 128, and block counts around
its four-block groups, its unrolled round and the cut of a split K loop (16 blocks, between
super-blocks of 8)."""
import numpy as np
import pytest

from test_oracle_gemv_cpu import int_matrix
from ziglm_amd import bridge as B
from ziglm_amd import synth

pytestmark = pytest.mark.gpu

# columns: 1-5 blocks (odd counts load single blocks), 16-18 and 31 (split), 24 (uneven halves)
COLS = {B.Q4_0: (32, 96, 128, 160, 512, 544, 992), B.Q8_0: (32, 64, 160, 512, 544, 992), B.BF16: (32, 96, 512, 992),
        B.Q4_K: (256, 512, 768), B.Q6_K: (256, 512, 768)}
CASES = [(q, c) for q in COLS for c in COLS[q]]


def operands(qtype, rows, cols, batch, seed):
    raw, wd = int_matrix(qtype, rows, cols, seed=seed, scale_pow=-1)
    x = np.random.default_rng(seed).integers(-3, 4, (batch, cols)).astype(np.float32)
    return raw, x, x.astype(np.float64) @ wd.T


@pytest.mark.parametrize("qtype,cols", CASES)
@pytest.mark.parametrize("rows,batch", [(1, 129), (31, 128), (33, 160), (127, 161), (129, 257)])
def test_f32_edges(dev, qtype, cols, rows, batch):
    raw, x, exact = operands(qtype, rows, cols, batch, rows + cols + batch)
    assert np.all(np.abs(exact) < 2 ** 24)
    y = dev.alloc(batch * rows * 4)
    y.fill(0xAB)
    dev.gemmEx(qtype, dev.from_numpy(raw), None, B.F32, dev.from_numpy(x), B.F32, y, batch, rows, cols)
    np.testing.assert_array_equal(y.to_numpy((batch, rows), np.float32), exact.astype(np.float32))


@pytest.mark.parametrize("qtype,cols", CASES)
@pytest.mark.parametrize("rows,batch", [(1, 1), (15, 31), (17, 33), (65, 130)])
def test_bf16_and_pair_edges(dev, qtype, cols, rows, batch):
    """bf16 activations into f32 outputs (exact), and the gate.up pair (both matrices the same one)
    against the product's own GeGLU: the same sums, so at most bf16's rounding apart."""
    raw, x, exact = operands(qtype, rows, cols, batch, rows + cols + batch)
    w = dev.from_numpy(raw)
    xb = dev.from_numpy(synth.f32_to_bf16(x))
    y = dev.alloc(batch * rows * 4)
    y.fill(0xAB)
    dev.gemmEx(qtype, w, None, B.BF16, xb, B.F32, y, batch, rows, cols)
    got = y.to_numpy((batch, rows), np.float32)
    np.testing.assert_array_equal(got, exact.astype(np.float32))
    g = dev.alloc(batch * rows * 4)
    dev.geglu(y, y, g, batch * rows)
    want = g.to_numpy((batch, rows), np.float32)
    p = dev.alloc(batch * rows * 2)
    dev.gemmEx(qtype, w, w, B.BF16, xb, B.BF16, p, batch, rows, cols)
    pair = synth.bf16_to_f32(p.to_numpy((batch, rows), np.uint16))
    # gelu and its product are the same f32 expression in both, up to a fused rounding (2^-23)
    np.testing.assert_allclose(pair, want, rtol=2.0 ** -8, atol=1e-30)


def rows_of(qtype, rows, cols, seed, some=61):
    """A matrix of `some` different rows repeated, and which of them each row is."""
    raw, wd = int_matrix(qtype, some, cols, seed=seed, scale_pow=-1)
    pick = np.arange(rows) % some
    return np.ascontiguousarray(raw).reshape(some, -1)[pick], wd, pick


def product(dev, qtype, w, wu, x, x_dtype, batch, rows, cols):
    """One hip_gemm_ex product of f32 activations, as they are, split beforehand or rounded to bf16."""
    xd, y = dev.from_numpy(synth.f32_to_bf16(x) if x_dtype == B.BF16 else x), dev.alloc(batch * rows * 4)
    y.fill(0xAB)
    if x_dtype == B.F32_TERMS:
        planes = dev.alloc(3 * batch * cols * 2)
        dev.splitTerms(xd, planes, batch * cols)
        xd = planes
    dev.gemmEx(qtype, w, wu, x_dtype, xd, B.F32, y, batch, rows, cols)
    return y.to_numpy((batch, rows), np.float32)


# tokens x rows of a workgroup's tile (gemm.hip launch_qt), with ragged last tiles in both dimensions:
LARGE = [(B.Q4_0, 160, 1990),                       # 64 x 128 (single blocks)
         (B.Q4_0, 128, 1990), (B.Q4_0, 640, 1990),  # 64 x 256, a group of blocks and more than a round
         (B.Q4_0, 4096, 1510),                      # 64 x 256 in two K halves (792 tiles)
         (B.Q8_0, 128, 1990), (B.Q8_0, 640, 1990), (B.Q8_0, 160, 1990),  # 128 x 128, groups and single blocks
         (B.Q8_0, 640, 300),                        # 64 x 128: single blocks (f32), groups (planes)
         (B.BF16, 640, 1990), (B.BF16, 4096, 1510),  # 64 x 256 (f32) and 128 x 128 (planes), 128 x 128
         (B.Q4_K, 256, 1990), (B.Q4_K, 768, 900)]   # 64 x 128: min terms on the matrix cores


@pytest.mark.parametrize("x_dtype", [B.F32, B.F32_TERMS, B.BF16])
@pytest.mark.parametrize("qtype,cols,batch", LARGE)
def test_large_tiles(dev, qtype, cols, batch, x_dtype):
    rows = 8200
    raw, wd, pick = rows_of(qtype, rows, cols, cols)
    x = np.random.default_rng(cols).integers(-3, 4, (batch, cols)).astype(np.float32)
    exact = x.astype(np.float64) @ wd.T
    assert np.all(np.abs(exact) < 2 ** 24)
    got = product(dev, qtype, dev.from_numpy(raw), None, x, x_dtype, batch, rows, cols)
    np.testing.assert_array_equal(got, exact.astype(np.float32)[:, pick])


@pytest.mark.parametrize("x_dtype", [B.F32, B.F32_TERMS])
@pytest.mark.parametrize("qtype,cols", [(B.Q8_0, 640), (B.BF16, 640), (B.BF16, 4096), (B.Q4_K, 768)])
def test_large_pair_tiles(dev, qtype, cols, x_dtype):
    """The gate.up pair on the same large tiles against the two exact products' GeGLU."""
    rows, batch = 4100, 1990
    raw, wd, pick = rows_of(qtype, 2 * rows, cols, cols)
    x = np.random.default_rng(cols).integers(-3, 4, (batch, cols)).astype(np.float32) / 64
    exact = (x.astype(np.float64) @ wd.T).astype(np.float32)[:, pick]
    w, wu = dev.from_numpy(np.ascontiguousarray(raw[:rows])), dev.from_numpy(np.ascontiguousarray(raw[rows:]))
    got = product(dev, qtype, w, wu, x, x_dtype, batch, rows, cols)
    want = dev.alloc(batch * rows * 4)
    dev.geglu(dev.from_numpy(np.ascontiguousarray(exact[:, :rows])), dev.from_numpy(np.ascontiguousarray(exact[:, rows:])),
              want, batch * rows)
    # gelu and its product are the same f32 expression in both, up to a fused rounding (2^-23)
    np.testing.assert_allclose(got, want.to_numpy((batch, rows), np.float32), rtol=2.0 ** -22, atol=1e-30)


SHARES = [(q, c) for q in (B.Q4_0, B.Q8_0, B.BF16) for c in (992, 1024, 1056, 1248, 1280, 2816)]
SHARES += [(q, c) for q in (B.Q4_K, B.Q6_K) for c in (1024, 1280, 2816)]


@pytest.mark.parametrize("qtype,cols", SHARES)
def test_k_shares(dev, qtype, cols):
    """K in two shares per workgroup, and from 32 blocks in four (two of them added into zeroed y):
    31 blocks (16 + 15), 32, 33, 39 (16 + 8 + 8 + 7), 40 and 88, on few and on more tiles."""
    for rows, batch in ((33, 129), (1025, 700)):
        raw, x, exact = operands(qtype, rows, cols, batch, rows + cols)
        assert np.all(np.abs(exact) < 2 ** 24)
        w, xd, y = dev.from_numpy(raw), dev.from_numpy(x), dev.alloc(batch * rows * 4)
        for _ in range(2):
            y.fill(0xAB)
            dev.gemmEx(qtype, w, None, B.F32, xd, B.F32, y, batch, rows, cols)
            np.testing.assert_array_equal(y.to_numpy((batch, rows), np.float32), exact.astype(np.float32))


@pytest.mark.parametrize("qtype,cols", [(B.Q6_K, 4352), (B.Q4_K, 1280), (B.Q8_0, 1056), (B.Q4_0, 4224)])
def test_teams_of_planes(dev, qtype, cols):
    """The two-team kernel on pre-split activations (Q6_K from 4096 columns)."""
    rows, batch = 100, 150
    raw, x, exact = operands(qtype, rows, cols, batch, cols)
    got = product(dev, qtype, dev.from_numpy(raw), None, x, B.F32_TERMS, batch, rows, cols)
    np.testing.assert_array_equal(got, exact.astype(np.float32))
