"""Small-batch products (k_gemm_skinny, reached by hip_gemm for the batches and shapes of its launch
rule) bit-exact on integer-valued operands, where every partial sum is an exact f32 integer times
a power of two: batches around the 8, 16 and 32 tokens of its operand packings and one past them,
ragged row tiles, block counts that share out unevenly over the waves and the two K halves. A
second call gives the same bits (the halves are two addends)."""
import numpy as np
import pytest

from test_oracle_gemv_cpu import int_matrix, random_matrix
from ziglm_amd import bridge as B

pytestmark = pytest.mark.gpu

GROUPED = (B.Q4_0, B.Q4_K, B.Q6_K)


def check(dev, qtype, rows, cols, batch):
    raw, wd = int_matrix(qtype, rows, cols, seed=rows + cols + batch, scale_pow=-1)
    x = np.random.default_rng(batch).integers(-2, 3, (batch, cols)).astype(np.float32)
    exact = x.astype(np.float64) @ wd.T
    assert np.all(np.abs(x).astype(np.float64) @ np.abs(wd).T < 2 ** 23)
    w, xd = dev.from_numpy(raw), dev.from_numpy(x)
    got = []
    for _ in range(2):
        y = dev.alloc(batch * rows * 4)
        y.fill(0xAB)
        dev.gemm(qtype, w, xd, y, batch, rows, cols)
        got.append(y.to_numpy((batch, rows), np.float32))
    np.testing.assert_array_equal(got[0], exact.astype(np.float32), err_msg=f"qtype={qtype} {rows}x{cols} b={batch}")
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


# two K halves: 4096 columns (32 groups of four blocks), 4352 (34: 17 a half, uneven over the waves)
@pytest.mark.parametrize("qtype,batches", [(B.Q4_0, (9, 16, 17, 24, 33, 128)), (B.Q4_K, (5, 8, 9, 16, 17, 24, 33, 128)),
                                           (B.Q6_K, (5, 8, 9, 16, 17, 31, 33, 128)), (B.Q8_0, (9, 16, 17, 33, 128)),
                                           (B.BF16, (64, 96, 128))])
@pytest.mark.parametrize("rows,cols", [(1, 4096), (33, 4352), (95, 4096)])
def test_deep(dev, qtype, batches, rows, cols):
    for batch in batches:
        check(dev, qtype, rows, cols, batch)


# many rows, a group of blocks or two of a wave's share
@pytest.mark.parametrize("qtype", GROUPED)
@pytest.mark.parametrize("rows,cols,batches", [(8193, 256, (3, 7, 8, 9, 15, 17, 32)), (5121, 768, (3, 16, 33, 63)),
                                               (2561, 256, (10, 17, 65, 127))])
def test_wide(dev, qtype, rows, cols, batches):
    for batch in batches:
        check(dev, qtype, rows, cols, batch)


# Two row tiles per wave (RT = 2), by operand packing (P = 4, 2, 1 for up to 8, 16, 32 tokens) and K halves;
# the launch rule gives: shallow rows RT = 2 where 64-row tiles x token tiles reach 160 and P < 4; deep ones
# where 32-row tiles x token tiles reach 160, in two halves where 64-row ones do not.
@pytest.mark.parametrize("qtype,rows,cols,batches",
                         [(q, 10241, 256, (9, 16, 17, 32)) for q in GROUPED] +            # P = 2, 1, no halves
                         [(q, 5153, 4096, (5, 8, 9, 16)) for q in GROUPED] +              # P = 4, 2, no halves
                         [(B.Q8_0, 5153, 4096, (9, 16, 17))] +                            # P = 2, 1, no halves
                         [(q, 2561, 4096, (33, 64)) for q in (*GROUPED, B.Q8_0)] +        # P = 1, two halves
                         [(B.BF16, 2561, 4096, (65, 96)), (B.BF16, 5153, 4352, (17, 32))])  # P = 1, halves and not
def test_two_row_tiles(dev, qtype, rows, cols, batches):
    for batch in batches:
        check(dev, qtype, rows, cols, batch)


@pytest.mark.parametrize("cols", [128, 384, 640])
def test_single_groups(dev, cols):
    for batch in (2, 12, 30):
        check(dev, B.Q4_0, 8192, cols, batch)


def test_infinite_activation_stays_in_its_token(dev):
    """Packed tokens share an operand's rows with their own other columns only."""
    rows, cols = 2048, 4096
    raw, wd = int_matrix(B.Q4_0, rows, cols, seed=1, scale_pow=-1)
    for batch in (6, 12, 20):
        x = np.random.default_rng(batch).integers(-2, 3, (batch, cols)).astype(np.float32)
        exact = (x.astype(np.float64) @ wd.T).astype(np.float32)
        x[3, 1000] = np.inf
        y = dev.alloc(batch * rows * 4)
        dev.gemm(B.Q4_0, dev.from_numpy(raw), dev.from_numpy(x), y, batch, rows, cols)
        got = y.to_numpy((batch, rows), np.float32)
        keep = np.arange(batch) != 3
        np.testing.assert_array_equal(got[keep], exact[keep])
        assert not np.any(np.isfinite(got[3]) & (got[3] == exact[3]))


# columns past 5120 (10240) and tokens below: products that the vector kernels can also take
@pytest.mark.parametrize("qtype,rows,cols,batch", [(B.Q6_K, 8192, 256, 3), (B.Q6_K, 8192, 256, 7), (B.Q6_K, 40, 4352, 6),
                                                   (B.Q8_0, 40, 5376, 9), (B.BF16, 2560, 10752, 17), (B.Q4_0, 40, 4352, 9),
                                                   (B.Q4_K, 40, 4352, 20), (B.Q6_K, 40, 4352, 33),
                                                   (B.Q8_0, 8192, 10496, 17), (B.BF16, 8192, 10496, 24),
                                                   (B.Q6_K, 8192, 10496, 33)])
def test_infinite_activations_give_what_f32_gives(dev, qtype, rows, cols, batch):
    """An infinite activation times a weight is an infinity of the product's sign (NaN for a zero
    weight, or where infinities of both signs meet), as in f32 arithmetic on the values; a value past
    bf16's largest is finite; the other tokens keep their exact sums."""
    some = min(rows, 64)  # different rows, repeated
    raw, wd = int_matrix(qtype, some, cols, seed=rows + cols, scale_pow=-1)
    raw, wd = np.tile(raw, (rows // some, 1)), np.tile(wd, (rows // some, 1))
    x = np.random.default_rng(batch).integers(-2, 3, (batch, cols)).astype(np.float32)
    keep = np.arange(3, batch)
    exact = x.astype(np.float64) @ wd.T
    x[0, cols - 7] = np.inf
    x[1, 5] = -np.inf
    x[1, cols // 2] = np.inf
    x[2] = 0
    x[2, 77] = np.float32(3.4e38)  # (bf16 rounds it to infinity); with f32 sums: w * x
    with np.errstate(invalid="ignore"):
        want = np.stack([np.inf * wd[:, cols - 7], -np.inf * wd[:, 5] + np.inf * wd[:, cols // 2]]).astype(np.float32)
    with np.errstate(over="ignore"):
        big = (wd[:, 77] * np.float64(x[2, 77])).astype(np.float32)
    y = dev.alloc(batch * rows * 4)
    dev.gemm(qtype, dev.from_numpy(raw), dev.from_numpy(x), y, batch, rows, cols)
    got = y.to_numpy((batch, rows), np.float32)
    np.testing.assert_array_equal(got[:2], want)
    np.testing.assert_array_equal(got[2], big)
    np.testing.assert_array_equal(got[keep], exact[keep].astype(np.float32))


@pytest.mark.parametrize("qtype,rows,cols,batches",
                         [(q, 40, 4352, (9, 20, 64, 96, 128)) for q in GROUPED] + [(q, 5121, 512, (5, 16, 40)) for q in GROUPED] +
                         [(B.Q8_0, 40, 4352, (9, 20, 64, 96, 128)), (B.BF16, 40, 4352, (64, 96, 128))] +
                         [(q, 2561, 4096, (65, 96)) for q in (*GROUPED, B.Q8_0, B.BF16)])
def test_split_activations_give_the_same_bits(dev, qtype, rows, cols, batches):
    """Activations split beforehand (F32_TERMS): hip_gemm's bits on the f32 activations wherever that
    runs this kernel."""
    raw, _ = int_matrix(qtype, rows, cols, seed=rows + cols, scale_pow=-1)
    w = dev.from_numpy(raw)
    for batch in batches:
        x = np.random.default_rng(batch).standard_normal((batch, cols)).astype(np.float32)
        xd, planes = dev.from_numpy(x), dev.alloc(3 * batch * cols * 2)
        dev.splitTerms(xd, planes, batch * cols)
        got = []
        for x_dtype, xs in ((B.F32, xd), (B.F32_TERMS, planes)):
            y = dev.alloc(batch * rows * 4)
            y.fill(0xAB)
            dev.gemmEx(qtype, w, None, x_dtype, xs, B.F32, y, batch, rows, cols)
            got.append(y.to_numpy((batch, rows), np.uint32))
        np.testing.assert_array_equal(got[0], got[1], err_msg=f"batch {batch}")


# the routes of few tokens with the longest sums: wide products on the GEMM (FINE tiles, in one and in two
# teams), deep ones on k_gemm_skinny
@pytest.mark.parametrize("qtype,rows,cols,batch", [
    (B.BF16, 8192, 2560, 33), (B.BF16, 8192, 10496, 17), (B.Q6_K, 8192, 2560, 33), (B.Q4_K, 8192, 10496, 48),
    (B.Q4_0, 8192, 10496, 80), (B.Q8_0, 8192, 10496, 80), (B.BF16, 2560, 21504, 17), (B.Q4_K, 192, 21504, 17),
    (B.Q4_K, 192, 21504, 64), (B.Q6_K, 192, 21504, 33), (B.Q4_0, 192, 21504, 48)])
def test_error_does_not_grow_with_depth(dev, qtype, rows, cols, batch):
    """A result is a total of short sums: its error (2-norms over all results) is that of a few f32
    roundings (2^-24, of which a random one costs 0.58 of the size rounded) at the result's size,
    whatever the depth: those of a block's products, about 1, of a chain of 8 or 16 block sums, about
    1.3, and of the result; 2.5 in all. One chain over 10496 columns is 3 (block sums) to 14 (single
    products, BF16) of them off."""
    some = 64  # different rows, repeated
    raw, wd = random_matrix(qtype, some, cols, seed=cols + batch)
    w = dev.from_numpy(np.tile(np.ascontiguousarray(raw).reshape(some, -1), (rows // some, 1)))
    x = np.random.default_rng(batch).standard_normal((batch, cols)).astype(np.float32)
    exact = x.astype(np.float64) @ wd.T
    y = dev.alloc(batch * rows * 4)
    dev.gemm(qtype, w, dev.from_numpy(x), y, batch, rows, cols)
    got = y.to_numpy((batch, rows // some, some), np.float32).astype(np.float64)
    err = np.linalg.norm(got - exact[:, None]) / (np.linalg.norm(exact) * (rows // some) ** 0.5)
    assert err <= 2.5 * 2.0 ** -24, err * 2 ** 24
