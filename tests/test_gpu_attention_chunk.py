"""Causal chunks on the matrix cores (k_attn_chunk, reached by hip_attention_batched for the larger
chunks) against float64 within the f32 attention bound: head sizes and head groups, ragged last
tiles of 16 query rows and 16-key blocks, windows and soft-cap, positions past the cache, and
infinite or NaN rows that only some of a tile's tokens see."""
import numpy as np
import pytest

from attn_ref import attention_f64
from ziglm_amd import synth

pytestmark = pytest.mark.gpu


def run(dev, q, kc, vc, layer, pos, max_seq, nh, nkv, d, scale, cap, window):
    T = q.shape[0]
    out = dev.alloc(T * nh * d * 4)
    out.fill(0xAB)
    dev.attentionBatched(dev.from_numpy(q), dev.from_numpy(kc), dev.from_numpy(vc), out, layer, pos, T, max_seq, nh, nkv,
                         d, nkv * d, scale, cap, window)
    return out.to_numpy((T, nh * d), np.float32)


def data(seed, T, nh, nkv, d, rows):
    return (synth.normal_f32(seed, "q", (T, nh * d), 0, 1), synth.normal_f32(seed, "k", (rows, nkv * d), 0, 1),
            synth.normal_f32(seed, "v", (rows, nkv * d), 0, 1))


# every shape launches the chunk kernel: 128 workgroups, or 8 heads per kv head and 16 rows of kv heads
@pytest.mark.parametrize("nh,nkv,d,T,pos", [(16, 16, 64, 129, 0), (8, 4, 256, 257, 0), (8, 4, 256, 260, 37),
                                            (8, 2, 128, 257, 30), (8, 1, 256, 17, 0), (8, 1, 256, 16, 250),
                                            (8, 1, 64, 31, 15), (16, 2, 256, 9, 100), (32, 16, 128, 65, 100)])
@pytest.mark.parametrize("cap,window", [(0.0, 0), (20.0, 0), (0.0, 33), (0.0, 16)])
def test_against_f64(dev, nh, nkv, d, T, pos, cap, window):
    max_seq, layer, scale = 320, 1, d ** -0.5
    q, kc, vc = data(nh + d + T, T, nh, nkv, d, 2 * max_seq)
    got = run(dev, q, kc, vc, layer, pos, max_seq, nh, nkv, d, scale, cap, window)
    for b in sorted({0, 1, 7, T // 2, T - 2, T - 1}):
        out, tol = attention_f64(q[b], kc, vc, layer * max_seq, pos + b, nh, nkv, d, scale, cap, window)
        assert np.all(np.abs(got[b] - out) <= tol), f"token {b}: {np.max(np.abs(got[b] - out) / tol)} of the bound"


def test_rows_past_the_cache_give_zeros(dev):
    nh, nkv, d, T, pos, max_seq = 8, 1, 128, 40, 90, 100
    q, kc, vc = data(3, T, nh, nkv, d, max_seq)
    got = run(dev, q, kc, vc, 0, pos, max_seq, nh, nkv, d, 0.1, 0.0, 0)
    assert np.all(got[10:] == 0.0)
    for b in (0, 9):
        out, tol = attention_f64(q[b], kc, vc, 0, pos + b, nh, nkv, d, 0.1)
        assert np.all(np.abs(got[b] - out) <= tol)


@pytest.mark.parametrize("window", [0, 24])
def test_values_that_only_some_tokens_see(dev, window):
    """Non-finite V rows (and K rows) of a token's successors, of rows before its window and of rows
    never written must not reach it; tokens that see an infinite V row show it."""
    nh, nkv, d, T, pos, max_seq = 8, 4, 256, 256, 0, 300
    q, kc, vc = data(4, T, nh, nkv, d, max_seq)
    bad = 131
    vc[bad] = np.inf
    kc[bad + 1] = np.nan
    vc[T:] = np.nan
    kc[T:] = np.nan
    got = run(dev, q, kc, vc, 0, pos, max_seq, nh, nkv, d, 0.05, 0.0, window)
    fine = [b for b in (0, 64, 128, 129, 130) + ((bad + 1 + 24, bad + 40, 255) if window else ())]
    for b in fine:
        out, tol = attention_f64(q[b], kc, vc, 0, b, nh, nkv, d, 0.05, 0.0, window)
        assert np.all(np.abs(got[b] - out) <= tol), b
    assert np.all(np.isinf(got[bad])) and np.all(np.isnan(got[bad + 1]))
