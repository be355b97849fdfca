// Prefill-sized GEMM on the matrix cores (gfx950 MFMA): Y[b][r] = sum_c W[r][c] * X[b][c] for
// Q4_0, Q8_0, F16, BF16 and F32 weights and f32 or bf16 activations (replaces
// cuda_bridge.cu:1179-1445, k_gemm_q4_0 / k_gemm_q8_0 / k_gemm_f16, used by ziglm's batched
// prefill at cuda_model.zig:1264-1383), with ziglm's CPU arithmetic (math.zig:440-616): weights
// dequantised exactly, activations kept in full, f32 sums. Outputs are f32 or bf16, and the
// gate.up pair of a GeGLU FFN runs as one launch that writes gelu(gate) * up (the reference's
// two prefill GEMMs and k_geglu, cuda_model.zig:1372-1387, cuda_bridge.cu:2247-2269): a tile holds
// its output rows of both matrices, an output's two sums meet by a lane shuffle (in k_gemm_dense
// through the LDS), and the gate and up outputs never reach HBM.
//
// Exact operands on a bf16 matrix core. The MFMA multiplies bf16 operands exactly into f32
// accumulators, so every operand is written as a short sum of bf16 terms that is exact or
// nearly so:
//   x (f32) = h + m + l, h = bf16(x), m = bf16(x - h), l = bf16(x - h - m): the three terms
//     carry x's 24 significant bits (the remainder is below 2^-24 |x|); bf16 activations are
//     one exact term (a third of the MFMAs and no split);
//   Q4_0 / Q8_0 quants (integers -8..7 / -127..127) are exact in bf16; the block's f16 scale d
//     multiplies the block's f32 partial sum, sum_k q_k x_k, afterwards (the CPU's
//     (q * d) * x products are all exact-integer-times-f16 values, so applying d after the sum
//     changes only the f32 rounding);
//   BF16 weights are exact; F16 weights (11 significant bits) are hi + lo, both exact in bf16;
//   F32 weights are split like x;
//   Q4_K (math.zig:440-496): a 32-column block is one sub-block j of a 256-column
//     super-block, value q * (d * sc_j) - dmin * m_j with q in 0..15. The codes enter as q - 8 (exact
//     in bf16): the block's partial sum_k (q_k - 8) x_k is scaled by A_j = d * sc_j and the min term
//     (dmin * m_j - 8 A_j) * sum_k x_k subtracted, with the per-token sums of x formed while staging x.
//     (With q itself the two parts of a value near the middle of the codes cancel and leave their
//     rounding: 10240 x 2560, 33 tokens, 2.4e-7 off against 1.7e-7.)
//   Q6_K (math.zig:556-616): value d * sc * (u - 32) with an int8 scale per 16 columns;
//     u - 32 is exact in bf16 and d * sc (exact in f32) scales each K = 16 half's partial
//     sum.
// The products of the terms are accumulated down to relative weight 2^-16 (h*w_hi, m*w_hi,
// l*w_hi, and for F16 / F32 the cross terms of the same size); the dropped ones are below
// 2^-24 of a product, so a dot product lies within the f32 rounding of the sum, like the
// decode GEMV's.
//
// Tiling (k_gemm_mfma: quantised and BF16 weights). A workgroup of 4 waves owns 32 WT tokens x 128 RT rows; a wave computes
// all of the tokens for its own 32 RT rows, as WT x RT tiles of v_mfma_f32_32x32x16_bf16 (tokens
// on the A side, so a lane's accumulators are one weight row: the block scale is one value per
// lane and tile, and stores of 32 lanes are 128 contiguous bytes of a token's output row). No two
// waves share a weight row, so a lane loads the codes of its row straight into registers in the
// B-operand layout and converts them there, once per workgroup, and only the activations go
// through the LDS: a step's LDS reads are the activation terms alone (staged through the LDS
// the weights were half of them, and their loop ran at 2-3 times the LDS traffic of this one).
// With GE a tile's 32 columns are 16 gate rows and the same 16 up rows, so gelu(gate) * up takes
// one lane shuffle.
// The K loop takes one 32-column block per step. The LDS holds block k as bf16 terms (rows
// permuted against bank conflicts, lds_chunk) in one of two buffers while the registers hold the
// raw bytes of the next blocks (more activation blocks ahead for the smaller tiles, whose steps
// are shorter than a memory round trip); block k + 1 is converted into the other buffer during
// block k's MFMAs, so a step takes one barrier. Activations load through a range-checked resource
// (tokens past the batch read zeros); weight rows past the end are the last row again, and nothing
// of them is stored. F16 and F32 weights are staged through the LDS instead (k_gemm_dense), and a
// few tokens take k_gemm_skinny.
#include "zl_common.h"
#include "zl_host.h"

namespace zl {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kKB = 32;       // columns per K step (one Q4_0 / Q8_0 block)
// A token's LDS row is the block's 32 columns of one term: 64 bytes, its four 16-byte chunks
// permuted by the row so that neither the reads (8 rows' same chunk a cycle) nor the writes (two
// whole rows a cycle) meet on a bank (counters: no conflict cycles; rows padded to 80 bytes had 32
// million in a 10240 x 2560 x 2048 product).
constexpr int kLdsRow = 32;
__device__ __forceinline__ int lds_chunk(int row, int c) { return row * kLdsRow + ((c ^ (row >> 2)) & 3) * 8; }

// Weight terms (bf16 planes) per type: Q4_0 / Q8_0 quants are exact in bf16 and their block
// scale multiplies each 32-column partial sum; BF16 weights are exact; F16 weights are two
// exact terms, F32 three. (Q4_0 products (u - 8) * d are also exact in two bf16 terms, which
// saves the per-block scale products at twice the MFMAs: measured slower, with f32
// activations 333 -> 438 us and with bf16 ones 191 -> 213 us for 10240 x 2560 x 2048.)
// Q6_K: its scale per 16-column half multiplies each K = 16 MFMA half's partial sum, the
// quants u - 32 one exact term. (sc * (u - 32) as two exact terms with one scale d per step
// instead: 5 term products, 10240 x 2560 x 2048 with f32 activations 555 against 453 us.)
// Q4_0 and Q8_0 rows whose block count is no multiple of four (see WGrp).
constexpr int kQ4_0Odd = 0x100 + HIP_BRIDGE_Q4_0, kQ8_0Odd = 0x100 + HIP_BRIDGE_Q8_0;
template <int QT>
constexpr bool is_q4_0() {
    return QT == HIP_BRIDGE_Q4_0 || QT == kQ4_0Odd;
}
template <int QT>
constexpr int w_terms() {
    return QT == HIP_BRIDGE_F16 ? 2 : QT == HIP_BRIDGE_F32 ? 3 : 1;
}
template <int QT>
constexpr bool w_scaled() {
    return is_q4_0<QT>() || QT == HIP_BRIDGE_Q8_0 || QT == kQ8_0Odd || QT == HIP_BRIDGE_Q4_K || QT == HIP_BRIDGE_Q6_K;
}
// bf16 (RNE) of two floats and the f32 values of the result.
__device__ __forceinline__ uint32_t bf16_pair(float a, float b, float& ra, float& rb) {
    const uint32_t p = pack_bf16x2(a, b);
    ra = bf16_lo(p);
    rb = bf16_hi(p);
    return p;
}

// x0, x1 -> three packed bf16 pairs (h, m, l).
__device__ __forceinline__ void split3(float x0, float x1, uint32_t* t) {
    float a, b;
    t[0] = bf16_pair(x0, x1, a, b);
    x0 -= a;
    x1 -= b;
    t[1] = bf16_pair(x0, x1, a, b);
    t[2] = pack_bf16x2(x0 - a, x1 - b);
}
// x0, x1 -> two packed bf16 pairs (hi, lo).
__device__ __forceinline__ void split2(float x0, float x1, uint32_t* t) {
    float a, b;
    t[0] = bf16_pair(x0, x1, a, b);
    t[1] = pack_bf16x2(x0 - a, x1 - b);
}

struct GemmArgs {
    const unsigned char* w;
    const unsigned char* wu;  // GeGLU: the up matrix (same type and shape as w)
    const void* x;            // f32 or bf16 [batch][cols]
    void* y;                  // f32 or bf16 [batch][rows]
    int64_t row_bytes;
    int rows, cols, batch;
    int y_bf16;
};

__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}
// Two f32 values that bf16 holds exactly -> a packed pair (the high halves).
__device__ __forceinline__ uint32_t pack_exact(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// The signed bytes of two words as 8 bf16 values, exact.
__device__ __forceinline__ bf16x8 bytes_s(uint32_t v, uint32_t w) {
    return __builtin_bit_cast(bf16x8, u32x4{pack_exact((float)(int8_t)v, (float)(int8_t)(v >> 8)),
                                            pack_exact((float)(int8_t)(v >> 16), (float)(int8_t)(v >> 24)),
                                            pack_exact((float)(int8_t)w, (float)(int8_t)(w >> 8)),
                                            pack_exact((float)(int8_t)(w >> 16), (float)(int8_t)(w >> 24))});
}
// a = {a of lanes 0-31, b of lanes 0-31}, b = {a of lanes 32-63, b of lanes 32-63}
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// A lane's share of a weight row: the 16 columns of each 32-column block that its half h =
// lane / 32 multiplies in the block's two MFMAs. wk(s, h) is the first of the 8 columns that
// half h takes in MFMA s; the activations are read from the LDS in the same order. Q4_0 holds
// columns c and c + 16 in one byte and Q6_K has a scale per 16 columns, so there MFMA s covers
// columns 16 s .. + 16; elsewhere a half takes 16 consecutive columns.
template <int QT>
__device__ __forceinline__ constexpr int wk(int s, int h) {
    return (is_q4_0<QT>() || QT == HIP_BRIDGE_Q6_K) ? 16 * s + 8 * h : 16 * h + 8 * s;
}

// 32-, 64- and 128-bit loads from 2-byte aligned addresses (block codes sit at offset 2 of 18-
// and 34-byte blocks; a 210-byte super-block may start anywhere), which gfx950 serves unaligned.
typedef uint32_t u32_a2 __attribute__((aligned(2)));
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
struct WSrc {  // the lane's weight row; offsets: the lane's, and a wave-uniform one
    const unsigned char* row;
    __device__ __forceinline__ u32x4 b128(uint32_t o, uint32_t so) const { return *(const u32x4_a2*)(row + so + o); }
    __device__ __forceinline__ u32x2 b64(uint32_t o, uint32_t so) const { return *(const u32x2_a2*)(row + so + o); }
    __device__ __forceinline__ uint32_t b32(uint32_t o, uint32_t so) const { return *(const u32_a2*)(row + so + o); }
    __device__ __forceinline__ uint32_t b16(uint32_t o, uint32_t so) const { return *(const uint16_t*)(row + so + o); }
};

// Raw bytes of G consecutive 32-column blocks (blocks kb .. kb + G, kb a multiple of G from the
// first block of the row): load() issues the loads, open() rearranges them once they are here,
// ops<S>(u) gives the B operands of block kb + u's MFMA S, and scale() the block's scale(s)
// (one per MFMA for Q6_K) and min factor (Q4_K). A lane's loads are few and wide: its row lies
// alone in its cache line, so an instruction costs as many cache accesses as it has rows
// whatever its width (Q8_0 with two loads per block: 2560 x 10240 at 700 tokens, bf16 activations,
// 285 us, in groups 159).
// Signed 4- and 6-bit codes are taken as 16 (u - 8) and 4 (u - 32), the signed bytes that a
// shift and a sign flip leave, so each costs one conversion; the power of two goes into the
// scale.
template <int QT>
struct WGrp;
template <>
struct WGrp<HIP_BRIDGE_Q4_0> {
    // Half h loads blocks 2 h and 2 h + 1 (36 bytes: f16 d, 16 code bytes, twice); open()
    // swaps code bytes between the halves so that each has bytes [8 h, + 8) of all four.
    static constexpr int G = 4;
    u32x4 a, b;
    uint32_t c;
    __device__ __forceinline__ void load(const WSrc& s, int kb, int h) {
        const uint32_t o = 36u * h, so = 18u * (uint32_t)kb;
        a = s.b128(o, so);
        b = s.b128(o + 16, so);
        c = s.b32(o + 32, so);
    }
    __device__ __forceinline__ void open() {
        // codes of the first block: the halfwords from byte 2 on; the second starts at byte 18
        uint32_t q0 = __builtin_amdgcn_alignbit(a.y, a.x, 16), q1 = __builtin_amdgcn_alignbit(a.z, a.y, 16);
        uint32_t q2 = __builtin_amdgcn_alignbit(a.w, a.z, 16), q3 = __builtin_amdgcn_alignbit(b.x, a.w, 16);
        uint32_t d0 = __builtin_amdgcn_perm(b.x, a.x, 0x07060100u), d1 = d0;  // both blocks' d
        swap_halves(q0, q2);
        swap_halves(q1, q3);
        uint32_t p0 = b.y, p1 = b.z, p2 = b.w, p3 = c;
        swap_halves(p0, p2);
        swap_halves(p1, p3);
        swap_halves(d0, d1);
        q[0][0] = q0 ^ 0x88888888u, q[0][1] = q1 ^ 0x88888888u;
        q[1][0] = p0 ^ 0x88888888u, q[1][1] = p1 ^ 0x88888888u;
        q[2][0] = q2 ^ 0x88888888u, q[2][1] = q3 ^ 0x88888888u;
        q[3][0] = p2 ^ 0x88888888u, q[3][1] = p3 ^ 0x88888888u;
        d[0] = d0, d[1] = d1;
    }
    uint32_t q[4][2], d[2];
    template <int S>
    __device__ __forceinline__ void ops(int u, bf16x8 (&o)[1]) const {
        // byte j: low nibble = element j, high nibble = element j + 16
        if constexpr (S == 0) o[0] = bytes_s((q[u][0] << 4) & 0xf0f0f0f0u, (q[u][1] << 4) & 0xf0f0f0f0u);
        else o[0] = bytes_s(q[u][0] & 0xf0f0f0f0u, q[u][1] & 0xf0f0f0f0u);
    }
    __device__ __forceinline__ void scale(int u, int, float (&dv)[2], float&) const {
        dv[0] = f16_bits_to_f32(u & 1 ? d[u >> 1] >> 16 : d[u >> 1] & 0xffffu) * 0.0625f;
    }
};
template <>
struct WGrp<kQ4_0Odd> {
    // Any block count: one block at a time (a group's loads would reach past the row).
    static constexpr int G = 1;
    u32x2 q;
    uint32_t d;
    __device__ __forceinline__ void load(const WSrc& s, int kb, int h) {
        const uint32_t so = 18u * (uint32_t)kb;
        d = s.b16(0, so);
        q = s.b64(2 + 8u * h, so);
    }
    __device__ __forceinline__ void open() {}
    template <int S>
    __device__ __forceinline__ void ops(int, bf16x8 (&o)[1]) const {
        const uint32_t x = q.x ^ 0x88888888u, y = q.y ^ 0x88888888u;
        if constexpr (S == 0) o[0] = bytes_s((x << 4) & 0xf0f0f0f0u, (y << 4) & 0xf0f0f0f0u);
        else o[0] = bytes_s(x & 0xf0f0f0f0u, y & 0xf0f0f0f0u);
    }
    __device__ __forceinline__ void scale(int, int, float (&dv)[2], float&) const {
        dv[0] = f16_bits_to_f32(d) * 0.0625f;
    }
};
template <>
struct WGrp<HIP_BRIDGE_Q8_0> {
    // Half h loads blocks 2 h and 2 h + 1 (68 bytes: f16 d, 32 codes, twice); open() swaps codes
    // between the halves so that each has columns [16 h, + 16) of all four.
    static constexpr int G = 4;
    u32x4 a[4];
    uint32_t e;
    __device__ __forceinline__ void load(const WSrc& s, int kb, int h) {
        const uint32_t o = 68u * h, so = 34u * (uint32_t)kb;
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = s.b128(o + 16u * i, so);
        e = s.b32(o + 64, so);
    }
    __device__ __forceinline__ void open() {
        auto w = [&](int i) { return i < 16 ? a[i >> 2][i & 3] : e; };
        // the first block's codes: the halfwords from byte 2 on; the second's start at byte 36
        uint32_t d0 = __builtin_amdgcn_perm(w(8), w(0), 0x07060100u), d1 = d0;  // both blocks' d
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t x = __builtin_amdgcn_alignbit(w(i + 1), w(i), 16), y = __builtin_amdgcn_alignbit(w(i + 5), w(i + 4), 16);
            swap_halves(x, y);
            q[0][i] = x, q[2][i] = y;
            x = w(9 + i), y = w(13 + i);
            swap_halves(x, y);
            q[1][i] = x, q[3][i] = y;
        }
        swap_halves(d0, d1);
        d[0] = d0, d[1] = d1;
    }
    uint32_t q[4][4], d[2];
    template <int S>
    __device__ __forceinline__ void ops(int u, bf16x8 (&o)[1]) const {
        o[0] = bytes_s(q[u][2 * S], q[u][2 * S + 1]);
    }
    __device__ __forceinline__ void scale(int u, int, float (&dv)[2], float&) const {
        dv[0] = f16_bits_to_f32(u & 1 ? d[u >> 1] >> 16 : d[u >> 1] & 0xffffu);
    }
};
template <>
struct WGrp<kQ8_0Odd> {
    static constexpr int G = 1;
    u32x4 q;
    uint32_t d;
    __device__ __forceinline__ void load(const WSrc& s, int kb, int h) {
        const uint32_t so = 34u * (uint32_t)kb;
        d = s.b16(0, so);
        q = s.b128(2 + 16u * h, so);
    }
    __device__ __forceinline__ void open() {}
    template <int S>
    __device__ __forceinline__ void ops(int, bf16x8 (&o)[1]) const {
        o[0] = bytes_s(q[2 * S], q[2 * S + 1]);
    }
    __device__ __forceinline__ void scale(int, int, float (&dv)[2], float&) const { dv[0] = f16_bits_to_f32(d); }
};
template <>
struct WGrp<HIP_BRIDGE_Q4_K> {
    // Half of a 144-byte super-block {f16 d, f16 dmin, scales[12], qs[128]} (types.zig:170-175):
    // sub-block j's 32 values are the low (j even) or high (j odd) nibbles of
    // qs[32 (j / 2) .. + 32)
    static constexpr int G = 4;
    u32x4 hd, q[2];
    __device__ __forceinline__ void load(const WSrc& s, int kb, int h) {
        const uint32_t so = 144u * (uint32_t)(kb >> 3), qo = 16u + 16u * h, sq = so + 16u * (uint32_t)(kb & 4);
        hd = s.b128(0, so);
        q[0] = s.b128(qo, sq);
        q[1] = s.b128(qo + 32, sq);
    }
    __device__ __forceinline__ void open() {}
    template <int S>
    __device__ __forceinline__ void ops(int u, bf16x8 (&o)[1]) const {
        const int sh = u & 1 ? 0 : 4;
        const uint32_t x = (q[u >> 1][2 * S] << sh) & 0xf0f0f0f0u, y = (q[u >> 1][2 * S + 1] << sh) & 0xf0f0f0f0u;
        o[0] = bytes_s(x ^ 0x80808080u, y ^ 0x80808080u);
    }
    __device__ __forceinline__ void scale(int u, int kb, float (&dv)[2], float& mn) const {
        // 6-bit scale and min of sub-block j (quant.zig:285-290): j < 4: scales[j] & 63 and
        // scales[j + 4] & 63; else the low / high nibble of scales[j + 4] with the top two
        // bits of scales[j - 4] / scales[j] above them
        const uint32_t b = 8u * (uint32_t)u;
        const uint32_t s0 = (hd.y >> b) & 0xffu, s1 = (hd.z >> b) & 0xffu, s2 = (hd.w >> b) & 0xffu;
        const uint32_t hi = 0u - (((uint32_t)kb >> 2) & 1u);  // j >= 4: all ones (masks: no branch)
        const uint32_t sc = (s0 & 63u & ~hi) | (((s2 & 15u) | ((s0 >> 6) << 4)) & hi);
        const uint32_t m = (s1 & 63u & ~hi) | (((s2 >> 4) | ((s1 >> 6) << 4)) & hi);
        const float A = f16_bits_to_f32(hd.x & 0xffffu) * (float)sc;
        dv[0] = A * 0.0625f;
        mn = fmaf(-8.0f, A, f16_bits_to_f32(hd.x >> 16) * (float)m);
    }
};
template <>
struct WGrp<HIP_BRIDGE_Q6_K> {
    // Half n of a 210-byte super-block {ql[128], qh[64], int8 scales[16], f16 d}
    // (types.zig:187-192): block t covers values [128 n + 32 t, + 32), value l of it takes the
    // low (t < 2) or high nibble of ql[64 n + 32 (t & 1) + l], bits 2t, 2t + 1 of qh[32 n + l]
    // and scale sc[8 n + l / 16 + 2 t] (quant.zig:357-385). Half h loads l in [16 h, + 16);
    // open() swaps 8 bytes so that MFMA s's words hold l in [16 s + 8 h, + 8).
    static constexpr int G = 4;
    u32x4 ql[2], qh;
    u32x2 sc;
    uint32_t d;
    __device__ __forceinline__ void load(const WSrc& s, int kb, int h) {
        const uint32_t so = 210u * (uint32_t)(kb >> 3), n = (uint32_t)(kb >> 2) & 1u, ho = 16u * h;
        ql[0] = s.b128(ho, so + 64 * n);
        ql[1] = s.b128(ho + 32, so + 64 * n);
        qh = s.b128(ho + 128, so + 32 * n);
        sc = s.b64(192, so + 8 * n);
        d = s.b16(208, so);
    }
    __device__ __forceinline__ void open() {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            u32x4& v = i < 2 ? ql[i & 1] : qh;
            uint32_t x = v.x, y = v.y, z = v.z, w = v.w;
            swap_halves(x, z);
            swap_halves(y, w);
            v = u32x4{x, y, z, w};
        }
    }
    template <int S>
    __device__ __forceinline__ void ops(int u, bf16x8 (&o)[1]) const {
        const int nsh = u < 2 ? 0 : 4, hsh = 2 * u;
        auto code = [&](uint32_t l, uint32_t hb) {  // 4 (u - 32) as signed bytes
            return ((((l >> nsh) & 0x0f0f0f0fu) << 2) | (((hb >> hsh) & 0x03030303u) << 6)) ^ 0x80808080u;
        };
        o[0] = bytes_s(code(ql[u & 1][2 * S], qh[2 * S]), code(ql[u & 1][2 * S + 1], qh[2 * S + 1]));
    }
    __device__ __forceinline__ void scale(int u, int, float (&dv)[2], float&) const {
        const float d4 = f16_bits_to_f32(d) * 0.25f;
        const uint32_t p = u < 2 ? sc.x >> (16 * u) : sc.y >> (16 * (u - 2));
        dv[0] = d4 * (float)(int8_t)p;
        dv[1] = d4 * (float)(int8_t)(p >> 8);
    }
};
template <>
struct WGrp<HIP_BRIDGE_BF16> {
    static constexpr int G = 1;
    u32x4 v[2];
    __device__ __forceinline__ void load(const WSrc& s, int kb, int h) {
        v[0] = s.b128(32u * h, 64u * (uint32_t)kb);
        v[1] = s.b128(32u * h + 16, 64u * (uint32_t)kb);
    }
    __device__ __forceinline__ void open() {}
    template <int S>
    __device__ __forceinline__ void ops(int, bf16x8 (&o)[1]) const {
        o[0] = __builtin_bit_cast(bf16x8, v[S]);
    }
    __device__ __forceinline__ void scale(int, int, float (&)[2], float&) const {}
};
// sum of w[c] * x[c] over columns [c0, c1) of a weight row, one column at a time: for sums that are
// not finite. An infinite x (or one that bf16 rounds to infinity) has the terms inf, inf - inf,
// inf - inf, so every product of its token is NaN on the matrix cores, and a block's sum of unscaled
// codes can overflow where the scaled products do not; this gives what f32 arithmetic on the values
// gives. Serial, some ms a call: the price of a result that has to be looked at, not of a usual one. A
// NaN ends it (a token of NaN, say a slot that holds none, costs next to nothing).
template <int QT>
__device__ float dot_columns(const unsigned char* row, const float* x, int c0, int c1) {
    float sum = 0.0f;
#pragma unroll 1
    for (int c = c0; c < c1; ++c) {
        float w;
        if constexpr (QT == HIP_BRIDGE_BF16) {
            w = bf16_lo(*(const uint16_t*)(row + 2 * (int64_t)c));
        } else if constexpr (QT == HIP_BRIDGE_Q8_0 || QT == kQ8_0Odd) {
            const unsigned char* b = row + (int64_t)(c / 32) * 34;
            w = (float)(int8_t)b[2 + c % 32] * f16_bits_to_f32(*(const uint16_t*)b);
        } else if constexpr (QT == HIP_BRIDGE_Q4_K) {  // (layouts: WGrp)
            const unsigned char* b = row + (int64_t)(c / 256) * 144;
            const int j = c / 32 % 8, s0 = b[4 + j % 4], s1 = b[8 + j % 4], s2 = b[12 + j % 4];
            const int sc = j < 4 ? s0 & 63 : (s2 & 15) | (s0 >> 6) << 4, m = j < 4 ? s1 & 63 : s2 >> 4 | (s1 >> 6) << 4;
            const int q = b[16 + 32 * (j / 2) + c % 32] >> (4 * (j & 1)) & 15;
            w = f16_bits_to_f32(*(const uint16_t*)b) * (float)sc * (float)q - f16_bits_to_f32(*(const uint16_t*)(b + 2)) * (float)m;
        } else if constexpr (QT == HIP_BRIDGE_Q6_K) {
            const unsigned char* b = row + (int64_t)(c / 256) * 210;
            const int n = c / 128 % 2, t = c / 32 % 4, l = c % 32;
            const int u = (b[64 * n + 32 * (t & 1) + l] >> (t < 2 ? 0 : 4) & 15) | (b[128 + 32 * n + l] >> (2 * t) & 3) << 4;
            w = f16_bits_to_f32(*(const uint16_t*)(b + 208)) * (float)(int8_t)b[192 + 8 * n + l / 16 + 2 * t] * (float)(u - 32);
        } else {
            const unsigned char* b = row + (int64_t)(c / 32) * 18;
            const int j = c % 32, q = b[2 + j % 16] >> (j < 16 ? 0 : 4) & 15;
            w = (float)(q - 8) * f16_bits_to_f32(*(const uint16_t*)b);
        }
        sum = fmaf(w, x[c], sum);
        if (!(sum == sum)) break;
    }
    return sum;
}

// The (x term, w term) products accumulated, largest first: down to relative size 2^-16
// (x in XT terms: 3 for f32 activations, 1 for bf16 ones, which are exact). Smallest first, the
// large products lose low bits of the small sum they are added to, always in one direction, so
// that the error grows with the depth: 2560 x 10240 Q4_0, 8 tokens, 1.0e-7 -> 2.3e-7 off.
template <int XT, int NW>
struct TermPairs;
template <>
struct TermPairs<3, 1> {
    static constexpr int n = 3;
    static constexpr int xt[3] = {0, 1, 2}, wt[3] = {0, 0, 0};
};
template <>
struct TermPairs<3, 2> {
    static constexpr int n = 5;
    static constexpr int xt[5] = {0, 1, 0, 2, 1}, wt[5] = {0, 0, 1, 0, 1};
};
template <>
struct TermPairs<3, 3> {
    static constexpr int n = 6;
    static constexpr int xt[6] = {0, 1, 0, 2, 1, 0}, wt[6] = {0, 0, 1, 0, 1, 2};
};
template <int NW>
struct TermPairs<1, NW> {
    static constexpr int n = NW;
    static constexpr int xt[3] = {0, 0, 0}, wt[3] = {0, 1, 2};
};

// XK: activation form (X_F32: f32, split into three terms while staging; X_BF16: bf16, one
// term; X_TERMS: three bf16 planes split beforehand, staged as they are). GE: gate.up GeGLU
// pairs (out = gelu(g) * u).
enum XKind { X_F32 = 0, X_BF16 = 1, X_TERMS = 2 };

constexpr int kFine = 8;  // K steps between additions to a compensated total (a power of two of rounds)
// Activation blocks a thread holds ahead: more for the smaller tiles, whose steps are shorter.
template <int WT>
constexpr int x_ahead() {
    return WT >= 4 ? 1 : WT >= 2 ? 2 : 4;
}

// total += part, with what the rounding lost carried on in `lost` (Kahan's sum)
__device__ __forceinline__ void add_kahan(float& total, float& lost, float part) {
    const float y = part - lost, t = total + y;
    lost = (t - total) - y;
    total = t;
}

// FINE (tiles of 32 tokens): the accumulators hold kFine steps and then join a compensated total, so
// that a deep product's error does not grow with its depth.
// TEAMS = 2: a second set of four waves takes the other half of the workgroup's K steps, with LDS
// buffers of its own, and its sums join the first's through the LDS at the end.
template <int QT, int XK, int WT, int RT, bool GE, int TEAMS, bool FINE>
__global__ __launch_bounds__(256 * TEAMS, 2) void k_gemm_mfma(GemmArgs a) {
    constexpr int NT = 256;                    // threads of a team: four waves
    constexpr int XT = XK == X_BF16 ? 1 : 3;  // activation terms
    constexpr int NW = w_terms<QT>();
    constexpr bool SCALED = w_scaled<QT>();
    constexpr bool HALVES = QT == HIP_BRIDGE_Q6_K;  // a scale per MFMA rather than per block
    constexpr bool SUMS = SCALED || FINE;           // a step's products form a sum of their own
    constexpr int BT = 32 * WT;                // tokens per workgroup
    constexpr int TR = GE ? 16 : 32;           // output rows per tile
    constexpr int OR = TR * 4 * RT;            // and per workgroup
    constexpr int XPLANE = BT * kLdsRow;
    // Q4_K: per-token sums of each K step's activations, four steps' worth.
    // The min terms are an f32 MFMA per tile and two blocks where a wave has several tiles (as FMAs they
    // are a fifth of the loop's vector instructions: 10240 x 2560 x 2048 f32 500 -> 463 us); for one tile the
    // MFMA's latency shows (1024 x 2560 at 1024 tokens 40.6 -> 47.6), so FMAs there.
    constexpr bool MIN = QT == HIP_BRIDGE_Q4_K, MIN_MFMA = MIN && WT * RT > 1;
    __shared__ __attribute__((aligned(16))) uint16_t s_x_all[TEAMS * 2 * XT * XPLANE];
    __shared__ __attribute__((aligned(16))) float s_xs_all[TEAMS][MIN ? 4 : 1][MIN ? BT : 1];

    const int team = TEAMS == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT);
    const int tid = (int)threadIdx.x - team * NT;
    uint16_t* const s_x = s_x_all + team * (2 * XT * XPLANE);
    auto& s_xs = s_xs_all[team];
    const int lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gx = (a.rows + OR - 1) / OR;
    const int r_base = ((int)blockIdx.x % gx) * OR, b_base = ((int)blockIdx.x / gx) * BT;
    // K steps [kbb, kbe): the share of this team and (gridDim.y = 2, f32 output, added into zeroed y)
    // workgroup row, cut between super-blocks; `steps`, of the team that has the most.
    const int nkb_all = a.cols / kKB, parts = (int)gridDim.y * TEAMS, p0 = (int)blockIdx.y * TEAMS;
    auto cut = [&](int p) { return p == parts ? nkb_all : (int)((int64_t)nkb_all * p / parts + 7) & ~7; };
    const int kbb = cut(p0 + team), kbe = cut(p0 + team + 1);
    const int steps = TEAMS == 1 ? kbe - kbb : max(cut(p0 + 1) - cut(p0), cut(p0 + TEAMS) - cut(p0 + TEAMS - 1));

    // X staging. f32 x: chunk c = tid + NT i is token c / 8, columns 4 (c % 8) .. (four
    // floats); bf16 x: token c / 4, columns 8 (c % 4) .. (eight bf16); term planes: the same
    // within each plane. Loads through range-checked resources over the workgroup's tokens.
    constexpr int XE = XK == X_F32 ? 4 : 8;          // elements per 16-byte chunk
    constexpr int XCPT = kKB / XE;                  // chunks per token per block (per plane)
    constexpr int XPL = XK == X_TERMS ? 3 : 1;      // planes loaded
    constexpr int XPP = (BT * XCPT + NT - 1) / NT;  // passes per plane
    constexpr int XCC = BT * XCPT;                  // chunks per plane; with more threads than
                                                    // chunks several hold (and write) the same one
    constexpr int NXI = XPL * XPP;                  // chunks per thread
    const int xes = XK == X_F32 ? 4 : 2;
    const int64_t tok_left = (int64_t)a.batch - b_base;
    const int64_t xbytes = (tok_left < BT ? tok_left : BT) * (int64_t)a.cols * xes;
    const uint32_t xrange = (uint32_t)(xbytes < 0xffffffffLL ? xbytes : 0xffffffffLL);
    const int64_t plane_bytes = (int64_t)a.batch * a.cols * xes;
    __amdgpu_buffer_rsrc_t rsx[XPL];
#pragma unroll
    for (int u = 0; u < XPL; ++u)
        rsx[u] = buf_rsrc((const unsigned char*)a.x + u * plane_bytes + (int64_t)b_base * a.cols * xes, xrange);
    constexpr int UX = x_ahead<WT>();
    constexpr int U = 4;  // K steps per unrolled round
    u32x4 xr[UX][NXI];
    uint32_t xoff[XPP];
#pragma unroll
    for (int i = 0; i < XPP; ++i) {
        const int cc = (tid + NT * i) % XCC;
        xoff[i] = (uint32_t)(((int64_t)(cc / XCPT) * a.cols + XE * (cc % XCPT)) * xes);
    }
    const int last = kbe - 1;
    const int lastg = last & ~3;  // the last group's first block (rows are whole groups where G > 1)
    auto load_x = [&](int kb, int q, u32x4 (&r)[NXI]) {
        r[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                             rsx[q / XPP], xoff[q % XPP], (uint32_t)(min(kb, last) * kKB * xes), 0));
    };
    float csum[XPP];
    auto store_x = [&](int kb, int buf, int q, const u32x4& v) {
        uint16_t* const sx = s_x + buf * (XT * XPLANE) + (q / XPP) * XPLANE;
        const int cc = (tid + NT * (q % XPP)) % XCC, tok = cc / XCPT, k = XE * (cc % XCPT);
        uint16_t* const dst = sx + lds_chunk(tok, k / 8) + k % 8;
        // (MIN) the token's sum over the step's 32 columns of one term: pairs, then the
        // XCPT consecutive lanes holding its chunks (8 of 4 f32 or 4 of 8 bf16: the same
        // tree over the 32 values); each of them writes it (a branch would cut the step in two).
        // Planes: a thread holds the same chunk of all three, whose sums it adds first.
        auto put_sum = [&](float cs) {
            if constexpr (XK == X_TERMS) {
                float& c = csum[q % XPP];
                c = q < XPP ? cs : c + cs;
                if (q >= 2 * XPP) s_xs[MIN ? kb & 3 : 0][tok] = group_sum<XCPT>(c);
            } else {
                s_xs[MIN ? kb & 3 : 0][tok] = group_sum<XCPT>(cs);
            }
        };
        if constexpr (XK == X_F32) {
            uint32_t t0[3], t1[3];
            split3(__uint_as_float(v.x), __uint_as_float(v.y), t0);
            split3(__uint_as_float(v.z), __uint_as_float(v.w), t1);
#pragma unroll
            for (int p = 0; p < 3; ++p)
                *reinterpret_cast<u32x2*>(dst + p * XPLANE) = u32x2{t0[p], t1[p]};
            if constexpr (MIN)
                put_sum((__uint_as_float(v.x) + __uint_as_float(v.y)) + (__uint_as_float(v.z) + __uint_as_float(v.w)));
        } else {
            *reinterpret_cast<u32x4*>(dst) = v;
            if constexpr (MIN)
                put_sum(((bf16_lo(v.x) + bf16_hi(v.x)) + (bf16_lo(v.y) + bf16_hi(v.y))) +
                        ((bf16_lo(v.z) + bf16_hi(v.z)) + (bf16_lo(v.w) + bf16_hi(v.w))));
        }
    };

    // W: RT tiles of 32 rows, a row per lane and half (the last row again past the end); GE: a
    // tile is 16 gate rows and the same 16 rows of the up matrix, so that an output's two sums
    // lie 16 lanes apart.
    const int trow = GE ? lane & 15 : lane & 31;
    const int wrow = r_base + TR * RT * wave;
    WSrc ws[RT];
#pragma unroll
    for (int j = 0; j < RT; ++j)
        ws[j].row = (GE && (lane & 16) ? a.wu : a.w) + (int64_t)min(wrow + TR * j + trow, a.rows - 1) * a.row_bytes;
    using WQ = WGrp<QT>;
    constexpr int G = WQ::G;
    constexpr int RING = G == 1 ? 2 : 1;  // G = 1: blocks in flight; else the next group
    WQ cur[RT], nxt[RING][RT];

    f32x16 acc[WT][RT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j) acc[i][j] = f32x16{};
    using TP = TermPairs<XT, NW>;
    constexpr int NP = TP::n;

    // Operands of the current step and, while it runs, of the next: [step parity].
    bf16x8 wb[2][RT][2][NW];
    float dv[2][RT][2], mn[2][RT];
#pragma unroll
    for (int j = 0; j < RT; ++j) dv[1][j][0] = dv[1][j][1] = mn[1][j] = 0.0f;
    // A unit is one chain of MFMAs into a partial sum that a scale then adds into the
    // accumulators: a block of one tile, or with HALVES each of its MFMAs.
    constexpr int UPT = HALVES ? 2 : 1, UNITS = WT * RT * UPT, NMU = 2 * NP / UPT;
    f32x16 part[2] = {f32x16{}, f32x16{}};
    f32x4 xsv[MIN ? 4 : 1];  // (min in FMAs) the unit's per-token sums
    // FMAs [r0, r1) of a finished unit: acc += d * part [- mn * (token sums)]
    auto scale_unit = [&](int unit, const f32x16& pt, int par, int kb, int r0, int r1) {
        const int tile = unit / UPT / RT, j = unit / UPT % RT;
        const float d = dv[par][j][HALVES ? unit & 1 : 0];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (r < r0 || r >= r1) continue;
            float v = acc[tile][j][r];
            if constexpr (MIN && !MIN_MFMA) {
                // lane (l, r) of a tile holds token 8 (r / 4) + 4 (l / 32) + r % 4
                if (r % 4 == 0) xsv[r >> 2] = *reinterpret_cast<const f32x4*>(&s_xs[kb & 3][32 * tile + 8 * (r >> 2) + 4 * h]);
                v = fmaf(-mn[par][j], xsv[r >> 2][r & 3], v);
            }
            acc[tile][j][r] = SCALED ? fmaf(d, pt[r], v) : v + pt[r];
        }
    };
    // Q4_K: acc -= (token sums) x (min factors) of blocks kb - 1 and kb, an f32 MFMA over the two (half
    // h's operands are block kb - 1 + h's; mn[par] is block kb's).
    auto min_pair = [&](int kb, int par) {
#pragma unroll
        for (int i = 0; i < WT; ++i) {
            const float xs = s_xs[(kb - 1 + h) & 3][32 * i + (lane & 31)];
#pragma unroll
            for (int j = 0; j < RT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xs, h ? -mn[par][j] : -mn[par ^ 1][j], acc[i][j], 0, 0, 0);
        }
    };

    f32x16 total = f32x16{}, lost = f32x16{};
    auto flush = [&]() {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float t = total[r], l = lost[r];
            add_kahan(t, l, acc[0][0][r]);
            total[r] = t, lost[r] = l, acc[0][0][r] = 0.0f;
        }
    };

    // One K step: block kb from LDS buffer `u & 1` with wb[u & 1]. Between its MFMAs, a slice
    // each, run the scale products of the unit before, the conversion of block kb + 1's
    // activations (into the other buffer) and weights, and the loads of the blocks after: the
    // matrix cores take 32 cycles per MFMA, in which the wave can issue about seven vector
    // instructions; left to themselves the conversion and the scale products form runs of their
    // own beside which the matrix cores idle (10240 x 2560 x 2048 Q4_0, f32: 356 us).
    int xlane[2];  // the lane's place in a tile's LDS rows, per MFMA
#pragma unroll
    for (int s = 0; s < 2; ++s) xlane[s] = lds_chunk(lane & 31, wk<QT>(s, h) / 8);
    auto step = [&](int u, int kb) {
        const int pc = u & 1, pn = pc ^ 1;
        const uint16_t* const sx = s_x + pc * (XT * XPLANE);
        bf16x8 xa[2][2][XT];
        auto read_tile = [&](int i) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int t = 0; t < XT; ++t)
                    xa[i & 1][s][t] = *reinterpret_cast<const bf16x8*>(sx + t * XPLANE + 32 * i * kLdsRow + xlane[s]);
        };
        constexpr int NS = WT * RT * 2 * NP;  // MFMAs (slices)
        auto w_item = [&](int j, int s) {     // block kb + 1's weights of tile j, MFMA s
            const int un = G == 1 ? 0 : (u + 1) & 3;
            WQ& q = G == 1 ? nxt[pn][j] : cur[j];
            if (s == 0) {
                if (G > 1 && un == 0) {
                    cur[j] = nxt[0][j];
                    cur[j].open();
                    nxt[0][j].load(ws[j], min(kb + 1 + G, lastg), h);
                }
                q.scale(un, kb + 1, dv[pn][j], mn[pn][j]);
                q.template ops<0>(un, wb[pn][j][0]);
            } else {
                q.template ops<1>(un, wb[pn][j][1]);
                if (G == 1) q.load(ws[j], min(kb + 3, last), h);
            }
        };
        read_tile(0);
        if constexpr (SUMS) scale_unit(UNITS - 1, part[(UNITS - 1) & 1], pn, kb - 1, 0, 16);
        if constexpr (MIN_MFMA) {
            if (u & 1) min_pair(kb, pc);  // (shares of K-quants are whole super-blocks)
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < WT; ++i) {
            if (i + 1 < WT) read_tile(i + 1);
#pragma unroll
            for (int j = 0; j < RT; ++j)
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        const int t = ((i * RT + j) * 2 + s) * NP + p;           // slice
                        const int unit = (i * RT + j) * UPT + (HALVES ? s : 0);  // and its place in its unit
                        const int m = HALVES ? p : s * NP + p;
                        const bf16x8 A = xa[i & 1][s][TP::xt[p]], Bv = wb[pc][j][s][TP::wt[p]];
                        if constexpr (SUMS)
                            part[unit & 1] =
                                __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, Bv, m == 0 ? f32x16{} : part[unit & 1], 0, 0, 0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, Bv, acc[i][j], 0, 0, 0);
                        if (SUMS && unit > 0) {
                            constexpr int M1 = NMU > 1 ? NMU - 1 : 1;
                            const int mm = NMU > 1 ? m - 1 : 0;
                            if (mm >= 0)
                                scale_unit(unit - 1, part[(unit - 1) & 1], pc, kb, 16 * mm / M1, 16 * (mm + 1) / M1);
                        }
#pragma unroll
                        for (int q = 0; q < NXI; ++q)
                            if (q * NS / NXI == t) {
                                store_x(kb + 1, pn, q, xr[(u + 1) % UX][q]);
                                load_x(kb + 1 + UX, q, xr[(u + 1) % UX]);
                            }
#pragma unroll
                        for (int w = 0; w < 2 * RT; ++w)  // after the last step's scale products
                            if ((2 * w + 1) * NS / (4 * RT) == t) w_item(w >> 1, w & 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
        }
        __syncthreads();  // block kb + 1 is in its buffer, and block kb's is free
    };

#pragma unroll
    for (int j = 0; j < RT; ++j) {
        cur[j].load(ws[j], kbb, h);
        if constexpr (G > 1) {
            nxt[0][j].load(ws[j], min(kbb + G, lastg), h);
        } else {
            nxt[1 % RING][j].load(ws[j], min(kbb + 1, last), h);
            nxt[0][j].load(ws[j], min(kbb + 2, last), h);
        }
    }
#pragma unroll
    for (int q = 0; q < NXI; ++q) load_x(kbb, q, xr[0]);
#pragma unroll
    for (int q = 0; q < NXI; ++q) store_x(kbb, 0, q, xr[0][q]);
#pragma unroll
    for (int b = 0; b < UX; ++b)
#pragma unroll
        for (int q = 0; q < NXI; ++q) load_x(kbb + 1 + b, q, xr[(b + 1) % UX]);
#pragma unroll
    for (int j = 0; j < RT; ++j) {
        cur[j].open();
        cur[j].scale(0, kbb, dv[0][j], mn[0][j]);
        cur[j].template ops<0>(0, wb[0][j][0]);
        cur[j].template ops<1>(0, wb[0][j][1]);
    }
    if constexpr (MIN && !MIN_MFMA) {  // the first step's scaling of "the unit before" adds 0 * 0
        if (tid < BT) s_xs[3][tid] = 0.0f;
    }
    __syncthreads();
    // A branch per step keeps each in a basic block of its own: unrolled into one, instruction
    // selection moves the scale products of several steps together, and their partial sums spill.
    for (int k0 = kbb; k0 < kbb + steps; k0 += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k0 + u < kbe) step(u, k0 + u);  // uniform
            else if (TEAMS > 1 && k0 + u < kbb + steps) __syncthreads();  // the other team's step
        }
        if (FINE && ((k0 + U) & (kFine - 1)) == 0) flush();
    }
    if constexpr (SUMS) {  // the last unit's scale products
        if ((kbe - kbb) & 1) scale_unit(UNITS - 1, part[(UNITS - 1) & 1], 0, kbe - 1, 0, 16);
        else scale_unit(UNITS - 1, part[(UNITS - 1) & 1], 1, kbe - 1, 0, 16);
    }
    if constexpr (FINE) {
        flush();
        acc[0][0] = total;
    }

    if constexpr (TEAMS > 1) {
        static_assert(TEAMS == 2 && sizeof(s_x_all) >= sizeof(acc) * NT);
        float* const sums = reinterpret_cast<float*>(s_x_all) + tid;  // (every step's barrier is behind)
#pragma unroll
        for (int q = 0; q < WT * RT * 16; ++q)
            if (team) sums[q * NT] = acc[q / 16 / RT][q / 16 % RT][q % 16];
        __syncthreads();
        if (team) return;
#pragma unroll
        for (int q = 0; q < WT * RT * 16; ++q) acc[q / 16 / RT][q / 16 % RT][q % 16] += sums[q * NT];
    }

    // Epilogue: lane (l, r) of tile (i, j) holds token 8 (r / 4) + 4 (l / 32) + r % 4 and row
    // l % 32.
    constexpr bool CHECK = FINE && XK == X_F32;  // sums that are not finite are formed again (dot_columns)
    uint32_t again = 0;
    if constexpr (CHECK) {
#pragma unroll
        for (int r = 0; r < 16; ++r) again |= !(fabsf(acc[0][0][r]) < INFINITY) ? 1u << r : 0u;
    }
    auto out = [&](auto put) {
#pragma unroll
        for (int j = 0; j < RT; ++j) {
            const int row = wrow + TR * j + trow;
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float v = acc[i][j][r];
                    if constexpr (GE) v = gelu_fast(v) * __shfl_xor(v, 16);
                    const int tok = b_base + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (tok < a.batch && row < a.rows && !(GE && (lane & 16)) && !(CHECK && again >> r & 1))
                        put((int64_t)tok * a.rows + row, v);
                }
        }
        if constexpr (CHECK) {
            for (; again; again &= again - 1) {
                const int r = __builtin_ctz(again), tok = b_base + 8 * (r >> 2) + 4 * h + (r & 3), row = wrow + trow;
                if (tok < a.batch && row < a.rows)
                    put((int64_t)tok * a.rows + row,
                        dot_columns<QT>(ws[0].row, (const float*)a.x + (int64_t)tok * a.cols, kKB * cut(p0), kKB * cut(p0 + TEAMS)));
            }
        }
    };
    if (a.y_bf16)
        out([&](int64_t o, float v) { ((uint16_t*)a.y)[o] = (uint16_t)(pack_bf16x2(v, 0.0f) & 0xffffu); });
    else if (gridDim.y > 1)  // two K halves into zeroed y: 0 + a + b in either order
        out([&](int64_t o, float v) { unsafeAtomicAdd((float*)a.y + o, v); });
    else
        out([&](int64_t o, float v) { ((float*)a.y)[o] = v; });
}

__global__ __launch_bounds__(256) void k_zero_f32(float* __restrict__ y, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) y[i] = 0.0f;
}
void launch_zero_f32(float* y, int64_t n, hipStream_t s) {
    k_zero_f32<<<(unsigned)std::min<int64_t>(cdiv(n, 256), 8192), 256, 0, s>>>(y, n);
}

// Two K halves per output tile (gridDim.y), added into zeroed y by float atomics: with exactly
// two addends (0 + a + b in either order) the sum does not depend on their order, so results stay
// bit-reproducible. f32 output only; 16 blocks at least, so that a cut between super-blocks
// leaves both halves some.
static unsigned split_k(const GemmArgs& a, bool ge, bool want, hipStream_t s) {
    if (!want || ge || a.y_bf16 || a.cols < 16 * kKB) return 1;
    launch_zero_f32((float*)a.y, (int64_t)a.batch * a.rows, s);
    return 2;
}

template <int QT, int XK, bool GE, int WT, int RT, int TEAMS = 1, bool FINE = false>
static void launch_tile(const GemmArgs& a, unsigned ky, hipStream_t s) {
    const dim3 grid((unsigned)(cdiv(a.rows, (GE ? 64 : 128) * RT) * cdiv(a.batch, 32 * WT)), ky);
    k_gemm_mfma<QT, XK, WT, RT, GE, TEAMS, FINE><<<grid, 256 * TEAMS, 0, s>>>(a);
}
// Workgroup tile (tokens x rows; GE: half the output rows), for 256 CUs that hold two workgroups
// each. Large tiles convert an operand for more MFMAs, small ones fill the chip. us at 10240 x 2560
// unless said:
//   bf16 activations: 128 x 128 from 1.5 workgroups per CU (2048 tokens Q4_0: 140, 64 x 128 151,
//     32 x 128 212), else 64 x 128 likewise, else 32 x 128; single blocks, two loads a step whatever the
//     tile, 128 x 128 from 80 tiles and 64 x 128 from 64 (10240 x 2592 at 200 tokens Q8_0 101 -> 51, Q4_0 60 -> 46; Q4_0 128 x 128 as other rows).
//   f32 (three-term) activations: 64 x 256 from three per CU for Q4_0 (it reads the LDS half as often
//     per MFMA; 2048 tokens 284, 128 x 128 336, 64 x 128 322), from 400 tiles for BF16 rows that are
//     not deep (700 tokens 123, 128 x 128 132, 64 x 128 147; gate.up 1024: 344, 361, 384; at 320 tiles, 512
//     tokens, 111 against 102). 128 x 128 from 448 tiles for Q8_0 (2048 tokens 367, 64 x 128 400;
//     21504 x 5376 gate.up 333: 590, 695; 320 tiles: 122, 116) and deep BF16 (21504 x 5376 at 333 tokens
//     274, 64 x 256 283, 64 x 128 302), unless a quarter more of it is padding. The K-quants' conversion
//     leaves no registers for either. Else 64 x 128 from 1.5 per CU, else 32 x 128 (512 tokens of 2048 x
//     2560: 39 us, 64 x 128 49); deep BF16 rows 64 x 128 from 160 tiles (2560 x 10240 at 512 tokens 129, 32
//     x 128 156; at 333, 120 tiles, 114 against 101).
//   planes: nothing to convert, so large tiles pay earlier. 128 x 128 from 320 tiles for Q8_0 and BF16
//     (512 tokens BF16 110, 64 x 128 122), 64 x 128 from 80 (BF16 at 200 tokens 63, 32 x 128 95; Q6_K 2560 x
//     10240 at 333 111, 136), but for Q4_0, whose 32 x 128 tiles are as fast (150 tokens 42, 44).
//   Q8_0 rows that are not deep take single blocks on 64 x 128 tiles of f32 activations: groups need
//     more registers and a swap of halves (512 tokens 116 against 124); deep ones are bound by the
//     loads (2560 x 10240 at 700 tokens 287 with single blocks, 166 with groups).
// Two K halves per tile (f32 output) where the tiles do not fill the CUs twice (512 tokens of 2048
// x 2560 39 -> 32 us, 1024 rows 38 -> 26), or four times for deep products (2560 x 10240 x 2048:
// 365 -> 341 us; at 333 tokens Q6_K 168 -> 117); at 333 tokens of 10240 x 2560 (480 tiles) the
// halves cost more than they fill (87 -> 97 us).
// Up to 128 tiles two halves leave each CU one workgroup or none, one wave per SIMD and a step's
// latency bare: each half then runs as two teams. us, without / with: 2560 x 10240 at 150 tokens Q4_0
// 85 / 63, Q4_K 101 / 78, Q8_0 98 / 82, Q6_K 98 / 86; 1024 x 2560 at 512 tokens Q4_0 25.5 / 22.7, Q4_K
// 29.0 / 26.2, Q8_0 25.2 / 23.3; 2048 x 2560 at 200 tokens Q4_0 24.1 / 21.2, Q6_K 27.7 / 28.3 (so deep
// ones only), BF16 25.5 / 28.2 (none); from 140 tiles on they lose (2048 x 2560 at 333 tokens 26.9 /
// 28.5; Q4_K 2560 x 10240 119 / 146). Pre-split planes take the same shares, so that they give the same
// sums (2560 x 10240 at 150 tokens Q4_0 73 / 62, Q4_K 123 / 95; 1024 x 2560 at 512 Q4_0 24.5 / 25.1).
// f32 products of few tokens take the compensated totals (FINE) where the kernels for small batches,
// whose sums are short chains, are closer to the exact product than the plain loop: from the batch at
// which hip_gemm takes this kernel to that where all of these shapes do, BF16 and Q6_K always, the
// others from the depth where those kernels change theirs.
static bool fine_sums(int qtype, int rows, int cols, int batch) {
    const bool wide = rows >= kWideRows, q6 = qtype == HIP_BRIDGE_Q6_K;
    const int below = qtype == HIP_BRIDGE_Q4_K ? (wide ? 128 : 96) : q6 ? (wide ? 64 : 96) : wide ? 96 : 128;
    return batch < below && batch >= gemm_mfma_min_batch(qtype, rows, cols) && (q6 || qtype == HIP_BRIDGE_BF16 || cols > (qtype == HIP_BRIDGE_Q4_K ? 5120 : 10240));
}
template <int QT, int XK, bool GE>
static void launch_qt(const GemmArgs& a, hipStream_t s) {
    constexpr bool Q8 = QT == HIP_BRIDGE_Q8_0 || QT == kQ8_0Odd, B16 = QT == HIP_BRIDGE_BF16, TERMS = XK == X_TERMS;
    constexpr bool F32 = XK != X_BF16 && !GE;
    auto wgs = [&](int wt, int rt) { return cdiv(a.rows, 128 * rt / (GE ? 2 : 1)) * cdiv(a.batch, 32 * wt); };
    const bool deep = a.cols >= kSplitMinCols;
    const bool fine = F32 && !a.y_bf16 && fine_sums(QT & 0xff, a.rows, a.cols, a.batch);
    const bool big = F32 && (QT == HIP_BRIDGE_Q4_0 || B16) && !fine && wgs(2, 2) >= 768;
    // The shares of K, from the tiles that f32 activations had the shares measured on, so that planes
    // and f32 activations give the same sums whichever tile they take
    constexpr bool ODD = QT == kQ4_0Odd || QT == kQ8_0Odd;
    const bool whole = cdiv(a.batch, 128) * 8 <= cdiv(a.batch, 64) * 5;  // 128 tokens: at most a quarter more padding
    int wt = fine ? 1 : big || wgs(2, 1) >= 384 ? 2 : 1;
    if (XK == X_BF16) {
        if (ODD) wt = whole && wgs(4, 1) >= (Q8 ? 80 : 384) ? 4 : a.batch > 32 && wgs(2, 1) >= 64 ? 2 : 1;
        else if (wgs(4, 1) >= 384) wt = 4;
    }
    const int64_t n = wgs(wt, big ? 2 : 1);
    if constexpr (F32 && !B16 && QT != kQ4_0Odd) {
        const bool pays = QT != HIP_BRIDGE_Q6_K || deep;
        if (wt == 1 && n <= 128 && pays && !a.y_bf16 && a.cols >= 32 * kKB) {
            const unsigned ky = split_k(a, GE, true, s);
            fine ? launch_tile<QT, XK, GE, 1, 1, 2, true>(a, ky, s) : launch_tile<QT, XK, GE, 1, 1, 2>(a, ky, s);
            return;
        }
    }
    const unsigned ky = split_k(a, GE, n < 384 || (n < 1024 && deep), s);
    if constexpr (F32) {
        if (fine) {
            launch_tile<QT, XK, GE, 1, 1, 1, true>(a, ky, s);
            return;
        }
    }
    int rt = big ? 2 : 1;
    if constexpr (XK != X_BF16) {
        if (wt == 1 && !fine && (TERMS || QT == kQ8_0Odd ? QT != HIP_BRIDGE_Q4_0 && a.batch > 32 && wgs(2, 1) >= 80 : B16 && deep && wgs(2, 1) >= 160)) wt = 2;
        if ((Q8 || B16) && whole && wgs(4, 1) >= (TERMS ? 320 : 448) && (Q8 || TERMS || deep)) wt = 4, rt = 1;
        else if (B16 && !TERMS && wgs(2, 2) >= 400 && !deep) wt = rt = 2;
        else if (B16 && TERMS) rt = 1;
    }
    if constexpr ((QT == HIP_BRIDGE_Q4_0 && F32) || (B16 && XK == X_F32)) {
        if (rt == 2) {
            launch_tile<QT, XK, GE, 2, 2>(a, ky, s);
            return;
        }
    }
    if constexpr (XK == X_BF16 || Q8 || B16) {
        if (wt == 4) {
            launch_tile<QT, XK, GE, 4, 1>(a, ky, s);
            return;
        }
    }
    if constexpr (Q8 && XK == X_F32) {
        if (wt == 2 && !deep) {
            launch_tile<kQ8_0Odd, XK, GE, 2, 1>(a, ky, s);
            return;
        }
    }
    if (wt == 2) launch_tile<QT, XK, GE, 2, 1>(a, ky, s);
    else launch_tile<QT, XK, GE, 1, 1>(a, ky, s);
}

// ---- dense weights ---------------------------------------------------------------------------
// F16 and F32 weights (two and three terms), and BF16 weights with bf16 activations. A dense row
// is 64-128 bytes per step, so fetching each lane's row into its registers touches a cache line
// per lane and instruction for 16 bytes of it; here the threads load half rows that neighbour
// each other and stage them through the LDS like the activations (BF16 x bf16, 2048 tokens:
// 10240 x 2560 149 us, rows in registers 160; gate.up 21504 x 5376 1807 against 2080. With f32
// activations the three terms hide the fetch and the register form is the faster one from 333
// tokens (111 -> 71 us) and equal at 2048, so BF16 weights take it there.)
// A 256-thread workgroup owns 64 WT tokens x 64 WR rows; its 4 waves form a 2 x 2 grid of WT x WR
// tiles of 32 x 32. The LDS holds block k's terms (rows padded to 80 bytes) while registers hold
// block k + 1's raw X and W; where two operand buffers fit two workgroups per CU a step takes one
// barrier.
constexpr int kDenseThreads = 256;
constexpr int kDenseRow = 40;  // bf16 per LDS row: 32 + 8 padding (80 bytes)
template <int QT>
struct DRaw {
    u32x4 v[QT == HIP_BRIDGE_F32 ? 4 : 2];  // elements [16h, 16h + 16) of a row's block
};
__device__ __forceinline__ u32x4 sel4(bool ok, u32x4 v) { return ok ? v : u32x4{0, 0, 0, 0}; }
// `blk` is always a valid address (the caller clamps the row); `ok` false gives zeros, selected
// after the loads so that no load sits under a branch.
template <int QT>
__device__ __forceinline__ void load_d(const unsigned char* blk, int h, bool ok, DRaw<QT>& r) {
    constexpr int n = QT == HIP_BRIDGE_F32 ? 4 : 2;
#pragma unroll
    for (int i = 0; i < n; ++i) r.v[i] = sel4(ok, ld16(blk + 16 * n * h + 16 * i));
}
template <int QT>
__device__ __forceinline__ void store_d(const DRaw<QT>& r, int h, uint16_t* sw, int plane, int row) {
    uint16_t* dst = sw + row * kDenseRow;
    if constexpr (QT == HIP_BRIDGE_BF16) {
        *reinterpret_cast<u32x4*>(dst + 16 * h) = r.v[0];
        *reinterpret_cast<u32x4*>(dst + 16 * h + 8) = r.v[1];
    } else if constexpr (QT == HIP_BRIDGE_F16) {
        uint32_t t[2][8];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t w4[4] = {r.v[i].x, r.v[i].y, r.v[i].z, r.v[i].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t s[2];
                split2(f16_bits_to_f32(w4[j] & 0xffffu), f16_bits_to_f32(w4[j] >> 16), s);
                t[0][4 * i + j] = s[0];
                t[1][4 * i + j] = s[1];
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            uint16_t* d = sw + u * plane + row * kDenseRow + 16 * h;
            *reinterpret_cast<u32x4*>(d) = u32x4{t[u][0], t[u][1], t[u][2], t[u][3]};
            *reinterpret_cast<u32x4*>(d + 8) = u32x4{t[u][4], t[u][5], t[u][6], t[u][7]};
        }
    } else {  // F32: elements [16h, 16h + 16)
        uint32_t t[3][8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t s[3];
            split3(__uint_as_float(r.v[i].x), __uint_as_float(r.v[i].y), s);
            t[0][2 * i] = s[0], t[1][2 * i] = s[1], t[2][2 * i] = s[2];
            split3(__uint_as_float(r.v[i].z), __uint_as_float(r.v[i].w), s);
            t[0][2 * i + 1] = s[0], t[1][2 * i + 1] = s[1], t[2][2 * i + 1] = s[2];
        }
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            uint16_t* d = sw + u * plane + row * kDenseRow + 16 * h;
            *reinterpret_cast<u32x4*>(d) = u32x4{t[u][0], t[u][1], t[u][2], t[u][3]};
            *reinterpret_cast<u32x4*>(d + 8) = u32x4{t[u][4], t[u][5], t[u][6], t[u][7]};
        }
    }
}

// Workgroups per CU the launch asks registers for: three (170 VGPRs a lane) for bf16
// activations when the LDS holds three, so a third wave per SIMD has MFMAs ready while the
// others read operands or wait at a barrier; two otherwise (the three-term activations' loop
// needs more registers: held to 170 it spills).
template <int QT, int XK, int WT, int WR>
constexpr int dense_wgs_per_cu() {
    constexpr int bt = 64 * WT, br = 64 * WR;
    constexpr int oper = (bt + w_terms<QT>() * br) * kDenseRow * 2;  // bf16 activations: one term
    return XK == X_BF16 && 2 * oper * 3 <= 160 * 1024 ? 3 : 2;
}

template <int QT, int XK, int WT, int WR, bool GE>
__global__ __launch_bounds__(kDenseThreads, (dense_wgs_per_cu<QT, XK, WT, WR>())) void k_gemm_dense(GemmArgs a) {
    constexpr int XT = XK == X_BF16 ? 1 : 3;  // activation terms
    constexpr int NW = w_terms<QT>();
    constexpr int BT = 2 * 32 * WT;  // tokens per workgroup
    constexpr int BR = 2 * 32 * WR;  // W rows per workgroup (GE: BR / 2 gate + BR / 2 up rows)
    constexpr int OR = GE ? BR / 2 : BR;  // output rows per workgroup
    constexpr int XPLANE = BT * kDenseRow, WPLANE = BR * kDenseRow;
    constexpr int OPER_BYTES = (XT * XPLANE + NW * WPLANE) * 2;
    // Two operand buffers (block kb read while block kb + 1 is written: one barrier per step)
    // when they fit two workgroups per CU in the 160 KB of LDS; else one.
    constexpr bool DB = 2 * OPER_BYTES <= 80 * 1024 && XK != X_F32;
    constexpr int NBUF = DB ? 2 : 1;
    constexpr int XCH_BYTES = GE ? 2 * WT * WR * 16 * kWave * 4 : 0;  // up accumulators, two waves
    constexpr int MAIN_BYTES = NBUF * OPER_BYTES > XCH_BYTES ? NBUF * OPER_BYTES : XCH_BYTES;
    __shared__ __attribute__((aligned(16))) unsigned char s_raw[MAIN_BYTES];
    auto sx_of = [&](int b) { return reinterpret_cast<uint16_t*>(s_raw + b * OPER_BYTES); };
    auto sw_of = [&](int b) { return reinterpret_cast<uint16_t*>(s_raw + b * OPER_BYTES) + XT * XPLANE; };

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int tile = blockIdx.x;
    const int gx = (a.rows + OR - 1) / OR;
    const int r_base = (tile % gx) * OR, b_base = (tile / gx) * BT;
    // K steps [kbb, kbe): all of them, or with a split launch (gridDim.y = 2, f32 output,
    // added into zeroed y) one half per workgroup row
    const int nkb_all = a.cols / kKB;
    const int kbb = (int)((int64_t)nkb_all * blockIdx.y / gridDim.y);
    const int kbe = (int)((int64_t)nkb_all * (blockIdx.y + 1) / gridDim.y);

    // X staging. f32 x: chunk c = tid + 256 i is token c / 8, columns 4 (c % 8) .. (four
    // floats); bf16 x: token c / 4, columns 8 (c % 4) .. (eight bf16); term planes: chunk c of
    // plane c / (4 BT), as bf16 x within the plane. Loads through range-checked resources over
    // the workgroup's tokens: tokens past the batch read zeros.
    constexpr int XE = XK == X_F32 ? 4 : 8;          // elements per 16-byte chunk
    constexpr int XCPT = kKB / XE;                  // chunks per token per block (per plane)
    constexpr int XPL = XK == X_TERMS ? 3 : 1;      // planes loaded
    constexpr int XCH = XPL * BT * XCPT / kDenseThreads;
    const int xes = XK == X_F32 ? 4 : 2;
    const int64_t tok_left = (int64_t)a.batch - b_base;
    const int64_t xbytes = (tok_left < BT ? tok_left : BT) * (int64_t)a.cols * xes;
    const uint32_t xrange = (uint32_t)(xbytes < 0xffffffffLL ? xbytes : 0xffffffffLL);
    const int64_t plane_bytes = (int64_t)a.batch * a.cols * xes;
    __amdgpu_buffer_rsrc_t rsx[XPL];
#pragma unroll
    for (int u = 0; u < XPL; ++u)
        rsx[u] = buf_rsrc((const unsigned char*)a.x + u * plane_bytes + (int64_t)b_base * a.cols * xes, xrange);
    u32x4 xr[XCH];
    // A plane is a whole number of 256-chunk passes, so pass i's plane is a constant of the
    // unrolled loop: the resource it selects stays in scalar registers (a plane index
    // computed from tid would make each load a loop over the lanes' distinct resources).
    static_assert((BT * XCPT) % kDenseThreads == 0, "X plane not a whole number of passes");
    auto load_x = [&](int kb) {
#pragma unroll
        for (int i = 0; i < XCH; ++i) {
            constexpr int PC = BT * XCPT;  // chunks per plane
            const int pl = kDenseThreads * i / PC, cc = tid + kDenseThreads * i % PC, tok = cc / XCPT;
            const uint32_t off = (uint32_t)(((int64_t)tok * a.cols + kb * kKB + XE * (cc % XCPT)) * xes);
            xr[i] = bldp<POL_DEFAULT>(rsx[pl], off);
        }
    };
    auto store_x = [&](int buf) {
        uint16_t* const sx = sx_of(buf);
#pragma unroll
        for (int i = 0; i < XCH; ++i) {
            constexpr int PC = BT * XCPT;
            const int pl = kDenseThreads * i / PC, cc = tid + kDenseThreads * i % PC;
            const int tok = cc / XCPT, k = XE * (cc % XCPT);
            if constexpr (XK == X_F32) {
                uint32_t t0[3], t1[3];
                split3(__uint_as_float(xr[i].x), __uint_as_float(xr[i].y), t0);
                split3(__uint_as_float(xr[i].z), __uint_as_float(xr[i].w), t1);
#pragma unroll
                for (int u = 0; u < 3; ++u)
                    *reinterpret_cast<u32x2*>(sx + u * XPLANE + tok * kDenseRow + k) = u32x2{t0[u], t1[u]};
            } else {
                *reinterpret_cast<u32x4*>(sx + pl * XPLANE + tok * kDenseRow + k) = xr[i];
            }
        }
    };
    // W staging: half rows (BR rows x 2 halves over 256 threads: BR / 128 passes, or the
    // first 2 BR threads when BR < 128). GE: tile rows [0, OR) are gate rows, [OR, BR) the
    // same rows of the up matrix.
    constexpr int WPASS = BR * 2 >= kDenseThreads ? BR * 2 / kDenseThreads : 1;
    constexpr int64_t blk_bytes = QT == HIP_BRIDGE_F32 ? 128 : 64;  // per K step
    DRaw<QT> wr[WPASS];
    auto load_wt = [&](int kb) {
        const int64_t boff = (int64_t)kb * blk_bytes;
#pragma unroll
        for (int i = 0; i < WPASS; ++i) {
            const int hr = tid + kDenseThreads * i, row = hr >> 1, h = hr & 1;
            const bool up = GE && row >= OR;
            const int gr = r_base + (up ? row - OR : row);
            const bool ok = hr < 2 * BR && gr < a.rows;
            const unsigned char* wm = up ? a.wu : a.w;
            load_d<QT>(wm + (int64_t)min(gr, a.rows - 1) * a.row_bytes + boff, h, ok, wr[i]);
        }
    };
    auto store_wt = [&](int buf) {
        uint16_t* const swb = sw_of(buf);
#pragma unroll
        for (int i = 0; i < WPASS; ++i) {
            const int hr = tid + kDenseThreads * i;
            if (2 * BR >= kDenseThreads || hr < 2 * BR) store_d<QT>(wr[i], hr & 1, swb, WPLANE, hr >> 1);
        }
    };

    const int wt0 = (wave >> 1) * 32 * WT;  // the wave's first token (within the workgroup)
    const int wr0 = (wave & 1) * 32 * WR;   // the wave's first W row (GE: wave & 1 = up)
    f32x16 acc[WT][WR];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WR; ++j) acc[i][j] = f32x16{};

    using TP = TermPairs<XT, NW>;
    constexpr int NP = TP::n;
    // One K step: block kb's operands from LDS buffer `buf` into registers, its MFMAs, then
    // `convert` (block kb + 1 into the LDS and the loads of kb + 2).
    auto step = [&](int buf, auto convert) {
        const uint16_t* const sx = sx_of(buf);
        const uint16_t* const sw = sw_of(buf);
        // with one buffer every wave holds all of block kb's operands before the barrier;
        // with two, each K = 16 half's operands are read just before its MFMAs (half the
        // registers)
        constexpr int KH = DB ? 1 : 2;
        bf16x8 xa[KH][WT][XT], wb[KH][WR][NW];
        auto read_ops = [&](int ks, int slot) {
            const int ko = 16 * ks + 8 * (lane >> 5);
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int u = 0; u < XT; ++u)
                    xa[slot][i][u] = *reinterpret_cast<const bf16x8*>(sx + u * XPLANE + (wt0 + 32 * i + (lane & 31)) * kDenseRow + ko);
#pragma unroll
            for (int j = 0; j < WR; ++j)
#pragma unroll
                for (int u = 0; u < NW; ++u)
                    wb[slot][j][u] = *reinterpret_cast<const bf16x8*>(sw + u * WPLANE + (wr0 + 32 * j + (lane & 31)) * kDenseRow + ko);
        };
        auto mfmas = [&](int ks, int slot) {
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WR; ++j)
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        const bf16x8 A = xa[slot][i][TP::xt[p]], Bv = wb[slot][j][TP::wt[p]];
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, Bv, acc[i][j], 0, 0, 0);
                    }
        };
        if constexpr (DB) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                read_ops(ks, 0);
                mfmas(ks, 0);
            }
        } else {
            read_ops(0, 0);
            read_ops(1, 1);
            __syncthreads();
            mfmas(0, 0);
            mfmas(1, 1);
        }
        convert();
    };

    // Pipeline. The raw registers hold block kb + 1 while the MFMAs of block kb run; they are
    // converted into the LDS (the other buffer with DB, else the same one once every wave has
    // read block kb's operands) and block kb + 2's loads are issued, so the matrix cores work
    // during the conversion rather than after it. Past the end: the last block again, unused.
    load_x(kbb);
    load_wt(kbb);
    store_x(0);
    store_wt(0);
    __syncthreads();
    load_x(min(kbb + 1, kbe - 1));
    load_wt(min(kbb + 1, kbe - 1));
    for (int it = 0; it < kbe - kbb; ++it) {
        const int kb = kbb + it;
        const int cur = DB ? (it & 1) : 0, nxt = DB ? (cur ^ 1) : 0;
        step(cur, [&]() {
            store_x(nxt);
            store_wt(nxt);
            load_x(min(kb + 2, kbe - 1));
            load_wt(min(kb + 2, kbe - 1));
        });
        __syncthreads();  // block kb + 1 is in the LDS (DB: and block kb's buffer is free)
    }

    // Epilogue: lane (l, r) of tile (i, j) holds token 8 (r / 4) + 4 (l / 32) + r % 4 and row
    // l % 32. GE: the up waves pass their accumulators through the (now free) LDS to the gate
    // waves of the same tokens, which write gelu(g) * u.
    if constexpr (GE) {
        float* const xch = reinterpret_cast<float*>(s_raw) + (wave >> 1) * (WT * WR * 16 * kWave);
        if (wave & 1) {
#pragma unroll
            for (int i = 0; i < WT; ++i)
#pragma unroll
                for (int j = 0; j < WR; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) xch[((i * WR + j) * 16 + r) * kWave + lane] = acc[i][j][r];
        }
        __syncthreads();
        if (wave & 1) return;
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < WR; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[i][j][r] = gelu_fast(acc[i][j][r]) * xch[((i * WR + j) * 16 + r) * kWave + lane];
    }
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WR; ++j) {
            const int row = r_base + (GE ? 0 : wr0) + 32 * j + (lane & 31);
            if (row >= a.rows) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int tok = b_base + wt0 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (tok < a.batch) {
                    if (a.y_bf16)
                        ((uint16_t*)a.y)[(int64_t)tok * a.rows + row] = (uint16_t)(pack_bf16x2(acc[i][j][r], 0.0f) & 0xffffu);
                    else if (gridDim.y > 1)  // two K halves into zeroed y: 0 + a + b in either order
                        unsafeAtomicAdd((float*)a.y + (int64_t)tok * a.rows + row, acc[i][j][r]);
                    else
                        ((float*)a.y)[(int64_t)tok * a.rows + row] = acc[i][j][r];
                }
            }
        }
}

// Workgroup tile: the largest of 128 x 128, 64 x 128 and 64 x 64 (tokens x W rows) that still
// gives at least two workgroups per CU (bigger tiles convert each operand for more MFMAs;
// smaller ones fill the chip at small batches). Deep products with f32 output that give fewer
// than two rounds of workgroups run each tile as two K halves.
template <int QT, int XK, bool GE>
static void launch_dense(const GemmArgs& a, hipStream_t s) {
    constexpr int64_t kFill = 512;
    auto wgs = [&](int bt, int br) { return cdiv(a.rows, GE ? br / 2 : br) * cdiv(a.batch, bt); };
    const int64_t n = wgs(128, 128) >= kFill ? wgs(128, 128) : wgs(64, 128) >= kFill ? wgs(64, 128) : wgs(64, 64);
    const unsigned ky = split_k(a, GE, n < 2 * kFill && a.cols >= kSplitMinCols, s);
    const dim3 grid((unsigned)n, ky);
    if (wgs(128, 128) >= kFill) {
        k_gemm_dense<QT, XK, 2, 2, GE><<<grid, kDenseThreads, 0, s>>>(a);
    } else if (wgs(64, 128) >= kFill) {
        k_gemm_dense<QT, XK, 1, 2, GE><<<grid, kDenseThreads, 0, s>>>(a);
    } else {
        k_gemm_dense<QT, XK, 1, 1, GE><<<grid, kDenseThreads, 0, s>>>(a);
    }
}

template <int QT>
static void launch_q(const GemmArgs& a, int xk, bool ge, hipStream_t s) {
    if constexpr (QT == HIP_BRIDGE_F16 || QT == HIP_BRIDGE_F32) {
        if (xk == X_F32) ge ? launch_dense<QT, X_F32, true>(a, s) : launch_dense<QT, X_F32, false>(a, s);
        else if (xk == X_BF16) ge ? launch_dense<QT, X_BF16, true>(a, s) : launch_dense<QT, X_BF16, false>(a, s);
        else ge ? launch_dense<QT, X_TERMS, true>(a, s) : launch_dense<QT, X_TERMS, false>(a, s);
    } else {
        if (xk == X_F32) {
            ge ? launch_qt<QT, X_F32, true>(a, s) : launch_qt<QT, X_F32, false>(a, s);
        } else if (xk == X_TERMS) {
            ge ? launch_qt<QT, X_TERMS, true>(a, s) : launch_qt<QT, X_TERMS, false>(a, s);
        } else if constexpr (QT == HIP_BRIDGE_BF16) {
            ge ? launch_dense<QT, X_BF16, true>(a, s) : launch_dense<QT, X_BF16, false>(a, s);
        } else {
            ge ? launch_qt<QT, X_BF16, true>(a, s) : launch_qt<QT, X_BF16, false>(a, s);
        }
    }
}

// ---- small batches -----------------------------------------------------------------------------
// Products of a few tokens (f32 activations and output): a matrix-vector product's traffic, one
// read of the weights, with every weight used for up to 32 tokens. A wave takes RT tiles of 32
// rows over a share of the blocks, alone: weights and activations go from memory straight into
// its registers in operand layout, blocks ahead of their use, are converted there, and the waves
// of a workgroup add their sums through the LDS at the end, so there is no barrier in the loop and
// a wave's round trips overlap. Tokens past the batch repeat the last one.
// Up to 32 / P tokens leave the A operand's other rows free, and those hold the same tokens' other
// columns: P = 2 (16 tokens) the block's second MFMA's, P = 4 (8 tokens) the next block's too. An
// MFMA then gives its own sums in 32 / P of its rows (the rest is dropped), and a lane splits
// and loads 1 / P of the activations: their split, 5.5 vector instructions a value, is what
// bounds the kernel beside the weights' conversion, not the loads' latency: two groups of weights or
// four activation loads ahead are slower nearly everywhere (10240 x 2560 Q4_0, weights not in cache, 8 tokens
// 13.5 -> 14.3 / 15.1 us; 2560 x 10240 Q6_K, 45 tokens 45 -> 53 / 46).
// XK: f32 activations, or the same split beforehand (X_TERMS), which gives the same bits.
template <int QT, int XK, int P, int RT>
__global__ __launch_bounds__(512, 2) void k_gemm_skinny(GemmArgs a) {
    constexpr bool SCALED = w_scaled<QT>(), HALVES = QT == HIP_BRIDGE_Q6_K, MIN = QT == HIP_BRIDGE_Q4_K;
    constexpr int TOK = 32 / P, VR = 16 / P;  // tokens; accumulator registers of an MFMA's own rows
    constexpr int MAXW = 8;                   // the most waves
    __shared__ __attribute__((aligned(16))) float s_red[MAXW * RT * VR * kWave];
    const int lane = threadIdx.x & 63, h = lane >> 5, c = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), ks = (int)blockDim.x / kWave;
    const int r_base = (int)blockIdx.x * 32 * RT, t_base = (int)blockIdx.y * TOK;
    // The wave's groups of four blocks: its share of all of them, or with gridDim.z = 2 of half
    const int ng = a.cols / (4 * kKB);
    const int z0 = (int)((int64_t)ng * blockIdx.z / gridDim.z), z1 = (int)((int64_t)ng * (blockIdx.z + 1) / gridDim.z);
    const int g0 = z0 + (int)((int64_t)(z1 - z0) * wave / ks), g1 = z0 + (int)((int64_t)(z1 - z0) * (wave + 1) / ks);
    const int lastb = 4 * g1 - 1;

    // The lane's columns of a block (P = 4: of a pair of blocks): MFMA s takes xr[2 s], [2 s + 1]
    // (P = 1) or the only two, the MFMA (and block) given by the lane's row group c / TOK
    constexpr int XS = P == 1 ? 2 : 1, XB = P == 4 ? 2 : 1;  // MFMAs held apart; blocks per load
    const int sub = c / TOK;
    const int64_t xat = (int64_t)min(t_base + c % TOK, a.batch - 1) * a.cols + (P == 1 ? 0 : wk<QT>(sub & 1, h)) + 32 * (sub >> 1);
    constexpr int XL = XK == X_TERMS ? 3 : 2;  // 128-bit loads of an MFMA's columns: planes, or halves
    const unsigned char* const xrow = (const unsigned char*)a.x + xat * (XK == X_TERMS ? 2 : 4);
    const int64_t plane_bytes = (int64_t)a.batch * a.cols * 2;
    WSrc ws[RT];
#pragma unroll
    for (int j = 0; j < RT; ++j) ws[j].row = a.w + (int64_t)min(r_base + 32 * j + c, a.rows - 1) * a.row_bytes;
    using WQ = WGrp<QT>;
    constexpr int G = WQ::G, RING = G == 1 ? 4 : 1;
    WQ cur[RT], nxt[RING][RT];
    constexpr int UX = 2;  // activation loads ahead
    u32x4 xr[UX][XS][XL];
    auto load_x = [&](int kb, u32x4 (&r)[XS][XL]) {
        const int at = 32 * min(kb, lastb + 1 - XB);
#pragma unroll
        for (int s = 0; s < XS; ++s) {
            const int col = at + (P == 1 ? wk<QT>(s, h) : 0);
#pragma unroll
            for (int q = 0; q < XL; ++q)
                r[s][q] = XK == X_TERMS ? ld16(xrow + 2 * (int64_t)col + q * plane_bytes) : ld16(xrow + 4 * (int64_t)col + 16 * q);
        }
    };
    f32x16 acc[RT];
#pragma unroll
    for (int j = 0; j < RT; ++j) acc[j] = f32x16{};
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;
    // The row groups' sums over FG groups of blocks (a share of up to WHOLE at once: 10240 x 2560 Q4_0, 8 tokens,
    // 12.4 us in two sums, 11.9 in one) join a total in the LDS, so that a deep product's error does not
    // grow with the length of a wave's share (BF16: a compensated total, shorter sums;
    // 5376 x 21504 at 24 tokens 1.27e-7 off without, the vector kernel 1.14e-7).
    constexpr bool KAHAN = QT == HIP_BRIDGE_BF16;
    constexpr int FG = KAHAN ? 1 : 4, WHOLE = HALVES && P == 1 ? 3 : 6, OWN = RT * VR * kWave;
    __shared__ float s_lost[KAHAN ? MAXW * OWN : 1];
    float *const total = s_red + wave * OWN + lane, *const lost = s_lost + (KAHAN ? wave * OWN + lane : 0);
    auto flush = [&](bool first) {
#pragma unroll
        for (int j = 0; j < RT; ++j) {
#pragma unroll
            for (int r = 0; r < VR; ++r) {
                float v = acc[j][r];
#pragma unroll
                for (int i = 1; i < P; ++i) v += acc[j][i * VR + r];
                const int at = (j * VR + r) * kWave;
                float t = v, l = 0.0f;
                if (!first) {
                    t = total[at];
                    if (KAHAN) {
                        l = lost[at];
                        add_kahan(t, l, v);
                    } else {
                        t += v;
                    }
                }
                total[at] = t;
                if (KAHAN) lost[at] = l;
            }
            acc[j] = f32x16{};
        }
    };

    if (g0 < g1) {
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
            for (int b = 0; b < RING; ++b) nxt[b][j].load(ws[j], min(4 * g0 + b, lastb), h);
#pragma unroll
        for (int b = 0; b < UX; ++b) load_x(4 * g0 + XB * b, xr[b]);
    }
    bool first = true;
    int stop = !KAHAN && g1 - g0 <= WHOLE ? g1 : min(g0 + FG, g1);
    for (int g = g0; g < g1; ++g) {
        bf16x8 xa[XS][3];
        f32x16 sx;  // (MIN) each row's sum over its columns
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kb = 4 * g + u;
            bf16x8 wb[RT][2][1];
            float dv[RT][2], mn[RT];
#pragma unroll
            for (int j = 0; j < RT; ++j) {
                if (G == 1 || u == 0) {
                    cur[j] = nxt[G == 1 ? u : 0][j];
                    cur[j].open();
                    nxt[G == 1 ? u : 0][j].load(ws[j], G == 1 ? min(kb + 4, lastb) : min(4 * g + 4, 4 * g1 - 4), h);
                }
                const int un = G == 1 ? 0 : u;
                cur[j].scale(un, kb, dv[j], mn[j]);
                cur[j].template ops<0>(un, wb[j][0]);
                cur[j].template ops<1>(un, wb[j][1]);
            }
            if (u % XB == 0) {
                u32x4(&xv)[XS][XL] = xr[u / XB % UX];
#pragma unroll
                for (int s = 0; s < XS; ++s) {
                    uint32_t v[4][3];
                    if constexpr (XK == X_F32) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            split3(__uint_as_float(xv[s][i / 2][2 * (i & 1)]), __uint_as_float(xv[s][i / 2][2 * (i & 1) + 1]), v[i]);
                    }
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        xa[s][q] = __builtin_bit_cast(bf16x8, XK == X_F32 ? u32x4{v[0][q], v[1][q], v[2][q], v[3][q]} : xv[s][q % XL]);
                }
                load_x(kb + UX * XB, xv);
                if constexpr (MIN) {
#pragma unroll
                    for (int s = 0; s < XS; ++s)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            sx = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[s][q], ones, s + q ? sx : f32x16{}, 0, 0, 0);
                }
            }
            // Chains of MFMAs: both of the block's (P = 1 with one scale), or one each, of which
            // the registers [v0, v0 + VR) are its own
#pragma unroll
            for (int j = 0; j < RT; ++j) {
                f32x16 part;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const bool start = s == 0 || HALVES || P > 1;
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        part = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa[s % XS][q], wb[j][s][0],
                                                                       q == 0 && start ? f32x16{} : part, 0, 0, 0);
                    if (HALVES || P > 1 || s == 1) {
                        const int v0 = P == 1 ? 0 : VR * (P == 4 ? 2 * (u & 1) + s : s);
#pragma unroll
                        for (int r = v0; r < v0 + VR; ++r) {
                            if constexpr (MIN) acc[j][r] = fmaf(-mn[j], sx[r], acc[j][r]);
                            acc[j][r] = SCALED ? fmaf(dv[j][HALVES ? s : 0], part[r], acc[j][r]) : acc[j][r] + part[r];
                        }
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // (else the loads sink to their uses)
        }
        if (g + 1 == stop) {  // uniform
            flush(first);
            first = false;
            stop = min(stop + FG, g1);
        }
    }
    if (first) flush(true);  // (no groups)

    // The waves' sums, in a tree of two halves: w and w + half, then those in order.
    const int half = (ks + 1) / 2;
    __syncthreads();
    for (int i = threadIdx.x; i < RT * VR * kWave; i += (int)blockDim.x) {
        const int tile = i / (VR * kWave), r = i / kWave % VR, l = i % kWave;
        float v = 0.0f;
        for (int w = 0; w < half; ++w) {
            const float lo = s_red[w * (RT * VR * kWave) + i], hi = w + half < ks ? s_red[(w + half) * (RT * VR * kWave) + i] : 0.0f;
            v = w ? v + (lo + hi) : lo + hi;
        }
        // register r of lane l: token 8 (r / 4) + 4 (l / 32) + r % 4, row l % 32
        const int tok = t_base + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3);
        const int row = r_base + 32 * tile + (l & 31);
        if (tok >= a.batch || row >= a.rows) continue;
        if (XK == X_F32 && !(fabsf(v) < INFINITY))
            v = dot_columns<QT>(a.w + (int64_t)row * a.row_bytes, (const float*)a.x + (int64_t)tok * a.cols, 4 * kKB * z0,
                                4 * kKB * z1);
        float* const y = (float*)a.y + (int64_t)tok * a.rows + row;
        if (gridDim.z > 1) unsafeAtomicAdd(y, v);  // two halves into zeroed y: 0 + a + b in either order
        else *y = v;
    }
}

// Row tiles per wave, waves and K halves. n1, n2: workgroups at one and two row tiles. Measured, us
// (Q4_0 unless said): 10240 x 2560, 8 tokens: one tile and 4 / 8 waves 12.0 / 13.8, two tiles
// 13.0; 16 tokens 16.1 / 17.9, 15.2; 32 tokens 25.5 / 28.1, 20.1 (two tiles share a split of x,
// worth it once that is large). 2560 x 10240, two halves added into zeroed y: 8 tokens 15.0, one
// tile and no halves 20.3; 48 tokens 45.7, two tiles 35.5; at 128 tokens two tiles fill the chip
// without halves, 57.3 against 66.6. 2048 x 2560, 16 tokens: 4 / 8 waves 8.7 / 9.6, halves 8.9;
// 48 tokens 15.0, halves 12.3.
template <int QT, int XK>
static void launch_skinny_t(const GemmArgs& a, hipStream_t s) {
    const int ng = a.cols / (4 * kKB);
    const int p = a.batch > 16 ? 1 : a.batch > 8 ? 2 : 4;
    const int64_t ttiles = cdiv(a.batch, 32 / p), n1 = cdiv(a.rows, 32) * ttiles, n2 = cdiv(a.rows, 64) * ttiles;
    const bool deep = a.cols >= kSplitMinCols;
    const int rt = deep ? (n1 >= 160 ? 2 : 1) : (p < 4 && n2 >= 160 ? 2 : 1);
    const unsigned kz = (deep ? (rt == 2 ? n2 : n1) : p == 1 ? n1 : 1024) < 160 ? 2 : 1;
    const int most = rt == 1 && kz == 1 ? 4 : 8;
    const int half = (int)cdiv(ng, (int)kz), share = (int)cdiv(half, most);  // groups of a half, of a wave
    const int ks = (int)cdiv(half, share);
    if (kz > 1) launch_zero_f32((float*)a.y, (int64_t)a.batch * a.rows, s);
    const dim3 grid((unsigned)cdiv(a.rows, 32 * rt), (unsigned)ttiles, kz);
    auto go = [&](auto p_c) {
        constexpr int PC = decltype(p_c)::value;
        if (rt == 1) k_gemm_skinny<QT, XK, PC, 1><<<grid, ks * kWave, 0, s>>>(a);
        else k_gemm_skinny<QT, XK, PC, 2><<<grid, ks * kWave, 0, s>>>(a);
    };
    if (p == 1) go(std::integral_constant<int, 1>{});
    else if (p == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 4>{});
}

// Where k_gemm_skinny is the fastest path for f32 x and y: below it the vector kernels and
// k_gemv_mb, above it k_gemm_mfma, which takes over early where the rows alone fill the chip
// (gemm_mfma_min_batch). us, this kernel / the best other, at n rows x columns:
//   Q4_0, Q4_K, Q6_K: at least 8192 rows to 32 tokens (10240 x 2560: Q4_0 2 tokens 11.7 / 18.3, 24
//     19.4 / 23.5, 40 32.4 / 25.7; Q6_K 2 tokens 16.1 / 13.1, 4 16.3 / 21.4; 262144 x 2560 Q6_K 4
//     tokens 247 / 471; 21504 x 5376 Q4_0 2 tokens 40 / 23, 3 40 / 41); at least 5120 to 64 tokens (6144 x
//     1536 Q4_K 64: 16.4 / 21.0, 128 30.5 / 24.5); deep ones from 5 to 128 tokens (2560 x 10240 Q4_0 4
//     tokens 13.6 / 12.4, 8 15.0 / 21.1, 96 36.2 / 78.9; 1536 x 6144 Q4_0 8 tokens 11.2 / 10.3, 9 11.6 /
//     13.6); the rest from 9 tokens on 1536 rows (2048 x 2560: 2 tokens 7.2 / 7.3, 16 8.7 / 10.0, 80 15.6 /
//     20.9; 256 x 1536 10 / 6), but
//       Q4_K of up to 2047 rows 33 to 64 and from 96 (1536 x 2048: 32 11.4 / 9.6, 45 11.5 / 13.5, 80 15.5 /
//       13.5), to 2559 from 49 (2048 x 2560: 9 11.2 / 8.5, 45 13.0 / 11.5, 63 13.1 / 17.7), above from 10;
//       Q6_K of up to 2047 rows 9 to 16 and as Q4_K (1536 x 2048: 32 12.0 / 10.4, 45 12.2 / 16.8);
//       Q4_0 of up to 2048 short rows not where k_gemv_mb's second (third) 16-token tile fills up (1536 x
//       2048: 24 10.3 / 10.4, 32 11.2 / 10.5, 33 11.3 / 15.4; 2048 x 1536: 45 9.9 / 9.4, 63 9.9 / 14.0);
//   Q8_0 and BF16: deep products of 9 to 128 tokens (2560 x 10240 Q8_0 9 30 / 43); BF16, whose blocks
//     take a load each, of 17 to 32 from 2560 rows (1536 x 6144, 24 22.6 / 16.0; 2560 x 10240 32.8 / 37.3; 48
//     tokens 48.0 / 42.1) and of 64 to 128.
//   From 2560 rows all but the K-quants to 96 tokens (2560 x 10240 at 112: Q4_0 58 / 59, Q8_0 68 / 69, BF16
//     85 / 94, Q4_K 61 / 73, Q6_K 74 / 85, and from planes, six loads a block where f32 takes four, Q4_0 82 /
//     62, BF16 128 / 88; 5376 x 4096 at 128: Q4_0 53 / 42, BF16 78 / 43).
//   All but BF16 leave 25 to 32 tokens of at most 2048 rows of up to 176 blocks to k_gemv_mb, whose two
//     halves are shortest there (2048 x 5376 at 32 tokens: Q4_0 17.6 / 16.6, Q8_0 18.4 / 16.8, Q4_K 18.0 /
//     15.5; 24 15.5 / 16.9, 16.3 / 18.3, 16.2 / 15.5).
static bool skinny_range(int qtype, int rows, int cols, int batch) {
    const bool q4 = qtype == HIP_BRIDGE_Q4_0, q4k = qtype == HIP_BRIDGE_Q4_K, q6 = qtype == HIP_BRIDGE_Q6_K;
    if (rows < kWideRows && cols >= kSplitMinCols) {  // deep
        if (batch > (rows >= 2560 && !q4k && !q6 ? 96 : 128)) return false;
        if (qtype == HIP_BRIDGE_BF16) return (batch >= 17 && batch <= 32 && rows >= 2560) || batch >= 64;
        if (rows <= 2048 && cols <= 176 * kKB && batch >= 25 && batch <= 32 && !q6) return false;
        if (qtype == HIP_BRIDGE_Q8_0) return batch >= 9;
        return (q4 || q4k || q6) && batch >= (q4 && rows < 2048 ? 9 : 5);
    }
    if (!(q4 || q4k || q6)) return false;
    if (rows >= kMidRows) return batch >= (q6 || (q4 && cols > 5120) ? 3 : 2) && batch <= (rows >= kWideRows ? 32 : 64);
    if (rows < 1536 || batch < 9 || batch > 127) return false;
    if (q4) return !(rows <= 2048 && cols <= 2048 && batch >= 25 && batch <= (cols <= 1536 ? 48 : 32));
    if (rows < 2048) return (q6 && batch <= 16) || (batch >= 33 && batch <= 64) || batch >= 96;
    return q6 || batch >= (rows < 2560 ? 49 : 10);
}

// Small-batch product, f32 x (or its F32_TERMS planes) and f32 y; false: not a shape, type or batch
// of this kernel (nothing launched).
bool launch_gemm_skinny(int qtype, const void* w, int64_t row_bytes, int x_dtype, const void* x, float* y, int rows,
                        int cols, int batch, hipStream_t s) {
    const bool kq = qtype == HIP_BRIDGE_Q4_K || qtype == HIP_BRIDGE_Q6_K;
    const uintptr_t wa = reinterpret_cast<uintptr_t>(w);
    if (!skinny_range(qtype, rows, cols, batch) || !w || !x || !y) return false;
    if (!aligned16(x) || cols % (kq ? 256 : 4 * kKB) != 0 || wa % (qtype == HIP_BRIDGE_BF16 ? 16 : 2) != 0) return false;
    const GemmArgs a{(const unsigned char*)w, nullptr, x, y, row_bytes, rows, cols, batch, 0};
    const bool terms = x_dtype == HIP_BRIDGE_F32_TERMS;
    auto go = [&](auto q_c) {
        constexpr int QT = decltype(q_c)::value;
        terms ? launch_skinny_t<QT, X_TERMS>(a, s) : launch_skinny_t<QT, X_F32>(a, s);
    };
    switch (qtype) {
        case HIP_BRIDGE_Q4_0: go(std::integral_constant<int, HIP_BRIDGE_Q4_0>{}); break;
        case HIP_BRIDGE_Q8_0: go(std::integral_constant<int, HIP_BRIDGE_Q8_0>{}); break;
        case HIP_BRIDGE_BF16: go(std::integral_constant<int, HIP_BRIDGE_BF16>{}); break;
        case HIP_BRIDGE_Q4_K: go(std::integral_constant<int, HIP_BRIDGE_Q4_K>{}); break;
        default: go(std::integral_constant<int, HIP_BRIDGE_Q6_K>{}); break;
    }
    check_launch();
    return true;
}

// 0 = launched; otherwise why not (the caller decides between a fallback and an error).
int launch_gemm_mfma_ex(int qtype, const void* w, const void* wu, int64_t row_bytes, int x_dtype, const void* x,
                        int y_dtype, void* y, int rows, int cols, int batch, hipStream_t s) {
    const bool kq = qtype == HIP_BRIDGE_Q4_K || qtype == HIP_BRIDGE_Q6_K;
    const bool types = qtype == HIP_BRIDGE_Q4_0 || qtype == HIP_BRIDGE_Q8_0 || qtype == HIP_BRIDGE_F16 ||
                       qtype == HIP_BRIDGE_BF16 || qtype == HIP_BRIDGE_F32 || kq;
    if (!types || (x_dtype != HIP_BRIDGE_F32 && x_dtype != HIP_BRIDGE_BF16 && x_dtype != HIP_BRIDGE_F32_TERMS) ||
        (y_dtype != HIP_BRIDGE_F32 && y_dtype != HIP_BRIDGE_BF16))
        return HIP_BRIDGE_EUNSUPPORTED;
    // dense rows must be 16-byte aligned for the 128-bit loads; block rows need 2 bytes
    const bool dense = qtype == HIP_BRIDGE_F16 || qtype == HIP_BRIDGE_BF16 || qtype == HIP_BRIDGE_F32;
    auto w_ok = [&](const void* p) {
        const uintptr_t wa = reinterpret_cast<uintptr_t>(p);
        return dense ? (wa % 16 == 0 && row_bytes % 16 == 0) : (wa % 2 == 0);
    };
    if (cols % (kq ? 256 : kKB) != 0 || !aligned16(x) || !w_ok(w) || (wu && !w_ok(wu))) return HIP_BRIDGE_EUNSUPPORTED;
    // 32-bit byte offsets within a token tile's activations (per plane)
    if ((int64_t)128 * cols * (x_dtype == HIP_BRIDGE_F32 ? 4 : 2) > 0xffffffffLL) return HIP_BRIDGE_EUNSUPPORTED;
    const GemmArgs a{(const unsigned char*)w, (const unsigned char*)wu, x, y, row_bytes, rows, cols, batch,
                     y_dtype == HIP_BRIDGE_BF16};
    const int xk = x_dtype == HIP_BRIDGE_BF16 ? X_BF16 : x_dtype == HIP_BRIDGE_F32_TERMS ? X_TERMS : X_F32;
    const bool ge = wu != nullptr;
    switch (qtype) {
        case HIP_BRIDGE_Q4_0:
            if (cols % (4 * kKB) == 0) launch_q<HIP_BRIDGE_Q4_0>(a, xk, ge, s);
            else launch_q<kQ4_0Odd>(a, xk, ge, s);
            break;
        case HIP_BRIDGE_Q8_0:
            if (cols % (4 * kKB) == 0) launch_q<HIP_BRIDGE_Q8_0>(a, xk, ge, s);
            else launch_q<kQ8_0Odd>(a, xk, ge, s);
            break;
        case HIP_BRIDGE_F16: launch_q<HIP_BRIDGE_F16>(a, xk, ge, s); break;
        case HIP_BRIDGE_BF16: launch_q<HIP_BRIDGE_BF16>(a, xk, ge, s); break;
        case HIP_BRIDGE_Q4_K: launch_q<HIP_BRIDGE_Q4_K>(a, xk, ge, s); break;
        case HIP_BRIDGE_Q6_K: launch_q<HIP_BRIDGE_Q6_K>(a, xk, ge, s); break;
        default: launch_q<HIP_BRIDGE_F32>(a, xk, ge, s); break;
    }
    check_launch();
    return 0;
}

// x (f32) -> three bf16 planes h, m, l (h = bf16(x), m = bf16(x - h), l = bf16(x - h - m)):
// the activation form the K loop stages without converting. Four elements per thread.
__global__ __launch_bounds__(256) void k_split_terms(const float* __restrict__ x, uint16_t* __restrict__ planes,
                                                     int64_t n) {
    const int64_t i4 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;  // n % 4 == 0
    if (i4 >= n) return;
    const u32x4 v = lds16(x + i4);
    uint32_t t0[3], t1[3];
    split3(__uint_as_float(v.x), __uint_as_float(v.y), t0);
    split3(__uint_as_float(v.z), __uint_as_float(v.w), t1);
#pragma unroll
    for (int u = 0; u < 3; ++u) *reinterpret_cast<u32x2*>(planes + u * n + i4) = u32x2{t0[u], t1[u]};
}

bool launch_gemm_mfma(int qtype, const void* w, int64_t row_bytes, const float* x, float* y, int rows, int cols,
                      int batch, hipStream_t s) {
    if (batch < gemm_mfma_min_batch(qtype, rows, cols) || !y) return false;
    return launch_gemm_mfma_ex(qtype, w, nullptr, row_bytes, HIP_BRIDGE_F32, x, HIP_BRIDGE_F32, y, rows, cols, batch,
                               s) == 0;
}

}  // namespace zl

using namespace zl;

extern "C" void hip_split_terms(const float* x, void* planes, int64_t n, HipStream_t stream) {
    if (n <= 0) return;
    if (!x || !planes) {
        set_error(HIP_BRIDGE_EINVAL);
        return;
    }
    if (!aligned16(x) || (reinterpret_cast<uintptr_t>(planes) & 7u) || n % 4) {
        set_error(HIP_BRIDGE_EUNSUPPORTED);
        return;
    }
    k_split_terms<<<(unsigned)cdiv(n, 1024), 256, 0, stream_of(stream)>>>(x, (uint16_t*)planes, n);
    check_launch();
}
