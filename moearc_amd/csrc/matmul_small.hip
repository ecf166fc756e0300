// Chunk-form projections for a few tokens: Y[t][r] = sum_c W[r][c] X[t][c] (+ bias[r]) for at most 64
// tokens, straight from the f32 activations in one launch. Bound by latency: the products of matmul.hip
// split the activations in a launch before, cut the reduction over grid z with one k-block in flight
// per wave, and added the slices in a launch after. 8 tokens of Q8_0 4096 x 2880 (12.6 MB) went from
// 21.9 to 8.8 us, of MXFP4 28.0 to 8.4, of Q4_K 4096 x 2048 25.4 to 6.6.
//
// Work-group: 16 weight rows and all tokens; its 8 waves cut the reduction between them (whole
// super-blocks for the K-quants) and meet once, in LDS, at the end. A wave has CK k-blocks of both
// operands in flight beside the CK it computes. Lane (q, n) holds k 8q .. 8q + 7 of weight row n (B
// operand of v_mfma_f32_16x16x32_f16), as loaded, and of token n (A operand, f16 hi + lo). D then has
// the weight row in its column, so a block's scale is one per-lane factor. Every work-group reads all
// activations through the L2, which is why this form ends where the larger tiles begin (the host's
// rule).
//
// Precision is matmul.hip's: x = hi + lo to 2^-22, payloads as exact f16 integers (E2M1 code points
// for MXFP4), each block's f32 sum scaled in f32. The K-quants' mins multiply the block's f32 sum of x.
#include "common.h"

namespace {

typedef float mms_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 mms_half4 __attribute__((ext_vector_type(4)));

constexpr uint32_t MMS_WAVES = MOEARC_MM_SMALL_WAVES;

// the bytes of two dwords -> f16 byte - BIAS (exact: under exponent 0x64 a byte is 1024 + its value)
template <int BIAS>
__device__ __forceinline__ half8_t mms_bytes(uint32_t w0, uint32_t w1) {
    half8_t r;
    const uint32_t w[2] = {w0, w1};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const half2_t off = {(_Float16) (1024.f + BIAS), (_Float16) (1024.f + BIAS)};
        const half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, w[i], 0x04010400u)) - off;
        const half2_t b = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, w[i], 0x04030402u)) - off;
        r[4 * i] = a[0];
        r[4 * i + 1] = a[1];
        r[4 * i + 2] = b[0];
        r[4 * i + 3] = b[1];
    }
    return r;
}

// Weights arrive in windows of WB k-blocks, S bytes of each row, as 16-byte pieces (the last one ends
// on the window's last byte): load j of a lane takes piece 4 j + lane % 4 of row lane / 4, 64
// contiguous bytes per four lanes. The pieces reach LDS at 16 bytes each, RS bytes per row, and the
// lanes read their operands from there: byte o of a window is at o, or at o + 16 NP - S in the last
// piece.
template <uint32_t TY>
struct MmsFmt {
    static constexpr uint32_t WB = TY == 1 ? 4 : 8;
    static constexpr uint32_t S = WB * 32u / moearc_mv_be(TY) * moearc_mv_bb(TY);
    static constexpr uint32_t NP = (S + 15u) / 16u, NI = (NP + 3u) / 4u;
    static constexpr uint32_t LAST = 16u * NP - S;
    static constexpr uint32_t RS = 16u * NP + (NP % 2u ? 0u : 16u);
};

// The 8 bytes at row + off + 8 q, off known at compile time.
__device__ __forceinline__ void mms_get8(uint32_t &d0, uint32_t &d1, const uint8_t *row, uint32_t off, uint32_t q) {
    const uint32_t *p = (const uint32_t *) (row + (off & ~3u) + 8u * q);
    if ((off & 3u) == 0u) {
        d0 = p[0];
        d1 = p[1];
    } else {
        const uint32_t w0 = p[0], w1 = p[1], w2 = p[2];
        d0 = __builtin_amdgcn_alignbyte(w1, w0, off & 3u);
        d1 = __builtin_amdgcn_alignbyte(w2, w1, off & 3u);
    }
}

__device__ __forceinline__ float mms_f16(uint32_t bits) { return (float) __builtin_bit_cast(_Float16, (uint16_t) bits); }

// The B operand of a window's k-block i from the lane's row, and its factors: s0 (and, Q4_K and Q5_K,
// the min s1; Q6_K, the second group's s1).
template <uint32_t TY>
__device__ __forceinline__ half8_t mms_operand(const uint8_t *row, uint32_t i, uint32_t lq, float &s0, float &s1) {
    uint32_t q0, q1;
    s0 = s1 = 0.f;
    if constexpr (TY == 1) {
        return __builtin_bit_cast(half8_t, *(const u32x4_t *) (row + 64u * i + 16u * lq));
    } else if constexpr (TY == 8) {
        s0 = mms_f16(*(const uint16_t *) (row + 34u * i));
        mms_get8(q0, q1, row, 34u * i + 2u, lq);
        return mms_bytes<128>(q0 ^ 0x80808080u, q1 ^ 0x80808080u);
    } else if constexpr (TY == 39) {
        const uint32_t e = row[17u * i];
        s0 = __uint_as_float(e ? e << 23 : 0x00400000u);  // 2^(e - 127)
        mms_get8(q0, q1, row, 17u * i + 1u + (i == 7u ? MmsFmt<TY>::LAST : 0u), lq & 1u);  // block 7: the last piece
        const uint32_t q[2] = {q0, q1};
        half8_t r;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t x = (q[j] >> (4u * (lq >> 1))) & 0x0F0F0F0Fu;
            const uint32_t y = x | (x >> 4);  // pairs in bytes 0 and 2
            const half2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(y, 1.0f, 0);
            const half2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(y, 1.0f, 2);
            r[4 * j] = p0[0];
            r[4 * j + 1] = p0[1];
            r[4 * j + 2] = p1[0];
            r[4 * j + 3] = p1[1];
        }
        return r;
    } else if constexpr (TY == 12 || TY == 13) {  // sub-block i of the super-block
        const u32x4_t hd = *(const u32x4_t *) row;  // get_scale_min_k4 (reference.rs:150-160)
        const uint32_t sh8 = 8u * (i & 3u);
        const uint32_t a1 = hd[1] >> sh8, a2 = hd[2] >> sh8, a3 = hd[3] >> sh8;
        const uint32_t sc = i < 4u ? a1 & 63u : (a3 & 15u) | (((a1 >> 6) & 3u) << 4);
        const uint32_t mn = i < 4u ? a2 & 63u : ((a3 >> 4) & 15u) | (((a2 >> 6) & 3u) << 4);
        s0 = mms_f16(hd[0] & 0xFFFFu) * (float) sc;
        s1 = mms_f16(hd[0] >> 16) * (float) mn;
        mms_get8(q0, q1, row, (TY == 12 ? 16u : 48u) + 32u * (i >> 1), lq);
        const uint32_t sh = 4u * (i & 1u);
        q0 = (q0 >> sh) & 0x0F0F0F0Fu;
        q1 = (q1 >> sh) & 0x0F0F0F0Fu;
        if constexpr (TY == 13) {
            uint32_t h0, h1;
            mms_get8(h0, h1, row, 16u, lq);
            q0 |= ((h0 >> i) & 0x01010101u) << 4;
            q1 |= ((h1 >> i) & 0x01010101u) << 4;
        }
        return mms_bytes<0>(q0, q1);
    } else {  // Q6_K: k-block i = (half n, quarter c) of the super-block
        const uint32_t n = i >> 2, c = i & 3u, shl = 4u * (c >> 1), shh = 2u * c;
        uint32_t h0, h1;
        mms_get8(q0, q1, row, 64u * n + 32u * (c & 1u), lq);
        mms_get8(h0, h1, row, 128u + 32u * n, lq);
        const uint32_t sc = *(const uint16_t *) (row + 192u + 8u * n + 2u * c);
        const float d = mms_f16(*(const uint16_t *) (row + 208u + MmsFmt<TY>::LAST));
        s0 = d * (float) (int8_t) sc;
        s1 = d * (float) (int8_t) (sc >> 8);
        return mms_bytes<32>(((q0 >> shl) & 0x0F0F0F0Fu) | (((h0 >> shh) & 0x03030303u) << 4),
                             ((q1 >> shl) & 0x0F0F0F0Fu) | (((h1 >> shh) & 0x03030303u) << 4));
    }
}

__device__ __forceinline__ float4_t mms_mfma(half8_t a, half8_t b, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t mms_token(uint32_t q, uint32_t k) { return 2u * q + (k & 1u) + 8u * (k >> 1); }

// T tiles of 16 tokens, CK k-blocks per batch of activation loads.
template <uint32_t TY, int T, int CK>
__device__ __forceinline__ void mms_body(const MatmulArgs &a) {
    using F = MmsFmt<TY>;
    constexpr uint32_t WB = F::WB;
    constexpr bool Q45 = TY == 12 || TY == 13;
    static_assert(WB % (2 * CK) == 0, "activation batches alternate within a window");
    // per wave: a window of weights; a k-block's activations in f16, [tile][hi, lo][16-byte slots], and at
    // the end the wave's sums, [tile][token][row n]
    __shared__ __attribute__((aligned(16))) uint8_t wlds[MMS_WAVES][16 * F::RS];
    __shared__ u32x4_t xlds[MMS_WAVES][T][2][64];
    const auto red = [&](uint32_t w, uint32_t t) { return (float *) xlds[w][t]; };
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, lq = lane >> 4;
    const MmSegView sg = mm_seg(a, blockIdx.x);
    const uint32_t r0 = 16u * sg.tile;
    // this wave's k-blocks kb0 .. end (as kb0 < nb_all ? min(kb_per, nb_all - kb0) : 0 the compiler dropped
    // the comparison); the host sends rows of at least WB
    const uint32_t nb_all = a.cols / 32u, kb0 = min(wave * a.kb_per, nb_all), end = min(kb0 + a.kb_per, nb_all);

    const uint8_t *wsrc = sg.w + (uint64_t) min(r0 + (lane >> 2), sg.rows - 1u) * sg.row_bytes;
    u32x4_t wreg[F::NI];
    auto wload = [&](uint32_t b) {  // the window that starts at block b
        const uint8_t *p = wsrc + (uint64_t) b * 32u / moearc_mv_be(TY) * moearc_mv_bb(TY);
#pragma unroll
        for (uint32_t j = 0; j < F::NI; ++j)
            __builtin_memcpy(&wreg[j], p + min(16u * (4u * j + (lane & 3u)), F::S - 16u), 16);
    };
    auto wput = [&]() {
#pragma unroll
        for (uint32_t j = 0; j < F::NI; ++j)
            *(u32x4_t *) (wlds[wave] + F::RS * (lane >> 2) + 16u * min(4u * j + (lane & 3u), F::NP - 1u)) = wreg[j];
    };
    // activation loads take whole 128-byte lines: load e of tile t, lane l: token 16 t + 8 e + l / 8,
    // floats 4 (l % 8) .. + 3 of the block. (In operand layout, 16 rows per load and a row's lanes 16
    // apart, a load of either operand cost 58 clocks at the L1 whatever it fetched: only neighbouring
    // lanes' addresses are joined. 16 tokens of Q8_0 4096 x 2880 took 15.0 us that way.) They reach
    // operand layout through LDS, as f16: token u's 16-byte slot q (k 8 q .. + 7) at q ^ (u / 4). Row 4 q + k
    // of the A operand, and of D, is token mms_token(q, k) of its tile, so that the tokens whose sums a lane's D
    // rows need (Q4_K, Q5_K) are those that its 16 lanes loaded.
    const float *x[T][2];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 2; ++e)
            x[t][e] = a.xs + (uint64_t) min(16u * t + 8u * e + (lane >> 3), a.n_tok - 1u) * a.cols + 4u * (lane & 7u);
    uint32_t put[2];  // in 8-byte halves of a slot
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const uint32_t u = 8u * e + (lane >> 3), c = lane & 7u;
        put[e] = 2u * (4u * u + ((c >> 1) ^ (u >> 2))) + (c & 1u);
    }
    const uint32_t un = mms_token(n >> 2, n & 3u), get = 4u * un + (lq ^ (un >> 2));
    struct Batch {
        mms_f4 x[CK][T][2];
    };
    auto xload = [&](Batch &o, uint32_t b0) {
#pragma unroll
        for (int i = 0; i < CK; ++i) {
            const uint32_t b = min(b0 + i, nb_all - 1u);
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int e = 0; e < 2; ++e) o.x[i][t][e] = *(const mms_f4 *) (x[t][e] + 32u * b);
        }
    };
    float4_t acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    const uint8_t *const wrow = wlds[wave] + F::RS * n;
    // blocks i0 .. i0 + CK - 1 of the window at ws, those of lo .. end
    auto compute = [&](const Batch &o, uint32_t ws, uint32_t i0, uint32_t lo_b) {
#pragma unroll
        for (int i = 0; i < CK; ++i) {
            const uint32_t b = ws + i0 + i;
            if (b < lo_b || b >= end) continue;  // uniform
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    mms_half4 hi, lo;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float v = o.x[i][t][e][k];
                        hi[k] = (_Float16) v;
                        lo[k] = (_Float16) (v - (float) hi[k]);
                    }
                    ((mms_half4 *) xlds[wave][t][0])[put[e]] = hi;
                    ((mms_half4 *) xlds[wave][t][1])[put[e]] = lo;
                }
            float sum[T][2];  // Q4_K, Q5_K: token 8 e + lane / 8's sum, over its eight lanes
            if constexpr (Q45) {
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const mms_f4 &v = o.x[i][t][e];
                        float s = (v[0] + v[1]) + (v[2] + v[3]);
                        s += dpp<0xB1>(s);
                        s += dpp<0x4E>(s);
                        sum[t][e] = s + dpp<0x141>(s);
                    }
            }
            __builtin_amdgcn_wave_barrier();
            float s0, s1;
            const half8_t bw = mms_operand<TY>(wrow, i0 + i, lq, s0, s1);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const half8_t hi = __builtin_bit_cast(half8_t, xlds[wave][t][0][get]);
                const half8_t lo = __builtin_bit_cast(half8_t, xlds[wave][t][1][get]);
                if constexpr (TY == 1) {
                    acc[t] = mms_mfma(lo, bw, mms_mfma(hi, bw, acc[t]));
                } else if constexpr (TY == 14) {
                    // the two 16-wide scale groups: lanes of k 0 .. 15 and 16 .. 31
                    const half8_t none = {};
                    const half8_t b0w = lq < 2u ? bw : none, b1w = lq < 2u ? none : bw;
                    const float4_t g0 = mms_mfma(lo, b0w, mms_mfma(hi, b0w, zero));
                    const float4_t g1 = mms_mfma(lo, b1w, mms_mfma(hi, b1w, zero));
#pragma unroll
                    for (int k = 0; k < 4; ++k) acc[t][k] = fmaf(s1, g1[k], fmaf(s0, g0[k], acc[t][k]));
                } else {
                    const float4_t s = mms_mfma(lo, bw, mms_mfma(hi, bw, zero));
#pragma unroll
                    for (int k = 0; k < 4; ++k) acc[t][k] = fmaf(s0, s[k], acc[t][k]);
                    if constexpr (Q45) {
                        // rows 4 lq .. + 3 of D: the tokens of lanes 0-7 and 8-15 of this lane's 16
                        acc[t][0] = fmaf(dpp<0x150>(sum[t][0]), -s1, acc[t][0]);
                        acc[t][1] = fmaf(dpp<0x158>(sum[t][0]), -s1, acc[t][1]);
                        acc[t][2] = fmaf(dpp<0x150>(sum[t][1]), -s1, acc[t][2]);
                        acc[t][3] = fmaf(dpp<0x158>(sum[t][1]), -s1, acc[t][3]);
                    }
                }
            }
        }
    };
    if (kb0 < end) {
        // windows of WB blocks from kb0; one that would pass the row's end starts earlier, its first
        // blocks skipped
        Batch p, q;
        uint32_t ws = min(kb0, nb_all - WB);
        wload(ws);
        xload(p, ws);
        for (uint32_t b = kb0; b < end; b += WB) {
            const uint32_t next = min(b + WB, nb_all - WB);
            __builtin_amdgcn_wave_barrier();
            wput();
            __builtin_amdgcn_wave_barrier();
            wload(next);
#pragma unroll
            for (uint32_t i = 0; i < WB; i += 2 * CK) {
                xload(q, ws + i + CK);
                __builtin_amdgcn_sched_barrier(0);
                compute(p, ws, i, b);
                __builtin_amdgcn_sched_barrier(0);
                xload(p, i + 2 * CK < WB ? ws + i + 2 * CK : next);
                __builtin_amdgcn_sched_barrier(0);
                compute(q, ws, i + CK, b);
                __builtin_amdgcn_sched_barrier(0);
            }
            ws = next;
        }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) red(wave, t)[16u * mms_token(lq, k) + n] = acc[t][k];
    __syncthreads();
    // element e of tile t: token 16 t + e / 16, row r0 + e % 16, the waves' sums in order
    for (uint32_t i = tid; i < 256u * T; i += 64u * MMS_WAVES) {
        const uint32_t t = i >> 8, e = i & 255u, tok = 16u * t + (e >> 4), r = r0 + (e & 15u);
        float s = red(0, t)[e];
#pragma unroll
        for (uint32_t v = 1; v < MMS_WAVES; ++v) s += red(v, t)[e];
        if (tok < a.n_tok && r < sg.rows) {
            float *yp = sg.y + (uint64_t) tok * sg.y_stride + r;
            const float y = sg.bias ? s + sg.bias[r] : s;
            *yp = a.accumulate ? *yp + y : y;
        }
    }
}

}  // namespace

#define MATMUL_SMALL(NAME, TY, CK1)                                                                          \
    extern "C" __global__ void __launch_bounds__(64 * MMS_WAVES, 4) moearc_matmul_small_##NAME##_t1_k(MatmulArgs a) { \
        mms_body<TY, 1, CK1>(a);                                                                             \
    }                                                                                                        \
    extern "C" __global__ void __launch_bounds__(64 * MMS_WAVES, 4) moearc_matmul_small_##NAME##_t2_k(MatmulArgs a) { \
        mms_body<TY, 2, 2>(a);                                                                               \
    }                                                                                                        \
    extern "C" __global__ void __launch_bounds__(64 * MMS_WAVES, 2) moearc_matmul_small_##NAME##_t3_k(MatmulArgs a) { \
        mms_body<TY, 3, 1>(a);                                                                               \
    }                                                                                                        \
    extern "C" __global__ void __launch_bounds__(64 * MMS_WAVES, 2) moearc_matmul_small_##NAME##_t4_k(MatmulArgs a) { \
        mms_body<TY, 4, 1>(a);                                                                               \
    }

MATMUL_SMALL(q8_0, 8, 4)
MATMUL_SMALL(f16, 1, 2)
MATMUL_SMALL(q4_k, 12, 4)
MATMUL_SMALL(q5_k, 13, 4)
MATMUL_SMALL(mxfp4, 39, 4)
MATMUL_SMALL(q6_k, 14, 4)
