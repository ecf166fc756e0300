// Split-K single-query paged attention on gfx950 MFMA: f16 or f32 KV, head_dim 64 (the gpt-oss shape:
// 64 query heads over 8 KV heads) or 128 (Qwen3-30B-A3B: 32 over 4).
//
// Semantics are moearc_attn_decode's (kernels.cpp:1837-1919): for each query head,
//     out = sum_j e^(s_j - M) V_j / (e^(sink - M) + sum_j e^(s_j - M)),  s_j = scale * q.K_j,
// over the span [kv_begin, n_kv) read through the block table.
//
// Work decomposition. A work-group of KB x WPK wavefronts owns KB consecutive KV heads of one
// split (a run of split_len consecutive keys) of one sequence, and serves every query head of each
// KV head's group from a single read of each K/V row -- the KV bytes cross HBM once, not once per
// query head. The split is walked in chunks of WPK * TILES 32-key tiles; wave (kl, sub) takes KV
// head kl and the sub-th run of TILES consecutive tiles of every chunk, so the work-group reads
// KB * 128 contiguous bytes of every key row of the chunk. A wave issues every load of its chunk
// (TILES tiles, 8 x 16 bytes per lane each) before it computes any of them: at TILES = 4 that is
// 32 KiB per wave in flight, and with 8 waves per CU the whole 256 KiB share of a CU in a 32K-key
// call is requested one block-table round trip after launch. The waves merge in LDS; a sequence
// whose span fits one split is finished there (sink applied, output written); otherwise each
// work-group writes per-head partial records (max, denominator, unnormalised output) and
// moearc_attn_decode_merge, the next launch on the stream, combines them.
//
// Per 32-key tile (one wave), all operands in registers, no LDS. For f16 and 64 channels (the other
// kinds differ in operand types and in P.V; see F16D128 and F32Kv):
//   loads   K and V rows go from HBM straight into MFMA A-operand layout: lane (g, m) loads 16
//           bytes, channels 8g..8g+7 (and 32+8g..) of key 16*blk + m.
//   QK^T    S^T[32 keys x 16 heads] = K . Q^T, 2 key blocks x 2 channel halves of
//           v_mfma_f32_16x16x32_f16. Q is split q = q_hi + q_lo into two f16 operands (after an
//           exact power-of-two normalisation), so the products see q to ~22 bits; K is exact f16.
//   softmax lane (g, n) holds head n's scores for keys 16*blk + 4g + r. exp2 with scale*log2(e)
//           folded into one multiplier; running max across the four lanes of a head.
//   V^T     the P.V product needs V with keys along the MFMA reduction axis. Multiplying the
//           natural-layout V block by a 0/1 selection matrix on the MFMA unit returns it in the
//           accumulator layout -- lane (g, n) gets channel n of keys 4g..4g+3 -- which is exactly
//           the A-operand layout P.V needs. Exact: each output is one f16 value times 1 plus zeros.
//   P.V     O^T[64 x 16] += V^T[64 x 32] . P^T[32 x 16], P^T straight from the softmax registers,
//           split p = p_hi + p_lo like q.
// Heads beyond the group (columns 8..15 when the group is 8) are computed and discarded: MFMA
// time is not the bound here, HBM is.
//
// The 128-channel and f32 kinds took the general kernel (decode_general.hip) before, a work-group per
// query head with neither splits nor a shared KV read: four sequences of 2K-8K keys at 32 heads over
// 4 KV heads of 128 f16 channels (34 MB) went from 2360 to 14.8 µs, 17 of 2K-30K reach 4.8 TB/s
// (123 µs, a large copy's rate), eight of 3K-30K over f32 caches 5.2-5.4 TB/s (106.6 and 112 µs).
// Their error against float64 is a quarter of that kernel's (2.8e-7 against 1.2e-6).
//
// Kernel arguments: the fields the first loads depend on (KV and block-table bases, q, sequence
// 0's span and split, the geometry) lead the argument list as scalars, which the dispatcher
// preloads into SGPRs (the code object is built with kernarg preloading), so the block-table
// loads leave with no kernel-argument round trip before them; the rest follows as a struct read
// on demand.
#include "common.h"

// Scores live in the log2 domain, x = scale * log2(e) * q.K. Probabilities enter the f16 MFMA
// operands as p * 2^LOG2_PSCALE relative to a per-head reference max m_ref that is only moved
// when a tile's max exceeds it by more than RESCALE_SLACK (the running sums are then rescaled
// once); so p * 2^7 <= 2^(7 + 8) = 32768 stays inside f16, and p_lo (the f16 residual of p_hi)
// stays a normal f16 down to p ~ 2^-10 of the reference, with a 2^-31 floor below that.
#define LOG2_PSCALE 7.0f
#define RESCALE_SLACK 8.0f

__device__ __forceinline__ float4_t mfma16(const half8_t a, const half8_t b, const float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ half8_t as_half8(const u32x4_t v) { return __builtin_bit_cast(half8_t, v); }

__device__ __forceinline__ float wave_max_16_32(float x) {
    x = fmaxf(x, __shfl_xor(x, 16));
    x = fmaxf(x, __shfl_xor(x, 32));
    return x;
}

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// What the running maximum of a head starts from where a key of -inf scores -inf (the 128-channel and f32
// kinds): below any score in the log2 domain, and finite, so that a first tile of such keys leaves weights of
// 0 and not NaN. The 64-channel f16 kind starts from -inf: its scores are finite or NaN, and its registers
// fall out the better for it (32 sequences of 1K-32K 207.8 -> 207.0 us, eight of 128K 377.6 -> 376.6).
#define M_START -3.0e38f

template <int NO>
struct SoftmaxState {
    float m;         // reference max (log2 domain), uniform over the 4 lanes of a head
    float l;         // running denominator in the m-frame, partial over this lane's keys
    float4_t O[NO];  // unnormalised output in the m-frame, in the kind's accumulator order
};

// The softmax of one 32-key tile: S[blk] lane (g, n) element i is the raw score of key
// j0 + 16 blk + 4g + i for head n, c the multiplier into the log2 domain. Moves the reference when
// it must and turns S into the weights * 2^LOG2_PSCALE.
template <int NO>
__device__ __forceinline__ void softmax_tile(SoftmaxState<NO> &st, float4_t (&S)[2], float c, uint32_t j0,
                                             uint32_t te, uint32_t g) {
    if (j0 + 32u > te) {  // the span's last, partial tile (uniform branch)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (j0 + 16u * (i >> 2) + 4u * g + (i & 3) >= te) S[i >> 2][i & 3] = -INFINITY;
    }
    float tmax = fmaxf(fmaxf(fmaxf(S[0][0], S[0][1]), fmaxf(S[0][2], S[0][3])),
                       fmaxf(fmaxf(S[1][0], S[1][1]), fmaxf(S[1][2], S[1][3])));
    tmax = wave_max_16_32(tmax) * c;
    // Move the reference only when some head's max outgrew it by more than the slack.
    if (__builtin_amdgcn_ballot_w64(tmax > st.m + RESCALE_SLACK) != 0) {
        const float m_new = fmaxf(st.m, tmax);
        const float corr = exp2_fast(st.m - m_new);  // first tile: exp2 of -inf or a huge negative, 0
        st.m = m_new;
        st.l *= corr;
#pragma unroll
        for (int mb = 0; mb < NO; ++mb) st.O[mb] *= corr;
    }
    const float bias = LOG2_PSCALE - st.m;
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float ps = exp2_fast(fmaf(S[i >> 2][i & 3], c, bias));
        psum += ps;
        S[i >> 2][i & 3] = ps;
    }
    st.l += psum;
}

// A head's q, normalised by a power of two (exact) so that a split into f16 pieces does not depend on
// the head's magnitude, and the score multiplier with that power folded in.
template <int NQ>
struct SplitQuery {
    float c;
    float v[8 * NQ];
    // lane (g, n): channels 32 i + 8 g .. + 7 of head n, 0 for columns past the group
    __device__ __forceinline__ void load(const float *q, uint32_t group, uint32_t dim, uint32_t g, uint32_t n) {
        const bool head_ok = n < group;
        const float *const qrow = q + (head_ok ? n : 0u) * dim;
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const float4_t x0 = *(const float4_t *) (qrow + 32 * i + 8 * g);
            const float4_t x1 = *(const float4_t *) (qrow + 32 * i + 8 * g + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[8 * i + e] = head_ok ? x0[e] : 0.f;
                v[8 * i + 4 + e] = head_ok ? x1[e] : 0.f;
            }
        }
    }
    // qexp and c for q 2^(top - qexp), whose largest channel is in [2^(top - 1), 2^top)
    __device__ __forceinline__ int normalise(float scale_log2e, int top) {
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < 8 * NQ; ++i) amax = fmaxf(amax, fabsf(v[i]));
        amax = wave_max_16_32(amax);
        int qexp = 0;
        if (amax > 0.f && amax < INFINITY) (void) frexpf(amax, &qexp);
        c = ldexpf(scale_log2e, qexp - top);  // score multiplier in the log2 domain
        return qexp;
    }
};

// ---- f16 cache, 64 channels ----------------------------------------------------------------------
struct F16D64 {
    static constexpr int D = 64, NO = 4, Q_LDS = 0;
    static constexpr float M0 = -INFINITY;
    using Elem = uint16_t;
    struct Tile {
        u32x4_t k[2][2];  // [key block][channel half], A-operand layout
        u32x4_t v[2][2];
    };
    struct Query : SplitQuery<2> {
        // q = hi + lo: 22 bits of the channels down to 2^-3 of the head's largest, 2^-25 of it below
        half8_t hi[2], lo[2];
        half8_t sel[2];  // selection operands: sel[s] lane (g, n) item i = 1 where 8g + i == 16s + n
        __device__ __forceinline__ void ready(float scale_log2e, uint32_t g, uint32_t n, uint32_t *) {
            const int qexp = normalise(scale_log2e, 1);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = ldexpf(v[8 * i + e], 1 - qexp);
                    const _Float16 h = (_Float16) x;
                    hi[i][e] = h;
                    lo[i][e] = (_Float16) (x - (float) h);
                }
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    sel[s][i] = (8u * g + i == 16u * s + n) ? (_Float16) 1.0f : (_Float16) 0.0f;
        }
    };
    // row[blk]: the physical row of this lane's key 16 blk + m16
    static __device__ __forceinline__ void load(Tile &r, const uint32_t (&row)[2], const Elem *k_pages,
                                                const Elem *v_pages, uint64_t row_elems, uint32_t kvh, uint32_t g,
                                                uint32_t) {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const uint64_t off = (uint64_t) row[blk] * row_elems + (uint64_t) kvh * 64u + 8u * g;
            const uint16_t *ks = k_pages + off;
            const uint16_t *vs = v_pages + off;
            r.k[blk][0] = *(const u32x4_t *) ks;
            r.k[blk][1] = *(const u32x4_t *) (ks + 32);
            r.v[blk][0] = *(const u32x4_t *) vs;
            r.v[blk][1] = *(const u32x4_t *) (vs + 32);
        }
    }
    static __device__ __forceinline__ void tile(SoftmaxState<NO> &st, Tile &r, const Query &q, uint32_t j0,
                                                uint32_t te, uint32_t g, uint32_t) {
        float4_t S[2];
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            float4_t s = (float4_t){0.f, 0.f, 0.f, 0.f};
            s = mfma16(as_half8(r.k[blk][0]), q.hi[0], s);
            s = mfma16(as_half8(r.k[blk][0]), q.lo[0], s);
            s = mfma16(as_half8(r.k[blk][1]), q.hi[1], s);
            s = mfma16(as_half8(r.k[blk][1]), q.lo[1], s);
            S[blk] = s;
        }
        softmax_tile(st, S, q.c, j0, te, g);
        half8_t phi, plo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float ps = S[i >> 2][i & 3];
            const _Float16 hi = (_Float16) ps;
            phi[i] = hi;
            plo[i] = (_Float16) (ps - (float) hi);
        }
        // V^T via the selection product, then P.V, one 16-channel block at a time
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
            const int hf = mb >> 1, sl = mb & 1;
            const float4_t z = (float4_t){0.f, 0.f, 0.f, 0.f};
            const float4_t t0 = mfma16(as_half8(r.v[0][hf]), q.sel[sl], z);  // keys 4g+i
            const float4_t t1 = mfma16(as_half8(r.v[1][hf]), q.sel[sl], z);  // keys 16+4g+i
            half8_t va;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                va[i] = (_Float16) t0[i];
                va[4 + i] = (_Float16) t1[i];
            }
            st.O[mb] = mfma16(va, phi, st.O[mb]);
            st.O[mb] = mfma16(va, plo, st.O[mb]);
        }
    }
    // O[mb] lane (g, n) element i: channel 16 mb + 4 g + i of head n
    static __device__ __forceinline__ void put(float *row, const SoftmaxState<NO> &st, uint32_t g) {
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) *(float4_t *) (row + 16u * mb + 4u * g) = st.O[mb];
    }
};

// Row numbers of the keys a lane takes of V (16 blk + 4 g + r): lane 4 g + r holds key 4 g + r's.
__device__ __forceinline__ uint32_t v_row(const uint32_t (&row)[2], int blk, uint32_t g, int r) {
    return __shfl(row[blk], (int) (4u * g + r));
}

// ---- f16 cache, 128 channels: HBM-bound like the 64-channel kind, 512 bytes per key and KV head.
// Scores as there, but with q whole in three f16 operands per 32 channels, q = hi + mid / 2^11 +
// lo / 2^22, each with sums of its own: f32's 24 bits for every channel down to 2^-28 of the head's
// largest (the general kernel multiplies in f32; two pieces kept about 7 bits of a channel 2^18 below the
// largest). FOLD, for groups of up to 8 heads: lo takes the idle columns 8 .. 15 of hi's product, so the
// third piece costs neither an MFMA nor a register. (In f32 MFMAs instead, four sequences of 2K-8K keys
// take 17.4 us for 15.7, and their 32-step chains err by 4.2e-7 for 2.5e-7.) For P.V, lane (g, m) loads channels
// 8 m .. 8 m + 7 of key 16 blk + 4 g + r: a 16-lane group reads a whole 256-byte row, and element e
// of the 16 lanes, widened to f32, is the A operand of a 16x16x4 f32 MFMA over keys {4 g + r} whose
// B operand is the softmax register r as it stands: no transposition, weights in f32, at the price of
// 4x the matrix time of the f16 product, which still leaves the matrix cores over half idle at the
// HBM rate.
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

template <bool FOLD_>
struct F16D128 {
    static constexpr bool FOLD = FOLD_;
    static constexpr float M0 = M_START;
    static constexpr int D = 128, NO = 8, Q_LDS = 256 * 4 * (FOLD ? 2 : 3) + 16;  // dwords: q's operands, the heads' c
    using Elem = uint16_t;
    struct Tile {
        u32x4_t k[2][4];  // [key block][channel quarter]
        u32x4_t v[2][4];  // [key block][r]: channels 8 m .. of key 4 g + r
    };
    // The four waves work for one KV head and make its operands together: a thread takes 4 channels of one
    // head, the 32 threads of a head share its largest channel, and the pieces meet in LDS. That is one
    // coalesced load; in operand layout, eight per wave of 64 scattered pieces each, q's loads and the third
    // piece's arithmetic in every wave cost more: four sequences of 2K-8K keys 15.9 us with the mid and low
    // pieces in LDS, 17.9 with FOLD, 14.8 this way (15.4 with two pieces), eight of 200-2000 13.0 -> 12.6.
    // At one query head per KV head, where the scattered load had one row to fetch, up to 2.5% longer.
    struct Query {
        static constexpr int ROUNDS = FOLD ? 1 : 2, PARTS = FOLD ? 2 : 3;  // heads / 8; hi (and lo), mid; or hi, mid, lo
        float c;
        float4_t raw[ROUNDS];
        half8_t hi[4], mid[FOLD ? 4 : 1];
        const half8_t *rest;  // !FOLD: mid and lo of 32 channels at [192 i], [192 i + 64], in LDS (registers would spill)
        bool own;             // FOLD: a column of the heads' hi and mid
        __device__ __forceinline__ void load(const float *q, uint32_t group, uint32_t, uint32_t, uint32_t) {
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const uint32_t head = 8u * r + (threadIdx.x >> 5);
                const float4_t x = *(const float4_t *) (q + min(head, group - 1u) * 128u + 4u * (threadIdx.x & 31u));
                raw[r] = head < group ? x : (float4_t){0.f, 0.f, 0.f, 0.f};
            }
        }
        __device__ __forceinline__ void ready(float scale_log2e, uint32_t g, uint32_t n, uint32_t *lds) {
            half4_t *const parts = (half4_t *) lds;       // 8-byte halves of the operands' 16-byte slots
            float *const c_of = (float *) (lds + Q_LDS - 16);
            const uint32_t d8 = threadIdx.x & 31u;        // channels 4 d8 .. + 3: slot [d8 / 8][part][d8 / 2 % 4], half d8 % 2
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                const uint32_t head = 8u * r + (threadIdx.x >> 5);
                float amax = fmaxf(fmaxf(fabsf(raw[r][0]), fabsf(raw[r][1])), fmaxf(fabsf(raw[r][2]), fabsf(raw[r][3])));
                amax = fmaxf(amax, dpp<0xB1>(amax));   // quads: lanes 1 0 3 2, then 2 3 0 1
                amax = fmaxf(amax, dpp<0x4E>(amax));
                amax = fmaxf(amax, dpp<0x141>(amax));  // eight lanes mirrored, then sixteen
                amax = fmaxf(amax, dpp<0x140>(amax));
                amax = fmaxf(amax, __shfl_xor(amax, 16));
                int qexp = 0;
                if (amax > 0.f && amax < INFINITY) (void) frexpf(amax, &qexp);
                if (d8 == 0u) c_of[head] = ldexpf(scale_log2e, qexp - 15);
                half4_t h, m, l;
#pragma unroll
                for (int e = 0; e < 4; ++e) {  // below 65504; the remainders are exact in f32
                    const float x = ldexpf(raw[r][e], 15 - qexp);
                    h[e] = (_Float16) x;
                    const float rem = (x - (float) h[e]) * 2048.f;
                    m[e] = (_Float16) rem;
                    l[e] = (_Float16) ((rem - (float) m[e]) * 2048.f);
                }
                const auto put = [&](uint32_t part, uint32_t column, const half4_t &v) {
                    parts[2u * (64u * (PARTS * (d8 >> 3) + part) + 16u * ((d8 >> 1) & 3u) + column) + (d8 & 1u)] = v;
                };
                put(0u, head, h);
                put(1u, head, m);
                if constexpr (FOLD) put(0u, head + 8u, l);  // (mid's columns past 8 hold anything, and are dropped)
                else put(2u, head, l);
            }
            // LDS alone is waited for: the first chunk's loads stay in flight
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            const half8_t *const at = (const half8_t *) lds + (16u * g + n);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                hi[i] = at[64 * PARTS * i];
                if constexpr (FOLD) mid[i] = at[64 * PARTS * i + 64];
            }
            rest = at + 64;
            own = n < 8u;
            c = c_of[FOLD ? n & 7u : n];
        }
    };
    static __device__ __forceinline__ void load(Tile &r, const uint32_t (&row)[2], const Elem *k_pages,
                                                const Elem *v_pages, uint64_t row_elems, uint32_t kvh, uint32_t g,
                                                uint32_t m16) {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const uint16_t *ks = k_pages + ((uint64_t) row[blk] * row_elems + (uint64_t) kvh * 128u + 8u * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) r.k[blk][i] = *(const u32x4_t *) (ks + 32 * i);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                r.v[blk][i] = *(const u32x4_t *) (v_pages + ((uint64_t) v_row(row, blk, g, i) * row_elems +
                                                             (uint64_t) kvh * 128u + 8u * m16));
        }
    }
    static __device__ __forceinline__ void tile(SoftmaxState<NO> &st, Tile &r, const Query &q, uint32_t j0,
                                                uint32_t te, uint32_t g, uint32_t) {
        float4_t S[2] = {}, t[2] = {}, u[2] = {};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                const half8_t k = as_half8(r.k[blk][i]);
                S[blk] = mfma16(k, q.hi[i], S[blk]);
                if constexpr (FOLD) {
                    t[blk] = mfma16(k, q.mid[i], t[blk]);
                } else {
                    t[blk] = mfma16(k, q.rest[192 * i], t[blk]);
                    u[blk] = mfma16(k, q.rest[192 * i + 64], u[blk]);
                }
            }
        // an infinite key (f16 overflow at the append) scores by q.hi's sign alone
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float s = S[i >> 2][i & 3];
            const float lo = FOLD ? dpp<0x128>(s) : u[i >> 2][i & 3];  // (rotated by 8 columns)
            const float full = fabsf(s) == INFINITY ? s : fmaf(fmaf(lo, 0x1p-11f, t[i >> 2][i & 3]), 0x1p-11f, s);
            S[i >> 2][i & 3] = !FOLD || q.own ? full : 0.f;
        }
        softmax_tile(st, S, q.c, j0, te, g);
        if (j0 + 32u > te) {  // keys past the span repeat its last row: weight 0, and no 0 * inf either
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (j0 + 16u * (i >> 2) + 4u * g + (i & 3) >= te) r.v[i >> 2][i & 3] = (u32x4_t){0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int blk = 0; blk < 2; ++blk)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const half8_t v = as_half8(r.v[blk][i]);
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    st.O[e] = __builtin_amdgcn_mfma_f32_16x16x4f32((float) v[e], S[blk][i], st.O[e], 0, 0, 0);
            }
    }
    // O[e] lane (g, n) element i: channel 8 (4 g + i) + e of head n
    static __device__ __forceinline__ void put(float *row, const SoftmaxState<NO> &st, uint32_t g) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
                *(float4_t *) (row + 32u * g + 8u * i + 4u * hf) =
                    (float4_t){st.O[4 * hf][i], st.O[4 * hf + 1][i], st.O[4 * hf + 2][i], st.O[4 * hf + 3][i]};
    }
};

// ---- f32 cache, 64 or 128 channels: everything in f32, on 16x16x4 f32 MFMAs. Both contractions
// take each lane's 16-byte loads as they come, four channels apart per instruction: scores with
// lane (g, m) holding channels 16 i + 4 g .. + 3 of key m, outputs with channels 64 hf + 4 m .. + 3
// of key 4 g + r (whole 256-byte row pieces per 16 lanes). 32 MFMAs per 16 keys and 64 channels:
// the matrix cores could take about three times the HBM rate.
template <int D_>
struct F32Kv {
    static constexpr float M0 = M_START;
    static constexpr int D = D_, NO = D / 16, NK = D / 16, NV = D / 64, Q_LDS = 0;
    using Elem = float;
    struct Tile {
        float4_t k[2][NK];     // [key block][16 channels]
        float4_t v[2][4][NV];  // [key block][r][64 channels]
    };
    struct Query {
        float4_t v[NK];  // lane (g, n): channels 16 i + 4 g .. + 3 of head n
        float c;
        __device__ __forceinline__ void load(const float *q, uint32_t group, uint32_t, uint32_t g, uint32_t n) {
            const bool head_ok = n < group;
            const float *const qrow = q + (head_ok ? n : 0u) * D;
#pragma unroll
            for (int i = 0; i < NK; ++i) {
                const float4_t x = *(const float4_t *) (qrow + 16 * i + 4 * g);
                v[i] = head_ok ? x : (float4_t){0.f, 0.f, 0.f, 0.f};
            }
        }
        __device__ __forceinline__ void ready(float scale_log2e, uint32_t, uint32_t, uint32_t *) { c = scale_log2e; }
    };
    static __device__ __forceinline__ void load(Tile &r, const uint32_t (&row)[2], const Elem *k_pages,
                                                const Elem *v_pages, uint64_t row_elems, uint32_t kvh, uint32_t g,
                                                uint32_t m16) {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const float *ks = k_pages + ((uint64_t) row[blk] * row_elems + (uint64_t) kvh * D + 4u * g);
#pragma unroll
            for (int i = 0; i < NK; ++i) r.k[blk][i] = *(const float4_t *) (ks + 16 * i);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float *vs = v_pages + ((uint64_t) v_row(row, blk, g, i) * row_elems + (uint64_t) kvh * D + 4u * m16);
#pragma unroll
                for (int hf = 0; hf < NV; ++hf) r.v[blk][i][hf] = *(const float4_t *) (vs + 64 * hf);
            }
        }
    }
    static __device__ __forceinline__ void tile(SoftmaxState<NO> &st, Tile &r, const Query &q, uint32_t j0,
                                                uint32_t te, uint32_t g, uint32_t) {
        float4_t S[2];
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            float4_t s = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NK; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s = __builtin_amdgcn_mfma_f32_16x16x4f32(r.k[blk][i][e], q.v[i][e], s, 0, 0, 0);
            S[blk] = s;
        }
        softmax_tile(st, S, q.c, j0, te, g);
        if (j0 + 32u > te) {  // keys past the span repeat its last row: weight 0, and no 0 * inf either
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int hf = 0; hf < NV; ++hf)
                    if (j0 + 16u * (i >> 2) + 4u * g + (i & 3) >= te)
                        r.v[i >> 2][i & 3][hf] = (float4_t){0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int blk = 0; blk < 2; ++blk)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int hf = 0; hf < NV; ++hf)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        st.O[4 * hf + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.v[blk][i][hf][e], S[blk][i],
                                                                                st.O[4 * hf + e], 0, 0, 0);
    }
    // O[4 hf + e] lane (g, n) element i: channel 64 hf + 4 (4 g + i) + e of head n
    static __device__ __forceinline__ void put(float *row, const SoftmaxState<NO> &st, uint32_t g) {
#pragma unroll
        for (int hf = 0; hf < NV; ++hf)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *(float4_t *) (row + 64u * hf + 16u * g + 4u * i) =
                    (float4_t){st.O[4 * hf][i], st.O[4 * hf + 1][i], st.O[4 * hf + 2][i], st.O[4 * hf + 3][i]};
    }
};

// The fixed record array of the allocation-free entry point (moearc_attn_decode_batched_noalloc):
// partial records live here instead of in the context's workspace. Each loaded instance of the code
// object -- one per context, on that context's device -- holds its own array for the life of the
// module; the host takes its device address from the module (hipModuleGetGlobal, the module form of
// hipGetSymbolAddress) once, at context creation, and passes that address to the kernels like any
// workspace. External linkage so the module can name it; nothing else refers to it. Nothing in it
// needs clearing: a call's merge reads only records its own split kernel wrote.
__device__ __align__(256) float moearc_decode_scratch[MOEARC_DECODE_SCRATCH_FLOATS];

// Agent-scope relaxed atomic stores for the partial records: global_store with sc1, written
// through to the device-coherent level, so the kernel-end release has no dirty L2 lines of them
// to write back.
__device__ __forceinline__ void st_agent(float *p, float v) {
    __hip_atomic_store((uint32_t *) p, __builtin_bit_cast(uint32_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Final normalisation with the sink (kernels.cpp:1864-1880), in the log2 domain and the m-frame:
// out = O 2^(M-Mt) / (L 2^(M-Mt) + 2^(sink*log2e - Mt + LOG2_PSCALE)), Mt = max(M, sink*log2e).
__device__ __forceinline__ float finish(float sink2, float M, float L, float acc) {
    const float Mt = fmaxf(M, sink2);
    const float fm = exp2_fast(M - Mt);
    const float den = L * fm + exp2_fast(sink2 - Mt + LOG2_PSCALE);
    return acc * fm / den;
}

__device__ __forceinline__ void store_out(void *out, uint32_t out_f16, uint64_t o, float r) {
    if (out_f16) ((_Float16 *) out)[o] = (_Float16) r;
    else ((float *) out)[o] = r;
}

// The split kernel. Geometry words: geo0 = pt_shift | MOEARC_DECODE_UNIFORM if every sequence has the
// same number of items | MOEARC_DECODE_MANY past 24 sequences | n_kv_heads << 16, geo1 = nkb | group << 16,
// nkb being the KV-head blocks (of KB heads) per work item.
template <class P, int KB, int WPK, int TILES>
__device__ __forceinline__ void decode_body(const typename P::Elem *k_pages, const typename P::Elem *v_pages,
                                            const uint32_t *bt0, const float *q0, uint32_t kvb0,
                                            uint32_t nkv0, uint32_t slen0, uint32_t next0,
                                            uint32_t geo0, uint32_t geo1, const DecodeArgs &a) {
    constexpr int WAVES = KB * WPK;
    constexpr uint32_t D = P::D;
    constexpr uint32_t CHUNK = 32u * TILES * WPK;  // keys of one chunk of the split
    // a head's D partial outputs per row, rows D + 4 floats apart: the float4 writes of a 16-lane pass
    // (16 heads, one channel quad each) then fall on 64 distinct banks (a stride of D floats put all
    // 16 heads on the same 16 banks)
    constexpr uint32_t OROW = D + 4u;
    __shared__ __attribute__((aligned(16))) float o_lds[WAVES][16 * OROW];
    __shared__ float m_lds[WAVES][16];
    __shared__ float l_lds[WAVES][16];
    __shared__ __attribute__((aligned(16))) uint32_t q_lds[P::Q_LDS ? P::Q_LDS : 1];
    static_assert(!P::Q_LDS || (KB == 1 && WPK == 4), "four waves that share q");

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t sh = geo0 & (MOEARC_DECODE_MANY - 1u), G = geo0 >> 16;
    const uint32_t nkb = geo1 & 0xFFFFu, group = geo1 >> 16;
    const uint32_t kbi = blockIdx.x % nkb;
    const uint32_t item = blockIdx.x / nkb;
    // Sequence 0 comes from the preloaded arguments; later sequences search the struct.
    uint32_t b = 0, ib = 0, next = next0, kvb = kvb0, nkv = nkv0;
    const uint32_t *bt = bt0;
    const float *qb = q0;
    if (item >= next) {
        // Where every sequence has as many splits as sequence 0 (windows: one), the item's number gives
        // the sequence; else a walk along item_begin, 40 ns per sequence of a chain that ends in the first
        // loads: 32 windows of 128 keys 6.07 -> 4.90 us, 24 at 128 channels 8.08 -> 7.43. (A lane per
        // sequence and a ballot, one vector round trip, lost up to 1.1 us to the walk at 2-24 ragged
        // sequences of 128 channels.)
        if (geo0 & MOEARC_DECODE_UNIFORM) {
            b = next0 == 1u ? item : item / next0;
            ib = b * next0;
            next = ib + next0;
            kvb = a.kv_begin[b];
            nkv = a.n_kv[b];
        } else {
            if (geo0 & MOEARC_DECODE_MANY) {
                // Past 24 sequences the walk's length outweighs two trips to the scalar cache, eight entries
                // each: every eighth, then the group's. 32 sequences of 200-2000 keys (graph replay)
                // 27.5 -> 26.5 us, 60: 37.4 -> 36.5; 8 and 17 lost 0.5-1% to the walk.
                static_assert(MOEARC_MAX_SEQS_PER_LAUNCH == 64, "eight groups of eight sequences");
                uint32_t g = 0;
#pragma unroll
                for (uint32_t i = 1; i < 8u; ++i) g += item >= a.item_begin[8u * i];
                b = 8u * g;
#pragma unroll
                for (uint32_t i = 1; i < 8u; ++i) b += item >= a.item_begin[8u * g + i];
            } else {
                do ++b; while (item >= a.item_begin[b + 1]);
            }
            ib = a.item_begin[b];
            next = a.item_begin[b + 1];
            kvb = a.kv_begin[b];
            nkv = a.n_kv[b];
        }
        bt = a.block_tables + (uint64_t) b * a.bt_stride;
        qb = a.q + (uint64_t) b * G * group * D;
    }
    const uint32_t split = item - ib;
    const uint32_t nsplit = next - ib;
    const uint32_t tb = kvb + split * slen0;
    const uint32_t te = min(nkv, tb + slen0);
    const uint32_t kl = wave % KB, sub = wave / KB;
    const uint32_t kvh_raw = kbi * KB + kl;
    const bool kvh_ok = kvh_raw < G;
    const uint32_t kvh = min(kvh_raw, G - 1u);
    const uint32_t g = lane >> 4, n = lane & 15u, m16 = lane & 15u;
    const bool head_ok = kvh_ok && n < group;
    const uint64_t row_elems = (uint64_t) G * D;
    const uint32_t pmask = (1u << sh) - 1u;

    // Block-table entries of this lane's keys in TILES tiles from key jw (j = jw + 32t + 16blk +
    // m16, clamped into the span: a tile past the span repeats its last key and computes to
    // nothing), then the physical rows once they have arrived.
    auto pages_of = [&](uint32_t jw_, uint32_t (&pid)[TILES][2]) {
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) pid[t][blk] = bt[min(jw_ + 32u * t + 16u * blk + m16, te - 1u) >> sh];
    };
    auto load_chunk = [&](uint32_t jw_, typename P::Tile (&r)[TILES], const uint32_t (&pid)[TILES][2]) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            uint32_t row[2];
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                const uint32_t j = min(jw_ + 32u * t + 16u * blk + m16, te - 1u);
                row[blk] = (pid[t][blk] << sh) | (j & pmask);
            }
            P::load(r[t], row, k_pages, v_pages, row_elems, kvh, g, m16);
        }
    };

    SoftmaxState<P::NO> st;
    st.m = P::M0;
    st.l = 0.f;
#pragma unroll
    for (int mb = 0; mb < P::NO; ++mb) st.O[mb] = (float4_t){0.f, 0.f, 0.f, 0.f};
    uint32_t jw = tb + 32u * TILES * sub;   // this wave's first tile
    const bool active = kvh_ok && jw < te;  // uniform per wave
    if (active) {
        // ---- start-up: q and the first chunk's block-table entries leave together; the chunk's KV
        // loads leave as soon as the entries arrive, before the q arithmetic.
        typename P::Query q;
        q.load(qb + (uint64_t) kvh * group * D, group, D, g, n);
        uint32_t pid[TILES][2];
        pages_of(jw, pid);
        typename P::Tile r[TILES];
        load_chunk(jw, r, pid);
        __builtin_amdgcn_sched_barrier(0);
        q.ready(a.scale_log2e, g, n, q_lds);

        // ---- key loop: every load of a chunk is issued before any of its tiles is computed, and
        // the next chunk's block-table entries leave before the computing starts. (The compiler
        // drains the next chunk's KV loads at the back edge; they were all issued together, so the
        // first tile would wait for nearly as long anyway.)
        for (;;) {
            const uint32_t jn = jw + CHUNK;
            const bool more = jn < te;  // uniform
            pages_of(more ? jn : jw, pid);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < TILES; ++t) P::tile(st, r[t], q, jw + 32u * t, te, g, n);
            if (!more) break;
            jw = jn;
            load_chunk(jw, r, pid);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else if constexpr (P::Q_LDS != 0) {  // a wave without keys makes its share of q and meets the others
        typename P::Query q;
        q.load(qb + (uint64_t) kvh * group * D, group, D, g, n);
        q.ready(a.scale_log2e, g, n, q_lds);
    }

    // ---- merge the WPK waves of each KV head in LDS ---------------------------------------------
    float l_run = st.l;
    l_run += __shfl_xor(l_run, 16);
    l_run += __shfl_xor(l_run, 32);
    if (head_ok) P::put(&o_lds[wave][n * OROW], st, g);
    if (g == 0) {
        m_lds[wave][n] = head_ok && active ? st.m : -INFINITY;
        l_lds[wave][n] = head_ok && active ? l_run : 0.f;
    }
    __syncthreads();

    // Threads take (KV head of the block, output element) pairs.
    const uint32_t n_out = group * D;
    const bool single = nsplit == 1u;
    const uint32_t H = G * group;
    for (uint32_t idx = threadIdx.x; idx < KB * n_out; idx += 64u * WAVES) {
        const uint32_t k2 = idx / n_out, e = idx - k2 * n_out;
        const uint32_t kv2 = kbi * KB + k2;
        if (kv2 >= G) break;
        const uint32_t hn = e / D, d = e % D;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < WPK; ++w) M = fmaxf(M, m_lds[w * KB + k2][hn]);
        float L = 0.f, acc = 0.f;
#pragma unroll
        for (int w = 0; w < WPK; ++w) {
            const uint32_t ww = w * KB + k2;
            const float mw = m_lds[ww][hn];
            const float f = mw == -INFINITY ? 0.f : exp2_fast(mw - M);  // a wave without keys drops out
            L += l_lds[ww][hn] * f;
            acc += o_lds[ww][hn * OROW + d] * f;
        }
        const uint32_t hh = kv2 * group + hn;
        if (single) {
            const float sink2 = a.sinks ? a.sinks[hh] * MOEARC_LOG2E : -INFINITY;
            store_out(a.out, a.out_f16, ((uint64_t) b * H + hh) * D + d, finish(sink2, M, L, acc));
        } else {
            // records, head-major: [head][work item], so a head's splits are contiguous
            const uint64_t r_i = (uint64_t) hh * a.n_items + item;
            st_agent(a.rec_o + r_i * D + d, acc);
            if (d == 0) {
                st_agent(a.rec_ml + 2u * r_i, M);
                st_agent(a.rec_ml + 2u * r_i + 1u, L);
            }
        }
    }
}

#define DECODE_KERNEL(NAME, P, KB, WPK, TILES, WAVES_EU)                                       \
    extern "C" __global__ __launch_bounds__(64 * KB * WPK, WAVES_EU) void                     \
        moearc_attn_decode_##NAME##_k##KB##w##WPK##t##TILES(                                   \
            const P::Elem *k_pages, const P::Elem *v_pages, const uint32_t *bt0,               \
            const float *q0, uint32_t kvb0, uint32_t nkv0, uint32_t slen0, uint32_t next0,     \
            uint32_t geo0, uint32_t geo1, const DecodeArgs a) {                                \
        decode_body<P, KB, WPK, TILES>(k_pages, v_pages, bt0, q0, kvb0, nkv0, slen0, next0,    \
                                       geo0, geo1, a);                                         \
    }

// Long spans: 8 waves, 32 KiB of K and V per wave in flight. Short spans: 4 waves on one KV head,
// 128-key chunks, many work-groups. The last number is the least waves per SIMD (the 128-channel
// f32 kind holds a 32 KiB tile per wave either way).
DECODE_KERNEL(f16d64, F16D64, 4, 2, 4, 2)
DECODE_KERNEL(f16d64, F16D64, 1, 4, 1, 4)
DECODE_KERNEL(f16d128, F16D128<true>, 1, 4, 1, 3)
DECODE_KERNEL(f16d128g16, F16D128<false>, 1, 4, 1, 3)
DECODE_KERNEL(f32d64, F32Kv<64>, 4, 2, 2, 2)
DECODE_KERNEL(f32d64, F32Kv<64>, 1, 4, 1, 4)
DECODE_KERNEL(f32d128, F32Kv<128>, 4, 2, 1, 2)
DECODE_KERNEL(f32d128, F32Kv<128>, 1, 4, 1, 2)

// (m, l, o) of two partial softmax sums over disjoint key sets, combined in the frame of the
// larger max; a side that saw no keys has m = -inf and drops out.
__device__ __forceinline__ void merge_partial4(float &m, float &l, float4_t &o, float m2, float l2,
                                               float4_t o2) {
    const float M = fmaxf(m, m2);
    const float f1 = m == -INFINITY ? 0.f : exp2_fast(m - M);
    const float f2 = m2 == -INFINITY ? 0.f : exp2_fast(m2 - M);
    m = M;
    l = l * f1 + l2 * f2;
    o = o * f1 + o2 * f2;
}

// Split merge. One 256-thread work-group per (query head, sequence) (one measured as fast as four
// at config 2's 128 splits, and a quarter of the work-groups): lane (split group sg, channel quad
// c4) owns channels 4c4..4c4+3 for the splits sg, sg + NSG, ...; it issues every load of a round (a
// 16-byte piece of each of MERGE_BATCH records and their (max, denominator) pairs) before using
// any, so up to NSG * MERGE_BATCH splits cost one memory round trip, and a head's records are
// contiguous. The split groups then combine by shuffles within a wave and through LDS across the
// four waves.
// Arguments: record bases, output, sinks and sequence 0's item count are preloaded scalars; the
// struct carries the other sequences' item ranges.
#define MERGE_BATCH 8

template <uint32_t D>
__device__ __forceinline__ void merge_body(const float *rec_o, const float *rec_ml, void *out,
                                           const float *sinks, uint32_t n_items, uint32_t next0,
                                           uint32_t n_heads, uint32_t out_f16, const MergeArgs &ma) {
    constexpr uint32_t QUADS = D / 4, NSG = MOEARC_MERGE_THREADS / QUADS;
    __shared__ float red[4][6][QUADS];  // [wave][m, l, o0..o3][channel quad]
    const uint32_t tid = threadIdx.x, c4 = tid % QUADS, sg = tid / QUADS, wave = tid >> 6;
    const uint32_t b = blockIdx.y, h = blockIdx.x;
    uint32_t ib0 = 0, ib1 = next0;
    if (b > 0) {
        ib0 = ma.item_begin[b];
        ib1 = ma.item_begin[b + 1];
    }
    const uint32_t nsplit = ib1 - ib0;
    if (nsplit <= 1u) return;  // finished by the split kernel itself
    // the sink, requested with the records and first used at the end (without sinks the load reads
    // a record word, ignored)
    const float sink_raw = *(sinks ? sinks + h : rec_ml);
    const uint32_t ch = 4u * c4;
    const uint64_t base = (uint64_t) h * n_items + ib0;
    float m_t = -INFINITY, l_t = 0.f;
    float4_t o_t = (float4_t){0.f, 0.f, 0.f, 0.f};
    for (uint32_t s0 = sg; s0 < nsplit; s0 += NSG * MERGE_BATCH) {
        float4_t v[MERGE_BATCH];
        float2_t ml[MERGE_BATCH];
#pragma unroll
        for (int k = 0; k < MERGE_BATCH; ++k) {
            const uint64_t s = base + min(s0 + NSG * (uint32_t) k, nsplit - 1u);
            v[k] = *(const float4_t *) (rec_o + s * D + ch);
            ml[k] = *(const float2_t *) (rec_ml + 2u * s);
        }
        __builtin_amdgcn_sched_barrier(0);  // every load of the round leaves before any is used
        float mr = m_t;
#pragma unroll
        for (int k = 0; k < MERGE_BATCH; ++k) mr = fmaxf(mr, ml[k][0]);  // duplicates are harmless
        const float corr = m_t == -INFINITY ? 0.f : exp2_fast(m_t - mr);
        l_t *= corr;
        o_t *= corr;
#pragma unroll
        for (int k = 0; k < MERGE_BATCH; ++k) {
            const bool live = s0 + NSG * (uint32_t) k < nsplit;
            const float f = live ? exp2_fast(ml[k][0] - mr) : 0.f;
            l_t = fmaf(ml[k][1], f, l_t);
            o_t += v[k] * f;
        }
        m_t = mr;
    }
    // the split groups of this wave (lanes equal modulo QUADS)
#pragma unroll
    for (uint32_t x = QUADS; x < 64u; x <<= 1) {
        float4_t o2;
#pragma unroll
        for (int i = 0; i < 4; ++i) o2[i] = __shfl_xor(o_t[i], x);
        merge_partial4(m_t, l_t, o_t, __shfl_xor(m_t, x), __shfl_xor(l_t, x), o2);
    }
    if ((tid & 63u) < QUADS) {
        red[wave][0][c4] = m_t;
        red[wave][1][c4] = l_t;
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][2 + i][c4] = o_t[i];
    }
    __syncthreads();
    if (tid < QUADS) {
#pragma unroll
        for (int w = 1; w < 4; ++w)
            merge_partial4(m_t, l_t, o_t, red[w][0][c4], red[w][1][c4],
                           (float4_t){red[w][2][c4], red[w][3][c4], red[w][4][c4], red[w][5][c4]});
        const float sink2 = sinks ? sink_raw * MOEARC_LOG2E : -INFINITY;
        const uint64_t o = ((uint64_t) b * n_heads + h) * D + ch;
        float r4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r4[i] = finish(sink2, m_t, l_t, o_t[i]);
        if (out_f16) {
            half2_t lo = {(_Float16) r4[0], (_Float16) r4[1]}, hi = {(_Float16) r4[2], (_Float16) r4[3]};
            *(half2_t *) ((_Float16 *) out + o) = lo;
            *(half2_t *) ((_Float16 *) out + o + 2) = hi;
        } else {
            *(float4_t *) ((float *) out + o) = (float4_t){r4[0], r4[1], r4[2], r4[3]};
        }
    }
}

#define MERGE_KERNEL(D)                                                                        \
    extern "C" __global__ __launch_bounds__(MOEARC_MERGE_THREADS) void                        \
        moearc_attn_decode_merge_d##D(const float *rec_o, const float *rec_ml, void *out,      \
                                      const float *sinks, uint32_t n_items, uint32_t next0,    \
                                      uint32_t n_heads, uint32_t out_f16, const MergeArgs ma) { \
        merge_body<D>(rec_o, rec_ml, out, sinks, n_items, next0, n_heads, out_f16, ma);        \
    }

MERGE_KERNEL(64)
MERGE_KERNEL(128)
