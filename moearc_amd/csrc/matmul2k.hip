// Chunk-form projections on v_mfma_f32_32x32x16_f16 for Q4_K and Q5_K weights: matmul2.hip's tiles,
// copies and operand order (its helpers are used here), with a super-block as the unit of scaling.
//
// A weight is d * sc * q - dmin * m: d and dmin f16 per super-block of 256, sc and m 6-bit integers
// per sub-block of 32, q 4 or 5 bits. sc * q is an integer of at most 63 * 31 = 1953 < 2048, exact in
// f16, so it is the matrix operand itself, and products of several sub-blocks add up in the matrix cores
// before d scales them. The operand costs what q alone did: the 0x64 exponent trick gives 1024 + q, and
// one packed f16 multiply-add, (1024 + q) * sc - 1024 * sc, exact, replaces the subtraction. The mins,
// sum over sub-blocks of m * (sum of x), are two 32x32x16 MFMAs per super-block and tile too: of the
// 8 sub-blocks' activation sums in four f16 pieces, sum / 64 = v0 + v1 / 2^11 + v2 / 2^22 + v3 / 2^33
// (moearc_split_sums_k), two side by side in a 16-wide k: v2 and v3 against m / 2^12 and m / 2^23, then v0
// and v1 against 2^10 m and m / 2, all exact in f16. v0 and v1 are 0 rather than subnormal (the matrix cores
// align a subnormal operand as if it were 2^-14, and its low bits drop out), so the pieces hold an f32 sum
// whole down to 2^-19, its first 23 bits down to 2^-30.
//
// What bounds it: with a scale and a min per sub-block (128 f32 multiply-adds per 16 MFMAs and wave,
// and 16-byte LDS reads of the sums for the mins) the vector unit did: 14.7 instructions per MFMA, issued for
// 46% of the cycles with the matrix cores busy for 25%. It is 6.8, 32% and 38% now (2048 tokens).
// Whole calls, split and sums included: 4096 x 2048 Q4_K over 2048 tokens 126 -> 96 us, over 1000 78 -> 56,
// over 128 28.8 -> 24.4; Q5_K 2048 x 4096 over 300 44 -> 34. The mins in two pieces and one MFMA, to 2^-23 of
// a sum, were 1.0-1.5% faster.
//
// Sums of a pair of sub-blocks go to the accumulators, d applied: the f32 rounding of the matrix cores'
// running sum grows with its length. Relative error against float64 (1000 tokens of N(0, 1), 2048
// columns): 2.4e-7 with a scale per sub-block; 1.9e-7 by pairs, and, with the mins in two pieces, 2.0e-7 by
// pairs, 2.2e-7 by four, 2.8e-7 by super-blocks, each twice as long about 1% faster. The low halves of the
// activations are multiplied first, while the sum is still small (2.1e-7 by pairs in hi, lo order).
#include "common.h"

namespace {

// LDS: three activation buffers as in matmul2.hip; two buffers of a pair of sub-blocks' 32 payload
// bytes per row (low nibbles: the first sub-block); two of a super-block's header per row (d, dmin,
// the 12 scale bytes; Q5_K: and the 32 bytes of fifth bits); one super-block's sums per token (v0 and v1; v2 and v3).
template <uint32_t TY, uint32_t KS = 1>  // KS: as mm2_body's
__device__ __forceinline__ void mm2k_body(const MatmulArgs &a) {
    constexpr bool Q5K = TY == 13;
    constexpr uint32_t SB = Q5K ? 176u : 144u, QS = Q5K ? 48u : 16u;  // super-block bytes, offset of its nibbles
    constexpr uint32_t HDR = Q5K ? 48u : 16u, NHDR = Q5K ? 2u : 1u;   // header bytes per row, copies per wave
    constexpr uint32_t PAIR = MM2_ROWS * 32u;
    constexpr uint32_t PAIR0 = MM2_NBUF * MM2_ACT, HDR0 = PAIR0 + 2u * PAIR, SUM0 = HDR0 + 2u * MM2_ROWS * HDR;
    constexpr uint32_t LDS = SUM0 + 2u * MM2_TOK * 32u;
    __shared__ __attribute__((aligned(1024))) uint8_t tiles[KS * LDS];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t group = KS == 2 ? wave8 >> 2 : 0u, wave = wave8 - 4u * group;
    const uint32_t n = lane & 31u, h = lane >> 5;
    const MmSegView sg = mm_seg(a, blockIdx.x);
    const uint32_t t0 = blockIdx.y * MM2_TOK, r0 = sg.tile * MM2_ROWS;
    // this work-group's k-slice: whole super-blocks, k-blocks kb0 .. kb0 + nb
    const Mm2Span span = mm2_span<KS, 8>(a, group);
    const uint32_t kb0 = span.kb0, nb = span.nb, nsb = nb >> 3;
    const uint32_t lds_all =
        __builtin_amdgcn_readfirstlane((uint32_t) (uintptr_t) (__attribute__((address_space(3))) uint8_t *) tiles);
    const uint32_t lds0 = lds_all + group * LDS;

    // ---- copy sources. Activations as in matmul2.hip: instruction i of wave w fills region R = 4 w + i.
    const uint16_t *xsrc[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t R = 4u * wave + i, tok = 16u * (R & 7u) + (lane >> 2);
        xsrc[i] = ((R >> 3) ? a.xl : a.xh) + (uint64_t) min(t0 + tok, a.n_tok - 1u) * a.cols + 32u * kb0 +
                  8u * ((lane & 3u) ^ mm2_swz(tok));
    }
    // Payload pairs and sums: slot q = 64 wave + lane is row (token) q / 2's 16-byte chunk
    // (q & 1) ^ ((q >> 4) & 1). Rows and tokens past the last repeat it.
    const uint32_t prow = (64u * wave + lane) >> 1, pchunk = (lane & 1u) ^ ((prow >> 3) & 1u);
    const uint64_t sb0 = SB * (uint64_t) (kb0 >> 3);
    const uint8_t *psrc = sg.w + (uint64_t) min(r0 + prow, sg.rows - 1u) * sg.row_bytes + sb0 + QS + 16u * pchunk;
    const uint8_t *ssrc = (const uint8_t *) a.xs + ((uint64_t) min(t0 + prow, a.n_tok - 1u) * (a.cols >> 8) + (kb0 >> 3)) * 64u +
                          16u * pchunk;
    // Headers: Q4_K row 64 (w & 1) + lane (waves 2 and 3 repeat 0 and 1); Q5_K instruction i of wave w
    // fills slots 64 min(2 w + i, 5) .. + 63, slot q being row q / 3's chunk q % 3.
    auto hslot = [&](uint32_t i) { return Q5K ? 64u * min(2u * wave + i, 5u) : 64u * (wave & 1u); };
    const uint8_t *hsrc[NHDR];
#pragma unroll
    for (uint32_t i = 0; i < NHDR; ++i) {
        const uint32_t q = hslot(i) + lane, r = Q5K ? q / 3u : q;
        hsrc[i] = sg.w + (uint64_t) min(r0 + r, sg.rows - 1u) * sg.row_bytes + sb0 + (Q5K ? 16u * (q % 3u) : 0u);
    }
    auto at = [&](uint32_t off) { return __builtin_amdgcn_readfirstlane(lds0 + off); };
    auto copy_act = [&](uint32_t b, uint32_t bufo) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) mm2_copy16(at(bufo + (4u * wave + i) * 1024u), xsrc[i] + 32u * b);
    };
    auto copy_pair = [&](uint32_t b, uint32_t par) {  // b even: of sub-blocks b and b + 1
        mm2_copy16(at(PAIR0 + par * PAIR + wave * 1024u), psrc + SB * (uint64_t) (b >> 3) + 16u * (b & 7u));
    };
    auto copy_hdr = [&](uint32_t s, uint32_t par) {
#pragma unroll
        for (uint32_t i = 0; i < NHDR; ++i)
            mm2_copy16(at(HDR0 + par * (MM2_ROWS * HDR) + 16u * hslot(i)), hsrc[i] + SB * (uint64_t) s);
    };

    // ---- operand addresses (activation buffer 0, pair buffer 0, header buffer 0)
    uint32_t aoff[2][2], poff[2], hoff[2], soff[2];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t tok = 64u * (wave & 1u) + 32u * i + n, rl = 64u * (wave >> 1) + 32u * i + n;
#pragma unroll
        for (uint32_t s = 0; s < 2; ++s) aoff[i][s] = lds0 + tok * 64u + 16u * ((2u * h + s) ^ mm2_swz(tok));
        poff[i] = lds0 + PAIR0 + 32u * rl + 16u * (h ^ ((rl >> 3) & 1u));
        hoff[i] = lds0 + HDR0 + HDR * rl;
        soff[i] = lds0 + SUM0 + 32u * tok + 16u * (h ^ ((tok >> 3) & 1u));
    }
    mm2_f32x16 acc[2][2], S[2][2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[tt][rt][j] = 0.f;

    copy_hdr(0u, 0u);
    copy_pair(0u, 0u);
    copy_act(0u, 0u);
    copy_act(1u, MM2_ACT);
    uint32_t bufo = 0u;              // k-block b's activation buffer, b % 3, as an offset
    for (uint32_t sb = 0; sb < nsb; ++sb) {
        const uint32_t hpar = sb & 1u;
        uint32_t dd[2], sc[2][2], mn[2][2];  // d | dmin << 16, the scales and mins of sub-blocks 0-3 and 4-7, one per byte
        u32x4_t kq[2];
        // Step k-block b = 8 sb + j: its copies have landed in every wave and every wave has read k-block
        // b - 1 (one barrier); request k-block b + 2 into b - 1's buffer, j even: the next pair, j = 1:
        // this super-block's sums, j = 4: the next super-block's header (past the end the last ones
        // again, which nothing reads); compute. In flight at step j: what step j - 1 requested.
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            const uint32_t b = 8u * sb + j;
            __builtin_amdgcn_sched_barrier(0);
            if (j == 5u) __builtin_amdgcn_s_waitcnt(mm2_vmcnt_lgkm0(5u + NHDR));
            else if (j == 2u) __builtin_amdgcn_s_waitcnt(mm2_vmcnt_lgkm0(6u));
            else if (j % 2u == 1u) __builtin_amdgcn_s_waitcnt(mm2_vmcnt_lgkm0(5u));
            else __builtin_amdgcn_s_waitcnt(mm2_vmcnt_lgkm0(4u));
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t prev = bufo == 0u ? 2u * MM2_ACT : bufo - MM2_ACT;
            copy_act(min(b + 2u, nb - 1u), prev);
            if (j % 2u == 0u) copy_pair(min(b + 2u, nb - 2u), ((j >> 1) + 1u) & 1u);
            if (j == 1u)
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i)
                    mm2_copy16(at(SUM0 + i * MM2_TOK * 32u + wave * 1024u), ssrc + 64u * (uint64_t) sb + 32u * i);
            if (j == 4u) copy_hdr(min(sb + 1u, nsb - 1u), hpar ^ 1u);
            __builtin_amdgcn_sched_barrier(0);

            half8_t ah[2][2], al[2][2], bw[2][2];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    ah[tt][s] = __builtin_bit_cast(half8_t, mm2_lds16(aoff[tt][s] + bufo));
                    al[tt][s] = __builtin_bit_cast(half8_t, mm2_lds16(aoff[tt][s] + bufo + MM2_HALF));
                }
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                if (j == 0u) {  // get_scale_min_k4 (reference.rs:150-160), four sub-blocks to a dword
                    const u32x4_t hd = mm2_lds16(hoff[rt] + hpar * (MM2_ROWS * HDR));
                    dd[rt] = hd[0];
                    sc[rt][0] = hd[1] & 0x3F3F3F3Fu;
                    mn[rt][0] = hd[2] & 0x3F3F3F3Fu;
                    sc[rt][1] = (hd[3] & 0x0F0F0F0Fu) | ((hd[1] >> 2) & 0x30303030u);
                    mn[rt][1] = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
                }
                if (j % 2u == 0u) kq[rt] = mm2_lds16(poff[rt] + ((j >> 1) & 1u) * PAIR);
                u32x4_t qh = {};
                if constexpr (Q5K) qh = mm2_lds16(hoff[rt] + hpar * (MM2_ROWS * HDR) + 16u + 16u * h);
                // sc as two f16, and -1024 sc
                const uint32_t s1k = __builtin_amdgcn_perm(0x64646464u, sc[rt][j >> 2], 0x04000400u | (j & 3u) << 16 | (j & 3u));
                const half2_t s2 = __builtin_bit_cast(half2_t, s1k) - half2_t{(_Float16) 1024.f, (_Float16) 1024.f};
                const half2_t s2n = s2 * half2_t{(_Float16) -1024.f, (_Float16) -1024.f};
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        uint32_t w = (kq[rt][2 * s + i] >> (j % 2u ? 4u : 0u)) & 0x0F0F0F0Fu;
                        if constexpr (Q5K) w |= (j >= 4u ? qh[2 * s + i] >> (j - 4u) : qh[2 * s + i] << (4u - j)) & 0x10101010u;
                        const half2_t h0 = __builtin_elementwise_fma(
                            __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)), s2, s2n);
                        const half2_t h1 = __builtin_elementwise_fma(
                            __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)), s2, s2n);
                        bw[rt][s][4 * i] = h0[0];
                        bw[rt][s][4 * i + 1] = h0[1];
                        bw[rt][s][4 * i + 2] = h1[0];
                        bw[rt][s][4 * i + 3] = h1[1];
                    }
            }
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    mm2_f32x16 c = {};
                    if (j % 2u == 1u) c = S[tt][rt];
#pragma unroll
                    for (int s = 0; s < 2; ++s) c = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[tt][s], bw[rt][s], c, 0, 0, 0);
#pragma unroll
                    for (int s = 0; s < 2; ++s) c = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[tt][s], bw[rt][s], c, 0, 0, 0);
                    if (j % 2u == 1u) {  // a pair's sum is complete
                        const float d = (float) __builtin_bit_cast(_Float16, (uint16_t) (dd[rt] & 0xFFFFu));
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[tt][rt][e] = fmaf(d, c[e], acc[tt][rt][e]);
                    } else {
                        S[tt][rt] = c;
                    }
                }
            if (j == 7u) {  // the super-block's mins and scale
                half8_t v01[2], v23[2];
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    v01[tt] = __builtin_bit_cast(half8_t, mm2_lds16(soff[tt]));
                    v23[tt] = __builtin_bit_cast(half8_t, mm2_lds16(soff[tt] + MM2_TOK * 32u));
                }
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) {
                    const half8_t m = mm2_u4_to_f16(mm2_u32x2{mn[rt][0], mn[rt][1]});
                    const half8_t m01 = m * (h ? (_Float16) 0.5f : (_Float16) 1024.f), m23 = m * (h ? (_Float16) 0x1p-23f : (_Float16) 0x1p-12f);
                    const float dm = -0.0625f * (float) __builtin_bit_cast(_Float16, (uint16_t) (dd[rt] >> 16));
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt) {
                        mm2_f32x16 M = {};
                        M = __builtin_amdgcn_mfma_f32_32x32x16_f16(v23[tt], m23, M, 0, 0, 0);
                        M = __builtin_amdgcn_mfma_f32_32x32x16_f16(v01[tt], m01, M, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            acc[tt][rt][e] = fmaf(dm, M[e], acc[tt][rt][e]);
                    }
                }
            }
            bufo = bufo == 2u * MM2_ACT ? 0u : bufo + MM2_ACT;
        }
    }
    if constexpr (KS == 2)
        for (uint32_t i = nb; i < span.most; ++i) __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_s_waitcnt(mm2_vmcnt(0));  // no copy outlives the work-group
    const uint32_t r = r0 + 64u * (wave >> 1) + n, tl = 64u * (wave & 1u) + 4u * h;
    if constexpr (KS == 2) {
        mm2_store_halves(a, sg, acc, group, wave, lane, lds_all, t0, r, tl);
    } else {
        mm2_store(a, sg, acc[0][0], acc[1][0], t0, r, tl);
        mm2_store(a, sg, acc[0][1], acc[1][1], t0, r + 32u, tl);
    }
}

}  // namespace

extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
moearc_matmul2_q4_k_k(MatmulArgs a) { mm2k_body<12>(a); }
extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
moearc_matmul2_q5_k_k(MatmulArgs a) { mm2k_body<13>(a); }
extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
moearc_matmul2x_q4_k_k(MatmulArgs a) { mm2k_body<12, 2>(a); }
extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
moearc_matmul2x_q5_k_k(MatmulArgs a) { mm2k_body<13, 2>(a); }

// The f16 hi / lo split of x (as moearc_split_f16_k) and, in the same pass, each super-block's eight
// 32-wide sums in f32 as the four f16 pieces of v = sum / 64 (an f16 sum of 32 activations could overflow):
// v0 = f16(v), v1 = f16 of the remainder times 2^11 and so on; the remainders are exact. A thread takes eight
// elements, four lanes a sub-block. xs: [n / 256][piece][8]. ALIGNED: x on 16 bytes, else element loads.
template <bool ALIGNED>
__device__ __forceinline__ void split_sums(const float *x, uint16_t *hi, uint16_t *lo, uint16_t *xs, uint64_t n8) {
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += (uint64_t) gridDim.x * blockDim.x) {
        float v[8];
        if constexpr (ALIGNED) {
            const float4_t va = ((const float4_t *) x)[2 * i], vb = ((const float4_t *) x)[2 * i + 1];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[k] = va[k];
                v[4 + k] = vb[k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = x[8 * i + k];
        }
        half8_t h, l;
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            h[k] = (_Float16) v[k];
            l[k] = (_Float16) (v[k] - (float) h[k]);
            t += v[k];
        }
        store_through16((u32x4_t *) hi + i, __builtin_bit_cast(u32x4_t, h));
        store_through16((u32x4_t *) lo + i, __builtin_bit_cast(u32x4_t, l));
        t += __shfl_xor(t, 1);  // n8 is a multiple of 32: a sub-block's four lanes are all here
        t += __shfl_xor(t, 2);
        t *= 0x1p-6f;
        _Float16 part[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            part[p] = p < 2 && fabsf(t) < 0x1p-14f ? (_Float16) 0.f : (_Float16) t;
            t = (t - (float) part[p]) * 2048.f;
        }
        const uint32_t p = (uint32_t) (i & 3u);
        xs[(i >> 5) * 32u + 8u * p + (uint32_t) ((i >> 2) & 7u)] =
            __builtin_bit_cast(uint16_t, p == 0u ? part[0] : p == 1u ? part[1] : p == 2u ? part[2] : part[3]);
    }
}
extern "C" __global__ void moearc_split_sums_k(const float *x, uint16_t *hi, uint16_t *lo, uint16_t *xs, uint64_t n8) {
    if ((uintptr_t) x % 16 == 0) split_sums<true>(x, hi, lo, xs, n8);
    else split_sums<false>(x, hi, lo, xs, n8);
}
