// Chunked prefill, single-f16 softmax weights: the default kernels (moearc_attn_prefill_g{1,2,4,8}).
//
// Semantics are those of prefill.hip (the reference engine's prefill, one decode per prompt token,
// moe.rs:1856-1862): query row i at absolute position p = pos0 + i attends keys [b(p), p], b(p) =
// max(0, p + 1 - n_swa) on a windowed layer and 0 otherwise, with the per-head sink in the
// denominator (kernels.cpp:1864-1880).
//
// Work decomposition. A work-group owns one KV head and 256 query rows, a row being one
// (token, head) pair of that KV head's group (GQA packing); each of its four waves owns 64 rows as
// two 32-row blocks, A and B, that share every K/V operand read from LDS. Two work-groups share a
// CU (two waves per SIMD). Work-group jj of a KV head takes query tile n-1-jj in its first half and
// tile jj-n/2 in its second, so the two work-groups that land on one CU carry a late (long) and an
// early (short) tile.
//
// Keys stream through LDS in 64-key tiles, four buffers, LDS-DMA copies (global_load_lds_dwordx4)
// two tiles ahead; each wave copies 16 keys of K and V per tile; one barrier per tile. Tiles start
// on a 32-key boundary and the loop may end after a tile's first chunk, so a work-group computes
// only chunks that hold some key of its rows' spans (a windowed work-group of 32 tokens: 5 chunks,
// not the 6 of 64-key-aligned tiles). (A tile's
// buffer is refilled only once both its chunks are finished: the step that opens tile t runs while
// tile t - 1's second chunk is still being computed, so it fills tile t - 2's buffer.)
//
// Per 32-key chunk j a wave runs four regions:
//   R1  S_B(j) = K(j).Q_B^T            4 MFMAs  |  exps of A(j)                       VALU
//       then the K operands of chunk j+1 are read from LDS
//   R2  O_A += V(j)^T.P_A(j)^T, l_A    6 MFMAs  |  f16 P_A(j), exponent inputs and rescale test of S_B(j)
//   R3  S_A(j+1) = K(j+1).Q_A^T        4 MFMAs  |  exps of B(j)
//   R4  O_B += V(j)^T.P_B(j)^T, l_B    6 MFMAs  |  f16 P_B(j), exponent inputs and rescale test of S_A(j+1)
//       then the V^T operands of chunk j+1 are read from LDS
// so each block's softmax runs beside the other block's matrix work, and LDS latency hides behind a
// region. Matrix layouts, LDS swizzles and operand reads are those of prefill.hip
// (v_mfma_f32_32x32x16_f16; lane (h, n) holds keys 8i + 4h + r of query row n). The key loop --
// tile copies, the four regions, masks and rescales -- is one asm statement generated by
// gen_prefill_loop.py (prefill_loop.inc) over a fixed register map: at ~210 live VGPRs the
// compiler's own allocation of this loop copies whole accumulator tuples at every join and spills.
//
// Pair balance: the two work-groups that share a CU (i and i + pair_half) would not end together --
// the issue arbiter favours the older one's waves -- so the second raises its priority for a number
// of chunks computed from both work-groups' chunk counts and drops it at that tile step.
//
// Softmax: the MFMA returns the raw scores q.k (exact f16 products, f32 sums) and one f32 FMA per
// score, s * c + (7 - m) with c = scale*log2(e), gives the base-2 exponent of its weight against the
// row's reference m (scaling q by c in f16 instead would round every q element once more, an error
// that grows with |q|.|k|: 6e-3 with a band of keys scaled by 6). m moves only when
// some exponent of a chunk reaches PFF_RESCALE_AT (the weight could leave f16's range): the test
// (a max3 tree and a compare into an SGPR pair) runs one region ahead, beside the other block's
// P.V, and the branch on it opens the region that exponentiates the block; the rescale recomputes
// the chunk's raw scores, takes the row maximum and rescales O, the sum and the bias. Each block's
// m starts at its row maximum over chunk 0 (the loop's prologue computes both blocks' first scores
// for it), so no block rescales at its first chunk. Chunks that
// cross a row's span boundary (or that a block does not see at all) are masked: masked weights are
// zero. The row sums l are taken on the matrix cores too, over the f16 weights the P.V product sees
// (two 16x16x32 MFMAs per block and chunk against a selection operand, in place of 16 VALU
// instructions), so a weight's f16 rounding cancels in the normalisation.
#include "common.h"

#define PFF_KT 64                // keys per LDS tile (two 32-key chunks)
#define PFF_NBUF 4               // tile buffers: copies run two tiles ahead
#define PFF_TILE (PFF_KT * 128)  // bytes of one K or V tile
#define PFF_BUF (2 * PFF_TILE)   // one buffer: K tile, V tile
// Exponent (log2 of a weight, 7 at the reference max) from which the chunk is rescaled first:
// 2^15 stays well inside f16 (65504) whatever the rounding of v_exp_f32.
#define PFF_RESCALE_AT 15.0f

typedef uint32_t u32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x8_t __attribute__((ext_vector_type(8)));

// registers the key loop writes beyond its in/out operands (m0, which its LDS copies set, is saved
// in s86 and restored before the statement ends)
#define PFF_CLOBBERS                                                                                 \
    "v64", "v65", "v66", "v67", "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", \
        "v78", "v79", "v80", "v81", "v82", "v83", "v84", "v85", "v86", "v87", "v88", "v89", "v90",    \
        "v91", "v92", "v93", "v94", "v95", "v160", "v161", "v162", "v163", "v164", "v165", "v166",   \
        "v167", "v168", "v169", "v170", "v171", "v172", "v173", "v174", "v175", "v176", "v177",       \
        "v178", "v179", "v180", "v181", "v182", "v183", "v184", "v185", "v186", "v187", "v188",       \
        "v189", "v190", "v191", "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199",       \
        "v200", "v201", "v202", "v203", "v204", "v205", "v206", "v207", "v226", "v227", "v228",       \
        "v229", "v244", "v245", "v246", "v247",                                                  \
        "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75", "s76",    \
        "s77", "s78", "s79", "s80", "s81", "s82", "s83", "s84", "s85", "s86", "vcc", "scc", "memory"

// SPLIT: the work-group takes a piece of its tile's key range (sp, launch_args.h), and leaves partial
// records unless the piece is the whole range. For chunks whose tiles leave CUs idle: a work-group's
// time is its chunk count (0.59 us per 32-key chunk alone on a CU) and about 10 us around it, so 200
// tokens behind 16301 keys (56 work-groups of 516 chunks) took 306 us and take 74.8 in 504 pieces,
// 16 behind 24000 443 -> 30.6, 300 behind 4000 84 -> 43.6 (64 query heads over 8 KV heads).
template <int GROUP, bool SPLIT>
__device__ __forceinline__ void prefill_fast_body(const PrefillArgs &a, const PrefillSplitArgs *sp) {
    constexpr uint32_t TOK = MOEARC_PREFILL_FAST_ROWS / GROUP;  // query tokens per work-group
    __shared__ __attribute__((aligned(1024))) uint8_t tiles[PFF_NBUF * PFF_BUF];

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t G = a.n_kv_heads;
    const uint32_t kvh = blockIdx.x % G;
    const uint32_t jj = blockIdx.x / G;
    const uint32_t nqt = a.n_qtiles, hq = (nqt + 1u) >> 1;
    uint32_t qt = jj < hq ? nqt - 1u - jj : jj - hq;
    uint32_t item = 0, piece = 0, pieces = 1;
    if constexpr (SPLIT) {
        // the tile that holds this item: lane t compares with tile t's first item (longest tiles first)
        item = sp->n_items - 1u - jj;
        const uint32_t first = sp->item_begin[lane];
        qt = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < nqt && first <= item)) - 1u;
        const uint32_t i0 = sp->item_begin[qt];
        piece = item - i0;
        pieces = sp->item_begin[qt + 1u] - i0;
    }
    const uint32_t q0 = qt * TOK, q_end = min(q0 + TOK, a.n_q);
    const uint32_t h = lane >> 5, n = lane & 31u;
    const uint32_t p_last = a.pos0 + q_end - 1u;
    auto win = [&](uint32_t p) -> uint32_t {
        return a.n_swa ? (p + 1u > a.n_swa ? p + 1u - a.n_swa : 0u) : 0u;
    };
    // Chunks of 32 keys from the one holding the first row's window start to the one holding the
    // last row's position; tiles of two chunks from there (the last tile may hold one chunk only).
    uint32_t key0 = win(a.pos0 + q0) / 32u * 32u;  // first key of chunk 0
    uint32_t nc = (p_last - key0) / 32u + 1u;      // 32-key chunks
    if constexpr (SPLIT) {
        const uint32_t c0 = nc * piece / pieces, c1 = nc * (piece + 1u) / pieces;  // the host bounds nc below 2^22
        key0 += 32u * c0;
        nc = c1 - c0;
    }
    const uint32_t ntiles = (nc + 1u) >> 1;

    // ---- pair balance: the dispatcher puts work-groups i and i + pair_half on one CU, and the issue
    // arbiter favours the older one's waves, so the first of a pair runs ahead and the second ends
    // alone at half occupancy. The second raises its waves' priority for boost_a * (its chunks) -
    // boost_b * (its partner's chunks) chunks and returns to the default at that tile step.
    uint32_t btile = 0;
    if constexpr (SPLIT) {  // pieces of nearly equal length
        if (a.pair_half && blockIdx.x >= a.pair_half) {
            btile = min(ntiles, (uint32_t) ((a.boost_a - a.boost_b) * 0.5f * (float) nc));
            if (btile) __builtin_amdgcn_s_setprio(1);
        }
    } else if (a.pair_half && blockIdx.x >= a.pair_half) {
        const uint32_t pb = blockIdx.x - a.pair_half, pjj = pb / G;
        const uint32_t pqt = pjj < hq ? nqt - 1u - pjj : pjj - hq;
        const uint32_t pq0 = pqt * TOK, pq_end = min(pq0 + TOK, a.n_q);
        const uint32_t pkey0 = win(a.pos0 + pq0) / 32u * 32u;
        const uint32_t pnc = (a.pos0 + pq_end - 1u - pkey0) / 32u + 1u;
        const float bc = a.boost_a * (float) nc - a.boost_b * (float) pnc;
        if (bc >= 2.f) {
            btile = min(ntiles, (uint32_t) (bc * 0.5f));
            __builtin_amdgcn_s_setprio(1);
        }
    }

    // ---- block-table entries of tiles 0 and 1 for this lane's two copy keys (16 wave + lane / 8
    // and 8 more; keys clamped to the last query position, tiles to the last tile), issued with the
    // query loads below so that both arrive in one memory round trip before the key loop starts
    const uint32_t kk0 = 16u * wave + (lane >> 3);
    u32x4_t pid01;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t key = key0 + 64u * min((uint32_t) t, ntiles - 1u) + kk0 + 8u * i;
            pid01[2 * t + i] = a.block_table[min(key, p_last) >> a.pt_shift];
        }

    // ---- per block: query operands (the caller's f16 q as it is: the MFMA's products are exact and
    // c = scale * log2 e is applied to each f32 score, so a score carries no rounding of q * c), and
    // the chunk range that needs no masks ---------------------------------------------------------
    const float c = a.scale_log2e;
    auto tok_of = [&](int X) { return q0 + (64u * wave + 32u * X + n) / GROUP; };
    auto hd_of = [&](int X) { return kvh * GROUP + (64u * wave + 32u * X + n) % GROUP; };
    u32x16_t Qp[2];
    uint32_t jlo[2], jn[2];
    uint32_t cm[2], span[2];
#pragma unroll
    for (int X = 0; X < 2; ++X) {
        const uint32_t tk = tok_of(X);
        const uint16_t *src =
            a.q + ((uint64_t) min(tk, a.n_q - 1u) * a.n_heads + hd_of(X)) * 64u + 8u * h;
        const bool ok = tk < q_end;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            u32x4_t v = *(const u32x4_t *) (src + 16 * t);
            if (!ok) v = (u32x4_t){0u, 0u, 0u, 0u};
#pragma unroll
            for (int e = 0; e < 4; ++e) Qp[X][4 * t + e] = v[e];
        }
        // Chunk j (keys key0 + 32 j ..) needs no masks for block X when its last key is at or
        // below the block's first row position and (windowed layers) its first key at or above
        // the block's last window start: j - jlo < jn (unsigned; jn = 0: every chunk is masked).
        const uint32_t r0 = 64u * wave + 32u * X;
        const uint32_t t0 = q0 + r0 / GROUP, t1 = q0 + (r0 + 31u) / GROUP;
        const uint32_t pmin = a.pos0 + min(t0, q_end - 1u), bmax = win(a.pos0 + min(t1, q_end - 1u));
        jlo[X] = 0u;
        jn[X] = 0u;
        if (pmin + 1u >= key0 + 32u) {
            const uint32_t hi = (pmin + 1u - key0) / 32u - 1u;
            jlo[X] = (a.n_swa != 0u && bmax > key0) ? (bmax - key0 + 31u) / 32u : 0u;
            jn[X] = hi >= jlo[X] ? hi - jlo[X] + 1u : 0u;
        }
        // this lane's row: key offset of chunk 0 relative to its window start, and its span
        const uint32_t rp = a.pos0 + min(tok_of(X), q_end - 1u), rb = win(rp);
        cm[X] = key0 + 4u * h - rb;
        span[X] = rp - rb;
    }

    float m_run[2], bias[2];  // bias = 7 - m: the exponent of a weight is s * c + bias
    float16_t O[2][2];
    // Row sums on the matrix cores: a 16x16x32 MFMA over a block's f16 weights (the very values the
    // P.V product sees) leaves row n's sum in register 0 of lane n < 32 (the key loop's `rowsum`);
    // `sel` is its A operand, ones in row 0 for lanes 0-15 and 32-47 and in row 4 for lanes 16-31
    // and 48-63 of the B operand.
    float4_t Lsum[2];
    u32x4_t sel;
    {
        const bool one = lane == 0u || lane == 32u || lane == 20u || lane == 52u;
#pragma unroll
        for (int e = 0; e < 4; ++e) sel[e] = one ? 0x3C003C00u : 0u;  // f16 (1, 1)
    }
#pragma unroll
    for (int X = 0; X < 2; ++X) {
        m_run[X] = PF_M_INIT;
        bias[X] = PF_LOG2_PSCALE - PF_M_INIT;
        Lsum[X] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            O[X][0][i] = 0.f;
            O[X][1][i] = 0.f;
        }
    }

    // ---- LDS operand addresses (buffer 0, chunk 0) ----------------------------------------------
    const uint32_t lds0 = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) uint8_t *) tiles;
    u32x4_t kbase;
#pragma unroll
    for (int t = 0; t < 4; ++t) kbase[t] = lds0 + k_off(n, 2u * t + h);
    u32x2_t vbase;
    {
        const uint32_t r = lane & 15u, qq = (lane >> 4) & 1u, vkey = 4u * h + (r >> 2);
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
            vbase[mb] = lds0 + PFF_TILE + v_off(vkey, 4u * mb + 2u * qq + ((r >> 1) & 1u)) + ((r & 1u) << 3);
    }

    // ---- tile copies: DMA instruction i of wave w fills keys 16w + 8i .. +7 of the K and V tiles;
    // lane L writes chunk slot L & 7 of key 16w + 8i + (L >> 3), which holds chunk (L & 7) ^ f(key).
    const uint32_t row_bytes = G * 128u;
    u32x4_t offs;    // uniform path: byte offsets from the tile's first row (K 0, K 1, V 0, V 1)
    u32x8_t bases;   // per-lane path: 64-bit pages base + this lane's chunk (K 0, K 1, V 0, V 1)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t kk = kk0 + 8u * i;
        const uint32_t ck = kvh * 128u + (((lane & 7u) ^ k_swz(kk)) << 4);
        const uint32_t cv = kvh * 128u + (((lane & 7u) ^ v_swz(kk)) << 4);
        offs[i] = kk * row_bytes + ck;
        offs[2 + i] = kk * row_bytes + cv;
        const uint64_t bk = (uint64_t) (uintptr_t) a.k_pages + ck, bv = (uint64_t) (uintptr_t) a.v_pages + cv;
        bases[2 * i] = (uint32_t) bk;
        bases[2 * i + 1] = (uint32_t) (bk >> 32);
        bases[4 + 2 * i] = (uint32_t) bv;
        bases[4 + 2 * i + 1] = (uint32_t) (bv >> 32);
    }
    const uint64_t btp = (uint64_t) (uintptr_t) a.block_table;
    const u32x2_t btb = {(uint32_t) btp, (uint32_t) (btp >> 32)};
    const uint32_t bperm = (lane ^ 32u) << 2;
    const uint64_t kp = (uint64_t) (uintptr_t) a.k_pages, vp = (uint64_t) (uintptr_t) a.v_pages;
    const uint32_t ldsw = __builtin_amdgcn_readfirstlane(lds0 + 16u * wave * 128u);

    // ---- the key loop (prefill_loop.inc) ---------------------------------------------------------
    asm volatile(
#include "prefill_loop.inc"
        : "+{v[0:15]}"(O[0][0]), "+{v[16:31]}"(O[0][1]), "+{v[32:47]}"(O[1][0]), "+{v[48:63]}"(O[1][1]),
          "+{v208}"(m_run[0]), "+{v209}"(m_run[1]), "+{v[100:103]}"(Lsum[0]), "+{v[104:107]}"(Lsum[1]),
          "+{v96}"(bias[0]), "+{v112}"(bias[1]), "+{v[222:225]}"(pid01)
        : "{v[128:143]}"(Qp[0]), "{v[144:159]}"(Qp[1]), "{v[212:215]}"(kbase), "{v[216:217]}"(vbase),
          "{v218}"(cm[0]), "{v219}"(span[0]), "{v220}"(cm[1]), "{v221}"(span[1]),
          "{v[230:233]}"(offs), "{v[234:241]}"(bases), "{v242}"(kk0), "{v243}"(bperm),
          "{v[248:249]}"(btb), "{v[108:111]}"(sel),
          [kplo] "s"(__builtin_amdgcn_readfirstlane((uint32_t) kp)),
          [kphi] "s"(__builtin_amdgcn_readfirstlane((uint32_t) (kp >> 32))),
          [vplo] "s"(__builtin_amdgcn_readfirstlane((uint32_t) vp)),
          [vphi] "s"(__builtin_amdgcn_readfirstlane((uint32_t) (vp >> 32))),
          [ntiles] "s"(__builtin_amdgcn_readfirstlane(ntiles)),
          [ntm1] "s"(__builtin_amdgcn_readfirstlane(ntiles - 1u)),
          [nc] "s"(__builtin_amdgcn_readfirstlane(nc)),
          [kb0] "s"(__builtin_amdgcn_readfirstlane(key0)),
          [plast] "s"(__builtin_amdgcn_readfirstlane(p_last)),
          [sh] "s"(__builtin_amdgcn_readfirstlane(a.pt_shift)),
          [pmask] "s"(__builtin_amdgcn_readfirstlane((1u << a.pt_shift) - 1u)),
          [rowb] "s"(__builtin_amdgcn_readfirstlane(row_bytes)),
          [ldsw] "s"(ldsw), [thr] "s"(__builtin_bit_cast(uint32_t, PFF_RESCALE_AT)),
          [cs] "s"(__builtin_amdgcn_readfirstlane(__builtin_bit_cast(uint32_t, c))),
          [jloa] "s"(__builtin_amdgcn_readfirstlane(jlo[0])), [jloa1] "s"(__builtin_amdgcn_readfirstlane(jlo[0] - 1u)),
          [jna] "s"(__builtin_amdgcn_readfirstlane(jn[0])),
          [jlob] "s"(__builtin_amdgcn_readfirstlane(jlo[1])), [jnb] "s"(__builtin_amdgcn_readfirstlane(jn[1])),
          [btile] "s"(__builtin_amdgcn_readfirstlane(btile))
        : PFF_CLOBBERS);

    // ---- finalise each block: row sum over the lane pair, the sink, the normalisation. The rows
    // leave through LDS, where the key loop is done: each wave stages its 64 normalised rows in f32
    // (256 bytes per row, 16-byte chunk c at position c ^ (row & 15): every 16-lane write or read
    // touches 64 distinct banks) and stores whole rows, 8 per instruction with f16 output and 4
    // with f32 -- instead of the accumulators' 8- or 16-byte pieces, which reach 32 rows (32 cache
    // lines) per store instruction.
    __builtin_amdgcn_s_waitcnt(0);  // the key loop's last copies have landed
    __syncthreads();                 // and no wave reads a K/V tile any more
    const uint32_t stage = lds0 + wave * (64u * 256u);
#pragma unroll
    for (int X = 0; X < 2; ++X) {
        const float L = Lsum[X][0] + __shfl_xor(Lsum[X][0], 32);  // lanes 32-63 hold 0 there
        const uint32_t hh = hd_of(X);
        const float sink2 = a.sinks ? a.sinks[hh] * MOEARC_LOG2E : -INFINITY;
        const float Mt = fmaxf(m_run[X], sink2);
        const float fm = __builtin_amdgcn_exp2f(m_run[X] - Mt);
        float inv = fm / (L * fm + __builtin_amdgcn_exp2f(sink2 - Mt + PF_LOG2_PSCALE));
        const uint32_t rho = 32u * X + n;  // row of the wave
        if constexpr (SPLIT) {
            if (pieces > 1u) {
                inv = 1.f;
                if (h == 0 && tok_of(X) < q_end)
                    *(float2_t *) (sp->rec_ml + 2u * (((uint64_t) item * G + kvh) * MOEARC_PREFILL_FAST_ROWS + 64u * wave + rho)) =
                        (float2_t){m_run[X], L};
            }
        }
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int jq = 0; jq < 4; ++jq) {
                // O reg 4jq + i = channel 32mb + 8jq + 4h + i of row n: 16-byte chunk 8mb + 2jq + h
                const float4_t v = {O[X][mb][4 * jq] * inv, O[X][mb][4 * jq + 1] * inv, O[X][mb][4 * jq + 2] * inv,
                                    O[X][mb][4 * jq + 3] * inv};
                const uint32_t c = 8u * mb + 2u * jq + h;
                *(__attribute__((address_space(3))) float4_t *) (uintptr_t) (stage + rho * 256u + 16u * (c ^ (rho & 15u))) = v;
            }
    }
    // (the reads below follow the writes in this wave's LDS order; other waves' rows are not read)
    if constexpr (SPLIT) {
        if (pieces > 1u) {
#pragma unroll
            for (int k = 0; k < 16; ++k) {  // lane L: row 4k + (L >> 4), channels 4 (L & 15) .. + 3
                const uint32_t rho = 4u * k + (lane >> 4), c = lane & 15u, r = 64u * wave + rho;
                const float4_t v = *(const __attribute__((address_space(3))) float4_t *) (uintptr_t) (
                    stage + rho * 256u + 16u * (c ^ (rho & 15u)));
                float *dst = sp->rec_o + ((((uint64_t) item * G + kvh) * MOEARC_PREFILL_FAST_ROWS + r) * 64u + 4u * c);
                if (q0 + r / GROUP < q_end) store_through16(dst, __builtin_bit_cast(u32x4_t, v));
            }
            return;
        }
    }
    auto out_row = [&](uint32_t rho) -> int64_t {  // element offset of a staged row, -1 past the chunk
        const uint32_t r = 64u * wave + rho, tk = q0 + r / GROUP;
        return tk < q_end ? (int64_t) (((uint64_t) tk * a.n_heads + kvh * GROUP + r % GROUP) * 64u) : -1;
    };
    if (a.out_f16) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {  // lane L: row 8k + (L >> 3), channels 8 (L & 7) .. + 7
            const uint32_t rho = 8u * k + (lane >> 3), j = lane & 7u;
            const float4_t lo = *(const __attribute__((address_space(3))) float4_t *) (uintptr_t) (
                stage + rho * 256u + 16u * ((2u * j) ^ (rho & 15u)));
            const float4_t hi = *(const __attribute__((address_space(3))) float4_t *) (uintptr_t) (
                stage + rho * 256u + 16u * ((2u * j + 1u) ^ (rho & 15u)));
            half8_t w;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                w[i] = (_Float16) lo[i];
                w[4 + i] = (_Float16) hi[i];
            }
            const int64_t o = out_row(rho);
            if (o >= 0) store_through16((_Float16 *) a.out + o + 8u * j, __builtin_bit_cast(u32x4_t, w));
            if (a.out_lo && o >= 0) {  // the split's low halves: f16(v - f32(hi)), as moearc_split_f16_k
                half8_t l;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    l[i] = (_Float16) (lo[i] - (float) w[i]);
                    l[4 + i] = (_Float16) (hi[i] - (float) w[4 + i]);
                }
                store_through16(a.out_lo + o + 8u * j, __builtin_bit_cast(u32x4_t, l));
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) {  // lane L: row 4k + (L >> 4), channels 4 (L & 15) .. + 3
            const uint32_t rho = 4u * k + (lane >> 4), c = lane & 15u;
            const float4_t v = *(const __attribute__((address_space(3))) float4_t *) (uintptr_t) (
                stage + rho * 256u + 16u * (c ^ (rho & 15u)));
            const int64_t o = out_row(rho);
            if (o >= 0) store_through16((float *) a.out + o + 4u * c, __builtin_bit_cast(u32x4_t, v));
        }
    }
}

#define PREFILL_FAST_KERNEL(GRP)                                                                 \
    extern "C" __global__ __launch_bounds__(MOEARC_PREFILL_THREADS)                              \
        __attribute__((amdgpu_waves_per_eu(2, 2))) void moearc_attn_prefill_g##GRP(const PrefillArgs a) { \
        prefill_fast_body<GRP, false>(a, nullptr);                                               \
    }                                                                                            \
    extern "C" __global__ __launch_bounds__(MOEARC_PREFILL_THREADS)                              \
        __attribute__((amdgpu_waves_per_eu(2, 2))) void moearc_attn_prefill_split_g##GRP(const PrefillSplitArgs s) { \
        prefill_fast_body<GRP, true>(s.a, &s);                                                   \
    }

PREFILL_FAST_KERNEL(1)
PREFILL_FAST_KERNEL(2)
PREFILL_FAST_KERNEL(4)
PREFILL_FAST_KERNEL(8)

// Combines the pieces of split tiles (launch_args.h): 16 lanes per (token, head) row, lane c taking
// channels 4c .. + 3 of each piece's record, eight pieces' loads in flight; then the sink, the
// normalisation and the store as the unsplit kernel's. Rows of unsplit tiles are left alone.
// Bound by the records' traffic: 33 MB of 504 pieces in 10-11 us.
extern "C" __global__ __launch_bounds__(256) void moearc_attn_prefill_merge_k(const PrefillSplitArgs s) {
    constexpr uint32_t B = 8;
    const PrefillArgs &a = s.a;
    const uint64_t row = (uint64_t) blockIdx.x * 16u + (threadIdx.x >> 4);
    const uint32_t c = threadIdx.x & 15u, H = a.n_heads, G = a.n_kv_heads, group = a.group;
    if (row >= (uint64_t) a.n_q * H) return;
    const uint32_t tk = (uint32_t) (row / H), hd = (uint32_t) (row % H), kvh = hd / group;
    const uint32_t qt = tk / s.tile_tokens, i0 = s.item_begin[qt], n = s.item_begin[qt + 1u] - i0;
    if (n <= 1u) return;
    const uint32_t r = (tk - qt * s.tile_tokens) * group + hd % group;
    const float sink2 = a.sinks ? a.sinks[hd] * MOEARC_LOG2E : -INFINITY;
    float m = PF_M_INIT, l = 0.f;
    float4_t o = (float4_t){0.f, 0.f, 0.f, 0.f};
    for (uint32_t p0 = 0; p0 < n; p0 += B) {
        float4_t v[B];
        float2_t ml[B];
#pragma unroll
        for (uint32_t k = 0; k < B; ++k) {
            const uint64_t at = ((uint64_t) (i0 + min(p0 + k, n - 1u)) * G + kvh) * MOEARC_PREFILL_FAST_ROWS + r;
            v[k] = *(const float4_t *) (s.rec_o + at * 64u + 4u * c);
            ml[k] = *(const float2_t *) (s.rec_ml + 2u * at);
        }
        float mn = m;
#pragma unroll
        for (uint32_t k = 0; k < B; ++k) mn = fmaxf(mn, ml[k][0]);  // repeats of the last are harmless
        const float corr = __builtin_amdgcn_exp2f(m - mn);
        l *= corr;
        o *= corr;
#pragma unroll
        for (uint32_t k = 0; k < B; ++k) {
            const float f = p0 + k < n ? __builtin_amdgcn_exp2f(ml[k][0] - mn) : 0.f;
            l = fmaf(ml[k][1], f, l);
            o += v[k] * f;
        }
        m = mn;
    }
    const float Mt = fmaxf(m, sink2);
    const float fm = __builtin_amdgcn_exp2f(m - Mt);
    o *= fm / (l * fm + __builtin_amdgcn_exp2f(sink2 - Mt + PF_LOG2_PSCALE));
    if (!a.out_f16) {
        *(float4_t *) ((float *) a.out + row * 64u + 4u * c) = o;
        return;
    }
    typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
    half4_t hi, lo;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        hi[i] = (_Float16) o[i];
        lo[i] = (_Float16) (o[i] - (float) hi[i]);  // as moearc_split_f16_k
    }
    *(half4_t *) ((_Float16 *) a.out + row * 64u + 4u * c) = hi;
    if (a.out_lo) *(half4_t *) ((_Float16 *) a.out_lo + row * 64u + 4u * c) = lo;
}
