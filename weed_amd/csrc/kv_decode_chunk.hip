// Decode attention for many rows per KV head -- chunks of query positions, large groups -- over the packed cache.
//
// The kernel of kv_decode_mfma_kernel.h takes sixteen (position, head) rows of a KV head per pass and unpacks the cache
// anew for every pass.  Here a workgroup of eight wavefronts unpacks a 64-token block ONCE, each wavefront an eighth of its
// matrix operands, into LDS (fp16, the operands in the order in which the matrix instructions take them: 32 KB per block at
// head_dim 128, two blocks, one barrier per block), and every wavefront takes two tiles of sixteen rows against them, so that
// an operand read from LDS serves both.  The matrix instructions (fp16 halves of queries and probabilities, as there) and the
// softmax are what is left: 4096 and some 2800 cycles per SIMD for a block and 256 rows of 128, of 7200 that it takes -- unpacking
// 1200, scores 1250, softmax 2100, values 1350 and the barrier, one after the other in both wavefronts of a SIMD.  What went (8900
// cycles): loads dword by dword (request_narrow), reloads of spilled addresses (`anew`; instances of their own for up to four bits
// a field), a masking and a subtraction per value in the split of the probabilities, the subtraction of the maximum per score, and
// trips through LDS for the maxima.  64 positions x 32 heads on 8 of 128, K 3 + V 4 bits, 16 sequences of 4096 to 8192 tokens 266 ->
// 235 us, of 8192 298 -> 264; of 4096, 4-bit cells 156 -> 143, 8-bit ones 175 -> 167.  (Half of the wavefronts half a block behind the
// others, so that softmax and matrix instructions of a SIMD run beside each other: 226 us for 224 as it is, with three buffers of V;
// unpacking between scores and softmax: 282, all of it scratch.)
// The partials' write-out is that of kv_decode_mfma_kernel.h for two tiles at a time: a change to one is due in the other.  The
// softmax there subtracts the maximum and masks the probabilities' high halves in instructions of their own: as it is here, passes
// gained 1 to 3 % and other calls lost 0.5 to 1 %.
// Beside the passes, before that: 16 sequences of 8192 tokens 360 -> 296 us, 4096 to 8192 294 -> 257; 64 sequences of 1500, 5-bit
// fields 571 -> 379, 8-bit uniform ones 529 -> 341.  Where it is used: see kTilesToShare.
// Against float64 its error is no larger than the passes' (16 sequences of 4096 to 8192 tokens, of the result's norm: Lloyd-Max 5.5e-7
// against 5.6e-7, 8-bit cells 6.3e-5 against 6.7e-5; queries of eight times the width 1.2e-6, 1.3e-6 and 3.5e-6, 3.6e-6).
// At 128 with tables 52 bytes a lane of two tiles' queries, sums and scores still go to scratch and back, 108 where a field has more
// than four bits; no other instance has any.
// Measured and dropped: one tile per wavefront (half the registers, twice the operand reads; 128 rows a workgroup: 132 rows 63 ->
// 89 us, 32 rows 43 -> 49), that with a block's scores multiplied between the softmax of the block before and its products with V
// between the scores' arithmetic (16 sequences of 8192 tokens 345 us), and with two blocks' packed words on their way instead of
// one (no different: memory is not what a block waits for); other priorities for one wavefront of each SIMD (no different).
//
// Queries come prepared (q_hi, q_lo, q_scale, q_sum) and partials leave as the other kernel's do, one per row and segment of a
// workgroup's run of blocks; the kernels ahead and behind are the same.
#include "kv_decode_mfma_kernel.h"

namespace weedhip_mfma {

// a less the fp16 value in h's low (high) half, exactly: one instruction (the compiler makes a conversion and a subtraction of it)
__device__ __forceinline__ float less_low_half(float a, uint32_t h)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
    return r;
}
__device__ __forceinline__ float less_high_half(float a, uint32_t h)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
    return r;
}

typedef float float2p __attribute__((ext_vector_type(2)));
typedef _Float16 half2p __attribute__((ext_vector_type(2)));

// A lane's number anew: what is derived from it in a loop is computed there, not kept in (or spilled from) registers around it.
__device__ __forceinline__ uint32_t anew(uint32_t lane)
{
    asm volatile("" : "+v"(lane));
    return lane;
}

constexpr uint32_t kSharedWaves = 8;
constexpr int kSharedTiles = 2; // tiles of sixteen rows per wavefront
static_assert(16 * kSharedTiles * kSharedWaves == mfma_decode_shared_rows);

// One operand: 8 fields of w bits, the first at bit `at` of x[0], as fp16 values.  Up to four bits a field they are 32 bits at
// most, and one piece of code cuts out the pairs of any width.
__device__ __forceinline__ uint4v lookup_operand(uint32_t w, const uint32_t (&x)[2], uint32_t at, uint32_t lane_byte)
{
    const uint32_t first = __builtin_amdgcn_alignbit(x[1], x[0], at);
    uint4v r;
#pragma unroll
    for (uint32_t pair = 0; pair < 4; ++pair) {
        r[pair] = lds_read((__builtin_amdgcn_ubfe(first, 2 * w * pair, 2 * w) << 8) + lane_byte);
    }
    return r;
}
// `third`: the dword behind x[1], read for seven bits only
__device__ __forceinline__ half8 unpack_operand(uint32_t w, const uint32_t (&x)[2], const uint32_t *third, uint32_t at, uint32_t lane_byte)
{
    if (w <= 4) {
        return __builtin_bit_cast(half8, lookup_operand(w, x, at, lane_byte));
    }
    const uint32_t first = __builtin_amdgcn_alignbit(x[1], x[0], at);
    const uint32_t y[2] = { first, w == 7 ? (uint32_t)__builtin_amdgcn_alignbit(*third, x[1], at) : x[1] >> at };
    switch (w) {
    case 5:
        return dequant_item<5, 2, 0>(y, lane_byte);
    case 6:
        return dequant_item<6, 2, 0>(y, lane_byte);
    case 7:
        return dequant_item<7, 2, 0>(y, lane_byte);
    default:
        return dequant_item<8, 2, 0>(y, lane_byte);
    }
}

// LDS: the lookup tables (from address 0, as the lookups want them), then two blocks of operands, then two blocks of row scales.
template <int D> constexpr uint32_t shared_block_bytes() { return 2U * (D / 8) * 1024U; }
template <int D> constexpr uint32_t shared_lds_bytes(uint32_t table_rows)
{
    return table_rows * kTableRowBytes + 2U * shared_block_bytes<D>() + 2U * 2U * 64U * 4U;
}

template <int D, bool LLOYD, bool NARROW>
__global__ void __launch_bounds__(64 * kSharedWaves) decode_shared_kernel(MfmaParams launch)
{
    constexpr int QT = kSharedTiles, KS = D / 32, JB = D / 16;
    constexpr int ITEMS = D / 8;                                  // operands per side and block (4 KS and 2 JB)
    constexpr int PER_WAVE = (ITEMS + kSharedWaves - 1) / kSharedWaves;
    MfmaParams p = launch;
    // the groups of rows that read the same blocks run next to each other on one XCD (see MfmaParams::grid_passes)
    const uint32_t octet = blockIdx.x >> 3, rows_group = octet % launch.grid_passes;
    const uint32_t unit = (octet / launch.grid_passes) * 8 + (blockIdx.x & 7);
    uint32_t g0 = unit * p.runs.unit_blocks;
    const uint32_t g1 = min(g0 + p.runs.unit_blocks, p.total_blocks);
    if (g0 >= g1) {
        return; // (the workgroups were rounded up to a multiple of eight)
    }
    p.head_first = rows_group * launch.tile_rows;
    p.G = min(launch.tile_rows, launch.group_total - p.head_first);

    extern __shared__ uint32_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t table_rows = mfma_table_rows(p.k.w, p.v.w);
    uint8_t *const operands = reinterpret_cast<uint8_t *>(lds) + table_rows * kTableRowBytes;
    float *const scales = reinterpret_cast<float *>(operands + 2 * shared_block_bytes<D>()); // [2][K, V][64]
    for (uint32_t i = tid; i < table_rows * (kTableRowBytes / 16); i += 64 * kSharedWaves) {
        const uint32_t w = p.table_image[i / 8];
        reinterpret_cast<uint4v *>(lds)[i] = uint4v{ w, w, w, w };
    }

    const auto blk_off_at = [&](uint32_t i) { return p.uniform_blocks ? i * p.uniform_blocks : p.blk_off[i]; };
    uint32_t seq = 0;
    if (p.uniform_blocks) {
        seq = g0 / (p.uniform_blocks * p.Hkv);
    } else {
        // the largest s with blk_off[s] * Hkv <= g0 (a sequence without tokens shares its offset with the next one)
        uint32_t hi = p.n_seq;
        while (hi - seq > 1) {
            const uint32_t mid = (seq + hi) / 2;
            if (p.blk_off[mid] * p.Hkv <= g0) {
                seq = mid;
            } else {
                hi = mid;
            }
        }
    }

    while (g0 < g1) {
        const uint32_t seq_first = blk_off_at(seq), nb_cap = blk_off_at(seq + 1) - seq_first;
        if (nb_cap == 0) {
            ++seq;
            continue;
        }
        const uint32_t rel = g0 - seq_first * p.Hkv, kvh = rel / nb_cap, b0 = rel - kvh * nb_cap;
        const uint32_t seg = min(nb_cap - b0, g1 - g0);
        const uint32_t slot = unit - (seq_first * p.Hkv + kvh * nb_cap) / p.runs.unit_blocks;
        const uint32_t L = (uint32_t)p.lens[seq]; // may be shorter than the cached length (prefix attention)
        const uint32_t b1 = min(b0 + seg, (L + 63) >> 6);
        const uint64_t region = (uint64_t)seq * p.Hkv + kvh;
        g0 += seg;

        // ---- this wavefront's share of the unpacking: operands wave, wave + 8, ... of each side.  A lane's run of a block
        //      is D w / 32 dwords; operand i begins at its bit 8 w i ----
        const uint8_t *kreg = p.k.fields + region * p.k.region_bytes, *vreg = p.v.fields + region * p.v.region_bytes;
        const float *alphas = nullptr;
        if constexpr (LLOYD) {
            alphas = (wave ? p.v.alpha : p.k.alpha) + region * p.padded;
        }
        uint32_t kx[PER_WAVE][2], vx[PER_WAVE][2];
        float alpha = 0.0f;
        auto request_side = [&](const uint8_t *reg, uint32_t w, uint32_t blk, uint32_t (&x)[PER_WAVE][2]) __attribute__((always_inline)) {
            const uint32_t run = D * w / 32; // dwords per lane
            const uint32_t *mine = reinterpret_cast<const uint32_t *>(reg + (uint64_t)blk * (8U * D * w)) + anew(lane) * run;
#pragma unroll
            for (int u = 0; u < PER_WAVE; ++u) {
                const uint32_t i = wave + kSharedWaves * u;
                const uint32_t dw = (8 * w * min(i, (uint32_t)ITEMS - 1)) >> 5;
                x[u][0] = mine[dw];
                x[u][1] = mine[min(dw + 1, run - 1)];
            }
        };
        // up to four bits a field: operands PER_WAVE wave .. PER_WAVE wave + PER_WAVE - 1, 64 bits from dword `first` of the run on in one load (a
        // load per dword of operands eight apart was four times the lines asked for: 660 to 1100 cycles a block)
        const auto first_dword = [&](uint32_t w) { return min((8 * w * PER_WAVE * wave) >> 5, D * w / 32 - 2); };
        auto request_narrow = [&](const uint8_t *reg, uint32_t w, uint32_t blk, uint32_t (&x)[2]) __attribute__((always_inline)) {
            typedef uint32_t uint2a __attribute__((ext_vector_type(2), aligned(4)));
            const uint32_t mine = 4 * (anew(lane) * (D * w / 32) + first_dword(w));
            const uint2a v = *reinterpret_cast<const uint2a *>(reg + (uint64_t)blk * (8U * D * w) + mine);
            x[0] = v[0];
            x[1] = v[1];
        };
        auto request = [&](uint32_t blk) __attribute__((always_inline)) {
            if constexpr (NARROW) {
                request_narrow(kreg, p.k.w, blk, kx[0]);
                request_narrow(vreg, p.v.w, blk, vx[0]);
            } else {
                request_side(kreg, p.k.w, blk, kx);
                request_side(vreg, p.v.w, blk, vx);
            }
            if constexpr (LLOYD) {
                if (wave < 2) {
                    alpha = alphas[blk * 64 + anew(lane)];
                }
            }
        };
        auto unpack = [&](uint32_t blk, uint32_t buf) __attribute__((always_inline)) {
            const uint32_t lane_ = anew(lane), vbase = (lane_ & 31) * 4, kbase = vbase + 128;
            uint4v *k_to = reinterpret_cast<uint4v *>(operands + buf * shared_block_bytes<D>()) + lane_, *v_to = k_to + ITEMS * 64;
            auto side = [&](const uint8_t *reg, uint32_t w, const uint32_t (&x)[PER_WAVE][2], uint32_t lane_byte, uint4v *to) __attribute__((always_inline)) {
                const uint32_t run = D * w / 32;
                const uint32_t *mine = reinterpret_cast<const uint32_t *>(reg + (uint64_t)blk * (8U * D * w)) + lane_ * run;
#pragma unroll
                for (int u = 0; u < PER_WAVE; ++u) {
                    const uint32_t i = wave + kSharedWaves * u, bit = 8 * w * i;
                    if (i < (uint32_t)ITEMS) {
                        const half8 v = unpack_operand(w, x[u], mine + min((bit >> 5) + 2, run - 1), bit & 31, lane_byte);
                        to[i * 64] = __builtin_bit_cast(uint4v, v);
                    }
                }
            };
            if constexpr (NARROW) {
                // (every lookup on its way before the first operand is put down)
                uint4v r[2][PER_WAVE];
                const auto cut = [&](uint32_t w, const uint32_t (&x)[2], int u, uint32_t lane_byte) __attribute__((always_inline)) {
                    const uint32_t at = 8 * w * (PER_WAVE * wave + u) - 32 * first_dword(w);
                    const uint32_t y[2] = { at < 32 ? x[0] : x[1], at < 32 ? x[1] : 0U };
                    return lookup_operand(w, y, at & 31, lane_byte);
                };
#pragma unroll
                for (int u = 0; u < PER_WAVE; ++u) {
                    r[0][u] = cut(p.k.w, kx[0], u, kbase);
                    r[1][u] = cut(p.v.w, vx[0], u, vbase);
                }
#pragma unroll
                for (int u = 0; u < PER_WAVE; ++u) {
                    const uint32_t i = PER_WAVE * wave + u;
                    if (i < (uint32_t)ITEMS) {
                        k_to[i * 64] = r[0][u];
                        v_to[i * 64] = r[1][u];
                    }
                }
            } else {
                side(kreg, p.k.w, kx, kbase, k_to);
                side(vreg, p.v.w, vx, vbase, v_to);
            }
            if constexpr (LLOYD) {
                if (wave < 2) {
                    scales[buf * 128 + wave * 64 + lane_] = alpha;
                }
            }
        };

        // ---- this wavefront's rows: tiles QT wave .. QT wave + QT - 1 of sixteen; lane c of a tile's column works on row c ----
        const bool works = QT * 16 * wave < p.G;
        half8 qop[QT][2][KS];
        float qscale[QT];
        float m_first[QT]; // what stands for a row's running maximum while it has seen nothing
        uint32_t hidden[QT];
        const uint32_t hidden_max = p.q_tokens - 1U;
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const uint32_t hs = 16 * (QT * wave + q) + c;
            const bool ok = hs < p.G;
            const uint32_t qh = q_head_of(p, kvh, ok ? hs : 0);
            const uint64_t row = (uint64_t)seq * p.Hq + qh, qbase = row * D + g * (D / 4);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                uint4v hi = { 0, 0, 0, 0 }, lo = { 0, 0, 0, 0 };
                if (ok) {
                    hi = *reinterpret_cast<const uint4v *>(p.q_hi + qbase + 8 * ks);
                    lo = *reinterpret_cast<const uint4v *>(p.q_lo + qbase + 8 * ks);
                }
                qop[q][0][ks] = __builtin_bit_cast(half8, hi);
                qop[q][1][ks] = __builtin_bit_cast(half8, lo);
            }
            qscale[q] = ok ? p.q_scale[row] : 0.0f;
            m_first[q] = (!LLOYD && ok) ? -__builtin_rintf(p.k.beta * p.q_sum[row]) : 0.0f;
            const uint32_t pair = p.head_first + hs; // index among the KV head's (position, head) pairs
            hidden[q] = (hidden_max && ok) ? hidden_max - (p.blocked ? pair % p.q_tokens : pair / p.real_group) : 0U;
        }
        // (the running maximum, its slack and `ep`: as in decode_mfma_kernel)
        constexpr float kSlack = 8.0f;
        int ep = 7;
        if constexpr (LLOYD) {
            uint32_t bits = 0;
#pragma unroll
            for (uint32_t i = 0; i < kScaleMaxSlots; ++i) {
                bits = max(bits, p.v.alpha_max[region * kScaleMaxSlots + i]);
            }
            ep = bits ? 133 - (int)((bits >> 23) & 0xff) : 0;
            ep = ep > 100 ? 100 : (ep < -100 ? -100 : ep);
        }
        const float unscale = __uint_as_float((uint32_t)(127 - ep) << 23); // 2^-ep
        // The running maximum of a row's scores, in whole log2 units: what a score is moved by, ep - m_run, what older sums are scaled
        // by and what the merge scales partials by are exact then, so no two runs of a row differ in what they took off their
        // scores.  (Taken as it was, off the sum of ep and what the uniform coder's constant part adds to every score of a row, it was
        // rounded to that sum's size: queries of one sign and 100 normal values' width, 4-bit cells, errors 3.6e-5 -> 4.1e-5
        // of the result's norm.  A softmax does not depend on that part; m_first takes it off a run's first scores, which are as
        // large as it otherwise and rounded accordingly.)
        float m_run[QT], l_run[QT];
        float4v O[QT][JB]; // lane (c, g), register r: row 4 g + r of the tile, coordinate 16 jb + c
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            m_run[q] = -INFINITY;
            l_run[q] = 0.0f;
#pragma unroll
            for (int jb = 0; jb < JB; ++jb) {
                O[q][jb] = float4v{ 0.0f, 0.0f, 0.0f, 0.0f };
            }
        }

        // operands are read kAhead ahead of the matrix instructions that take them
        constexpr int kAhead = 2, kRing = kAhead + 2;
        half8 pa[QT][2][2]; // probabilities as A operands: [tile][half of the block][high, low]
        float4v S[QT][4];
        auto scores = [&](uint32_t buf) __attribute__((always_inline)) {
            const uint4v *from = reinterpret_cast<const uint4v *>(operands + buf * shared_block_bytes<D>()) + anew(lane);
            half8 ring[kRing];
            auto read = [&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i < ITEMS) {
                    ring[i % kRing] = __builtin_bit_cast(half8, from[((i % 4) * KS + i / 4) * 64]);
                }
            };
            static_for<0, kAhead>(read);
            // (operand i: tokens 16 (i % 4) .. + 15, coordinates 32 (i / 4) .. + 31; two at a time, so that a sum is next added to
            // four instructions on)
            static_for<0, ITEMS / 2>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = 2 * decltype(ic)::value, t = i % 4, ks = i / 4;
                read(std::integral_constant<int, i + kAhead>{});
                read(std::integral_constant<int, i + 1 + kAhead>{});
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        const half8 a = ring[(i + n) % kRing];
#pragma unroll
                        for (int q = 0; q < QT; ++q) {
                            if (ks == 0 && half == 0) {
                                S[q][t + n] = float4v{ 0.0f, 0.0f, 0.0f, 0.0f };
                            }
                            S[q][t + n] = mfma16(a, qop[q][half][ks], S[q][t + n]);
                        }
                    }
                }
            });
        };
        auto softmax = [&](uint32_t blk, uint32_t buf) __attribute__((always_inline)) {
            const uint32_t g = anew(lane) >> 4;
            const float4v *ak = reinterpret_cast<const float4v *>(scales + buf * 128) + g, *av = ak + 16;
#pragma unroll
            for (int q = 0; q < QT; ++q) {
                const float shift = (float)ep - (m_run[q] == -INFINITY ? m_first[q] : m_run[q]);
                float C[4][4]; // token 16 t + 4 g + r, row c, in log2 units above the running maximum, plus ep
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float4v k_scale = LLOYD ? ak[4 * t] : float4v{ p.k.alpha_const, p.k.alpha_const, p.k.alpha_const, p.k.alpha_const };
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        C[t][r] = fmaf(S[q][t][r], k_scale[r] * qscale[q], shift);
                    }
                }
                if (blk * 64 + 64 + hidden_max > L) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (blk * 64 + 16 * t + 4 * g + r + hidden[q] >= L) {
                                C[t][r] = -INFINITY;
                            }
                        }
                    }
                }
                float most = -INFINITY;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        most = fmaxf(most, C[t][r]);
                    }
                }
                most = head_max<16>(most);
                if (__any(most > (m_run[q] == -INFINITY ? -INFINITY : kSlack + (float)ep))) {
                    // (a chunk's early positions can have a whole block hidden before anything was seen: still -inf)
                    const float m_was = m_run[q] == -INFINITY ? m_first[q] : m_run[q];
                    const float m_new = fmaxf(m_run[q], __builtin_ceilf(most + (m_was - (float)ep)));
                    const float lower = m_new == -INFINITY ? 0.0f : m_was - m_new;
                    const float scale = (m_run[q] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run[q] - m_new);
                    l_run[q] *= scale;
                    float sr[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        sr[r] = __shfl(scale, (int)(4 * g + r));
                    }
#pragma unroll
                    for (int jb = 0; jb < JB; ++jb) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            O[q][jb][r] *= sr[r];
                        }
                    }
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            C[t][r] += lower;
                        }
                    }
                    m_run[q] = m_new;
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    uint4v hi, lo;
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const int t = 2 * u + half;
                        const float4v v_scale = LLOYD ? av[4 * t] : float4v{ 1.0f, 1.0f, 1.0f, 1.0f };
                        float pv[4];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float e = __builtin_amdgcn_exp2f(C[t][r]); // exp2(-inf) = 0 masks the tail
                            l_run[q] += e;
                            pv[r] = e * v_scale[r];
                        }
#pragma unroll
                        for (int h2 = 0; h2 < 2; ++h2) {
                            // hi = top 11 significant bits (fp16, towards zero), lo = the rest (exact, from hi as it came out) to the nearest
                            const float a0 = pv[2 * h2], a1 = pv[2 * h2 + 1];
                            const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a0, a1));
                            hi[2 * half + h2] = h;
                            lo[2 * half + h2] = __builtin_bit_cast(uint32_t, __builtin_convertvector(float2p{ less_low_half(a0, h), less_high_half(a1, h) }, half2p));
                        }
                    }
                    pa[q][u][0] = __builtin_bit_cast(half8, hi);
                    pa[q][u][1] = __builtin_bit_cast(half8, lo);
                }
            }
        };
        auto values = [&](uint32_t buf) __attribute__((always_inline)) {
            const uint4v *from = reinterpret_cast<const uint4v *>(operands + buf * shared_block_bytes<D>()) + ITEMS * 64 + anew(lane);
            half8 ring[kRing];
            auto read = [&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                if constexpr (i < ITEMS) {
                    ring[i % kRing] = __builtin_bit_cast(half8, from[i * 64]);
                }
            };
            static_for<0, kAhead>(read);
            static_for<0, ITEMS / 2>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = 2 * decltype(ic)::value, u = i / JB, jb = i % JB;
                read(std::integral_constant<int, i + kAhead>{});
                read(std::integral_constant<int, i + 1 + kAhead>{});
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        const half8 b = ring[(i + n) % kRing];
#pragma unroll
                        for (int q = 0; q < QT; ++q) {
                            O[q][jb + n] = mfma16(pa[q][u][half], b, O[q][jb + n]);
                        }
                    }
                }
            });
        };

        // ---- the blocks: one in LDS, the next one's packed words in registers ----
        __syncthreads(); // the tables are there; nobody reads the last segment's operands any more
        if (b0 < b1) {
            request(b0);
            unpack(b0, 0);
            request(min(b0 + 1, b1 - 1));
        }
        __syncthreads();
        for (uint32_t blk = b0; blk < b1; ++blk) {
            const uint32_t buf = (blk - b0) & 1;
            if (blk + 1 < b1) {
                unpack(blk + 1, buf ^ 1);
                request(min(blk + 2, b1 - 1));
            }
            if (works) {
                scores(buf);
                softmax(blk, buf);
                values(buf);
            }
            __syncthreads();
        }

        // ---- this segment's un-normalised partial (m, l, o[d]) per row ----
        constexpr int PS = D + 2;
        const float o_mul = unscale * (LLOYD ? 1.0f : p.v.alpha_const);
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            const float l_row = head_sum<16>(l_run[q]) * unscale; // every lane of a row now holds its denominator
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t hs = 16 * (QT * wave + q) + 4 * g + r;
                const float l = __shfl(l_row, (int)(4 * g + r));
                if (hs < p.G) {
                    float *dst = p.partials + (((uint64_t)seq * p.Hq + q_head_of(p, kvh, hs)) * p.max_slots + slot) * PS;
#pragma unroll
                    for (int jb = 0; jb < JB; ++jb) {
                        // uniform coder: value = step * (code + 0.5) + lo, so add lo * sum(p)
                        dst[2 + 16 * jb + c] = fmaf(O[q][jb][r], o_mul, p.v.beta * l);
                    }
                }
            }
            const uint32_t hs = 16 * (QT * wave + q) + c;
            if (g == 0 && hs < p.G) {
                float *dst = p.partials + (((uint64_t)seq * p.Hq + q_head_of(p, kvh, hs)) * p.max_slots + slot) * PS;
                dst[0] = m_run[q];
                dst[1] = l_row;
            }
        }
        if (kvh + 1 == p.Hkv && b0 + seg == nb_cap) {
            ++seq;
        }
    }
}

template <int D, bool LLOYD, bool NARROW> int launch_shared(const MfmaParams &p, hipStream_t s)
{
    constexpr size_t most = shared_lds_bytes<D>(256);
    static_assert(most <= 160u * 1024u, "tables and blocks exceed a compute unit's LDS");
    // once per instance and process, whichever host thread gets here first (the others wait for it)
    static std::once_flag configured;
    static hipError_t config_status = hipSuccess;
    std::call_once(configured, [] {
        config_status = hipFuncSetAttribute((const void *)decode_shared_kernel<D, LLOYD, NARROW>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
    });
    WEED_HIP_CHECK(config_status);
    if (p.tile_rows > mfma_decode_shared_rows || p.tile_rows * p.grid_passes < p.group_total || p.runs.skew || p.merge.wg_regions ||
        p.merge.region_wgs || p.merge.general || p.query.q) {
        return fail(WEED_HIP_EDEVICE, "decode_shared: rows or runs that the kernel does not take");
    }
    const uint32_t units = (p.total_blocks + p.runs.unit_blocks - 1) / p.runs.unit_blocks;
    const uint32_t grid = (units + 7) / 8 * 8 * p.grid_passes;
    decode_shared_kernel<D, LLOYD, NARROW>
        <<<grid, 64 * kSharedWaves, shared_lds_bytes<D>(mfma_table_rows(p.k.w, p.v.w)), s>>>(p);
    WEED_HIP_LAUNCH_CHECK();
    return WEED_HIP_OK;
}
template <int D> int launch_shared_d(const MfmaParams &p, hipStream_t s)
{
    const bool narrow = p.k.w <= 4 && p.v.w <= 4; // (their instances need none of the registers that the other widths' unpacking takes)
    if (p.k.alpha != nullptr) {
        return narrow ? launch_shared<D, true, true>(p, s) : launch_shared<D, true, false>(p, s);
    }
    return narrow ? launch_shared<D, false, true>(p, s) : launch_shared<D, false, false>(p, s);
}

} // namespace weedhip_mfma

namespace weedhip {

int launch_mfma_decode_shared(const MfmaParams &p, uint32_t d, hipStream_t s)
{
    switch (d) {
    case 64:
        return weedhip_mfma::launch_shared_d<64>(p, s);
    case 96:
        return weedhip_mfma::launch_shared_d<96>(p, s);
    case 128:
        return weedhip_mfma::launch_shared_d<128>(p, s);
    }
    return fail(WEED_HIP_EINVAL, "decode_shared: head_dim %u", d);
}

} // namespace weedhip
