// Fused single-query decode attention over the packed cache.
//
// One call does what MultiHeadAttention::forward does between the cache rebuild and the output projection when
// T = 1 (src/modules/multihead_attention.cpp:259-348): un-pack K and V, rotate q, Q.K^T, divide by sqrt(d), softmax
// over each sequence's own length, P.V, un-rotate -- without ever materialising the dense K, V, K^T, the replicated
// GQA copies or the score matrix the reference builds.
//
// Launches: (1) rotate the queries; (2) one workgroup per (context split, kv head, sequence) produces an
// un-normalised partial (running max m, running sum l, o[d]) per query head; (3) merge the partials of all splits,
// normalise and un-rotate.
#include "kv_cache.h"
#include "kv_decode_mfma.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>

using namespace weedhip;
using namespace weedkv;

// Workspace of weed_hip_kv_decode_attn_noalloc: rotated queries, their fp16 halves, block offsets and the split
// partials of one call.  Every device the library runs on holds its own copy until the process ends; in host code the
// array's name is only a handle for hipGetSymbolAddress, the kernels get the address kept in g_scratch_dev.
constexpr size_t kStaticScratchBytes = 32u << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
void *g_scratch_dev[kMaxDevices] = {};
__global__ void __launch_bounds__(256) clear_words_kernel(uint32_t *p, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        p[i] = 0u;
    }
}
} // namespace

namespace weedhip {
// Called by weed_hip_init with `device_id` current: looks the device's copy of `scratch` up once.
int decode_scratch_setup(int device_id)
{
    if (device_id < 0 || device_id >= kMaxDevices) {
        return fail(WEED_HIP_EINVAL, "decode_scratch_setup: device %d outside [0, %d)", device_id, kMaxDevices);
    }
    if (!g_scratch_dev[device_id]) {
        void *ptr = nullptr;
        WEED_HIP_CHECK(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
        g_scratch_dev[device_id] = ptr;
    }
    return WEED_HIP_OK;
}
uint32_t *decode_scratch_counters()
{
    const int dev = current_device();
    return dev < 0 || dev >= kMaxDevices ? nullptr : static_cast<uint32_t *>(g_scratch_dev[dev]);
}

int decode_scratch_clear_counters()
{
    uint32_t *counters = decode_scratch_counters();
    if (!counters) {
        return WEED_HIP_OK; // the library has not been started on this device: nothing to clear
    }
    clear_words_kernel<<<(kMfmaMergeCounters + 255) / 256, 256, 0, stream()>>>(counters, kMfmaMergeCounters);
    WEED_HIP_LAUNCH_CHECK();
    return WEED_HIP_OK;
}
} // namespace weedhip

namespace {

constexpr int kGMax = 8;        // query heads of one kv head handled per pass
constexpr int kThreads = 256;
constexpr int kChunk = 256;     // tokens per inner iteration of the generic kernel

struct DecodeParams {
    SideParams k, v;
    const int32_t *lens;
    uint32_t padded;
    uint32_t d;      // head_dim as stored (a multiple of 32)
    uint32_t d_real; // the caller's head_dim (the scores are divided by its square root)
    uint32_t Hq, Hkv, G;
    int blocked; // 1: kv = h / G, 0: kv = h % Hkv (Weed)
    const float *q_rot; // [n_seq][Hq][d]
    float *partials;    // [n_seq][Hq][n_splits][d + 2]
    uint32_t n_splits, split_tokens;
};

__device__ __forceinline__ uint32_t q_head_of(const DecodeParams &p, uint32_t kvh, uint32_t g)
{
    return p.blocked ? (kvh * p.G + g) : (g * p.Hkv + kvh);
}

// blk_off[i] = number of 64-token blocks of the sequences before i, blk_off[n_seq] = all of them.  One workgroup of
// 256 threads: every thread sums a chunk, the chunk sums are scanned in LDS.
__device__ void block_offsets(const int32_t *__restrict__ lens, uint32_t n_seq, uint32_t *__restrict__ blk_off)
{
    __shared__ uint32_t chunk_sum[256];
    const uint32_t tid = threadIdx.x;
    const uint32_t per = (n_seq + 255) / 256;
    const uint32_t i0 = min(tid * per, n_seq), i1 = min(i0 + per, n_seq);
    uint32_t mine = 0;
    for (uint32_t i = i0; i < i1; ++i) {
        mine += ((uint32_t)lens[i] + 63u) >> 6;
    }
    chunk_sum[tid] = mine;
    __syncthreads();
    for (uint32_t k = 1; k < 256; k <<= 1) {
        const uint32_t add = tid >= k ? chunk_sum[tid - k] : 0;
        __syncthreads();
        chunk_sum[tid] += add;
        __syncthreads();
    }
    uint32_t run = chunk_sum[tid] - mine; // exclusive prefix of this thread's chunk
    for (uint32_t i = i0; i < i1; ++i) {
        blk_off[i] = run;
        run += ((uint32_t)lens[i] + 63u) >> 6;
    }
    if (tid == 255) {
        blk_off[n_seq] = chunk_sum[255];
    }
    __syncthreads();
}

// q_rot[s][h][:] = q[s][h][:] . Rk  (multihead_attention.cpp:276), or a plain gather when rotate == 0.
// For the matrix-core kernel the rotated query is also scaled by log2(e)/sqrt(d), divided by a power of two that
// brings it into [-1, 1], and split into fp16 hi + lo halves.
// `d`: head_dim as stored (a multiple of 32); `d_real` <= d: coordinates the caller's query has (zeros beyond them).
__global__ void __launch_bounds__(256) prep_q_kernel(const float *__restrict__ q, Geom3 g, uint32_t Hq, uint32_t d,
                                                     uint32_t d_real, const float *__restrict__ rot_t, int rotate,
                                                     float *__restrict__ q_rot, uint16_t *__restrict__ q_hi,
                                                     uint16_t *__restrict__ q_lo, float *__restrict__ q_scale,
                                                     float *__restrict__ q_sum, const int32_t *__restrict__ lens,
                                                     uint32_t n_seq, uint32_t *__restrict__ blk_off)
{
    __shared__ float qs[256];
    __shared__ float red_max[256];
    __shared__ float red_sum[256];
    const uint32_t h = blockIdx.x, s = blockIdx.y;
    const uint32_t tid = threadIdx.x;
    if (s == n_seq) {
        // the extra grid row: one of its workgroups builds the block offsets while the others rotate queries (as part
        // of a query's workgroup the scan would be the kernel's longest chain)
        if (blk_off && h == 0) {
            block_offsets(lens, n_seq, blk_off);
        }
        return;
    }
    if (tid < d) {
        qs[tid] = tid < d_real
                      ? q[(uint64_t)g.off + (uint64_t)s * g.s[0] + head_offset(g, h) + (uint64_t)tid * g.s[2]]
                      : 0.0f;
    }
    __syncthreads();
    float acc = 0.0f;
    if (tid < d) {
        if (rotate) {
            for (uint32_t i = 0; i < d; ++i) {
                acc = fmaf(qs[i], rot_t[tid + d * i], acc);
            }
        } else {
            acc = qs[tid];
        }
        q_rot[((uint64_t)s * Hq + h) * d + tid] = acc;
    }
    const float qc = acc * (1.4426950408889634f / sqrtf((float)d_real));
    red_max[tid] = fabsf(qc);
    red_sum[tid] = qc;
    __syncthreads();
    for (uint32_t k = 128; k > 0; k >>= 1) {
        if (tid < k) {
            red_max[tid] = fmaxf(red_max[tid], red_max[tid + k]);
            red_sum[tid] += red_sum[tid + k];
        }
        __syncthreads();
    }
    int e = 0;
    (void)frexpf(red_max[0], &e); // max = f * 2^e with f in [0.5, 1), so 2^e exceeds every |qc|
    e = e < -100 ? -100 : (e > 100 ? 100 : e);
    const float inv = ldexpf(1.0f, -e);
    if (tid < d) {
        const float qn = qc * inv;
        const _Float16 hi = (_Float16)qn;
        const _Float16 lo = (_Float16)(qn - (float)hi);
        q_hi[((uint64_t)s * Hq + h) * d + tid] = __builtin_bit_cast(uint16_t, hi);
        q_lo[((uint64_t)s * Hq + h) * d + tid] = __builtin_bit_cast(uint16_t, lo);
    }
    if (tid == 0) {
        q_scale[(uint64_t)s * Hq + h] = ldexpf(1.0f, e);
        q_sum[(uint64_t)s * Hq + h] = red_sum[0];
    }
}

__device__ __forceinline__ float wave_max(float v)
{
    for (int o = 32; o > 0; o >>= 1) {
        v = fmaxf(v, __shfl_xor(v, o));
    }
    return v;
}

__device__ __forceinline__ float wave_sum(float v)
{
    for (int o = 32; o > 0; o >>= 1) {
        v += __shfl_xor(v, o);
    }
    return v;
}

constexpr int kRowsPerWg = 4;

// The same as prep_q_kernel for kRowsPerWg (sequence, head) rows per workgroup: thread j owns output coordinate j of
// every row, so each element of the rotation is read once per workgroup instead of once per row.  Used when there
// are many rows (batched decode); results are identical (same order of fused multiply-adds).
__global__ void __launch_bounds__(256) prep_q_rows_kernel(const float *__restrict__ q, Geom3 g, uint32_t Hq, uint32_t d,
                                                          uint32_t d_real, uint32_t n_rows,
                                                          const float *__restrict__ rot_t, int rotate,
                                                          float *__restrict__ q_rot, uint16_t *__restrict__ q_hi,
                                                          uint16_t *__restrict__ q_lo, float *__restrict__ q_scale,
                                                          float *__restrict__ q_sum, const int32_t *__restrict__ lens,
                                                          uint32_t n_seq, uint32_t *__restrict__ blk_off)
{
    __shared__ float qs[kRowsPerWg][256];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t row0 = blockIdx.x * kRowsPerWg;
    // The rotation does not depend on the query: its first 64 elements per thread are requested before anything else,
    // so that they travel together with the query rows (one round trip to memory instead of two).  d is a multiple of
    // 64 here (the host checks).
    const bool rot_thread = rotate && tid < d;
    float x0[64];
    auto request = [&](float (&x)[64], uint32_t i0) {
#pragma unroll
        for (int u = 0; u < 64; ++u) {
            x[u] = rot_t[tid + d * (i0 + u)];
        }
    };
    if (blockIdx.x * kRowsPerWg >= n_rows) {
        // the extra workgroup behind the last rows: it builds the block offsets while the others rotate queries (as
        // part of a query's workgroup the scan would be the kernel's longest chain)
        if (blk_off) {
            block_offsets(lens, n_seq, blk_off);
        }
        return;
    }
    if (rot_thread) {
        request(x0, 0);
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWg; ++r) {
        const uint32_t row = row0 + r;
        float v = 0.0f;
        if (row < n_rows && tid < d_real) {
            const uint32_t s = row / Hq, h = row % Hq;
            v = q[(uint64_t)g.off + (uint64_t)s * g.s[0] + head_offset(g, h) + (uint64_t)tid * g.s[2]];
        }
        qs[r][tid] = v;
    }
    __syncthreads();
    float acc[kRowsPerWg];
#pragma unroll
    for (int r = 0; r < kRowsPerWg; ++r) {
        acc[r] = rotate ? 0.0f : qs[r][tid];
    }
    if (rot_thread) {
        // sixty-four elements at a time (same order of fused multiply-adds as the single-row kernel)
        for (uint32_t i0 = 0; i0 < d; i0 += 64) {
            if (i0) {
                request(x0, i0);
            }
#pragma unroll
            for (int u = 0; u < 64; ++u) {
#pragma unroll
                for (int r = 0; r < kRowsPerWg; ++r) {
                    acc[r] = fmaf(qs[r][i0 + u], x0[u], acc[r]);
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRowsPerWg; ++r) {
        qs[r][tid] = tid < d ? acc[r] : 0.0f;
    }
    __syncthreads();
    // one wavefront per row from here on
    for (uint32_t r = wave; r < (uint32_t)kRowsPerWg; r += 4) {
        const uint32_t row = row0 + r;
        if (row >= n_rows) {
            break;
        }
        const float k = 1.4426950408889634f / sqrtf((float)d_real);
        float mx = 0.0f, sum = 0.0f;
        for (uint32_t j = lane; j < d; j += 64) {
            const float qc = qs[r][j] * k;
            mx = fmaxf(mx, fabsf(qc));
            sum += qc;
        }
        mx = wave_max(mx);
        // the single-row kernel adds the coordinates pairwise over 256 slots; keep its summation tree: fold 64 lanes
        sum = wave_sum(sum);
        int e = 0;
        (void)frexpf(mx, &e);
        e = e < -100 ? -100 : (e > 100 ? 100 : e);
        const float inv = ldexpf(1.0f, -e);
        for (uint32_t j = lane; j < d; j += 64) {
            const float a = qs[r][j];
            const float qn = a * k * inv;
            const _Float16 hi = (_Float16)qn;
            const _Float16 lo = (_Float16)(qn - (float)hi);
            q_rot[(uint64_t)row * d + j] = a;
            q_hi[(uint64_t)row * d + j] = __builtin_bit_cast(uint16_t, hi);
            q_lo[(uint64_t)row * d + j] = __builtin_bit_cast(uint16_t, lo);
        }
        if (lane == 0) {
            q_scale[row] = ldexpf(1.0f, e);
            q_sum[row] = sum;
        }
    }
}

// ---- Queries and merges of many rows (chunks of positions, long lists of sequences) by tiles --------------------------
//
// Order in which the tiles take the (sequence, head) rows of a call: three nested dimensions, the fastest first, each with
// its extent, its step in the caller's tensor and its step in the row number s * Hq + hv.
struct RowOrder {
    uint32_t n0, n1;
    uint32_t x[3];   // elements of the caller's tensor
    uint32_t row[3]; // rows
};

__device__ __forceinline__ void row_of(const RowOrder &o, uint32_t e, uint32_t &row, uint64_t &at)
{
    const uint32_t rest = e / o.n0, i0 = e - rest * o.n0, i2 = rest / o.n1, i1 = rest - i2 * o.n1;
    row = i0 * o.row[0] + i1 * o.row[1] + i2 * o.row[2];
    at = (uint64_t)i0 * o.x[0] + (uint64_t)i1 * o.x[1] + (uint64_t)i2 * o.x[2];
}

// Rows per tile: two 32-row tiles of the matrix instruction up to head_dim 128, one above (32 KB of LDS either way).
constexpr uint32_t tile_rows_of(uint32_t nt) { return nt <= 4 ? 64u : 32u; }

typedef float float16acc __attribute__((ext_vector_type(16)));

// xs[R][d + 4] (in LDS) becomes xs . M with M[k][n] = m[n + d k], in place, on the fp32 matrix instruction
// (v_mfma_f32_32x32x2f32).  Four wavefronts share the (row tile, column tile) pairs; a wavefront keeps its column tile's
// part of M in registers for its row tiles.  The contraction index of an instruction may be any pair as long as both
// operands agree: step i of eight k takes 8 i + 4 (lane / 32) + j in its instruction j, so that the rows come from LDS
// in 16-byte pieces.  `b` comes with the wavefront's first column tile's first KC / 2 elements (load).
template <int NT> struct TileRotation {
    static constexpr uint32_t D = 32 * NT, R = tile_rows_of(NT), PITCH = D + 4;
    static constexpr uint32_t KC = NT <= 4 ? D : D / 2;                         // k per round of loads
    static constexpr uint32_t CW = NT >= 4 ? 4 : (NT >= 2 ? 2 : 1);             // wavefronts side by side over the columns
    static constexpr uint32_t RW = 4 / CW;                                      // ... and over the row tiles
    static constexpr uint32_t RT = (R / 32 + RW - 1) / RW;                      // row tiles per wavefront
    static constexpr uint32_t CT = (NT + CW - 1) / CW;                          // column tiles per wavefront

    static __device__ __forceinline__ void load(float (&b)[KC / 2], const float *__restrict__ m, uint32_t ct, uint32_t k0)
    {
        const uint32_t lane = threadIdx.x & 63;
        const float *src = m + 32 * ct + (lane & 31) + D * (k0 + 4 * (lane >> 5));
#pragma unroll
        for (uint32_t u = 0; u < KC / 2; ++u) {
            b[u] = src[D * (8 * (u / 4) + u % 4)];
        }
    }
    static __device__ __forceinline__ uint32_t first_column_tile() { return (threadIdx.x >> 6) % CW; }

    static __device__ __forceinline__ void run(float *xs, const float *__restrict__ m, float (&b)[KC / 2])
    {
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const uint32_t l32 = lane & 31, lk = lane >> 5, rw = wave / CW;
        float16acc acc[CT][RT];
#pragma unroll
        for (uint32_t c = 0; c < CT; ++c) {
            const uint32_t ct = wave % CW + c * CW;
#pragma unroll
            for (uint32_t t = 0; t < RT; ++t) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    acc[c][t][i] = 0.0f;
                }
            }
            if (ct < NT) {
#pragma unroll
                for (uint32_t k0 = 0; k0 < D; k0 += KC) {
                    if (c || k0) {
                        load(b, m, ct, k0);
                        // All of them requested before the first product: left alone, the compiler moves each load next to
                        // the product that takes it, a trip to the second-level cache per instruction (a tile at head_dim
                        // 96, 192 or 256 took 24, 43 or 53 us so, 8, 13 or 16 with the loads together).
#pragma unroll
                        for (uint32_t u = 0; u < KC / 2; ++u) {
                            asm volatile("" : "+v"(b[u]));
                        }
                    }
#pragma unroll
                    for (uint32_t t = 0; t < RT; ++t) {
                        const uint32_t rt = rw + t * RW;
                        if (rt < R / 32) {
                            const float *row = xs + (32 * rt + l32) * PITCH + k0 + 4 * lk;
#pragma unroll
                            for (uint32_t i = 0; i < KC / 8; ++i) {
                                const float4 a = *reinterpret_cast<const float4 *>(row + 8 * i);
                                acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b[4 * i], acc[c][t], 0, 0, 0);
                                acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b[4 * i + 1], acc[c][t], 0, 0, 0);
                                acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b[4 * i + 2], acc[c][t], 0, 0, 0);
                                acc[c][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b[4 * i + 3], acc[c][t], 0, 0, 0);
                            }
                        }
                    }
                }
            }
        }
        __syncthreads(); // everybody has read the rows
#pragma unroll
        for (uint32_t c = 0; c < CT; ++c) {
            const uint32_t ct = wave % CW + c * CW;
#pragma unroll
            for (uint32_t t = 0; t < RT; ++t) {
                const uint32_t rt = rw + t * RW;
                if (ct < NT && rt < R / 32) {
#pragma unroll
                    for (uint32_t i = 0; i < 16; ++i) {
                        xs[(32 * rt + 8 * (i / 4) + 4 * lk + i % 4) * PITCH + 32 * ct + l32] = acc[c][t][i];
                    }
                }
            }
        }
        __syncthreads();
    }
};

// How the rows of a tile lie in the caller's tensor: coordinates contiguous in 16-byte pieces (1), else (0) the lanes walk
// the rows, which the order above puts next to each other where the tensor does (a column-major layer's sequences).
template <int NT>
__device__ __forceinline__ void gather_tile(float *xs, const float *__restrict__ q, const uint64_t *at, uint32_t s_coord,
                                            int wide, uint32_t d_real)
{
    constexpr uint32_t D = 32 * NT, R = tile_rows_of(NT), PITCH = D + 4;
    const uint32_t tid = threadIdx.x;
    if (wide) {
        // eight lanes per row and 32 coordinates: a wavefront reads 128 consecutive bytes of eight rows
        const uint32_t j = 4 * (tid & 7);
#pragma unroll
        for (uint32_t r0 = 0; r0 < R; r0 += 32) {
            const uint32_t r = r0 + (tid >> 3);
            const uint64_t a = at[r];
            float4 v[NT];
#pragma unroll
            for (uint32_t c = 0; c < NT; ++c) {
                v[c] = (a != ~0ull && j + 32 * c < d_real) ? *reinterpret_cast<const float4 *>(q + a + j + 32 * c)
                                                          : float4{ 0.0f, 0.0f, 0.0f, 0.0f };
            }
#pragma unroll
            for (uint32_t c = 0; c < NT; ++c) {
                *reinterpret_cast<float4 *>(xs + r * PITCH + j + 32 * c) = v[c];
            }
        }
        return;
    }
    const uint32_t r = tid % R;
    const uint64_t a = at[r];
    constexpr uint32_t STEP = 256 / R; // coordinate quads taken at a time
#pragma unroll
    for (uint32_t c0 = 0; c0 < D / 4; c0 += 2 * STEP) {
        float v[2][4];
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u) {
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e) {
                const uint32_t j = 4 * (c0 + u * STEP + tid / R) + e;
                v[u][e] = (a != ~0ull && j < d_real) ? q[a + (uint64_t)j * s_coord] : 0.0f;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < 2; ++u) {
            const uint32_t c = c0 + u * STEP + tid / R;
            if (c < D / 4) {
                *reinterpret_cast<float4 *>(xs + r * PITCH + 4 * c) = float4{ v[u][0], v[u][1], v[u][2], v[u][3] };
            }
        }
    }
}

// prep_q_kernel for many rows, a tile of 32 or 64 of them per workgroup with the rotation on the matrix instruction (the
// row kernels above multiply 4 rows per 64 KB of the rotation on the vector unit, and a lane that walks the coordinates
// of a column-major query touches a cache line per element).  16 x 64 positions of 32 heads of 128: 64 us by rows,
// 18-20 here; 32 x 64 positions of a column-major query: 129 and 33 (the rows' bytes in and out take 6 and 12 us at 5.5 TB/s,
// the fp32 instruction's products 7 and 14).
template <int NT>
__global__ void __launch_bounds__(256) prep_q_tile_kernel(const float *__restrict__ q, uint32_t q_off, uint32_t s_coord,
                                                          RowOrder order, int wide, uint32_t d_real, uint32_t n_rows,
                                                          const float *__restrict__ rot_t, int rotate,
                                                          float *__restrict__ q_rot, uint16_t *__restrict__ q_hi,
                                                          uint16_t *__restrict__ q_lo, float *__restrict__ q_scale,
                                                          float *__restrict__ q_sum, const int32_t *__restrict__ lens,
                                                          uint32_t n_seq, uint32_t *__restrict__ blk_off)
{
    typedef TileRotation<NT> Rot;
    constexpr uint32_t D = Rot::D, R = Rot::R, PITCH = Rot::PITCH;
    __shared__ __attribute__((aligned(16))) float xs[R * PITCH];
    __shared__ uint64_t at_s[R];
    __shared__ uint32_t row_s[R];
    const uint32_t tid = threadIdx.x, e0 = blockIdx.x * R;
    if (e0 >= n_rows) { // the extra workgroup behind the last rows
        if (blk_off) {
            block_offsets(lens, n_seq, blk_off);
        }
        return;
    }
    float b[Rot::KC / 2];
    if (rotate) {
        Rot::load(b, rot_t, Rot::first_column_tile(), 0);
    }
    if (tid < R) {
        uint32_t row = 0;
        uint64_t at = ~0ull;
        if (e0 + tid < n_rows) {
            row_of(order, e0 + tid, row, at);
            at += q_off;
        }
        at_s[tid] = at;
        row_s[tid] = row;
    }
    __syncthreads();
    gather_tile<NT>(xs, q, at_s, s_coord, wide, d_real);
    __syncthreads();
    if (rotate) {
        Rot::run(xs, rot_t, b);
    }
    // eight lanes per row
    const uint32_t l8 = tid & 7;
    const float k = 1.4426950408889634f / sqrtf((float)d_real);
#pragma unroll
    for (uint32_t r0 = 0; r0 < R; r0 += 32) {
        const uint32_t r = r0 + (tid >> 3);
        float4 y[NT];
        float mx = 0.0f, sum = 0.0f;
#pragma unroll
        for (uint32_t c = 0; c < NT; ++c) {
            y[c] = *reinterpret_cast<const float4 *>(xs + r * PITCH + 4 * l8 + 32 * c);
            mx = fmaxf(fmaxf(mx, fmaxf(fabsf(y[c].x * k), fabsf(y[c].y * k))), fmaxf(fabsf(y[c].z * k), fabsf(y[c].w * k)));
            sum += (y[c].x * k + y[c].y * k) + (y[c].z * k + y[c].w * k);
        }
#pragma unroll
        for (int o = 4; o > 0; o >>= 1) {
            mx = fmaxf(mx, __shfl_xor(mx, o));
            sum += __shfl_xor(sum, o);
        }
        int e = 0;
        (void)frexpf(mx, &e);
        e = e < -100 ? -100 : (e > 100 ? 100 : e);
        const float inv = ldexpf(1.0f, -e);
        if (e0 + r < n_rows) {
            const uint32_t row = row_s[r];
#pragma unroll
            for (uint32_t c = 0; c < NT; ++c) {
                const float v[4] = { y[c].x, y[c].y, y[c].z, y[c].w };
                uint32_t hw[2], lw[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    uint32_t h2 = 0, l2 = 0;
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const float qn = v[2 * i + u] * k * inv;
                        const _Float16 hi = (_Float16)qn;
                        const _Float16 lo = (_Float16)(qn - (float)hi);
                        h2 |= (uint32_t)__builtin_bit_cast(uint16_t, hi) << (16 * u);
                        l2 |= (uint32_t)__builtin_bit_cast(uint16_t, lo) << (16 * u);
                    }
                    hw[i] = h2;
                    lw[i] = l2;
                }
                const uint64_t dst = (uint64_t)row * D + 4 * l8 + 32 * c;
                *reinterpret_cast<uint2 *>(q_hi + dst) = uint2{ hw[0], hw[1] };
                *reinterpret_cast<uint2 *>(q_lo + dst) = uint2{ lw[0], lw[1] };
                if (q_rot) {
                    *reinterpret_cast<float4 *>(q_rot + dst) = y[c];
                }
            }
            if (l8 == 0) {
                q_scale[row] = ldexpf(1.0f, e);
                q_sum[row] = sum;
            }
        }
    }
}

// Generic kernel: any head_dim that is a multiple of 32, any field width, any group size.
__global__ void __launch_bounds__(kThreads) decode_generic_kernel(DecodeParams p)
{
    __shared__ float q_s[kGMax * 256];
    __shared__ float qsum_s[kGMax];
    __shared__ float sc[kGMax * kChunk];
    __shared__ float m_s[kGMax], l_s[kGMax], scale_s[kGMax];
    __shared__ float o_s[kGMax * 256];
    __shared__ float ktab[256], vtab[256];

    const uint32_t split = blockIdx.x, kvh = blockIdx.y, seq = blockIdx.z;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t d = p.d;
    const uint32_t L = (uint32_t)p.lens[seq];
    const uint32_t n0 = split * p.split_tokens;
    const uint32_t n1 = min(L, n0 + p.split_tokens);
    const uint64_t region = (uint64_t)seq * p.Hkv + kvh;
    const float sqrt_d = sqrtf((float)p.d_real);
    const uint32_t parts = kThreads / d ? kThreads / d : 1;
    const uint32_t part = tid / d, jj = tid % d;
    const bool pv_active = part < parts;

    // fields wider than 5 bits exist in the uniform coder only, whose table is code + 0.5
    static_assert(kThreads == 256, "one table entry per thread");
    ktab[tid] = p.k.w > 5U ? (float)tid + 0.5f : p.k.table[tid & 31U];
    vtab[tid] = p.v.w > 5U ? (float)tid + 0.5f : p.v.table[tid & 31U];

    for (uint32_t hc = 0; hc < p.G; hc += kGMax) {
        const uint32_t gh = min((uint32_t)kGMax, p.G - hc);
        __syncthreads();
        for (uint32_t e = tid; e < gh * d; e += kThreads) {
            const uint32_t h = e / d, j = e % d;
            q_s[h * 256 + j] = p.q_rot[((uint64_t)seq * p.Hq + q_head_of(p, kvh, hc + h)) * d + j];
        }
        if (tid < kGMax) {
            m_s[tid] = -INFINITY;
            l_s[tid] = 0.0f;
        }
        __syncthreads();
        if (tid < gh) {
            float s = 0.0f;
            for (uint32_t j = 0; j < d; ++j) {
                s += q_s[tid * 256 + j];
            }
            qsum_s[tid] = s;
        }
        float o[kGMax];
#pragma unroll
        for (int h = 0; h < kGMax; ++h) {
            o[h] = 0.0f;
        }
        __syncthreads();

        for (uint32_t c0 = n0; c0 < n1; c0 += kChunk) {
            // ---- scores for token c0 + tid ----
            const uint32_t n = c0 + tid;
            float acc[kGMax];
#pragma unroll
            for (int h = 0; h < kGMax; ++h) {
                acc[h] = 0.0f;
            }
            if (n < n1) {
                const uint8_t *kbase = p.k.fields + region * p.k.region_bytes;
                for (uint32_t j0 = 0; j0 < d; j0 += 8) {
                    const uint8_t *item = kbase + k_field_pos(n, j0, d, p.k.w).byte;
                    for (uint32_t e = 0; e < 8; ++e) {
                        const float kv = ktab[item_get(item, e * p.k.w, p.k.w)];
#pragma unroll
                        for (int h = 0; h < kGMax; ++h) {
                            acc[h] = fmaf(q_s[h * 256 + j0 + e], kv, acc[h]);
                        }
                    }
                }
                const float a = p.k.alpha ? p.k.alpha[region * p.padded + n] : p.k.alpha_const;
#pragma unroll
                for (int h = 0; h < kGMax; ++h) {
                    if ((uint32_t)h < gh) {
                        sc[h * kChunk + tid] = (a * acc[h] + p.k.beta * qsum_s[h]) / sqrt_d;
                    }
                }
            } else {
#pragma unroll
                for (int h = 0; h < kGMax; ++h) {
                    sc[h * kChunk + tid] = -INFINITY;
                }
            }
            __syncthreads();
            // ---- running softmax statistics, one wave per head ----
            for (uint32_t h = wave; h < gh; h += kThreads / 64) {
                float v[kChunk / 64];
                float mx = -INFINITY;
#pragma unroll
                for (int k = 0; k < kChunk / 64; ++k) {
                    v[k] = sc[h * kChunk + lane + 64 * k];
                    mx = fmaxf(mx, v[k]);
                }
                mx = wave_max(mx);
                const float m_old = m_s[h];
                const float m_new = fmaxf(m_old, mx);
                float sum = 0.0f;
#pragma unroll
                for (int k = 0; k < kChunk / 64; ++k) {
                    const float e = (v[k] == -INFINITY) ? 0.0f : expf(v[k] - m_new);
                    sc[h * kChunk + lane + 64 * k] = e;
                    sum += e;
                }
                sum = wave_sum(sum);
                if (lane == 0) {
                    const float scale = (m_old == -INFINITY) ? 0.0f : expf(m_old - m_new);
                    scale_s[h] = scale;
                    l_s[h] = l_s[h] * scale + sum;
                    m_s[h] = m_new;
                }
            }
            __syncthreads();
            // ---- o += p . V, thread = (token slice, coordinate) ----
            if (pv_active) {
#pragma unroll
                for (int h = 0; h < kGMax; ++h) {
                    if ((uint32_t)h < gh) {
                        o[h] *= scale_s[h];
                    }
                }
                const uint32_t cnt = min((uint32_t)kChunk, n1 - c0);
                const uint8_t *vbase = p.v.fields + region * p.v.region_bytes;
                for (uint32_t nl = part; nl < cnt; nl += parts) {
                    const uint32_t nn = c0 + nl;
                    const FieldPos vp = v_field_pos(nn, jj, d, p.v.w);
                    const float a = p.v.alpha ? p.v.alpha[region * p.padded + nn] : p.v.alpha_const;
                    const float vv = fmaf(a, vtab[item_get(vbase + vp.byte, vp.bit, p.v.w)], p.v.beta);
#pragma unroll
                    for (int h = 0; h < kGMax; ++h) {
                        if ((uint32_t)h < gh) {
                            o[h] = fmaf(sc[h * kChunk + nl], vv, o[h]);
                        }
                    }
                }
            }
            __syncthreads();
        }

        // ---- fold the token slices together and emit the partial ----
        for (uint32_t r = 0; r < parts; ++r) {
            if (pv_active && part == r) {
#pragma unroll
                for (int h = 0; h < kGMax; ++h) {
                    if ((uint32_t)h < gh) {
                        o_s[h * 256 + jj] = (r ? o_s[h * 256 + jj] : 0.0f) + o[h];
                    }
                }
            }
            __syncthreads();
        }
        for (uint32_t e = tid; e < gh * d; e += kThreads) {
            const uint32_t h = e / d, j = e % d;
            const uint32_t qh = q_head_of(p, kvh, hc + h);
            float *dst = p.partials + (((uint64_t)seq * p.Hq + qh) * p.n_splits + split) * (d + 2);
            dst[2 + j] = o_s[h * 256 + j];
            if (j == 0) {
                dst[0] = m_s[h];
                dst[1] = l_s[h];
            }
        }
    }
}

// Merge the partials of all splits: out = sum_s e^(m_s - M) o_s / sum_s e^(m_s - M) l_s, then multiply by
// v_rotation^T (multihead_attention.cpp:343-348): out_i = sum_j O_j Rv[i + d*j].
constexpr uint32_t kMaxSlots = 1024; // partials per (sequence, head) that combine_kernel can weigh in one pass

// Run-length skew between the wavefront age classes of a workgroup, in percent of the mean run (see RunGeom): with
// two wavefronts per SIMD the older one gets 16 % more than the mean; with three the spread between oldest and
// youngest is wider (measured on the ragged batch: 16 % -> 47.8 us, 24-40 % -> 46.7-46.9 us, 48 % -> 48.2 us).
constexpr uint32_t kRunSkewPercent = 16, kRunSkewPercent3 = 28;
// Most regions that the blocks of one workgroup may lie in for the workgroups to merge their regions themselves in the
// general case (see decode_impl).
constexpr uint32_t kMostRegionsMergedByWorkgroup = 6;
// ... and most rows (region, head) of them: two passes of the merge (96 sequences of 2100 or 5000 tokens with four heads
// per kv head, five regions = 20 rows per workgroup: 59.2 and 116.8 us, against 51.2 and 111.9 with the merge kernel)
constexpr uint32_t kMostRowsMergedByWorkgroup = 16;

// Tuning knobs of the work partition.  The defaults come from the environment, read ONCE per process (at the first
// decode call or the first weed_hip_kv_decode_tuning): WEED_HIP_DECODE_WAVES (wavefronts the block list is cut for),
// WEED_HIP_DECODE_SKEW (percent), WEED_HIP_DECODE_SEARCH=1 (always find a wavefront's first region by search, even in
// a batch of equal contexts).
// Shortest and longest mean run for which neighbouring runs take their blocks in turns (see RunGeom::group_cycles).
constexpr uint32_t kFewestBlocksOfRunsInTurns = 4, kMostBlocksOfRunsInTurns = 32;
struct DecodeTuning {
    int wavefronts = 0;    // 0: as many as the device holds at once
    int skew_percent = -1; // < 0: kRunSkewPercent
    bool always_search = false;
    bool separate_merge = false; // always merge the partials with the second kernel
    bool separate_query = false; // always rotate the queries with the kernel ahead
    bool contiguous_runs = false; // never let neighbouring runs take turns (RunGeom::group_cycles)
    bool print_plan = false;      // WEED_HIP_DECODE_PLAN=1: every call writes its partition to stderr
};
DecodeTuning &decode_tuning()
{
    static DecodeTuning t = [] {
        DecodeTuning v;
        if (const char *env = std::getenv("WEED_HIP_DECODE_WAVES")) {
            v.wavefronts = std::max(0, std::atoi(env));
        }
        if (const char *env = std::getenv("WEED_HIP_DECODE_SKEW")) {
            v.skew_percent = std::atoi(env);
        }
        if (const char *env = std::getenv("WEED_HIP_DECODE_SEARCH")) {
            v.always_search = (std::atoi(env) & 1) != 0;
            v.separate_merge = (std::atoi(env) & 2) != 0;
            v.separate_query = (std::atoi(env) & 4) != 0;
            v.contiguous_runs = (std::atoi(env) & 8) != 0;
        }
        if (const char *env = std::getenv("WEED_HIP_DECODE_PLAN")) {
            v.print_plan = std::atoi(env) != 0;
        }
        return v;
    }();
    return t;
}

struct SlotGeom {
    const uint32_t *blk_off; // null: every (sequence, head) has `max_slots` valid partials
    uint32_t Hkv, G;
    RunGeom runs; // matrix-core kernel: how the block list was cut into per-wavefront runs
    int blocked;
    uint32_t uniform_blocks; // blocks per sequence when all sequences span the same number (blk_off is then not read:
                             // nothing may have computed it), else 0
};

// Partial slots of head h of sequence s: the wavefronts whose runs intersect the head's region, in order.
__device__ __forceinline__ uint32_t slots_of_row(const SlotGeom &sg, uint32_t s, uint32_t h)
{
    const uint32_t first_blk = sg.uniform_blocks ? s * sg.uniform_blocks : sg.blk_off[s];
    const uint32_t nb = sg.uniform_blocks ? sg.uniform_blocks : sg.blk_off[s + 1] - first_blk;
    if (nb == 0) {
        return 0;
    }
    const uint32_t kvh = sg.blocked ? h / sg.G : h % sg.Hkv;
    const uint32_t begin = first_blk * sg.Hkv + kvh * nb;
    return run_of_block(sg.runs, begin + nb - 1) - run_of_block(sg.runs, begin) + 1;
}

__global__ void combine_kernel(const float *__restrict__ partials, uint32_t Hq, uint32_t d, uint32_t d_real,
                               uint32_t max_slots, SlotGeom sg, const float *__restrict__ rv, int unrotate,
                               int log2_domain, float *__restrict__ out, Geom3 og)
{
    __shared__ float w_s[1024];
    __shared__ float o_sh[256];
    __shared__ float o_part[1024];
    __shared__ float red[2];
    const uint32_t h = blockIdx.x, s = blockIdx.y, tid = threadIdx.x;
    const float *base = partials + ((uint64_t)s * Hq + h) * max_slots * (d + 2);
    uint32_t n_splits = max_slots;
    if (sg.blk_off) {
        n_splits = slots_of_row(sg, s, h);
    }
    // n_splits <= 1024 is enforced by the host
    if (tid < 64) {
        float mx = -INFINITY;
        for (uint32_t k = tid; k < n_splits; k += 64) {
            mx = fmaxf(mx, base[(uint64_t)k * (d + 2)]);
        }
        mx = wave_max(mx);
        float sum = 0.0f;
        for (uint32_t k = tid; k < n_splits; k += 64) {
            const float m = base[(uint64_t)k * (d + 2)];
            const float w = (m == -INFINITY) ? 0.0f : (log2_domain ? exp2f(m - mx) : expf(m - mx));
            w_s[k] = w;
            sum = fmaf(w, base[(uint64_t)k * (d + 2) + 1], sum);
        }
        sum = wave_sum(sum);
        if (tid == 0) {
            red[0] = sum;
        }
    }
    __syncthreads();
    const float denom = red[0];
    {
        // thread groups of d2 (power of two >= d) threads take the partials in turn, then the groups are added up
        uint32_t d2 = 32;
        while (d2 < d) {
            d2 <<= 1;
        }
        const uint32_t grp = tid / d2, ngrp = blockDim.x / d2, j = tid % d2;
        float acc = 0.0f;
        if (j < d) {
            // eight partials at a time, so that their loads are in flight together
            for (uint32_t k0 = grp; k0 < n_splits; k0 += 8 * ngrp) {
                float y[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t k = k0 + u * ngrp;
                    y[u] = (k < n_splits && w_s[k] != 0.0f) ? base[(uint64_t)k * (d + 2) + 2 + j] : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t k = k0 + u * ngrp;
                    if (k < n_splits && w_s[k] != 0.0f) {
                        acc = fmaf(w_s[k], y[u], acc);
                    }
                }
            }
        }
        o_part[tid] = acc;
        __syncthreads();
        if (tid < d) {
            float tot = 0.0f;
            for (uint32_t gI = 0; gI < ngrp; ++gI) {
                tot += o_part[gI * d2 + tid];
            }
            o_sh[tid] = (denom > 0.0f) ? tot / denom : 0.0f;
        }
    }
    __syncthreads();
    if (tid >= d) {
        return;
    }
    float r;
    if (unrotate) {
        r = 0.0f;
        for (uint32_t j = 0; j < d; ++j) {
            r = fmaf(o_sh[j], rv[tid + d * j], r);
        }
    } else {
        r = o_sh[tid];
    }
    if (tid < d_real) {
        out[(uint64_t)og.off + (uint64_t)s * og.s[0] + head_offset(og, h) + (uint64_t)tid * og.s[2]] = r;
    }
}

// The same as combine_kernel for kRowsPerWg (sequence, head) rows per workgroup and at most 64 partials per row:
// thread j owns coordinate j of every row, so the rotation is read once per workgroup.
__global__ void __launch_bounds__(256) combine_rows_kernel(const float *__restrict__ partials, uint32_t Hq, uint32_t d,
                                                           uint32_t d_real, uint32_t max_slots, uint32_t n_rows,
                                                           SlotGeom sg,
                                                           const float *__restrict__ rv, int unrotate, int log2_domain,
                                                           float *__restrict__ out, Geom3 og)
{
    __shared__ float w_s[kRowsPerWg][64];
    __shared__ float denom_s[kRowsPerWg];
    __shared__ uint32_t n_s[kRowsPerWg];
    __shared__ float o_sh[kRowsPerWg][256];
    const uint32_t tid = threadIdx.x;
    const uint32_t row0 = blockIdx.x * kRowsPerWg;
    const uint32_t PS = d + 2;
    // The rotation does not depend on the partials: its first elements are requested before anything else, so that they
    // travel together with the partials.  d is a multiple of 64 here (the host checks).
    const bool rot_thread = unrotate && tid < d;
    float x0[64];
    auto request = [&](float (&x)[64], uint32_t j0) {
#pragma unroll
        for (int u = 0; u < 64; ++u) {
            x[u] = rv[tid + d * (j0 + u)];
        }
    };
    if (rot_thread) {
        request(x0, 0);
    }
    // Thread groups of d2 (power of two >= d) threads take the partials in turn.  The first four partials of every
    // group and row are requested here, before their weights are known (slots that turn out to be unused are read
    // and dropped), so that they travel together with the partials' headers.
    uint32_t d2 = 32;
    while (d2 < d) {
        d2 <<= 1;
    }
    const uint32_t grp = tid / d2, ngrp = 256 / d2, j = tid % d2;
    const bool col_ok = j < d;
    float x[kRowsPerWg][4];
#pragma unroll
    for (int r = 0; r < kRowsPerWg; ++r) {
        const float *base = partials + (uint64_t)(row0 + r) * max_slots * PS + 2 + j;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t k = grp + u * ngrp;
            x[r][u] = (col_ok && row0 + r < n_rows && k < max_slots) ? base[(uint64_t)k * PS] : 0.0f;
        }
    }
    {
        // one wavefront per row, one lane per partial: weights of the row's partials
        static_assert(kRowsPerWg == 4, "one 64-lane wavefront per row");
        const uint32_t r = tid >> 6, l = tid & 63;
        const uint32_t row = row0 + r;
        uint32_t n = 0;
        if (row < n_rows) {
            n = max_slots;
            if (sg.blk_off) {
                n = slots_of_row(sg, row / Hq, row % Hq);
            }
        }
        const float *base = partials + (uint64_t)row * max_slots * PS;
        float m0 = -INFINITY, l0 = 0.0f;
        if (l < n) {
            m0 = base[(uint64_t)l * PS];
            l0 = base[(uint64_t)l * PS + 1];
        }
        const float mx = wave_max(m0);
        const float w0 = (m0 == -INFINITY) ? 0.0f : (log2_domain ? exp2f(m0 - mx) : expf(m0 - mx));
        const float sum = wave_sum(w0 * l0);
        w_s[r][l] = w0;
        if (l == 0) {
            denom_s[r] = sum;
            n_s[r] = n;
        }
    }
    __syncthreads();
    {
        float acc[kRowsPerWg];
#pragma unroll
        for (int r = 0; r < kRowsPerWg; ++r) {
            const float *base = partials + (uint64_t)(row0 + r) * max_slots * PS + 2 + j;
            const uint32_t n = n_s[r];
            float a = 0.0f;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t k = grp + u * ngrp;
                // (an unused slot may hold anything, so it is skipped rather than weighted with zero)
                a = k < n ? fmaf(w_s[r][k], x[r][u], a) : a;
            }
            if (col_ok) {
                // further partials eight at a time, so that their loads are in flight together (ragged batches and
                // long contexts leave dozens of partials per row)
                for (uint32_t k0 = grp + 4 * ngrp; k0 < n; k0 += 8 * ngrp) {
                    float y[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const uint32_t k = k0 + u * ngrp;
                        y[u] = k < n ? base[(uint64_t)k * PS] : 0.0f;
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const uint32_t k = k0 + u * ngrp;
                        a = k < n ? fmaf(w_s[r][k], y[u], a) : a;
                    }
                }
            }
            acc[r] = a;
        }
        // add the groups up through LDS (o_sh doubles as the staging area: [row][group * d2 + j])
#pragma unroll
        for (int r = 0; r < kRowsPerWg; ++r) {
            o_sh[r][tid] = acc[r];
        }
        __syncthreads();
        float tot[kRowsPerWg];
#pragma unroll
        for (int r = 0; r < kRowsPerWg; ++r) {
            float t = 0.0f;
            if (tid < d) {
                for (uint32_t gI = 0; gI < ngrp; ++gI) {
                    t += o_sh[r][gI * d2 + tid];
                }
                const float den = denom_s[r];
                t = den > 0.0f ? t / den : 0.0f;
            }
            tot[r] = t;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRowsPerWg; ++r) {
            o_sh[r][tid] = tot[r];
        }
    }
    __syncthreads();
    if (tid >= d) {
        return;
    }
    float res[kRowsPerWg];
    if (unrotate) {
#pragma unroll
        for (int r = 0; r < kRowsPerWg; ++r) {
            res[r] = 0.0f;
        }
        for (uint32_t j0 = 0; j0 < d; j0 += 64) {
            if (j0) {
                request(x0, j0);
            }
#pragma unroll
            for (int u = 0; u < 64; ++u) {
#pragma unroll
                for (int r = 0; r < kRowsPerWg; ++r) {
                    res[r] = fmaf(o_sh[r][j0 + u], x0[u], res[r]);
                }
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < kRowsPerWg; ++r) {
            res[r] = o_sh[r][tid];
        }
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWg; ++r) {
        const uint32_t row = row0 + r;
        if (row < n_rows && tid < d_real) {
            const uint32_t s = row / Hq, h = row % Hq;
            out[(uint64_t)og.off + (uint64_t)s * og.s[0] + head_offset(og, h) + (uint64_t)tid * og.s[2]] = res[r];
        }
    }
}

// combine_kernel for many rows, a tile of them per workgroup like prep_q_tile_kernel (at most 64 partials per row).  16 x 64
// positions of 32 heads of 128 with seventeen partials each: 115 us by rows, 74 here (58 of them the partials' 290 MB), 23
// with the three partials that one round of workgroups leaves (pass_workgroups); 32 x 64 positions into a column-major
// tensor, one partial each: 240 and 43.
template <int NT>
__global__ void __launch_bounds__(256) combine_tile_kernel(const float *__restrict__ partials, uint32_t Hq, uint32_t d_real,
                                                           uint32_t max_slots, uint32_t n_rows, SlotGeom sg,
                                                           const float *__restrict__ rv, int unrotate, int log2_domain,
                                                           float *__restrict__ out, uint32_t o_off, uint32_t s_coord,
                                                           RowOrder order, int wide)
{
    typedef TileRotation<NT> Rot;
    constexpr uint32_t D = Rot::D, R = Rot::R, PITCH = Rot::PITCH, PS = D + 2;
    __shared__ __attribute__((aligned(16))) float xs[R * PITCH];
    __shared__ float w_s[R][64 + 1];
    __shared__ uint64_t at_s[R];
    __shared__ uint32_t row_s[R], n_s[R];
    __shared__ float inv_s[R];
    const uint32_t tid = threadIdx.x, e0 = blockIdx.x * R;
    float b[Rot::KC / 2];
    if (unrotate) {
        Rot::load(b, rv, Rot::first_column_tile(), 0);
    }
    if (tid < R) {
        uint32_t row = 0, n = 0;
        uint64_t at = ~0ull;
        if (e0 + tid < n_rows) {
            row_of(order, e0 + tid, row, at);
            at += o_off;
            n = sg.blk_off ? slots_of_row(sg, row / Hq, row % Hq) : max_slots;
        }
        at_s[tid] = at;
        row_s[tid] = row;
        n_s[tid] = n;
    }
    __syncthreads();
    {
        // weights: 256 / R lanes per row, each slot's maximum and sum requested before the first is looked at
        constexpr uint32_t L = 256 / R, U = 64 / L;
        const uint32_t r = tid / L, l = tid % L, n = n_s[r];
        const float *base = partials + (uint64_t)row_s[r] * max_slots * PS;
        float2 t[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (u * L < max_slots) {
                const uint32_t k = u * L + l;
                t[u] = *reinterpret_cast<const float2 *>(base + (uint64_t)(k < n ? k : 0U) * PS);
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (u * L + l < n) {
                mx = fmaxf(mx, t[u].x);
            }
        }
#pragma unroll
        for (uint32_t o = L / 2; o > 0; o >>= 1) {
            mx = fmaxf(mx, __shfl_xor(mx, (int)o));
        }
        float sum = 0.0f;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t k = u * L + l;
            if (k < n) {
                const float m = t[u].x;
                const float w = (m == -INFINITY) ? 0.0f : (log2_domain ? exp2f(m - mx) : expf(m - mx));
                w_s[r][k] = w;
                sum = fmaf(w, t[u].y, sum);
            }
        }
#pragma unroll
        for (uint32_t o = L / 2; o > 0; o >>= 1) {
            sum += __shfl_xor(sum, (int)o);
        }
        if (l == 0) {
            inv_s[r] = sum;
        }
    }
    __syncthreads();
    {
        // sixteen lanes per row, two coordinates each (the partials are 8-byte aligned), two rows at a time per thread
        const uint32_t l = tid & 15;
        for (uint32_t r0 = 0; r0 < R; r0 += 32) {
            float2 acc[2][NT];
            uint32_t n[2], most = 0;
            const float *base[2];
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                const uint32_t r = r0 + 16 * i + (tid >> 4);
                n[i] = n_s[r];
                most = max(most, n[i]);
                base[i] = partials + (uint64_t)row_s[r] * max_slots * PS + 2 + 2 * l;
#pragma unroll
                for (uint32_t c = 0; c < NT; ++c) {
                    acc[i][c] = float2{ 0.0f, 0.0f };
                }
            }
            constexpr uint32_t KU = NT <= 4 ? 4 : 2; // slots requested together
            for (uint32_t k0 = 0; k0 < most; k0 += KU) {
                float2 v[KU][2][NT];
#pragma unroll
                for (uint32_t u = 0; u < KU; ++u) {
                    if (u && k0 + u >= most) {
                        break;
                    }
#pragma unroll
                    for (uint32_t i = 0; i < 2; ++i) {
                        const float *slot = base[i] + (uint64_t)(k0 + u < n[i] ? k0 + u : 0U) * PS;
#pragma unroll
                        for (uint32_t c = 0; c < NT; ++c) {
                            v[u][i][c] = *reinterpret_cast<const float2 *>(slot + 32 * c);
                        }
                    }
                }
#pragma unroll
                for (uint32_t u = 0; u < KU; ++u) {
#pragma unroll
                    for (uint32_t i = 0; i < 2; ++i) {
                        // (an unused slot may hold anything, so it is skipped rather than weighted with zero)
                        const float w = k0 + u < n[i] ? w_s[r0 + 16 * i + (tid >> 4)][k0 + u] : 0.0f;
#pragma unroll
                        for (uint32_t c = 0; c < NT; ++c) {
                            acc[i][c].x = fmaf(w, w != 0.0f ? v[u][i][c].x : 0.0f, acc[i][c].x);
                            acc[i][c].y = fmaf(w, w != 0.0f ? v[u][i][c].y : 0.0f, acc[i][c].y);
                        }
                    }
                }
            }
#pragma unroll
            for (uint32_t i = 0; i < 2; ++i) {
                const uint32_t r = r0 + 16 * i + (tid >> 4);
                const float den = inv_s[r];
#pragma unroll
                for (uint32_t c = 0; c < NT; ++c) {
                    float2 t = acc[i][c];
                    t.x = den > 0.0f ? t.x / den : 0.0f;
                    t.y = den > 0.0f ? t.y / den : 0.0f;
                    *reinterpret_cast<float2 *>(xs + r * PITCH + 2 * l + 32 * c) = t;
                }
            }
        }
    }
    __syncthreads();
    if (unrotate) {
        Rot::run(xs, rv, b);
    }
    if (wide) {
        const uint32_t j = 4 * (tid & 7);
#pragma unroll
        for (uint32_t r0 = 0; r0 < R; r0 += 32) {
            const uint32_t r = r0 + (tid >> 3);
            const uint64_t a = at_s[r];
#pragma unroll
            for (uint32_t c = 0; c < NT; ++c) {
                if (a != ~0ull && j + 32 * c < d_real) {
                    *reinterpret_cast<float4 *>(out + a + j + 32 * c) =
                        *reinterpret_cast<const float4 *>(xs + r * PITCH + j + 32 * c);
                }
            }
        }
        return;
    }
    const uint32_t r = tid % R;
    const uint64_t a = at_s[r];
    if (a == ~0ull) {
        return;
    }
    for (uint32_t c = tid / R; c < D / 4; c += 256 / R) {
        const float4 v = *reinterpret_cast<const float4 *>(xs + r * PITCH + 4 * c);
        const float w[4] = { v.x, v.y, v.z, v.w };
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
            if (4 * c + e < d_real) {
                out[a + (uint64_t)(4 * c + e) * s_coord] = w[e];
            }
        }
    }
}

// From this many rows on the tiles of queries pay, at every head_dim and layout (4096 rows of 64, 96, 128, 192 or 256: 7.1,
// 14.7, 10.6, 14.8 and 21.1 us by rows, 5.6, 8.4, 9.3, 12.6 and 15.2 in tiles; a tile is one workgroup's chain of gather,
// rotate, store).  The merge's chain grows with the partials per row, half a microsecond each, while more rows shorten only
// the row kernel's share: where there is one (head_dims that are multiples of 64) a merge of s partials goes by tiles from
// 128 s rows more on (rows of 128: 4096 with 4, 9 or 25 partials 11.3, 12.1 and 16.6 us by rows, 12.6, 15.2 and 25.1 in
// tiles; 6144 with 4 or 13: 17.6 and 22.8 against 12.6 and 19.8; rows of 256: 4096 with 25 partials 32.9 and 35.6).
constexpr uint32_t kRowsForTiles = 4096;
constexpr uint32_t kRowsPerPartialForTiles = 128;

// The order in which the tiles walk a call's rows, and whether the rows' coordinates come in whole 16-byte pieces.  Rows
// that are contiguous are taken in the order of their numbers; else the dimension with the smallest step in the caller's
// tensor goes fastest, so that neighbouring lanes read neighbouring elements.
RowOrder row_order(const Geom3 &g, uint32_t n_seq, const void *base, uint32_t d_real, int &wide)
{
    struct Dim {
        uint32_t n, x, row;
    } dim[3] = { { g.heads, g.s[1], g.blocked ? g.tokens : 1u },
                 { g.tokens, g.ts, g.blocked ? 1u : g.heads },
                 { n_seq, g.s[0], g.heads * g.tokens } };
    wide = g.s[2] == 1 && d_real % 4 == 0 && ((g.off | g.s[0] | g.s[1] | (g.tokens > 1 ? g.ts : 0u)) & 3u) == 0 &&
        (reinterpret_cast<uintptr_t>(base) & 15) == 0;
    std::sort(dim, dim + 3, [&](const Dim &a, const Dim &b) { return wide ? a.row < b.row : (a.x != b.x ? a.x < b.x : a.row < b.row); });
    return RowOrder{ dim[0].n, dim[1].n, { dim[0].x, dim[1].x, dim[2].x }, { dim[0].row, dim[1].row, dim[2].row } };
}

template <typename F> void with_column_tiles(uint32_t d, F &&f) // f(std::integral_constant<int, d / 32>)
{
    switch (d / 32) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    default: f(std::integral_constant<int, 8>{}); break;
    }
}

// Workgroups per pass of a call whose passes share one launch.  They run in rounds of one workgroup per compute unit, and
// eight consecutive ones are spread over the eight XCDs, so a pass takes a multiple of eight and the passes together fill
// whole rounds: with 256 per pass, as for a single pass, sixteen passes were sixteen rounds of short runs, each with its
// queries, tables and partials to write and merge.  What a round costs beyond its blocks is about four and a half blocks
// per wavefront (16 sequences of 4096-8192 tokens, 64 positions, 32 heads on 8: 454 us in sixteen rounds, 383 in eight, 331
// in four, 302 in two, 296 in one; two passes over 4 x 8192-16384: 69 us in two rounds, 53 in one; twenty passes at
// head_dim 256: 189 us in 32 per pass or more, 102 in 24, 112 in 16, 95 in 8, which is one round).
uint32_t pass_workgroups(uint32_t passes, uint32_t blocks, uint32_t waves)
{
    uint32_t best = 8;
    double best_cost = 0.0;
    for (uint32_t per_pass = 8; per_pass <= 256; per_pass += 8) {
        const double rounds = std::ceil(passes * per_pass / 256.0);
        const double cost = rounds * (std::ceil((double)blocks / (per_pass * waves)) + 4.5);
        if (per_pass == 8 || cost < best_cost) {
            best = per_pass;
            best_cost = cost;
        }
    }
    return best;
}

// Where the workgroups share the unpacking of the cache: thirteen tiles of rows and more per group of sixteen, so that seven of a
// workgroup's eight wavefronts have rows (132 rows of 128 63 us by passes, 89 so), and as many blocks as it takes to earn what a
// workgroup's start (tables, LDS, one round of workgroups that waits for the slowest) and a region's start in it (queries, partials, the
// first block's way) cost more than by passes.  A block takes a workgroup the same time for 13 tiles as for 16, and the passes 13
// sixteenths: where the fields are cheap to unpack and a block's products long (96 and 128 coordinates) there is little to earn
// with few tiles, and the line rises with the cube of that.  Fields beyond four bits are dearer by passes, but for bytes, which take no
// table there, as uniform cells of up to four bits do: nothing to earn with either at 96, nor with bytes at 64.
// Measured on 800 drawn calls around the lines, 17 to 64 positions, 200 to 2000 rows per KV head (by passes -> shared, us; below a
// line by passes):
//   head_dim 128, fields up to 4 bits: 13 tiles, 19 sequences of 5500-10600 tokens 199 -> 180; 14 tiles, 4 of 13451 142 -> 148
//     (below); 16 tiles, 3 of 18000 164 -> 150, 16 of 4096 205 -> 180; 40 of 100-2500 239 -> 312 (below)
//   96: 13 tiles, 8 of 17800-37500 125 -> 137 and 15 tiles, 2 of 22900 116 -> 124 (both below), 13 tiles, 4 of 52600 198 -> 207 (the
//     furthest behind of those above); 16 tiles, 6 of 10300 148 -> 128
//   64: 13 tiles, 41 of 200-6600 212 -> 200; 15, 58 of 3257 167 -> 144; 32: of 6000 114 -> 117 (left to the passes)
//   5 to 7 bits at 64 and 96: 1.3 to 1.7 times as fast from the line on; bytes at 96 (by passes): 16 of 14657 124 -> 127, 2 of
//     39000-55000 182 -> 202, at 64 30 of 4700-9100 271 -> 283, 18 of 13800 188 -> 174; 4-bit cells at 96 (by passes): 4 of 36700-56000 180 -> 191
//   beyond 4 bits at 128: 8 of 3000, K and V 5 bits 143 -> 114, 8 bits 125 -> 100, V alone 5 bits 115 -> 106; 40 of 100 to 2500,
//     V alone 278 -> 293
constexpr uint32_t kTilesToShare = 13;
bool sharing_pays(uint32_t d, bool cells, uint32_t widest_field, uint32_t tiles, uint32_t groups, uint32_t wgs, uint64_t regions, uint64_t blocks)
{
    // (17 to 19 groups leave compute units idle, more than 32 take a second round: 4352 rows, 7 sequences of 7497 tokens, of 96
    // 315 -> 344 us, of 64 254 -> 270; with 11 groups, 176 workgroups, it is 232 -> 208 still, at 8 bits with 17 554 -> 429)
    if (widest_field <= 4 && (wgs * groups < 160 || wgs * groups > 256)) {
        return false;
    }
    if ((widest_field == 8 && d < 128) || (cells && widest_field <= 4 && d == 96)) {
        return false;
    }
    double workgroup = 20.0, region = 24.0; // in blocks
    if (widest_field > 4 && d == 128) {
        workgroup = 8.0, region = 15.0;
    } else if (widest_field <= 4 && d > 64) {
        const double room = 16.0 * groups / tiles;
        workgroup = (d == 96 ? 20.0 : 18.0) * room * room * room, region = 20.0;
    }
    return (double)blocks >= wgs * workgroup + (double)regions * region;
}

// `lens_dev` (optional): attend over these per-sequence lengths instead of the cached ones.
// `n_tokens` > 1: a chunk of query positions per sequence, the last `n_tokens` of the attended tokens being the
// chunk's own (position t sees all but the last n_tokens - 1 - t); q_tstride / o_tstride step between positions.
int decode_impl(const char *fn, weed_hip_kv_cache *c, int32_t n_q_heads, int32_t gqa_mapping, const float *q_dev,
                uint32_t q_off, const uint32_t q_stride[3], float *out_dev, uint32_t o_off, const uint32_t o_stride[3],
                uint32_t flags, const int32_t *lens_dev, uint32_t n_tokens = 1, uint32_t q_tstride = 0,
                uint32_t o_tstride = 0, uint8_t *fixed_ws = nullptr, size_t fixed_ws_bytes = 0)
{
    WEED_HIP_REQUIRE(c, "%s: null cache", fn);
    WEED_HIP_REQUIRE(q_dev && out_dev && q_stride && o_stride, "%s: null pointer", fn);
    // d: head_dim as stored (a multiple of 32, see weed_hip_kv_cache::dp); d_real: the caller's
    const uint32_t Hkv = (uint32_t)c->cfg.n_kv_heads, d = c->dp, S = (uint32_t)c->cfg.n_seq;
    const uint32_t d_real = (uint32_t)c->cfg.head_dim;
    WEED_HIP_REQUIRE(n_q_heads > 0 && (uint32_t)n_q_heads % Hkv == 0,
                     "%s: n_q_heads %d must be a positive multiple of n_kv_heads %u", fn, n_q_heads, Hkv);
    WEED_HIP_REQUIRE(gqa_mapping == WEED_HIP_GQA_WEED || gqa_mapping == WEED_HIP_GQA_BLOCKED,
                     "%s: unknown GQA mapping %d", fn, gqa_mapping);
    const bool rot_q = flags & WEED_HIP_ATTN_ROTATE_Q, unrot = flags & WEED_HIP_ATTN_UNROTATE_OUT;
    WEED_HIP_REQUIRE(!(rot_q || unrot) || c->has_rotations, "%s: rotation requested but no rotations are set", fn);
    // the kernels see (position, head) pairs as heads
    const uint32_t real_heads = (uint32_t)n_q_heads;
    const uint32_t Hq = real_heads * n_tokens;

    uint32_t max_len = 0;
    for (int32_t l : c->lens) {
        max_len = std::max(max_len, (uint32_t)l);
    }
    const uint32_t G = Hq / Hkv;
    // groups (or chunks: positions x heads) beyond a tile's rows take several passes of the matrix-core kernel
    const uint32_t tile_rows = mfma_decode_tile_rows(d);
    const uint32_t passes = (G + tile_rows - 1) / tile_rows;
    const uint32_t pass_heads = (G + passes - 1) / passes;
    const bool use_mfma = mfma_decode_supported(d, c->k.w, c->v.w, pass_heads);
    WEED_HIP_REQUIRE(n_tokens == 1 || use_mfma,
                     "%s: head_dim %u with fields of %u and %u bits is not served by the matrix-core kernel, which a "
                     "chunk of positions needs", fn, d, c->k.w, c->v.w);
    // ONE copy of the process-wide tuning for the whole plan: weed_hip_kv_decode_tuning may change it from another host
    // thread at any time, and a plan must not pair a block count chosen under one setting with a search mode of another.
    const DecodeTuning tune = decode_tuning();
    // Rows of a KV head that would take many passes share the unpacking of the cache instead (kv_decode_chunk.hip): groups of up to
    // 256 rows, one run of blocks per workgroup and one round of workgroups.  (See kTilesToShare.)
    const uint32_t row_tiles = (G + 15) / 16, most_tiles = mfma_decode_shared_rows / 16;
    const uint32_t row_groups = (row_tiles + most_tiles - 1) / most_tiles, group_rows = (row_tiles + row_groups - 1) / row_groups * 16;
    // (one round on every XCD: the groups of a run lie on one, which has 32 compute units.  256 / groups in all instead put 33 to
    // 36 workgroups on some of them with 3, 5, 6 or 7 groups, and those took two rounds: 648 rows of 96, 8 sequences of 5682
    // tokens 246 us, 145 so, 156 by passes; 640 rows of 128, 2 of 70414 780, 440 and 499.)
    const uint32_t group_wgs = 8 * std::max(1u, 32u / row_groups);
    bool shared = use_mfma && d >= 64 && d <= 128 && row_tiles >= kTilesToShare * row_groups && tune.wavefronts == 0;
    if (shared) {
        uint64_t blocks = 0;
        for (int32_t l : c->lens) {
            blocks += ((uint64_t)l + 63) / 64 * Hkv;
        }
        shared = sharing_pays(d, c->cfg.mode == WEED_HIP_KV_UNIFORM, std::max(c->k.w, c->v.w), row_tiles, row_groups, group_wgs,
                              (uint64_t)S * Hkv, blocks);
    }
    // workspace: rotated q (fp32), its fp16 hi / lo halves, per-head scale and sum, split partials
    const size_t n_q = (size_t)S * Hq * d;
    const size_t q_bytes = sizeof(float) * n_q;
    const size_t h_bytes = (sizeof(uint16_t) * n_q + 15) / 16 * 16;
    const size_t s_bytes = (sizeof(float) * (size_t)S * Hq + 15) / 16 * 16;
    const size_t off_bytes = (sizeof(uint32_t) * ((size_t)S + 1) + 15) / 16 * 16;
    // (the arrival counters of the kernel's own merge come first, at the same place whatever the shape, because they
    // have to be zero when a launch starts: they are cleared when the workspace is allocated and every launch leaves
    // them at zero; the static scratch starts as zeros)
    const size_t arrive_bytes = sizeof(uint32_t) * kMfmaMergeCounters;
    const auto workspace = [&](uint32_t slots) {
        return arrive_bytes + q_bytes + 2 * h_bytes + 2 * s_bytes + off_bytes + sizeof(float) * (size_t)S * Hq * slots * (d + 2);
    };
    uint32_t n_splits, split_tokens = 0;
    uint32_t total_blocks = 0;
    RunGeom runs = { 1, 0, 8, 0 };
    // Blocks per sequence as the partition counts them when that is more than the sequences have (see below), else 0.
    uint32_t virtual_blocks = 0;
    auto partition_blocks = [&](int32_t l) { return virtual_blocks ? virtual_blocks : ((uint32_t)l + 63u) >> 6; };
    if (use_mfma) {
        // every wavefront takes an equal run of 64-token blocks from the list of all regions' blocks; as many
        // wavefronts as the device holds at once
        runs.waves = mfma_decode_workgroup_waves(pass_heads, d, c->k.w, c->v.w);
        // Equal sequences of nb blocks: prefer a run length with which every workgroup holds whole regions (the
        // kernel then does the whole call by itself, see below): nb / (classes * q) blocks with q = 1, 2 or 4, that
        // is 4 / q regions per workgroup, provided the workgroups fill the compute units in at most two rounds.
        // A block count that no such run length divides is rounded up to the next one that one does (see below):
        // the partition then counts blocks at the end of every region that hold no tokens, which the kernel skips
        // as it skips those beyond a prefix length, and the wavefront they fall to has that much less to do -- far
        // cheaper than runs that straddle regions.
        uint32_t preferred_unit = 0;
        // Sequences with different block counts are counted alike, as the longest of them, within the same bounds.
        uint32_t most = 0, fewest = ~0u;
        uint64_t real_blocks = 0;
        for (int32_t l : c->lens) {
            most = std::max(most, ((uint32_t)l + 63u) >> 6);
            fewest = std::min(fewest, ((uint32_t)l + 63u) >> 6);
            real_blocks += ((uint32_t)l + 63u) >> 6;
        }
        // (The blocks without tokens may come to three quarters of those with, over the whole batch: a wavefront
        // whose run holds few tokens or none is done early and leaves the memory system to the others, so the call
        // takes about as long as its tokens' bytes take -- down to the time that the longest sequence's own
        // wavefronts need, which is what bounds the ratio.  Measured on 64 sequences with lengths drawn from
        // [4096, 8192]: 104.6 us with runs that straddle regions, 84.4 us counted alike; from [512, 8192], where the
        // partition would count 1.78 blocks per block with tokens: 76.3 against 73.9 us, a tie.)
        // Calls of less than a few dozen microseconds are all fixed cost, of which runs that straddle regions have
        // more: there the ratio may be four (16 sequences from [512, 8192]: 42 us against 33 us).  What bounds such
        // calls is the blocks as counted, which is what a wavefront of the longest sequence works through: 32
        // sequences with up to 8192 tokens each gain 8 to 17 us counted alike, 48 such sequences lose 5 to 44 us.
        const uint64_t counted_alike = (uint64_t)most * S * Hkv;
        const uint64_t most_counted = counted_alike > 32768 ? real_blocks * 7 / 4
            : counted_alike > 16384                         ? real_blocks * 5 / 2
                                                            : real_blocks * 4;
        // (counts beyond what a region's memory holds are fine: the kernel reads nothing behind a region's last block)
        // (and no further than 4096 blocks past the longest: the counts that qualify below recur every few hundred
        // blocks at most, so a search that has found none by then finds none, and the host's time stays bounded)
        const uint32_t reach = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(most_counted / S, fewest + 1),
                                                            std::min<uint64_t>((uint64_t)most + 4096, 1u << 24));
        // (instances that cannot merge their partials themselves gain from runs that stay inside regions as well)
        // (not for groups that take several passes: they do not merge in their workgroups, and every pass would walk
        // the blocks that the rounding adds -- 64 sequences of 2100 tokens, 64 heads on 2 kv heads of 224: 198 us with
        // the rounding, 160 without)
        const bool may_round =
            fewest != 0 && tune.wavefronts == 0 && !tune.separate_merge && !tune.always_search && passes == 1;
        {
            const uint32_t nb = most;
            // Fewer blocks than wavefronts and regions of no more blocks than a workgroup has wavefronts: the call is
            // all fixed cost, of which the rows that a workgroup rotates and merges one pass after the other are the
            // largest part, so as few regions per workgroup as one round of workgroups allows, however few of the
            // compute units they fill (3 to 96 sequences of 100 tokens with groups of eight: 27 us with four regions
            // per workgroup, 14 us with one).
            const bool tiny = real_blocks * Hkv <= (uint64_t)runs.waves * 256u && nb <= runs.waves;
            if (may_round && tiny) {
                const uint32_t classes = run_classes(runs), regions = S * Hkv;
                for (uint32_t q = 4; q >= 1 && !preferred_unit; q /= 2) {
                    if ((regions * q + 3) / 4 > 256) {
                        continue;
                    }
                    for (uint32_t cand = nb; cand <= reach; ++cand) {
                        if (cand % (classes * q) == 0) {
                            preferred_unit = cand / (classes * q);
                            virtual_blocks = cand == fewest ? 0 : cand;
                            break;
                        }
                    }
                }
            }
            if (may_round && !preferred_unit) {
                const uint32_t classes = run_classes(runs), regions = S * Hkv;
                for (uint32_t cand = nb; cand <= reach && !preferred_unit; ++cand) {
                    // (one or two rounds of workgroups; above head_dim 128, where a workgroup's queries and merges
                    // take longer and a compute unit holds one workgroup, one round only)
                    uint32_t best_rounds = d > 128 ? 2 : 3;
                    for (uint32_t q = 1; q <= 4; q *= 2) {
                        if (cand % (classes * q) != 0) {
                            continue;
                        }
                        const uint32_t wgs = (regions * q + 3) / 4, rounds = (wgs + 255) / 256;
                        if (rounds < best_rounds && wgs * 100 >= rounds * 256 * 95) {
                            best_rounds = rounds;
                            preferred_unit = cand / (classes * q);
                            virtual_blocks = cand == fewest ? 0 : cand;
                        }
                    }
                }
            }
        }
        uint64_t blocks = 0;
        for (int32_t l : c->lens) {
            blocks += partition_blocks(l);
        }
        blocks *= Hkv;
        WEED_HIP_REQUIRE(blocks < (1ull << 32), "%s: too many cached tokens for one launch", fn);
        total_blocks = (uint32_t)blocks;
        // one workgroup per compute unit, all passes of a call together
        const uint32_t target_units = tune.wavefronts > 0 ? (uint32_t)tune.wavefronts
            : passes > 1                                  ? runs.waves * pass_workgroups(passes, total_blocks, runs.waves)
                                                          : runs.waves * 256u;
        runs.unit_blocks = preferred_unit ? preferred_unit : std::max(1u, (total_blocks + target_units - 1) / target_units);
        // Small batches of long sequences, where a region is several workgroups' shares: the same rounding, to a
        // whole number of those shares.
        bool whole_shares = false;
        if (!preferred_unit && may_round) {
            for (uint32_t cand = most; cand <= reach; ++cand) {
                // (the run length that this count would get)
                const uint64_t all = (uint64_t)cand * S * Hkv;
                const uint32_t unit = (uint32_t)std::max<uint64_t>(1, (all + target_units - 1) / target_units);
                const uint32_t wg_blocks = runs.waves * unit;
                if (cand % wg_blocks == 0 && cand / wg_blocks <= 64 && all < (1ull << 32)) {
                    if (cand != fewest) {
                        virtual_blocks = cand;
                        total_blocks = (uint32_t)all;
                    }
                    runs.unit_blocks = unit;
                    whole_shares = true;
                    break;
                }
            }
        }
        // One workgroup per region instead, though that leaves compute units without one: its wavefronts' runs are longer,
        // but the region is merged in the workgroup's LDS instead of through memory by the last of its workgroups (2.6 us,
        // and up to 2.9 more with 256 workgroups arriving) or by runs that straddle regions (10.5 us).  A block more per
        // wavefront costs 1.7 us at 64 coordinates, 1.85 at 96, 2.6 at 128 and 3.3 above, a fifth less with uniform fields of
        // up to 4 bits, twice as much where both sides look their codes up in tables of 32 (all from both plans' times of
        // 500 drawn calls).
        // 32 heads on 8 of 128: 16 sequences of 600-1000 tokens 19.0 -> 16.0 us, 24 of 2000, whose runs straddled, 30.8 ->
        // 20.2; 12 heads of 64: one sequence of 1000 or 1500 tokens 11.9 and 12.2 -> 10.8.  Left as they are: 32 heads of
        // 128 at 2 + 3 bits over 2174 tokens (16.6 us, 18.3 so), 48 heads of 64 with signs, 5 + 5 bits, over 3040-3424 (15.7
        // and 21.4), 40 heads of 128 at 5 + 5 bits over 535 (17.4 and 19.1).
        if (!preferred_unit && may_round && (uint64_t)S * Hkv <= 256 &&
            mfma_decode_merges_whole_regions(pass_heads <= 4 ? 4u : (pass_heads <= 8 ? 8u : 16u), d, runs.waves)) {
            const uint32_t cand = (most + runs.waves - 1) / runs.waves * runs.waves, unit = cand / runs.waves;
            const uint32_t wg_blocks = runs.waves * runs.unit_blocks;
            const double wgs = std::min(256.0, std::ceil((double)total_blocks / wg_blocks));
            const double merge_us = whole_shares ? 2.6 + 2.9 * wgs / 256.0 : 10.5;
            const bool tables = c->cfg.mode == WEED_HIP_KV_LLOYDMAX;
            const int wide_sides = (c->k.w > 4 ? 1 : 0) + (c->v.w > 4 ? 1 : 0);
            const double block_us = (d <= 64 ? 1.7 : (d <= 96 ? 1.85 : (d <= 128 ? 2.6 : 3.3))) *
                (tables ? 1.0 + 0.5 * wide_sides : 0.8 + 0.1 * wide_sides);
            if (cand <= reach && (uint64_t)cand * S * Hkv < (1ull << 32) &&
                ((double)unit - runs.unit_blocks) * block_us < merge_us) {
                virtual_blocks = cand == fewest ? 0 : cand;
                runs.unit_blocks = unit;
                total_blocks = cand * S * Hkv;
            }
        }
        const uint32_t skew_pct = tune.skew_percent >= 0 ? (uint32_t)std::min(90, tune.skew_percent)
                                                         : (runs.waves == 12 ? kRunSkewPercent3 : kRunSkewPercent);
        const uint32_t nblk = virtual_blocks ? virtual_blocks : (max_len + 63) / 64;
        for (;;) {
            runs.skew = std::min(runs.unit_blocks - 1, (runs.unit_blocks * skew_pct + 50) / 100);
            const uint32_t shortest = runs.unit_blocks - runs.skew;
            n_splits = (nblk + shortest - 1) / shortest + 1; // partial slots per (sequence, head)
            if (n_splits <= kMaxSlots) {
                break;
            }
            // one very long region and few of them: longer runs (fewer wavefronts) keep the merge within its limit
            runs.unit_blocks += std::max(1u, runs.unit_blocks / 8);
        }
        if (shared) {
            // (a region of no more partials than the kernel behind merges by tiles)
            const RunGeom own = { std::max((total_blocks + group_wgs - 1) / group_wgs, (nblk + 62) / 63), 0, 8, 0 };
            const uint32_t own_splits = (nblk + own.unit_blocks - 1) / own.unit_blocks + 1;
            // These runs are up to twice as many as the passes' (256 workgroups' against 16 of eight wavefronts), and so are the
            // partials.  A call whose workspace holds the passes' only goes by passes: under capture, where it cannot grow, and a
            // call of one position up to the static scratch, which its twin that allocates nothing has, with the same bits.
            const auto only_passes_fit = [&](size_t room) { return workspace(own_splits) > room && workspace(n_splits) <= room; };
            shared = !(n_tokens == 1 && only_passes_fit(kStaticScratchBytes)) &&
                     !(!fixed_ws && only_passes_fit(c->dec_ws_bytes) && capturing());
            // So do few regions of very many blocks, whose runs the limit on partials makes so long that workgroups are missing (one
            // sequence of 230117 tokens, two KV heads of 96: 124 of them, 194 us against 129).
            shared = shared && 8ull * own.unit_blocks <= 9ull * ((total_blocks + group_wgs - 1) / group_wgs);
            if (shared) {
                runs = own;
                n_splits = own_splits;
            }
        }
    } else {
        // split the context so that the launch has a few workgroups per compute unit
        const uint32_t target_wgs = 2048;
        const uint32_t want = std::min((uint32_t)kMaxSlots, std::max(1u, target_wgs / (S * Hkv)));
        n_splits = std::max(1u, std::min((max_len + kChunk - 1) / kChunk, want));
        split_tokens = (max_len + n_splits - 1) / n_splits;
        split_tokens = std::max((uint32_t)kChunk, (split_tokens + kChunk - 1) / kChunk * kChunk);
        n_splits = std::max(1u, (max_len + split_tokens - 1) / split_tokens);
    }
    WEED_HIP_REQUIRE(n_splits <= kMaxSlots, "%s: internal split count %u too large", fn, n_splits);

    const size_t need = workspace(n_splits);
    if (fixed_ws) {
        // the caller's workspace (the static scratch): nothing is allocated, larger shapes are refused
        WEED_HIP_REQUIRE(need <= fixed_ws_bytes,
                         "%s: this shape needs %zu bytes of workspace, the static scratch holds %zu (use "
                         "weed_hip_kv_decode_attn)", fn, need, fixed_ws_bytes);
    } else if (need > c->dec_ws_bytes) {
        WEED_HIP_CHECK(hipStreamSynchronize(stream()));
        (void)hipFree(c->dec_ws);
        c->dec_ws = nullptr;
        c->dec_ws_bytes = 0;
        if (hipMalloc((void **)&c->dec_ws, need) != hipSuccess) {
            return fail(WEED_HIP_ENOMEM, "%s: workspace allocation of %zu bytes failed", fn, need);
        }
        c->dec_ws_bytes = need;
        WEED_HIP_CHECK(hipMemsetAsync(c->dec_ws, 0, arrive_bytes, stream()));
    }
    uint8_t *ws0 = fixed_ws ? fixed_ws : reinterpret_cast<uint8_t *>(c->dec_ws);
    uint32_t *arrive = reinterpret_cast<uint32_t *>(ws0);
    uint8_t *wsp = ws0 + arrive_bytes;
    const bool timed = !fixed_ws; // the timing scopes create events, which the allocation-free entry point must not
    float *q_rot = reinterpret_cast<float *>(wsp);
    uint16_t *q_hi = reinterpret_cast<uint16_t *>(wsp + q_bytes);
    uint16_t *q_lo = reinterpret_cast<uint16_t *>(wsp + q_bytes + h_bytes);
    float *q_scale = reinterpret_cast<float *>(wsp + q_bytes + 2 * h_bytes);
    float *q_sum = reinterpret_cast<float *>(wsp + q_bytes + 2 * h_bytes + s_bytes);
    uint32_t *blk_off = reinterpret_cast<uint32_t *>(wsp + q_bytes + 2 * h_bytes + 2 * s_bytes);
    float *partials = reinterpret_cast<float *>(wsp + q_bytes + 2 * h_bytes + 2 * s_bytes + off_bytes);

    const int blocked = gqa_mapping == WEED_HIP_GQA_BLOCKED ? 1 : 0;
    Geom3 qg = { q_off, { q_stride[0], q_stride[1], q_stride[2] }, n_tokens, real_heads, q_tstride, blocked };
    Geom3 og = { o_off, { o_stride[0], o_stride[1], o_stride[2] }, n_tokens, real_heads, o_tstride, blocked };
    const uint32_t n_rows = S * Hq;
    // the multi-row kernels pay off with many (sequence, head) rows; their rotation loops step by 64
    const bool many_rows = n_rows >= 512 && d % 64 == 0;
    const bool tiles = n_rows >= kRowsForTiles;

    // Blocks per sequence when all sequences span the same number, else 0.
    uint32_t uniform_blocks = 0;
    // The workgroups of the matrix-core kernel merge their regions themselves (wg_regions regions each, else 0) when
    // every workgroup's share of the block list is a whole number of regions and no run straddles a region boundary:
    // equal sequences of nb blocks each, nb a multiple of one cycle of the age classes' runs, and a workgroup's blocks
    // a multiple of nb.  They then also rotate their regions' queries themselves, and the call is ONE kernel.
    uint32_t wg_regions = 0, region_wgs = 0;
    bool general_merge = false;
    bool fused_query = false;
    if (use_mfma && total_blocks) {
        uniform_blocks = partition_blocks(c->lens[0]);
        for (int32_t l : c->lens) {
            if (partition_blocks(l) != uniform_blocks || tune.always_search) {
                uniform_blocks = 0;
                break;
            }
        }
        const uint32_t gp = pass_heads <= 4 ? 4u : (pass_heads <= 8 ? 8u : 16u);
        const uint32_t nb = uniform_blocks, cycle = run_classes(runs) * runs.unit_blocks;
        const uint32_t wg_blocks = runs.waves * runs.unit_blocks;
        // (Groups that take several passes of the kernel -- more than sixteen heads per kv head, more than eight at
        // head_dims above 128 -- go the three-kernel way: every pass would rotate its queries and merge at the end of
        // its workgroups, where one kernel ahead and one behind serve all passes.  Measured, 64 heads on 2 kv heads
        // of 128: 16 sequences of 8192 tokens 63.4 against 59.5 us, one sequence 57.7 against 37.2, two of 30000
        // tokens 105 against 58; 96 heads on 2: 91 against 61.)
        const bool may_merge = mfma_decode_merges_whole_regions(gp, d, runs.waves) && passes == 1;
        // (above head_dim 128 in one round of workgroups only: 64 sequences of 300 or 2100 tokens on 32 kv heads of
        // 256 in two rounds took 69 and 224 us against 61 and 216 with three kernels, where one round is 13 us ahead)
        if (may_merge && nb != 0 && nb % cycle == 0 && wg_blocks % nb == 0 && !tune.separate_merge &&
            (d <= 128 || (total_blocks + wg_blocks - 1) / wg_blocks <= 256)) {
            wg_regions = wg_blocks / nb;
        } else if (may_merge && nb != 0 && nb % wg_blocks == 0 && nb / wg_blocks >= 2 &&
                   nb / wg_blocks <= std::min(n_splits, 64u) && (size_t)S * Hkv <= kMfmaMergeCounters &&
                   !tune.separate_merge) {
            // small batches of long sequences: every region is a whole number of workgroups' shares
            region_wgs = nb / wg_blocks;
        }
        // Most regions that the blocks of one workgroup lie in (exact: the host knows the cached lengths).
        uint32_t wg_most_regions = wg_regions;
        bool every_sequence_has_tokens = true;
        if (wg_regions == 0) {
            // (a buffer of the cache object, so that a decode call allocates nothing on the host either)
            std::vector<uint64_t> &region_end = c->plan_region_end; // blocks up to and including region r
            region_end.clear();
            region_end.reserve((size_t)S * Hkv);
            uint64_t run = 0;
            for (int32_t l : c->lens) {
                const uint32_t b = partition_blocks(l);
                every_sequence_has_tokens = every_sequence_has_tokens && b != 0;
                for (uint32_t h = 0; h < Hkv; ++h) {
                    run += b;
                    region_end.push_back(run);
                }
            }
            size_t r = 0;
            for (uint64_t first = 0; first < total_blocks; first += wg_blocks) {
                const uint64_t last = std::min<uint64_t>(first + wg_blocks, total_blocks) - 1;
                while (region_end[r] <= first) {
                    ++r;
                }
                size_t r1 = r;
                while (region_end[r1] <= last) {
                    ++r1;
                }
                wg_most_regions = std::max(wg_most_regions, (uint32_t)(r1 - r + 1));
            }
        }
        // Anything else that the instance can merge: one slot per (run, region) in memory, an arrival counter per
        // region (ragged batches: up to 63 sequences, whose block offsets a wavefront keeps in one register).
        // A workgroup merges the regions that it completes one after the other, at its end, about 2 us each, where
        // the separate kernel merges all regions at once for 10 to 12 us: measured on batches that are half long and
        // half short sequences, the workgroups win up to 6 regions per workgroup, tie at 7 and lose from 8 on (5 to
        // 30 us at 8 to 17).  Nor do they where they could not rotate their queries as well (a kernel ahead and the
        // merges at the end: 3 to 200 sequences of 100 tokens with groups of eight, 27 us against 22 to 25).
        if (wg_regions == 0 && region_wgs == 0 && passes == 1 && mfma_decode_merges_in_general(gp, d, runs.waves) && every_sequence_has_tokens &&
            (nb != 0 || (S <= 63 && !tune.always_search)) && n_splits <= (d % 64 == 0 ? 64u : 24u) &&
            wg_most_regions <= kMostRegionsMergedByWorkgroup &&
            wg_most_regions * pass_heads <= std::min(kMostRowsMergedByWorkgroup, mfma_query_rows(d)) &&
            (size_t)S * Hkv <= kMfmaMergeCounters && !tune.separate_merge) {
            general_merge = true;
        }
        // A workgroup rotates the queries of the regions its blocks lie in itself when they are few enough for its
        // LDS (equal sequences, or the ragged batches above); nothing then runs ahead of the matrix-core kernel.
        fused_query = passes == 1 && (wg_regions != 0 || region_wgs != 0 || mfma_decode_merges_in_general(gp, d, runs.waves)) &&
                      (nb != 0 || general_merge) &&
                      wg_most_regions * pass_heads <= mfma_query_rows(d) && !tune.separate_query;
    }
    // Workgroups that merge whole regions or whole shares of a region: neighbouring runs take their blocks in turns
    // (see RunGeom), as many cycles' runs together as divide both a workgroup's share and a region, so that no group
    // crosses a region boundary.  (Measured on 1 to 256 sequences of 1024 to 16384 tokens: 1 to 6 % faster with runs
    // of 4 to 32 blocks, nothing with shorter ones, 1 to 1.5 % slower with runs of 64.  Not at head_dim 256, where
    // a block is twice the bytes: 64 sequences of 8192 tokens took 267 us with turns and 232 us without.)
    if ((wg_regions != 0 || region_wgs != 0) && runs.unit_blocks >= kFewestBlocksOfRunsInTurns &&
        runs.unit_blocks <= kMostBlocksOfRunsInTurns && !tune.contiguous_runs && d <= 128) {
        const uint32_t cycle = run_classes(runs) * runs.unit_blocks;
        uint32_t cycles = runs.waves / run_classes(runs);
        while (uniform_blocks % (cycles * cycle) != 0) {
            cycles /= 2; // (4, 2, 1: a region is whole cycles)
        }
        runs.group_cycles = cycles;
    }
    const bool fused_merge = wg_regions != 0 || region_wgs != 0 || general_merge;
    if (tune.print_plan) {
        std::fprintf(stderr,
                     "%s: S %u Hkv %u G %u d %u bits %u/%u  matrix cores %d  passes %u  blocks %u  run %u (skew %u, in turns %u) "
                     "x %u wavefronts  whole regions per workgroup %u  workgroups per region %u  general merge %d  "
                     "queries in the kernel %d  slots %u  groups that share the unpacking %u of %u rows\n",
                     fn, S, Hkv, G, d, c->k.w, c->v.w, (int)use_mfma, passes, total_blocks, runs.unit_blocks, runs.skew,
                     runs.group_cycles, runs.waves, wg_regions, region_wgs, (int)general_merge, (int)fused_query, n_splits,
                     shared ? row_groups : 0U, shared ? group_rows : 0U);
    }
    // (the kernels that take one (sequence, head) row per workgroup have the sequence on a 16-bit grid dimension)
    // (prep_q_kernel puts one more row on that dimension when it also builds the block offsets)
    WEED_HIP_REQUIRE(S + ((use_mfma && !fused_query && !many_rows) ? 1u : 0u) <= 65535u || (use_mfma && many_rows && n_splits <= 64),
                     "%s: %u sequences in one call are served only for head_dims that are multiples of 64 with "
                     "matrix-core instances; split the batch", fn, S);
    if (fused_query) {
        // (nothing runs ahead of the matrix-core kernel)
    } else if (tiles) {
        int wide = 0;
        const RowOrder order = row_order(qg, S, q_dev, d_real, wide);
        with_column_tiles(d, [&](auto nt) {
            constexpr int NT = decltype(nt)::value;
            constexpr uint32_t R = tile_rows_of(NT);
            prep_q_tile_kernel<NT><<<(n_rows + R - 1) / R + (use_mfma ? 1 : 0), 256, 0, stream()>>>(
                q_dev, q_off, qg.s[2], order, wide, d_real, n_rows, c->k.rot_t, rot_q ? 1 : 0, use_mfma ? nullptr : q_rot, q_hi,
                q_lo, q_scale, q_sum, c->lens_dev, S, use_mfma ? blk_off : nullptr);
        });
    } else if (many_rows) {
        prep_q_rows_kernel<<<(n_rows + kRowsPerWg - 1) / kRowsPerWg + (use_mfma ? 1 : 0), 256, 0, stream()>>>(
            q_dev, qg, Hq, d, d_real, n_rows, c->k.rot_t, rot_q ? 1 : 0, q_rot, q_hi, q_lo, q_scale, q_sum, c->lens_dev, S,
            use_mfma ? blk_off : nullptr);
    } else {
        prep_q_kernel<<<dim3(Hq, S + (use_mfma ? 1 : 0)), 256, 0, stream()>>>(q_dev, qg, Hq, d, d_real, c->k.rot_t, rot_q ? 1 : 0, q_rot, q_hi, q_lo,
                                                         q_scale, q_sum, c->lens_dev, S, use_mfma ? blk_off : nullptr);
    }
    WEED_HIP_LAUNCH_CHECK();

    if (use_mfma) {
        MfmaParams mp;
        const SideParams ks = side_params(c, 0), vs = side_params(c, 1);
        mp.k = MfmaSide{ ks.fields, ks.alpha, ks.region_bytes, ks.alpha_max, ks.alpha_const, ks.beta, ks.w };
        mp.v = MfmaSide{ vs.fields, vs.alpha, vs.region_bytes, vs.alpha_max, vs.alpha_const, vs.beta, vs.w };
        mp.table_image = c->table_image;
        mp.lens = lens_dev ? lens_dev : c->lens_dev;
        mp.padded = c->padded_tokens;
        mp.Hq = Hq;
        mp.Hkv = Hkv;
        mp.G = G;
        mp.blocked = gqa_mapping == WEED_HIP_GQA_BLOCKED;
        mp.q_tokens = n_tokens;
        mp.real_group = real_heads / Hkv;
        mp.q_hi = q_hi;
        mp.q_lo = q_lo;
        mp.q_scale = q_scale;
        mp.q_sum = q_sum;
        mp.partials = partials;
        mp.blk_off = blk_off;
        mp.n_seq = S;
        mp.total_blocks = total_blocks;
        mp.uniform_blocks = uniform_blocks;
        mp.merge = MfmaMerge{ wg_regions, region_wgs, general_merge ? 1u : 0u, arrive, d_real, out_dev, og, c->v.rot,
                              unrot ? 1 : 0 };
        mp.cached_lens = c->lens_dev;
        mp.query = MfmaQuery{ fused_query ? q_dev : nullptr, qg, c->k.rot_t, rot_q ? 1 : 0 };
        mp.runs = runs;
        mp.max_slots = n_splits;
        mp.group_total = G;
        mp.tile_rows = pass_heads;
        ProfileScope prof("kv_decode_attn", timed);
        mp.grid_passes = 0;
        if (shared) {
            mp.head_first = 0;
            mp.tile_rows = mp.G = group_rows;
            mp.grid_passes = row_groups;
            if (total_blocks) {
                WEED_HIP_TRY(launch_mfma_decode_shared(mp, d, stream()));
            }
        } else if (passes > 1 && total_blocks && !fused_merge && !fused_query) {
            // every pass in ONE launch: the passes' workgroups that read the same blocks run next to each other on one
            // XCD, so the cache is fetched from memory once instead of once per pass
            mp.grid_passes = passes;
            mp.head_first = 0;
            mp.G = pass_heads;
            WEED_HIP_TRY(launch_mfma_decode(mp, d, stream()));
        } else {
            for (uint32_t first = 0; total_blocks && first < G; first += pass_heads) {
                mp.head_first = first;
                mp.G = std::min(pass_heads, G - first);
                WEED_HIP_TRY(launch_mfma_decode(mp, d, stream()));
            }
        }
    } else {
        DecodeParams p;
        p.k = side_params(c, 0);
        p.v = side_params(c, 1);
        p.lens = lens_dev ? lens_dev : c->lens_dev;
        p.padded = c->padded_tokens;
        p.d = d;
        p.d_real = d_real;
        p.Hq = Hq;
        p.Hkv = Hkv;
        p.G = G;
        p.blocked = gqa_mapping == WEED_HIP_GQA_BLOCKED;
        p.q_rot = q_rot;
        p.partials = partials;
        p.n_splits = n_splits;
        p.split_tokens = split_tokens;
        ProfileScope prof("kv_decode_attn", timed);
        decode_generic_kernel<<<dim3(n_splits, Hkv, S), kThreads, 0, stream()>>>(p);
        WEED_HIP_LAUNCH_CHECK();
    }
    if (!fused_merge) {
        ProfileScope prof("kv_decode_combine", timed);
        const SlotGeom sg = { use_mfma ? blk_off : nullptr, Hkv, G, runs,
                              gqa_mapping == WEED_HIP_GQA_BLOCKED ? 1 : 0, uniform_blocks };
        if (tiles && n_splits <= 64 && (d % 64 != 0 || n_rows >= kRowsForTiles + kRowsPerPartialForTiles * n_splits)) {
            int wide = 0;
            const RowOrder order = row_order(og, S, out_dev, d_real, wide);
            with_column_tiles(d, [&](auto nt) {
                constexpr int NT = decltype(nt)::value;
                constexpr uint32_t R = tile_rows_of(NT);
                combine_tile_kernel<NT><<<(n_rows + R - 1) / R, 256, 0, stream()>>>(
                    partials, Hq, d_real, n_splits, n_rows, sg, c->v.rot, unrot ? 1 : 0, use_mfma ? 1 : 0, out_dev, o_off,
                    og.s[2], order, wide);
            });
        } else if (many_rows && n_splits <= 64) {
            combine_rows_kernel<<<(n_rows + kRowsPerWg - 1) / kRowsPerWg, 256, 0, stream()>>>(
                partials, Hq, d, d_real, n_splits, n_rows, sg, c->v.rot, unrot ? 1 : 0, use_mfma ? 1 : 0, out_dev, og);
        } else {
            combine_kernel<<<dim3(Hq, S), n_splits > 16 ? 1024 : 256, 0, stream()>>>(
                partials, Hq, d, d_real, n_splits, sg, c->v.rot, unrot ? 1 : 0, use_mfma ? 1 : 0, out_dev, og);
        }
        WEED_HIP_LAUNCH_CHECK();
    }
    return WEED_HIP_OK;
}

} // namespace

extern "C" int weed_hip_kv_decode_attn(weed_hip_kv_cache *c, int32_t n_q_heads, int32_t gqa_mapping, const float *q_dev,
                                       uint32_t q_off, const uint32_t q_stride[3], float *out_dev, uint32_t o_off,
                                       const uint32_t o_stride[3], uint32_t flags)
{
    return decode_impl("weed_hip_kv_decode_attn", c, n_q_heads, gqa_mapping, q_dev, q_off, q_stride, out_dev, o_off,
                       o_stride, flags, nullptr);
}

extern "C" int weed_hip_kv_decode_tuning(int32_t wavefronts, int32_t skew_percent, int32_t always_search)
{
    DecodeTuning &t = decode_tuning();
    t.wavefronts = std::max(0, wavefronts);
    t.skew_percent = skew_percent;
    t.always_search = (always_search & 1) != 0;
    t.separate_merge = (always_search & 2) != 0;
    t.separate_query = (always_search & 4) != 0;
    t.contiguous_runs = (always_search & 8) != 0;
    return WEED_HIP_OK;
}

extern "C" int weed_hip_kv_decode_attn_noalloc(weed_hip_kv_cache *c, int32_t n_q_heads, int32_t gqa_mapping,
                                               const float *q_dev, uint32_t q_off, const uint32_t q_stride[3],
                                               float *out_dev, uint32_t o_off, const uint32_t o_stride[3],
                                               uint32_t flags)
{
    const char *fn = "weed_hip_kv_decode_attn_noalloc";
    const int dev = current_device();
    WEED_HIP_REQUIRE(dev >= 0 && dev < kMaxDevices && g_scratch_dev[dev],
                     "%s: weed_hip_init has not run on the current device", fn);
    return decode_impl(fn, c, n_q_heads, gqa_mapping, q_dev, q_off, q_stride, out_dev, o_off, o_stride, flags, nullptr,
                       1, 0, 0, static_cast<uint8_t *>(g_scratch_dev[dev]), kStaticScratchBytes);
}

extern "C" int weed_hip_kv_decode_attn_prefix(weed_hip_kv_cache *c, const int32_t *lens_dev, int32_t n_q_heads,
                                              int32_t gqa_mapping, const float *q_dev, uint32_t q_off,
                                              const uint32_t q_stride[3], float *out_dev, uint32_t o_off,
                                              const uint32_t o_stride[3], uint32_t flags)
{
    const char *fn = "weed_hip_kv_decode_attn_prefix";
    WEED_HIP_REQUIRE(lens_dev, "%s: null length array", fn);
    return decode_impl(fn, c, n_q_heads, gqa_mapping, q_dev, q_off, q_stride, out_dev, o_off, o_stride, flags, lens_dev);
}

extern "C" int weed_hip_kv_decode_attn_chunk(weed_hip_kv_cache *c, const int32_t *lens_dev, int32_t n_tokens,
                                             int32_t n_q_heads, int32_t gqa_mapping, const float *q_dev, uint32_t q_off,
                                             const uint32_t q_stride[4], float *out_dev, uint32_t o_off,
                                             const uint32_t o_stride[4], uint32_t flags)
{
    const char *fn = "weed_hip_kv_decode_attn_chunk";
    WEED_HIP_REQUIRE(q_stride && o_stride, "%s: null pointer", fn);
    WEED_HIP_REQUIRE(n_tokens >= 1 && n_tokens <= 64, "%s: %d positions outside [1, 64]", fn, n_tokens);
    if (c && !lens_dev) {
        for (int32_t l : c->lens) {
            WEED_HIP_REQUIRE(l >= n_tokens, "%s: a sequence holds %d tokens, fewer than the chunk's %d", fn, l, n_tokens);
        }
    }
    const uint32_t qs3[3] = { q_stride[0], q_stride[2], q_stride[3] }, os3[3] = { o_stride[0], o_stride[2], o_stride[3] };
    return decode_impl(fn, c, n_q_heads, gqa_mapping, q_dev, q_off, qs3, out_dev, o_off, os3, flags, lens_dev,
                       (uint32_t)n_tokens, q_stride[1], o_stride[1]);
}
