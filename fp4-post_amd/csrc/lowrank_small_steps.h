// The two steps of the decode-sized rank-r projection (lowrank_small.hip) as device functions, so that a launch that has
// other small work to do for the same layer call can carry them in some of its blocks: the first step (partial sums of
// xv = x . v^T per K chunk) beside the activation's quantizer (nvfp4_quant.hip), the finishing step (adds the partial
// sums in chunk order, rounds to bf16 and applies s) beside the build of the activation's GEMM operands (metis_gemm.hip).
#pragma once
#include "metis_device.h"

namespace metis {

typedef __bf16 lr_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float lr_float4_t __attribute__((ext_vector_type(4)));
typedef float lr_float16_t __attribute__((ext_vector_type(16)));

constexpr int kLrMaxChunks = 128;
constexpr int kLrGroup = kLrMaxChunks / 4;     // chunks per thread of the finishing step

// K in chunks of *kc_out elements (a multiple of 64), at most kLrMaxChunks of them
inline int lowrank_small_chunks(int64_t K, int* kc_out)
{
    int64_t kc = 64;
    if ((K + kc - 1) / kc > kLrMaxChunks) kc = ((K + kLrMaxChunks - 1) / kLrMaxChunks + 63) / 64 * 64;
    *kc_out = (int)kc;
    return (int)((K + kc - 1) / kc);
}

// One wave of the first step: K chunk `chunk` (kc elements), RT tiles of 32 rows from 32 RT mtile on, columns 32 ct .. of R.  Every load
// touches 64 lines, which a compute unit's L1 looks up one a cycle: a step (4 + 4 RT loads) is bound by that and by one round trip to
// memory.  AHEAD: the next step is requested before this one is multiplied (32 more registers, which cost a launch with other work more
// than they give).
template <int RT, bool AHEAD>
__device__ __forceinline__ void lowrank_small_partial_wave(int chunk, int mtile, int ct, const uint16_t* __restrict__ x, int64_t ldx,
                                                           const uint16_t* __restrict__ v, int M, int R, int K, int kc, float* __restrict__ ws)
{
    const int lane = threadIdx.x & 63, hi = lane >> 5;
    const int m0 = mtile * (32 * RT);
    const int k0 = chunk * kc, k1 = min(k0 + kc, K);
    const uint16_t* vp = v + (int64_t)min(ct * 32 + (lane & 31), R - 1) * K + hi * 32;
    const uint16_t* xp[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) xp[i] = x + (int64_t)min(m0 + i * 32 + (lane & 31), M - 1) * ldx + hi * 32;
    lr_float16_t acc[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
    auto fetch = [&](uint4 (&rv)[4], uint4 (&rx)[RT][4], int k) {
#pragma unroll
        for (int q = 0; q < 4; ++q) rv[q] = reinterpret_cast<const uint4*>(vp + k)[q];
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) rx[i][q] = reinterpret_cast<const uint4*>(xp[i] + k)[q];
    };
    uint4 nv[4], nx[RT][4];
    if constexpr (AHEAD) fetch(nv, nx, k0);
    for (int k = k0; k < k1; k += 64) {                        // kc % 64 == 0 and K % 64 == 0
        uint4 rv[4], rx[RT][4];
        if constexpr (AHEAD) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                rv[q] = nv[q];
#pragma unroll
                for (int i = 0; i < RT; ++i) rx[i][q] = nx[i][q];
            }
            if (k + 64 < k1) fetch(nv, nx, k + 64);
        } else {
            fetch(rv, rx, k);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const lr_bf16x8_t fv = __builtin_bit_cast(lr_bf16x8_t, rv[q]);
#pragma unroll
            for (int i = 0; i < RT; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fv, __builtin_bit_cast(lr_bf16x8_t, rx[i][q]), acc[i], 0, 0, 0);
        }
    }
    // acc[i][e] of lane l: row m = m0 + 32 i + l % 32, column r = 32 ct + 8 (e / 4) + 4 (l / 32) + e % 4
    float* wp = ws + (size_t)chunk * M * R;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int m = m0 + i * 32 + (lane & 31);
        if (m >= M) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int r = ct * 32 + 8 * g + 4 * hi;
            if (r < R)                                          // R % 4 == 0
                *reinterpret_cast<float4*>(wp + (size_t)m * R + r) =
                    make_float4(acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]);
        }
    }
}

// The first step in a launch of 256-thread workgroups with other work: single tiles of 32 x 32, a workgroup with one wave for each, or
// (wide) four waves of 64 rows x 32 columns that share the rows' lines.  Microseconds with the quantizer, wide | single: 64 x 3584, R = 64
// 3.3 | 2.8, R = 128 4.3 | 3.0, 64 x 18944, R = 64 4.9 | 4.0, 5 x 18944, R = 128 4.5 | 3.2, 128 x 3584, R = 128 4.6 | 3.7, 128 x 8960, R = 128 6.1 | 5.2,
// 255 x 8960, R = 64 6.2 | 5.7, 192 x 18944, R = 32 5.7 | 5.6; where the compute units have more than ten steps of tiles each, re-reading V costs
// more: 192 x 8960, R = 128 6.6 | 8.3, 255 x 18944, R = 64 9.0 | 11.9.  (64 rows and fewer: 64 x 18944, R = 128 7.2 | 5.6.)  From five steps on it
// does so too where the wide workgroups fill one round of the compute units: 192 x 5120, R = 128 (240 of 256) 6.1 | 6.6, R = 96 5.3 | 5.4, 128 x 14336,
// R = 64 (224) 5.4 | 5.7, 255 x 3584, R = 96 (224) 5.1 | 5.4; but 192 x 3584, R = 128 (168) 5.5 | 5.2, 224 x 5120, R = 128 (320) 7.5 | 7.1, R = 32
// (one wave in four) 128 x 18944 (198) 5.4 | 5.1, 96 x 14336, R = 96 (224, half of their second rows empty) 6.0 | 5.7.
inline int lowrank_small_partial_blocks(int64_t M, int64_t R, int chunks, bool wide)
{
    return chunks * (int)(wide ? (M + 63) / 64 * ((R + 127) / 128) : (M + 31) / 32 * (R / 32));
}
inline bool lowrank_small_wide(int64_t M, int64_t R, int64_t K, int cus)
{
    const int64_t steps = (M + 31) / 32 * (R / 32) * (K / 64);
    int kc;
    const int blocks = lowrank_small_partial_blocks(M, R, lowrank_small_chunks(K, &kc), true);
    return M > 64 && (steps > 10 * (int64_t)cus || (M > 96 && R > 32 && steps >= 5 * (int64_t)cus && blocks > cus * 3 / 4 && blocks <= cus));
}
__device__ __forceinline__ void lowrank_small_partial_block(int block, int chunks, bool wide, const uint16_t* __restrict__ x, int64_t ldx,
                                                            const uint16_t* __restrict__ v, int M, int R, int K, int kc, float* __restrict__ ws)
{
    const int chunk = block % chunks, rest = block / chunks, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (wide) {
        const int mtiles = (M + 63) / 64, ct = rest / mtiles * 4 + wave;
        if (ct * 32 < R) lowrank_small_partial_wave<2, false>(chunk, rest % mtiles, ct, x, ldx, v, M, R, K, kc, ws);
    } else if (wave == 0) {
        lowrank_small_partial_wave<1, false>(chunk, rest / (R / 32), rest % (R / 32), x, ldx, v, M, R, K, kc, ws);
    }
}

// rounds four consecutive sums of the projection (element id of [M, R]) and applies s
__device__ __forceinline__ void lowrank_small_store(const float (&a)[4], int id, int r, const uint16_t* __restrict__ s, uint16_t* __restrict__ xv,
                                                    uint16_t* __restrict__ t)
{
    uint32_t h[4], u[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = bf16_bits(a[e]);
    *reinterpret_cast<uint2*>(xv + id) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    if (t) {
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = bf16_bits(__uint_as_float(h[e] << 16) * bf16_lo(s[r + e]));
        *reinterpret_cast<uint2*>(t + id) = make_uint2(u[0] | (u[1] << 16), u[2] | (u[3] << 16));
    }
}

// what lanes 16 .. 31 and 48 .. 63 hold, in lanes 0 .. 15 and 32 .. 47
__device__ __forceinline__ uint4 lr_from_odd_rows(uint4 a)
{
    return make_uint4(__builtin_amdgcn_permlane16_swap(a.x, a.x, false, false)[1], __builtin_amdgcn_permlane16_swap(a.y, a.y, false, false)[1],
                      __builtin_amdgcn_permlane16_swap(a.z, a.z, false, false)[1], __builtin_amdgcn_permlane16_swap(a.w, a.w, false, false)[1]);
}

// Both steps of 16 rows x 16 columns in one block of 1024 threads, for a launch with other work that waits for nothing of the projection; K <= 3072.
// Waves 4 g .. 4 g + 3 share the chunks of group g of the finishing step, a quarter each, requested together; the first of them adds the chunk sums of
// all four in chunk order.  A chunk is the four products of the first step on 32 x 32 tiles with 16 rows of either operand in lanes 0 .. 15 and
// 32 .. 47, so the bits are those of the two steps; the other lanes load half of those rows' elements and hand them over (v_permlane16_swap): their own
// rows of the product are nobody's.  Every thread of the block has to call it (two barriers inside).  Blocks: lowrank_small_project_blocks(M, R).
constexpr int kLrProjectThreads = 1024, kLrProjectK = 3072;
__device__ __forceinline__ void lowrank_small_project_block(int block, const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ v, int M,
                                                            int R, int K, const uint16_t* __restrict__ s, uint16_t* __restrict__ xv,
                                                            uint16_t* __restrict__ t)
{
    constexpr int MINE = kLrProjectK / 64 / 16;                // chunks of a wave
    __shared__ lr_float4_t sums[4][3][MINE][2][32], group[3][2][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l16 = lane & 15, hi = lane >> 5;
    const bool keeps = (lane & 16) == 0;
    const int slot = hi * 16 + l16;
    const int g = wave >> 2, w = wave & 3;
    const int r0 = block % (R / 16) * 16, m = block / (R / 16) * 16 + l16;
    const uint16_t* vp = v + (int64_t)(r0 + l16) * K + hi * 32 + (lane & 16);      // 32 bytes of a lane: pieces q = 0, 1 of the half chunk, or 2, 3
    const uint16_t* xp = x + (int64_t)min(m, M - 1) * ldx + hi * 32 + (lane & 16);
    const int chunks = K / 64, per = (chunks + 3) / 4, own = (per + 3) / 4;
    const int c0 = g * per + w * own, c1 = min(min(c0 + own, (g + 1) * per), chunks);
    uint4 rv[MINE][2], rx[MINE][2];
#pragma unroll
    for (int i = 0; i < MINE; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const bool live = c0 + i < c1;
            rv[i][q] = live ? *reinterpret_cast<const uint4*>(vp + (c0 + i) * 64 + 8 * q) : make_uint4(0u, 0u, 0u, 0u);
            rx[i][q] = live ? *reinterpret_cast<const uint4*>(xp + (c0 + i) * 64 + 8 * q) : make_uint4(0u, 0u, 0u, 0u);
        }
    // sums e of a lane: row m, columns r0 + 8 (e / 4) + 4 hi + e % 4, e < 8
    lr_float4_t total[2] = {(lr_float4_t)(0.0f), (lr_float4_t)(0.0f)};
    lr_float16_t acc[MINE];
#pragma unroll
    for (int i = 0; i < MINE; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < MINE; ++i) {
            const uint4 a = q < 2 ? rv[i][q] : lr_from_odd_rows(rv[i][q & 1]), b = q < 2 ? rx[i][q] : lr_from_odd_rows(rx[i][q & 1]);
            acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(lr_bf16x8_t, a), __builtin_bit_cast(lr_bf16x8_t, b), acc[i], 0, 0, 0);
        }
#pragma unroll
    for (int i = 0; i < MINE; ++i)                             // (a chunk past the end adds zeros)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const lr_float4_t a = {acc[i][4 * k], acc[i][4 * k + 1], acc[i][4 * k + 2], acc[i][4 * k + 3]};
            if (w == 0) total[k] += a;
            else if (keeps) sums[g][w - 1][i][k][slot] = a;
        }
    __syncthreads();
    if (w == 0) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < MINE; ++i)
#pragma unroll
                for (int k = 0; k < 2; ++k) total[k] += sums[g][p][i][k][slot];
        if (g > 0 && keeps) {
#pragma unroll
            for (int k = 0; k < 2; ++k) group[g - 1][k][slot] = total[k];
        }
    }
    __syncthreads();
    if (wave > 0 || !keeps || m >= M) return;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
        for (int i = 0; i < 3; ++i) total[k] += group[i][k][slot];
        const float a[4] = {total[k][0], total[k][1], total[k][2], total[k][3]};
        const int r = r0 + 8 * k + 4 * hi;
        lowrank_small_store(a, m * R + r, r, s, xv, t);
    }
}
inline int lowrank_small_project_blocks(int64_t M, int64_t R) { return (int)((M + 15) / 16 * (R / 16)); }

// One block of 256 threads: four threads per output quad (each a quarter of the chunks, folded in order), 64 quads.
// Every thread of the block has to call it (one barrier inside).
__device__ __forceinline__ void lowrank_small_finish_block(int block, const float* __restrict__ ws, int chunks, int MR, int R,
                                                           const uint16_t* __restrict__ s, uint16_t* __restrict__ xv,
                                                           uint16_t* __restrict__ t)
{
    __shared__ float4 fold[3][64];
    const int q = threadIdx.x & 63, g = threadIdx.x >> 6;      // output quad within the block, chunk group
    const int id = (block * 64 + q) * 4;                       // four consecutive elements of [M, R]
    const bool live = id < MR;
    const int per = (chunks + 3) / 4, c0 = g * per;            // this thread's chunks: [c0, c0 + per), per <= kLrGroup
    float4 p[kLrGroup];
#pragma unroll
    for (int c = 0; c < kLrGroup; ++c)
        p[c] = (live && c < per && c0 + c < chunks) ? *reinterpret_cast<const float4*>(ws + (size_t)(c0 + c) * MR + id)
                                                    : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 a = p[0];
#pragma unroll
    for (int c = 1; c < kLrGroup; ++c) { a.x += p[c].x; a.y += p[c].y; a.z += p[c].z; a.w += p[c].w; }
    if (g > 0) fold[g - 1][q] = a;
    __syncthreads();
    if (g > 0 || !live) return;
#pragma unroll
    for (int k = 0; k < 3; ++k) { const float4 b = fold[k][q]; a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; }
    const float sums[4] = {a.x, a.y, a.z, a.w};
    lowrank_small_store(sums, id, id % R, s, xv, t);
}

// One workgroup (256 threads) of the gradient of the rank-r scale vector: columns 8 block .. + 7 (scale_grad_kernel, lowrank_small.hip).
__device__ __forceinline__ void scale_grad_block(int block, const uint16_t* __restrict__ g, const uint16_t* __restrict__ xv, int L, int R,
                                                 void* __restrict__ out, int out_f32, float (&part)[8][256 + 4])
{
    constexpr int BATCH = 8;
    const int c0 = block * 8, tid = threadIdx.x;
    float acc[8] = {};
    for (int64_t l0 = tid; l0 < L; l0 += 256 * BATCH) {          // (64-bit: a step past the last row)
        uint4 a[BATCH], b[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const int64_t l = l0 + 256 * i;
            a[i] = b[i] = make_uint4(0u, 0u, 0u, 0u);             // (rows past the end add zeros)
            if (l < L) {
                a[i] = *reinterpret_cast<const uint4*>(g + l * R + c0);
                b[i] = *reinterpret_cast<const uint4*>(xv + l * R + c0);
            }
        }
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
            const uint32_t aw[4] = {a[i].x, a[i].y, a[i].z, a[i].w}, bw[4] = {b[i].x, b[i].y, b[i].z, b[i].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[2 * j] += rb(bf16_lo(aw[j]) * bf16_lo(bw[j]));
                acc[2 * j + 1] += rb(bf16_hi(aw[j]) * bf16_hi(bw[j]));
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) part[j][tid] = acc[j];
    __syncthreads();
    if (tid < 8) {
        float sum = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float4 v[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) v[t] = *reinterpret_cast<const float4*>(&part[tid][64 * q + 4 * t]);
#pragma unroll
            for (int t = 0; t < 16; ++t) sum = (((sum + v[t].x) + v[t].y) + v[t].z) + v[t].w;
        }
        if (out_f32) static_cast<float*>(out)[c0 + tid] = sum;
        else static_cast<uint16_t*>(out)[c0 + tid] = (uint16_t)bf16_bits(sum);
    }
}

}  // namespace metis
