// The mean mode's activation of few tokens in one launch: column mean over the rows, centred residual, its NVFP4 packing and the
// first step of the layer's rank-r projection (src/Metis/Metis/bitlinear.py:311-336).
#include "metis_device.h"
#include "metis_host.h"
#include "nvfp4_encode.h"
#include "lowrank_small_steps.h"

namespace metis {

// ---------------------------------------------------------------------------------------------
// The residual x - mean is quantized in blocks of 16 along a row, the mean runs down the columns: a workgroup that owns a strip of
// 32 columns and ALL rows has everything that its blocks need, so nothing has to leave the chip between the sum, the division
// and the encoder.  With a few hundred rows the strip is tens of KiB: the second read comes from L2.  What this replaces are
// dependent launches that leave the chip nearly empty (column sums, their finishing step, the centred quantizer, the
// projection's partial sums): latency-bound, 3 to 6 us each.
// The sums are taken in the order of the kernels that larger calls use, so the mean has their bits:
//   NORM = 0 (column_sum_kernel): slabs of rows_per_slab rows; in a slab four sums of every fourth row, (a + b) + (c + d); the
//            slabs in order.  A piece is one of a slab's four sums.
//   NORM = 1 (rmsnorm_colsum_rows_kernel and its finishing step): pieces of four consecutive rows in order; four sums of every
//            fourth piece, (a + b) + (c + d).
// A piece has at most four rows, all requested together; 64 pieces at a time, four lanes (16 bytes each) across the strip.
// Microseconds of device time, separate launches | this one (behind the norm: both with the norm's launch): 5 x 1536 8.8 | 3.4
// (10.6 | 6.2), 64 x 3584 11.3 | 3.5 (16.5 | 7.5), 411 x 1536 9.2 | 6.2 (12.5 | 10.4), 411 x 18944 14.0 | 9.6, 700 x 3584 13.2 | 8.5
// (20.4 | 15.7); 900 x 1536 10.1 | 10.3 (14.6 | 16.0), 1024 x 1024 9.1 | 10.2: narrow and longer, the strips no longer fill the chip.
// Workgroup ids are dealt out so that neighbouring strips, which share cache lines, run on the same XCD.
// ---------------------------------------------------------------------------------------------
constexpr uint32_t kStrip = 32, kMaxPieces = 256;

struct TokenMeanProjection {             // the first step of x . v^T rides in the workgroups behind the strips (R = 0: none)
    const uint16_t* v;
    float* ws;
    int R, kc, chunks, wide;
};

template <int NORM>
__global__ __launch_bounds__(256) void token_mean_quant_kernel(uint32_t strip_blocks, const uint16_t* __restrict__ x, uint32_t rows, uint32_t cols,
                                                               uint32_t pieces, uint32_t rows_per_slab, const uint16_t* __restrict__ cached,
                                                               float cached_count, uint16_t* __restrict__ mean, float* __restrict__ mean32,
                                                               uint2* __restrict__ codes, uint16_t* __restrict__ ws_amax,
                                                               uint32_t* __restrict__ ws_gmax, const TokenMeanProjection pr)
{
    if (blockIdx.x >= strip_blocks) {
        lowrank_small_partial_block((int)(blockIdx.x - strip_blocks), pr.chunks, pr.wide != 0, x, cols, pr.v, (int)rows, pr.R, (int)cols, pr.kc, pr.ws);
        return;
    }
    __shared__ __attribute__((aligned(16))) float sums[kMaxPieces][kStrip];
    __shared__ float chain[4][kStrip];
    __shared__ __attribute__((aligned(16))) float centre[kStrip];
    const uint32_t strips = (cols + kStrip - 1u) / kStrip, per_xcd = strip_blocks / 8u;
    const uint32_t strip = (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3);
    const uint32_t tid = threadIdx.x, c0 = strip * kStrip;
    float gmax = 0.0f;
    if (strip < strips) {                                       // the same for the whole workgroup
        // ---- sums of the pieces
        const uint32_t cl = (tid & 3u) * 8u;
        const bool live = c0 + cl < cols;                       // cols % 16 == 0: eight columns exist together
        for (uint32_t p = tid >> 2; p < pieces; p += 64u) {
            const uint32_t first = NORM ? 4u * p : (p >> 2) * rows_per_slab + (p & 3u), step = NORM ? 1u : 4u;
            const uint32_t end = min(NORM ? 4u * p + 4u : ((p >> 2) + 1u) * rows_per_slab, rows);
            uint4 w[4];
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) {
                const uint32_t r = first + i * step;
                w[i] = make_uint4(0u, 0u, 0u, 0u);
                if (live && r < end) w[i] = *reinterpret_cast<const uint4*>(x + (size_t)r * cols + c0 + cl);
            }
            float a[8] = {};
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) {                  // (a row that is not there adds +0)
                a[0] += bf16_lo(w[i].x); a[1] += bf16_hi(w[i].x); a[2] += bf16_lo(w[i].y); a[3] += bf16_hi(w[i].y);
                a[4] += bf16_lo(w[i].z); a[5] += bf16_hi(w[i].z); a[6] += bf16_lo(w[i].w); a[7] += bf16_hi(w[i].w);
            }
            *reinterpret_cast<float4*>(&sums[p][cl]) = make_float4(a[0], a[1], a[2], a[3]);
            *reinterpret_cast<float4*>(&sums[p][cl + 4u]) = make_float4(a[4], a[5], a[6], a[7]);
        }
        __syncthreads();
        // ---- the column's sum: its four chains side by side (NORM), or the slabs' sums first, then in order
        const uint32_t c = tid & (kStrip - 1u), g = tid / kStrip;
        if constexpr (NORM != 0) {
            if (g < 4u) {
                float s = 0.0f;
#pragma unroll 8
                for (uint32_t p = g; p < pieces; p += 4u) s += sums[p][c];
                chain[g][c] = s;
            }
        } else {
            for (uint32_t k = g; k < pieces / 4u; k += 256u / kStrip)    // (a slab's four sums are read and replaced by one thread)
                sums[4u * k][c] = (sums[4u * k][c] + sums[4u * k + 1u][c]) + (sums[4u * k + 2u][c] + sums[4u * k + 3u][c]);
        }
        __syncthreads();
        if (g == 0u) {
            float s = 0.0f;
            if constexpr (NORM != 0) {
                s = (chain[0][c] + chain[1][c]) + (chain[2][c] + chain[3][c]);
            } else {
#pragma unroll 8
                for (uint32_t k = 0; k < pieces / 4u; ++k) s += sums[4u * k][c];
            }
            float m = rb(s / (float)rows);
            if (c0 + c < cols) {
                if (cached) {                                    // the weighted running mean of single-token calls, each operation rounded (316-323)
                    const float a = rb(__uint_as_float((uint32_t)cached[c0 + c] << 16) * cached_count), b = rb(m * (float)rows);
                    m = rb(rb(a + b) / (cached_count + (float)rows));
                }
                mean[c0 + c] = (uint16_t)bf16_bits(m);
                mean32[c0 + c] = m;
            }
            centre[c] = m;
        }
        __syncthreads();
        // ---- the strip's blocks: two per row, thread = block, the next one requested ahead
        const uint32_t b = tid & 1u, cb = c0 + b * 16u;
        if (cb < cols) {
            float cen[kBlock];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 f = *reinterpret_cast<const float4*>(&centre[b * 16u + 4 * q]);
                cen[4 * q] = f.x; cen[4 * q + 1] = f.y; cen[4 * q + 2] = f.z; cen[4 * q + 3] = f.w;
            }
            uint4 n0 = make_uint4(0u, 0u, 0u, 0u), n1 = n0;
            auto request = [&](uint32_t r) {
                const uint4* src = reinterpret_cast<const uint4*>(x + (size_t)r * cols + cb);
                n0 = src[0]; n1 = src[1];
            };
            uint32_t r = tid >> 1;
            if (r < rows) request(r);
            for (; r < rows; r += 128u) {
                float v[kBlock];
                unpack16(n0, n1, v);
                if (r + 128u < rows) request(r + 128u);
#pragma unroll
                for (int j = 0; j < kBlock; ++j) v[j] = rb(v[j] - cen[j]);
                const float am = block_amax(v);
                gmax = fmaxf(gmax, am);
                const size_t at = ((size_t)r * cols + cb) / kBlock;
                ws_amax[at] = (uint16_t)(__float_as_uint(am) >> 16);
                codes[at] = encode_rne_pb16(v, block_scalar<1>(am));
            }
        }
    }
    publish_group_max(gmax, ws_gmax, kDeferredPartials, blockIdx.x, strip_blocks);
}

// the pieces of a call: column_mean's slabs (nvfp4_gemv.hip), or rmsnorm_colmean's workgroups (rmsnorm_quant.hip)
static bool token_mean_pieces(int64_t rows, int64_t cols, int after_norm, uint32_t* pieces, uint32_t* rows_per_slab)
{
    if (rows <= 0 || cols <= 0 || cols % kBlock) return false;
    if ((cols + kStrip - 1) / kStrip > (int64_t)kDeferredPartials - 8) return false;
    if (after_norm) {
        if (rows > 4 * (int64_t)kMaxPieces || rmsnorm_colmean_groups(rows) * 4 < rows) return false;
        *pieces = (uint32_t)((rows + 3) / 4);
        *rows_per_slab = 0;
        return true;
    }
    int64_t per = 0;
    const int64_t slabs = column_mean_slabs(rows, cols, &per);
    if (per > 16 || slabs * 4 > (int64_t)kMaxPieces) return false;
    *pieces = (uint32_t)(slabs * 4);
    *rows_per_slab = (uint32_t)per;
    return true;
}

int token_mean_quant_applies(int64_t rows, int64_t cols, int after_norm)
{
    uint32_t p, r;
    return token_mean_pieces(rows, cols, after_norm, &p, &r) ? 1 : 0;
}

int token_mean_quant(const void* x, int64_t rows, int64_t cols, int after_norm, const void* cached, int64_t cached_count, void* mean, float* mean32,
                     void* codes, void* deferred, size_t bytes, const void* v, int64_t R, void* lr_workspace, size_t lr_workspace_bytes, hipStream_t st)
{
    if (rows <= 0 || cols <= 0) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    uint32_t pieces, per;
    if (!token_mean_pieces(rows, cols, after_norm, &pieces, &per)) return METIS_E_TOO_LARGE;
    if (!x || !mean || !mean32 || !codes || ((uintptr_t)x % 16) || ((uintptr_t)mean % 4) || ((uintptr_t)mean32 % 4) || ((uintptr_t)codes % 8)) return METIS_E_ARG;
    if (cached && (cached_count < 0 || cached_count > (1 << 24) || ((uintptr_t)cached % 2))) return METIS_E_ARG;
    const uint32_t strip_blocks = (uint32_t)(((cols + kStrip - 1) / kStrip + 7) / 8 * 8);
    TokenMeanProjection pr = {};
    int more = 0;
    if (v) {
        if (rows >= 256 || cols % 64 || R <= 0 || R % 32 || R > 256) return METIS_E_SHAPE;
        if (((uintptr_t)v % 16)) return METIS_E_ARG;
        if (!lr_workspace || ((uintptr_t)lr_workspace % 16) || lr_workspace_bytes < lowrank_small_workspace_bytes(rows, R, cols)) return METIS_E_WORKSPACE;
        pr.v = (const uint16_t*)v;
        pr.ws = (float*)lr_workspace;
        pr.R = (int)R;
        pr.chunks = lowrank_small_chunks(cols, &pr.kc);
        // A workgroup of this launch holds the strips' LDS, whatever it does: four to a compute unit.  Single tiles, one wave in four, as long as they and
        // the strips are on the device together; beyond, four waves of 64 rows.  Microseconds, four waves | single: 64 x 8960, R = 160 (704 of them, and
        // 280 strips) 6.5 | 5.0, 48 x 8960, R = 128 6.0 | 4.9, 96 x 8960, R = 96 (910) 5.8 | 5.2, 128 x 1536, R = 256 5.1 | 4.8, 192 x 1536, R = 128 (624)
        // 5.2 | 5.4; 160 x 8960, R = 64 (980) 5.8 | 6.1, 160 x 18944, R = 32 (1087) 6.6 | 7.5, 1 x 14336, R = 256 (1344) 4.5 | 5.0, 64 x 18944, R = 256 8.8 | 11.7.
        const int single = lowrank_small_partial_blocks(rows, R, pr.chunks, false);
        pr.wide = 4 * ((int64_t)strip_blocks + single) > 15 * (int64_t)device_cus();
        more = pr.wide ? lowrank_small_partial_blocks(rows, R, pr.chunks, true) : single;
    }
    Workspace ws;
    if (const int rc = carve_deferred(deferred, bytes, rows, cols, &ws)) return rc;
#define METIS_TM(N) hipLaunchKernelGGL((token_mean_quant_kernel<N>), dim3(strip_blocks + (unsigned)more), dim3(256), 0, st, strip_blocks, \
        (const uint16_t*)x, (uint32_t)rows, (uint32_t)cols, pieces, per, (const uint16_t*)cached, (float)cached_count, (uint16_t*)mean, mean32, \
        (uint2*)codes, ws.amax, ws.gmax, pr)
    if (after_norm) METIS_TM(1); else METIS_TM(0);
#undef METIS_TM
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

}  // namespace metis
