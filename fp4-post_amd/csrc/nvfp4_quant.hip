// NVFP4 quantizer kernels for gfx950: block-16 absmax -> E2M1 codes + E4M3 block scales + a
// binary32 tensor scale, round-to-nearest or stochastic rounding, row- or column-blocked.
//
// Replaces the eager op chain of src/Metis/Metis/quant.py:6-36 (RNE) and 273-308 + 137-147
// (stochastic rounding).  HBM-bound integer/byte work: one coalesced read of the bf16 input,
// 0.5 B/element of codes and 1/16 B/element of scales written.
//
// Two-phase structure forced by the arithmetic: the codes depend only on the block's own raw
// scalar (quant.py:27), the scale bytes on the tensor-wide maximum (quant.py:21-23).  Phase 1
// writes codes, parks each block's maximum (2 B per block as bf16; 4 B as binary32 for data that is not
// bf16-valued) and publishes one partial maximum per workgroup; phase 2 turns the parked maxima into E4M3 bytes.
#include "metis_device.h"
#include "metis_host.h"
#include "nvfp4_encode.h"
#include "grid_max.h"
#include "lowrank_small_steps.h"
#include <atomic>
#include <stdio.h>
#include <stdlib.h>
#include <type_traits>

namespace metis {

// ---------------------------------------------------------------------------------------------
// Phase 1, row-blocked: codes + parked block maxima + per-workgroup maximum.  One block of 16 per
// thread per iteration: thread i <-> block i (32 contiguous bytes, two 16-byte loads).
// ---------------------------------------------------------------------------------------------
// WIDE (binary32 arithmetic only): the values to encode are binary32 values that need not be bf16 values,
// because the input tensor is binary32 (in_f32) and/or a binary32 centre is subtracted first.  The short cuts
// of the bf16 path (div6, the block-level guards of the hardware conversion) are proven for bf16 values only, so
// these instantiations take the block scalar by IEEE division, test every quotient before trusting the hardware
// conversion (encode_rne_wide), and park the block maxima as binary32.
//
// center (optional): one value per column, subtracted before anything else: x - center rounded to the
// arithmetic's dtype, the centred residual of the reference's mean mode (src/Metis/Metis/bitlinear.py:
// 330-333).  binary32 [cols] in binary32 arithmetic (always WIDE then), bf16 [cols] in bf16 arithmetic.
// Round-to-nearest rows of a contiguous bf16 tensor, the shape every activation and weight has: a kernel of its own
// so that its loop carries no row/column arithmetic at all.  Software-pipelined: the next DEPTH blocks' bytes are in
// flight while the current block is encoded.  Binary32 arithmetic takes the two-operation quotient for every block
// maximum the staged table clears (nvfp4_encode.h).
typedef uint32_t metis_u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t metis_u32x4_t __attribute__((ext_vector_type(4)));
template <int MODE> __device__ __forceinline__ uint2 encode_row_block(const float (&v)[kBlock], float am, const uint32_t* table)
{
    if constexpr (MODE == 0) {
        uint32_t w[2];
        encode_rne_p32_tbl<kBlock>(v, am, block_scalar<0>(am), table, w);
        return make_uint2(w[0], w[1]);
    } else {
        return encode_rne_pb16(v, block_scalar<1>(am));
    }
}

// (workgroup `block` of `grid`: a launch may give other blocks to other work)
template <int MODE, int DEPTH>
__device__ __forceinline__ void quant_codes_contig_block(uint32_t block, uint32_t grid, const uint4* __restrict__ x,
                                                         uint2* __restrict__ codes, uint16_t* __restrict__ ws_amax,
                                                         uint32_t* __restrict__ ws_gmax, uint32_t nblocks, uint32_t fill_to)
{
    __shared__ uint32_t table[MODE == 0 ? kQuotientTableWords : 4];
    float gmax = 0.0f;
    const uint32_t step = grid * 256u;
    uint32_t i = block * 256u + threadIdx.x;
    uint4 c0[DEPTH], c1[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        const uint32_t j = i + d * step;
        c0[d] = c1[d] = make_uint4(0u, 0u, 0u, 0u);
        if (j < nblocks) { c0[d] = x[2 * (size_t)j]; c1[d] = x[2 * (size_t)j + 1]; }
    }
    if constexpr (MODE == 0) stage_quotient_table(table);
    while (i < nblocks) {
        const uint4 a0 = c0[0], a1 = c1[0];
#pragma unroll
        for (int d = 0; d + 1 < DEPTH; ++d) { c0[d] = c0[d + 1]; c1[d] = c1[d + 1]; }
        const uint32_t nxt = i + DEPTH * step;
        if (nxt < nblocks) { c0[DEPTH - 1] = x[2 * (size_t)nxt]; c1[DEPTH - 1] = x[2 * (size_t)nxt + 1]; }
        float v[kBlock];
        unpack16(a0, a1, v);
        const float am = block_amax(v);
        gmax = fmaxf(gmax, am);
        ws_amax[i] = (uint16_t)(__float_as_uint(am) >> 16);        // read again soon by whoever forms the scale bytes
        const uint2 cw = encode_row_block<MODE>(v, am, table);
        __builtin_nontemporal_store((metis_u32x2_t){cw.x, cw.y}, reinterpret_cast<metis_u32x2_t*>(codes) + i);
        i += step;
    }
    publish_group_max(gmax, ws_gmax, fill_to, block, grid);
}

template <int MODE, int DEPTH = 1>
__global__ __launch_bounds__(256) void quant_codes_contig_kernel(const uint4* __restrict__ x, uint2* __restrict__ codes,
                                                                 uint16_t* __restrict__ ws_amax, uint32_t* __restrict__ ws_gmax,
                                                                 uint32_t nblocks, uint32_t fill_to)
{
    quant_codes_contig_block<MODE, DEPTH>(blockIdx.x, gridDim.x, x, codes, ws_amax, ws_gmax, nblocks, fill_to);
}

// A decode-sized activation's quantizer (scale bytes deferred) and the first step of its rank-r projection
// (lowrank_small_steps.h) in one launch: both only read x.  Blocks 0 .. qgrid-1 quantize, the others form the partial sums.
template <int MODE>
__global__ __launch_bounds__(256) void decode_quant_partial_kernel(uint32_t qgrid, const uint4* __restrict__ x, uint2* __restrict__ codes,
                                                                   uint16_t* __restrict__ ws_amax, uint32_t* __restrict__ ws_gmax,
                                                                   uint32_t nblocks, uint32_t fill_to, int64_t ldx,
                                                                   const uint16_t* __restrict__ v, int M, int R, int K, int kc, int chunks,
                                                                   int wide, float* __restrict__ lr_ws)
{
    if (blockIdx.x < qgrid) {
        quant_codes_contig_block<MODE, 1>(blockIdx.x, qgrid, x, codes, ws_amax, ws_gmax, nblocks, fill_to);
        return;
    }
    lowrank_small_partial_block((int)(blockIdx.x - qgrid), chunks, wide != 0, reinterpret_cast<const uint16_t*>(x), ldx, v, M, R, K, kc, lr_ws);
}

// The same loop with a centre subtracted first (mean mode, src/Metis/Metis/bitlinear.py:311-336: the tensor that is
// quantized is x - me with the column mean me): contiguous bf16 rows of at most 4096 columns, the centre staged once per
// workgroup in LDS (binary32 [cols] in binary32 arithmetic, bf16 values widened in bf16 arithmetic).  In binary32 arithmetic
// the residuals are binary32 values that need not be bf16 values: the per-quotient encoder and binary32 block maxima, as
// quant_codes_kernel<0, false, true>; in bf16 arithmetic the residual is rounded to bf16 and encoded as any bf16 block.
// A block's column position advances by a fixed amount modulo the row length: no division in the loop.
constexpr int kCentreMaxCols = 4096;
template <int MODE>
__global__ __launch_bounds__(256) void quant_codes_contig_centered_kernel(const uint4* __restrict__ x, const void* __restrict__ center,
                                                                          uint2* __restrict__ codes, void* __restrict__ ws_amax_v,
                                                                          uint32_t* __restrict__ ws_gmax, uint32_t nblocks,
                                                                          uint32_t nbpr, uint32_t fill_to)
{
    // quarter q of block b at cen[q][b]: the 16-byte reads of consecutive lanes (consecutive blocks) are consecutive in LDS
    // (block after block, a lane's four reads would be 64 bytes apart from its neighbour's: four lanes per bank)
    __shared__ float4 cen[4][kCentreMaxCols / kBlock];
    for (uint32_t c = threadIdx.x; c < nbpr * kBlock; c += 256u)
        reinterpret_cast<float*>(&cen[(c % kBlock) / 4u][c / kBlock])[c % 4u] =
            MODE == 0 ? static_cast<const float*>(center)[c] : bf16_lo(static_cast<const uint16_t*>(center)[c]);
    __syncthreads();
    float gmax = 0.0f;
    const uint32_t step = gridDim.x * 256u, step_mod = step % nbpr;
    uint32_t i = blockIdx.x * 256u + threadIdx.x;
    uint32_t cb = i % nbpr;
    uint4 c0 = make_uint4(0u, 0u, 0u, 0u), c1 = c0;
    if (i < nblocks) { c0 = x[2 * (size_t)i]; c1 = x[2 * (size_t)i + 1]; }
    while (i < nblocks) {
        const uint4 a0 = c0, a1 = c1;
        const uint32_t nxt = i + step;
        if (nxt < nblocks) { c0 = x[2 * (size_t)nxt]; c1 = x[2 * (size_t)nxt + 1]; }
        float v[kBlock];
        unpack16(a0, a1, v);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 f = cen[q][cb];
            if constexpr (MODE == 0) {
                v[4 * q] -= f.x; v[4 * q + 1] -= f.y; v[4 * q + 2] -= f.z; v[4 * q + 3] -= f.w;
            } else {
                v[4 * q] = rb(v[4 * q] - f.x); v[4 * q + 1] = rb(v[4 * q + 1] - f.y);
                v[4 * q + 2] = rb(v[4 * q + 2] - f.z); v[4 * q + 3] = rb(v[4 * q + 3] - f.w);
            }
        }
        const float am = block_amax(v);
        gmax = fmaxf(gmax, am);
        uint2 cw;
        if constexpr (MODE == 0) {
            static_cast<float*>(ws_amax_v)[i] = am;
            cw = encode_rne_wide(v, block_scalar_ieee(am));
        } else {
            static_cast<uint16_t*>(ws_amax_v)[i] = (uint16_t)(__float_as_uint(am) >> 16);
            cw = encode_rne_pb16(v, block_scalar<1>(am));
        }
        __builtin_nontemporal_store((metis_u32x2_t){cw.x, cw.y}, reinterpret_cast<metis_u32x2_t*>(codes) + i);
        i = nxt;
        cb += step_mod;
        cb = cb >= nbpr ? cb - nbpr : cb;
    }
    publish_group_max(gmax, ws_gmax, fill_to);
}

// HAD: every block is rotated first (NV recipe, hadamard16_forward): the rotated tensor is what gets quantized, as in
// `_quantize_wgrad_operand` and `_get_quantized_weight` of src/Metis/Metis/bitlinear.py:395-405, 577-585.  In bf16
// arithmetic the rotated values are rounded to bf16 (the reference's rotation returns the input dtype); in binary32
// arithmetic they are binary32 values that need not be bf16 values, hence WIDE.
// copy (HAD, binary32 input): the tensor itself rounded to bf16, [rows, cols] contiguous: the rank-r branch of the backward pass reads
// a binary32 output gradient in bf16, and a conversion of its own would read all of it once more (45 us at 4096 x 8960; the step of
// that projection, 1536 -> 8960, under the NV recipe: 597 us with it, 582 with the copy from here).
template <int MODE, bool SR, bool WIDE = false, bool HAD = false>
__global__ __launch_bounds__(256) void quant_codes_kernel(
    const void* __restrict__ xv, uint32_t rows, uint32_t cols, int64_t ld, const void* __restrict__ noise,
    uint64_t seed, uint64_t offset, uint2* __restrict__ codes, void* __restrict__ ws_amax_v,
    uint32_t* __restrict__ ws_gmax, uint32_t nblocks, int in_f32, const void* __restrict__ center, uint32_t sign_mask,
    uint32_t fill_to, uint4* __restrict__ copy = nullptr)
{
    static_assert(!WIDE || MODE == 0, "binary32 values imply binary32 arithmetic");
    static_assert(!HAD || WIDE || MODE == 1, "rotated binary32 values are not bf16 values");
    const uint16_t* __restrict__ x = static_cast<const uint16_t*>(xv);
    uint16_t* __restrict__ ws_amax = static_cast<uint16_t*>(ws_amax_v);
    float gmax = 0.0f;
    const uint32_t nbpr = cols / kBlock;      // row layout: blocks per row
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < nblocks; i += gridDim.x * 256u) {
        float v[kBlock], u[kBlock] = {};
        const uint32_t row = i / nbpr, cb = i - row * nbpr;
        if (WIDE && in_f32) {
            const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(xv) + (int64_t)row * ld + (int64_t)cb * kBlock);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float4 f = p[c];
                v[4 * c] = f.x; v[4 * c + 1] = f.y; v[4 * c + 2] = f.z; v[4 * c + 3] = f.w;
            }
            if constexpr (HAD) {
                if (copy) {
                    copy[2 * (size_t)i] = make_uint4(rb_pair(v[0], v[1]), rb_pair(v[2], v[3]), rb_pair(v[4], v[5]), rb_pair(v[6], v[7]));
                    copy[2 * (size_t)i + 1] = make_uint4(rb_pair(v[8], v[9]), rb_pair(v[10], v[11]), rb_pair(v[12], v[13]), rb_pair(v[14], v[15]));
                }
            }
        } else {
            const uint4* p = reinterpret_cast<const uint4*>(x + (int64_t)row * ld + (int64_t)cb * kBlock);
            unpack16(p[0], p[1], v);
        }
        if (center) {
            if constexpr (MODE == 0) {
                const float4* cp = reinterpret_cast<const float4*>(static_cast<const float*>(center) + (size_t)cb * kBlock);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float4 f = cp[c];
                    v[4 * c] -= f.x; v[4 * c + 1] -= f.y; v[4 * c + 2] -= f.z; v[4 * c + 3] -= f.w;
                }
            } else {
                const uint4* cp = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(center) + (size_t)cb * kBlock);
                float cv[kBlock];
                unpack16(cp[0], cp[1], cv);
#pragma unroll
                for (int j = 0; j < kBlock; ++j) v[j] = rb(v[j] - cv[j]);
            }
        }
        if constexpr (HAD) {
            hadamard16_forward(v, sign_mask);
            if constexpr (MODE == 1) {
#pragma unroll
                for (int j = 0; j < kBlock; ++j) v[j] = rb(v[j]);
            }
        }
        if (SR && noise) {
#pragma unroll
            for (int j = 0; j < kBlock; ++j) {
                int64_t e = (int64_t)i * kBlock + j;
                u[j] = MODE ? bf16_lo(((const uint16_t*)noise)[e]) : ((const float*)noise)[e];
            }
        }
        const float am = block_amax(v);
        gmax = fmaxf(gmax, am);
        if constexpr (WIDE) {
            static_cast<float*>(ws_amax_v)[i] = am;
            const float sc = block_scalar_ieee(am);
            if constexpr (SR) codes[i] = !noise ? encode_sr_hardware<0, true>(v, sc, seed, offset, i) : encode_literal<0, true>(v, sc, u);
            else codes[i] = encode_rne_wide(v, sc);
        } else {
            ws_amax[i] = (uint16_t)(__float_as_uint(am) >> 16);      // am is a bf16 value
            // caller-supplied noise: the reference's literal sequence; own stream: hardware stochastic rounding
            codes[i] = (SR && !noise) ? encode_sr_hardware<MODE>(v, block_scalar<MODE>(am), seed, offset, i)
                                      : encode_block<MODE, SR>(v, block_scalar<MODE>(am), u);
        }
    }
    publish_group_max(gmax, ws_gmax, fill_to);
}

// ---------------------------------------------------------------------------------------------
// Phase 1, column-blocked: blocks run down 16 consecutive rows of one column and the packed tensor
// is stored transposed ([cols, rows/2] codes, [cols, rows/16] scales).  A workgroup owns a tile of
// 256 rows x 64 columns: thread t encodes blocks 4g..4g+3 (g = t / 64) of column t % 64, every load
// instruction reading 64 consecutive columns of one row.  Codes and block maxima are transposed
// through LDS so that they leave as 32-byte (8-byte) pieces of the 128 (32) contiguous bytes each
// column owns in the tile, instead of one scattered 8-byte and 2-byte store per lane.
// Rows from `valid` on (valid < rows: a ragged token count padded to the contraction step) are not read: their residual is
// zero, as if the tensor had been copied and filled up with rows equal to the centre.  Without those copies of x and dY a
// training step of an MLP on 2103 tokens (3584 -> 18944, mean mode) takes 4061 instead of 4338 us.
// ---------------------------------------------------------------------------------------------
constexpr int kColTileBlocks = 16, kColTileCols = 64;
// a finished tile leaves LDS: thread t takes column t / 4, blocks 4 (t % 4) .. +3: 32 contiguous bytes of codes, 8 of maxima
template <bool QUADS = true, typename amax_t>
__device__ __forceinline__ void store_col_tile(const uint2 (&s_codes)[kColTileCols][kColTileBlocks + 1], const amax_t (&s_amax)[kColTileCols][kColTileBlocks + 2],
                                               uint2* __restrict__ codes, amax_t* __restrict__ amax, uint32_t tc, uint32_t tr, uint32_t cols, uint32_t nbc)
{
    // A full tile of a packing with whole quads of blocks per column: a column's sixteen blocks are 128 consecutive bytes of codes, two per
    // lane, and their maxima go four to a lane.  Block by block (eight stores of 8 and 2 bytes a thread, each touching a quarter of its
    // lines) every column kernel waited for its stores.  Both launches, bf16 arithmetic: 18944 x 3584 58.1 -> 51.8 us, 4096 x 14336
    // 50.3 -> 43.6; stochastic 4096 x 8960 34.6 -> 30.6; both packings of 4096 x 8960 45.2 -> 40.5, of 2112 x 18944 59.6 -> 51.2.
    // (QUADS: without it both packings of a binary32 tensor, which have no register left for it.)
    typedef uint32_t quad_t __attribute__((ext_vector_type(4), aligned(8)));
    const uint32_t oc = threadIdx.x >> 2, part = threadIdx.x & 3u;
    const uint32_t c2 = tc * kColTileCols + oc, b0 = tr * kColTileBlocks + part * 4u;
    if (QUADS && nbc % 4u == 0u && (tr + 1u) * kColTileBlocks <= nbc) {             // (the same for the workgroup)
#pragma unroll
        for (uint32_t i = 0; i < 2u; ++i) {
            const uint32_t cl = i * 32u + (threadIdx.x >> 3), pair = (threadIdx.x & 7u) * 2u, c3 = tc * kColTileCols + cl;
            const uint2 lo = s_codes[cl][pair], hi = s_codes[cl][pair + 1u];
            if (c3 < cols) *reinterpret_cast<quad_t*>(codes + (int64_t)c3 * nbc + tr * kColTileBlocks + pair) = (quad_t){lo.x, lo.y, hi.x, hi.y};
        }
        if (c2 < cols) {
            struct __attribute__((aligned(4 * sizeof(amax_t)))) four_t { amax_t a[4]; } f;
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) f.a[i] = s_amax[oc][part * 4u + i];
            *reinterpret_cast<four_t*>(amax + (int64_t)c2 * nbc + b0) = f;
        }
        return;
    }
    if (c2 >= cols) return;
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
        if (b0 + i < nbc) {
            const int64_t ob = (int64_t)c2 * nbc + b0 + i;
            codes[ob] = s_codes[oc][part * 4u + i];
            amax[ob] = s_amax[oc][part * 4u + i];
        }
    }
}
// F32IN (WIDE only): the input tensor itself is binary32; a compile-time choice, so that the sixteen loads of a block are
// issued back to back (decided at run time, element by element, the bf16 input of a centred call took twice as long).
template <int MODE, bool SR, bool WIDE = false, bool F32IN = false>
__global__ __launch_bounds__(256) void quant_codes_col_kernel(
    const void* __restrict__ xv, uint32_t rows, uint32_t cols, int64_t ld, const void* __restrict__ noise,
    uint64_t seed, uint64_t offset, uint2* __restrict__ codes, void* __restrict__ ws_amax_v,
    uint32_t* __restrict__ ws_gmax, uint32_t tiles_c, uint32_t tiles_total, const void* __restrict__ center, uint32_t valid)
{
    static_assert(!F32IN || WIDE, "binary32 input implies binary32 values");
    static_assert(!WIDE || MODE == 0, "binary32 values imply binary32 arithmetic");
    using amax_t = typename std::conditional<WIDE, float, uint16_t>::type;   // parked block maximum
    const uint16_t* __restrict__ x = static_cast<const uint16_t*>(xv);
    amax_t* __restrict__ ws_amax = static_cast<amax_t*>(ws_amax_v);
    __shared__ uint2 s_codes[kColTileCols][kColTileBlocks + 1];
    __shared__ amax_t s_amax[kColTileCols][kColTileBlocks + 2];
    const uint32_t nbc = rows / kBlock;                       // blocks per column
    const uint32_t cl = threadIdx.x & 63u, g = threadIdx.x >> 6;
    float gmax = 0.0f;
    for (uint32_t tile = blockIdx.x; tile < tiles_total; tile += gridDim.x) {
        const uint32_t tr = tile / tiles_c, tc = tile - tr * tiles_c;
        const uint32_t c = tc * kColTileCols + cl;
#pragma unroll 1
        for (uint32_t k = 0; k < 4u; ++k) {
            const uint32_t bl = g * 4u + k, b = tr * kColTileBlocks + bl;
            uint2 packed = make_uint2(0u, 0u);
            float am = 0.0f;
            if (c < cols && b < nbc) {
                float v[kBlock], u[kBlock] = {};
                const uint32_t have = valid > b * kBlock ? valid - b * kBlock : 0u;   // rows of this block that x has (the same for the wave)
                if (have >= (uint32_t)kBlock) {
#pragma unroll
                    for (int j = 0; j < kBlock; ++j) {
                        if constexpr (F32IN) v[j] = static_cast<const float*>(xv)[(int64_t)(b * kBlock + j) * ld + c];
                        else v[j] = bf16_lo(x[(int64_t)(b * kBlock + j) * ld + c]);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < kBlock; ++j) {
                        v[j] = 0.0f;
                        if ((uint32_t)j < have) {
                            if constexpr (F32IN) v[j] = static_cast<const float*>(xv)[(int64_t)(b * kBlock + j) * ld + c];
                            else v[j] = bf16_lo(x[(int64_t)(b * kBlock + j) * ld + c]);
                        }
                    }
                }
                if (center) {                                  // one centre per column: the same for the whole block
                    if constexpr (MODE == 0) {
                        const float cen = static_cast<const float*>(center)[c];
#pragma unroll
                        for (int j = 0; j < kBlock; ++j) v[j] -= cen;
                    } else {
                        const float cen = bf16_lo(static_cast<const uint16_t*>(center)[c]);
#pragma unroll
                        for (int j = 0; j < kBlock; ++j) v[j] = rb(v[j] - cen);
                    }
                    if (have < (uint32_t)kBlock) {
#pragma unroll
                        for (int j = 0; j < kBlock; ++j) v[j] = (uint32_t)j < have ? v[j] : 0.0f;
                    }
                }
                if (SR && noise) {
#pragma unroll
                    for (int j = 0; j < kBlock; ++j) {
                        int64_t e = (int64_t)(b * kBlock + j) * cols + c;
                        u[j] = MODE ? bf16_lo(((const uint16_t*)noise)[e]) : ((const float*)noise)[e];
                    }
                }
                am = block_amax(v);
                gmax = fmaxf(gmax, am);
                if constexpr (WIDE) {
                    const float sc = block_scalar_ieee(am);
                    if constexpr (SR) packed = !noise ? encode_sr_hardware<0, true>(v, sc, seed, offset, (int64_t)c * nbc + b)
                                                      : encode_literal<0, true>(v, sc, u);
                    else packed = encode_rne_wide(v, sc);
                } else {
                    packed = (SR && !noise) ? encode_sr_hardware<MODE>(v, block_scalar<MODE>(am), seed, offset, (int64_t)c * nbc + b)
                                            : encode_block<MODE, SR>(v, block_scalar<MODE>(am), u);
                }
            }
            s_codes[cl][bl] = packed;
            if constexpr (WIDE) s_amax[cl][bl] = am;
            else s_amax[cl][bl] = (uint16_t)(__float_as_uint(am) >> 16);
        }
        __syncthreads();
        store_col_tile(s_codes, s_amax, codes, ws_amax, tc, tr, cols, nbc);
        __syncthreads();
    }
    publish_group_max(gmax, ws_gmax);
}

// Column `lane` of a 16 x 64 slab of bf16 values in LDS (rows of `words` words), as binary32 values: four transposing reads, in each of
// which a group of sixteen lanes hands in 4 rows x 16 columns in pieces of four and takes out four rows of a column each.  (Sixteen reads of
// a word that two lanes share, shifted and masked, are twice the vector instructions: both packings of 8192 x 4096 with a centre
// 47.8 -> 44.0 us; the column kernel gains with fewer workgroups, see kColPerCu.)
__device__ __forceinline__ void column_of_slab(const uint32_t* slab, int words, uint32_t lane, float (&v)[kBlock])
{
    typedef short short4_t __attribute__((ext_vector_type(4)));
    typedef short4_t __attribute__((address_space(3))) * lds_ptr_t;
    const uint32_t* p = slab + ((lane >> 2) & 3u) * words + (lane >> 4) * 8u + (lane & 3u) * 2u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint2 d = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p + 4 * q * words)));
        v[4 * q] = __uint_as_float(d.x << 16);
        v[4 * q + 1] = __uint_as_float(d.x & 0xffff0000u);
        v[4 * q + 2] = __uint_as_float(d.y << 16);
        v[4 * q + 3] = __uint_as_float(d.y & 0xffff0000u);
    }
}

// The same with whole 16-byte loads: a wave requests its next 16-row slab of the tile (consecutive lanes consecutive 16-byte
// chunks) while it encodes the current one, and turns it in LDS -- written as loaded, read back as columns, as
// quant_codes_both_kernel does.  A lane's sixteen 2-byte loads per block, each waited for in place, left the kernel above at
// 3 TB/s; now the vector units (Philox, or the encoder and the turning) and HBM bound it together.  Needs 16-byte-aligned rows (ld and cols multiples of 16 bytes) and
// takes no caller noise; same bytes.  Binary32 arithmetic on bf16 values takes its quotients in two operations under the table of block
// maxima, as the row kernel does (18944 x 3584 with scale bytes 82 -> 64 us).  TABLE = false: without it, for tensors of up to 48 rows, of whose tiles one
// wave in four has blocks: the table takes it longer to read than to do without (16 x 64 3.70 | 3.42 us, 32 x 1024 4.92 | 4.71; 64 x 3584 5.50 | 5.48, 256 x 1536
// 5.28 | 5.44).
// Five workgroups per compute unit: enough loads in flight, and fewer partial lines open at once in each die's L2 than with eight.
// With scale bytes, eight | six | five | four: 18944 x 3584 51.5 | 50.0 | 48.3 | 48.2 us, 4096 x 14336 44.2 | 43.2 | 41.5 | 40.0,
// stochastic 2112 x 18944 36.6 | 35.6 | 34.1 | 34.2; binary32 arithmetic, bound by its encoder, 4096 x 14336 52.9 | 56.2 | 54.5 | 57.2,
// 18944 x 3584 64.5 | 61.2 | 64.4 | 67.7.
constexpr int kColPerCu = 5;
template <int MODE, bool SR, bool WIDE = false, bool F32IN = false, bool TABLE = true>
__global__ __launch_bounds__(256) void quant_codes_col_slab_kernel(
    const void* __restrict__ xv, uint32_t rows, uint32_t cols, int64_t ld, uint64_t seed, uint64_t offset, uint2* __restrict__ codes,
    void* __restrict__ ws_amax_v, uint32_t* __restrict__ ws_gmax, uint32_t tiles_c, uint32_t tiles_total, const void* __restrict__ center, uint32_t valid)
{
    static_assert(!F32IN || WIDE, "binary32 input implies binary32 values");
    static_assert(!WIDE || MODE == 0, "binary32 values imply binary32 arithmetic");
    using amax_t = typename std::conditional<WIDE, float, uint16_t>::type;   // parked block maximum
    using elem_t = typename std::conditional<F32IN, float, uint16_t>::type;
    const elem_t* __restrict__ x = static_cast<const elem_t*>(xv);
    amax_t* __restrict__ ws_amax = static_cast<amax_t*>(ws_amax_v);
    __shared__ uint2 s_codes[kColTileCols][kColTileBlocks + 1];
    __shared__ amax_t s_amax[kColTileCols][kColTileBlocks + 2];
    constexpr int kSlabWords = F32IN ? kColTileCols + 4 : kColTileCols / 2;
    __shared__ __attribute__((aligned(16))) uint32_t slab[4][kBlock][kSlabWords];
    constexpr int NQ = F32IN ? 4 : 2, CPR = F32IN ? 16 : 8, RPI = 64 / CPR, EPC = F32IN ? 4 : 8;   // loads per lane, chunks per slab row, rows per load, elements per chunk
    const uint32_t nbc = rows / kBlock;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t g = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lrow = lane / CPR, lch = lane % CPR;
    const elem_t* const xl = x + (int64_t)lrow * ld + lch * EPC;
    auto fetch = [&](uint32_t tile, uint32_t k, uint4 (&q)[NQ]) {
        const uint32_t tr = tile / tiles_c, tc = tile - tr * tiles_c;
        const uint32_t row0 = (tr * kColTileBlocks + g * 4u + k) * kBlock, col0 = tc * kColTileCols;
        const elem_t* p = xl + (int64_t)row0 * ld + col0;
        if (tile < tiles_total && row0 + kBlock <= valid && col0 + kColTileCols <= cols) {     // (the same for the wave)
#pragma unroll
            for (int i = 0; i < NQ; ++i) q[i] = *reinterpret_cast<const uint4*>(p + (int64_t)(i * RPI) * ld);
        } else {
            const bool in = tile < tiles_total && col0 + lch * EPC < cols;
#pragma unroll
            for (int i = 0; i < NQ; ++i)
                q[i] = in && row0 + i * RPI + lrow < valid ? *reinterpret_cast<const uint4*>(p + (int64_t)(i * RPI) * ld) : make_uint4(0u, 0u, 0u, 0u);
        }
    };
    constexpr bool kTable = TABLE && MODE == 0 && !SR && !WIDE;
    __shared__ uint32_t table[kTable ? kQuotientTableWords : 1];
    float gmax = 0.0f;
    uint4 cur[NQ], nxt[NQ];
    fetch(blockIdx.x, 0u, cur);
    if constexpr (kTable) stage_quotient_table(table);
    for (uint32_t tile = blockIdx.x; tile < tiles_total; tile += gridDim.x) {
        const uint32_t tr = tile / tiles_c, tc = tile - tr * tiles_c;
        const uint32_t c = tc * kColTileCols + lane;
        float cen = 0.0f;                                      // one centre per column: the same for all its blocks
        if (center && c < cols) cen = MODE == 0 ? static_cast<const float*>(center)[c] : bf16_lo(static_cast<const uint16_t*>(center)[c]);
#pragma unroll 1
        for (uint32_t k = 0; k < 4u; ++k) {
            fetch(k < 3u ? tile : tile + gridDim.x, k < 3u ? k + 1u : 0u, nxt);
            const uint32_t bl = g * 4u + k, b = tr * kColTileBlocks + bl;
            // a wave's LDS operations complete in the order issued: the barriers only keep the compiler from moving them
#pragma unroll
            for (int i = 0; i < NQ; ++i) *reinterpret_cast<uint4*>(&slab[g][i * RPI + lrow][lch * 4u]) = cur[i];
            __builtin_amdgcn_wave_barrier();
            float v[kBlock];
            if constexpr (F32IN) {
#pragma unroll
                for (int j = 0; j < kBlock; ++j) v[j] = __uint_as_float(slab[g][j][lane]);
            } else {
                column_of_slab(&slab[g][0][0], kSlabWords, lane, v);
            }
            __builtin_amdgcn_wave_barrier();
            uint2 packed = make_uint2(0u, 0u);
            float am = 0.0f;
            if (c < cols && b < nbc) {
                if (center) {
#pragma unroll
                    for (int j = 0; j < kBlock; ++j) v[j] = MODE == 0 ? v[j] - cen : rb(v[j] - cen);
                    const uint32_t have = valid > b * kBlock ? valid - b * kBlock : 0u;
                    if (have < (uint32_t)kBlock) {
#pragma unroll
                        for (int j = 0; j < kBlock; ++j) v[j] = (uint32_t)j < have ? v[j] : 0.0f;
                    }
                }
                const float none[kBlock] = {};
                am = block_amax(v);
                gmax = fmaxf(gmax, am);
                if constexpr (WIDE) {
                    const float sc = block_scalar_ieee(am);
                    if constexpr (SR) packed = encode_sr_hardware<0, true>(v, sc, seed, offset, (int64_t)c * nbc + b);
                    else packed = encode_rne_wide(v, sc);
                } else {
                    if constexpr (SR) packed = encode_sr_hardware<MODE>(v, block_scalar<MODE>(am), seed, offset, (int64_t)c * nbc + b);
                    else if constexpr (kTable) {
                        uint32_t w[2];
                        encode_rne_p32_tbl<kBlock>(v, am, block_scalar<MODE>(am), table, w);
                        packed = make_uint2(w[0], w[1]);
                    } else packed = encode_block<MODE, false>(v, block_scalar<MODE>(am), none);
                }
            }
            s_codes[lane][bl] = packed;
            if constexpr (WIDE) s_amax[lane][bl] = am;
            else s_amax[lane][bl] = (uint16_t)(__float_as_uint(am) >> 16);
#pragma unroll
            for (int i = 0; i < NQ; ++i) cur[i] = nxt[i];
        }
        __syncthreads();
        store_col_tile(s_codes, s_amax, codes, ws_amax, tc, tr, cols, nbc);
        __syncthreads();
    }
    publish_group_max(gmax, ws_gmax);
}

// ---------------------------------------------------------------------------------------------
// Phase 1 of BOTH packings of one tensor in one pass: the weight-gradient and input-gradient GEMMs of the backward
// pass contract the output gradient over different dimensions, so dY is packed twice -- blocks along its last
// dimension (rows) and blocks down its columns (src/Metis/Metis/bitlinear.py:488-510 re-quantizes grad_output for
// each product).  Stochastic rounding on the library's own stream; the two packings draw from their own offsets, so the
// results are those of quant_codes_kernel<.., SR> and quant_codes_col_kernel<.., SR> called one after the other.
// Same tile as the column kernel (256 rows x 64 columns per workgroup, wave g takes 16-row slabs 4g .. 4g+3): a lane
// holds one column of a slab; the slab also goes through LDS (68-word rows) and comes back as row blocks, lane l
// taking row l / 4, block l % 4.  Both packings share the tensor maximum, hence one partial maximum per workgroup.
// copy (binary32 input): the tensor rounded to bf16 as well, as in quant_codes_kernel.
// CEN: one value per column is subtracted first (the mean mode's output gradient), bf16 in bf16 arithmetic, binary32 for a binary32
// tensor; rows past `valid` have a zero residual.  The MLP step of 2103 tokens, 3584 -> 18944: 3824 us with two
// passes over each dY, 3806 with one (the encoders bound it, not the second read).
// ---------------------------------------------------------------------------------------------
// (Five waves per SIMD asked for where the compiler gives them anyway, bf16 without a centre, cost it two registers: 18944 x 3584 60.9 -> 63.2.)
constexpr uint32_t kBothRun = 16;
template <int MODE, bool WIDE = false, bool CEN = false>
__global__ __launch_bounds__(256, CEN ? 4 : WIDE ? 5 : 1) void quant_codes_both_kernel(
    const void* __restrict__ xv, uint32_t rows, uint32_t cols, int64_t ld, uint64_t seed, uint64_t offset_row, uint64_t offset_col,
    uint2* __restrict__ codes_row, void* __restrict__ amax_row_v, uint2* __restrict__ codes_col, void* __restrict__ amax_col_v,
    uint32_t* __restrict__ ws_gmax, uint32_t tiles_c, uint32_t tiles_total, uint32_t valid, uint16_t* __restrict__ copy = nullptr,
    const void* __restrict__ center = nullptr)
{
    static_assert(!WIDE || MODE == 0, "binary32 values imply binary32 arithmetic");
    using amax_t = typename std::conditional<WIDE, float, uint16_t>::type;
    amax_t* __restrict__ amax_row = static_cast<amax_t*>(amax_row_v);
    amax_t* __restrict__ amax_col = static_cast<amax_t*>(amax_col_v);
    __shared__ uint2 s_codes[kColTileCols][kColTileBlocks + 1];
    __shared__ amax_t s_amax[kColTileCols][kColTileBlocks + 2];
    // one 16 x 64 slab per wave, in the input's own width: binary32 words, or bf16 pairs as loaded
    constexpr int kSlabWords = WIDE ? kColTileCols + 4 : kColTileCols / 2 + 4;
    __shared__ __attribute__((aligned(16))) uint32_t slab[4][kBlock][kSlabWords];
    const uint32_t nbc = rows / kBlock, nbpr = cols / kBlock;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t g = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t rr = lane >> 2, cb = lane & 3u;            // as a row block: row rr of the slab, block cb of its 64 columns
    float gmax = 0.0f;
    auto parked = [](float am) -> amax_t {
        if constexpr (WIDE) return am;
        else return (uint16_t)(__float_as_uint(am) >> 16);
    };
    // A tile's row blocks are 32 bytes of a row of codes, and 8 bytes of a row of maxima: kBothRun tiles side by side
    // complete whole 128-byte lines.  Workgroups go round the eight dies in turn, each die with an L2 of its own that
    // merges partial lines; so the workgroups of one die take a run of kBothRun neighbouring tiles at a time.
    const uint32_t span = 8u * kBothRun, padded = (tiles_total + span - 1) / span * span;
    auto tile_of = [&](uint32_t wid) { return wid / span * span + (wid % 8u) * kBothRun + (wid / 8u) % kBothRun; };
    // slab k of workgroup item wid, as the wave loads it: instruction i covers RPI whole rows of the slab, consecutive lanes
    // consecutive 16-byte chunks (every instruction reads whole lines); zeros beyond the tensor.  The next slab's loads are
    // issued before the current one is encoded (one slab ahead, across tiles).
    constexpr int NQ = WIDE ? 4 : 2, CPR = WIDE ? 16 : 8, RPI = 64 / CPR;   // loads per lane, 16-byte chunks per slab row, rows per load
    static_assert(NQ * RPI == kBlock, "the instructions of a wave cover the 16 rows of a slab");
    const uint32_t lrow = lane / CPR, lch = lane % CPR;        // row within an instruction's rows, 16-byte chunk of the row
    using elem_t = typename std::conditional<WIDE, float, uint16_t>::type;
    const elem_t* const xl = static_cast<const elem_t*>(xv) + (int64_t)lrow * ld + lch * (WIDE ? 4u : 8u);
    auto fetch = [&](uint32_t wid, uint32_t k, uint4 (&q)[NQ]) {
        const uint32_t tile = tile_of(wid);
        const bool live = wid < padded && tile < tiles_total;
        const uint32_t tr = tile / tiles_c, tc = tile - tr * tiles_c;
        const uint32_t row0 = (tr * kColTileBlocks + g * 4u + k) * kBlock, col0 = tc * kColTileCols;
        const elem_t* p = xl + (int64_t)row0 * ld + col0;
        if (live && row0 + kBlock <= valid && col0 + kColTileCols <= cols) {       // the same for the wave: no masks, no zeros
#pragma unroll
            for (int i = 0; i < NQ; ++i) q[i] = *reinterpret_cast<const uint4*>(p + (int64_t)(i * RPI) * ld);
        } else {
            const bool in = live && col0 + lch * (WIDE ? 4u : 8u) < cols;
#pragma unroll
            for (int i = 0; i < NQ; ++i)                         // rows from `valid` on are zero, as in quant_codes_col_kernel
                q[i] = in && row0 + i * RPI + lrow < valid ? *reinterpret_cast<const uint4*>(p + (int64_t)(i * RPI) * ld) : make_uint4(0u, 0u, 0u, 0u);
        }
    };
    uint4 cur[NQ], nxt[NQ];
    fetch(blockIdx.x, 0u, cur);
    for (uint32_t wid = blockIdx.x; wid < padded; wid += gridDim.x) {
        const uint32_t tile = tile_of(wid);
        const bool live = tile < tiles_total;                  // the same for the whole workgroup
        const uint32_t tr = tile / tiles_c, tc = tile - tr * tiles_c;
        const uint32_t c = tc * kColTileCols + lane;
        const uint32_t cbg = tc * 4u + cb;
        // the centre of the lane's row block (as stored) and of its column
        uint4 crow[CEN ? (WIDE ? 4 : 2) : 1];
        float ccol = 0.0f;
        if constexpr (CEN) {
#pragma unroll
            for (int q = 0; q < (WIDE ? 4 : 2); ++q)
                crow[q] = live && cbg < nbpr ? reinterpret_cast<const uint4*>(center)[(size_t)cbg * (WIDE ? 4 : 2) + q] : make_uint4(0u, 0u, 0u, 0u);
            if (live && c < cols) ccol = WIDE ? static_cast<const float*>(center)[c] : bf16_lo(static_cast<const uint16_t*>(center)[c]);
        }
#pragma unroll 1
        for (uint32_t k = 0; k < 4u; ++k) {
            if (k < 3u) fetch(wid, k + 1u, nxt);
            else fetch(wid + gridDim.x, 0u, nxt);
            if (live) {
                const uint32_t bl = g * 4u + k, b = tr * kColTileBlocks + bl;
                // to this wave's slab in LDS as loaded, and back as columns.  A wave's LDS operations complete in the
                // order issued, so no wait lies between its own writes and reads: the barriers only keep the compiler
                // from moving them.
                float w[kBlock], v[kBlock];
                const bool have_row = b < nbc && cbg < nbpr;
#pragma unroll
                for (int i = 0; i < NQ; ++i) *reinterpret_cast<uint4*>(&slab[g][i * RPI + lrow][lch * 4u]) = cur[i];
                __builtin_amdgcn_wave_barrier();
                if constexpr (WIDE) {
                    const uint32_t col = tc * kColTileCols + lch * 4u;
                    if (copy && col < cols) {                  // as loaded: 128 consecutive bytes of a row per 16 lanes
#pragma unroll
                        for (int i = 0; i < NQ; ++i) {
                            const uint32_t row = b * kBlock + i * RPI + lrow;
                            if (row < valid)
                                *reinterpret_cast<uint2*>(copy + (size_t)row * cols + col) =
                                    make_uint2(rb_pair(__uint_as_float(cur[i].x), __uint_as_float(cur[i].y)), rb_pair(__uint_as_float(cur[i].z), __uint_as_float(cur[i].w)));
                        }
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint4 f = *reinterpret_cast<const uint4*>(&slab[g][rr][cb * kBlock + 4 * q]);
                        w[4 * q] = __uint_as_float(f.x); w[4 * q + 1] = __uint_as_float(f.y);
                        w[4 * q + 2] = __uint_as_float(f.z); w[4 * q + 3] = __uint_as_float(f.w);
                    }
#pragma unroll
                    for (int j = 0; j < kBlock; ++j) v[j] = __uint_as_float(slab[g][j][lane]);
                } else {
                    unpack16(*reinterpret_cast<const uint4*>(&slab[g][rr][cb * 8u]), *reinterpret_cast<const uint4*>(&slab[g][rr][cb * 8u + 4u]), w);
                    column_of_slab(&slab[g][0][0], kSlabWords, lane, v);
                }
                __builtin_amdgcn_wave_barrier();
                if constexpr (CEN) {
                    const bool row_in = b * kBlock + rr < valid;
                    float cr[kBlock];
                    if constexpr (WIDE) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            cr[4 * q] = __uint_as_float(crow[q].x); cr[4 * q + 1] = __uint_as_float(crow[q].y);
                            cr[4 * q + 2] = __uint_as_float(crow[q].z); cr[4 * q + 3] = __uint_as_float(crow[q].w);
                        }
                    } else {
                        unpack16(crow[0], crow[WIDE ? 0 : 1], cr);
                    }
#pragma unroll
                    for (int j = 0; j < kBlock; ++j) {
                        w[j] = row_in ? rd<MODE>(w[j] - cr[j]) : 0.0f;
                        v[j] = b * kBlock + j < valid ? rd<MODE>(v[j] - ccol) : 0.0f;
                    }
                }
                if (have_row) {
                    const float amr = block_amax(w);
                    gmax = fmaxf(gmax, amr);
                    const int64_t ir = (int64_t)(b * kBlock + rr) * nbpr + cbg;
                    uint2 pr;
                    if constexpr (WIDE) pr = encode_sr_hardware<0, true>(w, block_scalar_ieee(amr), seed, offset_row, ir);
                    else pr = encode_sr_hardware<MODE>(w, block_scalar<MODE>(amr), seed, offset_row, ir);
                    codes_row[ir] = pr;
                    amax_row[ir] = parked(amr);
                }
                uint2 packed = make_uint2(0u, 0u);
                float am = 0.0f;
                if (c < cols && b < nbc) {
                    am = block_amax(v);
                    if constexpr (WIDE) packed = encode_sr_hardware<0, true>(v, block_scalar_ieee(am), seed, offset_col, (int64_t)c * nbc + b);
                    else packed = encode_sr_hardware<MODE>(v, block_scalar<MODE>(am), seed, offset_col, (int64_t)c * nbc + b);
                }
                s_codes[lane][bl] = packed;
                s_amax[lane][bl] = parked(am);
            }
#pragma unroll
            for (int i = 0; i < NQ; ++i) cur[i] = nxt[i];
        }
        if (!live) continue;
        __syncthreads();
        store_col_tile<!WIDE || CEN>(s_codes, s_amax, codes_col, amax_col, tc, tr, cols, nbc);
        __syncthreads();
    }
    publish_group_max(gmax, ws_gmax);
}

// ---------------------------------------------------------------------------------------------
// Phase 2: tensor unit and E4M3 scale bytes (quant.py:21-23), four blocks per thread.
// Every workgroup folds the published partial maxima itself (a few KB from L2).
// ---------------------------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(256) void quant_scales_kernel(const uint16_t* __restrict__ ws_amax,
                                                           const uint32_t* __restrict__ ws_gmax, uint32_t ngroups,
                                                           uint8_t* __restrict__ scales, float* __restrict__ unit_out,
                                                           uint32_t nblocks, const uint16_t* __restrict__ ws_amax2 = nullptr,
                                                           uint8_t* __restrict__ scales2 = nullptr, float* __restrict__ unit_out2 = nullptr)
{
    // grid row 1 (if launched): a second packing of the same tensor (same partial maxima, its own parked block maxima)
    if (blockIdx.y) { ws_amax = ws_amax2; scales = scales2; unit_out = unit_out2; }
    const uint32_t nocts = nblocks / 8u;
    const uint32_t step = gridDim.x * 256u;
    uint32_t q = blockIdx.x * 256u + threadIdx.x;
    // first eight parked maxima are requested before the reduction so that both round trips overlap
    uint4 a = make_uint4(0u, 0u, 0u, 0u);
    if (q < nocts) a = reinterpret_cast<const uint4*>(ws_amax)[q];
    const float amax = fold_group_maxima(ws_gmax, ngroups);
    // max over blocks of scalar(amax_block) = scalar(max amax_block): the scalar map is monotone
    const float unit = tensor_unit_of<MODE>(amax);
    if (blockIdx.x == 0 && threadIdx.x == 0) *unit_out = unit;

    const ScaleBytes<MODE, false> bytes(unit);
    while (q < nocts) {
        const uint32_t nxt = q + step;
        uint4 n = a;
        if (nxt < nocts) n = reinterpret_cast<const uint4*>(ws_amax)[nxt];
        const float am[8] = {bf16_lo(a.x), bf16_hi(a.x), bf16_lo(a.y), bf16_hi(a.y), bf16_lo(a.z), bf16_hi(a.z), bf16_lo(a.w), bf16_hi(a.w)};
        uint32_t o[2];
        bytes(am, o);
        reinterpret_cast<uint2*>(scales)[q] = make_uint2(o[0], o[1]);
        a = n; q = nxt;
    }
    // ragged tail (block count not a multiple of eight)
    for (uint32_t k = nocts * 8u + blockIdx.x * 256u + threadIdx.x; k < nblocks; k += step) {
        const float s = block_scalar<MODE>(__uint_as_float((uint32_t)ws_amax[k] << 16));
        scales[k] = (uint8_t)e4m3_byte(rd<MODE>(s / unit));
    }
}

// Phase 2 for a decode-sized activation (fewer than 256 rows, cols % 256 == 0): unit and scale bytes as above, and the
// packed tensor once more in the decode layout that the decode-sized GEMM streams as whole lines (gemm_common.h): block
// (tile of 32 rows, step of 256 elements) = four KiB of codes, piece j of lane l = (h << 5 | row) at j * 1024 + l * 16,
// then 512 scale bytes, lane l at 4096 + l * 8.  One workgroup per block at a time: thread (j, l) moves a piece, and the
// threads with j == 0 form the eight scale bytes of their lane.  Rows past the tensor are zero.
template <int MODE>
__global__ __launch_bounds__(256) void quant_scales_decode_kernel(const uint16_t* __restrict__ ws_amax, const uint32_t* __restrict__ ws_gmax,
                                                                  uint32_t ngroups, const uint8_t* __restrict__ codes,
                                                                  uint8_t* __restrict__ scales, float* __restrict__ unit_out,
                                                                  uint8_t* __restrict__ decode, int rows, int cols, int blocks)
{
    const float unit = tensor_unit_of<MODE>(fold_group_maxima(ws_gmax, ngroups));
    if (blockIdx.x == 0 && threadIdx.x == 0) *unit_out = unit;
    const int iters = cols / 256, l = threadIdx.x & 63, j = threadIdx.x >> 6, h = l >> 5;
    for (int b = blockIdx.x; b < blocks; b += gridDim.x) {
        const int tile = b / iters, it = b - tile * iters;
        const int row = tile * 32 + (l & 31);
        uint8_t* dst = decode + (int64_t)b * kDecodeBlock;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (row < rows) v = *reinterpret_cast<const uint4*>(codes + (int64_t)row * (cols / 2) + it * 128 + h * 64 + 16 * j);
        *reinterpret_cast<uint4*>(dst + j * 1024 + l * 16) = v;
        if (j == 0) {
            uint2 o = make_uint2(0u, 0u);
            if (row < rows) {
                const int64_t kb = (int64_t)row * (cols / kBlock) + it * 16 + h * 8;
                const uint4 a = *reinterpret_cast<const uint4*>(ws_amax + kb);
                uint32_t by[8];
                const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    by[2 * q] = scale_byte_of<MODE>(w[q] & 0xffffu, unit);
                    by[2 * q + 1] = scale_byte_of<MODE>(w[q] >> 16, unit);
                }
                o.x = by[0] | (by[1] << 8) | (by[2] << 16) | (by[3] << 24);
                o.y = by[4] | (by[5] << 8) | (by[6] << 16) | (by[7] << 24);
                *reinterpret_cast<uint2*>(scales + kb) = o;
            }
            *reinterpret_cast<uint2*>(dst + 4096 + l * 8) = o;
        }
    }
}

// Phase 2 for parked binary32 maxima (binary32 input), four blocks per thread.
__global__ __launch_bounds__(256) void quant_scales_f32_kernel(const float* __restrict__ ws_amax,
                                                               const uint32_t* __restrict__ ws_gmax, uint32_t ngroups,
                                                               uint8_t* __restrict__ scales, float* __restrict__ unit_out,
                                                               uint32_t nblocks, bool divide, const float* __restrict__ ws_amax2 = nullptr,
                                                               uint8_t* __restrict__ scales2 = nullptr, float* __restrict__ unit_out2 = nullptr)
{
    if (blockIdx.y) { ws_amax = ws_amax2; scales = scales2; unit_out = unit_out2; }
    const uint32_t nquads = nblocks / 4u, step = gridDim.x * 256u;
    uint32_t q = blockIdx.x * 256u + threadIdx.x;
    // the next quad is always requested ahead, the first one before the reduction
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (q < nquads) a = reinterpret_cast<const float4*>(ws_amax)[q];
    const float amax = fold_group_maxima(ws_gmax, ngroups);
    const float unit = block_scalar_ieee(amax) / 448.0f;      // the scalar map is monotone: max of scalars = scalar of max
    if (blockIdx.x == 0 && threadIdx.x == 0) *unit_out = unit;
    const ScaleBytes<0, true> bytes(unit);
    while (q < nquads) {
        const uint32_t nxt = q + step;
        float4 n = a;
        if (nxt < nquads) n = reinterpret_cast<const float4*>(ws_amax)[nxt];
        const float am[4] = {a.x, a.y, a.z, a.w};
        uint32_t o[1];
        bytes(am, o, divide);
        reinterpret_cast<uint32_t*>(scales)[q] = o[0];
        a = n; q = nxt;
    }
    for (uint32_t k = nquads * 4u + blockIdx.x * 256u + threadIdx.x; k < nblocks; k += step)
        scales[k] = (uint8_t)e4m3_byte(block_scalar_ieee(ws_amax[k]) / unit);
}

// ---------------------------------------------------------------------------------------------
// Single-launch variant for round-to-nearest rows of a contiguous bf16 tensor: both phases in one kernel.  Each thread
// keeps the maxima of its (at most NB) blocks in registers across a grid-wide maximum, so in the ordinary case neither
// the parked maxima nor a second launch are needed.
//
// The grid-wide maximum is the protocol of grid_max.h; a workgroup that leaves parks its block maxima in the workspace, and what it
// leaves behind are its scale bytes.
// ---------------------------------------------------------------------------------------------
// One block in flight ahead of the one being encoded (as in phase 1 of the two-launch path), block maxima kept in
// registers, and the arrival placed before the encoding of the thread's last block so that the tree's latency is covered.
template <int MODE, int NB>
__global__ __launch_bounds__(256) void quant_fused_kernel(const uint16_t* __restrict__ x, uint2* __restrict__ codes,
                                                          uint8_t* __restrict__ scales, float* __restrict__ unit_out,
                                                          uint32_t* __restrict__ sync, uint16_t* __restrict__ parked,
                                                          uint32_t nblocks, uint32_t spin_limit)
{
    __shared__ GridMaxState sh;
    const uint64_t tag = grid_max_begin(sync);
    const uint32_t stride = gridDim.x * 256u;
    const uint32_t i0 = blockIdx.x * 256u + threadIdx.x;
    const uint4* xp = reinterpret_cast<const uint4*>(x);
    uint4 c0 = make_uint4(0u, 0u, 0u, 0u), c1 = c0;
    if (i0 < nblocks) { c0 = xp[2 * (size_t)i0]; c1 = xp[2 * (size_t)i0 + 1]; }
    float am[NB];
    float gmax = 0.0f;
    const float none[kBlock] = {};
    constexpr int TAIL = NB >= 2 ? 2 : 1;                          // blocks encoded after the arrival
#pragma unroll
    for (int k = 0; k < NB - TAIL; ++k) {
        const uint32_t i = i0 + k * stride;
        uint4 n0 = make_uint4(0u, 0u, 0u, 0u), n1 = n0;
        if (i + stride < nblocks) { n0 = xp[2 * (size_t)(i + stride)]; n1 = xp[2 * (size_t)(i + stride) + 1]; }
        float v[kBlock];
        unpack16(c0, c1, v);
        am[k] = block_amax(v);
        gmax = fmaxf(gmax, am[k]);
        if (i < nblocks) codes[i] = encode_block<MODE, false>(v, block_scalar<MODE>(am[k]), none);
        c0 = n0; c1 = n1;
    }
    {
        // the last blocks: all their maxima first, then the arrival, then their encoding -- a few microseconds of vector
        // work between the arrival and the wait, which is what the tree and the last workgroup's word need to get round
        const uint32_t ia = i0 + (NB - TAIL) * stride, ib = ia + stride;
        uint4 d0 = make_uint4(0u, 0u, 0u, 0u), d1 = d0;
        if (TAIL == 2 && ib < nblocks) { d0 = xp[2 * (size_t)ib]; d1 = xp[2 * (size_t)ib + 1]; }
        float va[kBlock], vb[kBlock];
        unpack16(c0, c1, va);
        am[NB - TAIL] = block_amax(va);
        gmax = fmaxf(gmax, am[NB - TAIL]);
        if (TAIL == 2) {
            unpack16(d0, d1, vb);
            am[NB - 1] = block_amax(vb);
            gmax = fmaxf(gmax, am[NB - 1]);
        }
        grid_max_arrive(gmax, sync, sh);
        if (ia < nblocks) codes[ia] = encode_block<MODE, false>(va, block_scalar<MODE>(am[NB - TAIL]), none);
        if (TAIL == 2 && ib < nblocks) codes[ib] = encode_block<MODE, false>(vb, block_scalar<MODE>(am[NB - 1]), none);
    }
    auto scale_bytes = [&](float amax) {
        const float unit = rd<MODE>(block_scalar<MODE>(amax) / 448.0f);      // quant.py:21-22
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            const uint32_t i = i0 + k * stride;
            if (i < nblocks) scales[i] = (uint8_t)e4m3_byte(rd<MODE>(block_scalar<MODE>(am[k]) / unit));   // quant.py:23
        }
        return unit;
    };
    __syncthreads();                                               // thread 0 is through the tree: sh.last, sh.result
    const uint32_t j = blockIdx.x % kGroups;
    if (!sh.last) {
        // ---- wait for the last workgroup's word, a bounded number of polls
        if (threadIdx.x < 64) {
            uint64_t w = 0;
            uint32_t polls = 0;
            bool have = false;
            for (;;) {
                w = METIS_AT_LOAD(sync_result(sync, j));
                have = is_result(w, tag);
                if (have || ++polls > spin_limit) break;
                __builtin_amdgcn_s_sleep(2);
            }
            if (threadIdx.x == 0) {
                sh.known = have ? 1u : 0u;
                sh.result = __uint_as_float(((uint32_t)w & 0xffffu) << 16);
            }
        }
        __syncthreads();
        if (!sh.known) {
            // ---- leave: park the block maxima, raise the flag, tell the group's word -- unless the result is there by now
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const uint32_t i = i0 + k * stride;
                if (i < nblocks) parked[i] = (uint16_t)(__float_as_uint(am[k]) >> 16);
            }
            __threadfence();
            __syncthreads();
            if (threadIdx.x == 0) {
                METIS_AT_STORE(sync_left_flag(sync, blockIdx.x), (uint32_t)tag);
                __threadfence();                                   // maxima and flag are out before the marker can be seen
                uint64_t w = METIS_AT_LOAD(sync_result(sync, j));
                for (;;) {
                    if (is_result(w, tag)) {
                        sh.known = 1u;
                        sh.result = __uint_as_float(((uint32_t)w & 0xffffu) << 16);
                        break;
                    }
                    if (is_left_marker(w, tag) || METIS_AT_CAS(sync_result(sync, j), &w, result_word(tag, 1u, 0u))) break;
                }
            }
            __syncthreads();
            if (!sh.known) return;                                 // the last workgroup writes this workgroup's scale bytes
        }
        scale_bytes(sh.result);
        return;
    }
    // ---- the last workgroup to arrive: publish, then look after workgroups that have left
    const float amax = sh.result;
    const uint32_t ngroups = gridDim.x < kGroups ? gridDim.x : kGroups;
    bool somebody_left = false;
    if (threadIdx.x < ngroups)
        somebody_left = is_left_marker(METIS_AT_XCHG(sync_result(sync, threadIdx.x), result_word(tag, 0u, __float_as_uint(amax) >> 16)), tag);
    if (threadIdx.x == 0) sh.nleft = 0u;
    const float unit = scale_bytes(amax);
    if (threadIdx.x == 0) *unit_out = unit;
    if (__syncthreads_or(somebody_left)) {
        __threadfence();                                           // their parked maxima and flags were out before their markers
        for (uint32_t slab = 0; slab < gridDim.x; slab += 256u) {
            const uint32_t b = slab + threadIdx.x;
            if (b < gridDim.x && METIS_AT_LOAD(sync_left_flag(sync, b)) == (uint32_t)tag) sh.left[atomicAdd(&sh.nleft, 1u)] = b;
            __syncthreads();
            const uint32_t nd = sh.nleft;
            for (uint32_t d = 0; d < nd; ++d) {
                const uint32_t base = sh.left[d] * 256u + threadIdx.x;
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    const uint32_t i = base + k * stride;
                    if (i < nblocks) {
                        const float a = __uint_as_float((uint32_t)parked[i] << 16);
                        scales[i] = (uint8_t)e4m3_byte(rd<MODE>(block_scalar<MODE>(a) / unit));
                    }
                }
            }
            __syncthreads();
            if (threadIdx.x == 0) sh.nleft = 0u;
            __syncthreads();
        }
    }
    if (threadIdx.x == 0) METIS_AT_STORE(sync_generation(sync), tag);
}

// ---------------------------------------------------------------------------------------------
// Dequantize: ((v * sign) / 2) * (e4m3 * unit), quant.py:23-24 and 32-35.  Eight elements per thread.
// ---------------------------------------------------------------------------------------------
template <int MODE, int OUT_F32>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ codes, const uint8_t* __restrict__ scales,
                                                      const float* __restrict__ unit_p, void* __restrict__ out, int64_t noct)
{
    const float unit = *unit_p;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < noct; i += (int64_t)gridDim.x * 256) {
        const uint32_t c = codes[i];
        const float dq = rd<MODE>(e4m3_value(scales[i >> 1]) * unit);
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t nib = (c >> (4 * j)) & 0xfu, r = nib & 7u;
            // expand (quant.py:32-34): r + relu(r-4) + 2 relu(r-6)
            float v = (float)(r + (r > 4u ? r - 4u : 0u) + (r > 6u ? 2u * (r - 6u) : 0u));
            v = (nib & 8u) ? -v : v;
            o[j] = rd<MODE>((v * 0.5f) * dq);
        }
        if (OUT_F32) {
            float4* p = reinterpret_cast<float4*>(out) + i * 2;
            p[0] = make_float4(o[0], o[1], o[2], o[3]);
            p[1] = make_float4(o[4], o[5], o[6], o[7]);
        } else {
            uint4 w;
            w.x = bf16_bits(o[0]) | (bf16_bits(o[1]) << 16);
            w.y = bf16_bits(o[2]) | (bf16_bits(o[3]) << 16);
            w.z = bf16_bits(o[4]) | (bf16_bits(o[5]) << 16);
            w.w = bf16_bits(o[6]) | (bf16_bits(o[7]) << 16);
            reinterpret_cast<uint4*>(out)[i] = w;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Phase 2 with the dequantized tensor (the round trip of quant.py:6-36: codes, scale bytes AND the dequantized values
// from one call): tensor unit, E4M3 bytes and out = ((v * sign) / 2) * (e4m3 * unit) in one pass over the codes and the
// parked maxima.  A lane owns half a block (one word of codes, 16 bytes of output), so every load and store instruction
// of a wave covers consecutive bytes; the hardware converter turns two codes into their binary32 values (E2M1 = v / 2
// with its sign).  The scale bytes of a wave's 32 blocks leave as eight dwords.
// ---------------------------------------------------------------------------------------------
// WIDE: a binary32 tensor (maxima parked as binary32, IEEE divisions), dequantized to binary32.
typedef float metis_f32x2_t __attribute__((ext_vector_type(2)));
typedef float metis_f32x4_t __attribute__((ext_vector_type(4)));
template <int MODE, bool WIDE = false>
__global__ __launch_bounds__(256) void quant_scales_dequant_kernel(const uint32_t* __restrict__ codes,
                                                                   const typename std::conditional<WIDE, float, uint16_t>::type* __restrict__ ws_amax,
                                                                   const uint32_t* __restrict__ ws_gmax, uint32_t ngroups,
                                                                   uint8_t* __restrict__ scales, float* __restrict__ unit_out,
                                                                   metis_u32x4_t* __restrict__ out, uint32_t nhalves)
{
    static_assert(!WIDE || MODE == 0, "binary32 values imply binary32 arithmetic");
    using amax_t = typename std::conditional<WIDE, float, uint32_t>::type;
    const uint32_t step = gridDim.x * 256u;
    uint32_t i = blockIdx.x * 256u + threadIdx.x;               // half-block index
    uint32_t cw = 0u;
    amax_t aw = 0;
    if (i < nhalves) { cw = codes[i]; aw = ws_amax[i >> 1]; }
    const float amax = fold_group_maxima(ws_gmax, ngroups);
    float unit;
    if constexpr (WIDE) unit = block_scalar_ieee(amax) / 448.0f;
    else unit = tensor_unit_of<MODE>(amax);
    if (blockIdx.x == 0 && threadIdx.x == 0) *unit_out = unit;
    const uint32_t lane = threadIdx.x & 63u;
    while (i < nhalves) {
        const uint32_t nxt = i + step;
        uint32_t ncw = 0u;
        amax_t naw = 0;
        if (nxt < nhalves) { ncw = codes[nxt]; naw = ws_amax[nxt >> 1]; }
        uint32_t byte;
        if constexpr (WIDE) byte = e4m3_byte(block_scalar_ieee(aw) / unit);
        else byte = scale_byte_of<MODE>(aw, unit);
        const float dq = rd<MODE>(e4m3_value(byte) * unit);
        if constexpr (WIDE) {
            metis_f32x4_t* o = reinterpret_cast<metis_f32x4_t*>(out) + 2 * (size_t)i;
            const metis_f32x2_t v0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 0), v1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 1),
                                v2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 2), v3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, 3);
            o[0] = (metis_f32x4_t){v0.x * dq, v0.y * dq, v1.x * dq, v1.y * dq};
            o[1] = (metis_f32x4_t){v2.x * dq, v2.y * dq, v3.x * dq, v3.y * dq};
        } else {
        uint32_t w[4];
#define METIS_DQ_PAIR(J)                                                                                  \
        {                                                                                                 \
            const metis_f32x2_t v = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(cw, 1.0f, J);                \
            w[J] = rb_pair(rd<MODE>(v.x * dq), rd<MODE>(v.y * dq));                                       \
        }
        METIS_DQ_PAIR(0) METIS_DQ_PAIR(1) METIS_DQ_PAIR(2) METIS_DQ_PAIR(3)
#undef METIS_DQ_PAIR
        __builtin_nontemporal_store((metis_u32x4_t){w[0], w[1], w[2], w[3]}, out + i);
        }
        // scale bytes: the wave's 32 blocks; lane 8 j + {0, 2, 4, 6} hold the bytes of dword j
        const uint32_t b1 = __shfl(byte, (lane & ~7u) + 2u, 64), b2 = __shfl(byte, (lane & ~7u) + 4u, 64), b3 = __shfl(byte, (lane & ~7u) + 6u, 64);
        if ((lane & 7u) == 0u) {
            const uint32_t blk = i >> 1;                          // first of four consecutive blocks
            if (2u * (blk + 3u) < nhalves) *reinterpret_cast<uint32_t*>(scales + blk) = byte | (b1 << 8) | (b2 << 16) | (b3 << 24);
            else {
                const uint32_t bs[4] = {byte, b1, b2, b3};
                for (uint32_t j = 0; j < 4u && 2u * (blk + j) < nhalves; ++j) scales[blk + j] = (uint8_t)bs[j];
            }
        }
        cw = ncw; aw = naw; i = nxt;
    }
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
static int grid_for(uint32_t work_items, int per_cu = 8)           // 8 workgroups of 256 per CU are resident
{
    int64_t g = ((int64_t)work_items + 255) / 256;
    const int64_t cap = (int64_t)device_cus() * per_cu;
    if (g > cap) g = cap;
    if (g > kMaxGroups) g = kMaxGroups;
    return g < 1 ? 1 : (int)g;
}

int launch_scales_decode(int mode, const Workspace& ws, uint32_t ngroups, const void* codes, void* scales, float* unit, int64_t rows,
                         int64_t cols, void* decode, hipStream_t st)
{
    if (rows <= 0 || rows >= 256 || cols <= 0 || cols % 256 || (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16)) return METIS_E_ARG;
    if (!decode || ((uintptr_t)decode % 16) || ((uintptr_t)scales % 8) || ((uintptr_t)codes % 16)) return METIS_E_ARG;
    const int blocks = (int)(((rows + 31) / 32) * (cols / 256));
    const int cap = device_cus() * 8;
    const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
    if (mode == 0)
        hipLaunchKernelGGL((quant_scales_decode_kernel<0>), grid, dim3(256), 0, st, ws.amax, ws.gmax, ngroups, (const uint8_t*)codes,
                           (uint8_t*)scales, unit, (uint8_t*)decode, (int)rows, (int)cols, blocks);
    else
        hipLaunchKernelGGL((quant_scales_decode_kernel<1>), grid, dim3(256), 0, st, ws.amax, ws.gmax, ngroups, (const uint8_t*)codes,
                           (uint8_t*)scales, unit, (uint8_t*)decode, (int)rows, (int)cols, blocks);
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

int launch_scales(int mode, const Workspace& ws, uint32_t ngroups, void* scales, float* unit, uint32_t nblocks,
                  hipStream_t st, const void* amax2, void* scales2, float* unit2)
{
    const int g2 = grid_for((nblocks + 7) / 8);
    const dim3 grid((unsigned)g2, amax2 ? 2u : 1u);            // a second packing of the same tensor rides in grid row 1
    // Binary32 maxima: divisions below 2048 blocks, where one workgroup of few waves does it all (ScaleBytes).  Microseconds of the launch, divisions |
    // quotients by three operations first: 16 x 64 2.05 | 2.16, 5 x 1536 2.23 | 2.34; 32 x 1024 2.46 | 2.41, 512 x 4096 3.51 | 3.40.
    if (mode == METIS_MODE_P32_F32)
        hipLaunchKernelGGL(quant_scales_f32_kernel, grid, dim3(256), 0, st, (const float*)ws.amax, ws.gmax, ngroups,
                           (uint8_t*)scales, unit, nblocks, nblocks < 2048u, (const float*)amax2, (uint8_t*)scales2, unit2);
    else if (mode == 0)
        hipLaunchKernelGGL((quant_scales_kernel<0>), grid, dim3(256), 0, st, ws.amax, ws.gmax, ngroups,
                           (uint8_t*)scales, unit, nblocks, (const uint16_t*)amax2, (uint8_t*)scales2, unit2);
    else
        hipLaunchKernelGGL((quant_scales_kernel<1>), grid, dim3(256), 0, st, ws.amax, ws.gmax, ngroups,
                           (uint8_t*)scales, unit, nblocks, (const uint16_t*)amax2, (uint8_t*)scales2, unit2);
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

// Workgroups per compute unit of the contiguous row quantizer: four waves per SIMD hide the memory latency as well as eight
// do, the last round of blocks (encoded with nothing left to overlap) is half as long, and half as many partial maxima
// are folded later.
constexpr int kContigPerCu = 4;

// Co-resident workgroups of the single-launch kernel on the current device (0 = unknown).
template <int MODE, int NB>
static int fused_capacity()
{
    static int cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    if (cached[dev] == 0) {
        int per_cu = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, quant_fused_kernel<MODE, NB>, 256, 0);
        cached[dev] = (e != hipSuccess || per_cu <= 0) ? -1 : per_cu * device_cus();
    }
    return cached[dev] < 0 ? 0 : cached[dev];
}

template <int MODE, int NB>
static int try_fused(const void* x, void* codes, void* scales, float* unit, const Workspace& ws, uint32_t nblocks,
                     hipStream_t st, uint32_t spin_limit)
{
    int cap = fused_capacity<MODE, NB>();
    if (cap > kFusedMaxGrid) cap = kFusedMaxGrid;
    const int64_t need = ((int64_t)nblocks + 256 * NB - 1) / (256 * NB);
    if (cap <= 0 || need > cap) return 1;                      // does not fit: caller picks another path
    hipLaunchKernelGGL((quant_fused_kernel<MODE, NB>), dim3((unsigned)need), dim3(256), 0, st, (const uint16_t*)x,
                       (uint2*)codes, (uint8_t*)scales, unit, ws.sync, ws.amax, nblocks, spin_limit);
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

template <int MODE>
static int launch_fused(const void* x, void* codes, void* scales, float* unit, const Workspace& ws, uint32_t nblocks,
                        hipStream_t st, uint32_t spin_limit)
{
    int rc = try_fused<MODE, 1>(x, codes, scales, unit, ws, nblocks, st, spin_limit);
    if (rc == 1) rc = try_fused<MODE, 2>(x, codes, scales, unit, ws, nblocks, st, spin_limit);
    if (rc == 1) rc = try_fused<MODE, 4>(x, codes, scales, unit, ws, nblocks, st, spin_limit);
    if (rc == 1) rc = try_fused<MODE, 8>(x, codes, scales, unit, ws, nblocks, st, spin_limit);
    return rc;
}

template <int MODE>
static void launch_contig(const void* x, void* codes, const Workspace& ws, uint32_t nblocks, uint32_t fill_to, int grid, hipStream_t st)
{
    if (measure_int("METIS_Q_DEPTH", 1) == 2)
        hipLaunchKernelGGL((quant_codes_contig_kernel<MODE, 2>), dim3(grid), dim3(256), 0, st, (const uint4*)x, (uint2*)codes, ws.amax,
                           ws.gmax, nblocks, fill_to);
    else
        hipLaunchKernelGGL((quant_codes_contig_kernel<MODE, 1>), dim3(grid), dim3(256), 0, st, (const uint4*)x, (uint2*)codes, ws.amax,
                           ws.gmax, nblocks, fill_to);
}

template <int MODE, bool SR, bool COL, bool WIDE = false, bool HAD = false>
static int launch_quant(const void* x, int64_t rows, int64_t cols, int64_t ld, const void* noise, uint64_t seed,
                        uint64_t offset, void* codes, void* scales, float* unit, const Workspace& ws, hipStream_t st,
                        int in_f32 = 0, const void* center = nullptr, uint32_t sign_mask = 0, void* decode = nullptr, int64_t valid = -1,
                        void* copy = nullptr)
{
    static_assert(!HAD || !COL, "the rotation runs along the last dimension, as the row blocks do");
    const uint32_t nblocks = (uint32_t)(rows * cols / kBlock);
    if constexpr (COL) {
        const uint32_t tiles_r = (uint32_t)((rows / kBlock + kColTileBlocks - 1) / kColTileBlocks);
        const uint32_t tiles_c = (uint32_t)((cols + kColTileCols - 1) / kColTileCols);
        const int64_t tiles = (int64_t)tiles_r * tiles_c;
        int64_t g = tiles;
        const int64_t cap = (int64_t)device_cus() * kColPerCu;
        if (g > cap) g = cap;
        if (g > kMaxGroups) g = kMaxGroups;
        const int per16 = (WIDE && in_f32) ? 4 : 8;              // elements of 16 bytes
        if (!noise && cols % per16 == 0 && ld % per16 == 0 && (uintptr_t)x % 16 == 0) {
            // with scale bytes, one element | 16 bytes per load (both with narrow stores): 18944 x 3584 round to nearest 62.0 | 58.3 us,
            // 4096 x 8960 stochastic 35.7 | 30.4, 2112 x 18944 stochastic with a centre 45.6 | 36.7
#define METIS_QCS(F, T) hipLaunchKernelGGL((quant_codes_col_slab_kernel<MODE, SR, WIDE, F, T>), dim3((unsigned)g), dim3(256), 0, st, x, (uint32_t)rows, \
                                        (uint32_t)cols, ld, seed, offset, (uint2*)codes, (void*)ws.amax, ws.gmax, tiles_c, (uint32_t)tiles, center, \
                                        (uint32_t)(valid < 0 ? rows : valid))
            constexpr bool table = MODE == 0 && !SR && !WIDE;
            if (WIDE && in_f32) METIS_QCS(WIDE, false);
            else if (rows < 64) METIS_QCS(false, false);
            else METIS_QCS(false, table);
#undef METIS_QCS
        } else if (WIDE && in_f32)
            hipLaunchKernelGGL((quant_codes_col_kernel<MODE, SR, WIDE, WIDE>), dim3((unsigned)g), dim3(256), 0, st, x,
                               (uint32_t)rows, (uint32_t)cols, ld, noise, seed, offset, (uint2*)codes, (void*)ws.amax, ws.gmax, tiles_c,
                               (uint32_t)tiles, center, (uint32_t)(valid < 0 ? rows : valid));
        else
            hipLaunchKernelGGL((quant_codes_col_kernel<MODE, SR, WIDE, false>), dim3((unsigned)g), dim3(256), 0, st, x,
                               (uint32_t)rows, (uint32_t)cols, ld, noise, seed, offset, (uint2*)codes, (void*)ws.amax, ws.gmax, tiles_c,
                               (uint32_t)tiles, center, (uint32_t)(valid < 0 ? rows : valid));
        return launch_scales(WIDE ? METIS_MODE_P32_F32 : MODE, ws, (uint32_t)g, scales, unit, nblocks, st);
    } else {
        if constexpr (!SR && !HAD && (WIDE ? MODE == 0 : MODE == 1)) {
            if (center && !in_f32 && ld == cols && cols <= kCentreMaxCols) {   // mean mode on contiguous bf16 rows
                if (decode) return METIS_E_ARG;
                const int gc = grid_for(nblocks, kContigPerCu);
                hipLaunchKernelGGL((quant_codes_contig_centered_kernel<MODE>), dim3(gc), dim3(256), 0, st, (const uint4*)x, center,
                                   (uint2*)codes, (void*)ws.amax, ws.gmax, nblocks, (uint32_t)(cols / kBlock), 0u);
                return launch_scales(WIDE ? METIS_MODE_P32_F32 : MODE, ws, (uint32_t)gc, scales, unit, nblocks, st);
            }
        }
        if constexpr (!SR && !WIDE && !HAD) {
            if (!center && ld == cols) {
                const int gc = grid_for(nblocks, measure_int("METIS_Q_WGPC", kContigPerCu));
                launch_contig<MODE>(x, codes, ws, nblocks, 0u, gc, st);
                if (decode) return launch_scales_decode(MODE, ws, (uint32_t)gc, codes, scales, unit, rows, cols, decode, st);
                return launch_scales(MODE, ws, (uint32_t)gc, scales, unit, nblocks, st);
            }
        }
        if (decode) return METIS_E_ARG;                         // only contiguous bf16 rows, round to nearest, come with the decode layout
        const int g1 = grid_for(nblocks);
        hipLaunchKernelGGL((quant_codes_kernel<MODE, SR, WIDE, HAD>), dim3(g1), dim3(256), 0, st, x, (uint32_t)rows,
                           (uint32_t)cols, ld, noise, seed, offset, (uint2*)codes, (void*)ws.amax, ws.gmax, nblocks, in_f32, center,
                           sign_mask, 0u, (uint4*)copy);
        return launch_scales(WIDE ? METIS_MODE_P32_F32 : MODE, ws, (uint32_t)g1, scales, unit, nblocks, st);
    }
}

int quantize(const void* x, int64_t rows, int64_t cols, int64_t ld, int mode, bool sr, bool col, const void* noise,
             uint64_t seed, uint64_t offset, void* codes, void* scales, float* unit, void* workspace,
             size_t workspace_bytes, hipStream_t st, const void* center, bool resident, uint32_t spin_limit, void* decode, int64_t valid)
{
    if (rows < 0 || cols < 0 || ld < cols) return METIS_E_ARG;
    if (valid >= 0 && (!col || valid > rows || noise)) return METIS_E_ARG;
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16 && mode != METIS_MODE_P32_F32) return METIS_E_ARG;
    const bool f32in = mode == METIS_MODE_P32_F32;
    if ((col ? rows : cols) % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;              // nothing to read or write, unit untouched
    if (!x || !codes || !scales || !unit) return METIS_E_ARG;
    if (rows * cols / kBlock >= (int64_t)1 << 31) return METIS_E_ARG;
    if (!col && ((ld % (f32in ? 4 : 8)) || ((uintptr_t)x % 16))) return METIS_E_ARG;     // 16-byte vector loads
    if (col && f32in && ((uintptr_t)x % 4)) return METIS_E_ARG;
    if (center && ((uintptr_t)center % 16)) return METIS_E_ARG;
    const bool wide = f32in || (center && mode == METIS_MODE_P32);   // a binary32 centre leaves binary32 residuals
    if (((uintptr_t)codes % 8) || ((uintptr_t)scales % 8)) return METIS_E_ARG;
    Workspace ws;
    int rc = carve_workspace(workspace, workspace_bytes, rows, cols, &ws);
    if (rc != METIS_OK) return rc;
    if (decode && (sr || col || wide || center || ld != cols || rows >= 256 || cols % 256)) return METIS_E_ARG;
    if (resident && !decode && !sr && !col && !wide && !center && ld == cols) {   // opt-in single-launch path; falls through when it does not fit
        const uint32_t nblocks = (uint32_t)(rows * cols / kBlock);
        if (spin_limit == 0) spin_limit = kSpinLimit;
        rc = mode == 0 ? launch_fused<0>(x, codes, scales, unit, ws, nblocks, st, spin_limit)
                       : launch_fused<1>(x, codes, scales, unit, ws, nblocks, st, spin_limit);
        if (rc != 1) return rc;
    }
#define METIS_Q(M, S, C) return launch_quant<M, S, C>(x, rows, cols, ld, noise, seed, offset, codes, scales, unit, ws, st, 0, center, 0u, decode, valid)
#define METIS_QF(S, C) return launch_quant<0, S, C, true>(x, rows, cols, ld, noise, seed, offset, codes, scales, unit, ws, st, f32in, center, 0u, nullptr, valid)
    if (wide) {
        if (!sr) { if (!col) METIS_QF(false, false); else METIS_QF(false, true); }
        else { if (!col) METIS_QF(true, false); else METIS_QF(true, true); }
    }
#undef METIS_QF
    if (mode == 0) {
        if (!sr) { if (!col) METIS_Q(0, false, false); else METIS_Q(0, false, true); }
        else { if (!col) METIS_Q(0, true, false); else METIS_Q(0, true, true); }
    } else {
        if (!sr) { if (!col) METIS_Q(1, false, false); else METIS_Q(1, false, true); }
        else { if (!col) METIS_Q(1, true, false); else METIS_Q(1, true, true); }
    }
#undef METIS_Q
}

// The round trip of quant.py:6-36 from one call: codes, scale bytes, unit and the dequantized bf16 tensor, two launches
// (phase 1 as in quantize(); phase 2 forms bytes and dequantized values together).  Contiguous bf16 rows, round to nearest.
int quantize_dequantize_row(const void* x, int64_t rows, int64_t cols, int mode, void* codes, void* scales, float* unit, void* out,
                            void* workspace, size_t workspace_bytes, hipStream_t st)
{
    if (rows < 0 || cols < 0) return METIS_E_ARG;
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16 && mode != METIS_MODE_P32_F32) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!x || !codes || !scales || !unit || !out) return METIS_E_ARG;
    if (rows * cols / kBlock >= (int64_t)1 << 30) return METIS_E_ARG;
    if (((uintptr_t)x % 16) || ((uintptr_t)out % 16) || ((uintptr_t)codes % 8) || ((uintptr_t)scales % 8)) return METIS_E_ARG;
    Workspace ws;
    if (const int rc = carve_workspace(workspace, workspace_bytes, rows, cols, &ws)) return rc;
    const uint32_t nblocks = (uint32_t)(rows * cols / kBlock);
    const bool f32in = mode == METIS_MODE_P32_F32;
    const int g1 = f32in ? grid_for(nblocks) : grid_for(nblocks, kContigPerCu);
    if (f32in)
        hipLaunchKernelGGL((quant_codes_kernel<0, false, true>), dim3(g1), dim3(256), 0, st, x, (uint32_t)rows, (uint32_t)cols, cols, (const void*)nullptr,
                           (uint64_t)0, (uint64_t)0, (uint2*)codes, (void*)ws.amax, ws.gmax, nblocks, 1, (const void*)nullptr, 0u, 0u);
    else if (mode == 0) launch_contig<0>(x, codes, ws, nblocks, 0u, g1, st);
    else launch_contig<1>(x, codes, ws, nblocks, 0u, g1, st);
    if (hipGetLastError() != hipSuccess) return METIS_E_LAUNCH;
    const uint32_t nhalves = nblocks * 2u;
    // whole waves of 32 blocks per iteration: the stride is a multiple of 64 halves by construction (256 threads)
    const int g2 = grid_for((nhalves + 3) / 4);                 // four halves per thread
    if (f32in)
        hipLaunchKernelGGL((quant_scales_dequant_kernel<0, true>), dim3(g2), dim3(256), 0, st, (const uint32_t*)codes, (const float*)ws.amax, ws.gmax,
                           (uint32_t)g1, (uint8_t*)scales, unit, (metis_u32x4_t*)out, nhalves);
    else if (mode == 0)
        hipLaunchKernelGGL((quant_scales_dequant_kernel<0>), dim3(g2), dim3(256), 0, st, (const uint32_t*)codes, ws.amax, ws.gmax, (uint32_t)g1,
                           (uint8_t*)scales, unit, (metis_u32x4_t*)out, nhalves);
    else
        hipLaunchKernelGGL((quant_scales_dequant_kernel<1>), dim3(g2), dim3(256), 0, st, (const uint32_t*)codes, ws.amax, ws.gmax, (uint32_t)g1,
                           (uint8_t*)scales, unit, (metis_u32x4_t*)out, nhalves);
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

// Workgroups of quant_codes_both_kernel that the current device holds at once (its LDS slabs bound them): the grid is
// no larger, so that every workgroup starts at once.  How many tiles each then has is a matter of the spans (quantize_both_sr).
template <int MODE, bool WIDE, bool CEN>
static int both_capacity()
{
    static int cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    if (cached[dev] == 0) {
        int per_cu = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, quant_codes_both_kernel<MODE, WIDE, CEN>, 256, 0);
        cached[dev] = (e != hipSuccess || per_cu <= 0) ? -1 : per_cu * device_cus();
    }
    return cached[dev] < 0 ? device_cus() * 4 : cached[dev];
}

// ---------------------------------------------------------------------------------------------
// Both packings of one tensor (rows and columns) with stochastic rounding, one pass over x; then phase 2 for each.
// The workspace holds two areas of parked maxima: 2 x workspace_bytes(rows, cols).
// ---------------------------------------------------------------------------------------------
int quantize_both_sr(const void* x, int64_t rows, int64_t cols, int64_t ld, int mode, uint64_t seed, uint64_t offset_row,
                     uint64_t offset_col, void* codes_row, void* scales_row, float* unit_row, void* codes_col, void* scales_col,
                     float* unit_col, void* workspace, size_t bytes, hipStream_t st, int64_t valid, void* copy, const void* center)
{
    if (rows < 0 || cols < 0 || ld < cols || valid > rows) return METIS_E_ARG;
    if (copy && (mode != METIS_MODE_P32_F32 || ((uintptr_t)copy % 16))) return METIS_E_ARG;
    if (center && ((mode != METIS_MODE_P32_F32 && mode != METIS_MODE_PB16) || ((uintptr_t)center % 16))) return METIS_E_ARG;   // (a binary32 centre leaves binary32 residuals)
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16 && mode != METIS_MODE_P32_F32) return METIS_E_ARG;
    const bool f32in = mode == METIS_MODE_P32_F32;
    if (rows % kBlock || cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!x || !codes_row || !scales_row || !unit_row || !codes_col || !scales_col || !unit_col) return METIS_E_ARG;
    if (rows * cols / kBlock >= (int64_t)1 << 31) return METIS_E_ARG;
    if ((ld % (f32in ? 4 : 8)) || ((uintptr_t)x % 16)) return METIS_E_ARG;                 // 16-byte vector loads
    if (((uintptr_t)codes_row % 8) || ((uintptr_t)scales_row % 8) || ((uintptr_t)codes_col % 8) || ((uintptr_t)scales_col % 8)) return METIS_E_ARG;
    const size_t one = workspace_bytes(rows, cols);
    if (!workspace || ((uintptr_t)workspace % 256) || bytes < 2 * one) return METIS_E_WORKSPACE;
    Workspace wr, wc;
    if (const int rc = carve_workspace(workspace, one, rows, cols, &wr)) return rc;
    if (const int rc = carve_workspace(static_cast<char*>(workspace) + one, one, rows, cols, &wc)) return rc;
    wc.gmax = wr.gmax;                                         // one tensor, one maximum: both packings fold the same partials
    const uint32_t nblocks = (uint32_t)(rows * cols / kBlock);
    const uint32_t tiles_r = (uint32_t)((rows / kBlock + kColTileBlocks - 1) / kColTileBlocks);
    const uint32_t tiles_c = (uint32_t)((cols + kColTileCols - 1) / kColTileCols);
    const int64_t tiles = (int64_t)tiles_r * tiles_c;
    // One workgroup for every place of the last, partly filled, span of eight runs while they all fit the device: a grid of as many
    // workgroups as tiles left the tiles behind the empty places to workgroups that had one already (two of 16 workgroups took all of
    // 256 x 1024).  With the scale bytes, bf16 arithmetic, before -> now: 256 x 1024 42.3 -> 9.9 us, 512 x 1536 19.5 -> 10.0, 512 x 8960
    // 16.3 -> 13.1, 1488 x 3648 16.9 -> 14.0, 2048 x 8960 26.2 -> 23.9; whole spans and tensors beyond the device's capacity as before.
    const int64_t span = 8 * kBothRun;
    int64_t g = (tiles + span - 1) / span * span;
    const int64_t cap = center ? (f32in ? both_capacity<0, true, true>() : both_capacity<1, false, true>())
                               : f32in ? both_capacity<0, true, false>() : mode == 0 ? both_capacity<0, false, false>() : both_capacity<1, false, false>();
    if (g > cap) g = cap;
    if (g > kMaxGroups) g = kMaxGroups;
#define METIS_QB(M, W, C) hipLaunchKernelGGL((quant_codes_both_kernel<M, W, C>), dim3((unsigned)g), dim3(256), 0, st, x, (uint32_t)rows, \
                                          (uint32_t)cols, ld, seed, offset_row, offset_col, (uint2*)codes_row, (void*)wr.amax, (uint2*)codes_col, \
                                          (void*)wc.amax, wr.gmax, tiles_c, (uint32_t)tiles, (uint32_t)(valid < 0 ? rows : valid), (uint16_t*)copy, center)
    if (center) { if (f32in) METIS_QB(0, true, true); else METIS_QB(1, false, true); }
    else if (f32in) METIS_QB(0, true, false);
    else if (mode == 0) METIS_QB(0, false, false);
    else METIS_QB(1, false, false);
#undef METIS_QB
    if (hipGetLastError() != hipSuccess) return METIS_E_LAUNCH;
    const int pm = f32in ? METIS_MODE_P32_F32 : mode;
    return launch_scales(pm, wr, (uint32_t)g, scales_row, unit_row, nblocks, st, wc.amax, scales_col, unit_col);   // one launch for both
}

// ---------------------------------------------------------------------------------------------
// Deferred scale bytes.  The codes of a block depend on the block alone, the scale bytes on the tensor maximum: a
// consumer that runs after the quantizer anyway (the tiled expansion ahead of a GEMM) can form them from the parked
// block maxima, and the quantizer is then ONE launch.  The caller owns the parked data: [0, 8 KiB) the partial maxima
// (kDeferredPartials entries), then one bf16 maximum per block.  Round-to-nearest rows of a contiguous bf16 tensor.
// ---------------------------------------------------------------------------------------------
size_t deferred_bytes(int64_t rows, int64_t cols)
{
    if (rows <= 0 || cols <= 0) return 0;
    const size_t nblocks = (size_t)((rows * cols + 15) / 16);
    return kDeferredPartials * 4 + ((nblocks * 2 + 255) / 256) * 256;
}

int carve_deferred(void* p, size_t bytes, int64_t rows, int64_t cols, Workspace* ws)
{
    if (!p || ((uintptr_t)p % 256) || bytes < deferred_bytes(rows, cols)) return METIS_E_WORKSPACE;
    ws->gmax = static_cast<uint32_t*>(p);
    ws->sync = nullptr;
    ws->amax = reinterpret_cast<uint16_t*>(static_cast<char*>(p) + kDeferredPartials * 4);
    return METIS_OK;
}

int deferred_grid(uint32_t work_items, int per_cu)
{
    const int g = grid_for(work_items, per_cu);
    return g > (int)kDeferredPartials ? (int)kDeferredPartials : g;
}

// center (bf16 arithmetic only: a binary32 centre leaves residuals whose maxima are not bf16 values): one bf16 value per
// column subtracted first, as quantize() does for the mean mode.
int quantize_row_deferred(const void* x, int64_t rows, int64_t cols, int mode, const void* center, void* codes, void* deferred,
                          size_t bytes, hipStream_t st)
{
    if (rows < 0 || cols < 0) return METIS_E_ARG;
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16) return METIS_E_ARG;
    if (center && (mode != METIS_MODE_PB16 || ((uintptr_t)center % 16))) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!x || !codes || ((uintptr_t)x % 16) || ((uintptr_t)codes % 8)) return METIS_E_ARG;
    if (rows * cols / kBlock >= (int64_t)1 << 31) return METIS_E_ARG;
    Workspace ws;
    if (const int rc = carve_deferred(deferred, bytes, rows, cols, &ws)) return rc;
    const uint32_t nblocks = (uint32_t)(rows * cols / kBlock);
    const int g1 = deferred_grid(nblocks, center ? 8 : measure_int("METIS_Q_WGPC", kContigPerCu));
    if (center && cols <= kCentreMaxCols)
        hipLaunchKernelGGL((quant_codes_contig_centered_kernel<1>), dim3(g1), dim3(256), 0, st, (const uint4*)x, center, (uint2*)codes,
                           (void*)ws.amax, ws.gmax, nblocks, (uint32_t)(cols / kBlock), kDeferredPartials);
    else if (center)
        hipLaunchKernelGGL((quant_codes_kernel<1, false, false, false>), dim3(g1), dim3(256), 0, st, x, (uint32_t)rows, (uint32_t)cols,
                           cols, nullptr, (uint64_t)0, (uint64_t)0, (uint2*)codes, (void*)ws.amax, ws.gmax, nblocks, 0, center, 0u,
                           kDeferredPartials);
    else if (mode == 0)
        launch_contig<0>(x, codes, ws, nblocks, kDeferredPartials, g1, st);
    else
        launch_contig<1>(x, codes, ws, nblocks, kDeferredPartials, g1, st);
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

// quantize_row_deferred of a decode-sized contiguous bf16 activation and, in the same launch, the first step of its
// rank-r projection onto v [R, cols]: partial sums per K chunk into lr_workspace (lowrank_small's workspace), for a
// finishing step that runs later (decode_prepare_deferred with x = nullptr).
int quantize_row_deferred_partial(const void* x, int64_t rows, int64_t cols, int mode, void* codes, void* deferred, size_t bytes,
                                  const void* v, int64_t R, void* lr_workspace, size_t lr_workspace_bytes, hipStream_t st)
{
    if (rows < 0 || cols < 0 || R <= 0) return METIS_E_ARG;
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16) return METIS_E_ARG;
    if (rows == 0 || rows >= 256 || cols == 0 || cols % 64 || R % 32 || R > 128) return METIS_E_SHAPE;
    if (!x || !codes || !v || ((uintptr_t)x % 16) || ((uintptr_t)codes % 8) || ((uintptr_t)v % 16)) return METIS_E_ARG;
    if (!lr_workspace || ((uintptr_t)lr_workspace % 16) || lr_workspace_bytes < lowrank_small_workspace_bytes(rows, R, cols))
        return METIS_E_WORKSPACE;
    Workspace ws;
    if (const int rc = carve_deferred(deferred, bytes, rows, cols, &ws)) return rc;
    const uint32_t nblocks = (uint32_t)(rows * cols / kBlock);
    const int g1 = deferred_grid(nblocks, kContigPerCu);
    int kc;
    const int chunks = lowrank_small_chunks(cols, &kc);
    const bool wide = lowrank_small_wide(rows, R, cols, device_cus());
    const int g = g1 + lowrank_small_partial_blocks(rows, R, chunks, wide);
#define METIS_QP(MODE) hipLaunchKernelGGL((decode_quant_partial_kernel<MODE>), dim3(g), dim3(256), 0, st, (uint32_t)g1, (const uint4*)x, \
                                          (uint2*)codes, ws.amax, ws.gmax, nblocks, kDeferredPartials, cols, (const uint16_t*)v, \
                                          (int)rows, (int)R, (int)cols, kc, chunks, (int)wide, (float*)lr_workspace)
    if (mode == 0) METIS_QP(0); else METIS_QP(1);
#undef METIS_QP
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

// phase 2 on parked data, whenever somebody wants the bytes after all
int deferred_scales(const void* deferred, int64_t rows, int64_t cols, int mode, void* scales, float* unit, hipStream_t st)
{
    if (rows < 0 || cols < 0 || (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16)) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!scales || !unit || ((uintptr_t)scales % 8)) return METIS_E_ARG;
    Workspace ws;
    if (const int rc = carve_deferred(const_cast<void*>(deferred), deferred_bytes(rows, cols), rows, cols, &ws)) return rc;
    return launch_scales(mode, ws, kDeferredPartials, scales, unit, (uint32_t)(rows * cols / kBlock), st);
}

// ---------------------------------------------------------------------------------------------
// "svd" mode of the activation / output-gradient decomposition (src/Metis/Metis/bitlinear.py:283-303): the tensor that is
// quantized is x - ker with ker = (U diag(s)) V of rank r, and the caller goes on with ker + QDQ(x - ker).  Every element of ker
// is the chain
//     acc = 0;  acc = fma(us[i][k], v[k][j], acc)  for k = 0 .. r-1 in that order, in binary32
// (bf16 arithmetic: exact products of bf16 factors, the sum rounded to bf16 once, as a bf16 matrix product with
// binary32 accumulation does) -- a fixed order, so that a CPU restatement reproduces the bits.  v_mfma_f32_32x32x2_f32 is that
// chain for its two values of k (k = 0 from lanes 0..31, then k = 1 from lanes 32..63, each a fused multiply-add, subnormals
// included; the tests hold it to the restatement bit for bit).
//
// A wave forms 32 rows x 64 columns and needs neither LDS nor a barrier: V's operand is a row of V as it lies (coalesced words), U's
// are 16 bytes a lane along the rank, put in order by two half swaps, and 8 half swaps turn a lane's 16 sums into one block of 16
// columns, ready for the encoder.  The four waves of a workgroup lie side by side: they read the same rows of U from L1 and write
// whole lines of codes.  Then the residual x - ker (rounded to the arithmetic's type) is encoded like any other block; the codes and
// the parked block maxima go where the row quantizer puts them, and ker is written out only when the caller wants the dense result.
//
// What bounds it: the SIMDs.  Binary32 MFMAs reach 137 TFLOP/s alone and vector FMAs 96, but the two do not run side by side (63 + 63
// when mixed in one wave).  At 4096 x 3584, r = 64 the matrix units are busy 12 and the vector units 9 of the kernel's 27 us; 1.75 of two rounds of
// workgroups are filled.  Call
// with its scales launch, in a graph, vector FMAs from LDS tiles before -> now: binary32 4096 x 3584 r = 64 39.5 -> 35.1 us (30.9 with the scale bytes as they are formed now), r = 32
// 28.3 -> 26.7, 1000 x 2048 r = 64 19.1 -> 10.6, 128 x 1024 r = 32 13.4 -> 8.7; bf16 4096 x 3584 r = 64 39.3 -> 33.4, 2048 x 1536 r = 64
// 19.7 -> 13.4.  64 rows a wave: 13.7 at 1000 x 2048 (half as many waves), 36.5 at the largest; x requested before the products: 38.1
// (U's lines leave L1 meanwhile).
// ---------------------------------------------------------------------------------------------
constexpr int kLrRows = 32, kLrCols = 256, kLrRanks = 16;
typedef float lr_acc_t __attribute__((ext_vector_type(16)));

// lanes 32..63 of a against lanes 0..31 of b
__device__ __forceinline__ void swap_halves(float& a, float& b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

template <int MODE, bool F32IN>
__global__ __launch_bounds__(256, 4) void quant_lowrank_residual_kernel(
    const void* __restrict__ xv, const void* __restrict__ usv, const void* __restrict__ vtv, uint32_t rows, uint32_t cols,
    uint32_t rank, uint2* __restrict__ codes, void* __restrict__ ws_amax_v, uint32_t* __restrict__ ws_gmax,
    void* __restrict__ ker_out, uint32_t tiles_c, uint32_t tiles)
{
    static_assert(MODE == 0 || !F32IN, "bf16 arithmetic reads bf16 tensors");
    typedef typename std::conditional<MODE == 0, float, uint16_t>::type factor_t;
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 31u, hi = lane >> 5;
    const uint32_t nbpr = cols / kBlock;
    float gmax = 0.0f;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t tr = tile / tiles_c, tc = tile - tr * tiles_c;
        const uint32_t row0 = tr * kLrRows, col0 = tc * kLrCols + wave * 64u;
        if (col0 >= cols) continue;                             // (no barrier inside the loop)
        // rows and columns beyond the tensor read its last ones: their products are not used
        const factor_t* pv[2];
#pragma unroll
        for (uint32_t b = 0; b < 2; ++b) pv[b] = static_cast<const factor_t*>(vtv) + (size_t)hi * cols + min(col0 + 32u * b + j, cols - 1u);
        const factor_t* pu = static_cast<const factor_t*>(usv) + (size_t)min(row0 + j, rows - 1u) * rank + hi * 4u;
        factor_t nv[2][4];                                      // V of ranks k0 + 2 s + hi
        typedef typename std::conditional<MODE == 0, float4, uint2>::type four_t;
        four_t nu;                                              // U diag(s) of ranks k0 + 4 hi ..
        auto fetch = [&]() {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int s = 0; s < 4; ++s) nv[b][s] = pv[b][(size_t)(2 * s) * cols];
                pv[b] += (size_t)8 * cols;
            }
            nu = *reinterpret_cast<const four_t*>(pu);
            pu += 8;
        };
        lr_acc_t acc[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[b][e] = 0.0f;
        fetch();
        for (uint32_t k0 = 0; k0 < rank; k0 += 8) {
            float fv[2][4];
            float4 u;
            if constexpr (MODE == 0) u = nu;
            else u = make_float4(bf16_lo(nu.x), bf16_hi(nu.x), bf16_lo(nu.y), bf16_hi(nu.y));
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if constexpr (MODE == 0) fv[b][s] = nv[b][s];
                    else fv[b][s] = __uint_as_float((uint32_t)nv[b][s] << 16);
                }
            // (k0, k0 + 4), (k0 + 1, k0 + 5) -> (k0, k0 + 1), (k0 + 4, k0 + 5), and likewise the other pair
            swap_halves(u.x, u.y);
            swap_halves(u.z, u.w);
            const float fu[4] = {u.x, u.z, u.y, u.w};
            if (k0 + 8 < rank) fetch();
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int b = 0; b < 2; ++b) acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(fv[b][s], fu[s], acc[b], 0, 0, 0);
        }
        const uint32_t row = row0 + j;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            // a lane holds columns 8 q + 4 hi + (0..3) of its row, q = 0..3: after the swaps the lower lanes have columns 0..15, the upper
            // ones 16..31 of the 32
            float ker[kBlock];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float lo = acc[b][e], up = acc[b][e + 8];
                swap_halves(lo, up);
                ker[(e & 4) * 2 + (e & 3)] = lo;
                ker[(e & 4) * 2 + (e & 3) + 4] = up;
            }
            const uint32_t cbg = col0 / kBlock + 2u * b + hi;
            if (row >= rows || cbg >= nbpr) continue;
            const size_t e0 = (size_t)row * cols + (size_t)cbg * kBlock;
            float v[kBlock];
            if constexpr (F32IN) {
                const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(xv) + e0);
#pragma unroll
                for (int q = 0; q < 4; ++q) { const float4 f = p[q]; v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w; }
            } else {
                const uint4* p = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(xv) + e0);
                unpack16(p[0], p[1], v);
            }
            if constexpr (MODE == 0) {
                if (ker_out) {
                    float4* o = reinterpret_cast<float4*>(static_cast<float*>(ker_out) + e0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) o[q] = make_float4(ker[4 * q], ker[4 * q + 1], ker[4 * q + 2], ker[4 * q + 3]);
                }
#pragma unroll
                for (int i = 0; i < kBlock; ++i) v[i] -= ker[i];
            } else {
                uint32_t kw[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) kw[i] = bf16_bits(ker[2 * i]) | (bf16_bits(ker[2 * i + 1]) << 16);
                if (ker_out) {
                    uint4* o = reinterpret_cast<uint4*>(static_cast<uint16_t*>(ker_out) + e0);
                    o[0] = make_uint4(kw[0], kw[1], kw[2], kw[3]);
                    o[1] = make_uint4(kw[4], kw[5], kw[6], kw[7]);
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    v[2 * i] = rb(v[2 * i] - bf16_lo(kw[i]));
                    v[2 * i + 1] = rb(v[2 * i + 1] - bf16_hi(kw[i]));
                }
            }
            const float am = block_amax(v);
            gmax = fmaxf(gmax, am);
            const uint32_t blk = row * nbpr + cbg;
            if constexpr (MODE == 0) {
                static_cast<float*>(ws_amax_v)[blk] = am;
                codes[blk] = encode_rne_wide(v, block_scalar_ieee(am));
            } else {
                const float none[kBlock] = {};
                static_cast<uint16_t*>(ws_amax_v)[blk] = (uint16_t)(__float_as_uint(am) >> 16);
                codes[blk] = encode_block<1, false>(v, block_scalar<1>(am), none);
            }
        }
    }
    publish_group_max(gmax, ws_gmax, 0u);
}

// out = ker + QDQ(x - ker), in place on the buffer that holds ker (bitlinear.py:301-303): eight elements per thread
template <int MODE>
__global__ __launch_bounds__(256) void lowrank_add_dequant_kernel(const uint32_t* __restrict__ codes, const uint8_t* __restrict__ scales,
                                                                  const float* __restrict__ unit_p, void* __restrict__ out, int64_t noct)
{
    const float unit = *unit_p;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < noct; i += (int64_t)gridDim.x * 256) {
        const uint32_t c = codes[i];
        const float dq = rd<MODE>(e4m3_value(scales[i >> 1]) * unit);
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t nib = (c >> (4 * j)) & 0xfu, r = nib & 7u;
            float v = (float)(r + (r > 4u ? r - 4u : 0u) + (r > 6u ? 2u * (r - 6u) : 0u));
            v = (nib & 8u) ? -v : v;
            o[j] = rd<MODE>((v * 0.5f) * dq);
        }
        if constexpr (MODE == 0) {
            float4* p = reinterpret_cast<float4*>(out) + i * 2;
            const float4 a = p[0], b = p[1];
            p[0] = make_float4(a.x + o[0], a.y + o[1], a.z + o[2], a.w + o[3]);
            p[1] = make_float4(b.x + o[4], b.y + o[5], b.z + o[6], b.w + o[7]);
        } else {
            uint4* p = reinterpret_cast<uint4*>(out) + i;
            const uint4 k = *p;
            uint4 w;
            w.x = rb_pair(bf16_lo(k.x) + o[0], bf16_hi(k.x) + o[1]);
            w.y = rb_pair(bf16_lo(k.y) + o[2], bf16_hi(k.y) + o[3]);
            w.z = rb_pair(bf16_lo(k.z) + o[4], bf16_hi(k.z) + o[5]);
            w.w = rb_pair(bf16_lo(k.w) + o[6], bf16_hi(k.w) + o[7]);
            *p = w;
        }
    }
}

int quantize_lowrank_residual(const void* x, bool x_f32, const void* us, const void* vt, int64_t rows, int64_t cols, int rank, int mode,
                              void* codes, void* scales, float* unit, void* dense, void* workspace, size_t workspace_bytes,
                              hipStream_t st)
{
    if (rows < 0 || cols < 0 || rank <= 0) return METIS_E_ARG;
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16) return METIS_E_ARG;
    if (x_f32 && mode != METIS_MODE_P32) return METIS_E_ARG;
    if (cols % kBlock || rank % kLrRanks) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!x || !us || !vt || !codes || !scales || !unit) return METIS_E_ARG;
    if (((uintptr_t)x % 16) || ((uintptr_t)us % 16) || ((uintptr_t)vt % 16) || ((uintptr_t)dense % 16) || ((uintptr_t)codes % 8) ||
        ((uintptr_t)scales % 8))
        return METIS_E_ARG;
    if (rows * cols / kBlock >= (int64_t)1 << 31) return METIS_E_ARG;
    Workspace ws;
    if (const int rc = carve_workspace(workspace, workspace_bytes, rows, cols, &ws)) return rc;
    const uint32_t tiles_c = (uint32_t)((cols + kLrCols - 1) / kLrCols);
    const int64_t tiles = (int64_t)((rows + kLrRows - 1) / kLrRows) * tiles_c;
    int64_t g = tiles;
    if (g > kMaxGroups) g = kMaxGroups;
    const uint32_t nblocks = (uint32_t)(rows * cols / kBlock);
#define METIS_LR(M, F)                                                                                                          \
    hipLaunchKernelGGL((quant_lowrank_residual_kernel<M, F>), dim3((unsigned)g), dim3(256), 0, st, x, us, vt, (uint32_t)rows,      \
                       (uint32_t)cols, (uint32_t)rank, (uint2*)codes, (void*)ws.amax, ws.gmax, dense, tiles_c, (uint32_t)tiles)
    if (mode == METIS_MODE_PB16) METIS_LR(1, false);
    else if (x_f32) METIS_LR(0, true);
    else METIS_LR(0, false);
#undef METIS_LR
    if (hipGetLastError() != hipSuccess) return METIS_E_LAUNCH;
    if (const int rc = launch_scales(mode == METIS_MODE_P32 ? METIS_MODE_P32_F32 : METIS_MODE_PB16, ws, (uint32_t)g, scales, unit, nblocks, st,
                                     nullptr, nullptr, nullptr))
        return rc;
    if (dense) {
        const int64_t noct = rows * cols / 8;
        const int g3 = grid_for((uint32_t)noct);                 // noct < 2^32: nblocks < 2^31
        if (mode == METIS_MODE_P32)
            hipLaunchKernelGGL((lowrank_add_dequant_kernel<0>), dim3(g3), dim3(256), 0, st, (const uint32_t*)codes, (const uint8_t*)scales, unit, dense, noct);
        else
            hipLaunchKernelGGL((lowrank_add_dequant_kernel<1>), dim3(g3), dim3(256), 0, st, (const uint32_t*)codes, (const uint8_t*)scales, unit, dense, noct);
        if (hipGetLastError() != hipSuccess) return METIS_E_LAUNCH;
    }
    return METIS_OK;
}

// ---------------------------------------------------------------------------------------------
// NV recipe: rotate every tile of 16 along the last dimension, then quantize the rotated tensor (row blocks = tiles),
// in one pass over x.  Round to nearest, or stochastic rounding on the library's own stream.
// ---------------------------------------------------------------------------------------------
int quantize_rht(const void* x, int64_t rows, int64_t cols, int64_t ld, int mode, uint32_t sign_mask, bool sr, uint64_t seed,
                 uint64_t offset, void* codes, void* scales, float* unit, void* workspace, size_t workspace_bytes, hipStream_t st, void* copy)
{
    if (rows < 0 || cols < 0 || ld < cols || sign_mask > 0xffffu) return METIS_E_ARG;
    if (copy && (mode != METIS_MODE_P32_F32 || ((uintptr_t)copy % 16))) return METIS_E_ARG;
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16 && mode != METIS_MODE_P32_F32) return METIS_E_ARG;
    const bool f32in = mode == METIS_MODE_P32_F32;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!x || !codes || !scales || !unit) return METIS_E_ARG;
    if (rows * cols / kBlock >= (int64_t)1 << 31) return METIS_E_ARG;
    if ((ld % (f32in ? 4 : 8)) || ((uintptr_t)x % 16)) return METIS_E_ARG;
    if (((uintptr_t)codes % 8) || ((uintptr_t)scales % 8)) return METIS_E_ARG;
    Workspace ws;
    if (const int rc = carve_workspace(workspace, workspace_bytes, rows, cols, &ws)) return rc;
#define METIS_QH(M, S, W) return launch_quant<M, S, false, W, true>(x, rows, cols, ld, nullptr, seed, offset, codes, scales, unit, ws, st, \
                                                                    f32in, nullptr, sign_mask, nullptr, -1, copy)
    if (mode == METIS_MODE_PB16) { if (sr) METIS_QH(1, true, false); else METIS_QH(1, false, false); }
    if (sr) METIS_QH(0, true, true); else METIS_QH(0, false, true);
#undef METIS_QH
}

// The rotation alone, bf16 or binary32 in and out (same dtype): out = rotate(x) or its inverse, tile by tile.
template <int F32, int INVERSE>
__global__ __launch_bounds__(256) void hadamard16_kernel(const void* __restrict__ xv, void* __restrict__ outv, int64_t ntiles,
                                                         int64_t tiles_per_row, int64_t ldx, int64_t ldo, uint32_t sign_mask)
{
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < ntiles; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / tiles_per_row, cb = i - row * tiles_per_row;
        float v[kBlock];
        if (F32) {
            const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(xv) + row * ldx + cb * kBlock);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float4 f = p[c];
                v[4 * c] = f.x; v[4 * c + 1] = f.y; v[4 * c + 2] = f.z; v[4 * c + 3] = f.w;
            }
        } else {
            const uint4* p = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(xv) + row * ldx + cb * kBlock);
            unpack16(p[0], p[1], v);
        }
        if (INVERSE) hadamard16_inverse(v, sign_mask);
        else hadamard16_forward(v, sign_mask);
        if (F32) {
            float4* o = reinterpret_cast<float4*>(static_cast<float*>(outv) + row * ldo + cb * kBlock);
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
        } else {
            uint32_t w[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) w[j] = bf16_bits(v[2 * j]) | (bf16_bits(v[2 * j + 1]) << 16);
            uint4* o = reinterpret_cast<uint4*>(static_cast<uint16_t*>(outv) + row * ldo + cb * kBlock);
            o[0] = make_uint4(w[0], w[1], w[2], w[3]);
            o[1] = make_uint4(w[4], w[5], w[6], w[7]);
        }
    }
}

int hadamard16(const void* x, int64_t rows, int64_t cols, int64_t ldx, int dtype, int inverse, uint32_t sign_mask, void* out,
               int64_t ldo, hipStream_t st)
{
    if (rows < 0 || cols < 0 || ldx < cols || ldo < cols || sign_mask > 0xffffu) return METIS_E_ARG;
    if (dtype != METIS_DTYPE_BF16 && dtype != METIS_DTYPE_F32) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    const int al = dtype == METIS_DTYPE_F32 ? 4 : 8;
    if (!x || !out || (ldx % al) || (ldo % al) || ((uintptr_t)x % 16) || ((uintptr_t)out % 16)) return METIS_E_ARG;
    const int64_t tpr = cols / kBlock, ntiles = rows * tpr;
    int64_t g = (ntiles + 255) / 256;
    const int64_t cap = (int64_t)device_cus() * 16;
    if (g > cap) g = cap;
#define METIS_H(F, I) hipLaunchKernelGGL((hadamard16_kernel<F, I>), dim3((unsigned)g), dim3(256), 0, st, x, out, ntiles, tpr, ldx, ldo, sign_mask)
    if (dtype == METIS_DTYPE_F32) { if (inverse) METIS_H(1, 1); else METIS_H(1, 0); }
    else { if (inverse) METIS_H(0, 1); else METIS_H(0, 0); }
#undef METIS_H
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

// ---------------------------------------------------------------------------------------------
// Allocation-free variant of the row quantizer: the workspace (per-workgroup maxima, reduction words,
// parked block maxima) is a file-scope device array instead of caller memory, for callers that cannot
// allocate (HIP graph capture, serving loops).  Every device the library runs on holds its own copy of
// the array at its own address until the process ends; the address is looked up once per device, with
// that device current, and host code only ever uses that address, never the array's name.
// ---------------------------------------------------------------------------------------------
constexpr int64_t kStaticMaxElements = (int64_t)1 << 26;         // 64 Mi elements, e.g. [16384, 4096]
constexpr size_t kStaticScratchBytes = kWsGmaxBytes + kWsSyncBytes + (size_t)(kStaticMaxElements / kBlock) * 4;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

static int static_scratch(void** out)
{
    static std::atomic<void*> ptrs[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return METIS_E_DEVICE;
    void* p = ptrs[dev].load(std::memory_order_acquire);
    if (!p) {
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
            (void)hipGetLastError();
            return METIS_E_DEVICE;
        }
        ptrs[dev].store(p, std::memory_order_release);         // two racing first calls store the same address
    }
    *out = p;
    return METIS_OK;
}

int quantize_row_static(const void* x, int64_t rows, int64_t cols, int64_t ld, int mode, void* codes, void* scales,
                        float* unit, hipStream_t st)
{
    if (rows < 0 || cols < 0) return METIS_E_ARG;
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16 && mode != METIS_MODE_P32_F32) return METIS_E_ARG;
    if (rows > 0 && cols > kStaticMaxElements / rows) return METIS_E_TOO_LARGE;
    static_assert(kStaticScratchBytes >= kWsGmaxBytes + kWsSyncBytes + (size_t)(kStaticMaxElements / kBlock) * 4, "scratch too small");
    void* ws = nullptr;
    if (const int rc = static_scratch(&ws)) return rc;
    // the two-launch path: nothing in the scratch has to start at zero (phase 1 rewrites every word phase 2 reads)
    return quantize(x, rows, cols, ld, mode, false, false, nullptr, 0, 0, codes, scales, unit, ws, kStaticScratchBytes, st);
}

int dequantize(const void* codes, const void* scales, const float* unit, int64_t rows, int64_t cols, int mode, void* out,
               int out_dtype, hipStream_t st)
{
    if (rows < 0 || cols < 0) return METIS_E_ARG;
    if (mode == METIS_MODE_P32_F32) mode = METIS_MODE_P32;     // same arithmetic, the packed format does not know its source
    if (mode != METIS_MODE_P32 && mode != METIS_MODE_PB16) return METIS_E_ARG;
    if (out_dtype != METIS_DTYPE_BF16 && out_dtype != METIS_DTYPE_F32) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!codes || !scales || !unit || !out) return METIS_E_ARG;
    if (((uintptr_t)codes % 4) || ((uintptr_t)out % 16)) return METIS_E_ARG;
    const int64_t noct = rows * cols / 8;
    if (noct == 0) return METIS_OK;
    int64_t g = (noct + 255) / 256;
    const int64_t cap = (int64_t)device_cus() * 16;
    if (g > cap) g = cap;
#define METIS_D(M, F) hipLaunchKernelGGL((dequant_kernel<M, F>), dim3((int)g), dim3(256), 0, st, (const uint32_t*)codes, \
                                         (const uint8_t*)scales, unit, out, noct)
    if (mode == 0) { if (out_dtype == METIS_DTYPE_F32) METIS_D(0, 1); else METIS_D(0, 0); }
    else { if (out_dtype == METIS_DTYPE_F32) METIS_D(1, 1); else METIS_D(1, 0); }
#undef METIS_D
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

}  // namespace metis
