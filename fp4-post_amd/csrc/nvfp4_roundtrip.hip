// The NVFP4 round trip as VALUES: out = dequantize(quantize(x)), same shape and type as x, with no packed tensor left behind
// (quant_func[...].quantize_dequantize, src/Metis/Metis/quant.py:6-36 / 392-433).
#include "metis_device.h"
#include "metis_host.h"
#include "nvfp4_encode.h"
#include <type_traits>

namespace metis {

// ---------------------------------------------------------------------------------------------
// A code depends on its block, the value it stands for also on the tensor maximum, so x is seen twice.  quantize_dequantize_row
// (nvfp4_quant.hip) writes codes and parked maxima in between; here nothing is written but the result:
//   pass 1: one partial maximum per workgroup, nothing but a read of x
//   pass 2: unit from the partial maxima; every half block (one lane) from x to its dequantized values in registers
// HBM-bound, 6 B (bf16) or 12 B (binary32) per element against 5.3 and 9.5 with the packed form in between, but with a first pass
// that neither encodes nor stores.  Microseconds, packed form | this: bf16 1024 x 4096 11.0 | 7.9, 4096 x 4096 22.0 | 17.7,
// 8192 x 4096 36.2 | 35.2 (35.8 | 36.5 where the input changes from call to call), 12288 x 4096 50.5 | 50.7; binary32 1024 x 4096 13.9 | 11.2, 2048 x 4096 20.4 | 18.3, 3072 x 4096 25.8 |
// 27.2, 8192 x 4096 56 | 63.6: the caller keeps the packed form for the largest tensors (ops.roundtrip_pays).
// A small tensor takes ONE launch: each workgroup folds the maximum of the whole tensor itself, from L2.
// The values are those of quantize + dequantize bit for bit: the same maxima, the same encoders, the same products.
// ---------------------------------------------------------------------------------------------
typedef uint32_t rt_u32x4_t __attribute__((ext_vector_type(4)));
typedef float rt_f32x2_t __attribute__((ext_vector_type(2)));
typedef float rt_f32x4_t __attribute__((ext_vector_type(4)));

// half a block: 8 bf16 values (one 16-byte load) or 8 binary32 values (two)
template <bool F32> struct HalfBlock { uint4 w[F32 ? 2 : 1]; };
template <bool F32> __device__ __forceinline__ HalfBlock<F32> load_half(const uint4* __restrict__ x, uint32_t i)
{
    HalfBlock<F32> h;
#pragma unroll
    for (int k = 0; k < (F32 ? 2 : 1); ++k) h.w[k] = x[(size_t)i * (F32 ? 2 : 1) + k];
    return h;
}
template <bool F32> __device__ __forceinline__ void unpack_half(const HalfBlock<F32>& h, float (&v)[8])
{
    if constexpr (F32) {
        const uint32_t w[8] = {h.w[0].x, h.w[0].y, h.w[0].z, h.w[0].w, h.w[1].x, h.w[1].y, h.w[1].z, h.w[1].w};
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = __uint_as_float(w[j]);
    } else {
        const uint32_t w[4] = {h.w[0].x, h.w[0].y, h.w[0].z, h.w[0].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) { v[2 * j] = bf16_lo(w[j]); v[2 * j + 1] = bf16_hi(w[j]); }
    }
}
__device__ __forceinline__ float amax8(const float (&v)[8], float m)
{
#pragma unroll
    for (int j = 0; j < 8; j += 2) m = amax3(m, v[j], v[j + 1]);
    return m;
}

// the largest |x| of half blocks first, first + step, ... < nhalves, four of them in flight
template <bool F32, int AHEAD>
__device__ __forceinline__ float fold_magnitudes(const uint4* __restrict__ x, uint32_t first, uint32_t step, uint32_t nhalves)
{
    float m = 0.0f, v[8];
    uint64_t i = first;
    for (; i + (uint64_t)(AHEAD - 1) * step < nhalves; i += (uint64_t)AHEAD * step) {
        HalfBlock<F32> h[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) h[k] = load_half<F32>(x, (uint32_t)(i + (uint64_t)k * step));
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) { unpack_half<F32>(h[k], v); m = amax8(v, m); }
    }
    for (; i < nhalves; i += step) { unpack_half<F32>(load_half<F32>(x, (uint32_t)i), v); m = amax8(v, m); }
    return m;
}

template <bool F32>
__global__ __launch_bounds__(256) void tensor_amax_kernel(const uint4* __restrict__ x, uint32_t nhalves, uint32_t* __restrict__ partial)
{
    publish_group_max(fold_magnitudes<F32, F32 ? 2 : 4>(x, blockIdx.x * 256u + threadIdx.x, gridDim.x * 256u, nhalves), partial);
}

// the dequantized values of half blocks i, i + step, ...: the next one is requested before the current one is encoded
template <int MODE, bool F32>
__device__ __forceinline__ void roundtrip_halves(const uint4* __restrict__ x, void* __restrict__ out, uint32_t i, uint32_t step, uint32_t nhalves, float amax)
{
    float unit;
    if constexpr (F32) unit = amax_unit_ieee(amax);
    else unit = tensor_unit_of<MODE>(amax);
    HalfBlock<F32> cur = {};
    if (i < nhalves) cur = load_half<F32>(x, i);
    while (i < nhalves) {
        const uint32_t nxt = i + step;                          // nhalves < 2^31: no wrap
        HalfBlock<F32> ahead = {};
        if (nxt < nhalves) ahead = load_half<F32>(x, nxt);
        float v[8];
        unpack_half<F32>(cur, v);
        float am = amax8(v, 0.0f);
        // the neighbouring lane holds the other half of the block (quad_perm 1,0,3,2)
        am = fmaxf(am, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, am), 0xB1, 0xf, 0xf, false)));
        uint32_t c[1], byte;
        if constexpr (F32) {
            const float s = block_scalar_ieee(am);
            encode_rne_wide_n<8>(v, s, c);
            byte = e4m3_byte(s / unit);
        } else {
            encode_rne_pb16_n<8>(v, block_scalar<1>(am), c);
            byte = scale_byte_of<1>(__float_as_uint(am) >> 16, unit);
        }
        const float dq = rd<MODE>(e4m3_value(byte) * unit);
        const rt_f32x2_t d0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[0], 1.0f, 0), d1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[0], 1.0f, 1),
                         d2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[0], 1.0f, 2), d3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c[0], 1.0f, 3);
        if constexpr (F32) {
            rt_f32x4_t* o = static_cast<rt_f32x4_t*>(out) + 2 * (size_t)i;
            o[0] = (rt_f32x4_t){d0.x * dq, d0.y * dq, d1.x * dq, d1.y * dq};
            o[1] = (rt_f32x4_t){d2.x * dq, d2.y * dq, d3.x * dq, d3.y * dq};
        } else {
            const rt_u32x4_t o = {rb_pair(d0.x * dq, d0.y * dq), rb_pair(d1.x * dq, d1.y * dq), rb_pair(d2.x * dq, d2.y * dq), rb_pair(d3.x * dq, d3.y * dq)};
            __builtin_nontemporal_store(o, static_cast<rt_u32x4_t*>(out) + i);
        }
        cur = ahead; i = nxt;
    }
}

template <int MODE, bool F32>
__global__ __launch_bounds__(256) void roundtrip_kernel(const uint4* __restrict__ x, void* __restrict__ out, uint32_t nhalves,
                                                        const uint32_t* __restrict__ partial, uint32_t npartial)
{
    __shared__ float smax[4];
    float m = 0.0f;
    for (uint32_t g = threadIdx.x; g < npartial; g += 256u) m = fmaxf(m, __uint_as_float(partial[g]));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) smax[threadIdx.x >> 6] = m;
    __syncthreads();
    roundtrip_halves<MODE, F32>(x, out, blockIdx.x * 256u + threadIdx.x, gridDim.x * 256u, nhalves,
                                fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3])));
}

constexpr int kRoundtripSmallThreads = 512;
template <int MODE, bool F32>
__global__ __launch_bounds__(kRoundtripSmallThreads) void roundtrip_small_kernel(const uint4* __restrict__ x, void* __restrict__ out, uint32_t nhalves)
{
    __shared__ float smax[kRoundtripSmallThreads / 64];
    const float m = wave_max(fold_magnitudes<F32, F32 ? 4 : 8>(x, threadIdx.x, kRoundtripSmallThreads, nhalves));
    if ((threadIdx.x & 63) == 0) smax[threadIdx.x >> 6] = m;
    __syncthreads();
    float amax = smax[0];
#pragma unroll
    for (int w = 1; w < kRoundtripSmallThreads / 64; ++w) amax = fmaxf(amax, smax[w]);
    roundtrip_halves<MODE, F32>(x, out, blockIdx.x * kRoundtripSmallThreads + threadIdx.x, gridDim.x * kRoundtripSmallThreads, nhalves, amax);
}

// One launch while every workgroup's own read of the whole tensor costs no more than the second launch would: device time, one |
// two launches: bf16 64 x 1024 3.6 | 5.4 us, 77 x 1536 4.8 | 5.4, 192 x 1024 5.6 | 5.5; binary32 (twice the bytes) 64 x 1024 4.5 |
// 5.3, 77 x 1536 5.9 | 5.4, 128 x 1024 6.2 | 5.4, 192 x 1024 8.1 | 5.5.  The second launch also costs the host 4 us (6.7 | 11.5 us
// per eager call), which is what such a call is bound by: the line lies a little beyond equal device time.
static bool one_launch(int64_t nhalves, bool f32) { return nhalves <= (f32 ? 16384 : 24576); }
constexpr int kRoundtripPartials = 2048;
size_t roundtrip_workspace_bytes(int64_t rows, int64_t cols, int mode)
{
    if (rows <= 0 || cols <= 0 || one_launch(rows * cols / 8, mode == METIS_MODE_P32_F32)) return 0;
    return kRoundtripPartials * sizeof(uint32_t);
}

int roundtrip(const void* x, int64_t rows, int64_t cols, int mode, void* out, void* workspace, size_t bytes, hipStream_t st)
{
    if (rows < 0 || cols < 0) return METIS_E_ARG;
    if (mode != METIS_MODE_PB16 && mode != METIS_MODE_P32_F32) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!x || !out || ((uintptr_t)x % 16) || ((uintptr_t)out % 16)) return METIS_E_ARG;
    if (rows > (((int64_t)1 << 34) - 1) / cols) return METIS_E_ARG;      // half blocks are counted in 31 bits
    const uint32_t nhalves = (uint32_t)(rows * cols / 8);
    const bool f32 = mode == METIS_MODE_P32_F32;
    const uint4* xv = static_cast<const uint4*>(x);
    if (one_launch(nhalves, f32)) {
        const unsigned g = (nhalves + kRoundtripSmallThreads - 1) / kRoundtripSmallThreads;
        if (f32) hipLaunchKernelGGL((roundtrip_small_kernel<0, true>), dim3(g), dim3(kRoundtripSmallThreads), 0, st, xv, out, nhalves);
        else hipLaunchKernelGGL((roundtrip_small_kernel<1, false>), dim3(g), dim3(kRoundtripSmallThreads), 0, st, xv, out, nhalves);
        return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
    }
    if (!workspace || ((uintptr_t)workspace % 16) || bytes < roundtrip_workspace_bytes(rows, cols, mode)) return METIS_E_WORKSPACE;
    uint32_t* partial = static_cast<uint32_t*>(workspace);
    auto grid = [&](int per_thread) {                           // eight workgroups per compute unit are resident
        int64_t g = ((int64_t)nhalves + 256 * per_thread - 1) / (256 * per_thread);
        const int64_t cap = (int64_t)device_cus() * 8;
        if (g > cap) g = cap;
        return (unsigned)(g > kRoundtripPartials ? kRoundtripPartials : g);
    };
    const unsigned g1 = grid(f32 ? 2 : 4), g2 = grid(2);
    if (f32) {
        hipLaunchKernelGGL(tensor_amax_kernel<true>, dim3(g1), dim3(256), 0, st, xv, nhalves, partial);
        hipLaunchKernelGGL((roundtrip_kernel<0, true>), dim3(g2), dim3(256), 0, st, xv, out, nhalves, partial, g1);
    } else {
        hipLaunchKernelGGL(tensor_amax_kernel<false>, dim3(g1), dim3(256), 0, st, xv, nhalves, partial);
        hipLaunchKernelGGL((roundtrip_kernel<1, false>), dim3(g2), dim3(256), 0, st, xv, out, nhalves, partial, g1);
    }
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

}  // namespace metis
