// The NVFP4 round trip as VALUES: out = dequantize(quantize(x)), same shape and type as x, with no packed tensor left behind
// (quant_func[...].quantize_dequantize, src/Metis/Metis/quant.py:6-36 / 392-433).
#include "metis_device.h"
#include "metis_host.h"
#include "nvfp4_encode.h"
#include "grid_max.h"

namespace metis {

// ---------------------------------------------------------------------------------------------
// A code depends on its block, the value it stands for also on the tensor maximum.  Between the two nothing has to leave the chip:
//   small tensors: each workgroup folds the maximum of the whole tensor itself, from L2, then takes its own blocks;
//   others, while the codes fit half of the registers: every workgroup reads and encodes its blocks, the maximum is taken over the grid,
//   and the codes are decoded where they are.
// One launch either way (behind one that clears the area of the grid's maximum where the call is captured, ops.py).  (Codes and parked maxima through memory, quantize_dequantize_row, move 5.3 B per bf16 element and 9.5 B per
// binary32 element instead of 4 and 8, and take a second launch.)
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

// the largest |x| of half blocks first, first + step, ... < nhalves, eight loads in flight
template <bool F32>
__device__ __forceinline__ float fold_magnitudes(const uint4* __restrict__ x, uint32_t first, uint32_t step, uint32_t nhalves)
{
    constexpr int AHEAD = F32 ? 4 : 8;
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

// a half block's codes, and the maximum of its block
template <bool F32>
__device__ __forceinline__ uint32_t encode_half(const HalfBlock<F32>& h, float& am)
{
    float v[8];
    unpack_half<F32>(h, v);
    am = amax8(v, 0.0f);
    // the neighbouring lane holds the other half of the block (quad_perm 1,0,3,2)
    am = fmaxf(am, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, am), 0xB1, 0xf, 0xf, false)));
    uint32_t c[1];
    if constexpr (F32) encode_rne_wide_n<8>(v, block_scalar_ieee(am), c);
    else encode_rne_pb16_n<8>(v, block_scalar<1>(am), c);
    return c[0];
}
// the dequantized values of half block i
template <bool F32>
__device__ __forceinline__ void decode_half(uint32_t c, float am, float unit, void* __restrict__ out, uint32_t i)
{
    uint32_t byte;
    if constexpr (F32) byte = e4m3_byte(block_scalar_ieee(am) / unit);
    else byte = scale_byte_of<1>(__float_as_uint(am) >> 16, unit);
    const float dq = rd<(F32 ? 0 : 1)>(e4m3_value(byte) * unit);
    const rt_f32x2_t d0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 0), d1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 1),
                     d2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 2), d3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(c, 1.0f, 3);
    if constexpr (F32) {
        rt_f32x4_t* o = static_cast<rt_f32x4_t*>(out) + 2 * (size_t)i;
        o[0] = (rt_f32x4_t){d0.x * dq, d0.y * dq, d1.x * dq, d1.y * dq};
        o[1] = (rt_f32x4_t){d2.x * dq, d2.y * dq, d3.x * dq, d3.y * dq};
    } else {
        const rt_u32x4_t o = {rb_pair(d0.x * dq, d0.y * dq), rb_pair(d1.x * dq, d1.y * dq), rb_pair(d2.x * dq, d2.y * dq), rb_pair(d3.x * dq, d3.y * dq)};
        __builtin_nontemporal_store(o, static_cast<rt_u32x4_t*>(out) + i);
    }
}
template <bool F32> __device__ __forceinline__ float roundtrip_unit(float amax) { return F32 ? amax_unit_ieee(amax) : tensor_unit_of<1>(amax); }

// the dequantized values of half blocks i, i + step, ...: the next one is requested before the current one is encoded
template <bool F32>
__device__ __forceinline__ void roundtrip_halves(const uint4* __restrict__ x, void* __restrict__ out, uint32_t i, uint32_t step, uint32_t nhalves, float amax)
{
    const float unit = roundtrip_unit<F32>(amax);
    HalfBlock<F32> cur = {};
    if (i < nhalves) cur = load_half<F32>(x, i);
    while (i < nhalves) {
        const uint32_t nxt = i + step;                          // nhalves < 2^31: no wrap
        HalfBlock<F32> ahead = {};
        if (nxt < nhalves) ahead = load_half<F32>(x, nxt);
        float am;
        const uint32_t c = encode_half<F32>(cur, am);
        decode_half<F32>(c, am, unit, out, i);
        cur = ahead; i = nxt;
    }
}

constexpr int kRoundtripSmallThreads = 512;
template <bool F32>
__global__ __launch_bounds__(kRoundtripSmallThreads) void roundtrip_small_kernel(const uint4* __restrict__ x, void* __restrict__ out, uint32_t nhalves)
{
    __shared__ float smax[kRoundtripSmallThreads / 64];
    const float m = wave_max(fold_magnitudes<F32>(x, threadIdx.x, kRoundtripSmallThreads, nhalves));
    if ((threadIdx.x & 63) == 0) smax[threadIdx.x >> 6] = m;
    __syncthreads();
    float amax = smax[0];
#pragma unroll
    for (int w = 1; w < kRoundtripSmallThreads / 64; ++w) amax = fmaxf(amax, smax[w]);
    roundtrip_halves<F32>(x, out, blockIdx.x * kRoundtripSmallThreads + threadIdx.x, gridDim.x * kRoundtripSmallThreads, nhalves, amax);
}

// ---------------------------------------------------------------------------------------------
// A tensor whose codes fit half of the chip's registers: read once and encoded on the way (a half block leaves one word of codes and its
// block's maximum, a third of itself in bf16, a quarter in binary32), the maximum taken over the grid (grid_max.h), then decoded
// and written: 4 or 8 B per element, nothing in between.  HBM-bound, with the wait for the grid's maximum (about 4 us) between the read
// and the write.  Microseconds between events, packed form through memory in two launches | this: bf16 2048 x 4096 24.1 | 13.6, 4096 x 4096
// 25.0 | 20.5, 8192 x 4096 39.2 | 31.4; binary32 3072 x 4096 29.0 | 25.4, 4096 x 4096 34.7 | 30.2.  (x itself kept in registers and
// encoded after the wait: 8192 x 4096 32.0.  x read a second time in a second launch: 35.2.)
//
// The grid is at most HALF of what the device holds (more half blocks to a thread instead).  Workgroups that wait keep their places, so
// a grid that needs every place of the device makes no progress until whatever else runs has left all of it, and several of them in parts
// on the device wait for each other until they give up; then one workgroup writes everything that was left, in milliseconds.  Per call
// beside other work, packed form | half of the device | all of it: bf16 8192 x 4096 beside copies of 2 GiB 80 us | 56 | 881, binary32 4096 x
// 4096 beside exp of 512 Mi elements 65 | 50 | 4850; one call on each of three streams, together 97 | 72 | 7165 and 85 | 70 | 3314.
// Three quarters of the device (bf16 12288 x 4096): three streams 956, packed form 140.  Alone, back to back, all of the device | half:
// bf16 4096 x 4096 17.5 | 18.4, 5120 x 4096 20.6 | 22.2, 8192 x 4096 31.0 | 30.6.  Tensors beyond take the packed form: bf16
// 12288 x 4096 51.4 where all of the device gave 41.6, binary32 8192 x 4096 58.3 where it gave 45.9.
// A workgroup that cannot wait any longer leaves its values to the last one, which reads x again.
// ---------------------------------------------------------------------------------------------
template <bool F32, int NH>
__global__ __launch_bounds__(256, 4) void roundtrip_resident_kernel(const uint4* __restrict__ x, void* __restrict__ out, uint32_t nhalves,
                                                                    uint32_t* __restrict__ sync, uint32_t spin_limit)
{
    using Word = ResultWord<F32>;
    __shared__ GridMaxState sh;
    const uint64_t tag = grid_max_begin(sync);
    const uint32_t step = gridDim.x * 256u, first = blockIdx.x * 256u + threadIdx.x;
    constexpr int AHEAD = F32 ? 2 : 4;                             // half blocks in flight
    uint32_t c[NH], am[F32 ? NH : NH / 2];                         // (bf16: two maxima to a register)
    auto maximum = [&](int k) { return __uint_as_float(F32 ? am[k] : (k & 1) ? am[k / 2] & 0xffff0000u : am[k / 2] << 16); };
    HalfBlock<F32> ring[AHEAD];
    auto request = [&](int k) {
        const uint32_t i = first + k * step;
        ring[k % AHEAD] = {};
        if (i < nhalves) ring[k % AHEAD] = load_half<F32>(x, i);
    };
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) request(k);
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < NH; ++k) {
        float a;
        c[k] = encode_half<F32>(ring[k % AHEAD], a);
        m = fmaxf(m, a);
        if constexpr (F32) am[k] = __float_as_uint(a);
        else if (k & 1) am[k / 2] |= __float_as_uint(a);           // (a bf16 value: its low half is zero)
        else am[k / 2] = __float_as_uint(a) >> 16;
        if (k + AHEAD < NH) request(k + AHEAD);
        __builtin_amdgcn_sched_barrier(0);                         // loads stay where they are issued
    }
    grid_max_arrive(m, sync, sh);
    __syncthreads();                                               // thread 0 is through the tree: sh.last, sh.result
    const uint32_t j = blockIdx.x % kGroups;
    bool somebody_left = false;
    const bool last = sh.last != 0u;
    if (last) {
        const uint32_t ngroups = gridDim.x < kGroups ? gridDim.x : kGroups;
        if (threadIdx.x < ngroups) somebody_left = Word::has_marker(METIS_AT_XCHG(Word::slot(sync, threadIdx.x), Word::result(tag, sh.result)), tag);
        if (threadIdx.x == 0) sh.nleft = 0u;
    } else {
        if (threadIdx.x < 64) {
            uint64_t w = 0;
            uint32_t polls = 0;
            bool have = false;
            for (;;) {
                w = METIS_AT_LOAD(Word::slot(sync, j));
                have = Word::has_result(w, tag);
                if (have || ++polls > spin_limit) break;
                __builtin_amdgcn_s_sleep(2);
            }
            if (threadIdx.x == 0) {
                if (!have) {                                       // leave, unless the result is there by now
                    METIS_AT_STORE(sync_left_flag(sync, blockIdx.x), (uint32_t)tag);
                    __threadfence();                               // the flag is out before the marker can be seen
                    w = METIS_AT_LOAD(Word::slot(sync, j));
                    for (;;) {
                        have = Word::has_result(w, tag);
                        if (have || Word::has_marker(w, tag) || METIS_AT_CAS(Word::slot(sync, j), &w, Word::marker(tag))) break;
                    }
                }
                sh.known = have ? 1u : 0u;
                sh.result = Word::value(w);
            }
        }
        __syncthreads();
        if (!sh.known) return;                                     // the last workgroup writes this workgroup's values
    }
    const float unit = roundtrip_unit<F32>(sh.result);
#pragma unroll
    for (int k = 0; k < NH; ++k) {
        const uint32_t i = first + k * step;
        if (i < nhalves) decode_half<F32>(c[k], maximum(k), unit, out, i);
    }
    if (!last) return;
    if (__syncthreads_or(somebody_left)) {
        __threadfence();                                           // their flags were out before their markers
        for (uint32_t slab = 0; slab < gridDim.x; slab += 256u) {
            const uint32_t b = slab + threadIdx.x;
            if (b < gridDim.x && METIS_AT_LOAD(sync_left_flag(sync, b)) == (uint32_t)tag) sh.left[atomicAdd(&sh.nleft, 1u)] = b;
            __syncthreads();
            const uint32_t nd = sh.nleft;
            for (uint32_t d = 0; d < nd; ++d) {
#pragma unroll 1
                for (int k = 0; k < NH; ++k) {
                    const uint32_t i = sh.left[d] * 256u + threadIdx.x + k * step;
                    if (i < nhalves) {
                        float a;
                        const uint32_t w = encode_half<F32>(load_half<F32>(x, i), a);
                        decode_half<F32>(w, a, unit, out, i);
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

// Workgroups of the resident kernel that the current device holds at once (0: unknown)
template <bool F32, int NH>
static int resident_capacity()
{
    static int cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    if (cached[dev] == 0) {
        int per_cu = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, roundtrip_resident_kernel<F32, NH>, 256, 0);
        cached[dev] = (e != hipSuccess || per_cu <= 0) ? -1 : per_cu * device_cus();
    }
    return cached[dev] < 0 ? 0 : (cached[dev] > kFusedMaxGrid ? kFusedMaxGrid : cached[dev]);
}
template <bool F32, int NH>
static int64_t resident_grid(uint32_t nhalves) { return ((int64_t)nhalves + 256 * NH - 1) / (256 * NH); }
template <bool F32, int NH>
static bool resident_fits(uint32_t nhalves) { return resident_grid<F32, NH>(nhalves) <= resident_capacity<F32, NH>() / 2; }   // (why half: beside the kernel)

// half blocks per thread of the widest grid that fits, 0: none does
template <bool F32>
static int resident_halves(uint32_t nhalves)
{
    return resident_fits<F32, 4>(nhalves) ? 4 : resident_fits<F32, 8>(nhalves) ? 8 : resident_fits<F32, 16>(nhalves) ? 16 : 0;
}

template <bool F32>
static void launch_resident(int nh, const uint4* x, void* out, uint32_t nhalves, uint32_t* sync, uint32_t spin_limit, hipStream_t st)
{
#define METIS_RT(NH) hipLaunchKernelGGL((roundtrip_resident_kernel<F32, NH>), dim3((unsigned)resident_grid<F32, NH>(nhalves)), dim3(256), 0, st, x, out, \
                                        nhalves, sync, spin_limit)
    if (nh == 4) METIS_RT(4); else if (nh == 8) METIS_RT(8); else METIS_RT(16);
#undef METIS_RT
}

// The whole-tensor fold while it costs no more than taking the maximum over the grid: up to 256 Ki elements in bf16, 144 Ki in binary32,
// twice the bytes to fold.  Device time, fold | grid: bf16 128 x 1024 4.6 | 6.6 us, 192 x 1024 5.6 | 6.6, 256 x 1024 6.55 | 6.65, 272 x 1024
// 7.1 | 6.9, 320 x 1024 7.6 | 6.7; binary32 77 x 1536 5.8 | 6.6, 128 x 1024 6.2 | 6.7, 144 x 1024 6.6 | 6.9, 152 x 1024 7.0 | 6.8, 192 x 1024
// 8.0 | 6.8.
static bool small_tensor(int64_t nhalves, bool f32) { return nhalves <= (f32 ? 18432 : 32768); }

// What a call of these sizes takes: half blocks per thread of the resident kernel in *nh (0: the fold), or why it is refused.
static int roundtrip_form(int64_t rows, int64_t cols, int mode, int* nh)
{
    *nh = 0;
    if (rows < 0 || cols < 0) return METIS_E_ARG;
    if (mode != METIS_MODE_PB16 && mode != METIS_MODE_P32_F32) return METIS_E_ARG;
    if (cols % kBlock) return METIS_E_SHAPE;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (rows > ((int64_t)1 << 31) / cols) return METIS_E_TOO_LARGE;
    const uint32_t nhalves = (uint32_t)(rows * cols / 8);
    const bool f32 = mode == METIS_MODE_P32_F32;
    if (small_tensor(nhalves, f32)) return METIS_OK;
    *nh = f32 ? resident_halves<true>(nhalves) : resident_halves<false>(nhalves);
    return *nh ? METIS_OK : METIS_E_TOO_LARGE;
}

int roundtrip_applies(int64_t rows, int64_t cols, int mode, size_t* bytes)
{
    int nh;
    const int rc = roundtrip_form(rows, cols, mode, &nh);
    if (bytes) *bytes = nh ? workspace_bytes(1, kBlock) : 0;
    return rc;
}

int roundtrip(const void* x, int64_t rows, int64_t cols, int mode, void* out, void* workspace, size_t bytes, uint32_t spin_limit, hipStream_t st)
{
    int nh;
    if (const int rc = roundtrip_form(rows, cols, mode, &nh)) return rc;
    if (rows == 0 || cols == 0) return METIS_OK;
    if (!x || !out || ((uintptr_t)x % 16) || ((uintptr_t)out % 16)) return METIS_E_ARG;
    const uint32_t nhalves = (uint32_t)(rows * cols / 8);
    const bool f32 = mode == METIS_MODE_P32_F32;
    const uint4* xv = static_cast<const uint4*>(x);
    if (nh == 0) {
        const unsigned g = (nhalves + kRoundtripSmallThreads - 1) / kRoundtripSmallThreads;
        if (f32) hipLaunchKernelGGL(roundtrip_small_kernel<true>, dim3(g), dim3(kRoundtripSmallThreads), 0, st, xv, out, nhalves);
        else hipLaunchKernelGGL(roundtrip_small_kernel<false>, dim3(g), dim3(kRoundtripSmallThreads), 0, st, xv, out, nhalves);
        return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
    }
    Workspace ws;
    if (const int rc = carve_workspace(workspace, bytes, 1, kBlock, &ws)) return rc;
    if (spin_limit == 0) spin_limit = kSpinLimit;
    if (f32) launch_resident<true>(nh, xv, out, nhalves, ws.sync, spin_limit, st);
    else launch_resident<false>(nh, xv, out, nhalves, ws.sync, spin_limit, st);
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

}  // namespace metis
