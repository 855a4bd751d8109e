// Decode-sized block-scaled GEMM for many column tiles in bf16 arithmetic (32 < M < 256 rows, K % 256 == 0, ready activation operands, cached
// weights in the decode layout): the activation travels once per workgroup through LDS instead of once per column tile through L1.
//
//   out[M,N] = round(round(round(sum_k A[m,k] B[n,k]) + bias[n]) + sum_j T[m,j] U[n,j])        (bf16 roundings of the reference's all-bf16 forward)
//
// Same contraction, order of sums and roundings as skinny_tile<PB16> (metis_gemm.hip), so the same bits, where its workgroups fill the device once.
// A workgroup of twelve waves, one per compute unit, owns up to five tiles of 32 columns and 64 rows.  Two waves per column tile halve K between
// them; two loader waves copy the activation's operands for either half (skinny_operand_kernel: one KiB per row tile and 16 elements of K) by
// direct loads into a ring of two stages of 256 elements of K.  A compute wave streams its weight blocks straight into registers, a step ahead of
// their use.  156 KiB of LDS.
//
// What bounds it: SIMD issue.  16 elements of K of a tile are 18 vector instructions (expansion) and two MFMAs, 60 ns of a SIMD together (they
// overlap only in part: a probe with nothing else takes the same), 2.9 us per step where a SIMD has three compute waves.  skinny_tile reads 543 MB
// of operands through L1 for the 76 MB of weights of 64 x 3584 -> 37888.
// Microseconds in a graph, skinny_tile | this kernel: 64 x 3584 -> 2 x 18944 (r = 64) 35.9 | 30.9, 64 x 3584 -> 32768 31.3 | 25.6, 192 x 3584 -> 37888
// 93.8 | 88.6, 33 x 1024 -> 40960 18.5 | 12.5, 64 x 1024 -> 24608 12.5 | 10.1.  On the way: low-rank operands fetched by the compute waves before the
// first step 2.5 more (their latency ahead of everything), after the last 1.5 more; a fifth tile spread over four waves of its own for even
// SIMDs, other distances of the LDS reads, s_setprio, two steps unrolled: no change.
#include "gemm_common.h"

namespace metis {

constexpr int DW_NT = 5;                                       // column tiles per workgroup
constexpr int DW_WAVES = 2 * DW_NT + 2;
constexpr int DW_HALF = 32 * 1024, DW_STAGE = 2 * DW_HALF;     // bytes of a stage for one half of K, for both
constexpr int DW_LR = 4;                                       // products of 16 low-rank columns whose operands are staged
constexpr int DW_LDS = 2 * DW_STAGE + (DW_NT + 2) * DW_LR * 1024;

// one KiB, 16 bytes from each lane's address, to consecutive bytes of LDS
__device__ __forceinline__ void dw_direct_load(const void* src, uint32_t dst)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(dst) : "memory");
}
// own direct loads landed
__device__ __forceinline__ void dw_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// own LDS reads and writes done, then the workgroup's barrier; global loads in flight stay in flight
__device__ __forceinline__ void dw_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16 products of 16 elements of K each for two row tiles: weights of the run rw, activation operands at sp (KiB m of row tile i at (16 i + m) KiB).
// The operands of product m + 2 are requested and the weights of product m + 1 expanded beside the MFMAs of product m.
__device__ __forceinline__ void dw_products(const RunRegs<4>& rw, const uint8_t* sp, float ub, float16_t (&acc)[2])
{
    constexpr int AHEAD = 2, N = 16, VALU = 18;                // vector instructions of one expansion
    bf16x8_t fa[N][2];
    auto read = [&](int m) {
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[m][i] = *reinterpret_cast<const bf16x8_t*>(sp + (i * 16 + m) * 1024);
    };
#pragma unroll
    for (int m = 0; m < AHEAD; ++m) read(m);
    bf16x8_t fw = run_operand_bf16<4>(rw, 0, ub);
#pragma unroll
    for (int m = 0; m < N; ++m) {
        if (m + AHEAD < N) read(m + AHEAD);
        const bf16x8_t cur = fw;
        if (m + 1 < N) fw = run_operand_bf16<4>(rw, m + 1, ub);
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur, fa[m][i], acc[i], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * AHEAD, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);
#pragma unroll
    for (int m = 0; m < N; ++m) {
        if (m + AHEAD < N) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (m + 1 < N) __builtin_amdgcn_sched_group_barrier(0x002, VALU / 2, 0);
        }
    }
}

// column tile `at` of the group: its matrix, and its first column there
__device__ __forceinline__ SkinnyMember dw_member(const SkinnyGroup& grp, int at, int& n)
{
    SkinnyMember mm = grp.m[0];
    int start = 0;
#pragma unroll
    for (int i = 1; i < kMaxGroupMembers; ++i)
        if (i < grp.count && at >= grp.m[i - 1].tile_end) { mm = grp.m[i]; start = grp.m[i - 1].tile_end; }
    n = (at - start) * 32;
    return mm;
}

template <int OUT_F32>
__global__ __launch_bounds__(64 * DW_WAVES) void gemm_decode_wide_kernel(const uint8_t* a_ops, int M, int K, const SkinnyGroup grp, int tiles,
                                                                         int per_wg)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t dw_lds[];
    const int lane = threadIdx.x & 63, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int m0 = (int)blockIdx.y * 64;
    const int iters = K / 256, mid = 4 * iters / 8;            // steps of 256 elements; eighths of K 0..3 | 4..7
    const int nsteps = iters - mid;                            // of the longer half
    const int h = wave & 1, j = wave >> 1;                     // half of K, column tile (DW_NT: the loaders)
    const int first = h ? mid : 0, hlen = h ? iters - mid : mid;
    const int tile0 = (int)blockIdx.x * per_wg, tile = tile0 + j;
    // The first 64 low-rank columns' operands of the first tile's matrix are staged behind the ring: KiB (j, c) of U, then (i, c) of T.
    uint8_t* lr = dw_lds + 2 * DW_STAGE;
    int n_first;
    const SkinnyMember mm0 = dw_member(grp, tile0, n_first);

    // Every wave passes the same barriers: one per step, two behind the loop.
    if (j == DW_NT) {                                          // ---- loader of half h
        auto issue = [&](int step) {
            if (step >= hlen) return;
            const uint32_t slot = (uint32_t)(uintptr_t)dw_lds + (uint32_t)((step & 1) * DW_STAGE + h * DW_HALF);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint8_t* src = a_ops + (int64_t)((m0 / 32 + i) * iters + first + step) * 16 * 1024 + lane * 16;
#pragma unroll
                for (int k = 0; k < 16; ++k) dw_direct_load(src + k * 1024, slot + (uint32_t)(i * 16 + k) * 1024u);
            }
        };
        issue(0);
        for (int step = 0; step < nsteps; ++step) {
            dw_landed();
            dw_barrier();
            issue(step + 1);                                   // that slot held step - 1, which every wave has left
            if (step != 0) continue;
            for (int c = 2 * h; c < 2 * h + 2 && c * 16 < mm0.r; ++c) {
                const uint32_t dst = (uint32_t)(uintptr_t)lr + (uint32_t)c * 1024u;
                const int jj = c * 16 + hi * 8;
                for (int i = 0; i < 2; ++i)
                    dw_direct_load(mm0.t + (int64_t)min(m0 + i * 32 + (lane & 31), M - 1) * mm0.ldt + jj, dst + (uint32_t)((DW_NT + i) * DW_LR) * 1024u);
                for (int k = 0; k < per_wg && n_first + 32 * k < mm0.N; ++k)
                    dw_direct_load(mm0.u + (int64_t)min(n_first + 32 * k + (lane & 31), mm0.N - 1) * mm0.r + jj, dst + (uint32_t)(k * DW_LR) * 1024u);
            }
        }
        dw_landed();
        dw_barrier();
        dw_barrier();
        return;
    }

    // ---- compute wave: half h of K of column tile j; it finishes row tile h
    const bool live = j < per_wg && tile < tiles;
    int n0;
    const SkinnyMember mm = dw_member(grp, tile, n0);
    const int len = live ? hlen : 0;
    const uint8_t* cp = mm.b_codes + ((int64_t)(n0 / 32) * iters + first) * kDecodeBlock + lane * 16;
    const uint8_t* xp = cp + 4096 - lane * 8;
    const float ub = *mm.b_unit;
    float16_t acc[2], total[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = total[i][e] = 0.0f;
    RunRegs<4> next;
    if (len > 0) load_run_strided<4>(next, cp, 1024, xp);
    for (int step = 0; step < nsteps; ++step) {
        const RunRegs<4> rw = next;
        if (step + 1 < len) load_run_strided<4>(next, cp + (int64_t)(step + 1) * kDecodeBlock, 1024, xp + (int64_t)(step + 1) * kDecodeBlock);
        dw_barrier();
        if (step >= len) continue;
        dw_products(rw, dw_lds + (step & 1) * DW_STAGE + h * DW_HALF + lane * 16, ub, acc);
        const int at = first + step + 1;                       // the end of an eighth of K: its sums join the half's
        bool edge = false;
#pragma unroll
        for (int k = 1; k <= 4; ++k) edge |= at == (4 * h + k) * iters / 8;
        if (edge) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) { total[i][e] += acc[i][e]; acc[i][e] = 0.0f; }
        }
    }
    const int m = m0 + h * 32 + (lane & 31);
    const bool biased = live && mm.bias;
    float bias[16];                                            // on its way during the exchange
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int n = n0 + 8 * (e >> 2) + 4 * hi + (e & 3);
        bias[e] = biased && n < mm.N ? bias_value(mm.bias, mm.bias_f32, n) : 0.0f;
    }
    dw_barrier();                                              // the ring is free
    // the tile's waves hand each other the sums of the row tile that they do not finish (slots of 4 KiB: tile, row tile)
    float* red = reinterpret_cast<float*>(dw_lds) + j * 2 * 16 * 64 + lane;
    if (live) {
#pragma unroll
        for (int e = 0; e < 16; ++e) red[((1 - h) * 16 + e) * 64] = h ? total[0][e] : total[1][e];
    }
    // low-rank products, 32 columns at a time, each slice's sums added to those before it
    float16_t low;
#pragma unroll
    for (int e = 0; e < 16; ++e) low[e] = 0.0f;
    const bool staged = mm.out == mm0.out;
    const int nrow = min(n0 + (lane & 31), mm.N - 1), mrow = min(m, M - 1);
    for (int j0 = 0; j0 < (live ? mm.r : 0); j0 += 32) {
        float16_t p;
#pragma unroll
        for (int e = 0; e < 16; ++e) p[e] = 0.0f;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int jj = j0 + k * 16 + hi * 8, c = j0 / 16 + k;
            bf16x8_t fu, ft;
            if (staged && c < DW_LR) {
                fu = *reinterpret_cast<const bf16x8_t*>(lr + (j * DW_LR + c) * 1024 + lane * 16);
                ft = *reinterpret_cast<const bf16x8_t*>(lr + ((DW_NT + h) * DW_LR + c) * 1024 + lane * 16);
            } else {
                fu = *reinterpret_cast<const bf16x8_t*>(mm.u + (int64_t)nrow * mm.r + jj);
                ft = *reinterpret_cast<const bf16x8_t*>(mm.t + (int64_t)mrow * mm.ldt + jj);
            }
            p = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fu, ft, p, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) low[e] += p[e];
    }
    dw_barrier();
    if (!live || m >= M) return;
    // total[h][e] of lane l: row m = l % 32, column n = 8 (e / 4) + 4 (l / 32) + e % 4
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int n = n0 + 8 * g + 4 * hi;
        if (n >= mm.N) continue;                               // N % 4 == 0 is required
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = 4 * g + k;
            v[k] = rb((h ? total[1][e] : total[0][e]) + red[(h * 16 + e) * 64]);   // the reference's bf16 matmul result, then its bf16 bias add
            if (biased) v[k] = rb(v[k] + bias[e]);
            v[k] += low[e];
            if (OUT_F32) v[k] = rb(v[k]);                      // a binary32 buffer still receives bf16 values
        }
        if (OUT_F32) {
            *reinterpret_cast<float4*>((float*)mm.out + (int64_t)m * mm.N + n) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            uint2 w;
            w.x = rb_pair(v[0], v[1]);
            w.y = rb_pair(v[2], v[3]);
            *reinterpret_cast<uint2*>((uint16_t*)mm.out + (int64_t)m * mm.N + n) = w;
        }
    }
}

// Column tiles per workgroup where the kernel takes a call, 0 where skinny_tile keeps it: more than three tiles per compute unit, so that a
// workgroup's tiles share what the activation's way through LDS costs, and at most five, one round of workgroups per 64 rows.  Beyond 64 rows the
// rounds must also be nine tenths full (255 x 2048 -> 28000, 0.85 full: 58.5 | 62.4).  Microseconds, skinny_tile | this kernel, K = 3584, M = 64 and
// 192: 2 tiles per unit 17.0 | 16.0 and 41.6 | 44.2, 3 23.8 | 22.4 and 63.9 | 64.4, 4 31.3 | 25.6 and 82.9 | 73.3, 4.6 36.0 | 30.9 and
// 93.8 | 88.6, 6 42.8 | 49.5 and 120 | 109; K = 1024, M = 64: 3 11.8 | 10.8, 4 14.0 | 11.3, 6 21.3 | 24.7.  Up to 32 rows an expansion feeds one
// MFMA and the two are even (32 x 3584 -> 37888 24.0 | 24.6).
int decode_wide_tiles(int64_t M, int64_t tiles)
{
    const int64_t cus = device_cus(), rows = (M + 63) / 64;
    if (M <= 32 || cus <= 0 || tiles <= 3 * cus || tiles > DW_NT * cus) return 0;
    const int64_t per_wg = (tiles + cus - 1) / cus, rounds = ((tiles + per_wg - 1) / per_wg * rows + cus - 1) / cus;
    return rows == 1 || 10 * tiles * rows >= 9 * rounds * cus * per_wg ? (int)per_wg : 0;
}

int launch_decode_wide(const void* a_ops, int64_t M, int64_t K, const SkinnyGroup& grp, int tiles, int per_wg, int out_dtype, hipStream_t st)
{
    const dim3 grid((unsigned)((tiles + per_wg - 1) / per_wg), (unsigned)((M + 63) / 64));
    static bool done[2][64];
#define METIS_DW(O) do { if (const int rc = allow_dynamic_lds((const void*)gemm_decode_wide_kernel<O>, DW_LDS, done[O])) return rc; \
    hipLaunchKernelGGL(gemm_decode_wide_kernel<O>, grid, dim3(64 * DW_WAVES), DW_LDS, st, (const uint8_t*)a_ops, (int)M, (int)K, grp, tiles, \
                       per_wg); } while (0)
    if (out_dtype == METIS_DTYPE_F32) METIS_DW(1); else METIS_DW(0);
#undef METIS_DW
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

}  // namespace metis
