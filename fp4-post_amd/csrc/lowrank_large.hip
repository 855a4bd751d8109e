// Rank-r products of the low-rank branch at training / prefill sizes (256 rows and more), bf16 operands, binary32
// accumulation on MFMA.  Both are bound by one pass over the tall operand in HBM.
//
//   lowrank_nt:  xv[M, R] = x[M, K] . v[R, K]^T,  t = bf16(xv * s)      `vlinear(x)` and `torch.mul(self.s, y)` of
//                BitLinear.forward with V in bf16 (src/Metis/Metis/bitlinear.py:752-756);
//                with v = U^T also dY . U of the backward pass
//   lowrank_tn:  out[C, R] = sum_l a[l, C] . b[l, R]                     the two products of the backward pass that
//                contract over tokens: dY^T . (xv * s) -> grad of U, x^T . g_xv -> grad of V (written transposed)
//
// lowrank_nt: a workgroup owns 32 rows of x and walks K in stages of 64 or 128.  The x rows and the R rows of v of a stage (v
// from L2 after the first workgroup touched it) go straight from memory to LDS, into a ring of two to four stages, so that no
// wave waits for the loads it issued last; the waves share a stage's quarters of 64 k and the column tiles.  (Staged through
// registers two steps ahead, with two barriers per step and the encoder between them, the loads in flight per compute unit were
// what its registers held: 16384 x 3584, R = 64 25.7 -> 23.4 us, 8192 x 4096 22.2 -> 15.9; with the quantizer 40.9 -> 32.4 and
// 27.9 -> 26.4, 4096 x 8960 31.2 -> 26.6.  The read of x alone at 5 TB/s: 23.5 and 13.4 from HBM; with codes and maxima written 30.8
// and 17.6.)  Bound by memory; with a wide V by what a compute unit takes in, about 46 bytes a nanosecond, of which x is one part in
// 1 + R / 32.  Where several workgroups would share a compute unit, one therefore owns two row tiles and fetches v once for both:
// 16384 x 18944, R = 64, with the quantizer 248 -> 205 us, 16384 x 3584, R = 192 53 -> 48.5, from flushed caches 89 -> 74.  The order
// of an element's sums depends on its row tile, so the two are chosen among those that start at the same step of K (nt_pair).
//
// lowrank_tn: the contraction runs down the rows of both operands, so each has to be turned: a workgroup owns 64
// columns of a and one slice of the tokens; a step of 64 tokens is loaded row by row (coalesced) and staged in LDS as it
// is; the MFMA fragments (8 consecutive tokens of one column) are read with the transposing LDS read of gfx950.  Token
// slices give every compute unit work; their binary32 partial results go to a caller workspace and a second kernel adds
// them in slice order.
#include "metis_device.h"
#include "metis_host.h"
#include "nvfp4_encode.h"
#include "gemm_common.h"
#include "lowrank_small_steps.h"

namespace metis {

constexpr int NT_ROWS = 32;                      // rows of a row tile of x
// A form of the kernel: TILES row tiles per workgroup, KS k per stage, NS stages in the ring; one thread per block of 16 of x.
template <int TILES, int RT, int KS, int NS> struct NtForm {
    static constexpr int kRows = TILES * NT_ROWS, kThreads = kRows * KS / 16, kWaves = kThreads / 64;
    static constexpr int kRowBytes = KS * 2, kRowsPerPiece = 1024 / kRowBytes, kChunks = kRowBytes / 16;
    static constexpr int kStage = (kRows + RT * 32) * kRowBytes;              // bytes of a stage: x rows, then v rows
    static constexpr int kLoads = kStage / 1024 / kWaves, kXLoads = kRows / kRowsPerPiece / kWaves;   // 1 KiB loads per wave and stage; those of x
    // K is walked in steps of 256, whose quarters of 64 have sums of their own: the waves share the quarters of a stage and the
    // column tiles; a step is kStages stages, with a set of sums for each.
    static constexpr int kQuarters = KS / 64, kStages = 4 / kQuarters;
    static constexpr int kColGroups = kWaves / kQuarters / TILES, kColTiles = (RT + kColGroups - 1) / kColGroups;
    static constexpr int kRed = kStages * (kQuarters - 1) * TILES * RT * 4096 + 64;   // partial sums of the waves, then their maxima
    static constexpr int kLds = NS * kStage > kRed ? NS * kStage : kRed;
    static_assert((KS == 64 || KS == 128) && kColGroups * kQuarters * TILES == kWaves && kStage % (1024 * kWaves) == 0 && kXLoads >= 1,
                  "every wave loads whole pieces and multiplies a quarter");
};
// The factors of up to four projections of the same x, their columns side by side in xv and t: a group's members hand in
// their own V and s (stacked copies would have to be made anew whenever one of them changes).
struct NtFactors {
    const uint16_t* v[kTiledMembers];
    const uint16_t* s[kTiledMembers];
    int end[kTiledMembers];                                    // columns up to and with this member; a multiple of 32
};
__device__ __forceinline__ int nt_member(const NtFactors& f, int col)
{
    int i = 0;
#pragma unroll
    for (int q = 0; q + 1 < kTiledMembers; ++q) i += col >= f.end[q];
    return i;
}
__device__ __forceinline__ const uint16_t* nt_pick(const uint16_t* const (&p)[kTiledMembers], int i)
{
    return i == 0 ? p[0] : i == 1 ? p[1] : i == 2 ? p[2] : p[3];
}
// s of column col
__device__ __forceinline__ const uint16_t* nt_s(const NtFactors& f, int col)
{
    const int i = nt_member(f, col);
    return nt_pick(f.s, i) + (col - (i == 0 ? 0 : i == 1 ? f.end[0] : i == 2 ? f.end[1] : f.end[2]));
}
__device__ __forceinline__ const uint16_t* nt_v(const NtFactors& f, int col, int64_t K)
{
    const int i = nt_member(f, col);
    return nt_pick(f.v, i) + (col - (i == 0 ? 0 : i == 1 ? f.end[0] : i == 2 ? f.end[1] : f.end[2])) * K;
}
// The step of its K range that row tile b starts at, of `steps`.
constexpr int NT_ROTATE = 5;
__device__ __forceinline__ int nt_first_step(int b, int steps) { return (int)((unsigned)b * NT_ROTATE % (unsigned)steps); }
// The row tiles at the places `at` and `at + 1` of all `tiles`, ordered by the step that they start at; that step of the first, and
// how many steps later the second starts: none within a class, between neighbouring classes one, or five where 5 divides `steps` (up to five where
// some classes are empty).  An odd one out is returned twice.
// Tiles b and b + p start alike, with p = steps or, if 5 divides it, steps / 5; tiles = a p + e: the p classes have a members, the
// first e of them one more.  Class c = i / 5 (mod p; or i itself) is the i-th in the order; a lane looks at one class.
__device__ __forceinline__ void nt_pair(int at, int tiles, int steps, int* tile0, int* tile1, int* rot, int* lag)
{
    *tile0 = *tile1 = at;
    if (steps <= 0) { if (at + 1 < tiles) *tile1 = at + 1; return; }
    const bool fives = steps % NT_ROTATE == 0;
    const int p = fives ? steps / NT_ROTATE : steps, a = tiles / p, e = tiles % p, lane = threadIdx.x & 63;
    const int inverse[NT_ROTATE] = {0, 4, 2, 3, 1};             // times p, plus 1: a multiple of 5
    const unsigned fifth = fives ? 1u : (unsigned)(inverse[p % NT_ROTATE] * p + 1) / NT_ROTATE;
    int larger = 0, found = 0;
    for (int i0 = 0; i0 < p && found < 2; i0 += 64) {
        const int i = i0 + lane, c = (int)((unsigned)i * fifth % (unsigned)p);
        const unsigned long long more = __ballot(i < p && c < e);
        const int begin = i * a + larger + __popcll(more & ((1ull << lane) - 1)), end = begin + a + (int)((more >> lane) & 1);
        larger += __popcll(more);
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const unsigned long long hit = __ballot(i < p && at + w >= begin && at + w < end);
            if (!hit) continue;
            const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)hit) - 1);
            const int t = __builtin_amdgcn_readlane(c, l) + p * (at + w - __builtin_amdgcn_readlane(begin, l));
            const int r = fives ? (i0 + l) * NT_ROTATE : i0 + l;
            if (w == 0) { *tile0 = *tile1 = t; *rot = r; }
            else { *tile1 = t; *lag = r - *rot; }
            ++found;
        }
    }
}
// Leaves at most VM of the wave's vector memory operations in flight.  Assembly with a memory clobber: no load or store of
// the loop may move across it, the counts at its uses rely on that.
template <int VM> __device__ __forceinline__ void nt_wait()
{
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(VM) : "memory");
}

// K slices: a tensor of a few thousand rows has too few row tiles to keep every compute unit's loads in flight.  gridDim.y
// workgroups then share a row tile, each walking its own range of stages; their binary32 partial sums go to a caller
// workspace ([slice][row][R]) and lowrank_nt_finish_kernel adds them in slice order.  One slice: written directly.
//
// QMODE >= 0: the same pass also quantizes x (round to nearest, rows; METIS_MODE_P32 or _PB16 arithmetic): a stage holds one
// block of 16 per thread, read back from LDS -- E2M1 codes, the block maximum parked as bf16, one partial tensor maximum per
// workgroup: what quant_codes_contig_kernel leaves for a consumer that forms the scale bytes itself.
// Every form adds an element's products in the same order -- the four quarters of each step of 256 k in sums of their own, the
// steps from the row tile's own first one on, the quarters' sums at the end, in order -- so that a column of v gives the same
// bits alone and beside any others, with and without the quantizer.
// TAIL: K % 256 != 0.
template <int TILES, int RT, int QMODE, int KS, int NS, bool TAIL>
__global__ __launch_bounds__(TILES * NT_ROWS * KS / 16) void lowrank_nt_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const NtFactors fac, uint16_t* __restrict__ xv, uint16_t* __restrict__ t, int M, int K, float* __restrict__ part, uint2* __restrict__ codes,
    uint16_t* __restrict__ q_amax, uint32_t* __restrict__ q_gmax, uint32_t fill_to, int R)
{
    using F = NtForm<TILES, RT, KS, NS>;
    const int col0 = QMODE < 0 ? (int)blockIdx.z * RT * 32 : 0; // R: all columns; the workgroup's are RT * 32 of them from here on
    constexpr int STAGE = F::kStage, LPW = F::kLoads, XL = F::kXLoads, RPP = F::kRowsPerPiece, RB = F::kRowBytes;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];     // the ring, then the waves' partial sums
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // TAIL (K % 64 == 0): the last step is cut.  A stage that begins past the end fetches the step's first again, the lanes of a
    // half that does its other half; the quarters past the end multiply zeros, and the threads of such blocks encode the ones that
    // were fetched once more (the same bytes).
    // A template parameter: the branch would keep product and encoder from being interleaved (8192 x 4096: 27.4 -> 35.6 us).
    constexpr int NH = F::kStages;
    const int steps_all = (K + 255) / 256;
    const int per = (steps_all + (int)gridDim.y - 1) / (int)gridDim.y;
    const int first = (int)blockIdx.y * per, wide_steps = max(0, min(steps_all, first + per) - first);
    // Every row tile starts at a different step of its K range and wraps around: at any moment the workgroups then read
    // different column stripes of x instead of the same one.  With rows a multiple of 4 KiB long, pieces at the same offset
    // of every row can fall on the same few memory channels.  The binary32 sums of a tile are therefore added in an order
    // that depends on the tile, the same for every call.  (An offset of 5 steps per tile: 8192 x 4096 from flushed caches 31 us,
    // 39 without; other row lengths within 2 %.)
    // Two row tiles: they share the walk and the pieces of v, and each keeps its own order.  nt_pair picks tiles that start at the
    // same step or `lag` (at most five) steps apart; the second then joins that much after the first and goes on as long after it.
    int tile0 = (int)blockIdx.x, tile1 = (int)blockIdx.x, rot = 0, lag = 0;
    if constexpr (TILES == 2) nt_pair(2 * (int)blockIdx.x, (M + NT_ROWS - 1) / NT_ROWS, wide_steps, &tile0, &tile1, &rot, &lag);
    else rot = wide_steps > 0 ? nt_first_step(tile0, wide_steps) : 0;
    const int steps = (wide_steps + lag) * NH;                  // stages
    auto kof = [&](int st) {
        int q = st / NH + rot;
        if (q >= wide_steps) q -= wide_steps;
        if (TILES == 2 && q >= wide_steps) q -= wide_steps;
        return (first + q) * 256 + st % NH * KS;
    };
    // row r of the workgroup's
    auto row_of = [&](int r) { return TILES == 2 ? (r < NT_ROWS ? tile0 * NT_ROWS : (tile1 - 1) * NT_ROWS) + r : tile0 * NT_ROWS + r; };
    auto fetched = [&](int k0) { return TAIL && k0 >= K ? k0 & ~255 : k0; };   // where the stage at k0 is fetched from

    // ---- loads go straight to LDS: piece p = j * waves + wave of a stage is 1 KiB, whole rows of x | v.  The 16-byte chunk c
    // of row q lies at position c ^ swz(q) of the row, so that the fragment reads (32 rows at the same chunk) spread over all
    // banks; the lanes of a piece fetch their chunks in that order.
    // Written as assembly with waits placed by hand: the compiler would order every LDS read behind all loads in flight.
    auto swz = [](int row) { return KS == 64 ? (row >> 1) & 7 : row & 15; };
    const uint16_t* src[LPW];                                   // (64-bit: a stage spans up to 256 rows of any length)
    uint32_t upper = 0u;                                        // bit j: the lane's chunk of load j lies in the second 64 k
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
        const int row = ((j < XL ? j : j - XL) * F::kWaves + wave) * RPP + lane / F::kChunks;
        const int chunk = (lane % F::kChunks) ^ swz(row);
        src[j] = (j < XL ? x + (int64_t)min(row_of(row), M - 1) * ldx : nt_v(fac, col0 + row, K)) + chunk * 8;
        upper |= (uint32_t)(chunk >> 3) << j;
    }
    auto issue = [&](int slot, int st) {
        const int k0 = fetched(kof(st));
        const bool cut = TAIL && KS == 128 && k0 + KS > K;
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const uint32_t dst = (uint32_t)(slot * STAGE + (j * F::kWaves + wave) * 1024);
            const uint16_t* g = src[j] + k0;
            if (cut) g -= ((upper >> j) & 1u) * 64u;
            asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" :: "v"(g), "s"(dst) : "memory");
        }
    };

    constexpr int CT = F::kColTiles;
    float16_t acc[NH][CT];
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[h][j][e] = 0.0f;
    // wave: quarter of the stage, column group; lane l of an operand: row l % 32, chunk 2 ks + l / 32 of the quarter.
    // (An odd number of column tiles: the second group's last is its neighbour's again, and not written.)
    const int rt = TILES == 2 ? wave / (F::kWaves / 2) : 0;     // row tile
    const int qi = wave % F::kQuarters, cg = wave / F::kQuarters % F::kColGroups;
    const int lr = lane & 31;
    int foff[4], coff[CT];
    const int xoff = rt * NT_ROWS * RB;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) foff[ks] = lr * RB + (((qi * 8 + ks * 2 + (lane >> 5)) ^ swz(lr)) * 16);
#pragma unroll
    for (int j = 0; j < CT; ++j) coff[j] = (F::kRows + min(cg * CT + j, RT - 1) * 32) * RB;
    auto multiply = [&](int slot, int step, int k0, float16_t (&sums)[CT]) {
        // selects, not branches: product and encoder stay interleaved
        const bool out = (TAIL && k0 + qi * 64 >= K) || (TILES == 2 && (rt ? step < lag : step >= wide_steps));
        const unsigned char* b = lds + slot * STAGE;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            bf16x8_t fa = *reinterpret_cast<const bf16x8_t*>(b + xoff + foff[ks]);
            if (out) fa = bf16x8_t{};
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                bf16x8_t fb = *reinterpret_cast<const bf16x8_t*>(b + coff[j] + foff[ks]);
                if (out) fb = bf16x8_t{};
                sums[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb, fa, sums[j], 0, 0, 0);
            }
        }
    };
    // a thread encodes one block of the stage, consecutive threads consecutive blocks of a row.  Rows past the tensor repeat its last row: the stores below are
    // never skipped, which the counted waits rely on (the same bytes to the same place).
    float gmax = 0.0f;
    const int erow = tid / (KS / 16), eblk = tid % (KS / 16), eswz = swz(erow);
    const int64_t eib = (int64_t)min(row_of(erow), M - 1) * (K / kBlock);
    auto encode = [&](int slot, int k0) {
        if constexpr (QMODE >= 0) {
            const unsigned char* b = lds + slot * STAGE + erow * RB;
            const int blk = (TAIL && k0 + eblk * kBlock >= K) ? eblk - 4 : eblk;
            const uint4 c0 = *reinterpret_cast<const uint4*>(b + ((2 * blk) ^ eswz) * 16);
            const uint4 c1 = *reinterpret_cast<const uint4*>(b + ((2 * blk + 1) ^ eswz) * 16);
            float val[kBlock];
            const float none[kBlock] = {};
            unpack16(c0, c1, val);
            const float am = block_amax(val);
            gmax = fmaxf(gmax, am);
            const int64_t ib = eib + k0 / kBlock + blk;
            q_amax[ib] = (uint16_t)(__float_as_uint(am) >> 16);
            codes[ib] = encode_block<QMODE < 0 ? 0 : QMODE, false>(val, block_scalar<QMODE < 0 ? 0 : QMODE>(am), none);
        }
    };

    // ---- stage st lies in slot st % NS.  Per stage: wait for its own loads (a stage is requested NS - 1 iterations ahead),
    // barrier, request stage st + NS - 1 into the slot that everybody left before the barrier, multiply, encode.
    // The counter also counts the two stores of an encoded stage: (NS - 1) iterations of them follow a stage's loads.
    constexpr int STORES = QMODE >= 0 ? 2 : 0;
#pragma unroll
    for (int p = 0; p < NS - 1; ++p)
        if (p < steps) issue(p, p);
    int slot = 0;
    for (int step = 0; step < steps; step += NH) {
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const int st = step + h;
            if (st + NS - 1 > steps) nt_wait<0>();             // fewer stages behind it than counted below
            else if (st < NS - 1) nt_wait<(NS - 2) * LPW>();
            else nt_wait<(NS - 2) * LPW + (NS - 1) * STORES>();
            __syncthreads();
            if (st + NS - 1 < steps) issue(slot == 0 ? NS - 1 : slot - 1, st + NS - 1);
            const int k0 = kof(st);
            multiply(slot, step / NH, k0, acc[h]);
            encode(slot, fetched(k0));
            slot = slot + 1 == NS ? 0 : slot + 1;
        }
    }
    if constexpr (NH * CT > 12) {                               // R = 256: 256 sums per lane, left in the accumulation registers until they are read
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int j = 0; j < CT; ++j) asm volatile("" : "+a"(acc[h][j]));
    }
    __syncthreads();                                            // the ring is free
    float* red = reinterpret_cast<float*>(lds);                 // [stage of the step][column tile][e][lane], then the waves' maxima
    auto red_at = [&](int h, int jt, int e) -> float& { return red[(((rt * NH + h) * RT + jt) * 16 + e) * 64 + lane]; };
    constexpr int MAXIMA = F::kStages * (F::kQuarters - 1) * TILES * RT * 1024;
    if constexpr (QMODE >= 0) {
        float* smax = red + MAXIMA;
        const float wm = wave_max(gmax);
        if (lane == 0) smax[wave] = wm;
    }
    // acc[h][j][e] of lane l: row m0 + l % 32, column 32 (cg CT + j) + 8 (e / 4) + 4 (l / 32) + e % 4.  The odd quarters
    // join the even ones in LDS.
    if (qi > 0) {
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int j = 0; j < CT; ++j)
                if (cg * CT + j < RT) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) red_at(h, cg * CT + j, e) = acc[h][j][e];
                }
    }
    __syncthreads();
    if constexpr (QMODE >= 0) {
        const float* smax = red + MAXIMA;
        const uint32_t gid = blockIdx.y * gridDim.x + blockIdx.x, gsize = gridDim.x * gridDim.y;
        if (tid == 0) {
            float wm = smax[0];
#pragma unroll
            for (int w = 1; w < F::kWaves; ++w) wm = fmaxf(wm, smax[w]);
            q_gmax[gid] = __float_as_uint(wm);
        }
        for (uint32_t j = gsize + gid * F::kThreads + tid; j < fill_to; j += gsize * F::kThreads) q_gmax[j] = 0u;
    }
    const int m = row_of(rt * NT_ROWS + lr);
    if (qi > 0 || m >= M || (TILES == 2 && rt && tile1 == tile0)) return;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        const int jt = cg * CT + j;
        if (jt >= RT) break;
        const uint16_t* sj = t && !part ? nt_s(fac, col0 + jt * 32) : nullptr;     // the 32 columns belong to one member
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int col = col0 + jt * 32 + 8 * g + 4 * (lane >> 5);
            float sum[4];
            uint32_t h[4], ts[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] = acc[0][j][4 * g + e];
#pragma unroll
                for (int h = 0; h < NH; ++h) {
                    if (h) sum[e] += acc[h][j][4 * g + e];
                    if constexpr (F::kQuarters > 1) sum[e] += red_at(h, jt, 4 * g + e);
                }
            }
            if (part) {                                         // one of several slices: the finishing kernel rounds
                *reinterpret_cast<float4*>(part + ((int64_t)blockIdx.y * M + m) * R + col) = make_float4(sum[0], sum[1], sum[2], sum[3]);
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                h[e] = bf16_bits(sum[e]);
                if (t) ts[e] = bf16_bits(__uint_as_float(h[e] << 16) * bf16_lo(sj[8 * g + 4 * (lane >> 5) + e]));
            }
            *reinterpret_cast<uint2*>(xv + (int64_t)m * R + col) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            if (t) *reinterpret_cast<uint2*>(t + (int64_t)m * R + col) = make_uint2(ts[0] | (ts[1] << 16), ts[2] | (ts[3] << 16));
        }
    }
}

// xv = bf16(sum over slices, ascending), t = bf16(xv * s): four columns per thread.  A round trip to the memory behind the slices' L2s and
// little else: s and eight slices are requested together.  Both launches, one slice after the other | now: 256 x 18944, R = 64 (sixteen slices) 12.1 |
// 8.9 us, 411 x 8960 9.3 | 7.9, 800 x 18944 17.8 | 15.3, 2103 x 18944 22.7 | 21.4; 1024 x 3584, R = 32 (three) 7.1 | 7.1.  (Workgroups of 64: 7.3.)
__global__ __launch_bounds__(256) void lowrank_nt_finish_kernel(const float* __restrict__ part, int slices, int64_t MR, uint32_t R,
                                                                const NtFactors fac, uint16_t* __restrict__ xv, uint16_t* __restrict__ t)
{
    constexpr int BATCH = 8;
    const uint32_t quad = blockIdx.x * 256u + threadIdx.x;
    const int64_t i = (int64_t)quad * 4;
    if (i >= MR) return;
    uint16_t sv[4] = {0, 0, 0, 0};
    if (t) {
        const uint16_t* s = nt_s(fac, (int)(quad % (R / 4u)) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) sv[e] = s[e];
    }
    float4 a = *reinterpret_cast<const float4*>(part + i);
    for (int k0 = 1; k0 < slices; k0 += BATCH) {
        float4 b[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k)
            if (k0 + k < slices) b[k] = *reinterpret_cast<const float4*>(part + (int64_t)(k0 + k) * MR + i);
#pragma unroll
        for (int k = 0; k < BATCH; ++k)
            if (k0 + k < slices) { a.x += b[k].x; a.y += b[k].y; a.z += b[k].z; a.w += b[k].w; }
    }
    const uint32_t h[4] = {bf16_bits(a.x), bf16_bits(a.y), bf16_bits(a.z), bf16_bits(a.w)};
    *reinterpret_cast<uint2*>(xv + i) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    if (t) {
        uint32_t ts[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) ts[e] = bf16_bits(__uint_as_float(h[e] << 16) * bf16_lo(sv[e]));
        *reinterpret_cast<uint2*>(t + i) = make_uint2(ts[0] | (ts[1] << 16), ts[2] | (ts[3] << 16));
    }
}

// K slices for M rows: none when 32-row tiles give every compute unit a workgroup; otherwise two such tiles per compute unit or a few
// more, at least 1024 k per slice, and never more workgroups than the quantizer's partial maxima have room for.
static int nt_slices(int64_t M, int64_t K, size_t workspace_bytes, int64_t R)
{
    const int64_t tiles = (M + 31) / 32, steps = (K + 255) / 256, cus = device_cus();
    if (tiles >= cus) return 1;
    int64_t sl = (2 * cus + tiles - 1) / tiles;
    if (sl > steps / 4) sl = steps / 4;
    if (sl * tiles > (int64_t)kDeferredPartials) sl = (int64_t)kDeferredPartials / tiles;
    if (sl > 16) sl = 16;
    while (sl > 1 && (size_t)(sl * M * R * 4) > workspace_bytes) --sl;
    return sl < 1 ? 1 : (int)sl;
}

size_t lowrank_nt_workspace_bytes(int64_t M, int64_t R, int64_t K)
{
    if (M <= 0 || R <= 0 || K <= 0) return 0;
    const int sl = nt_slices(M, K, (size_t)-1, R);
    return sl > 1 ? (size_t)sl * M * R * 4 : 0;
}

// Whether the row tiles go in pairs (stages of 128 k, three, from 192 columns on two), which fetch v half as often.  Only where single tiles would
// share compute units, and where a pair's walk is not much longer than a tile's: the workgroup whose two tiles start `lag` steps apart ends the
// launch.  They pay where x no longer fits the memory-side cache, or V's pieces are most of what a unit takes in.  Microseconds, single | pairs, on
// an x just read and, after the dash, on one from HBM; lags in brackets where there is one:
//   R = 192  16384 x 3584 50 | 44 - 94 | 80, 8704 x 2048 (1 of 8) 35 | 30 - 54 | 50, 8225 x 3840 51 | 44 - 96 | 77, 8225 x 5120 (5 of 20) 62 | 61 - 116 | 101;
//            8225 x 2560 (5 of 10) 38 | 41 - 70 | 66, 8225 x 320 (1 of 2) 18.0 | 18.6, 8225 x 128 14.4 | 15.3
//   R = 256  16384 x 3584 61 | 54 - 112 | 87, 8704 x 1536 (1 of 6) 34 | 32 - 57 | 49;  16384 x 1024 31 | 33, 16384 x 320 25 | 28, 12345 x 2560 (5 of 10) 50 | 55
//   R = 128  16384 x 3584 35.3 | 34.5 - 72 | 65, 8225 x 3072 (1 of 12) 29.5 | 28.8 - 56 | 49, 8225 x 7680 (5 of 30) 63 | 60 - 117 | 98, 16384 x 5120 47 | 44 - 98 | 88;
//            rows of whole 4 KiB 8225 x 4096 33.2 | 34.9, 16384 x 2048 24.1 | 24.8, 8225 x 8192 56 | 58; short ones 8704 x 1536 (1 of 6) 19.3 | 19.9,
//            16384 x 1024 17.6 | 18.3; lags 10240 x 3840 (5 of 15) 37 | 39, 12345 x 5120 (5 of 20) 46.6 | 47.8
//   beyond 120 M elements  R = 128 16384 x 8960 106 | 87 - 152 | 140, R = 96 8225 x 14592 126 | 91 - 186 | 144, R = 64 12000 x 18944 143 | 121 - 191 | 169;
//            16384 x 7680 (5 of 30) R = 96 59.6 | 63.3, R = 64 46.6 | 47.0; below 120 M, R = 64 16384 x 6400 41 | 43
//   R = 32   10240 x 14336 73 | 66 - 138 | 124, 16384 x 8960 59 | 55;  8225 x 14592 49 | 57, 9000 x 14336 52 | 54, 16384 x 6400 35 | 40
//   with the quantizer, R = 64: 8225 x 14592 150 | 127 - 190 | 162, 16384 x 18944 247 | 213 - 288 | 247;  R = 32 8225 x 18944 142 | 156 - 186 | 180,
//            16384 x 8960 94 | 102 - 139 | 143, 12000 x 18944 165 | 169 - 210 | 201
static bool nt_pairs(int64_t tiles, int64_t M, int64_t R, int64_t K, bool quantizes)
{
    if (tiles <= device_cus() || K > 1 << 20) return false;
    const int64_t steps = (K + 255) / 256;
    const bool fives = steps % NT_ROTATE == 0;
    const int64_t p = fives ? steps / NT_ROTATE : steps;         // classes of tiles that start alike (nt_pair)
    const int64_t lag = p == 1 || tiles % (2 * p) == 0 ? 0 : fives || tiles < p ? NT_ROTATE : 1;
    if (R == 32 && quantizes) return false;
    if (M * K > (R == 32 ? 140000000 : 120000000) && 7 * lag <= steps) return true;
    if (R >= 192) return K > 1024 && 3 * lag <= steps;
    return R == 128 && K > 2560 && K % 2048 != 0 && 6 * lag <= steps;
}

// Columns per workgroup without the quantizer, for `groups` workgroups per column range.  Where these leave compute units
// idle, the time is that of one workgroup's stages, and a stage of R columns takes the longer the more of v it fetches and
// multiplies (and the wide forms' rings hold only two of them): workgroups of 32 or 64 columns side by side (gridDim.z) read x
// again from L2 and finish sooner, with the same bits.  Microseconds at 32 | 64 | all R columns:
//   411 x 1536, R = 192 (13 groups)    7.2 | 8.5 | 17.7         1024 x 3584, R = 192 (96)   11.4 | 10.4 | 14.8
//   2103 x 1536, R = 128 (66)          9.2 | 8.7 | 13.6         1500 x 3584, R = 192 (141)  18.5 | 14.4 | 15.8
//   800 x 3584, R = 128 (75)          10.0 | 9.3 | 12.1         8192 x 4096, R = 192 (256)  53.3 | 37.5 | 40.1
//   4096 x 1536, R = 96 (128)          8.8 |  -  | 11.9         1500 x 8960, R = 128 (376)  22.6 | 20.8 | 18.3
//   2103 x 3584, R = 96 (198)         15.0 |  -  | 11.9         800 x 18944, R = 256 (400)  47.0 | 38.2 | 31.1
//   2103 x 3584, R = 64 (198)         10.5 |  -  | 9.6          4096 x 8960, R = 128 (512)  48.9 | 32.6 | 25.6
// 32 columns up to about a workgroup per compute unit (a rank that has no half of 64 columns: up to 7/4), 64 up to one row group each.
static int nt_column_group(int64_t groups, int64_t R)
{
    const int64_t cus = device_cus();
    if (groups * (R / 32) * 8 <= cus * (R % 64 ? 14 : 9)) return 32;
    return R % 64 == 0 && groups <= cus ? 64 : (int)R;
}

template <int TILES, int RT, int QMODE, int KS, int NS, bool TAIL>
static int launch_nt(int slices, hipStream_t st, const void* x, int64_t ldx, const NtFactors& fac, void* xv, void* t, int64_t M, int64_t R, int64_t K,
                     float* part, void* codes, uint16_t* amax, uint32_t* gmax)
{
    using F = NtForm<TILES, RT, KS, NS>;
    static bool attr_set[64] = {};
    if (const int rc = allow_dynamic_lds((const void*)lowrank_nt_kernel<TILES, RT, QMODE, KS, NS, TAIL>, F::kLds, attr_set)) return rc;
    hipLaunchKernelGGL((lowrank_nt_kernel<TILES, RT, QMODE, KS, NS, TAIL>), dim3((unsigned)((M + F::kRows - 1) / F::kRows), (unsigned)slices, (unsigned)(R / (RT * 32))), dim3(F::kThreads), F::kLds, st,
                       (const uint16_t*)x, ldx, fac, (uint16_t*)xv, (uint16_t*)t, (int)M, (int)K, part, (uint2*)codes, amax, gmax, (uint32_t)kDeferredPartials, (int)R);
    return METIS_OK;
}

// qmode < 0: the product alone.  qmode = METIS_MODE_P32 / _PB16: x (contiguous rows, ldx == K) is quantized on the way,
// codes and the deferred data (partial maxima, parked block maxima) as quantize_row_deferred leaves them.
int lowrank_nt(const void* x, int64_t ldx, const void* v, int64_t M, int64_t R, int64_t K, const void* s, void* xv, void* t,
               hipStream_t st, void* workspace, size_t workspace_bytes, int qmode, void* codes, void* deferred, size_t deferred_size)
{
    if (R <= 0) return METIS_E_ARG;
    const LowrankFactor one = {v, s, R};
    return lowrank_nt_grouped(x, ldx, M, K, &one, 1, xv, t, st, workspace, workspace_bytes, qmode, codes, deferred, deferred_size);
}

int lowrank_nt_grouped(const void* x, int64_t ldx, int64_t M, int64_t K, const LowrankFactor* factors, int count, void* xv, void* t, hipStream_t st,
                       void* workspace, size_t workspace_bytes, int qmode, void* codes, void* deferred, size_t deferred_size)
{
    if (M < 0 || K <= 0 || ldx < K || !factors || count < 1 || count > kTiledMembers) return METIS_E_ARG;
    int64_t R = 0;
    for (int i = 0; i < count; ++i) {
        if (factors[i].r <= 0 || factors[i].r % 32 || factors[i].r > 256) return METIS_E_SHAPE;
        R += factors[i].r;
    }
    if ((R != 32 && R != 64 && R != 96 && R != 128 && R != 192 && R != 256) || K % 64 || ldx % 8) return METIS_E_SHAPE;
    if (M == 0) return METIS_OK;
    if (M > INT32_MAX - 64 || K > INT32_MAX) return METIS_E_ARG;
    if (!x || !xv || ((uintptr_t)x % 16) || ((uintptr_t)xv % 8) || ((uintptr_t)t % 8)) return METIS_E_ARG;
    NtFactors fac = {};
    int col = 0;
    for (int i = 0; i < kTiledMembers; ++i) {
        if (i < count) {
            const LowrankFactor& f = factors[i];
            if (!f.v || (t && !f.s) || ((uintptr_t)f.v % 16) || ((uintptr_t)f.s % 2)) return METIS_E_ARG;
            fac.v[i] = (const uint16_t*)f.v;
            fac.s[i] = (const uint16_t*)f.s;
            col += (int)f.r;
        }
        fac.end[i] = col;
    }
    if (workspace && ((uintptr_t)workspace % 16)) return METIS_E_WORKSPACE;
    Workspace q = {nullptr, nullptr, nullptr};
    if (qmode >= 0) {
        if (qmode != METIS_MODE_P32 && qmode != METIS_MODE_PB16) return METIS_E_ARG;
        if (R > 64) return METIS_E_SHAPE;
        if (ldx != K || !codes || ((uintptr_t)codes % 8)) return METIS_E_ARG;
        if ((M + 31) / 32 > (int64_t)kDeferredPartials) return METIS_E_TOO_LARGE;
        if (M * K / kBlock >= (int64_t)1 << 31) return METIS_E_ARG;
        if (const int rc = carve_deferred(deferred, deferred_size, M, K, &q)) return rc;
    }
    const int slices = workspace ? nt_slices(M, K, workspace_bytes, R) : 1;
    float* part = slices > 1 ? static_cast<float*>(workspace) : nullptr;
    int rc = METIS_OK;
    // Stages of 128 k, three in the ring (two with the quantizer, whose vector work wants more workgroups per compute unit, and where
    // V is wide).  From 96 columns on and with more than one workgroup for a compute unit, stages of 64 k, so that two fit beside
    // each other.  Microseconds, 128 k | 64 k:
    //   R = 96   4096 x 8960 28 | 22, 16384 x 3584 37 | 30, 8192 x 4096 (one workgroup each) 21.7 | 27
    //   R = 128  4096 x 8960 33 | 25, 16384 x 3584 44 | 34, 8192 x 4096 25 | 28
    //   R = 192  4096 x 8960 44 | 36, 16384 x 3584 62 | 48, 8192 x 4096 40 | 47;   R = 256  54 | 48, 75 | 59, 47 | 54
    // An x of more than the memory-side cache wants its rows in longer pieces: 8000 x 18944, R = 128 114 | 138, R = 96 99 | 107; from
    // 192 columns on V's share outweighs that (16384 x 18944 433 | 361).
    //   with the quantizer, R = 64, three | two stages of 128 k: 411 x 1536 12.8 | 11.7, 16384 x 3584 33.4 | 31.7; three where a compute
    //   unit has one workgroup and x comes from HBM: 8192 x 14336 91 | 105
    const int64_t tiles = (M + NT_ROWS - 1) / NT_ROWS, groups = tiles * slices;
    const bool tail = K % 256 != 0, shared = groups > device_cus() && (R > 128 || M * K <= (int64_t)1 << 27);
    const bool pairs = slices == 1 && nt_pairs(tiles, M, R, K, qmode >= 0);
#define METIS_NT(T, RT, Q, KS, NS) do { if (tail) rc = launch_nt<T, RT, Q, KS, NS, true>(slices, st, x, ldx, fac, xv, t, M, R, K, part, codes, q.amax, q.gmax); \
                                        else rc = launch_nt<T, RT, Q, KS, NS, false>(slices, st, x, ldx, fac, xv, t, M, R, K, part, codes, q.amax, q.gmax); } while (0)
#define METIS_NTS(RT, NS, NS64) do { if (pairs) METIS_NT(2, RT, -1, 128, NS); else if (shared) METIS_NT(1, RT, -1, 64, NS64); else METIS_NT(1, RT, -1, 128, NS); } while (0)
    const int width = qmode < 0 ? nt_column_group(groups, R) : (int)R;
    const bool deep = groups <= device_cus() && M * K >= 100000000;
#define METIS_NTQ1(RT, Q) do { if (deep) METIS_NT(1, RT, Q, 128, 3); else METIS_NT(1, RT, Q, 128, 2); } while (0)
#define METIS_NTQ(RT, Q) do { if (pairs) METIS_NT(2, RT, Q, 128, 3); else METIS_NTQ1(RT, Q); } while (0)
#define METIS_NTC(RT) do { if (pairs) METIS_NT(2, RT, -1, 128, 3); else METIS_NT(1, RT, -1, 128, 3); } while (0)
    if (qmode == METIS_MODE_P32) { if (R == 32) METIS_NTQ1(1, 0); else METIS_NTQ(2, 0); }
    else if (qmode >= 0) { if (R == 32) METIS_NTQ1(1, 1); else METIS_NTQ(2, 1); }
    else if (width == 32) METIS_NTC(1);
    else if (width == 64) METIS_NTC(2);
    else if (width == 96) METIS_NTS(3, 3, 4);
    else if (width == 128) METIS_NTS(4, 3, 4);
    else if (width == 192) METIS_NTS(6, 2, 2);
    else METIS_NTS(8, 2, 2);
#undef METIS_NTC
#undef METIS_NTS
#undef METIS_NTQ
#undef METIS_NTQ1
#undef METIS_NT
    if (rc) return rc;
    if (hipGetLastError() != hipSuccess) return METIS_E_LAUNCH;
    if (slices > 1) {
        const int64_t MR = M * R;
        hipLaunchKernelGGL(lowrank_nt_finish_kernel, dim3((unsigned)((MR / 4 + 255) / 256)), dim3(256), 0, st, part, slices, MR, (uint32_t)R, fac,
                           (uint16_t*)xv, (uint16_t*)t);
        if (hipGetLastError() != hipSuccess) return METIS_E_LAUNCH;
    }
    return METIS_OK;
}

// ---------------------------------------------------------------------------------------------
// out[C, R] = sum_l a[l, C] b[l, R]
// ---------------------------------------------------------------------------------------------
// One contraction of a launch, and where its result goes.
struct TnProblem {
    const uint16_t *a, *b;
    int64_t lda;
    int C, groups, slices, per;                                // groups of 64 columns, slices of `per` steps of 64 tokens
    float* part;
    void* out;
    int out_f32, transpose;
};

// One workgroup: 64 columns of a, one slice of the tokens.
template <int RT>
__device__ __forceinline__ void lowrank_tn_block(const TnProblem& p, int block, int L)
{
    const uint16_t *__restrict__ a = p.a, *__restrict__ b = p.b;
    const int64_t lda = p.lda;
    const int C = p.C, steps_per_slice = p.per;
    float* __restrict__ part = p.part;
    constexpr int R = RT * 32;
    // Staged as loaded, token by token, in slabs of 32 columns: [slab][token][32], 64 bytes per token and slab.  The MFMA
    // fragments (8 consecutive tokens of one column) come out of LDS through the transposing read of gfx950
    // (ds_read_b64_tr_b16: the sixteen lanes of a group hand in sixteen addresses of 4 halves each and lane l receives
    // element l % 4 of the pieces of lanes l / 4, l / 4 + 4, l / 4 + 8, l / 4 + 12 -- established with a probe on the
    // device.  With lane i handing in the piece (token i / 4, columns 4 (i % 4) ..), lane l gets column l of four
    // consecutive tokens), so nothing is scattered element by element.  Rows of 64 bytes keep both the 16-byte writes and the
    // transposing reads free of bank conflicts (rows r .. r + 3 and the two 32-byte halves of a row fall on different banks).
    __shared__ __attribute__((aligned(16))) uint16_t at[2][64 * 32];          // [column slab][token][column]
    __shared__ __attribute__((aligned(16))) uint16_t bt[RT][64 * 32];         // [r slab][token][r]
    __shared__ __attribute__((aligned(16))) float red[2][RT][16][64];         // the two waves that take the second half of each step
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c0 = block % p.groups * 64, slice = block / p.groups;
    const int steps_all = (L + 63) / 64;
    const int s0 = slice * steps_per_slice, s1 = min(s0 + steps_per_slice, steps_all);
    // loading: thread -> token tid / 8 (+ 32), 16-byte chunk tid % 8 of the 64 columns; for b, R / 8 chunks per token
    const int lrow = tid >> 3, lch = tid & 7;
    const bool col_live = c0 + lch * 8 < C;                     // C % 8 == 0: a chunk is inside or outside
    constexpr int BCH = R / 8;                                  // 16-byte chunks per token of b: 4, 8 or 16
    constexpr int BPT = 64 * BCH / 256;                         // b chunks per thread: 1, 2 or 4
    uint4 ra[2][2], rbv[2][BPT];
    auto fetch = [&](uint4 (&ra)[2], uint4 (&rbv)[BPT], int st) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int l = st * 64 + i * 32 + lrow;
            ra[i] = (l < L && col_live) ? *reinterpret_cast<const uint4*>(a + (int64_t)l * lda + c0 + lch * 8) : make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int i = 0; i < BPT; ++i) {
            const int id = i * 256 + tid, l = st * 64 + id / BCH, ch = id % BCH;
            rbv[i] = l < L ? *reinterpret_cast<const uint4*>(b + (int64_t)l * R + ch * 8) : make_uint4(0u, 0u, 0u, 0u);
        }
    };
    auto stage = [&](const uint4 (&ra)[2], const uint4 (&rbv)[BPT]) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            *reinterpret_cast<uint4*>(&at[lch >> 2][(i * 32 + lrow) * 32 + (lch & 3) * 8]) = ra[i];
#pragma unroll
        for (int i = 0; i < BPT; ++i) {
            const int id = i * 256 + tid, tok = id / BCH, ch = id % BCH;
            *reinterpret_cast<uint4*>(&bt[ch >> 2][tok * 32 + (ch & 3) * 8]) = rbv[i];
        }
    };
    float16_t acc[RT];
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
    // wave -> 32 columns (wave % 2) and the first or second half (wave / 2) of every 64-token step
    const int ct = wave & 1, kh = wave >> 1;
    // lane l of the MFMA holds column l % 32 and the tokens 8 (l / 32) .. + 7 of a 16-token step; in its group of sixteen
    // lanes it hands in the piece (token i / 4, columns 16 (l / 16 % 2) + 4 (i % 4) ..), i = l % 16
    typedef short short4_t __attribute__((ext_vector_type(4)));
    typedef short short8_t __attribute__((ext_vector_type(8)));
    const int piece = ((lane & 15) >> 2) * 32 + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
    auto fragment = [&](const uint16_t* slab, int tok0) -> bf16x8_t {
        typedef short4_t __attribute__((address_space(3))) * lds_ptr_t;
        const uint16_t* p = slab + tok0 * 32 + piece;
        const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)p);
        const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr_t)(p + 4 * 32));
        const short8_t v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return __builtin_bit_cast(bf16x8_t, v);
    };
    auto multiply = [&]() {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int tok0 = (kh * 4 + ks * 2 + (lane >> 5)) * 8;
            const bf16x8_t fa = fragment(at[ct], tok0);
#pragma unroll
            for (int j = 0; j < RT; ++j) {
                const bf16x8_t fb = fragment(bt[j], tok0);
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb, fa, acc[j], 0, 0, 0);
            }
        }
    };
    // two steps in flight while a third is multiplied
    if (s0 < s1) fetch(ra[0], rbv[0], s0);
    if (s0 + 1 < s1) fetch(ra[1], rbv[1], s0 + 1);
    for (int st = s0; st < s1; st += 2) {
        stage(ra[0], rbv[0]);
        __syncthreads();
        if (st + 2 < s1) fetch(ra[0], rbv[0], st + 2);
        multiply();
        __syncthreads();
        if (st + 1 < s1) {
            stage(ra[1], rbv[1]);
            __syncthreads();
            if (st + 3 < s1) fetch(ra[1], rbv[1], st + 3);
            multiply();
            __syncthreads();
        }
    }
    // acc[j][e] of lane l: column c0 + 32 ct + l % 32, r = 32 j + 8 (e / 4) + 4 (l / 32) + e % 4; halves of the steps add up
    if (kh == 1) {
#pragma unroll
        for (int j = 0; j < RT; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) red[ct][j][e][lane] = acc[j][e];
    }
    __syncthreads();
    if (kh == 1) return;
    const int c = c0 + ct * 32 + (lane & 31);
    if (c >= C) return;
    float* dst = part + ((int64_t)slice * C + c) * R;
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float4 o;
            o.x = acc[j][4 * g] + red[ct][j][4 * g][lane];
            o.y = acc[j][4 * g + 1] + red[ct][j][4 * g + 1][lane];
            o.z = acc[j][4 * g + 2] + red[ct][j][4 * g + 2][lane];
            o.w = acc[j][4 * g + 3] + red[ct][j][4 * g + 3][lane];
            *reinterpret_cast<float4*>(dst + j * 32 + 8 * g + 4 * (lane >> 5)) = o;
        }
}

// The two contractions of a layer's backward pass (dY^T t for U, x^T g_xv for V) and the gradient of its scale vector in one
// launch: they need nothing of each other.  scale_grad's few workgroups come first: they are a serial chain, not work.
template <int RT>
__global__ __launch_bounds__(256) void lowrank_tn_kernel(const TnProblem p0, const TnProblem p1, int L, int scale_blocks, const uint16_t* __restrict__ g,
                                                         const uint16_t* __restrict__ xv, void* __restrict__ scale_out, int scale_f32)
{
    if ((int)blockIdx.x < scale_blocks) {
        __shared__ __attribute__((aligned(16))) float chains[8][256 + 4];
        scale_grad_block((int)blockIdx.x, g, xv, L, RT * 32, scale_out, scale_f32, chains);
        return;
    }
    const int b = (int)blockIdx.x - scale_blocks, first = p0.groups * p0.slices;
    lowrank_tn_block<RT>(b < first ? p0 : p1, b < first ? b : b - first, L);
}

// Adds the token slices in order; out [C, R] or, transposed, [R, C]; bf16 or binary32.  A thread has four consecutive r of a column, so
// that a wave reads whole lines of the partial sums; transposed, a workgroup turns its columns through LDS and writes 32 or 64 bytes (bf16)
// of a row at a time.  (The lanes over the output's columns fetched 16 bytes of every line, and each line once per quad of r.)  What bounds
// it is what a compute unit takes in and one round trip to the memory behind the slices' L2s: eight slices are requested together.
// With the launch before it, both contractions of a layer, tokens x N, K, R, lanes over the output's columns | now: 4096 x 1536, 8960, 32 33.2 | 23.1 us,
// 4096 x 8960, 1536, 32 28.0 | 23.5, 2103 x 3584, 18944, 64 46.3 | 32.7, 2103 x 18944, 3584, 64 36.5 | 33.0, 8192 x 4096, 4096, 64 49.3 | 45.3,
// 1000 x 2048, 2568, 128 21.6 | 17.1, 411 x 1536, 8960, 64 14.7 | 11.0.  From a rank of 64 on 32 columns to a workgroup leave compute units idle.
// No load stands under a condition of its lane's (a lane past the end reads the last quad), and none of a whole batch under any: the eight would wait
// for each other.  One contraction, the loads of live lanes under their condition | now: 4608 x 1536, R = 32 (18 slices) 13.0 | 9.4 us, 20000 x 64,
// R = 64 (63) 26.7 | 11.9, 20000 x 256, R = 128 transposed (63) 45.7 | 23.3; 2103 x 3584, R = 64 (7) 13.6 | 12.8.
template <int N, int BATCH>
__device__ __forceinline__ void tn_sum_slices(const TnProblem& p, const float* const (&src)[N], int64_t CR, float4 (&sum)[N])
{
    const int slices = p.slices;
#pragma unroll
    for (int u = 0; u < N; ++u) sum[u] = *reinterpret_cast<const float4*>(src[u]);
    auto add = [&](int z0, auto in) {                            // in(i): there is a slice z0 + i
        float4 v[BATCH][N];
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (in(i)) {
#pragma unroll
                for (int u = 0; u < N; ++u) v[i][u] = *reinterpret_cast<const float4*>(src[u] + (int64_t)(z0 + i) * CR);
            }
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (in(i)) {
#pragma unroll
                for (int u = 0; u < N; ++u) { sum[u].x += v[i][u].x; sum[u].y += v[i][u].y; sum[u].z += v[i][u].z; sum[u].w += v[i][u].w; }
            }
    };
    int z0 = 1;
    for (; z0 + BATCH <= slices; z0 += BATCH) add(z0, [](int) { return true; });
    if (z0 < slices) add(z0, [&](int i) { return z0 + i < slices; });
}
__device__ __forceinline__ void tn_store_quad(const TnProblem& p, int64_t o, const float4 f)    // four consecutive elements of the output
{
    typedef uint32_t pair_t __attribute__((ext_vector_type(2), aligned(4)));
    typedef uint32_t quad_t __attribute__((ext_vector_type(4), aligned(4)));
    if (p.out_f32)
        *reinterpret_cast<quad_t*>(static_cast<float*>(p.out) + o) =
            (quad_t){__float_as_uint(f.x), __float_as_uint(f.y), __float_as_uint(f.z), __float_as_uint(f.w)};
    else
        *reinterpret_cast<pair_t*>(static_cast<uint16_t*>(p.out) + o) =
            (pair_t){bf16_bits(f.x) | (bf16_bits(f.y) << 16), bf16_bits(f.z) | (bf16_bits(f.w) << 16)};
}
constexpr int tn_turn(int rt) { return rt == 1 ? 32 : 16; }     // columns that a workgroup turns, 256 quads and more
template <int RT>
__global__ __launch_bounds__(256) void lowrank_tn_finish_kernel(const TnProblem p0, const TnProblem p1, int first)
{
    constexpr int R = RT * 32, TN_TURN = tn_turn(RT), Q = RT * TN_TURN / 32;
    __shared__ float turn[R][TN_TURN + 1];
    const bool second = (int)blockIdx.x >= first;
    const TnProblem& p = second ? p1 : p0;
    const int block = (int)blockIdx.x - (second ? first : 0), tid = (int)threadIdx.x;
    const int64_t CR = (int64_t)p.C * R;
    if (!p.transpose) {
        const int64_t o = ((int64_t)block * 256 + tid) * 4;
        const float* const src[1] = {p.part + (o < CR ? o : CR - 4)};
        float4 sum[1];
        tn_sum_slices<1, 8>(p, src, CR, sum);
        if (o < CR) tn_store_quad(p, o, sum[0]);
        return;
    }
    const int64_t c0 = (int64_t)block * TN_TURN;
    const float* src[Q];
    float4 sum[Q];
#pragma unroll
    for (int u = 0; u < Q; ++u) {
        const int64_t o = c0 * R + (int64_t)(u * 256 + tid) * 4;     // (the columns of a workgroup are one piece of each slice)
        src[u] = p.part + (o < CR ? o : CR - 4);
    }
    tn_sum_slices<Q, 8>(p, src, CR, sum);
#pragma unroll
    for (int u = 0; u < Q; ++u) {
        const int c = (u * 256 + tid) / (R / 4), r = (u * 256 + tid) % (R / 4) * 4;
        turn[r][c] = sum[u].x; turn[r + 1][c] = sum[u].y; turn[r + 2][c] = sum[u].z; turn[r + 3][c] = sum[u].w;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < Q; ++u) {
        const int r = (u * 256 + tid) / (TN_TURN / 4), c = (u * 256 + tid) % (TN_TURN / 4) * 4;
        if (c0 + c < p.C)                                            // (C is a multiple of 8)
            tn_store_quad(p, (int64_t)r * p.C + c0 + c, make_float4(turn[r][c], turn[r][c + 1], turn[r][c + 2], turn[r][c + 3]));
    }
}

static int tn_slices(int64_t L, int64_t C, int* steps_per_slice)
{
    const int64_t steps = (L + 63) / 64, groups = (C + 63) / 64;
    int64_t want = (4 * (int64_t)device_cus() + groups - 1) / groups;       // four workgroups per compute unit
    if (want > steps / 4) want = steps / 4;                                 // at least four steps per slice
    if (want < 1) want = 1;
    const int64_t per = (steps + want - 1) / want;
    *steps_per_slice = (int)per;
    return (int)((steps + per - 1) / per);
}

size_t lowrank_tn_workspace_bytes(int64_t L, int64_t C, int64_t R)
{
    if (L <= 0 || C <= 0 || R <= 0) return 0;
    int per;
    return (size_t)tn_slices(L, C, &per) * (size_t)C * (size_t)R * sizeof(float);
}

static int tn_problem(const void* a, int64_t lda, const void* b, int64_t L, int64_t C, int64_t R, void* out, int out_dtype, int transpose,
                      void* workspace, size_t workspace_bytes, TnProblem* p)
{
    if (L < 0 || C <= 0 || R <= 0 || lda < C) return METIS_E_ARG;
    if (out_dtype != METIS_DTYPE_BF16 && out_dtype != METIS_DTYPE_F32) return METIS_E_ARG;
    if ((R != 32 && R != 64 && R != 128) || C % 8 || lda % 8) return METIS_E_SHAPE;
    if (L > INT32_MAX - 64 || C > INT32_MAX - 64) return METIS_E_ARG;
    if (!a || !b || !out) return METIS_E_ARG;
    if (((uintptr_t)a % 16) || ((uintptr_t)b % 16) || ((uintptr_t)out % 4)) return METIS_E_ARG;
    if (!workspace || ((uintptr_t)workspace % 16) || workspace_bytes < lowrank_tn_workspace_bytes(L, C, R)) return METIS_E_WORKSPACE;
    *p = TnProblem{(const uint16_t*)a, (const uint16_t*)b, lda, (int)C, (int)((C + 63) / 64), 0, 0, (float*)workspace, out,
                   out_dtype == METIS_DTYPE_F32, transpose};
    p->slices = tn_slices(L, C, &p->per);
    return METIS_OK;
}

static int launch_tn(const TnProblem& p0, const TnProblem& p1, int L, int R, int scale_blocks, const void* g, const void* xv, void* scale_out,
                     int scale_f32, hipStream_t st)
{
    const int64_t blocks = scale_blocks + (int64_t)p0.groups * p0.slices + (int64_t)p1.groups * p1.slices;
    if (blocks > INT32_MAX) return METIS_E_ARG;
    auto finishing = [&](const TnProblem& p) {
        const int64_t per = p.transpose ? tn_turn(R / 32) : 256 * 4 / R;          // columns to a workgroup; R divides 1024
        return p.C ? ((int64_t)p.C + per - 1) / per : 0;
    };
    const int64_t f0 = finishing(p0), f1 = finishing(p1);
#define METIS_TN(RT) do { hipLaunchKernelGGL((lowrank_tn_kernel<RT>), dim3((unsigned)blocks), dim3(256), 0, st, p0, p1, L, scale_blocks, (const uint16_t*)g, \
                                             (const uint16_t*)xv, scale_out, scale_f32); \
                          if (hipGetLastError() != hipSuccess) return METIS_E_LAUNCH; \
                          hipLaunchKernelGGL((lowrank_tn_finish_kernel<RT>), dim3((unsigned)(f0 + f1)), dim3(256), 0, st, p0, p1, (int)f0); } while (0)
    if (R == 32) METIS_TN(1);
    else if (R == 64) METIS_TN(2);
    else METIS_TN(4);
#undef METIS_TN
    return hipGetLastError() == hipSuccess ? METIS_OK : METIS_E_LAUNCH;
}

int lowrank_tn(const void* a, int64_t lda, const void* b, int64_t L, int64_t C, int64_t R, void* out, int out_dtype, int transpose,
               void* workspace, size_t workspace_bytes, hipStream_t st)
{
    TnProblem p;
    if (const int rc = tn_problem(a, lda, b, L, C, R, out, out_dtype, transpose, workspace, workspace_bytes, &p)) return rc;
    return launch_tn(p, TnProblem{}, (int)L, (int)R, 0, nullptr, nullptr, nullptr, 0, st);
}

size_t lowrank_backward_workspace_bytes(int64_t L, int64_t N, int64_t K, int64_t R)
{
    return (lowrank_tn_workspace_bytes(L, N, R) + 255) / 256 * 256 + lowrank_tn_workspace_bytes(L, K, R);
}

// One launch and one finishing launch in place of two of each and scale_grad's.  The step of an MLP with 4096 tokens, 1536 -> 8960,
// R = 32: 1627 -> 1593 us; 2103 tokens, 3584 -> 18944, R = 64: 3779 -> 3740; one projection 1536 -> 8960 in binary32: 592 -> 580.
int lowrank_backward(const void* dy, int64_t lddy, const void* t, int64_t N, const void* x, int64_t ldx, const void* gxv, int64_t K, int64_t L, int64_t R,
                     void* gu, int gu_dtype, void* gv, int gv_dtype, const void* gt, const void* xv, void* gs, int gs_dtype, void* workspace,
                     size_t workspace_bytes, hipStream_t st)
{
    const size_t one = (lowrank_tn_workspace_bytes(L, N, R) + 255) / 256 * 256;
    if (L <= 0) return METIS_E_ARG;
    if (!workspace || workspace_bytes < lowrank_backward_workspace_bytes(L, N, K, R)) return METIS_E_WORKSPACE;
    TnProblem p0, p1;
    if (const int rc = tn_problem(dy, lddy, t, L, N, R, gu, gu_dtype, 0, workspace, one, &p0)) return rc;
    if (const int rc = tn_problem(x, ldx, gxv, L, K, R, gv, gv_dtype, 1, static_cast<char*>(workspace) + one, workspace_bytes - one, &p1)) return rc;
    if (!gt || !xv || !gs || ((uintptr_t)gt % 16) || ((uintptr_t)xv % 16) || ((uintptr_t)gs % 4)) return METIS_E_ARG;
    if (gs_dtype != METIS_DTYPE_BF16 && gs_dtype != METIS_DTYPE_F32) return METIS_E_ARG;
    return launch_tn(p0, p1, (int)L, (int)R, (int)R / 8, gt, xv, gs, gs_dtype == METIS_DTYPE_F32, st);
}

}  // namespace metis
