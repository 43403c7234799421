// W4A4 GEMM main loop for launches with many rows: 256 x 128 tiles, a wavefront owns 64 rows x 128 columns.
//
// Activations as fp6 codes with their scales in the loop's order (act_blocked == 2, ascales_blocked; K a multiple of 512),
// signed or not.  Per output the same matrix instructions, FMAs and order of sums as gemm_w4a4_f8_kernel: identical bits.
//
// What bounds it: power.  A loop of nothing but this kernel's two matrix instructions and sixteen FMAs per 32 x 32 block
// and group, in registers, takes 36 ns per SIMD on zeros and 43 on random codes (the clock falls); this loop takes 51 with
// two workgroups on a CU.  With 32 rows to a wavefront (the 128-row tiles' loop) it is 70: every weight operand is read from
// LDS for one matrix instruction and the CU fetches 7.75 KB for eight steps where this one fetches 11.5 KB for sixteen.
// us before / now (bf16, rank 32): 4608 x 9216, K = 3072: 133.0 / 122.1, with Q/K norm + RoPE 138.4 / 127.2; 12288 columns with
// GELU 204.0 / 197.6; K = 12288, 3072 columns 179.6 / 158.1; 8192 x 9216 227 / 209; 1201 x 9216 with Q/K norm 41.5 / 37.4.
//
//  * Two sets of result registers: the group product of step q + 1 is issued before the FMAs of step q and its scale product
//    between their halves.  A wavefront alone on its SIMD then takes 59 ns a step (77 with one set and the same loads), so a
//    CU that is left with one workgroup is hardly slower than one with two.  The last step of a stage waits for the next
//    one's operands, meets the other wavefronts and reads its first operands before its own FMAs: no bubble at the barrier.
//  * 128 accumulators, 64 result registers and 24 of activations leave 40 of the 256 that two wavefronts per SIMD allow, and one
//    spilled register costs a wait for every load in flight: lane offsets are recomputed where they are used, activation
//    scales wait in LDS, an activation operand is refilled as soon as its group is through, and the matrix instruction runs
//    without block scales (codes count as code / 8, so the sums are 1/64 of the result: an exact factor, put back at the end).
//  * LDS objects are split so that nothing is read from one that a load in flight writes to: the compiler waits for every
//    load before such a read (the scales of even and odd pairs of stages, with one object: 162 against 158 us at K = 12288).
//  * Tiles of 128 rows (32 to a wavefront, same code) fill the last round: see the rule at wide_whole.
#include <algorithm>
#include <type_traits>

#include "gemm_w4a4_tile.h"
#include "gemm_w4a4_wide.h"

namespace svdq {

constexpr int WBM = 256;                          // activation rows of a whole tile: four wavefronts x 64
constexpr int WIDE_GROUP_M = 4;                   // m-tiles per raster band (1024 rows, as with the 128-row tiles)
constexpr int PAIR_BLK = 2 * AUX_LBLK;            // scales of a weight block's 32 rows for a pair of stages
constexpr int AS_SLOT_BYTES = NWAVES * 1024;      // activation scales of four stages: 64 rows x 16 bytes per wavefront

struct WideLds {  // the kernel's LDS objects
    uint8_t *buf0, *buf1;  // weight codes of even and odd stages
    uint8_t *aux0, *aux1;  // weight scales of even and odd pairs of stages
    uint8_t *epi, *as;     // epilogue operands; activation scales: two slots of four stages, then zeros
};

// Of an XCD's `tiles` 256-row tiles, how many run whole; the others, the last ones, run as two workgroups of 128 rows.
// A launch takes as long as the CU with the most work, and a CU does its tiles at nearly the same rate one or two at a time:
// 27 us for one tile of K = 3072, then 21 more for each (288 tiles of 256 rows on 256 CUs 43 us, 504 49, 576 68).  Where the
// last round has tiles for half of the CUs at most, halves take that round from 21 us to 11 (1152 tiles 111.5 / 105.6, 1296 131.9
// / 121.7, 576 67.7 / 58.6); for more than half of them some CU has two halves and both are slower than a whole (432 tiles,
// K = 12288: 184 with halves, 156 without).  An XCD with less than one tile to a CU (launches that the rule at wide_takes leaves to
// the 128-row kernels, unless set_variant forces them here) has 128-row tiles only: 216 tiles 28.1 / 25.9.
__host__ __device__ inline int wide_whole(int tiles, int cus_per_xcd) {
    const int whole = tiles / cus_per_xcd * cus_per_xcd;
    return whole == 0 || 2 * (tiles - whole) <= cus_per_xcd ? whole : tiles;
}

// One tile: RB x 32 rows to a wavefront (2: 256-row tile, 1: 128-row tile) x 128 columns.
template <typename T, int EPI, int RB>
__device__ __forceinline__ void wide_tile(const svdq_gemm_args &a, const WideLds &l, int m0, int n0, int pid_n, int wm, int lane) {
    constexpr int NQ = 8 * RB;  // steps per stage: (group, weight block, row block)
    const int l32 = lane & 31, half = lane >> 5;
    const int G = a.K / GROUP, nstages = G / 2;

    const int nblk = min(n0 / 32 + wm, (a.N + 31) / 32 - 1);
    const __amdgpu_buffer_rsrc_t rW = g_buffer((const uint8_t *)a.wgt_planes + (size_t)nblk * nstages * (WPL_BLOCKS * BLK_BYTES));
    const __amdgpu_buffer_rsrc_t rX =
        g_buffer((const uint8_t *)a.wgt_planes + planes_code_bytes(a.N, a.K) + (size_t)nblk * (nstages + 1) * AUX_BLK);
    // Lane offsets other than 16 * lane are made from it where they are used (fresh() keeps them out of registers in between)
    const uint32_t l16 = (uint32_t)lane * 16u;
    auto fresh = [&]() {
        uint32_t t = l16;
        asm volatile("" : "+v"(t));
        return t;
    };
    auto dma = [&](int s, uint8_t *dst, int i) {
        g_load16_lds(rW, dst + (wm * WPL_BLOCKS + i) * BLK_BYTES, l16, (uint32_t)s * (uint32_t)(WPL_BLOCKS * BLK_BYTES) + (uint32_t)(i * BLK_BYTES));
    };
    auto dma_aux = [&](int s, uint8_t *dst) {  // stages s and s + 1
        const uint32_t t = fresh();
        g_load16_lds(rX, dst + wm * PAIR_BLK, t - (t >> 2), (uint32_t)s * (uint32_t)AUX_BLK);
    };
    const int lastblk = ((a.M + 31) >> 5) - 1;
    const int rb0 = min((m0 >> 5) + RB * wm, lastblk), rb1 = min((m0 >> 5) + RB * wm + RB - 1, lastblk);
    const __amdgpu_buffer_rsrc_t rAct = g_buffer((const uint8_t *)a.act + (size_t)rb0 * G * 1536);
    const __amdgpu_buffer_rsrc_t rAS = g_buffer((const uint8_t *)a.ascales + (size_t)rb0 * (G >> 3) * 512);
    const uint32_t dAct = (uint32_t)(rb1 - rb0) * (uint32_t)G * 1536u;
    const uint32_t dS = (uint32_t)(rb1 - rb0) * (uint32_t)(G >> 3) * 512u;
    v8i a6[2][RB];  // [group][row block]
    auto load_act = [&](int s, int gg) {
        const uint32_t l8 = 1024u + (fresh() >> 1);
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const uint32_t off = (uint32_t)(2 * s + gg) * 1536u + (rb ? dAct : 0u);
            const v4i lo = g_load128(rAct, l16, off);
            const v2i hi = g_load64(rAct, l8, off);
            a6[gg][rb] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], 0, 0};
        }
    };
    auto load_as = [&](int s4, int slot) {
        const uint32_t t = fresh();
        g_load16_lds(rAS, l.as + slot * AS_SLOT_BYTES + wm * 1024, (t & 511u) + (t >> 9) * dS, (uint32_t)s4 * 512u);
    };

    v16f acc[RB][NBN];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int bn = 0; bn < NBN; bn++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[rb][bn][i] = 0.0f;
    const v16f z16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    v16f P[2], S[2];
    v8i w8[2];
    v2i wsp[2];
    int scv[RB];
    auto read_w8 = [&](const uint8_t *base, int b) -> v8i {
        const int gg = b >> 2, bn = b & 3;
        const v4i lo = *(const v4i *)(base + l16 + (bn * WPL_BLOCKS + gg) * BLK_BYTES);
        const v2i hi = *(const v2i *)(base + l16 + (bn * WPL_BLOCKS + 2) * BLK_BYTES + gg * 8);
        return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], 0, 0};
    };
    const uint32_t rrow = (uint32_t)l32 * AUX_LROW;
    auto read_ws = [&](int st, int bn) -> v2i {  // scales of both groups, and a finite value that meets a zero
        return *(const v2i *)((st & 2 ? l.aux1 : l.aux0) + bn * PAIR_BLK + (st & 1) * AUX_LBLK + 8 + rrow);
    };
    auto read_as = [&](int slot, int st) {  // lanes 32-63 read zeros
        const uint32_t t = fresh();
        const uint32_t o = t < 512u ? t + (uint32_t)(slot * AS_SLOT_BYTES + wm * 1024) : (uint32_t)(2 * AS_SLOT_BYTES);
#pragma unroll
        for (int rb = 0; rb < RB; rb++) scv[rb] = *(const int *)(l.as + o + rb * 512 + 4 * st);
    };
    auto scales = [&](int q) -> v16f {
        return mfma32_16bit_k8<T>(wsp[(q / RB) & 1], (v2i){q / (4 * RB) ? scv[q % RB] & (int)0xFFFF0000 : scv[q % RB] & 0xFFFF, 0}, z16);
    };
    auto group = [&](int q) -> v16f {
        return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w8[(q / RB) & 1], a6[q / (4 * RB)][q % RB], z16, 2, 2, 0, 0, 0, 0);
    };
    auto wait_and_meet = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * RB, 15));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    load_act(0, 0);
    load_as(0, 0);
#pragma unroll
    for (int i = 0; i < WPL_BLOCKS; i++) dma(0, l.buf0, i);
    dma_aux(0, l.aux0);
    fetch_epilogue_operands<EPI>(a, l.epi, n0, wm, lane);
    __builtin_amdgcn_sched_barrier(0);
    load_act(0, 1);
    __builtin_amdgcn_sched_barrier(0);
    wait_and_meet();
    read_as(0, 0);
    wsp[0] = read_ws(0, 0);
    w8[0] = read_w8(l.buf0, 0);
    S[0] = scales(0);
    P[0] = group(0);
    if (RB == 1) {
        wsp[1] = read_ws(0, 1);
        w8[1] = read_w8(l.buf0, 1);
    }

    int par = 0;  // parity of the four stages
    auto stage = [&](auto st_tag, int s) {
        constexpr int ST = decltype(st_tag)::value, ST1 = (ST + 1) & 3;
        uint8_t *base = (ST & 1) ? l.buf1 : l.buf0;
        uint8_t *other = (ST & 1) ? l.buf0 : l.buf1;
        const int sn = min(s + 1, nstages - 1);
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int c = q & 1, n = c ^ 1, bn = (q / RB) & 3, rb = q % RB;
            const bool last = q == NQ - 1, reads = q % RB == 0;
            const int b = RB == 2 ? q / 2 + 1 : q + 2;  // the next operand to read
            if (!last) {
                P[n] = group(q + 1);
            } else {
                wait_and_meet();
                if (ST == 3) par ^= 1;
                read_as(par, ST1);
                wsp[0] = read_ws(ST1, 0);
                w8[0] = read_w8(other, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!last && reads && b < 8) w8[b & 1] = read_w8(base, b);
            if (q < WPL_BLOCKS) dma(sn, other, q);
            if (q == 3 && !(ST & 1)) dma_aux(min(s + 2, nstages - 2), ST & 2 ? l.aux0 : l.aux1);
            if (q == 4 && ST == 0) load_as(min((s >> 2) + 1, (nstages >> 2) - 1), par ^ 1);
            if (q == 4 * RB - 2) load_act(sn, 0);
            if (q == 8 * RB - 2) load_act(sn, 1);
#pragma unroll
            for (int i = 0; i < 8; i++) acc[rb][bn][i] = __builtin_fmaf(P[c][i], S[c][i], acc[rb][bn][i]);
            __builtin_amdgcn_sched_barrier(0);
            S[n] = scales(last ? 0 : q + 1);
            if (last) P[n] = group(0);
            __builtin_amdgcn_sched_barrier(0);
            if (!last && reads && b < 8) wsp[b & 1] = read_ws(ST, b & 3);
            if (last && RB == 1) {
                wsp[1] = read_ws(ST1, 1);
                w8[1] = read_w8(other, 1);
            }
#pragma unroll
            for (int i = 8; i < 16; i++) acc[rb][bn][i] = __builtin_fmaf(P[c][i], S[c][i], acc[rb][bn][i]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int s = 0; s < nstages; s += 4) {
        stage(std::integral_constant<int, 0>{}, s);
        stage(std::integral_constant<int, 1>{}, s + 1);
        stage(std::integral_constant<int, 2>{}, s + 2);
        stage(std::integral_constant<int, 3>{}, s + 3);
    }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int bn = 0; bn < NBN; bn++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[rb][bn][i] *= 64.0f;  // codes went in as code / 8
    uint8_t *priv = wm == 0 ? l.buf0 : wm == 1 ? l.buf1 : wm == 2 ? l.aux0 : l.as;
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        tile_epilogue<T, EPI, true>(a, acc[rb], priv, l.epi, m0 + 32 * RB * wm, n0, pid_n, rb, lane);
        // the second block reads its operands again: kept over the first one's epilogue they spill
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <typename T, int EPI>
__global__ __launch_bounds__(NTHREADS, 2) void gemm_w4a4_wide_kernel(svdq_gemm_args a, int rows, int cus_per_xcd) {
    __shared__ __align__(16) uint8_t sbuf0[F8_STAGE_BYTES];
    __shared__ __align__(16) uint8_t sbuf1[F8_STAGE_BYTES];
    __shared__ __align__(16) uint8_t saux0[PRIV_BYTES];  // four weight blocks' scales of two stages; later a wavefront's epilogue memory
    __shared__ __align__(16) uint8_t saux1[NBN * PAIR_BLK];
    __shared__ __align__(16) uint8_t sepi[EPI_LDS_BYTES];
    __shared__ __align__(16) uint8_t sas[2 * AS_SLOT_BYTES + 1024];  // two slots, then zeros
    const int lane = threadIdx.x & 63;
    const int wm = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    const int tiles_m = (rows + WBM - 1) / WBM, tiles_n = (a.N + BN - 1) / BN, tiles = tiles_m * tiles_n;
    const int xcd = blockIdx.x % NUM_XCD, loc = blockIdx.x / NUM_XCD;
    const int per = tiles / NUM_XCD, rem = tiles % NUM_XCD;
    const int cnt = per + (xcd < rem), start = xcd * per + min(xcd, rem);
    const int whole = wide_whole(cnt, cus_per_xcd);
    const bool halves = loc >= whole;
    const int t = halves ? whole + ((loc - whole) >> 1) : loc;
    if (t >= cnt) return;
    const int id = start + t;  // XCD-contiguous ranges of tiles, then the m-banded raster of tile_ids
    const int band = WIDE_GROUP_M * tiles_n;
    const int first_m = (id / band) * WIDE_GROUP_M;
    const int gm = min(tiles_m - first_m, WIDE_GROUP_M);
    const int pid_m = first_m + (id % band) % gm, pid_n = (id % band) / gm;
    const int m0 = pid_m * WBM + (halves ? ((loc - whole) & 1) * (WBM / 2) : 0), n0 = pid_n * BN;
    if (m0 >= rows) return;
    if (threadIdx.x < 64) *(v4i *)(sas + 2 * AS_SLOT_BYTES + threadIdx.x * 16) = (v4i){0, 0, 0, 0};
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(63, 0));
    const WideLds l = {sbuf0, sbuf1, saux0, saux1, sepi, sas};
    if (halves || rows - m0 <= WBM / 2)
        wide_tile<T, EPI, 1>(a, l, m0, n0, pid_n, wm, lane);
    else
        wide_tile<T, EPI, 2>(a, l, m0, n0, pid_n, wm, lane);
}

// Rows a launch has to run: the requantizing epilogues write all M rows, the others those below actual_m only.
static int wide_rows(const svdq_gemm_args &a) {
    const bool quant = a.epilogue == SVDQ_EPI_GELU_QUANT || a.epilogue == SVDQ_EPI_SWIGLU_QUANT;
    return quant ? a.M : a.actual_m;
}

template <typename T>
static void launch_wide(const svdq_gemm_args &a, int cus, hipStream_t s) {
    const int rows = wide_rows(a), tiles = ((rows + WBM - 1) / WBM) * ((a.N + BN - 1) / BN);
    const int per_xcd = std::max(cus / NUM_XCD, 1);
    auto workgroups = [&](int t) { return 2 * t - wide_whole(t, per_xcd); };
    const int most = std::max(workgroups(tiles / NUM_XCD), workgroups((tiles + NUM_XCD - 1) / NUM_XCD));
    const dim3 grid((unsigned)most * NUM_XCD), block(NTHREADS);
    switch (a.epilogue) {
        case SVDQ_EPI_PLAIN:
            hipLaunchKernelGGL((gemm_w4a4_wide_kernel<T, SVDQ_EPI_PLAIN>), grid, block, 0, s, a, rows, per_xcd);
            break;
        case SVDQ_EPI_QK_NORM_ROPE:
            hipLaunchKernelGGL((gemm_w4a4_wide_kernel<T, SVDQ_EPI_QK_NORM_ROPE>), grid, block, 0, s, a, rows, per_xcd);
            break;
        case SVDQ_EPI_GELU_QUANT:
            hipLaunchKernelGGL((gemm_w4a4_wide_kernel<T, SVDQ_EPI_GELU_QUANT>), grid, block, 0, s, a, rows, per_xcd);
            break;
        case SVDQ_EPI_SWIGLU_QUANT:
            hipLaunchKernelGGL((gemm_w4a4_wide_kernel<T, SVDQ_EPI_SWIGLU_QUANT>), grid, block, 0, s, a, rows, per_xcd);
            break;
    }
}

bool wide_runs(const svdq_gemm_args &a) {  // (offsets of a wavefront's two row blocks are 32 bits)
    return a.act_blocked == 2 && a.ascales_blocked && (uint64_t)(a.K / GROUP) * 3072 < (1ull << 32);
}

// Tiles of 256 rows pay where there is one for every CU (below, every tile runs as two of 128 rows, and the kernel built for those is
// the faster one) and where K is long for the epilogue: the loop gains 10 to 20 % of its time, but a wavefront takes its two row blocks
// through the epilogue one after the other, with two workgroups on a CU where the 128-row kernel has three to hide it.  Between two
// and three rounds of tiles (the 128-row kernel: about one and a half to two of its own) K has to be longer.  us, here / the faster
// 128-row build (bf16):
//   plain, rank 32, 3072 columns: K = 3072, 2560 rows (240 tiles) 29.4 / 28.7, 2688 (264) 34.0 / 39.0;  K = 12288 97.6 / 95.4 and
//     110.8 / 132.9;  9216 columns, 2200 rows (648 tiles): K = 512 21.7 / 20.0, K = 1024 30.2 / 30.3;  3072 x 4608, K = 512 14.0 / 15.5
//   Q/K norm + RoPE, 4608 columns: 3072 rows (432 tiles), K = 1024 rank 32 23.2 / 24.9, 128 37.5 / 38.7;  8192 rows, K = 512
//     36.8 / 35.0;  4608 rows (648 tiles): rank 32 K = 1024 35.1 / 34.1, K = 1536 44.6 / 44.8, rank 128 K = 1536 64.2 / 63.2, K = 2048 73.2 / 73.5
//   GELU, 6144 columns, 3072 rows: rank 32 K = 2048 60.4 / 59.4, K = 3072 75.8 / 76.6;  rank 128 K = 3072 121.5 / 117.2, K = 4608 144.3 / 143.2
//   SwiGLU, 4096 columns, 4608 rows: rank 32 K = 1024 40.2 / 39.7, K = 2048 55.7 / 56.4;  rank 128 K = 1536 90.4 / 88.7, K = 2048 97.1 / 96.9
bool wide_takes(const svdq_gemm_args &a, int cus) {
    const long tiles = (long)((wide_rows(a) + WBM - 1) / WBM) * ((a.N + BN - 1) / BN);
    if (tiles < cus) return false;
    const bool between = tiles > 2L * cus && tiles < 3L * cus;
    switch (a.epilogue) {
        case SVDQ_EPI_QK_NORM_ROPE: return a.K >= 1024 + (between ? 8 * a.R : 0);
        case SVDQ_EPI_GELU_QUANT: return a.K >= 1900 + 18 * a.R2;
        case SVDQ_EPI_SWIGLU_QUANT: return a.K >= 1024 + 8 * a.R2;
        default: return a.K >= 1024 || !between;
    }
}

void launch_gemm_wide(const svdq_gemm_args &a, int cus, hipStream_t s) {
    if (a.dtype == SVDQ_BF16)
        launch_wide<BF16>(a, cus, s);
    else
        launch_wide<FP16>(a, cus, s);
}
}  // namespace svdq
