// W4A4 GEMM for launches with few rows: a workgroup owns 32 rows x 128 columns and its eight or four wavefronts split K, or 64 rows x
// 128 columns, and four wavefronts split K over either half of them.
//
// F6ACT: activations as fp6 codes (act_blocked == 2), signed or not; otherwise unsigned nibbles, as the (M, K / 2) matrix or
// in lane order, unpacked to fp8 codes: the same integers and the same sums, so that all hand-over forms of unsigned
// activations give the same bits.  (Signed nibbles need the offset correction and stay with the tiles.)  Same arithmetic as
// gemm_w4a4_f8_kernel (per group one fp6 x fp6 or fp6 x fp8 matrix instruction = the exact integer dot product, one 16-bit
// matrix instruction = the product of the two scales, one fp32 FMA per output); only the order of the fp32 sums over groups
// differs (a partial sum per wavefront; the same order with 32 and 64 rows to a workgroup).  Against 64-bit sums it is the closer one: of 512 x 3072
// outputs in fp16 (K = 3072) 989 are not the correctly rounded value, 1086 with the tiles; K = 12288, 333 rows: 1053 and 1366.
//
// Why: with 128 x 128 tiles a prompt's 512 rows give a 3072-wide layer 96 workgroups on 256 CUs, each alone on its CU with
// one wavefront per SIMD and a barrier per 128 k.  Here the same layer has 384 workgroups and a wavefront runs a quarter of
// K (an eighth where no CU gets a second workgroup).  A CU with two workgroups, or with one of eight wavefronts, has two
// wavefronts per SIMD.  Between one and two of them per CU most launches run as half as many workgroups of 64 rows (split64_takes).
// What bounds the 32-row form: every workgroup streams its own copy of the weight tile from L2 (there is no second row block in it to
// share it with), in all about 11 TB/s at K = 12288 and 512 rows, the rate the tiles' loop is delivered at too and less than half of 64
// bytes per clock and CU.  That is why large launches stay with the tiles.  The epilogue is one wavefront's for each row block; the
// others have ended.
//
//  * Nothing is shared between the wavefronts of a workgroup inside the loop, so weights go straight to registers (they lie
//    in the matrix instruction's lane order) and there is neither LDS nor a barrier in it; a stage (two groups) is
//    requested one stage ahead: 16 KB in flight per wavefront (32 rows).
//  * Wavefront w of those along K takes stages w, w + WAVES, ...: the workgroup reads a contiguous stretch of the weight at a time.
//  * The partial tiles meet in LDS: one wavefront (w < 4 for column block w with 32 rows, each of the eight with 64) adds up a 32 x 32 block in a
//    fixed order (the result does not depend on timing); the sums of a row block go to one wavefront, which owns its whole
//    32 x 128 tile for the epilogue as in the other kernels.
//  * Workgroups of one column tile are neighbours on one XCD, so that a weight tile is fetched into one L2.
#include <algorithm>
#include <type_traits>

#include "gemm_w4a4_split.h"
#include "gemm_w4a4_tile.h"

namespace svdq {

constexpr int SK_BLOCK_BYTES = 16 * 64 * 4;  // one 32 x 32 fp32 block, 16 registers of 64 lanes

template <typename T, int EPI, int WAVES, bool F6ACT>
__global__ __launch_bounds__(WAVES * 64, 2) void gemm_w4a4_split_kernel(svdq_gemm_args a, int tiles_m) {
    static_assert(WAVES >= NBN && NBN == NWAVES, "wavefront w < 4 adds up column block w");
    __shared__ __align__(16) uint8_t sred[NBN * (WAVES - 1) * SK_BLOCK_BYTES];  // [column block][the other wavefronts]
    __shared__ __align__(16) uint8_t sepi[EPI_LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;

    // XCD-contiguous renumbering (ids are dealt round-robin over the XCDs), then the row blocks of a column tile in a row
    const int nb = gridDim.x, xcd = blockIdx.x % NUM_XCD, loc = blockIdx.x / NUM_XCD;
    const int per = (nb + NUM_XCD - 1) / NUM_XCD, rem = nb % NUM_XCD;
    const int id = ((rem == 0 || xcd < rem) ? xcd * per : rem * per + (xcd - rem) * (per - 1)) + loc;
    const int pid_m = id % tiles_m, pid_n = id / tiles_m;
    const int m0 = pid_m * 32, n0 = pid_n * BN;
    const int G = a.K / GROUP, nst = (G + 1) / 2;
    const int count = (nst - wave + WAVES - 1) / WAVES;  // this wavefront's stages (none where K is short)

    // operands, all through raw buffers: base in SGPRs + per-lane offset + scalar offset of block and stage.  A column block
    // past N re-reads the last one (its outputs are never stored).
    const int b0 = n0 / 32, blast = (a.N + 31) / 32 - 1;
    const __amdgpu_buffer_rsrc_t rW = g_buffer((const uint8_t *)a.wgt_planes + (size_t)b0 * nst * (WPL_BLOCKS * BLK_BYTES));
    const __amdgpu_buffer_rsrc_t rX =
        g_buffer((const uint8_t *)a.wgt_planes + planes_code_bytes(a.N, a.K) + (size_t)b0 * (nst + 1) * AUX_BLK);
    const bool ablk = F6ACT || a.act_blocked != 0;
    const uint32_t sA = F6ACT ? 1536u : ablk ? 1024u : 32u;  // a step of one group
    const int mrow = min(m0 + l32, a.M - 1);
    const __amdgpu_buffer_rsrc_t rA = g_buffer((const uint8_t *)a.act + (ablk ? (size_t)pid_m * G * sA : (size_t)m0 * a.ld_act));
    const uint32_t oA = ablk ? (uint32_t)lane * 16u : (uint32_t)(mrow - m0) * (uint32_t)a.ld_act + half * 16;
    // activation scales: with ascales_blocked eight groups of a row lie side by side, 512 bytes per 32 rows
    const bool sblk = a.ascales_blocked != 0;
    const __amdgpu_buffer_rsrc_t rS = g_buffer((const uint8_t *)a.ascales + (sblk ? (size_t)pid_m * (G >> 3) * 512 : 0));
    const uint32_t s1 = sblk ? 2u : 2u * (uint32_t)a.ld_ascales, s8 = sblk ? 512u : 8u * s1;  // steps of one and of eight groups
    const uint32_t oS = sblk ? (uint32_t)l32 * 16u : 2u * (uint32_t)mrow;
    uint32_t wblk[NBN], xblk[NBN];
#pragma unroll
    for (int bn = 0; bn < NBN; bn++) {
        const uint32_t b = (uint32_t)(min(b0 + bn, blast) - b0);
        wblk[bn] = b * (uint32_t)nst * (uint32_t)(WPL_BLOCKS * BLK_BYTES);
        xblk[bn] = b * (uint32_t)(nst + 1) * (uint32_t)AUX_BLK;
    }
    const uint32_t l16 = (uint32_t)lane * 16u, l8 = 1024u + (uint32_t)lane * 8u;
    const uint32_t oX = (uint32_t)l32 * AUX_ROW + 8u;

    v4i w[2][NBN][WPL_BLOCKS], alo[2][2];
    v2i ahi[2][2];
    int ws[2][NBN];
    uint16_t as[2][2];
    auto load = [&](auto set_tag, int i) {  // the wavefront's i-th stage
        constexpr int S = decltype(set_tag)::value;
        const uint32_t s = (uint32_t)(i * WAVES + wave);
#pragma unroll
        for (int gg = 0; gg < 2; gg++) {  // a group past the end (K / 64 odd) re-reads the last one: its weights are zeros
            const uint32_t g = min(2 * s + gg, (uint32_t)G - 1);
            alo[S][gg] = g_load128(rA, oA, g * sA);
            if constexpr (F6ACT) ahi[S][gg] = g_load64(rA, l8, g * sA);
            as[S][gg] = g_load16(rS, oS, (g >> 3) * s8 + (g & 7) * s1);
        }
#pragma unroll
        for (int bn = 0; bn < NBN; bn++) ws[S][bn] = __builtin_amdgcn_raw_buffer_load_b32(rX, (int)oX, (int)(xblk[bn] + s * AUX_BLK), 0);
#pragma unroll
        for (int bn = 0; bn < NBN; bn++)
#pragma unroll
            for (int p = 0; p < WPL_BLOCKS; p++)
                w[S][bn][p] = g_load128(rW, l16, wblk[bn] + s * (uint32_t)(WPL_BLOCKS * BLK_BYTES) + (uint32_t)(p * BLK_BYTES));
        __builtin_amdgcn_sched_barrier(0);
    };

    v16f acc[NBN];
#pragma unroll
    for (int bn = 0; bn < NBN; bn++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[bn][i] = 0.0f;
    const v16f z16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    auto compute = [&](auto set_tag) {
        constexpr int S = decltype(set_tag)::value;
        // scale product of group gg: the activation side carries its scale in that group's K slot and zeros elsewhere
        const v2i sa[2] = {(v2i){half ? 0 : (int)as[S][0], 0}, (v2i){half ? 0 : (int)((uint32_t)as[S][1] << 16), 0}};
        v8i am[2];
#pragma unroll
        for (int gg = 0; gg < 2; gg++) {
            if constexpr (F6ACT) {
                am[gg] = (v8i){alo[S][gg][0], alo[S][gg][1], alo[S][gg][2], alo[S][gg][3], ahi[S][gg][0], ahi[S][gg][1], 0, 0};
            } else {  // even nibbles, then odd ones, as in gemm_w4a4_f8_kernel
                const v4i e = alo[S][gg] & 0x0F0F0F0F, o = (alo[S][gg] >> 4) & 0x0F0F0F0F;
                am[gg] = (v8i){e[0], e[1], e[2], e[3], o[0], o[1], o[2], o[3]};
            }
        }
#pragma unroll
        for (int b = 0; b < 2 * NBN; b++) {
            const int gg = b & 1, bn = b >> 1;
            const v8i w6 = {w[S][bn][gg][0], w[S][bn][gg][1], w[S][bn][gg][2], w[S][bn][gg][3], w[S][bn][2][2 * gg], w[S][bn][2][2 * gg + 1], 0, 0};
            const v16f sc = mfma32_16bit_k8<T>((v2i){ws[S][bn], 0}, sa[gg], z16);
            v16f p;
            if constexpr (F6ACT)
                p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w6, am[gg], z16, 2, 2, 0, F6_SCALE, 0, F6_SCALE);
            else
                p = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w6, am[gg], z16, 2, 0, 0, F6_SCALE, 0, F8_SCALE);
#pragma unroll
            for (int i = 0; i < 16; i++) acc[bn][i] = __builtin_fmaf(p[i], sc[i], acc[bn][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<int, 0> S0;
    const std::integral_constant<int, 1> S1;
    if (count > 0) load(S0, 0);
    if (wave < NWAVES) fetch_epilogue_operands<EPI>(a, sepi, n0, wave, lane);
    int i = 0;
    for (; i + 1 < count; i += 2) {  // past the end: the last stage again
        load(S1, i + 1);
        compute(S0);
        load(S0, min(i + 2, count - 1));
        compute(S1);
    }
    if (i < count) compute(S0);

    // ---- partial sums: block bn of wavefront v lands at slot (bn, v < bn ? v : v - 1) ----------------------------------
#pragma unroll
    for (int bn = 0; bn < NBN; bn++)
        if (bn != wave) {
            uint8_t *p = sred + (bn * (WAVES - 1) + (wave < bn ? wave : wave - 1)) * SK_BLOCK_BYTES + lane * 16;
#pragma unroll
            for (int j = 0; j < 4; j++) *(v4f *)(p + j * 1024) = (v4f){acc[bn][4 * j], acc[bn][4 * j + 1], acc[bn][4 * j + 2], acc[bn][4 * j + 3]};
        }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));  // (also: this wavefront's share of the epilogue operands has landed)
    __syncthreads();
    if (wave < NBN) {
        v16f mine = acc[0];
#pragma unroll
        for (int bn = 1; bn < NBN; bn++)
            if (bn == wave) mine = acc[bn];
        uint8_t *p = sred + wave * (WAVES - 1) * SK_BLOCK_BYTES + lane * 16;
#pragma unroll
        for (int v = 0; v < WAVES - 1; v++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f t = *(const v4f *)(p + v * SK_BLOCK_BYTES + j * 1024);
#pragma unroll
                for (int e = 0; e < 4; e++) mine[4 * j + e] += t[e];
            }
        if (wave != 0) {
#pragma unroll
            for (int j = 0; j < 4; j++) *(v4f *)(p + j * 1024) = (v4f){mine[4 * j], mine[4 * j + 1], mine[4 * j + 2], mine[4 * j + 3]};
        } else {
            acc[0] = mine;
        }
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int bn = 1; bn < NBN; bn++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const v4f t = *(const v4f *)(sred + bn * (WAVES - 1) * SK_BLOCK_BYTES + lane * 16 + j * 1024);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[bn][4 * j + e] = t[e];
        }
    // block 0's slots (12 KB or more) were read before the second barrier: wavefront 0's private epilogue memory
    static_assert(PRIV_BYTES <= (WAVES - 1) * SK_BLOCK_BYTES, "the epilogue's private memory must not reach the sums of block 1");
    tile_epilogue<T, EPI, true>(a, acc, sred, sepi, m0, n0, pid_n, 0, lane);
}

// The same over 64 rows x 128 columns: eight wavefronts, of which four split K over the left and four over the right 64 columns.
// A wavefront owns 64 x 64, so an operand that comes from L2 feeds two matrix instructions, and two steps' matrix instructions and FMAs
// overlap (two sets of result registers).  SB: activation scales in the loop's order (with F6ACT).
//
// What bounds it: the issue of loads.  They are replaced where they are used up (a weight or activation operand by that of the
// wavefront's next stage), and scales come for two stages at a time: the lanes of one half hold the scales of a stage, those of the other
// half the scales of the wavefront's next one, and the activation side is zero in the half whose stage it is not.  (One load per
// stage and scale, of lanes that all hold the same: 512 x 3072, K = 12288 40.2 us, 29.0 without scales.)
// us, 32-row workgroups / these (bf16, rank 32, fp6 codes with blocked scales): K = 3072: 512 x 3072 14.8 / 11.4, 333 x 4096 14.7 / 11.4,
// 64 x 18432 17.4 / 13.1; K = 12288: 333 x 3072 40.4 / 31.0, 512 x 3072 41.4 / 31.2; K = 2048: 1000 x 2048 12.1 / 9.5.  Of the 31.2 the
// matrix instructions and FMAs alone are 20.  Partial sums added pairwise by half of the wavefronts, then a quarter, with three barriers
// instead of two: 512 x 3072 at K = 3072 12.1, at K = 12288 31.9.
template <typename T, int EPI, bool F6ACT, bool SB>
__global__ __launch_bounds__(512, 2) void gemm_w4a4_split64_kernel(svdq_gemm_args a, int tiles_m) {
    static_assert(F6ACT || !SB, "blocked scales come with fp6 codes");
    constexpr int RB = 2, CB = 2, WC = NBN / CB, KS = 8 / WC;  // blocks of a wavefront, column halves, wavefronts that split K
    __shared__ __align__(16) uint8_t sred[KS * RB * NBN * SK_BLOCK_BYTES];  // [wavefront along K][row block][column block]
    __shared__ __align__(16) uint8_t sepi[EPI_LDS_BYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wc = wave % WC, ks = wave / WC;
    const int l32 = lane & 31, half = lane >> 5;

    // XCD-contiguous renumbering, then the row blocks of a column tile in a row
    const int nb = gridDim.x, xcd = blockIdx.x % NUM_XCD, loc = blockIdx.x / NUM_XCD;
    const int id = xcd * (nb / NUM_XCD) + min(xcd, nb % NUM_XCD) + loc;
    const int pid_m = id % tiles_m, pid_n = id / tiles_m;
    const int m0 = pid_m * 32 * RB, n0 = pid_n * BN;
    const int G = a.K / GROUP, nst = (G + 1) / 2;
    const int count = (nst - ks + KS - 1) / KS;  // this wavefront's stages, two at least (split64_takes)

    // column blocks past N and row blocks past M re-read the last one (their outputs are never stored)
    const int blast = (a.N + 31) / 32 - 1, b0 = min(n0 / 32 + wc * CB, blast);
    const __amdgpu_buffer_rsrc_t rW = g_buffer((const uint8_t *)a.wgt_planes + (size_t)b0 * nst * (WPL_BLOCKS * BLK_BYTES));
    const __amdgpu_buffer_rsrc_t rX =
        g_buffer((const uint8_t *)a.wgt_planes + planes_code_bytes(a.N, a.K) + (size_t)b0 * (nst + 1) * AUX_BLK);
    const bool ablk = F6ACT || a.act_blocked != 0;
    const uint32_t sA = F6ACT ? 1536u : ablk ? 1024u : 32u;  // a step of one group
    const int mblast = (a.M - 1) >> 5, mb0 = m0 >> 5;
    const __amdgpu_buffer_rsrc_t rA = g_buffer((const uint8_t *)a.act + (ablk ? (size_t)mb0 * G * sA : (size_t)m0 * a.ld_act));
    const __amdgpu_buffer_rsrc_t rS = g_buffer((const uint8_t *)a.ascales + (SB ? (size_t)mb0 * (G >> 3) * 512 : 0));
    const uint32_t l16 = (uint32_t)lane * 16u, l8 = 1024u + (uint32_t)lane * 8u;
    uint32_t oA[RB], uA[RB], oS[RB], wblk[CB], xblk[CB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        const int blk = min(mb0 + rb, mblast), row = min(blk * 32 + l32, a.M - 1);
        uA[rb] = ablk ? (uint32_t)(blk - mb0) * (uint32_t)G * sA : 0u;
        oA[rb] = ablk ? l16 : (uint32_t)(row - m0) * (uint32_t)a.ld_act + half * 16;
        oS[rb] = SB ? (uint32_t)(blk - mb0) * (uint32_t)(G >> 3) * 512u + (uint32_t)l32 * 16u : 2u * (uint32_t)row;
    }
#pragma unroll
    for (int bn = 0; bn < CB; bn++) {
        const uint32_t b = (uint32_t)(min(n0 / 32 + wc * CB + bn, blast) - b0);
        wblk[bn] = b * (uint32_t)nst * (uint32_t)(WPL_BLOCKS * BLK_BYTES);
        xblk[bn] = b * (uint32_t)(nst + 1) * (uint32_t)AUX_BLK;
    }

    v4i w[CB][WPL_BLOCKS], alo[2][RB];
    v2i ahi[2][RB];
    int ws[2][CB], as2[2][RB];       // [set of two stages]; as2: both groups' scales (SB)
    uint16_t as1[2][2][RB];          // likewise one by one
    auto stage_of = [&](int i) { return (uint32_t)(min(i, count - 1) * KS + ks); };  // past the end: the last one again
    auto load_w = [&](int i, int bn, int p) {
        w[bn][p] = g_load128(rW, l16, wblk[bn] + stage_of(i) * (uint32_t)(WPL_BLOCKS * BLK_BYTES) + (uint32_t)(p * BLK_BYTES));
    };
    auto load_a = [&](int i, int gg, int rb) {  // a group past the end (K / 64 odd) re-reads the last one: its weights are zeros
        const uint32_t g = min(2 * stage_of(i) + gg, (uint32_t)G - 1);
        alo[gg][rb] = g_load128(rA, oA[rb], uA[rb] + g * sA);
        if constexpr (F6ACT) ahi[gg][rb] = g_load64(rA, l8, uA[rb] + g * sA);
    };
    auto load_scales = [&](int i, int set) {  // of stages i and i + 1
        const uint32_t s = half ? stage_of(i + 1) : stage_of(i);
        const uint32_t oX = (uint32_t)l32 * AUX_ROW + 8u + s * (uint32_t)AUX_BLK;
#pragma unroll
        for (int bn = 0; bn < CB; bn++) ws[set][bn] = __builtin_amdgcn_raw_buffer_load_b32(rX, (int)oX, (int)xblk[bn], 0);
        if constexpr (SB) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++) as2[set][rb] = __builtin_amdgcn_raw_buffer_load_b32(rS, (int)(oS[rb] + (s >> 2) * 512u + (s & 3u) * 4u), 0, 0);
        } else {
#pragma unroll
            for (int gg = 0; gg < 2; gg++) {
                const uint32_t o = min(2 * s + gg, (uint32_t)G - 1) * 2u * (uint32_t)a.ld_ascales;
#pragma unroll
                for (int rb = 0; rb < RB; rb++) as1[set][gg][rb] = g_load16(rS, oS[rb] + o, 0);
            }
        }
    };

    v16f acc[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int bn = 0; bn < CB; bn++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[rb][bn][i] = 0.0f;
    const v16f z16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    constexpr int NQ = 2 * CB * RB;  // steps of a stage: (group, column block, row block)
    v16f P[2], S[2];
    auto scales = [&](int q, int set, int par) -> v16f {  // par: first or second stage of the set
        const int gg = q / (CB * RB), bn = (q / RB) % CB, rb = q % RB;
        uint32_t v;
        if constexpr (SB)
            v = gg ? (uint32_t)as2[set][rb] & 0xFFFF0000u : (uint32_t)as2[set][rb] & 0xFFFFu;
        else
            v = gg ? (uint32_t)as1[set][1][rb] << 16 : (uint32_t)as1[set][0][rb];
        return mfma32_16bit_k8<T>((v2i){ws[set][bn], 0}, (v2i){half == par ? (int)v : 0, 0}, z16);
    };
    auto group = [&](int q) -> v16f {
        const int gg = q / (CB * RB), bn = (q / RB) % CB, rb = q % RB;
        const v8i w6 = {w[bn][gg][0], w[bn][gg][1], w[bn][gg][2], w[bn][gg][3], w[bn][2][2 * gg], w[bn][2][2 * gg + 1], 0, 0};
        if constexpr (F6ACT) {
            const v8i am = {alo[gg][rb][0], alo[gg][rb][1], alo[gg][rb][2], alo[gg][rb][3], ahi[gg][rb][0], ahi[gg][rb][1], 0, 0};
            return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w6, am, z16, 2, 2, 0, F6_SCALE, 0, F6_SCALE);
        } else {  // even nibbles, then odd ones, as in gemm_w4a4_f8_kernel
            const v4i e = alo[gg][rb] & 0x0F0F0F0F, o = (alo[gg][rb] >> 4) & 0x0F0F0F0F;
            const v8i am = {e[0], e[1], e[2], e[3], o[0], o[1], o[2], o[3]};
            return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w6, am, z16, 2, 0, 0, F6_SCALE, 0, F8_SCALE);
        }
    };
    auto stage = [&](auto par_tag, auto set_tag, int i) {
        constexpr int PAR = decltype(par_tag)::value, SET = decltype(set_tag)::value;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int gg = q / (CB * RB), bn = (q / RB) % CB, rb = q % RB, c = q & 1, n = c ^ 1;
            const bool last = q == NQ - 1;
            if (!last) P[n] = group(q + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (PAR == 0 && q == 0) load_scales(i + 2, SET ^ 1);
            if (rb == RB - 1) {
                load_w(i + 1, bn, gg);
                if (gg == 1) load_w(i + 1, bn, 2);
            }
            if (bn == CB - 1) load_a(i + 1, gg, rb);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 8; e++) acc[rb][bn][e] = __builtin_fmaf(P[c][e], S[c][e], acc[rb][bn][e]);
            __builtin_amdgcn_sched_barrier(0);
            S[n] = last ? scales(0, PAR ? SET ^ 1 : SET, PAR ^ 1) : scales(q + 1, SET, PAR);
            if (last) P[n] = group(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 8; e < 16; e++) acc[rb][bn][e] = __builtin_fmaf(P[c][e], S[c][e], acc[rb][bn][e]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    const std::integral_constant<int, 0> I0;
    const std::integral_constant<int, 1> I1;
    load_scales(0, 0);
#pragma unroll
    for (int gg = 0; gg < 2; gg++) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) load_a(0, gg, rb);
#pragma unroll
        for (int bn = 0; bn < CB; bn++) {
            load_w(0, bn, gg);
            if (gg == 0) load_w(0, bn, 2);
        }
    }
    if (wave < NWAVES) fetch_epilogue_operands<EPI>(a, sepi, n0, wave, lane);
    S[0] = scales(0, 0, 0);
    P[0] = group(0);
    int i = 0;
    for (; i + 3 < count; i += 4) {
        stage(I0, I0, i);
        stage(I1, I0, i + 1);
        stage(I0, I1, i + 2);
        stage(I1, I1, i + 3);
    }
    const int left = count - i;  // 0 .. 3
    if (left >= 1) stage(I0, I0, i);
    if (left >= 2) stage(I1, I0, i + 1);
    if (left >= 3) stage(I0, I1, i + 2);

    // ---- partial sums: every wavefront adds up one block, in the order of gemm_w4a4_split_kernel (of column block bn: wavefront bn's
    // first, then the others'), so that an output has the same bits as there; then a row block to a wavefront
    auto slot = [&](int k, int r, int b) { return sred + ((k * RB + r) * NBN + b) * SK_BLOCK_BYTES + lane * 16; };
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int bn = 0; bn < CB; bn++) {
            uint8_t *p = slot(ks, rb, wc * CB + bn);
#pragma unroll
            for (int j = 0; j < 4; j++) *(v4f *)(p + j * 1024) = (v4f){acc[rb][bn][4 * j], acc[rb][bn][4 * j + 1], acc[rb][bn][4 * j + 2], acc[rb][bn][4 * j + 3]};
        }
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));  // (also: this wavefront's share of the epilogue operands has landed)
    __syncthreads();
    {
        static_assert(KS == RB * CB && KS == NBN, "a block to a wavefront, a wavefront along K that a column block's sum begins with");
        const int rb = ks / CB, b = wc * CB + ks % CB;
        v4f sum[4];
#pragma unroll
        for (int j = 0; j < 4; j++) sum[j] = *(const v4f *)(slot(b, rb, b) + j * 1024);
#pragma unroll
        for (int v = 0; v < KS - 1; v++) {
            const uint8_t *p = slot(v < b ? v : v + 1, rb, b);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f t = *(const v4f *)(p + j * 1024);
#pragma unroll
                for (int e = 0; e < 4; e++) sum[j][e] += t[e];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) *(v4f *)(slot(0, rb, b) + j * 1024) = sum[j];
    }
    __syncthreads();
    if (wave >= RB || m0 + 32 * wave >= a.M) return;
    v16f mine[NBN];
#pragma unroll
    for (int bn = 0; bn < NBN; bn++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const v4f t = *(const v4f *)(slot(0, wave, bn) + j * 1024);
#pragma unroll
            for (int e = 0; e < 4; e++) mine[bn][4 * j + e] = t[e];
        }
    static_assert(PRIV_BYTES <= NBN * SK_BLOCK_BYTES, "the epilogue's private memory lies in the row block's own sums");
    tile_epilogue<T, EPI, true>(a, mine, sred + wave * NBN * SK_BLOCK_BYTES, sepi, m0, n0, pid_n, wave, lane);
}

template <typename T, int WAVES, bool F6ACT>
static void launch_split(const svdq_gemm_args &a, int tiles_m, hipStream_t s) {
    const dim3 grid((unsigned)tiles_m * (unsigned)((a.N + BN - 1) / BN)), block(WAVES * 64);
    switch (a.epilogue) {
        case SVDQ_EPI_PLAIN:
            hipLaunchKernelGGL((gemm_w4a4_split_kernel<T, SVDQ_EPI_PLAIN, WAVES, F6ACT>), grid, block, 0, s, a, tiles_m);
            break;
        case SVDQ_EPI_QK_NORM_ROPE:
            hipLaunchKernelGGL((gemm_w4a4_split_kernel<T, SVDQ_EPI_QK_NORM_ROPE, WAVES, F6ACT>), grid, block, 0, s, a, tiles_m);
            break;
        case SVDQ_EPI_GELU_QUANT:
            hipLaunchKernelGGL((gemm_w4a4_split_kernel<T, SVDQ_EPI_GELU_QUANT, WAVES, F6ACT>), grid, block, 0, s, a, tiles_m);
            break;
        case SVDQ_EPI_SWIGLU_QUANT:
            hipLaunchKernelGGL((gemm_w4a4_split_kernel<T, SVDQ_EPI_SWIGLU_QUANT, WAVES, F6ACT>), grid, block, 0, s, a, tiles_m);
            break;
    }
}

// Row blocks a launch has to run: the requantizing epilogues write all M rows, the others those below actual_m only.
static int row_blocks(const svdq_gemm_args &a) {
    const bool quant = a.epilogue == SVDQ_EPI_GELU_QUANT || a.epilogue == SVDQ_EPI_SWIGLU_QUANT;
    return ((quant ? a.M : a.actual_m) + 31) / 32;
}

template <typename T, bool F6ACT, bool SB>
static void launch_split64(const svdq_gemm_args &a, int tiles_m, hipStream_t s) {
    const dim3 grid((unsigned)tiles_m * (unsigned)((a.N + BN - 1) / BN)), block(512);
    switch (a.epilogue) {
        case SVDQ_EPI_PLAIN:
            hipLaunchKernelGGL((gemm_w4a4_split64_kernel<T, SVDQ_EPI_PLAIN, F6ACT, SB>), grid, block, 0, s, a, tiles_m);
            break;
        case SVDQ_EPI_QK_NORM_ROPE:
            hipLaunchKernelGGL((gemm_w4a4_split64_kernel<T, SVDQ_EPI_QK_NORM_ROPE, F6ACT, SB>), grid, block, 0, s, a, tiles_m);
            break;
        case SVDQ_EPI_GELU_QUANT:
            hipLaunchKernelGGL((gemm_w4a4_split64_kernel<T, SVDQ_EPI_GELU_QUANT, F6ACT, SB>), grid, block, 0, s, a, tiles_m);
            break;
        case SVDQ_EPI_SWIGLU_QUANT:
            hipLaunchKernelGGL((gemm_w4a4_split64_kernel<T, SVDQ_EPI_SWIGLU_QUANT, F6ACT, SB>), grid, block, 0, s, a, tiles_m);
            break;
    }
}

// Workgroups of 64 rows, of those launches that split K over four wavefronts, where all of them find a CU of their own (beyond that the
// 32-row ones, two to a CU, divide the rows better) and every wavefront has two stages (with one the refills in it are for nothing; the
// kernel relies on it).  Time against
// the 32-row workgroups over 687 launches of 64 to 2048 rows, both types, PLAIN | GELU at rank 128: K = 128 1.00 to 1.06 | 1.00 to 1.03, 512
// 1.08 to 1.15 | 1.02 to 1.06, 1024 0.89 to 0.92 | 0.86 to 0.95, 3072 0.78 to 0.84 | 0.79 to 0.90, 12288 0.75 to 0.81 | 0.75 to 0.81.
static bool split64_takes(const svdq_gemm_args &a, int cus) {
    return a.K > 14 * GROUP && (long)((row_blocks(a) + 1) / 2) * ((a.N + BN - 1) / BN) <= cus;
}

template <typename T>
static void launch_split_type(const svdq_gemm_args &a, int wavefronts, int cus, hipStream_t s) {
    const int tiles_m = row_blocks(a), pairs = (tiles_m + 1) / 2;
    if (wavefronts == 4 && split64_takes(a, cus)) {
        if (a.act_blocked != 2)
            launch_split64<T, false, false>(a, pairs, s);
        else if (a.ascales_blocked)
            launch_split64<T, true, true>(a, pairs, s);
        else
            launch_split64<T, true, false>(a, pairs, s);
    } else if (a.act_blocked == 2) {
        wavefronts == 8 ? launch_split<T, 8, true>(a, tiles_m, s) : launch_split<T, 4, true>(a, tiles_m, s);
    } else {
        wavefronts == 8 ? launch_split<T, 8, false>(a, tiles_m, s) : launch_split<T, 4, false>(a, tiles_m, s);
    }
}

// Rows and columns: two workgroups of 32 rows fit a CU (256 registers a wavefront).  Up to that many the split is faster than the tiles,
// beyond it each further round streams the weight tiles again.  The lines of this rule were measured on 32-row workgroups of four
// wavefronts; those of 64 rows are faster still.  PLAIN launch in us, 32-row workgroups / the faster tile build (bf16, rank 32):
//   K = 3072,  N = 3072:  512 rows (384 workgroups) 15.5 / 18.3;  768 rows (576) 24.2 / 18.5
//   K = 12288, N = 3072:  512 rows 42.1 / 63.4;  768 rows 70.7 / 63.5
//   K = 2048,  N = 2048:  1024 rows (512) 13.5 / 13.7;  1536 rows (768) 20.0 / 14.0
// With at most one workgroup per CU eight wavefronts share its K, so that every SIMD still has two (K = 12288, N = 3072, 256
// rows: 26.2 us with eight, 32.9 with four, 64.0 as tiles; K = 6144, N = 1536, 512 rows: 16.5, 19.1, 32.6).
//
// K and rank: the exchange of the partial tiles costs 0.6 us, which the split has to save elsewhere: on the loop, where K is
// long, or on the low-rank product, whose serial steps over 16 ranks each more and smaller workgroups run faster.  Time against
// the tiles, PLAIN, 256 x 3072 (eight wavefronts) | 512 x 3072 (four, which run more stages each beside a second workgroup):
//   rank 32:  K = 128 1.10 | 1.11;  256 1.01 | 1.08;  512 0.92 | 1.01;  1024 0.78 | 1.14;  1280 0.75 | 0.99;  2048 0.77 | 0.96
//   rank 64:  K = 128 0.97 | 1.05;  256 0.91 | 1.00;  512 0.85 | 0.93;  1024 0.74 | 1.06;  1280 0.72 | 0.94;  2048 0.74 | 0.94
//   rank 128: K = 128 0.82 | 0.91;  256 0.79 | 0.88;  512 0.75 | 0.84;  1024 0.68 | 0.95;  1280 0.67 | 0.86;  2048 0.69 | 0.89
// The other epilogues lie within 0.1 of these.  At rank 32 and four wavefronts SwiGLU wins from K = 1280 on (0.97), Q/K norm +
// RoPE from 1344 (0.95; 1280 1.01), GELU from 1600 (0.98; 1536 1.02, and 1.04 at rank 16).  The dips at K = 1024 and 2048 lie at
// column blocks of a weight tile 24 and 48 KB apart; the second one counts for Q/K norm + RoPE (1.05) and GELU (1.03) only.
int split_wavefronts(const svdq_gemm_args &a, int cus) {
    const long wgs = (long)row_blocks(a) * ((a.N + BN - 1) / BN);
    if (wgs > 2L * cus || (uint64_t)NBN * (a.K / 128 + 1) * (WPL_BLOCKS * BLK_BYTES) >= (1ull << 32)) return 0;
    const int stages = (a.K / GROUP + 1) / 2;
    const bool gelu = a.epilogue == SVDQ_EPI_GELU_QUANT, swiglu = a.epilogue == SVDQ_EPI_SWIGLU_QUANT, qk = a.epilogue == SVDQ_EPI_QK_NORM_ROPE;
    const int rank = gelu || swiglu ? std::min(a.R, a.R2) : a.R;
    if (wgs <= cus) return stages >= 3 || rank >= 64 ? 8 : 0;
    if (rank >= 128) return 4;
    const int from = rank >= 64 ? 3 : gelu ? 13 : qk ? 11 : 10;
    return stages >= from && stages != 8 && !(stages == 16 && (gelu || qk)) ? 4 : 0;
}

void launch_gemm_split(const svdq_gemm_args &a, int wavefronts, int cus, hipStream_t s) {
    if (a.dtype == SVDQ_BF16)
        launch_split_type<BF16>(a, wavefronts, cus, s);
    else
        launch_split_type<FP16>(a, wavefronts, cus, s);
}

}  // namespace svdq
