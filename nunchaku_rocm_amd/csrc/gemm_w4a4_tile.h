// What the W4A4 GEMM kernels share: tile geometry, the layout of pre-split weights, buffer loads, and the epilogues.
#pragma once

#include "svdq_common.h"

namespace svdq {

constexpr int BM = 128, BN = 128;     // workgroup tile (activation rows x weight rows)
constexpr int KSTAGE = 128;           // K per LDS stage = two scale groups
constexpr int BLK_BYTES = 64 * 16;    // one MFMA operand block (32 rows x 16 bytes per lane) of one group, lane-linear
constexpr int NWAVES = 4, NTHREADS = NWAVES * 64;  // one wavefront per 32 activation rows
constexpr int NBN = BN / 32;                        // 32-row weight blocks per wavefront: it owns 32 x 128 outputs
// the first 32 ranks of the tile's lora_up, fetched next to stage 0: [2 c][4 blocks] 1 KB blocks in MFMA lane order,
// then the tile's 128 bias values, then the 128 RMSNorm weights of the tile's head (Q/K norm + RoPE epilogue)
constexpr int LORA_UP_BYTES = 8 * BLK_BYTES;
constexpr int EPI_NORM_OFF = LORA_UP_BYTES + BN * 2;
constexpr int EPI_LDS_BYTES = EPI_NORM_OFF + 128 * 2;
constexpr int TP_PITCH = 36;                        // floats per row of the accumulator transposition tile
constexpr int PRIV_BYTES = 32 * BN * 2;             // a wavefront's private epilogue memory: its 32 output rows of 256 bytes
static_assert(32 * TP_PITCH * 4 <= PRIV_BYTES, "the transposition tile of one block does not fit");
constexpr int GROUP_M_TILES = 8;      // m-tiles per raster band
constexpr int NUM_XCD = 8;

// ---- fp8 kernel
constexpr int F8_SCALE = (int)0x88888888;  // e8m0 block scale 2^9 in every byte: an fp8 code c (value c * 2^-9) counts as c
constexpr int F6_SCALE = (int)0x82828282;  // e8m0 block scale 2^3: an fp6 (e2m3) code c <= 15 (value c / 8) counts as c
// Pre-split weights, per (block of 32 rows, stage of two groups): three 1 KB blocks in MFMA lane order.  A lane's 32
// weights of a group are 32 six-bit codes = six registers: blocks 0 and 1 hold registers 0-3 of the stage's first and
// second group (16 bytes per lane), block 2 registers 4-5 of both (8 + 8 bytes per lane).
constexpr int WPL_BLOCKS = 3;
constexpr int F8_STAGE_BYTES = NBN * WPL_BLOCKS * BLK_BYTES;  // 12288
// ... and, per (block of 32 rows, stage), 32 rows of six 16-bit values: the two pieces (hi + lo) of
// D = -ws * (8 * sum of the group's even weights - 7 * sum of its odd weights) for the stage's two groups, then the two
// weight scales.  A 12-byte-per-lane global -> LDS load puts lane l's bytes at 16 l, so in LDS a row takes 16 bytes; they
// sit in a ring of eight stages per block; one load brings a stage and the one after it (64 lanes = two stages' rows)
// into an even slot and its neighbour.
constexpr int AUX_ROW = 12;                                  // bytes per row and stage in memory
constexpr int AUX_BLK = 32 * AUX_ROW;                        // 384
constexpr int AUX_LROW = 16;                                 // ... and in LDS
constexpr int AUX_LBLK = 32 * AUX_LROW;                      // 512
constexpr int AUX_SLOTS = 8;
constexpr int AUX_NBLK_BYTES = AUX_SLOTS * AUX_LBLK;         // 4096
constexpr int F8_RING_BYTES = NBN * AUX_NBLK_BYTES;          // 16384: after the loop two wavefronts' private memory
static_assert(2 * PRIV_BYTES <= F8_RING_BYTES, "two wavefronts' private epilogue memory must fit the ring");
static_assert(PRIV_BYTES <= F8_STAGE_BYTES, "a wavefront's private epilogue memory must fit a staging buffer");
constexpr int PLANES_STATUS_BYTES = 16;  // trailing status word of a pre-split weight

__host__ __device__ inline size_t planes_code_bytes(int N, int K) {
    return (size_t)((N + 31) / 32) * (size_t)((K / GROUP + 1) / 2) * (WPL_BLOCKS * BLK_BYTES);
}
__host__ __device__ inline size_t planes_aux_bytes(int N, int K) {  // one stage of padding per block of rows
    return (size_t)((N + 31) / 32) * (size_t)((K / GROUP + 1) / 2 + 1) * AUX_BLK;
}

// Register loads of the fp8 loop go through raw buffers: address = descriptor base + scalar offset (the group or stage)
// + 32-bit lane offset, so no vector instruction computes an address.  The range covers everything (offsets are clamped
// where rows or columns run out).
__device__ inline __amdgpu_buffer_rsrc_t g_buffer(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)0xFFFFFFFFu, 0x00020000);  // raw buffer, 32-bit data format
}
__device__ inline uint16_t g_load16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, (int)lane_off, (int)uniform_off, 0);
}
__device__ inline v4i g_load128(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_off, (int)uniform_off, 0));
}

__device__ inline v2i g_load64(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    return __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(r, (int)lane_off, (int)uniform_off, 0));
}

// Block loads global -> LDS through a raw buffer: the 64 lanes' 16 (or 12) bytes at base + lane offset + scalar offset land at
// lds + 16 * lane; base and scalar offset live in SGPRs, so the loop's block loads need no vector address arithmetic.
__device__ inline void g_load16_lds(__amdgpu_buffer_rsrc_t r, uint8_t *lds, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (SVDQ_AS3 void *)lds, 16, (int)lane_off, (int)uniform_off, 0, 0);
}
__device__ inline void g_load4_lds(__amdgpu_buffer_rsrc_t r, uint8_t *lds, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (SVDQ_AS3 void *)lds, 4, (int)lane_off, (int)uniform_off, 0, 0);
}
__device__ inline void g_load12_lds(__amdgpu_buffer_rsrc_t r, uint8_t *lds, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (SVDQ_AS3 void *)lds, 12, (int)lane_off, (int)uniform_off, 0, 0);
}

// (pid_m, pid_n) of this workgroup: XCD-contiguous renumbering, then m-banded raster.
__device__ inline void tile_ids(int tiles_m, int tiles_n, int &pid_m, int &pid_n) {
    const int nb = gridDim.x;
    const int bid = blockIdx.x;
    const int xcd = bid % NUM_XCD, loc = bid / NUM_XCD;
    const int per = (nb + NUM_XCD - 1) / NUM_XCD, rem = nb % NUM_XCD;
    const int start = (rem == 0 || xcd < rem) ? xcd * per : rem * per + (xcd - rem) * (per - 1);
    const int id = start + loc;
    const int band = GROUP_M_TILES * tiles_n;
    const int first_m = (id / band) * GROUP_M_TILES;
    const int gm = min(tiles_m - first_m, GROUP_M_TILES);
    pid_m = first_m + (id % band) % gm;
    pid_n = (id % band) / gm;
}

// Row strides of lora_up below this: the offsets of 32 of its rows fit 32 bits.
constexpr int LORA_UP_LD32 = 1 << 26;

// Epilogue operands every wavefront of the tile needs, fetched global -> LDS next to stage 0: the tile's 128 bias
// values, the first 32 ranks of lora_up and (Q/K norm + RoPE epilogue, Q and K tiles) the head's 128 norm weights.
// (Buffer loads: next to a global_load_lds in flight the compiler waits for every load before the first register load's
// use in a loop that follows.)
template <int EPI>
__device__ inline void fetch_epilogue_operands(const svdq_gemm_args &a, uint8_t *sepi, int n0, int wm, int lane) {
    const int l32 = lane & 31, half = lane >> 5;
    if constexpr (EPI == SVDQ_EPI_QK_NORM_ROPE) {
        const int part = n0 / (a.N / 3);
        if (part < 2 && wm == 2)  // 64 lanes x 4 bytes
            g_load4_lds(g_buffer(part == 0 ? a.norm_q : a.norm_k), sepi + EPI_NORM_OFF, 4u * (uint32_t)lane, 0);
    }
    if (a.bias != nullptr && wm == 3)  // 64 lanes x 4 bytes = the tile's 128 bias values
        g_load4_lds(g_buffer((const uint16_t *)a.bias + n0), sepi + LORA_UP_BYTES, 2u * (uint32_t)min(2 * lane, a.N - 2 - n0), 0);
    if (a.R > 0) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int q = wm * 2 + i, c = q >> 2, blk = q & 3;  // wave-uniform
            const int r0 = min(n0 + blk * 32, a.N - 1);         // the block's first row: its rows are 32-bit offsets from there
            const __amdgpu_buffer_rsrc_t r = g_buffer((const uint16_t *)a.lora_up + (size_t)r0 * a.ld_lora_up);
            const uint32_t row = (uint32_t)(min(n0 + blk * 32 + l32, a.N - 1) - r0);
            if (16 * c >= a.R) continue;
            if (__builtin_expect(a.ld_lora_up < LORA_UP_LD32, 1)) {
                g_load16_lds(r, sepi + q * BLK_BYTES, row * 2u * (uint32_t)a.ld_lora_up + (uint32_t)(32 * c + 16 * half), 0);
            } else {  // rows too far apart: one by one (a lane's 16 bytes land at its place whoever else is masked off; through registers
                      // the fp8 loop's kernels spill up to three more)
#pragma unroll 1
                for (int i32 = 0; i32 < 32; i32++)
                    if (l32 == i32)
                        g_load16_lds(g_buffer((const uint16_t *)a.lora_up + (size_t)min(r0 + i32, a.N - 1) * a.ld_lora_up), sepi + q * BLK_BYTES,
                                     (uint32_t)(32 * c + 16 * half), 0);
            }
        }
    }
}

// Requantized activations as fp6 codes in the consuming GEMM's lane order (qout_blocked == 2).  A lane of the epilogue
// owns, of its row's group of 64 values, the runs k = 8 t + 4 half .. + 3 (t = 0 .. 7): codes p = 4 t + 2 half, + 1 of the
// consuming lane of K half 0 (its even k) and the same codes of the lane of K half 1 (its odd k), i.e. one 12-bit piece
// per t and consuming lane, at bit 24 t + 12 half of that lane's 192.  f6_pack_unit places four pieces (96 bits);
// f6_swap_unit trades the two half-filled units with lane ^ 32 (all lanes of the wavefront must be active) -- every lane
// ends up with all of one consuming lane's 24 bytes -- and f6_store writes their first 16 at 16 l and their last 8 at
// 1024 + 8 l of the (row block, group)'s 1536, l = 32 half + row % 32.
__device__ inline void f6_pack_unit(uint32_t p0, uint32_t p1, uint32_t p2, uint32_t p3, uint32_t sh, uint32_t (&d)[3]) {
    const uint64_t lo = ((uint64_t)p0 | ((uint64_t)p1 << 24)) << sh, hi = ((uint64_t)p2 | ((uint64_t)p3 << 24)) << sh;
    d[0] = (uint32_t)lo;
    d[1] = (uint32_t)(lo >> 32) | ((uint32_t)hi << 16);
    d[2] = (uint32_t)(hi >> 16);
}
__device__ inline void f6_swap_unit(const uint32_t (&v0)[3], const uint32_t (&v1)[3], uint32_t *r) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const auto sw = __builtin_amdgcn_permlane32_swap(v0[i], v1[i], false, false);
        r[i] = sw[0] | sw[1];
    }
}
__device__ inline void f6_store(const uint32_t (&r)[6], uint8_t *blk, int lane, bool ok) {
    if (ok) {
        *(v4i *)(blk + 16 * lane) = (v4i){(int)r[0], (int)r[1], (int)r[2], (int)r[3]};
        *(v2i *)(blk + 1024 + 8 * lane) = (v2i){(int)r[4], (int)r[5]};
    }
}

// Everything after the main loop, for one wavefront: acc[bn][i] holds out[m = mw0 + 8 (i >> 2) + 4 half + (i & 3)]
// [n = n0 + 32 bn + lane % 32] without LoRA-up and bias -- or, with ROWS_IN_LANES (a main loop that passes the weights as
// the matrix instruction's first operand), out[m = mw0 + lane % 32][n = n0 + 32 bn + 8 (i >> 2) + 4 half + (i & 3)],
// which is the orientation every row-wise epilogue wants: the turn through LDS below is then not needed.  `priv` is PRIV_BYTES of LDS nobody else touches from here on;
// `sepi` holds what fetch_epilogue_operands brought.  No workgroup barrier inside.
template <typename T, int EPI, bool ROWS_IN_LANES = false>
__device__ __forceinline__ void tile_epilogue(const svdq_gemm_args &a, v16f (&acc)[NBN], uint8_t *priv, const uint8_t *sepi,
                                              int m0, int n0, int pid_n, int wm, int lane) {
    const int l32 = lane & 31, half = lane >> 5;
    const int mw0 = m0 + wm * 32;

    // Q/K RMSNorm + RoPE: the lane's rotary entries of a 32-column block are fetched two blocks ahead of their use, the
    // first two blocks' before the transposition (issued one load at a time next to the arithmetic, as the compiler orders
    // them under this register pressure, the sixteen dependent L2 round trips took 6 % of the launch); the head's norm
    // weights came into LDS next to stage 0.
    const int qk_part = EPI == SVDQ_EPI_QK_NORM_ROPE ? n0 / (a.N / 3) : 2;  // 0 = Q, 1 = K, 2 = V or no such epilogue
    v4f qk_sc[2][4];
    auto qk_fetch = [&](int bn, int buf) {
        if (a.rotary_blocked != nullptr) {
            // re-laid-out table: the 64 lanes of a load read 1 KB in a row.  (From the (rows, 128) table a load fetches
            // 32-byte pieces of 32 different rows; at the QKV shape that was 8 of the epilogue's 11 us.)
            const int rb = min(mw0 >> 5, (a.actual_m + 31) / 32 - 1);
            const v4f *p = (const v4f *)a.rotary_blocked + ((size_t)rb * 16 + bn * 4) * 64 + lane;
#pragma unroll
            for (int j = 0; j < 4; j++) qk_sc[buf][j] = p[j * 64];
            return;
        }
        const int m = mw0 + l32;
        const float *rot = a.rotary + (size_t)(m < a.actual_m ? m : 0) * a.ld_rotary;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int d = bn * 32 + 8 * j + 4 * half;  // channel within the head
            qk_sc[buf][j] = *(const v4f *)(rot + d);  // (sin, cos, sin, cos)
        }
    };


    // ---- LoRA-up and bias, still in the main loop's orientation (lane = weight row, registers = activation rows) ----
    // The bias and the first 32 ranks of lora_up were fetched into LDS next to stage 0 and arrived long ago; the
    // wavefront's own rows of lora_act and ranks beyond 32 come from global memory, all loads of a 32-rank pass issued
    // before their first use.  Rows past N / M hold copies of the last row: they only reach outputs that are never stored.
    if (a.R > 0) {
        const uint16_t *lu = (const uint16_t *)a.lora_up;
        const float *la = a.lora_act + (size_t)min(mw0 + l32, a.M - 1) * a.ld_lora_act + half * 8;
        for (int r0 = 0; r0 < a.R; r0 += 32) {
            const bool two = r0 + 16 < a.R;  // uniform: the second 16 ranks of this pass exist
            v4i ua[2][NBN];
            v4f uf[2][2];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                if (c == 1 && !two) break;
                uf[c][0] = *(const v4f *)(la + r0 + 16 * c);
                uf[c][1] = *(const v4f *)(la + r0 + 16 * c + 4);
#pragma unroll
                for (int blk = 0; blk < NBN; blk++) {
                    if (r0 == 0)
                        ua[c][blk] = *(const v4i *)(sepi + (c * 4 + blk) * BLK_BYTES + lane * 16);
                    else
                        ua[c][blk] = *(const v4i *)(lu + (size_t)min(n0 + blk * 32 + l32, a.N - 1) * a.ld_lora_up + r0 + 16 * c + half * 8);
                }
            }
#pragma unroll
            for (int c = 0; c < 2; c++) {
                if (c == 1 && !two) break;
                const v4f f0 = uf[c][0], f1 = uf[c][1];
                v4i ub;
                ub[0] = (int)pack2<T>(f0[0], f0[1]);
                ub[1] = (int)pack2<T>(f0[2], f0[3]);
                ub[2] = (int)pack2<T>(f1[0], f1[1]);
                ub[3] = (int)pack2<T>(f1[2], f1[3]);
#pragma unroll
                for (int bn = 0; bn < NBN; bn++)
                    acc[bn] = ROWS_IN_LANES ? mfma32_16bit<T>(ua[c][bn], ub, acc[bn]) : mfma32_16bit<T>(ub, ua[c][bn], acc[bn]);
            }
        }
    }
    if (a.bias != nullptr) {
#pragma unroll
        for (int bn = 0; bn < NBN; bn++) {
            if constexpr (ROWS_IN_LANES) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint2 b4 = *(const uint2 *)(sepi + LORA_UP_BYTES + (bn * 32 + 8 * j + 4 * half) * 2);
                    acc[bn][4 * j + 0] += T::lo_f32(b4.x);
                    acc[bn][4 * j + 1] += T::hi_f32(b4.x);
                    acc[bn][4 * j + 2] += T::lo_f32(b4.y);
                    acc[bn][4 * j + 3] += T::hi_f32(b4.y);
                }
            } else {
                const float b = T::to_f32(*(const uint16_t *)(sepi + LORA_UP_BYTES + (bn * 32 + l32) * 2));
#pragma unroll
                for (int i = 0; i < 16; i++) acc[bn][i] += b;
            }
        }
    }

    if constexpr (EPI == SVDQ_EPI_QK_NORM_ROPE) {
        if (qk_part < 2) {  // measured: issued ahead of LoRA-up as well, the launch takes 0.6 % longer
            qk_fetch(0, 0);
            qk_fetch(1, 1);
        }
    }

    // ---- transposition: lane = weight row -> lane = activation row ---------------------------------------------
    // One 32x32 block at a time through the private tile (the LDS operations of one wavefront complete in order).
    // Afterwards lane (m = lane % 32, half) holds columns 32 bn + 8 j + 4 half + e of row m in acc[bn][4 j + e]: row-wise
    // epilogue work is in-lane plus one exchange with lane ^ 32, and no epilogue needs another wavefront's data.
    if constexpr (!ROWS_IN_LANES) {
        float *tp = (float *)priv;
#pragma unroll
        for (int bn = 0; bn < NBN; bn++) {
#pragma unroll
            for (int i = 0; i < 16; i++) tp[(8 * (i >> 2) + 4 * half + (i & 3)) * TP_PITCH + l32] = acc[bn][i];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const v4f v = *(const v4f *)(tp + l32 * TP_PITCH + 8 * j + 4 * half);
                acc[bn][4 * j + 0] = v[0];
                acc[bn][4 * j + 1] = v[1];
                acc[bn][4 * j + 2] = v[2];
                acc[bn][4 * j + 3] = v[3];
            }
        }
    }

    // Output rows go out through LDS: in registers a lane holds 4 consecutive columns of one row, which stored directly
    // is an 8-byte piece per row and lane; staged as the wavefront's [32 rows][256 bytes] tile, each store instruction
    // writes four contiguous 256-byte row segments instead.  16-byte chunk c of row r sits at chunk c ^ (r & 15), its two
    // 8-byte halves swapped for rows 16-31: writes and reads are free of bank conflicts.
    auto store_out = [&]() {
#pragma unroll
        for (int bn = 0; bn < NBN; bn++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                uint2 v;
                v.x = pack2<T>(acc[bn][4 * j], acc[bn][4 * j + 1]);
                v.y = pack2<T>(acc[bn][4 * j + 2], acc[bn][4 * j + 3]);
                *(uint2 *)(priv + l32 * (BN * 2) + (((4 * bn + j) ^ (l32 & 15)) << 4) + 8 * (half ^ (l32 >> 4))) = v;
            }
        uint16_t *out = (uint16_t *)a.out;
        const int c = lane & 15, n = n0 + c * 8;
#pragma unroll
        for (int pass = 0; pass < 8; pass++) {
            const int r = 4 * pass + (lane >> 4), m = mw0 + r;  // rows 16-31 are passes 4-7
            v4i q = *(const v4i *)(priv + r * (BN * 2) + ((c ^ (r & 15)) << 4));
            if (pass >= 4) q = (v4i){q[2], q[3], q[0], q[1]};
            if (m < a.actual_m && n < a.N)
                // streamed: the 85 MB of a QKV output do not fit any cache level of the CU, and lines left dirty in L2 have
                // to be written back before the next kernel on the stream starts (measured: 1 % of the launch)
                __builtin_nontemporal_store(q, (v4i *)(out + (size_t)m * a.ld_out + n));
        }
    };

    if (EPI == SVDQ_EPI_PLAIN) {
        store_out();
        return;
    }

    if (EPI == SVDQ_EPI_QK_NORM_ROPE) {
        // the 128-wide tile is one head, all of it in this wavefront; part 0 = Q, 1 = K, 2 = V (untouched)
        if (qk_part < 2) {
            float ss = 0.0f;
#pragma unroll
            for (int bn = 0; bn < NBN; bn++)
#pragma unroll
                for (int i = 0; i < 16; i++) ss += acc[bn][i] * acc[bn][i];
            ss += __shfl_xor(ss, 32);
            const float rstd = 1.0f / sqrtf(ss / 128.0f + a.eps);
#pragma unroll
            for (int bn = 0; bn < NBN; bn++) {
                const int buf = bn & 1;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint2 wb = *(const uint2 *)(sepi + EPI_NORM_OFF + (bn * 32 + 8 * j + 4 * half) * 2);
                    const v4f sc = qk_sc[buf][j];
                    const float x0 = acc[bn][4 * j + 0] * rstd * T::lo_f32(wb.x);
                    const float x1 = acc[bn][4 * j + 1] * rstd * T::hi_f32(wb.x);
                    const float x2 = acc[bn][4 * j + 2] * rstd * T::lo_f32(wb.y);
                    const float x3 = acc[bn][4 * j + 3] * rstd * T::hi_f32(wb.y);
                    acc[bn][4 * j + 0] = x0 * sc[1] - x1 * sc[0];
                    acc[bn][4 * j + 1] = x0 * sc[0] + x1 * sc[1];
                    acc[bn][4 * j + 2] = x2 * sc[3] - x3 * sc[2];
                    acc[bn][4 * j + 3] = x2 * sc[2] + x3 * sc[3];
                }
                if (bn + 2 < NBN) qk_fetch(bn + 2, buf);  // behind the block's last use of this buffer
            }
        }
        store_out();
        return;
    }

    if (EPI == SVDQ_EPI_GELU_QUANT) {
        const uint16_t *ldt = (const uint16_t *)a.lora_down_t;
        // needed further down, issued before the GELU arithmetic: the next layer's smoothing factors of columns lane and
        // 64 + lane
        uint16_t smv[2] = {0, 0};
        const bool has_sm = a.smooth_next != nullptr;
        if (has_sm) {
#pragma unroll
            for (int t = 0; t < 2; t++) smv[t] = ((const uint16_t *)a.smooth_next)[min(n0 + 64 * t + lane, a.N - 1)];
        }
        if (a.out != nullptr) store_out();  // pre-GELU output, when asked for
#pragma unroll
        for (int bn = 0; bn < NBN; bn++) {
#pragma unroll
            for (int i = 0; i < 16; i++) acc[bn][i] = gelu_tanh(acc[bn][i]);
            __builtin_amdgcn_sched_barrier(0);  // (all 64 at once spill where the wavefront owns a second row block)
        }

        // next layer's LoRA-down on the un-shifted, un-smoothed GELU output rounded to T:
        // D[r][m] = sum_n ldT[r][n] * x[n][m] over the tile's 128 columns; registers [8 s, 8 s + 8) of a block are one
        // MFMA's B operand.  One partial per n-tile, summed in tile order by lora_part_reduce_kernel.
        for (int rc = 0; rc < a.R2; rc += 32) {
            v16f d;
#pragma unroll
            for (int i = 0; i < 16; i++) d[i] = 0.0f;
            const int r = rc + l32;
#pragma unroll
            for (int bn = 0; bn < NBN; bn++) {
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    // (fetched ahead of the GELU arithmetic, all at once or two column blocks ahead, these loads spill
                    // registers and the launch is no faster: the other workgroups of the CU cover their latency)
                    v4i la = (v4i){0, 0, 0, 0};
                    if (a.lora_down_blocked != nullptr) {
                        // re-laid-out copy: the operand of this instruction is 1 KB in lane order (from the (R2, N) copy a
                        // lane fetches two 8-byte pieces of its rank's row, 32 rows to a load instruction)
                        la = ((const v4i *)a.lora_down_blocked)[(((size_t)pid_n * ((a.R2 + 31) / 32) + rc / 32) * 8 + bn * 2 + s) * 64 + lane];
                    } else if (r < a.R2) {
                        const uint16_t *lp = ldt + (size_t)r * a.N + n0 + bn * 32 + 16 * s + 4 * half;
                        const uint2 q0 = *(const uint2 *)lp, q1 = *(const uint2 *)(lp + 8);
                        la = (v4i){(int)q0.x, (int)q0.y, (int)q1.x, (int)q1.y};
                    }
                    v4i xb;
#pragma unroll
                    for (int e = 0; e < 4; e++) xb[e] = (int)pack2<T>(acc[bn][8 * s + 2 * e], acc[bn][8 * s + 2 * e + 1]);
                    d = mfma32_16bit<T>(la, xb, d);
                }
            }
            const int m = mw0 + l32;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int rr = rc + 8 * j + 4 * half;
                if (m < a.M && rr < a.R2)
                    *(v4f *)(a.scratch + ((size_t)pid_n * a.M + m) * a.R2 + rr) = (v4f){d[4 * j], d[4 * j + 1], d[4 * j + 2], d[4 * j + 3]};
            }
        }

        // +shift, * 1/smooth, unsigned per-64 quantization: the wavefront's 128 columns are two groups
        float *lds_rs = (float *)priv;  // [BN], this wavefront's own copy
#pragma unroll
        for (int t = 0; t < 2; t++) lds_rs[64 * t + lane] = has_sm ? 1.0f / T::to_f32(smv[t]) : 1.0f;
        const int m = mw0 + l32;
#pragma unroll
        for (int gi = 0; gi < 2; gi++) {
            const int g = (n0 + 64 * gi) / GROUP;
            float gmax = 0.0f;
#pragma unroll
            for (int b2 = 0; b2 < 2; b2++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int bn = 2 * gi + b2;
                    const v4f rs = *(const v4f *)(lds_rs + bn * 32 + 8 * j + 4 * half);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float v = (acc[bn][4 * j + e] + a.shift) * rs[e];
                        acc[bn][4 * j + e] = v;
                        gmax = fmaxf(gmax, v);
                    }
                }
            gmax = max_with_lane_xor32(gmax);
            const float scale = gmax / 15.0f;
            const float safe = (scale == 0.0f) ? 1.0f : scale;
            const float rq = 1.0f / safe;
            if (half == 0 && m < a.M && n0 + 64 * gi < a.N)  // (oscales_blocked: the consuming GEMM's ascales_blocked layout)
                ((uint16_t *)a.oscales)[a.oscales_blocked ? ((size_t)(m >> 5) * (a.N / (8 * GROUP)) + (g >> 3)) * 256 + (m & 31) * 8 + (g & 7)
                                                          : (size_t)g * a.ld_oscales + m] = T::from_f32(scale);
            if (a.qout_blocked == 2) {
                uint32_t vec[6];
#pragma unroll
                for (int b2 = 0; b2 < 2; b2++) {
                    const int bn = 2 * gi + b2;
                    uint32_t pc[2][4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        uint32_t c[4];
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            c[e] = __float_as_uint(__builtin_amdgcn_fmed3f(acc[bn][4 * j + e] * rq, 0.0f, 15.0f) + RNE_MAGIC) & 0xFu;
                        pc[0][j] = c[0] | (c[2] << 6);
                        pc[1][j] = c[1] | (c[3] << 6);
                    }
                    uint32_t d0[3], d1[3];
                    f6_pack_unit(pc[0][0], pc[0][1], pc[0][2], pc[0][3], 12u * half, d0);
                    f6_pack_unit(pc[1][0], pc[1][1], pc[1][2], pc[1][3], 12u * half, d1);
                    f6_swap_unit(d0, d1, vec + 3 * b2);
                }
                f6_store(vec, (uint8_t *)a.qout + ((size_t)(m >> 5) * (a.N / GROUP) + g) * 1536, 32 * half + (m & 31), m < a.M);
                continue;
            }
#pragma unroll
            for (int b2 = 0; b2 < 2; b2++) {
                const int bn = 2 * gi + b2;
                uint32_t mine[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    uint32_t w = 0;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float q = __builtin_amdgcn_fmed3f(acc[bn][4 * j + e] * rq, 0.0f, 15.0f) + RNE_MAGIC;
                        w |= (__float_as_uint(q) & 0xFu) << (4 * e);
                    }
                    mine[j] = w;  // 16 bits: columns 8 j + 4 half + 0..3
                }
                // lane and lane ^ 32 hold alternating 16-bit pieces of one 16-byte run (dword j = piece of half 0 in
                // the low 16 bits, piece of half 1 in the high 16 bits); trade so half 0 stores dwords 0-1 and half 1
                // stores dwords 2-3
                uint32_t dw[2];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const uint32_t keep = half ? mine[2 + t] : mine[t];
                    const uint32_t send = half ? mine[t] : mine[2 + t];
                    const uint32_t theirs = __shfl_xor(send, 32);
                    dw[t] = half ? (theirs | (keep << 16)) : (keep | (theirs << 16));
                }
                if (m < a.M) {
                    // (qout_blocked: where lane (m % 32, bn % 2) of the consuming GEMM's row block and group reads its 16 bytes)
                    uint8_t *dst = a.qout_blocked
                                       ? (uint8_t *)a.qout + ((size_t)(m >> 5) * (a.N / GROUP) + g) * 1024 + (((bn & 1) * 32 + (m & 31)) * 16 + 8 * half)
                                       : (uint8_t *)a.qout + (size_t)m * a.ld_qout + (n0 + bn * 32) / 2 + 8 * half;
                    *(uint2 *)dst = make_uint2(dw[0], dw[1]);
                }
            }
        }
        return;
    }

    if (EPI == SVDQ_EPI_SWIGLU_QUANT) {
        // Output columns come in 16-blocks [gate | up]: registers j = 0, 1 of a 32-column block are gate values and
        // j = 2, 3 the matching up values, so y = silu(gate) * up is formed in-lane.  The tile's 128 columns give 64
        // y columns = one quantization group, all of it in this wavefront.
        const int H = a.N / 2;
        const uint16_t *ldt = (const uint16_t *)a.lora_down_t;
        const int yt0 = n0 / 2;  // first y column of the tile
        uint16_t smv = 0;
        const bool has_sm = a.smooth_next != nullptr;
        if (has_sm) smv = ((const uint16_t *)a.smooth_next)[min(yt0 + lane, H - 1)];
        float y[NBN][8];  // [bn][4 j + e]: y column 16 bn + 8 j + 4 half + e of the tile's 64
#pragma unroll
        for (int bn = 0; bn < NBN; bn++)
#pragma unroll
            for (int i = 0; i < 8; i++) y[bn][i] = silu(acc[bn][i]) * acc[bn][8 + i];
        const int m = mw0 + l32;
        for (int rc = 0; rc < a.R2; rc += 32) {
            v16f d;
#pragma unroll
            for (int i = 0; i < 16; i++) d[i] = 0.0f;
            const int r = rc + l32;
#pragma unroll
            for (int s = 0; s < NBN; s++) {
                v4i la = (v4i){0, 0, 0, 0};
                if (r < a.R2) {
                    const uint16_t *lp = ldt + (size_t)r * H + yt0 + 16 * s + 4 * half;
                    const uint2 q0 = *(const uint2 *)lp, q1 = *(const uint2 *)(lp + 8);
                    la = (v4i){(int)q0.x, (int)q0.y, (int)q1.x, (int)q1.y};
                }
                v4i xb;
#pragma unroll
                for (int e = 0; e < 4; e++) xb[e] = (int)pack2<T>(y[s][2 * e], y[s][2 * e + 1]);
                d = mfma32_16bit<T>(la, xb, d);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int rr = rc + 8 * j + 4 * half;
                if (m < a.M && rr < a.R2)
                    *(v4f *)(a.scratch + ((size_t)pid_n * a.M + m) * a.R2 + rr) = (v4f){d[4 * j], d[4 * j + 1], d[4 * j + 2], d[4 * j + 3]};
            }
        }

        // * 1/smooth, signed per-64 quantization over the tile's 64 y columns
        float *lds_rs = (float *)priv;  // [64], this wavefront's own copy
        lds_rs[lane] = has_sm ? 1.0f / T::to_f32(smv) : 1.0f;
        float gmax = 0.0f;
#pragma unroll
        for (int bn = 0; bn < NBN; bn++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const v4f rs = *(const v4f *)(lds_rs + 16 * bn + 8 * j + 4 * half);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float v = (y[bn][4 * j + e] + a.shift) * rs[e];
                    y[bn][4 * j + e] = v;
                    gmax = fmaxf(gmax, fabsf(v));
                }
            }
        gmax = max_with_lane_xor32(gmax);
        const float scale = gmax / 7.0f;
        const float safe = (scale == 0.0f) ? 1.0f : scale;
        const float rq = 1.0f / safe;
        if (half == 0 && m < a.M) {
            const int g = yt0 / GROUP;
            ((uint16_t *)a.oscales)[a.oscales_blocked ? ((size_t)(m >> 5) * (H / (8 * GROUP)) + (g >> 3)) * 256 + (m & 31) * 8 + (g & 7)
                                                      : (size_t)g * a.ld_oscales + m] = T::from_f32(scale);
        }
        if (a.qout_blocked == 2) {
            // sign | magnitude: the magnitude rounds as the value does; the magic constant gets 32 more for a negative one
            uint32_t vec[6];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                uint32_t pc[2][4];
#pragma unroll
                for (int t = 0; t < 4; t++) {  // piece 4 u + t: block bn = 2 u + t / 2, register run j = t % 2
                    uint32_t c[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float q = __builtin_amdgcn_fmed3f(y[2 * u + (t >> 1)][4 * (t & 1) + e] * rq, -8.0f, 7.0f);
                        const uint32_t mg = ((uint32_t)((int)__float_as_uint(q) >> 31) & 32u) | (uint32_t)RNE_MAGIC_BITS;
                        c[e] = __float_as_uint(__builtin_fabsf(q) + __uint_as_float(mg)) & 0x3Fu;
                    }
                    pc[0][t] = c[0] | (c[2] << 6);
                    pc[1][t] = c[1] | (c[3] << 6);
                }
                uint32_t d0[3], d1[3];
                f6_pack_unit(pc[0][0], pc[0][1], pc[0][2], pc[0][3], 12u * half, d0);
                f6_pack_unit(pc[1][0], pc[1][1], pc[1][2], pc[1][3], 12u * half, d1);
                f6_swap_unit(d0, d1, vec + 3 * u);
            }
            f6_store(vec, (uint8_t *)a.qout + ((size_t)(m >> 5) * (H / GROUP) + yt0 / GROUP) * 1536, 32 * half + (m & 31), m < a.M);
            return;
        }
#pragma unroll
        for (int bn = 0; bn < NBN; bn++) {
            uint32_t mine[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                uint32_t w = 0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float q = __builtin_amdgcn_fmed3f(y[bn][4 * j + e] * rq, -8.0f, 7.0f) + RNE_MAGIC;
                    w |= (__float_as_uint(q) & 0xFu) << (4 * e);
                }
                mine[j] = w;  // 16 bits: y columns 16 bn + 8 j + 4 half + 0..3
            }
            // dword j of the block's 8-byte run = piece of half 0 (low 16 bits) | piece of half 1 (high 16 bits);
            // half h keeps dword h
            const uint32_t keep = half ? mine[1] : mine[0];
            const uint32_t send = half ? mine[0] : mine[1];
            const uint32_t theirs = __shfl_xor(send, 32);
            const uint32_t dw = half ? (theirs | (keep << 16)) : (keep | (theirs << 16));
            if (m < a.M) {
                // (qout_blocked: the tile's 64 y columns are one group of the consuming GEMM; byte 8 bn + 4 half of its 32)
                uint8_t *dst = a.qout_blocked
                                   ? (uint8_t *)a.qout + ((size_t)(m >> 5) * (H / GROUP) + yt0 / GROUP) * 1024 + (((bn >> 1) * 32 + (m & 31)) * 16 + 8 * (bn & 1) + 4 * half)
                                   : (uint8_t *)a.qout + (size_t)m * a.ld_qout + (yt0 + 16 * bn) / 2 + 4 * half;
                *(uint32_t *)dst = dw;
            }
        }
        return;
    }
}

}  // namespace svdq
