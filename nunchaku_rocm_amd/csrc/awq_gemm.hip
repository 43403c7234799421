// AWQ W4A16 GEMM for gfx950: out = x . T(q * s + z)^T on TinyChat-packed weights, decoded in registers on the way to the
// matrix instruction.
//
// Arithmetic (reference: nunchaku/ops/triton/awq.py:48-79 awq_dequantize, :232-251 awq_gemm_w4a16): a weight is
// q * s + z in fp32, rounded to T; products and sums are the 16-bit matrix instruction's (fp32 accumulation).
//
// What bounds it: the vector instructions that decode a weight (2.4 each) beside the matrix instructions.  Every workgroup
// decodes its own channels, so the ratio falls with the rows it covers: 4.75 vector instructions per matrix instruction at
// 128 rows, where two wavefronts of a SIMD issue both at about 70 % of the matrix rate.  The alternative, a dense (N, K)
// matrix in memory and a library product, writes and reads back four times the packed bytes first.  Measured, K = 4096,
// bf16: M = 512, N = 10240 46 us against 75 for decode + library product (decode alone 26), N = 4096 24 against 43.
//
// Split.  A weight goes from memory to the matrix instruction in registers: the 16 bytes of (channel, half of a group
// of 64) hold, per nibble plane, eight consecutive k -- one lane's operand.  So a wavefront owns 64 channels (two
// 32-channel operands), no other wavefront decodes them, and only the activations go through LDS.  A workgroup is NS
// channel slices x 2 halves of K: wavefront (ns, kp) multiplies rows x 64 channels over its 64 of a stage's 128 k, and
// the two K halves of a slice are added through LDS at the end.  With K split inside the workgroup an operand read from
// LDS feeds two matrix instructions while the workgroup stays narrow, which is what a launch of few rows needs to cover
// the chip.  MB = 32-row blocks of activations per workgroup.
// Activations: rows x 128 k of T per stage, [row][256 bytes] with the row's sixteen 16-byte chunks XOR-swizzled by
// row % 16 (operand reads are conflict free), fetched memory -> LDS directly, two stages ahead (one stage ahead the same
// launch waited 9 us for them); weights into registers two stages ahead.
#include "svdq_common.h"

namespace svdq {

constexpr int AG_K = 128;
constexpr int AG_ROW = AG_K * 2;  // bytes of a row's stage

// Decodes the weights T(q * s + z) of nibble planes par and par + 2 in one dword (two k of each plane: int16 2 d in the low
// half).  A nibble c in a byte is the fp8 (e4m3) code of c * 2^-9 (subnormals and the first binade are one linear run), so
// the hardware's fp8 -> fp32 conversion with scale 2^9 turns two of them into exact floats in one instruction; masked to
// one nibble per byte, a half dword holds the same k of both planes.
template <typename T>
__device__ inline void ag_decode(int w, int par, float s, float z, int &lo_plane, int &hi_plane) {
    const int p = (int)(((uint32_t)w >> (4 * par)) & 0x0F0F0F0Fu);
    const auto a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(p, 512.0f, false), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(p, 512.0f, true);
    lo_plane = (int)pack2<T>(__builtin_fmaf(a[0], s, z), __builtin_fmaf(b[0], s, z));
    hi_plane = (int)pack2<T>(__builtin_fmaf(a[1], s, z), __builtin_fmaf(b[1], s, z));
}

__device__ inline __amdgpu_buffer_rsrc_t ag_buffer(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)0xFFFFFFFFu, 0x00020000);
}
// lane l's 16 bytes at base + lane offset + uniform offset -> lds + 16 l, or -> registers
__device__ inline void ag_load_lds(__amdgpu_buffer_rsrc_t r, uint8_t *lds, uint32_t lane_off, uint32_t uniform_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (SVDQ_AS3 void *)lds, 16, (int)lane_off, (int)uniform_off, 0, 0);
}
__device__ inline v4i ag_load128(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_off, (int)uniform_off, 0));
}
__device__ inline uint16_t ag_load16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, (int)lane_off, 0, 0);
}

template <typename T, int MB, int NS>
__global__ __launch_bounds__(NS * 128, MB == 4 && NS == 2 ? 1 : 2) void awq_gemm_kernel(const uint16_t *__restrict__ x, const uint8_t *__restrict__ qw,
                                                                 const uint16_t *__restrict__ scales, const uint16_t *__restrict__ zeros,
                                                                 uint16_t *__restrict__ out, int M, int N, int K, int ld_x, int ld_scales,
                                                                 int ld_out, int tiles_m, uint32_t gmagic) {
    constexpr int BMR = 32 * MB;                     // rows of the tile
    constexpr int STAGE = BMR * AG_ROW;              // 32, 16 or 8 KB
    constexpr int AG_N = 64 * NS, NWAVES = 2 * NS;   // channels, wavefronts
    constexpr int XLOADS = STAGE / 1024 / NWAVES;    // block loads per wavefront and stage
    constexpr int XCH = 32 * 64 * 4;                 // a wavefront's exchange region: one row block of its slice in fp32
    // an LDS object per stage: the compiler then knows that a block load into one cannot touch what is read from another
    constexpr int REGIONS = STAGE / XCH > (NWAVES + 2) / 3 ? STAGE / XCH : (NWAVES + 2) / 3;  // exchange regions per object
    constexpr int SMEM = STAGE > REGIONS * XCH ? STAGE : REGIONS * XCH;
    __shared__ __align__(16) uint8_t smem0[SMEM], smem1[SMEM], smem2[SMEM];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), ns = wave % NS, kp = wave / NS;
    const int l32 = lane & 31, half = lane >> 5;
    // workgroup -> tile: each XCD (ids are dealt round-robin over eight) takes a contiguous range, row tiles innermost,
    // so that the row tiles of a weight slice read it through one L2
    const int nb = gridDim.x, xcd = blockIdx.x & 7, per = nb / 8, rem = nb % 8;
    const int id = xcd * per + min(xcd, rem) + (int)(blockIdx.x >> 3);
    const int m0 = (id % tiles_m) * BMR, n0 = (id / tiles_m) * AG_N;
    const int nstages = K / AG_K, G64 = K / GROUP;  // whole stages; K / 64 odd: half a stage behind them
    const int slast = (G64 - 1) / 2;

    // ---- activations: lane l of block load i fetches chunk (l % 16) ^ (row % 16) of row 4 i + l / 16 -----------------
    const __amdgpu_buffer_rsrc_t rX = ag_buffer(x + (size_t)m0 * ld_x);
    uint32_t xoff[XLOADS];
#pragma unroll
    for (int j = 0; j < XLOADS; j++) {
        const int row = 4 * (wave * XLOADS + j) + (lane >> 4);
        xoff[j] = (uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)ld_x * 2u + (uint32_t)(((lane & 15) ^ (row & 15)) * 16);
    }
    auto issue_x = [&](int s, uint8_t *buf) {
        const bool tail = s >= nstages;  // half a stage: its second 128 bytes of a row do not exist, the first are read again
#pragma unroll
        for (int j = 0; j < XLOADS; j++) {
            const uint32_t second = (uint32_t)(((lane >> 3) & 1) ^ (((wave * XLOADS + j) >> 1) & 1)) * 128u;  // chunk & 8
            ag_load_lds(rX, buf + (wave * XLOADS + j) * 1024, xoff[j] - (tail ? second : 0u), (uint32_t)s * AG_ROW);
        }
    };

    // ---- weights: per 32-channel block 16 bytes (lane = channel, half of the group of 64), a scale and a zero --------
    const __amdgpu_buffer_rsrc_t rW = ag_buffer(qw + (size_t)(n0 >> 2) * K * 2), rS = ag_buffer(scales), rZ = ag_buffer(zeros);
    uint32_t woff[2], soff[2];
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const int n = min(n0 + ns * 64 + b * 32 + l32, N - 1);
        woff[b] = (uint32_t)((n >> 2) - (n0 >> 2)) * (uint32_t)K * 2u + 32u * (n & 3) + 16u * half;
        soff[b] = 2u * (uint32_t)n;
    }
    struct W {
        v4i q[2];
        uint16_t s[2], z[2];
    };
    auto load_w = [&](int s, W &w) {
        const int c = min(2 * s + kp, G64 - 1);
        // scale group of this lane's 32 k: (2 c + half) / (group / 32) as a multiplication by ceil(2^31 / (group / 32))
        const uint32_t g = __umulhi(2u * (uint32_t)(2 * c + half), gmagic) * (uint32_t)ld_scales * 2u;
#pragma unroll
        for (int b = 0; b < 2; b++) {
            w.q[b] = ag_load128(rW, woff[b], (uint32_t)c * 128u);
            w.s[b] = ag_load16(rS, soff[b] + g);
            w.z[b] = ag_load16(rZ, soff[b] + g);
        }
    };

    v16f acc[2][MB];
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int m = 0; m < MB; m++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[b][m][i] = 0.0f;

    // A stage is eight slots of MB matrix instructions: (plane, channel block) in the order of planes 0, 2, 1, 3.  Behind
    // each a quarter of the next two planes' weights is decoded, and the next plane's activations are read once the
    // second channel block is through with the current ones.  The last four slots do so for the next stage, whose
    // activations a barrier in the middle of this stage has released: no slot waits for a stage to begin.
    v4i xa[MB], wd[2][2][2];  // wd[planes 0, 2 / 1, 3][which of the two][channel block]
    auto read_x = [&](const uint8_t *base, int pl, int m) {
        xa[m] = *(const v4i *)(base + (m * 32 + l32) * AG_ROW + (((8 * kp + 4 * half + pl) ^ (l32 & 15)) * 16));
    };
    auto decode = [&](const W &w, int par, int b, int d0) {
        const float fs = T::to_f32(w.s[b]), fz = T::to_f32(w.z[b]);
#pragma unroll
        for (int d = d0; d < d0 + 2; d++) {
            int lo, hi;
            ag_decode<T>(w.q[b][d], par, fs, fz, lo, hi);
            wd[par][0][b][d] = lo;
            wd[par][1][b][d] = hi;
        }
    };
    constexpr int PLANE[4] = {0, 2, 1, 3};
    W wa, wb;
    auto stage = [&](int s, const uint8_t *cur, const uint8_t *nxt, uint8_t *fill, W &w, const W &wn) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int par = u >> 2, pi = (u >> 1) & 1, b = u & 1;
            __builtin_amdgcn_sched_barrier(0);
            if (u == 4) {
                // this wavefront's activations of stage s + 1 have landed: nothing younger is outstanding.  (The weights are asked
                // for behind the wait.  A wait that leaves their six loads out would count loads that the compiler may drop or
                // move; asked for before or after, a launch takes the same time.)  Behind the barrier everybody's have landed, and
                // nobody reads stage s - 1 any more: its buffer takes stage s + 2 (past the end: the last stage again)
                __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 15));
                load_w(min(s + 2, slast), w);  // all of them decoded: their registers take the stage after next
                __builtin_amdgcn_s_barrier();
                issue_x(min(s + 2, slast), fill);
            }
#pragma unroll
            for (int m = 0; m < MB; m++) {
                acc[b][m] = mfma32_16bit<T>(wd[par][pi][b], xa[m], acc[b][m]);
                if (b == 1) read_x(u < 7 ? cur : nxt, PLANE[((u >> 1) + 1) & 3], m);
            }
            decode(par == 0 ? w : wn, par ^ 1, pi, 2 * b);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // The first wait leaves out the block loads of stage 1 and nothing else: they are kept, and kept the youngest.
    issue_x(0, smem0);
    load_w(0, wa);
    load_w(min(1, slast), wb);
    __builtin_amdgcn_sched_barrier(0);
    issue_x(min(1, slast), smem1);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(XLOADS, 15));
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int m = 0; m < MB; m++) read_x(smem0, 0, m);
#pragma unroll
    for (int u = 0; u < 4; u++) decode(wa, 0, u >> 1, 2 * (u & 1));
    int s = 0;
    for (; s + 6 <= nstages; s += 6) {
        stage(s, smem0, smem1, smem2, wa, wb);
        stage(s + 1, smem1, smem2, smem0, wb, wa);
        stage(s + 2, smem2, smem0, smem1, wa, wb);
        stage(s + 3, smem0, smem1, smem2, wb, wa);
        stage(s + 4, smem1, smem2, smem0, wa, wb);
        stage(s + 5, smem2, smem0, smem1, wb, wa);
    }
    const int left = nstages - s;  // 0 .. 5
    if (left >= 1) stage(s, smem0, smem1, smem2, wa, wb);
    if (left >= 2) stage(s + 1, smem1, smem2, smem0, wb, wa);
    if (left >= 3) stage(s + 2, smem2, smem0, smem1, wa, wb);
    if (left >= 4) stage(s + 3, smem0, smem1, smem2, wb, wa);
    if (left >= 5) stage(s + 4, smem1, smem2, smem0, wa, wb);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));  // every load has landed, the redundant ones of the last stages too
    __syncthreads();
    if ((G64 & 1) && kp == 0) {  // half a stage: the first K half's 64 k, which the last slot has begun to read and decode
        const uint8_t *cur = left % 3 == 0 ? smem0 : left % 3 == 1 ? smem1 : smem2;
        const W w = (left & 1) ? wb : wa;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int par = u >> 2, pi = (u >> 1) & 1, b = u & 1;
#pragma unroll
            for (int m = 0; m < MB; m++) {
                acc[b][m] = mfma32_16bit<T>(wd[par][pi][b], xa[m], acc[b][m]);
                if (b == 1 && u < 7) read_x(cur, PLANE[(u >> 1) + 1], m);
            }
            if (par == 0) decode(w, 1, pi, 2 * b);
        }
    }
    __syncthreads();

    // ---- the two K halves of a slice are added: a wavefront hands every other row block to its partner and finishes the
    // blocks in between (with one block the second half hands it over); lane = row, registers walk channels
    auto region = [&](int w) { return (float *)((w < REGIONS ? smem0 : w < 2 * REGIONS ? smem1 : smem2) + (w % REGIONS) * XCH); };
    float *xw = region(wave);
    const float *xr = region(wave ^ NS);
    auto at = [&](int b, int j) { return l32 * 64 + (((8 * b + 2 * j + half) ^ (l32 & 15)) << 2); };
#pragma unroll
    for (int h = 0; h < MB; h += 2) {
        if (MB > 1 || kp == 1) {
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v4f v;
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = MB > 1 && kp == 0 ? acc[b][MB > 1 ? h + 1 : h][4 * j + e] : acc[b][h][4 * j + e];
                    *(v4f *)(xw + at(b, j)) = v;
                }
        }
        __syncthreads();
        if (MB > 1 || kp == 0) {
            const int m = m0 + (h + (MB > 1 ? kp : 0)) * 32 + l32;
            uint16_t *orow = out + (size_t)min(m, M - 1) * ld_out;
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const v4f o = *(const v4f *)(xr + at(b, j));
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = o[e] + (MB > 1 && kp == 1 ? acc[b][MB > 1 ? h + 1 : h][4 * j + e] : acc[b][h][4 * j + e]);
                    const int n = n0 + ns * 64 + 32 * b + 8 * j + 4 * half;
                    if (m < M && n < N) *(uint2 *)(orow + n) = make_uint2(pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3]));
                }
        }
        if (h + 2 < MB) __syncthreads();
    }
}

// Rows and channels of a workgroup's tile, by the workgroups of the most loaded CU: microseconds of one such workgroup at
// K = 4096 (alone on its CU, each further one), measured on 80 to 1280 workgroups.  Tall and wide tiles decode a weight for
// more rows; small ones keep CUs from idling (M = 512: N = 4096 23.6 us with 64 x 128 tiles against 43.9 with 128 x 256,
// N = 10240 53.9 against 46.5; M = 1024, N = 4096 36.4 with 128 x 128).
struct AwqTile {
    int rows, channels;
};
static AwqTile awq_gemm_tile(int M, int N, int cus) {
    auto cost = [&](AwqTile t, double first, double next) {
        const long wgs = (long)((M + t.rows - 1) / t.rows) * ((N + t.channels - 1) / t.channels), per_cu = (wgs + cus - 1) / cus;
        return first + (double)(per_cu - 1) * next;
    };
    AwqTile best = {128, 256};
    double least = cost(best, 42, 50);
    auto consider = [&](AwqTile t, double first, double next) {
        const double c = cost(t, first, next);
        if (c < least) best = t, least = c;
    };
    consider({128, 128}, 28, 34);
    consider({64, 128}, 21, 16.5);
    consider({32, 128}, 19, 12.5);
    return best;
}

template <typename T>
static void launch_awq_gemm(const svdq_awq_gemv_args &a, int group, hipStream_t s) {
    auto go = [&](auto mtag, auto ntag) {
        constexpr int MB = decltype(mtag)::value, NS = decltype(ntag)::value;
        const int tiles_m = (a.M + 32 * MB - 1) / (32 * MB), tiles_n = (a.N + 64 * NS - 1) / (64 * NS);
        hipLaunchKernelGGL((awq_gemm_kernel<T, MB, NS>), dim3((unsigned)tiles_m * (unsigned)tiles_n), dim3(NS * 128), 0, s, (const uint16_t *)a.x,
                           (const uint8_t *)a.qweight, (const uint16_t *)a.scales, (const uint16_t *)a.zeros, (uint16_t *)a.out, a.M, a.N, a.K,
                           a.ld_x, a.ld_scales, a.ld_out, tiles_m, (uint32_t)(((1ull << 31) + group / 32 - 1) / (group / 32)));
    };
    constexpr std::integral_constant<int, 1> c1{};
    constexpr std::integral_constant<int, 2> c2{};
    constexpr std::integral_constant<int, 4> c4{};
    const AwqTile t = awq_gemm_tile(a.M, a.N, cu_count());
    if (t.channels == 256)
        go(c4, c4);
    else if (t.rows == 128)
        go(c4, c2);
    else if (t.rows == 64)
        go(c2, c2);
    else
        go(c1, c2);
}

}  // namespace svdq

using namespace svdq;

extern "C" int svdq_awq_gemm_tile(int32_t M, int32_t N, int32_t cus) {
    if (M <= 0 || N <= 0) return 0;
    const AwqTile t = awq_gemm_tile(M, N, cus > 0 ? cus : cu_count());
    return t.rows << 16 | t.channels;
}

extern "C" int svdq_awq_gemm_w4a16(const svdq_awq_gemv_args *args, int32_t group_size, void *stream) {
    if (!args) {
        set_error("svdq_awq_gemm_w4a16: null args");
        return SVDQ_E_INVALID;
    }
    const svdq_awq_gemv_args &a = *args;
    if (a.dtype != SVDQ_BF16 && a.dtype != SVDQ_FP16) {
        set_error("svdq_awq_gemm_w4a16: dtype %d", a.dtype);
        return SVDQ_E_INVALID;
    }
    if (a.M < 0 || a.N <= 0 || a.N % 4 || a.K <= 0 || a.K % GROUP || group_size <= 0 || group_size % 32 || a.K % group_size) {
        set_error("svdq_awq_gemm_w4a16: M=%d N=%d K=%d group_size=%d needs N %% 4 == 0, K %% 64 == 0, group_size %% 32 == 0 dividing K", a.M, a.N,
                  a.K, group_size);
        return SVDQ_E_INVALID;
    }
    if (!a.x || !a.qweight || !a.scales || !a.zeros || !a.out || ((uintptr_t)a.x & 15) || a.ld_x % 8 || a.ld_x < a.K ||
        ((uintptr_t)a.qweight & 15) || a.ld_scales < a.N || ((uintptr_t)a.out & 7) || a.ld_out % 4 || a.ld_out < a.N) {
        set_error("svdq_awq_gemm_w4a16: x rows and qweight must be 16-byte, out rows 8-byte aligned; leading dimensions >= row length");
        return SVDQ_E_INVALID;
    }
    if ((size_t)128 * a.ld_x * 2 >= ((size_t)1 << 31) || (size_t)(a.K / group_size) * a.ld_scales * 2 >= ((size_t)1 << 32) || (size_t)((a.M + 31) / 32) * ((a.N + 127) / 128) >= ((size_t)1 << 31)) {
        set_error("svdq_awq_gemm_w4a16: M=%d N=%d ld_x=%d ld_scales=%d: too large for 32-bit offsets", a.M, a.N, a.ld_x, a.ld_scales);
        return SVDQ_E_UNSUPPORTED;
    }
    if (a.M == 0) return SVDQ_OK;
    if (a.dtype == SVDQ_BF16)
        launch_awq_gemm<BF16>(a, group_size, (hipStream_t)stream);
    else
        launch_awq_gemm<FP16>(a, group_size, (hipStream_t)stream);
    return check_launch("svdq_awq_gemm_w4a16");
}
