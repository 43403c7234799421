// Unmasked scaled-dot-product attention (flash-attention forward) for gfx950, head dimension 128 or 64.
//
// Arithmetic (reference: nunchaku/ops/triton/attention.py:37-169): q is multiplied by scale * log2(e) and rounded to
// the 16-bit type; per block of keys S = q k^T in fp32, online softmax with exp2 (a row reference m and row sum l),
// P rounded to the 16-bit type, O = O * 2^(m_old - m_new) + P v in fp32; at the end O / l, stored as
// (B, Tq, H * 128).  Two choices the mathematics leaves open differ from the reference: the reference m is only moved
// when a row maximum exceeds it by more than 8 (P then lies in (0, 2^8] instead of (0, 1]: the same O / l, since P, O
// and l all carry the same power of two), and l sums the rounded P the matrix instruction sees, not the unrounded one.
//
// How it maps to CDNA4:
//  * Everything is computed transposed.  S^T = K Q^T puts the keys in the MFMA's A operand and the queries in its B
//    operand, so in the 32x32 accumulator a lane owns ONE query (column) and its registers walk the keys: the row
//    maximum and row sum of the softmax are in-lane reductions plus one exchange with lane ^ 32
//    (v_permlane32_swap), and the rescaling of the output accumulator is a per-lane scalar.  O^T = V^T P^T then
//    takes P^T as its B operand straight from those accumulator registers (eight values of a lane are the eight
//    k-slots the operand wants: keys 4 h .. 4 h + 3 and 8 + 4 h .. 8 + 4 h + 3 of a 16-key chunk for the lanes of
//    half h), with no trip through LDS.
//  * The S^T accumulator starts at minus the row reference, so the scores leave the matrix instruction ready for
//    exp2: no subtraction per score.
//  * V is never transposed in memory: K and V tiles (64 keys x 2 D bytes each) stream buffer -> LDS directly
//    (buffer_load_dwordx4 ... lds, whole rows per load, per-lane offsets fixed and the tile chosen by the scalar
//    buffer base, 16-byte chunks XOR-swizzled so that the operand reads are conflict free), two tiles in flight, one
//    barrier per 64 keys; the V^T operand comes out of the V tile through the transposing LDS read of gfx950
//    (ds_read_b64_tr_b16: sixteen lanes pass the addresses of four rows x 16 columns and lane l receives column l
//    of the four rows), two reads per operand.
//  * Four wavefronts of 32 queries, two workgroups per CU, or eight and one (wide_queries); Q stays in registers (pre-scaled), the output
//    accumulator is D / 2 registers.  The keys are walked 32 at a time in a software pipeline: the products of the next and
//    of the previous 32 keys are issued beside the softmax of the current ones (see the comment in the kernel).
//  * Workgroups of one head run on one XCD (when the head count is a multiple of 8), so K and V of a head are
//    fetched into one L2 only.
#include <type_traits>

#include "svdq_common.h"

namespace svdq {

constexpr int AT_BK = 64;  // keys per tile

// Geometry for head dimension D (128 or 64).  K and V tiles are [key][2 D bytes]; every block load moves 1 KB
// (64 lanes x 16 bytes) = whole rows; 16-byte chunks are XOR-swizzled by the row so that the operand reads touch every
// bank once.  K (32 rows x one chunk per half-wave): rows of 256 bytes by row & 15, rows of 128 bytes (two rows span
// the 64 banks) by row / 2 & 7.  V (a transposing read = 4 rows x 32 bytes per 16 lanes, two such groups with
// neighbouring 32-byte column slots per half-wave): the eight (row, slot) pairs of a half-wave must land in eight
// different 32-byte slots of the 256 bytes the banks span, so the 64-byte quarter of a row is swizzled by row & 3
// (256-byte rows) or the 64-byte half by row / 2 & 1 (128-byte rows, where rows r and r + 1 already differ by half
// the banks).
template <int D, int WAVES>
struct AtGeo {
    static constexpr int NC = D / 16;               // 16-wide k chunks of q k^T = matrix instructions per 32-key half
    static constexpr int NDT = D / 32;              // 32-row d tiles of O^T
    static constexpr int KROW = 2 * D;              // bytes per key row
    static constexpr int KCH = KROW / 16;           // chunks per key row (16 or 8)
    static constexpr int KT_BYTES = AT_BK * KROW;   // K tile
    static constexpr int VT_BYTES = KT_BYTES;       // V tile
    static constexpr int STAGE = KT_BYTES + VT_BYTES;
    static constexpr int LOADS = KT_BYTES / 1024 / WAVES;  // block loads per wavefront and tile, of K and of V alike
    static constexpr int OPITCH = 2 * D + 16;       // staged output row
    __host__ __device__ static constexpr int kswz(int row) { return KROW == 256 ? (row & 15) : ((row >> 1) & 7); }
    __host__ __device__ static constexpr int vswz(int row) { return KROW == 256 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); }
};

constexpr uint32_t AT_RSRC_FLAGS = 0x00020000;  // raw buffer, 32-bit data format (gfx9 family)

// 16 bytes per lane from a raw buffer (`bytes` long from `base`; reads past it return zero) straight into LDS at
// lds + 16 * lane.  Plain functions, so that the kernel template below calls no target builtin with dependent operands.
__device__ inline __amdgpu_buffer_rsrc_t at_buffer(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)bytes, AT_RSRC_FLAGS);
}
__device__ inline void at_load16_lds(__amdgpu_buffer_rsrc_t r, uint8_t *lds, uint32_t lane_off, uint32_t wave_off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (SVDQ_AS3 void *)lds, 16, lane_off, wave_off, 0, 0);
}
// four rows x one column of a [row][col] 16-bit matrix in LDS: the sixteen lanes of a group pass the addresses of
// (row r = lane % 16 / 4, columns 4 (lane % 4) .. + 3) and lane l of the group receives column l of rows 0 .. 3
typedef short v4s16 __attribute__((ext_vector_type(4)));
typedef int v2i32 __attribute__((ext_vector_type(2)));
__device__ inline v2i32 at_read_tr(const uint8_t *p) {
    return __builtin_bit_cast(v2i32, __builtin_amdgcn_ds_read_tr16_b64_v4i16((SVDQ_AS3 v4s16 *)p));
}
constexpr float AT_LAZY = 8.0f;                 // the accumulator is rescaled when a row maximum grew by more than this

template <typename T, int D, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void attention_kernel(svdq_attention_args a, int ntile, int xcd_heads) {
    using G = AtGeo<D, WAVES>;
    constexpr int AT_BQ = 32 * WAVES;  // queries per workgroup
    constexpr int NC = G::NC, NDT = G::NDT, LOADS = G::LOADS;
    // Two separate LDS objects, one per stage, and a main loop unrolled over them: the compiler then knows that a tile
    // load into one stage cannot touch what is being read from the other.  With one object and a run-time stage offset
    // it made every LDS read wait for all loads in flight, i.e. for the tile that was requested just before.
    static_assert(WAVES % 4 == 0 && 64 * G::OPITCH <= G::STAGE, "the output tile is staged as two halves of 64 rows, one per stage");
    __shared__ __align__(16) uint8_t smem0[G::STAGE];
    __shared__ __align__(16) uint8_t smem1[G::STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    // workgroup -> (batch * head, query tile).  Workgroups are dealt to the eight XCDs round-robin; when the head count
    // allows it, a head's query tiles all land on one XCD so that its K and V stay in that XCD's L2.
    int bh, qt;
    if (xcd_heads) {
        const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
        bh = (j / ntile) * 8 + xcd;
        qt = j % ntile;
    } else {
        bh = blockIdx.x / ntile;
        qt = blockIdx.x % ntile;
    }
    const int b = bh / a.H, h = bh % a.H;
    const int q0 = qt * AT_BQ;

    // ---- Q^T operand: lane (q, half) holds q[16 c + 8 half, +8) for c < NC, scaled and rounded to T ---------------
    const int qrow = min(q0 + wave * 32 + l32, a.Tq - 1);
    const uint16_t *qp = (const uint16_t *)a.q + (long)b * a.sqb + (long)h * a.sqh + (long)qrow * a.sqm + 8 * half;
    const float qscale = a.scale * 1.4426950408889634f;
    v4i qop[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const v4i raw = *(const v4i *)(qp + 16 * c);
#pragma unroll
        for (int e = 0; e < 4; e++)
            qop[c][e] = (int)pack2<T>(T::lo_f32((uint32_t)raw[e]) * qscale, T::hi_f32((uint32_t)raw[e]) * qscale);
    }

    // ---- tile loads (buffer -> LDS, 16 bytes per lane): lane l of load i fetches one chunk of key row
    // (64 / KCH) i + l / KCH of K and of V alike.  LOADS K and LOADS V loads per wavefront and tile.  The per-lane
    // offsets never change; the tile is selected by the (scalar) buffer base, and key rows past the end lie outside
    // the buffers' ranges and arrive as zeros.
    const uint8_t *kbase = (const uint8_t *)a.k + ((long)b * a.skb + (long)h * a.skh) * 2;
    const uint8_t *vbase = (const uint8_t *)a.v + ((long)b * a.svb + (long)h * a.svh) * 2;
    const uint32_t kbytes = (uint32_t)(((long)(a.Tkv - 1) * a.skn + D) * 2);
    const uint32_t vbytes = (uint32_t)(((long)(a.Tkv - 1) * a.svn + D) * 2);
    const uint32_t ktile = (uint32_t)(AT_BK * a.skn * 2), vtile = (uint32_t)(AT_BK * a.svn * 2);
    uint32_t kvo[LOADS], vvo[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; j++) {
        const int i = wave * LOADS + j;
        const int row = (64 / G::KCH) * i + lane / G::KCH;
        kvo[j] = (uint32_t)row * (uint32_t)(a.skn * 2) + (uint32_t)(((lane % G::KCH) ^ G::kswz(row)) * 16);
        vvo[j] = (uint32_t)row * (uint32_t)(a.svn * 2) + (uint32_t)(((lane % G::KCH) ^ G::vswz(row)) * 16);
    }
    auto issue_k = [&](int blk, uint8_t *stage, int j) {
        const uint32_t off = (uint32_t)blk * ktile;
        at_load16_lds(at_buffer(kbase + off, kbytes - off), stage + (wave * G::LOADS + j) * 1024, kvo[j], 0);
    };
    auto issue_v = [&](int blk, uint8_t *stage, int j) {
        const uint32_t off = (uint32_t)blk * vtile;
        at_load16_lds(at_buffer(vbase + off, vbytes - off), stage + G::KT_BYTES + (wave * G::LOADS + j) * 1024, vvo[j], 0);
    };

    // operand read offsets.  K rows 32 t + l32 (chunk 2 c + half).  V^T operand of d tile dt and 16-key chunk c: lane
    // (half, dq = lane / 16 % 2, r = lane % 16 / 4, c4 = lane % 4) passes the address of V[16 c + 4 half + r (+ 8 for
    // the second read)][32 dt + 16 dq + 4 c4] and receives d = 32 dt + lane % 32, keys 4 half .. + 3 (8 + 4 half .. + 3)
    int koff[NC], vtoff[NDT];
#pragma unroll
    for (int c = 0; c < NC; c++) koff[c] = l32 * G::KROW + (((2 * c + half) ^ G::kswz(l32)) * 16);
    {
        const int dq = (lane >> 4) & 1, r = (lane & 15) >> 2, c4 = lane & 3, key = 4 * half + r;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
            vtoff[dt] = G::KT_BYTES + key * G::KROW + (((4 * dt + 2 * dq + (c4 >> 1)) ^ G::vswz(key)) * 16) + 8 * (c4 & 1);
    }
    // (keys 16 c + 8 + key have the same swizzle as key: both leave key % 4 and, for 128-byte rows, key / 2 % 2 alone)
    auto read_v = [&](const uint8_t *st, int dt, int c) {
        const v2i32 lo = at_read_tr(st + vtoff[dt] + c * (16 * G::KROW));
        const v2i32 hi = at_read_tr(st + vtoff[dt] + c * (16 * G::KROW) + 8 * G::KROW);
        return v4i{lo[0], lo[1], hi[0], hi[1]};
    };

    v16f acc_o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc_o[dt][i] = 0.0f;
    // Scores come out of the matrix instructions already relative to the row's reference: the accumulator of S^T starts
    // at -bias (cinit), so p = 2^s' with s' = s - bias needs no subtraction.  bias trails the true row maximum by at
    // most AT_LAZY (it only moves when a maximum exceeds it by more than that), which keeps p <= 2^AT_LAZY.
    // The bias itself only lives in cinit; gap = reference - bias: 0 once a reference exists, -inf before the first keys.
    float gap = -INFINITY, l_run = 0.0f;
    v16f cinit;
#pragma unroll
    for (int i = 0; i < 16; i++) cinit[i] = 0.0f;

    const int nblk = (a.Tkv + AT_BK - 1) / AT_BK, nhalf = (a.Tkv + 31) / 32;
    // Software pipeline over halves of 32 keys.  Iteration j issues three independent strands side by side:
    //   S(j + 1) = K[j + 1] Q^T      |  softmax of S(j)  |      O^T += V^T[j - 1] P(j - 1)^T
    // in 2 NC slots of one matrix instruction, its share of the softmax and the read that refills the operand registers it
    // has just used with the operand of RING matrix instructions of its strand later.  Stage t & 1 holds V of tile t and K of
    // tile t + 1; the operands are read from it between the middle of tile t's first iteration, where a barrier releases it and
    // the other stage begins to fill, and the middle of tile t + 1's.  The compiler is kept from regrouping the slots.
    // What bounds it is power.  us with the softmax beside one of the two products only / this way (bf16, workgroups of 128 queries): D = 128, 24
    // heads x 4608 253 / 232, 24 x 2000 58 / 52; D = 64, 40 x 4096 172 / 166.  Scores of the next tile that are there when the reference moves
    // get the difference subtracted; started anew from the new bias (the last bit of a few outputs in a million) keys whose size
    // grows along the sequence took 280 instead of 263.
    // Priority: the second iteration of a tile goes first (s_setprio), which keeps the two wavefronts of a SIMD out of step: 242 / 236.
    constexpr int RING = NC / 2;
    static_assert(NC == 2 * NDT, "as many matrix instructions per half in either product");
#pragma unroll
    for (int j = 0; j < LOADS; j++) issue_k(0, smem1, j);  // K of tile 0: read before the first barrier in the loop
#pragma unroll
    for (int j = 0; j < LOADS; j++) issue_v(0, smem0, j);
#pragma unroll
    for (int j = 0; j < LOADS; j++) issue_k(min(1, nblk - 1), smem0, j);
    // V of half -1: zeros (the keys that are read of it: the last sixteen rows of the stage's V)
    if (tid < 16 * G::KCH) *(v4i *)(smem1 + G::KT_BYTES + 48 * G::KROW + 16 * tid) = (v4i){0, 0, 0, 0};
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(2 * LOADS, 0));
    __builtin_amdgcn_s_barrier();
    v4i rk[RING], rv[RING];  // operand c of a half in c % RING; of V^T operand c: rows 32 (c % NDT).., 16-key chunk c / NDT
    v16f sc[2];
    {
        v4i k0[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) k0[c] = *(const v4i *)(smem1 + koff[c]);
#pragma unroll
        for (int c = 0; c < NC; c++) sc[0] = mfma32_16bit<T>(k0[c], qop[c], c == 0 ? cinit : sc[0]);
    }
#pragma unroll
    for (int c = 0; c < RING; c++) rk[c] = *(const v4i *)(smem1 + 32 * G::KROW + koff[c]), rv[c] = (v4i){0, 0, 0, 0};
    v4i pop[2][2];  // [parity of the half][16-key chunk]: P^T operand = accumulator quads 2 cc, 2 cc + 1 of S
#pragma unroll
    for (int c = 0; c < 2; c++) pop[1][c] = (v4i){0, 0, 0, 0};

    auto max3 = [](float x, float y, float z) {
        float r;
        asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "v"(z));
        return r;
    };
    auto iteration = [&](auto half_tag, auto stage_tag, int blk) {  // half half_tag of tile blk, which lives in stage stage_tag
        constexpr int H = decltype(half_tag)::value, PAR = decltype(stage_tag)::value, NU = 2 * NC;
        const uint8_t *st = PAR ? smem1 : smem0;
        uint8_t *other = PAR ? smem0 : smem1;  // the stage before this one, then the next
        v16f &cur = sc[H], &nxt = sc[H ^ 1];
        const int key0 = blk * AT_BK + 32 * H;
        if (key0 + 32 > a.Tkv) {  // keys past the end count as -inf
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (key0 + 8 * (i >> 2) + 4 * half + (i & 3) >= a.Tkv) cur[i] = -INFINITY;
        }
        float mx, shift = 0.0f, alpha = 1.0f, rs = 0.0f;  // rs: this half's row sum, at the new reference
        bool need = false, moved = false;
        // the softmax in sixteen pieces: row maximum of the half (16 scores of this lane, 16 of lane ^ 32) relative to the bias;
        // when it exceeds the allowance, shift = how far the reference moves, alpha = the factor that moves the accumulator there
        // (0 before the first keys); then two scores at a time to packed P values, whose rounded sum is the row sum's share
        auto piece = [&](int v) {
            if (v == 0) {
                mx = max3(cur[0], cur[1], cur[2]);
                mx = max3(mx, cur[3], cur[4]);
            } else if (v < 4) {
                mx = max3(mx, cur[4 * v + 1], cur[4 * v + 2]);
                mx = max3(mx, cur[4 * v + 3], cur[v == 3 ? 15 : 4 * v + 4]);
            } else if (v == 4) {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
                mx = max3(__uint_as_float(sw[0]), __uint_as_float(sw[1]), __uint_as_float(sw[1]));
                need = mx > gap + AT_LAZY;
                moved = __builtin_amdgcn_ballot_w64(need) != 0;
            } else if (v == 5) {
                if (moved) {
                    shift = need ? mx : 0.0f;
                    alpha = __builtin_amdgcn_exp2f(need ? gap - mx : 0.0f);
                    gap = need ? 0.0f : gap;
#pragma unroll
                    for (int i = 0; i < 16; i++) cur[i] -= shift;
                }
            } else if (v < 14) {
                const int k = v - 6;
                uint32_t p = pack2<T>(__builtin_amdgcn_exp2f(cur[2 * k]), __builtin_amdgcn_exp2f(cur[2 * k + 1]));
                asm volatile("" : "+v"(p));  // (not moved to its use in the next iteration)
                pop[H][k >> 2][k & 3] = (int)p;
                rs = T::sum2(p, rs);
            }
        };
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(H);
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const int c = u >> 1, r = c % RING;
#pragma unroll
            for (int v = u * 16 / NU; v < (u + 1) * 16 / NU; v++) piece(v);
            __builtin_amdgcn_sched_barrier(0);
            const bool early = c < RING;
            if (H == 0 && u == NC) {  // my loads of this stage have landed, my reads of the other are done
                __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            if ((u & 1) == 0) {
                nxt = mfma32_16bit<T>(rk[r], qop[c], c == 0 ? cinit : nxt);
                if (early)  // the rest of half j + 1, then the first operands of half j + 2
                    rk[r] = *(const v4i *)((H ? st : other + 32 * G::KROW) + koff[c + RING]);
                else
                    rk[r] = *(const v4i *)(st + H * (32 * G::KROW) + koff[c - RING]);
            } else {
                acc_o[c % NDT] = mfma32_16bit<T>(rv[r], pop[H ^ 1][c / NDT], acc_o[c % NDT]);
                if (early)  // the rest of half j - 1, then the first operands of half j
                    rv[r] = read_v(H ? st : other, (c + RING) % NDT, 2 * (H ^ 1) + (c + RING) / NDT);
                else
                    rv[r] = read_v(st, (c - RING) % NDT, 2 * H + (c - RING) / NDT);
            }
            static_assert(2 * LOADS <= NC, "the block loads fit the second half of an iteration");
            if (H == 0 && u >= NC && u - NC < 2 * LOADS) {
                if (u & 1)
                    issue_k(min(blk + 2, nblk - 1), other, (u - NC) >> 1);
                else
                    issue_v(min(blk + 1, nblk - 1), other, (u - NC) >> 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (moved) {  // accumulator, row sum and the scores already computed to the new reference, later ones start from it
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc_o[dt][i] *= alpha;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                nxt[i] -= shift;
                cinit[i] -= shift;
            }
        }
        l_run += rs;
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<int, 0> I0;
    const std::integral_constant<int, 1> I1;
    auto last_pv = [&](const uint8_t *st, auto half_tag) {  // O^T += V^T P^T of the last half
        constexpr int H = decltype(half_tag)::value;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const v4i v = c < RING ? rv[c % RING] : read_v(st, c % NDT, 2 * H + c / NDT);
            acc_o[c % NDT] = mfma32_16bit<T>(v, pop[H][c / NDT], acc_o[c % NDT]);
        }
    };
    {
        int blk = 0;
        for (; 2 * blk + 4 <= nhalf; blk += 2) {
            iteration(I0, I0, blk);
            iteration(I1, I0, blk);
            iteration(I0, I1, blk + 1);
            iteration(I1, I1, blk + 1);
        }
        const int left = nhalf - 2 * blk;  // 0 .. 3
        if (left >= 1) iteration(I0, I0, blk);
        if (left >= 2) iteration(I1, I0, blk);
        if (left == 3) iteration(I0, I1, blk + 1);
        if (left == 0)
            last_pv(smem1, I1);
        else if (left == 1)
            last_pv(smem0, I0);
        else if (left == 2)
            last_pv(smem0, I1);
        else
            last_pv(smem1, I0);
    }

    // ---- O = O^T / l, staged through LDS so that rows leave as 256-byte segments -------------------------------------
    l_run += __shfl_xor(l_run, 32);
    const float inv = 1.0f / (l_run == 0.0f ? 1.0f : l_run);
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));  // the redundant last tile load has landed
    uint16_t *op = (uint16_t *)a.o + (long)b * a.sob + (long)h * D;
    constexpr int OCH = D / 8, OROWS = 64 * WAVES / OCH;  // 16-byte chunks per output row, rows per pass
    const int c = tid % OCH;
#pragma unroll
    for (int part = 0; part < WAVES / 4; part++) {  // 128 rows at a time
        __syncthreads();
        if (WAVES == 4 || wave >> 2 == part) {
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    uint2 w;
                    w.x = pack2<T>(acc_o[dt][4 * j] * inv, acc_o[dt][4 * j + 1] * inv);
                    w.y = pack2<T>(acc_o[dt][4 * j + 2] * inv, acc_o[dt][4 * j + 3] * inv);
                    *(uint2 *)((wave & 2 ? smem1 : smem0) + ((wave & 1) * 32 + l32) * G::OPITCH + (32 * dt + 8 * j + 4 * half) * 2) = w;
                }
        }
        __syncthreads();
#pragma unroll
        for (int pass = 0; pass < 128 / OROWS; pass++) {
            const int row = pass * OROWS + tid / OCH, q = q0 + 128 * part + row;
            if (q < a.Tq) *(v4i *)(op + (long)q * a.som + 8 * c) = *(const v4i *)((row < 64 ? smem0 : smem1) + (row & 63) * G::OPITCH + c * 16);
        }
    }
}

// Whether workgroups of 256 queries (eight wavefronts, one workgroup to a CU) are the faster ones than two of 128 to a CU: they fetch a
// tile of K and V once for eight wavefronts and not for four, which at head dimension 128 is 2 to 7 % of a launch.  A round of them
// counts 0.97 of a round of two workgroups of 128, and one workgroup of 128 alone on a CU 0.565 (28 heads x 4608: 504 workgroups of
// 256 252.8 us, 1008 of 128 258.7; 7 heads, 252 of 128 73, 126 of 256 93).  With few keys a launch is mostly beginnings and ends of
// workgroups, which two to a CU hide from each other: beyond one round 77 keys 1.00 to 1.16 of the time, 512 1.02 to 1.10, 2500 0.96
// to 0.97; within one, 256 keys at 480 workgroups of 128 1.015, at 432 0.99.  us, 128 / 256 queries (bf16): 24 x 4608 234 / 225, 24 x 2000
// 52.5 / 49.9, 24 x 8192 672 / 658, 10 x 4608 112 / 108, 20 x 3000 87.8 / 87.0.  Head dimension 64: 40 x 4096 169 / 192.
static bool wide_queries(const svdq_attention_args &a, int cus) {
    if (a.D != 128) return false;
    const long wg4 = (long)((a.Tq + 127) / 128) * a.H * a.B, wg8 = (long)((a.Tq + 255) / 256) * a.H * a.B;
    const long deep = (wg4 + cus - 1) / cus, rounds = (wg8 + cus - 1) / cus;  // workgroups of 128 on the fullest CU
    if (0.97 * (double)rounds >= (double)(deep / 2) + (deep % 2 ? 0.565 : 0.0)) return false;
    return rounds > 1 ? a.Tkv >= 2048 : a.Tkv >= 1024 || 4 * wg4 <= 7L * cus;
}

template <typename T, int D, int WAVES>
static void launch_attention(const svdq_attention_args &a, hipStream_t s) {
    const int ntile = (a.Tq + 32 * WAVES - 1) / (32 * WAVES), xcd_heads = (a.B * a.H) % 8 == 0;
    hipLaunchKernelGGL((attention_kernel<T, D, WAVES>), dim3((unsigned)(ntile * a.H * a.B)), dim3(64 * WAVES), 0, s, a, ntile, xcd_heads);
}
template <typename T>
static void launch_attention(const svdq_attention_args &a, hipStream_t s) {
    if (wide_queries(a, cu_count()))
        launch_attention<T, 128, 8>(a, s);
    else if (a.D == 128)
        launch_attention<T, 128, 4>(a, s);
    else
        launch_attention<T, 64, 4>(a, s);
}

}  // namespace svdq

using namespace svdq;

extern "C" int svdq_attention_queries(const svdq_attention_args *args, int32_t cus) {
    return args && args->B > 0 && args->H > 0 && args->Tq > 0 && wide_queries(*args, cus > 0 ? cus : cu_count()) ? 256 : 128;
}

extern "C" int svdq_attention_fp16(const svdq_attention_args *args, void *stream) {
    if (!args) {
        set_error("svdq_attention_fp16: null args");
        return SVDQ_E_INVALID;
    }
    const svdq_attention_args &a = *args;
    if (a.dtype != SVDQ_BF16 && a.dtype != SVDQ_FP16) {
        set_error("svdq_attention_fp16: dtype %d", a.dtype);
        return SVDQ_E_INVALID;
    }
    if (a.D != 128 && a.D != 64) {
        set_error("svdq_attention_fp16: head dimension %d is not supported (128 and 64 only)", a.D);
        return SVDQ_E_UNSUPPORTED;
    }
    if (a.B <= 0 || a.H <= 0 || a.Tq < 0 || a.Tkv <= 0 || a.B > 65535 || a.H > 65535) {
        set_error("svdq_attention_fp16: bad shape B=%d H=%d Tq=%d Tkv=%d", a.B, a.H, a.Tq, a.Tkv);
        return SVDQ_E_INVALID;
    }
    if (!a.q || !a.k || !a.v || !a.o) {
        set_error("svdq_attention_fp16: null tensor");
        return SVDQ_E_INVALID;
    }
    auto al = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
    if (!al(a.q) || !al(a.k) || !al(a.v) || !al(a.o) || a.sqm % 8 || a.sqh % 8 || a.sqb % 8 || a.skn % 8 ||
        a.skh % 8 || a.skb % 8 || a.svn % 8 || a.svh % 8 || a.svb % 8 || a.som % 8 || a.sob % 8) {
        set_error("svdq_attention_fp16: tensors and their row / head / batch strides must be 16-byte aligned");
        return SVDQ_E_INVALID;
    }
    if (a.Tq == 0) return SVDQ_OK;
    const int Tpad = (a.Tkv + AT_BK - 1) / AT_BK * AT_BK;
    if (((size_t)Tpad * a.svn + a.D) * 2 >= ((size_t)1 << 31) || ((size_t)Tpad * a.skn + a.D) * 2 >= ((size_t)1 << 31) ||
        (size_t)a.B * a.H * ((a.Tq + 127) / 128) >= ((size_t)1 << 31)) {
        set_error("svdq_attention_fp16: Tq=%d Tkv=%d key / value stride %lld / %lld: too large for 32-bit tile offsets", a.Tq, a.Tkv,
                  (long long)a.skn, (long long)a.svn);
        return SVDQ_E_UNSUPPORTED;
    }
    if (a.skn < a.D || a.svn < a.D) {
        set_error("svdq_attention_fp16: key or value rows overlap (stride %lld / %lld < head dimension)", (long long)a.skn, (long long)a.svn);
        return SVDQ_E_INVALID;
    }
    hipStream_t s = (hipStream_t)stream;
    if (a.dtype == SVDQ_BF16)
        launch_attention<BF16>(a, s);
    else
        launch_attention<FP16>(a, s);
    return check_launch("svdq_attention_fp16");
}
