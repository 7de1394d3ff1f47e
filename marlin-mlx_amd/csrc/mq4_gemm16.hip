// Prefill-shaped (large M) MLX-affine Q4 GEMM for gfx950 with the weights
// dequantized to fp16 in registers and fed to the fp16 MFMA.
//
// Same call sites as mq4_gemm.hip: qmatmul (src/model/marlin.cpp:18-25)
// inside mlp_forward (:31-35) over all S prompt tokens, with the rms_norm in
// front (:141, :12-16) and the swiglu (:27-29) fused in; used for both
// products of mq4_mlp_residual: gate/up with the SwiGLU epilogue, and down
// with the residual add (:142), whole or in K parts whose fp32 sums
// kpart_residual_kernel adds in order.
//
//   Y[M, N] = X[M, K] . W[N, K]^T,  W[n, k] = s[n, g] * q[n, k] + b[n, g],  g = k / 64
//
// mq4_gemm.hip keeps both MFMA operands exact (x and 128 + q in bf16) and
// folds every group into the fp32 result with the VALU, two instructions per
// output and group: at 64 x 64 outputs per wave that fold is as long as the
// group's MFMAs, and the kernel is VALU-bound.  Here each weight is formed
// once as w = fp16(s q + b), one rounding (v_pk_fma_f16 on exact fp16 q, s
// and b), and the MFMA accumulates x . w straight into the result: no fold.
// s q + b of a bf16 scale and bias and a 4-bit q mostly fits fp16's 11-bit
// significand, so most weights are exact; on 0.02-std Gaussian weights the
// product's error is 2.4e-6 of the output rms (max 1.5e-4), against about
// 1e-5 for the exact-operand kernel's fp32 fold.  Scales and biases convert
// to fp16 exactly in its normal range (beyond 65504 a weight would not be
// finite; below 2^-14 the conversion is subnormal, an absolute error under
// 2^-25).
//
// The activations are an fp16 copy of the bf16 operand in the MFMA pair
// order (launch_pair_rows16: normalized x), each row scaled by a power of two
// 2^-e (e = 0 unless the row holds values of 2^15 or more) that the epilogue
// multiplies back exactly, so any bf16 input stays finite.  A bf16 value
// converts to fp16 exactly unless it lies below 2^-14 (2^-14 + e), where
// fp16 is subnormal: an absolute error under 2^-25 of the row's scale.
//
// Work decomposition:
//  * A wave takes 32 RI rows and 64 weight columns (gate/up: 32 gate and the
//    same 32 up columns) as RI x 2 v_mfma_f32_32x32x16_f16 tiles and
//    dequantizes its own weights: 13 VALU per packed word of eight (a
//    v_and_or_b32 forms two fp16 1024 + q, a v_pk_add_f16 takes the 1024 off,
//    a v_pk_fma_f16 applies s and b to the pair, one shift per word).  What a
//    wave issues bounds it: 112 VALU per k group against 8 RI MFMAs of 14 ns
//    (one wave per SIMD issues a VALU every 2.4 ns, two waves one every
//    2.0 ns, MFMAs of either wave running beside them), so RI = 4 wherever
//    the rows fill it, and as little else in the loop as possible: 8 groups
//    unrolled, every LDS address a constant, scales and biases read once per
//    8 groups.
//  * The ring and the schedule are in gemm16_tile, the tile shapes and the
//    rule that picks one in tile_for.  At full load (M = 8192) the card holds
//    the clock at 1.7-1.8 GHz (2.4 at most) with the socket at 1334 W of its
//    1400 W cap, and MFMAs are busy 57% of the cycles; a large library product
//    runs at 1.9-2.0 GHz and 1395 W, 59% busy.  So power management sets the
//    pace there, and fewer instructions per product are what is left.
//  * Per 64-k group, the activations (each row's eight 16-byte chunks
//    XOR-swizzled by (row / 2) % 8: the 16 lanes of a ds_read_b128 phase, 16
//    rows at one chunk, cover the 64 banks once) and the packed weights (per
//    32 columns one DMA instruction, lane l reading k-half l / 32 of column
//    l % 32, so that the stage holds each k-half's 32 columns in consecutive
//    slots) go to LDS by DMA; the columns' scales and biases follow every
//    eight groups (16 bytes per column, two slots).  Barriers carry no memory
//    fence.  (Per-group DMA of the scales, four bytes from 64 columns per
//    instruction, made the kernel bound by L2 requests.)
//  * Activations are stored by k group, [group][row][64], so that a tile's
//    group is one contiguous run.
//  * The operand layout is mq4_gemm.hip's: lane l of a tile holds row (or
//    weight column) l % 32 and k-half l / 32; MFMA step ks takes word ks of
//    the half, whose nibble pairs (q_p, q_{p+4}) meet the activations in the
//    pair order (x_p, x_{p+4}) of the pre-pass.  The weights are the MFMA's
//    row operand and the activations its column operand, so that a result
//    lane holds one activation row and four runs of four consecutive weight
//    columns: the epilogue reads one row scale per 32 rows and writes 8-byte
//    runs.
#include <type_traits>

#include "mq4_device.h"
#include "mq4_gemm.h"
#include "mq4_gemv.h"
#include "mq4_host.h"
#include "mq4_stage.h"

namespace mq4 {

namespace g16 {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int NJ = 2;                     // 32-column MFMA tiles per wave (SwiGLU: a gate and an up tile)

// A block of KW teams of WR x WC waves, each wave 32 RI rows x 64 weight
// columns; the teams compute the same tile over their own parts of K.
template <int WR, int WC, int RI, int KW>
struct Shape {
    static constexpr int NW = WR * WC, THREADS = 64 * NW * KW;
    static constexpr int TBM = 32 * RI * WR;            // rows per block
    static constexpr int BNW = 32 * NJ * WC;            // weight columns per block
    static constexpr int A_I = TBM / 8 / NW;            // activation DMA instructions per wave and group
    static constexpr int B_I = BNW / 32 / NW;           // weight DMA instructions per wave and group
    static constexpr int SB_I = 2 * BNW / 64 / NW;      // scale/bias DMA instructions per wave and 8 groups
    static constexpr int LUT_I = SILU_LUT_N / 512 / (NW * KW); // SiLU table DMA instructions per wave
    static_assert(A_I * 8 * NW == TBM && B_I * 32 * NW == BNW && SB_I * 64 * NW == 2 * BNW &&
                      LUT_I * 512 * NW * KW == SILU_LUT_N,
                  "every wave issues the same DMA");
};

// One k group: activations [row][chunk ^ ((row >> 1) & 7)] (fp16 pairs) and
// packed weights [32-column block][k-half][column].
template <int TBM, int BNW>
struct Stage {
    uint4 a[TBM * 8];
    uint4 b[2 * BNW];
};
// A team's ring: S stages; scales and biases of 8 groups, [scales |
// biases][weight column], 16 bytes (groups 8 t .. 8 t + 7) each, two slots.
template <int TBM, int BNW, int S>
struct Ring {
    Stage<TBM, BNW> st[S];
    uint4 sb[2][2][BNW];
};
template <int EPI, int TBM, int BNW, int S, int KW>
struct Smem {
    Ring<TBM, BNW, S> ring[KW];
    __align__(16) uint16_t lut[EPI == GEMM_SWIGLU ? SILU_LUT_N : 8];
};

// A bf16 value (its float bits) as a pair of the same fp16 (round to nearest
// even; exact for bf16 values of fp16's normal range).
__device__ __forceinline__ h2_t bf16_to_h2(uint32_t float_bits) {
    const _Float16 v = (_Float16)__uint_as_float(float_bits);
    return (h2_t){v, v};
}

__device__ __forceinline__ uint32_t word_of(const uint4& v, int i) {
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

// (s & m) | c in one v_and_or_b32, the mask in an SGPR and the exponent
// bits in a VGPR, both set up once by the caller: the nibbles m selects in
// each 16-bit half as fp16 mantissa bits under c's exponents.  (Not as asm:
// see weight_operand_k in mq4_gemm.hip.)
__device__ __forceinline__ uint32_t nib_pair_h(uint32_t s, uint32_t m, uint32_t c) {
    return (s & m) | c;
}

// The eight fp16 weights fp16(s q + b) of one packed word, in the nibble-pair
// order (q0, q4), (q1, q5), (q2, q6), (q3, q7).  Pairs 0 and 2 are the low
// nibbles of each half of w and of w >> 8, under the exponent of 1024 (fp16
// 1024 + q); pairs 1 and 3 are their high nibbles, left in place (bits 4-7
// of the half) under the exponent of 64, whose mantissa step is 1/16 (fp16
// 64 + q): one shift per word instead of three.  m_lo / c_lo = 0x000f000f /
// 0x64006400, m_hi / c_hi = 0x00f000f0 / 0x54005400.
__device__ __forceinline__ h8_t dequant_word(uint32_t w, h2_t s2, h2_t b2, uint32_t m_lo, uint32_t c_lo,
                                             uint32_t m_hi, uint32_t c_hi) {
    const h2_t k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    const h2_t k64 = {(_Float16)64.0f, (_Float16)64.0f};
    const uint32_t w8 = w >> 8;
    const h2_t q[4] = {__builtin_bit_cast(h2_t, nib_pair_h(w, m_lo, c_lo)) - k1024,      // exact
                       __builtin_bit_cast(h2_t, nib_pair_h(w, m_hi, c_hi)) - k64,
                       __builtin_bit_cast(h2_t, nib_pair_h(w8, m_lo, c_lo)) - k1024,
                       __builtin_bit_cast(h2_t, nib_pair_h(w8, m_hi, c_hi)) - k64};
    uint32_t out[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) out[p] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q[p], s2, b2));
    return __builtin_bit_cast(h8_t, make_uint4(out[0], out[1], out[2], out[3]));
}

// Column of an 8-column chunk whose pair-order position (2 (c % 4) + c / 4)
// is r.
__device__ __forceinline__ int perm8(int r) { return 4 * (r & 1) + (r >> 1); }

// One block's tile: rows m0 .. m0 + TBM - 1, weight columns of n0 .., K part
// kpart of S_K (split again over the block's KW teams).
template <int EPI, int WR, int WC, int RI, int S, int KW, class Sm>
__device__ __forceinline__ void gemm16_tile(const Gemm16Args& p, Sm& smem_all, int n0, int m0, int kpart, int S_K) {
#pragma clang fp contract(off)
    using Sh = Shape<WR, WC, RI, KW>;
    static_assert(EPI == GEMM_SWIGLU || EPI == GEMM_RESIDUAL, "the epilogues of mq4_mlp_residual");
    constexpr int NMAT = EPI == GEMM_SWIGLU ? 2 : 1;
    constexpr int TBM = Sh::TBM, BNW = Sh::BNW, A_I = Sh::A_I, B_I = Sh::B_I, SB_I = Sh::SB_I;
    constexpr int BN = BNW / NMAT;                       // output columns per block
    constexpr int D = A_I + B_I;                         // DMA instructions per wave and stage
    static_assert((S == 2 || S == 4) && D * (S - 1) < 64, "ring depth");

    const int tid = threadIdx.x, lane = tid & 63;
    const int bwave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int team = bwave / Sh::NW, wave = bwave % Sh::NW;
    const int wr_ = wave / WC, wc = wave % WC;           // wave row and wave column of the block
    const int h = lane >> 5, col = lane & 31;
    const int M = p.M, N = p.N, K = p.K, G = K / 64;
    const int GL = G / (S_K * KW), g0 = (kpart * KW + team) * GL;   // this team's groups g0 .. g0 + GL - 1
    auto& smem = smem_all.ring[team];

    // ---- DMA sources: wave-uniform pointers, moved along K one group per
    // step, plus 32-bit lane byte offsets ----
    const int64_t xg = (int64_t)M * 128;               // bytes of one group's rows
    const char* xp = reinterpret_cast<const char*>(p.x) + g0 * xg;
    uint32_t aoff[A_I];
#pragma unroll
    for (int t = 0; t < A_I; ++t) {
        const int slot = (wave * A_I + t) * 64 + lane;
        const int r = slot >> 3, c = (slot & 7) ^ ((r >> 1) & 7);
        const int row = (m0 + r) < M ? (m0 + r) : (M - 1);
        aoff[t] = (uint32_t)(row * 128 + c * 16);
    }
    // weight column r of the block -> matrix and output row (rows past N
    // repeat row N - 1, never stored)
    auto wrow_of = [&](int r) -> int {
        const int n = NMAT == 2 ? n0 + (r % (BNW / 2)) : n0 + r;
        return n < N ? n : N - 1;
    };
    auto mat_of = [&](int r) -> const QMat& { return (NMAT == 2 && r >= BNW / 2) ? p.B : p.A; };
    // packed weights: instruction t covers 32 weight columns, lane l takes
    // k-half l / 32 of column l % 32 (its group's 32 bytes as two 16-byte
    // halves), so the stage holds [32-column block][k-half][column] and the
    // operand reads of a k-half are 32 consecutive 16-byte slots
    const char* bp[B_I];
    uint32_t boff[B_I];
#pragma unroll
    for (int t = 0; t < B_I; ++t) {
        const int r0 = (wave * B_I + t) * 32;
        bp[t] = reinterpret_cast<const char*>(mat_of(r0).wq) + (int64_t)g0 * 32;
        boff[t] = (uint32_t)((int64_t)wrow_of(r0 + (lane & 31)) * (K / 2) + (lane >> 5) * 16);
    }
    // scales and biases: 16 bytes (8 groups) of one weight column per lane
    const char* sbp[SB_I];
    uint32_t sboff[SB_I];
#pragma unroll
    for (int t = 0; t < SB_I; ++t) {
        const int u0 = (wave * SB_I + t) * 64, sel = u0 / BNW, r0 = u0 % BNW;
        sbp[t] = reinterpret_cast<const char*>(sel ? mat_of(r0).b : mat_of(r0).s) + (int64_t)(g0 / 8) * 16;
        sboff[t] = (uint32_t)((int64_t)wrow_of(r0 + lane) * G * 2);
    }
    // LDS byte addresses of this wave's DMA blocks in stage 0 and slot 0
    const uint32_t a_lds = stage::lds_addr(&smem.st[0].a[0]) + (uint32_t)(wave * A_I * 1024);
    const uint32_t b_lds = stage::lds_addr(&smem.st[0].b[0]) + (uint32_t)(wave * B_I * 1024);
    const uint32_t sb_lds = stage::lds_addr(&smem.sb[0][0][0]) + (uint32_t)(wave * SB_I * 1024);
    constexpr uint32_t STG = sizeof(smem.st[0]), SBS = sizeof(smem.sb[0]);
    // the group xp / bp point at -> ring stage `slot`; then the pointers move
    // on by `step` groups (0 at the end of K: the last group again)
    auto issue = [&](int slot, int step) {
#pragma unroll
        for (int t = 0; t < A_I; ++t) stage::dma16_m0(xp, aoff[t], a_lds + slot * STG + t * 1024);
#pragma unroll
        for (int t = 0; t < B_I; ++t) stage::dma16_m0(bp[t], boff[t], b_lds + slot * STG + t * 1024);
        xp += step * xg;
#pragma unroll
        for (int t = 0; t < B_I; ++t) bp[t] += step * 32;
    };
    auto issue_sb = [&](uint32_t slot, int step) {     // the next eight groups' scales and biases
#pragma unroll
        for (int t = 0; t < SB_I; ++t) {
            stage::dma16_m0(sbp[t], sboff[t], sb_lds + slot * SBS + t * 1024);
            sbp[t] += step * 16;
        }
    };

    // ---- this lane's weight columns (block-relative) of tiles j = 0, 1 ----
    // Weight column c of a tile is MFMA row c, except for outputs in the
    // pair order: there MFMA row 8 b + r holds column 8 b + perm8(r), so that
    // the four consecutive MFMA rows of a result lane are four consecutive
    // positions of the pair order.
    const bool f16_out = EPI == GEMM_SWIGLU && p.yscale != 0.0f;
    const bool paired_out = EPI == GEMM_SWIGLU && !f16_out && p.ysum != nullptr;
    const int ccol = f16_out || paired_out ? ((col & ~7) | perm8(col & 7)) : col;
    int wr[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) wr[j] = NMAT == 2 ? j * (BNW / 2) + wc * 32 + ccol : wc * (32 * NJ) + j * 32 + ccol;
    // LDS operand addresses (in uint4) within a stage: activation chunk
    // 4 h + ks of row wr_ RI 32 + col (row tile i: + 256 i), packed words of
    // column wr[j]
    uint32_t arow[4], brow[NJ];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) arow[ks] = (uint32_t)((wr_ * RI * 32 + col) * 8 + ((4 * h + ks) ^ ((col >> 1) & 7)));
#pragma unroll
    for (int j = 0; j < NJ; ++j) brow[j] = (uint32_t)((wr[j] >> 5) * 64 + h * 32 + (wr[j] & 31));

    uint32_t nib_mask, nib_exp, nib_mask_hi, nib_exp_hi;   // the nibble-pair constants, set up once
    asm("s_mov_b32 %0, 0x000f000f" : "=s"(nib_mask));
    asm("v_mov_b32 %0, 0x64006400" : "=v"(nib_exp));
    asm("s_mov_b32 %0, 0x00f000f0" : "=s"(nib_mask_hi));
    asm("v_mov_b32 %0, 0x54005400" : "=v"(nib_exp_hi));

    f32x16_t acc[RI][NJ];
#pragma unroll
    for (int i = 0; i < RI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    uint4 bw[NJ];                                      // a group's packed words
    uint4 sv[NJ], bv[NJ];                              // eight groups' scales and biases
    h2_t s2[NJ], b2[NJ];                               // a group's, as fp16 pairs
    auto read_w = [&](int slot) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) bw[j] = smem.st[slot].b[brow[j]];
    };
    auto read_sb = [&](uint32_t slot) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            sv[j] = smem.sb[slot][0][wr[j]];
            bv[j] = smem.sb[slot][1][wr[j]];
        }
    };
    auto group_sb = [&](int u) {                       // group u of the eight
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            s2[j] = bf16_to_h2(u & 1 ? word_of(sv[j], u >> 1) & 0xffff0000u : word_of(sv[j], u >> 1) << 16);
            b2[j] = bf16_to_h2(u & 1 ? word_of(bv[j], u >> 1) & 0xffff0000u : word_of(bv[j], u >> 1) << 16);
        }
    };
    auto read_a = [&](int slot, int ks, h8_t (&a)[RI]) {
#pragma unroll
        for (int i = 0; i < RI; ++i) a[i] = __builtin_bit_cast(h8_t, smem.st[slot].a[arow[ks] + 256 * i]);
    };
    auto dequant = [&](int ks, h8_t (&bo)[NJ]) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            bo[j] = dequant_word(word_of(bw[j], ks), s2[j], b2[j], nib_mask, nib_exp, nib_mask_hi, nib_exp_hi);
    };
    // The weights are the MFMA row operand and the activations the column
    // operand: result lane l of tile (i, j) holds activation row i 32 + l % 32.
    auto mfmas = [&](const h8_t (&a)[RI], const h8_t (&bo)[NJ]) {
#pragma unroll
        for (int i = 0; i < RI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bo[j], a[i], acc[i][j], 0, 0, 0);
    };
    auto interleave = [] {                             // one LDS read and the dequantization per MFMA
#pragma unroll
        for (int m = 0; m < RI * NJ; ++m) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                   // MFMA
            if (m < RI) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // LDS read
            __builtin_amdgcn_sched_group_barrier(0x002, 28 / (RI * NJ), 0);      // VALU
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- prologue: the table, the first scales and S stages in flight ----
    if constexpr (EPI == GEMM_SWIGLU) {
#pragma unroll
        for (int t = 0; t < Sh::LUT_I; ++t)
            stage::dma16_m0(p.silu_lut, (uint32_t)((bwave * Sh::LUT_I + t) * 1024 + lane * 16),
                            stage::lds_addr(smem_all.lut) + (uint32_t)((bwave * Sh::LUT_I + t) * 1024));
    }
    const int nblk = GL / 8;                           // eight-group blocks of this K part
    issue_sb(0, nblk > 1 ? 1 : 0);
#pragma unroll
    for (int s = 0; s < S; ++s) issue(s, 1);           // GL >= 8 > S
    wait_vmcnt<D * (S - 1)>();
    lds_barrier();                                     // stage 0 (and the table) is in for every wave
    h8_t a0[RI], a1[RI], w0[NJ], w1[NJ];
    read_w(0);
    read_sb(0);
    read_a(0, 0, a0);
    group_sb(0);
    dequant(0, w0);

    // Step u of an eight-group block computes its group from stage u % S
    // (S divides 8: every LDS address in the step is a constant).  MFMA step
    // ks + 1's activation reads and dequantization are issued during step
    // ks's MFMAs (two operand sets); before the last MFMA step the waves meet
    // (each has read all of the stage, and has waited for its own DMA of the
    // next one), so that during it the next group's operands are read and the
    // group S ahead goes into the free stage: a step never starts by waiting
    // for its operands.  Every step issues D DMA instructions (past the end:
    // the last group again, into a stage that nobody reads), so one constant
    // vmcnt serves every step; a block's scales and biases go out just before
    // its first group.
    for (int t8 = 0; t8 < nblk; ++t8) {
        const bool more = t8 + 1 < nblk;               // another block follows
        const int inc = more ? 1 : 0, sb_inc = t8 + 2 < nblk ? 1 : 0;
        const uint32_t nsb = (uint32_t)(t8 + 1) & 1;
        auto step = [&](auto uc) {
            constexpr int u = decltype(uc)::value, cs = u % S, ns = (u + 1) % S;
            mfmas(a0, w0);
            read_a(cs, 1, a1);
            dequant(1, w1);
            interleave();
            mfmas(a1, w1);
            read_a(cs, 2, a0);
            dequant(2, w0);
            interleave();
            mfmas(a0, w0);
            read_a(cs, 3, a1);
            dequant(3, w1);
            interleave();
            wait_vmcnt<D * (S - 2)>();
            lds_barrier();
            read_w(ns);
            if constexpr (u == 7) read_sb(nsb);        // past the end: stale bytes, not used
            read_a(ns, 0, a0);
            issue(cs, u + S + 1 < 8 ? 1 : inc);
            if constexpr (u == 7 - S) issue_sb(nsb, sb_inc);
            mfmas(a1, w1);
            group_sb((u + 1) & 7);
            dequant(0, w0);
            __builtin_amdgcn_sched_barrier(0);
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        step(std::integral_constant<int, 4>{});
        step(std::integral_constant<int, 5>{});
        step(std::integral_constant<int, 6>{});
        step(std::integral_constant<int, 7>{});
    }
    wait_vmcnt<0>();                                 // no DMA outstanding past the loop

    // Teams: each takes over OWN of every wave's row tiles, adding the teams'
    // sums in team order; they travel through LDS (the rings, free now), each
    // lane's 16 values of a tile as four 16-byte slots.
    constexpr int OWN = KW <= RI ? RI / KW : 1;
    auto mine = [&](int i) { return KW == 1 || i / OWN == team; };   // row tiles this wave writes
    if constexpr (KW > 1) {
        static_assert(KW >= RI || RI % KW == 0, "whole row tiles per team");
        constexpr int CAP = KW <= RI ? RI - OWN : RI;  // row tiles a team hands over, at most
        f32x4_t* ex = reinterpret_cast<f32x4_t*>(&smem_all.ring[0]);
        static_assert((size_t)KW * Sh::NW * CAP * NJ * 4 * 64 * 16 <= sizeof(smem_all.ring), "exchange area");
        auto slot = [&](int k, int i) {
            return (((k * Sh::NW + wave) * CAP + (KW <= RI && i / OWN > k ? i - OWN : i)) * NJ) * 4 * 64 + lane;
        };
        lds_barrier();                                 // every wave is done with its ring
#pragma unroll
        for (int i = 0; i < RI; ++i) {
            if (mine(i)) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    ex[slot(team, i) + (j * 4 + q) * 64] = (f32x4_t){acc[i][j][4 * q], acc[i][j][4 * q + 1],
                                                                    acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        }
        lds_barrier();
#pragma unroll
        for (int i = 0; i < RI; ++i) {
            if (!mine(i)) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    f32x4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int k = 0; k < KW; ++k) {
                        const f32x4_t own = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                             acc[i][j][4 * q + 3]};
                        const f32x4_t v = k == i / OWN ? own : ex[slot(k, i) + (j * 4 + q) * 64];
                        sum = k == 0 ? v : sum + v;
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][4 * q + r] = sum[r];
                }
        }
    }

    // ---- epilogue: result lane l of tile (i, j) holds activation row
    // i 32 + l % 32 and MFMA rows (e / 4) 8 + (l / 32) 4 + e % 4 of tile j:
    // four runs of four consecutive output columns (natural order, or the
    // pair-order positions 4 (l / 32) .. + 3 of an 8-column chunk), each
    // stored as one 8-byte (16 for fp32) write.
    // SwiGLU with ysum: h also goes to an LDS tile in natural column order
    // (the ring stages, free once every wave is past its last group), for
    // the group sums of its rows.
    constexpr int TS = BN + 8;                                     // bf16 per epilogue tile row
    uint16_t* tile = reinterpret_cast<uint16_t*>(&smem_all.ring[0]);   // [TBM][TS] bf16
    static_assert(EPI != GEMM_SWIGLU || TBM * TS * 2 <= (int)sizeof(smem_all.ring), "epilogue tile");
    // whole-run vector stores: N % 4 == 0 and 8-byte aligned y and res
    // (16-byte aligned fp32 parts)
    const bool vec = N % 4 == 0 &&
                     (S_K > 1 ? reinterpret_cast<uintptr_t>(p.part) % 16 == 0
                            : reinterpret_cast<uintptr_t>(p.y) % 8 == 0 &&
                                  (EPI != GEMM_RESIDUAL || reinterpret_cast<uintptr_t>(p.res) % 8 == 0));
    const float ascale = p.ascale != 0.0f ? p.ascale : 1.0f;
    // The lane's row scales, loaded together (one wait, not one per row
    // tile).
    float scv[RI];
#pragma unroll
    for (int i = 0; i < RI; ++i) {
        const int row = m0 + (wr_ * RI + i) * 32 + col;
        scv[i] = (p.xscale && row < M ? p.xscale[row] : 1.0f) * ascale;
    }
    // One-part residual epilogue: the residual runs of all row tiles
    // are loaded before the first is written (one wait, not one per run).
    // In place (res == y) every element is read and written by the same
    // lane, the read first.
    const bool res_runs = EPI == GEMM_RESIDUAL && S_K == 1;
    uint2 resv[RI][4 * NJ];
    const bool res_whole = vec && n0 + BN <= N;          // every run of the block: one 8-byte load
    auto load_res = [&](int i, uint2 (&rv)[4 * NJ]) {
        const int row = m0 + (wr_ * RI + i) * 32 + col;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int eg = 0; eg < 4; ++eg) {
                const int cb = n0 + wc * (32 * NJ) + j * 32 + eg * 8 + h * 4;
                uint2 t = make_uint2(0u, 0u);
                if (row < M && cb < N) {
                    const uint16_t* r = p.res + (int64_t)row * N + cb;
                    if (vec && cb + 3 < N) {
                        t = *reinterpret_cast<const uint2*>(r);
                    } else {
                        uint32_t e[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q) e[q] = cb + q < N ? r[q] : 0u;
                        t = make_uint2(e[0] | (e[1] << 16), e[2] | (e[3] << 16));
                    }
                }
                rv[j * 4 + eg] = t;
            }
    };
    if (res_runs) {
        if (res_whole) {
            // rows past M read row M - 1 (never stored): no branch between
            // the loads
#pragma unroll
            for (int i = 0; i < RI; ++i) {
                if (!mine(i)) continue;
                const int row = m0 + (wr_ * RI + i) * 32 + col;
                const uint16_t* r = p.res + (int64_t)(row < M ? row : M - 1) * N + n0 + wc * (32 * NJ) + h * 4;
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int eg = 0; eg < 4; ++eg)
                        resv[i][j * 4 + eg] = *reinterpret_cast<const uint2*>(r + j * 32 + eg * 8);
            }
        } else {
#pragma unroll
            for (int i = 0; i < RI; ++i)
                if (mine(i)) load_res(i, resv[i]);
        }
    }
    // One wait for the row scales and residual runs, before the first branch
    // of the epilogue: past it the compiler's waits at branch joins would
    // count this tile's stores and drain them.
    wait_vmcnt<0>();
    auto emit = [&](int i) {
        const int rl = (wr_ * RI + i) * 32 + col, row = m0 + rl;
        if (row >= M) return;
        const float sc = scv[i];
        const int64_t rowo = (int64_t)row * N;
        // SwiGLU of the lane's 16 (gate, up) pairs of this tile row
        uint32_t hv[16];
        if (EPI == GEMM_SWIGLU) {
            float ga[16], ua[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                ga[e] = acc[i][0][e] * sc;
                ua[e] = acc[i][1][e] * sc;
            }
            swiglu_bf16_lut_batch<16>(ga, ua, hv, smem_all.lut);
        }
#pragma unroll
        for (int j = 0; j < (NMAT == 2 ? 1 : NJ); ++j) {
#pragma unroll
            for (int eg = 0; eg < 4; ++eg) {
                const int cl = (NMAT == 2 ? wc * 32 : wc * (32 * NJ) + j * 32) + eg * 8 + h * 4;
                const int cb = n0 + cl;                             // first column (position) of the run
                if (cb >= N) continue;
                const bool whole = vec && cb + 3 < N;
                if (EPI == GEMM_SWIGLU) {
                    uint32_t o[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint32_t v = hv[eg * 4 + q];
                        o[q] = v;
                        if (paired_out) tile[rl * TS + (cl & ~7) + perm8(h * 4 + q)] = (uint16_t)v;
                        if (f16_out) {
                            // exact for |h| within [2^-14, 65504] / yscale
                            const float hv = fminf(fmaxf(bf16_to_f32(v) * p.yscale, -65504.0f), 65504.0f);
                            o[q] = __builtin_bit_cast(uint16_t, (_Float16)hv);
                        }
                    }
                    uint16_t* y = reinterpret_cast<uint16_t*>(p.y) +
                                  (f16_out ? ((int64_t)(cb >> 6) * M + row) * 64 + (cb & 63) : rowo + cb);
                    if (whole) {
                        *reinterpret_cast<uint2*>(y) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (cb + q < N) y[q] = (uint16_t)o[q];
                    }
                    continue;
                }
                float v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) v[q] = acc[i][j][eg * 4 + q] * sc;
                if (S_K > 1) {
                    float* y = p.part + (int64_t)kpart * M * N + rowo + cb;
                    if (whole) {
                        *reinterpret_cast<float4*>(y) = make_float4(v[0], v[1], v[2], v[3]);
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (cb + q < N) y[q] = v[q];
                    }
                    continue;
                }
                uint32_t o[4];
                uint16_t* y = reinterpret_cast<uint16_t*>(p.y) + rowo + cb;
                const uint2 t = resv[i][j * 4 + eg];
                const uint32_t rv[4] = {t.x & 0xffffu, t.x >> 16, t.y & 0xffffu, t.y >> 16};
#pragma unroll
                for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16(bf16_to_f32(rv[q]) + round_bf16(v[q]));
                if (whole) {
                    *reinterpret_cast<uint2*>(y) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        if (cb + q < N) y[q] = (uint16_t)o[q];
                }
            }
        }
    };
    if (paired_out) __syncthreads();                               // every wave is done with the stages
#pragma unroll
    for (int i = 0; i < RI; ++i)
        if (mine(i)) emit(i);
    if constexpr (EPI == GEMM_SWIGLU) {
        if (paired_out) {
            // ysum of group n0 / 64 + gi of row rl: a task per row, group and
            // half (32 values summed left to right), then the two halves are
            // added (the order of mq4_gemm.hip's paired SwiGLU output)
            constexpr int GI = BN / 64;
            __syncthreads();
            for (int t = tid; t < TBM * GI * 2; t += Sh::THREADS) {
                const int rl = t / (2 * GI), gi = (t >> 1) % GI, hf = t & 1;
                float sum = 0.0f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint4 v = *reinterpret_cast<const uint4*>(&tile[rl * TS + gi * 64 + hf * 32 + c * 8]);
                    const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        sum += bf16_to_f32(w4[q] & 0xffffu);
                        sum += bf16_to_f32(w4[q] >> 16);
                    }
                }
                const float other = __shfl_xor(sum, 1);
                if (hf == 0 && m0 + rl < M) p.ysum[(int64_t)((n0 >> 6) + gi) * M + m0 + rl] = sum + other;
            }
        }
    }
}

// XCD-aware tile order (block b runs on XCD b % 8).  With many column blocks
// (a multiple of 8) XCD x takes a fixed eighth of them for every row block,
// so its weights stay in its own L2.  With few, that leaves one or two
// columns per XCD and every XCD reads all of the activations (four times the
// weights' bytes per tile): there XCD x takes a contiguous run of the row-major tile order instead.
constexpr int kRowRunCols = 16;
__device__ __forceinline__ void tile_of(int b, int T, int NB, int& nb, int& mb) {
    const int x = b & 7, s = b >> 3;
    if ((NB & 7) == 0 && NB > kRowRunCols) {
        const int per = NB >> 3;
        nb = (s % per) * 8 + x;
        mb = s / per;
    } else {
        const int q = T >> 3, r = T & 7;
        const int t = x * q + (x < r ? x : r) + s;
        nb = t % NB;
        mb = t / NB;
    }
}

// WPE: waves per SIMD the registers are sized for.
template <int EPI, int WR, int WC, int RI, int S, int KW, int WPE>
__global__ __launch_bounds__(64 * WR * WC * KW, WPE) void q4_gemm16_kernel(Gemm16Args p) {
    using Sh = Shape<WR, WC, RI, KW>;
    constexpr int BN = Sh::BNW / (EPI == GEMM_SWIGLU ? 2 : 1);
    __shared__ Smem<EPI, Sh::TBM, Sh::BNW, S, KW> smem;
    static_assert(sizeof(smem) <= 160 * 1024, "LDS of a CU");
    // K parts (GEMM_RESIDUAL): block b takes part b / tiles
    const int S_K = EPI == GEMM_RESIDUAL && p.ksplit > 1 ? p.ksplit : 1;
    int bt = blockIdx.x, kpart = 0;
    if (S_K > 1) {
        const int tiles = (int)gridDim.x / S_K;
        kpart = bt / tiles;
        bt -= kpart * tiles;
    }
    int nb, mb;
    tile_of(bt, (int)gridDim.x / S_K, (p.N + BN - 1) / BN, nb, mb);
    gemm16_tile<EPI, WR, WC, RI, S, KW>(p, smem, nb * BN, mb * Sh::TBM, kpart, S_K);
}

// ---------------------------------------------------------------------------
// Activation pre-pass: one wave per row.  Pass 1 forms the row's sum of
// squares (with the norm; the per-element formula of mq4_rms_norm) and the
// largest |x (1 + w)| (|x| without the norm); pass 2 writes bf16(x r (1 + w))
// (or x), scaled by 2^-e and converted to fp16, in the pair order and by k
// group ([group][row][64]), and xscale[m] = 2^e.  e is the smallest such that the scaled row stays below
// 2^15 (0 for every normalized row whose values stay below 2^15).  With CAP >
// 0 (K <= 512 CAP) a lane keeps its chunks of x and of the norm weight in
// registers between the passes (all loads issued first), so the row is read
// once; the sums keep the chunk order of the reloading form (CAP = 0).  With
// lut, the blocks past the rows' write the SiLU table (silu_lut_entry), one
// entry per thread.
template <bool NORM, int CAP>
__global__ __launch_bounds__(256) void pair_rows16_kernel(const uint16_t* __restrict__ x, int M, int K,
                                                          const uint16_t* __restrict__ nw, float eps,
                                                          uint16_t* __restrict__ xp, float* __restrict__ xscale,
                                                          uint16_t* __restrict__ lut) {
#pragma clang fp contract(off)
    const int row_blocks = (M + 3) / 4;
    if ((int)blockIdx.x >= row_blocks) {
        const uint32_t i = (blockIdx.x - (uint32_t)row_blocks) * 256u + threadIdx.x;
        if (i < (uint32_t)SILU_LUT_N) lut[i] = (uint16_t)silu_lut_entry(i);
        return;
    }
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (m >= M) return;                                  // whole waves
    const int CH = K / 8;
    const uint4* src = reinterpret_cast<const uint4*>(x + (int64_t)m * K);
    const uint4* nw4 = reinterpret_cast<const uint4*>(nw);
    uint4* dst = reinterpret_cast<uint4*>(xp) + (int64_t)m * 8;       // chunk c: + (c / 8) M 8 + c % 8
    constexpr int NC = CAP > 0 ? CAP : 1;
    uint4 xc[NC], wc[NC];
    if (CAP > 0) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int c = lane + 64 * i;
            if (c < CH) {
                xc[i] = src[c];
                wc[i] = NORM ? nw4[c] : make_uint4(0, 0, 0, 0);
            }
        }
    }
    float ss = 0.0f, big = 0.0f;
    auto scan = [&](const uint4& v, const uint4& wv) {
        const uint32_t vw[4] = {v.x, v.y, v.z, v.w};
        const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (NORM) ss = sumsq_word(ss, vw[q]);
            const float a0 = bf16_to_f32(vw[q] & 0xffffu), a1 = bf16_to_f32(vw[q] >> 16);
            const float f0 = NORM ? 1.0f + bf16_to_f32(ww[q] & 0xffffu) : 1.0f;
            const float f1 = NORM ? 1.0f + bf16_to_f32(ww[q] >> 16) : 1.0f;
            big = fmaxf(big, fmaxf(fabsf(a0 * f0), fabsf(a1 * f1)));
        }
    };
    if (CAP > 0) {
#pragma unroll
        for (int i = 0; i < NC; ++i)
            if (lane + 64 * i < CH) scan(xc[i], wc[i]);
    } else {
        for (int c = lane; c < CH; c += 64) scan(src[c], NORM ? nw4[c] : make_uint4(0, 0, 0, 0));
    }
    float r = 1.0f;
    if (NORM) r = rms_inv(wave_sum(ss), K, eps);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) big = fmaxf(big, __shfl_xor(big, off));
    big *= NORM ? r : 1.0f;
    // the largest output is below big * (1 + 2^-8) (one bf16 rounding)
    int e = 0;
    while (!(big * 1.01f < 32768.0f * __builtin_ldexpf(1.0f, e)) && e < 200) ++e;
    const float down = __builtin_ldexpf(1.0f, -e);
    if (lane == 0) xscale[m] = __builtin_ldexpf(1.0f, e);
    auto emit = [&](int c, uint4 v, const uint4& w) {
        if (NORM)
            v = make_uint4(norm_word(v.x, w.x, r), norm_word(v.y, w.y, r), norm_word(v.z, w.z, r),
                           norm_word(v.w, w.w, r));
        uint32_t pr[4];
        pair_chunk(v, pr, 0.0f);
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const h2_t hv = {(_Float16)(bf16_to_f32(pr[q] & 0xffffu) * down),
                             (_Float16)(bf16_to_f32(pr[q] >> 16) * down)};
            o[q] = __builtin_bit_cast(uint32_t, hv);
        }
        dst[(int64_t)(c >> 3) * M * 8 + (c & 7)] = make_uint4(o[0], o[1], o[2], o[3]);
    };
    if (CAP > 0) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int c = lane + 64 * i;
            if (c < CH) emit(c, xc[i], wc[i]);
        }
    } else {
        for (int c = lane; c < CH; c += 64) emit(c, src[c], NORM ? nw4[c] : make_uint4(0, 0, 0, 0));
    }
}

// y = bf16(res + round_bf16(part[0] + part[1] + ... + part[S - 1])), the
// parts added in order: 4 elements per thread (MN % 4 == 0, 16-byte aligned
// parts, 8-byte aligned res and y), S <= 6.
__global__ __launch_bounds__(256) void kpart_residual_kernel(const float* __restrict__ part, int S, int64_t MN,
                                                             const uint16_t* __restrict__ res,
                                                             uint16_t* __restrict__ y) {
#pragma clang fp contract(off)
    const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (e >= MN) return;
    // every load issued before the first add (S <= 6 parts)
    float4 v[6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if (k < S) v[k] = *reinterpret_cast<const float4*>(part + (int64_t)k * MN + e);
    const uint2 r = *reinterpret_cast<const uint2*>(res + e);
    float4 sum = v[0];
#pragma unroll
    for (int k = 1; k < 6; ++k) {
        if (k < S) {
            sum.x += v[k].x;
            sum.y += v[k].y;
            sum.z += v[k].z;
            sum.w += v[k].w;
        }
    }
    const float sv[4] = {sum.x, sum.y, sum.z, sum.w};
    const uint32_t rv[4] = {r.x & 0xffffu, r.x >> 16, r.y & 0xffffu, r.y >> 16};
    uint32_t o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = f32_to_bf16(bf16_to_f32(rv[q]) + round_bf16(sv[q]));
    *reinterpret_cast<uint2*>(y + e) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
}

}  // namespace g16

int launch_pair_rows16(const uint16_t* x, int M, int K, const uint16_t* norm_w, float eps, uint16_t* xp,
                       float* xscale, uint16_t* silu_lut, hipStream_t st) {
    if (M < 1 || K % 512 != 0) return -1;
    const unsigned blocks = (unsigned)((M + 3) / 4) + (silu_lut ? (unsigned)(SILU_LUT_N / 256) : 0u);
    // rows of at most 4 chunks per lane (K <= 2048) read once
    const bool cached = K / 512 <= 4;
    if (norm_w && cached)
        hipLaunchKernelGGL((g16::pair_rows16_kernel<true, 4>), dim3(blocks), dim3(256), 0, st, x, M, K, norm_w, eps,
                           xp, xscale, silu_lut);
    else if (norm_w)
        hipLaunchKernelGGL((g16::pair_rows16_kernel<true, 0>), dim3(blocks), dim3(256), 0, st, x, M, K, norm_w, eps,
                           xp, xscale, silu_lut);
    else if (cached)
        hipLaunchKernelGGL((g16::pair_rows16_kernel<false, 4>), dim3(blocks), dim3(256), 0, st, x, M, K, norm_w, eps,
                           xp, xscale, silu_lut);
    else
        hipLaunchKernelGGL((g16::pair_rows16_kernel<false, 0>), dim3(blocks), dim3(256), 0, st, x, M, K, norm_w, eps,
                           xp, xscale, silu_lut);
    return 0;
}

namespace g16 {

// The tile of a product: rows x weight columns (gate/up: half of them each).
//   T64x128:  two teams of 2 waves (64 x 64 each) on halves of K, 4 stages
//   T128x128: 4 waves of 64 x 64, 4 stages
//   T128x256: 4 waves of 128 x 64, 2 stages, two blocks per CU
//   T256x256: 8 waves of 128 x 64, 2 stages
// Few rows leave CUs idle and each block serial: the smallest tile whose
// blocks are all resident at one per CU.  Many rows: the fewest VALU per
// MFMA, which is 128 rows per wave.  Measured, us per kernel (gate/up 2 x
// 6144 x 2048, and down 2048 x 6144 in the parts of gemm16_parts):
//   M      gate/up, 64x128 / 128x128 / 128x256    down, the same / 256x256
//   40     13.5 / 20.4 / 28.0                     10.4 / 12.1 (6 parts)
//   203    26.8 / 20.7 / 32.2                     16.6 (3) / 15.2 (6) / 79 (1)
//   400    38.6 / 40.1 / 33.5                     21.7 (2) / 20.2 (4)
//   1960   152 / 124 / 102                        76 / 62 / 86 / 119 (1 part)
//   2560   -   / -   / 123                        104 (128x128) / 90 / 125
//   6000   -   / -   / 275 (256x256: 294)         174 (128x128) / 160 / 150
// (every shape in one stage less and the dequantization waiting for its
// operands, 128 x 256 and 128 x 128 tiles: 33 / 37 / 36 / 107 / 141 / 310 us
// gate/up and 17 / 19 / 21 / 73 / 105 / 189 us down.)
enum Tile { T64x128, T128x128, T128x256, T256x256 };
Tile tile_for(int64_t M, int64_t N, int64_t K, int epi) {
    const int64_t cols = epi == GEMM_SWIGLU ? 2 * N : N, cus = num_cus();
    auto blocks = [&](int r, int c) { return ((M + r - 1) / r) * ((cols + c - 1) / c); };
    const bool teams = (K / 64) % 16 == 0;             // eight-group blocks in each half of K
    if (teams && (epi == GEMM_SWIGLU ? blocks(64, 128) <= cus : M <= 128)) return T64x128;
    if (blocks(128, 128) <= cus) return T128x128;
    if (epi == GEMM_SWIGLU || blocks(128, 256) <= cus) return T128x256;
    return T256x256;
}

}  // namespace g16

// The most K parts, up to `most` (whole eight-group blocks per part and team),
// whose blocks stay within one per CU.
int gemm16_parts(int64_t M, int64_t N, int64_t K, int most) {
    const g16::Tile t = g16::tile_for(M, N, K, GEMM_RESIDUAL);
    const int64_t r = t == g16::T64x128 ? 64 : t == g16::T256x256 ? 256 : 128;
    const int64_t c = t == g16::T64x128 || t == g16::T128x128 ? 128 : 256;
    const int64_t blocks = ((M + r - 1) / r) * ((N + c - 1) / c), teams = t == g16::T64x128 ? 2 : 1;
    int S = 1;
    for (int s : {2, 3, 4, 6})
        if (s <= most && (K / 512) % (s * teams) == 0 && blocks * s <= (int64_t)num_cus()) S = s;
    return S;
}

int launch_q4_gemm16(const Gemm16Args& a, int epi, hipStream_t st) {
    // 32-bit byte offsets in the kernel; whole blocks of 8 groups (K % 512,
    // the scale/bias DMA) with scale/bias rows 16-byte aligned
    const bool fits32 = (int64_t)a.M * a.K * 2 <= 0xFFFFFFFFLL && (int64_t)a.N * a.K / 2 <= 0xFFFFFFFFLL;
    auto a16 = [](const QMat& q) { return reinterpret_cast<uintptr_t>(q.s) % 16 == 0 && reinterpret_cast<uintptr_t>(q.b) % 16 == 0; };
    if (epi != GEMM_SWIGLU && epi != GEMM_RESIDUAL) return -1;
    if (!fits32 || a.K % 512 != 0 || a.M < 1 || a.N < 1 || !a16(a.A) || (epi == GEMM_SWIGLU && !a16(a.B))) return -1;
    if (a.ysum && (epi != GEMM_SWIGLU || a.yscale != 0.0f || a.N % 128 != 0)) return -1;
    if (a.yscale != 0.0f && (epi != GEMM_SWIGLU || a.N % 8 != 0)) return -1;
    if (epi == GEMM_SWIGLU && (!a.silu_lut || !aligned(a.silu_lut, 16))) return -1;
    // K parts: GEMM_RESIDUAL only, at most 6, whole 8-group scale slots per
    // part, fp32 parts [ksplit][M][N] (16-byte aligned, N % 4 == 0) combined
    // by a second kernel
    const int S = a.ksplit > 1 ? a.ksplit : 1;
    if (S > 1 && (epi != GEMM_RESIDUAL || S > 6 || (a.K / 64) % (8 * S) != 0 || !a.part ||
                  reinterpret_cast<uintptr_t>(a.part) % 16 != 0 || a.N % 4 != 0 || !aligned(a.res, 8) ||
                  !aligned(a.y, 8)))
        return -1;
    const unsigned cols = (unsigned)(epi == GEMM_SWIGLU ? 2 * a.N : a.N);
    auto go = [&](auto kern, int threads, int tbm, int bnw) {
        const unsigned blocks = (cols + bnw - 1) / bnw * (unsigned)((a.M + tbm - 1) / tbm) * S;
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(threads), 0, st, a);
    };
    using namespace g16;
    const Tile t = tile_for(a.M, a.N, a.K, epi);
    if (t == T64x128 && (a.K / 64) % (16 * S) != 0) return -1;
    if (epi == GEMM_SWIGLU) {
        switch (t) {
            case T64x128: go(q4_gemm16_kernel<GEMM_SWIGLU, 1, 2, 2, 4, 2, 1>, 256, 64, 128); break;
            case T128x128: go(q4_gemm16_kernel<GEMM_SWIGLU, 2, 2, 2, 4, 1, 1>, 256, 128, 128); break;
            default: go(q4_gemm16_kernel<GEMM_SWIGLU, 1, 4, 4, 2, 1, 2>, 256, 128, 256); break;
        }
        return 0;
    }
    switch (t) {
        case T64x128: go(q4_gemm16_kernel<GEMM_RESIDUAL, 1, 2, 2, 4, 2, 1>, 256, 64, 128); break;
        case T128x128: go(q4_gemm16_kernel<GEMM_RESIDUAL, 2, 2, 2, 4, 1, 1>, 256, 128, 128); break;
        case T128x256: go(q4_gemm16_kernel<GEMM_RESIDUAL, 1, 4, 4, 2, 1, 2>, 256, 128, 256); break;
        case T256x256: go(q4_gemm16_kernel<GEMM_RESIDUAL, 2, 4, 4, 2, 1, 2>, 512, 256, 256); break;
    }
    if (S > 1) {
        const int64_t MN = (int64_t)a.M * a.N;
        hipLaunchKernelGGL(g16::kpart_residual_kernel, dim3((unsigned)((MN / 4 + 255) / 256)), dim3(256), 0, st,
                           a.part, S, MN, a.res, reinterpret_cast<uint16_t*>(a.y));
    }
    return 0;
}

}  // namespace mq4
