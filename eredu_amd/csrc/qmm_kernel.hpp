// The kernel of the prefill-shaped quantized matmul (M > 16, 16-bit activations,
// transpose = true) on gfx950 matrix cores; qmm.hip plans and launches it, the
// qmm_t*.hip files hold its variants by tile shape.
#pragma once
//
// y = x . W^T with W[n, k] = s[n, k/gs] * q[n, k] + b[n, k/gs]
// (safemlx/src/ops/quantization.rs:190-226, QuantizedLinear's layout).
//
// Work layout.  A workgroup of 8 waves owns a 128 (m) x 256 (n) output tile
// and walks K (or one split of it) in steps of two 64-wide chunks.  The waves
// form two K-groups of 4 that take alternate chunks (even, odd), so that every
// SIMD runs two waves (one's dequantization and memory waits overlap the
// other's MFMAs) while a wave keeps a large output block; at the end the
// second K-group adds its sums into the first through LDS.  Wave w of a
// K-group owns the 64 columns [64w, 64w + 64) and all 128 rows: 4 x 2 tiles of
// v_mfma_f32_32x32x16_bf16 with f32 accumulators.  Outputs with too few such
// tiles to fill the GPU without splitting K into short pieces take 128 x 128,
// 96 x 128 or 64 x 128 tiles instead (wave w: columns [32w, 32w + 32); the
// planner, qmm_plan, chooses).
//
//  * Everything the loop reads goes straight from memory to LDS
//    (buffer_load ... lds): a step's activations (two buffers) and its codes
//    (kept as packed codes; up to four steps ahead).  Codes gathered by the
//    waves themselves -- a lane per row and 16 bytes, so 32 cache lines an
//    instruction -- kept the texture units busy for 80 % of the launch; a load
//    to LDS reads 64 or 128 contiguous bytes of a row with adjacent lanes.
//  * A lane then reads its row's 32 codes of a chunk (row n = l % 32 of a
//    32-column block, k from 32 * (l / 32)) and turns code word t into the B
//    operand of MFMA step t: w = s*q + b is one f32 FMA per code and one
//    v_cvt_pk_bf16_f32 per pair, used by the 4 row blocks of the tile.
//  * A operand of step t for lane (m, kb) = x[m][k0 + 32 kb + 8 t .. + 8],
//    matching the codes the B lane (n, kb) holds for step t.
//  * Schedule: the next k-step's A reads and dequantization are placed between
//    the MFMAs of the current one, a few instructions after each (fixed with
//    scheduling barriers), and the step's loads between those of its last
//    k-step, where a burst of loads would hold the MFMAs up behind the texture
//    queue.  One barrier per step, ahead of its last k-step: by then every
//    wave has read the step's activations and codes, so their buffers can be
//    refilled, and the next step's have landed, so the next operands can be
//    prepared under the last MFMAs.  What bounds it now: the matrix cores are
//    busy for 40 % of the cycles at M = 512 and 55 % at M = 4096 (14336 x 4096);
//    between them the dequantization takes issue slots, and both together hold
//    the clock at 1.66 GHz with many rows.
//  * Measured, M = 512, weights rotated from HBM, against two chunks' codes
//    loaded to registers at the head of each step, the K-groups in opposite
//    phase and (except group 64) a 2-byte load per parameter: 14336 x 4096
//    4-bit group 64 72.2 -> 65.6 us, group 32 94.3 -> 67.3, group 128 87.3 ->
//    62.5, 8-bit group 64 90.3 -> 75.4, group 32 115.3 -> 76.5, group 128
//    103.6 -> 69.7; M = 4096, 4096 x 14336, 4-bit group 64 442 -> 405 us
//    (1190 TFLOP/s).
//  * All global reads are buffer loads: rows past M or N read as zero, so any
//    M and N work (K is a multiple of 64, checked by the dispatcher).
//  * Split K: when the output has too few tiles to fill the GPU, each tile's K
//    is split over several workgroups that write f32 partial tiles to a
//    workspace; a second kernel sums the splits in a fixed order (results do
//    not depend on timing) and rounds once to bf16.
//  * Tiles are assigned so that the workgroups one XCD receives cover few
//    row blocks of x (which then stay in that XCD's L2).
//  * MXFP4 (scale type E8M0T: group 32, E8M0 scale bytes, no biases): the
//    same tiles and pipeline; each lane's 32 codes become B operands through
//    v_cvt_scalef32_pk_bf16_fp4 with the group's scale folded in (exact).
#include <utility>

#include "eq_common.hpp"
#include "qmm_plan.hpp"

namespace eq {

typedef uint32_t q_u32x4 __attribute__((ext_vector_type(4)));

constexpr int kQmmThreads = 512;               // two K-groups of 4 waves

// Steps of codes a kernel variant holds in LDS ahead of their use, which is
// also its main loop's unroll and its parameter windows' length.
constexpr int qmm_ring(int bits, int tn) { return tn == 2 && bits == 8 ? 2 : 4; }

typedef _Float16 q_f16x8 __attribute__((ext_vector_type(8)));

// Activation types of the prefill kernel: the 16-bit type both MFMA operands
// take (the dequantized weights are rounded to it), the MFMA and the output.
template <typename XT>
struct QmmAct;
template <>
struct QmmAct<BF16T> {
    __device__ static __forceinline__ uint32_t pack(float a, float b) { return pack_bf16x2(a, b); }
    __device__ static __forceinline__ f32x16 mfma(q_u32x4 wq, bf16x8 a, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wq), a, c, 0, 0, 0);
    }
    __device__ static __forceinline__ uint16_t out(float v) { return uint16_t(f32_to_bf16_bits(v)); }
};
template <>
struct QmmAct<F16T> {
    // two f32 -> one word of f16 (a low), round to nearest even (v_cvt_pk_f16_f32)
    __device__ static __forceinline__ uint32_t pack(float a, float b) {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
    }
    __device__ static __forceinline__ f32x16 mfma(q_u32x4 wq, bf16x8 a, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(q_f16x8, wq), __builtin_bit_cast(q_f16x8, a),
                                                      c, 0, 0, 0);
    }
    __device__ static __forceinline__ uint16_t out(float v) { return uint16_t(f32_to_f16_bits(v)); }
};

// Every LDS operation of the wave done and at most N memory operations in flight.
template <int N>
__device__ __forceinline__ void wait_lds_and_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

// f(0), f(1), ... f(N - 1), the index a constant of each call: loops whose
// register arrays must not wait for the optimiser's unrolling to be split up.
template <typename F, int... I>
__device__ __forceinline__ void unrolled_calls(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unrolled(F f) {
    unrolled_calls(f, std::make_integer_sequence<int, N>{});
}

template <typename ST>
__device__ __forceinline__ float qmm_param(uint32_t bits);
template <>
__device__ __forceinline__ float qmm_param<BF16T>(uint32_t bits) { return bf16_bits_to_f32(bits & 0xffffu); }
template <>
__device__ __forceinline__ float qmm_param<F16T>(uint32_t bits) { return f16_bits_to_f32(bits & 0xffffu); }

struct QmmArgs {
    uint16_t* y;
    float* ws;  // split K: f32 partial tiles, [split][M][N]; null: y
    const uint16_t* x;
    const uint32_t* w;
    const uint16_t* s;
    const uint16_t* b;  // may be null
    int M, N, K, ldy, mtiles, ntiles, splits, cps;  // cps: chunks per split; ldy: y row stride
    // Grouped (routed experts, no split K): row tile tm is entry groups[tm] =
    // {expert, first row, rows, row offset} of a device-built list; x and y rows
    // [first, first + rows) belong to the expert, whose weights, scales and biases
    // follow the previous expert's.  Entry groups[mtiles] holds how many of the
    // mtiles are in use.  Null: one plain problem.
    const int4* groups;
    // Grouped: y row r multiplies x row lhs[r] (null: row r, or row 0 of a
    // single one) of x_rows; an index outside them reads zeros.
    const int32_t* lhs;
    int x_rows;
};

// PW (parameters as whole words: every row of scales and biases 4-byte
// aligned; otherwise each is a 2-byte load).  Group size 16: the two groups of
// a lane's codes in one load.  Group sizes 32, 64 and 128 (WIN): windows --
// instead of a load per parameter, column and step, which touches one cache
// line per row each, the workgroup stages the scales and biases of a window of
// U steps of both K-groups for all of its columns in LDS: one lane per (array,
// column, 16 bytes), stored word-major so that a lane reads its column's word
// of a step without bank conflicts.
//
// TM x TN: 32-row blocks and 32-column blocks of each wave's output block;
// the workgroup's tile is 32 TM rows x 128 TN columns (4 x 2: 128 x 256, the
// default; 4 x 1 and 2 x 1: 128 x 128 and 64 x 128, for outputs with too few
// large tiles to fill the GPU, which then need no split of K or fewer splits;
// 3 x 1: 96 x 128).  A 2 x 1 workgroup of 4-bit codes leaves room for a second
// one on its CU (64-80 KiB of LDS, 80 registers; with 8-bit codes 96-112 KiB):
// routed experts of 32 rows 252 -> 218 us.
template <int BITS, int GS, typename ST, bool PW, typename XT, int TM, int TN>
__global__ __launch_bounds__(kQmmThreads) __attribute__((amdgpu_waves_per_eu(2, TM == 2 ? 4 : 2))) void qmm_mfma_kernel(
    const QmmArgs args) {
    constexpr int BM = 32 * TM, BN = 128 * TN, LBUF = BM * kBK * 2;  // LBUF: bytes per K-group buffer
    static_assert((TM == 4 && TN == 2) || (TM >= 2 && TM <= 4 && TN == 1), "tile shapes");
    // Steps of codes in LDS, and the unroll of the main loop.
    constexpr int U = qmm_ring(BITS, TN);
    constexpr int CBUF = BN * 16 * BITS;  // bytes of codes of one step (a chunk of each K-group)
    // Activation buffers of two steps and code buffers of U.  Separate arrays,
    // so that the compiler's LDS alias scopes tell the buffers apart and a read
    // of one does not wait for the loads still landing in another.
    __shared__ __attribute__((aligned(16))) char abuf0[2 * LBUF], abuf1[2 * LBUF];
    __shared__ __attribute__((aligned(16))) char cbuf0[CBUF], cbuf1[CBUF], cbuf2[U == 4 ? CBUF : 16],
        cbuf3[U == 4 ? CBUF : 16];
    constexpr bool MX = __is_same(ST, E8M0T);
    constexpr uint32_t PB = MX ? 1u : 2u;  // bytes per scale / bias
    static_assert(!MX || (BITS == 4 && GS == 32 && !PW), "MXFP4: 4-bit codes, group 32");
    static_assert(!MX || std::is_same<XT, BF16T>::value, "MXFP4 prefill takes bf16 activations");
    static_assert(GS == 16 || GS == 32 || GS == 64 || GS == 128, "group sizes");
    constexpr bool WIN = PW && GS != 16;
    constexpr int NPL = GS == 16 && !PW ? 2 : 1;  // loads per parameter, column and step (without windows)
    const int N = args.N, K = args.K, G = K / GS;
    int M = args.M;

    // Tile and split of this workgroup: the workgroups of one XCD (id % 8)
    // take a contiguous run of row-major tiles, i.e. few row blocks of x.  Grouped:
    // an eighth of the tiles in use; with runs over the whole list, which must
    // have room for a part tile per expert, the last XCDs got none (8 experts of
    // 7168 x 4096, 8-bit, 128 routes to two of them 77 -> 29 us, to all 100 -> 75;
    // 128 experts of 768 x 2048, 4-bit, 4096 routes 60 -> 45).
    const int T = args.mtiles * args.ntiles * args.splits;
    int bid = blockIdx.x;
    if (args.groups) {
        const int used = args.groups[args.mtiles].x * args.ntiles, run = (used + 7) >> 3, at = bid >> 3;
        bid = (bid & 7) * run + at;
        if (at >= run || bid >= used) return;  // (the whole workgroup, before any barrier)
    } else if ((T & 7) == 0) {
        bid = (bid & 7) * (T >> 3) + (bid >> 3);
    }
    const int split = bid % args.splits, tile = bid / args.splits;
    const int tm = tile / args.ntiles, tn = tile % args.ntiles;
    int m0 = tm * BM;
    const int n0 = tn * BN;
    const uint16_t* xp = args.x;
    const uint32_t* wp = args.w;
    const char* sp = reinterpret_cast<const char*>(args.s);
    const char* bp = reinterpret_cast<const char*>(args.b);
    uint16_t* yp = args.y;
    int first = 0, x_rows = M;
    if (args.groups) {
        const int4 gd = args.groups[tm];
        first = gd.y, x_rows = args.x_rows;
        yp += int64_t(gd.y) * args.ldy;
        M = gd.z;
        m0 = gd.w;
        wp += int64_t(gd.x) * N * (K * BITS / 32);
        sp += int64_t(gd.x) * N * G * PB;
        if (bp) bp += int64_t(gd.x) * N * G * PB;
    }
    const int nchunks = K / kBK;
    const int c_begin = split * args.cps, c_end = min(nchunks, c_begin + args.cps);
    const int nloc = c_end - c_begin;  // >= 1 (the planner leaves no split empty)

    const int lane = threadIdx.x & 63;
    const int kgrp = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 8);  // K-group: chunks 2i + kgrp
    const int tid = threadIdx.x & 255;                                         // thread within the K-group
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);                 // column quarter
    const int l32 = lane & 31, kb = lane >> 5;
    const int gofs = kgrp * LBUF;  // this K-group's part of each ring buffer
    const int steps = (nloc + 1) / 2;         // chunks of the first K-group
    const int mine = (nloc - kgrp + 1) / 2;   // of this one (the second may have one fewer, or none)

    const __amdgpu_buffer_rsrc_t xr = raw_rsrc(xp, uint32_t(x_rows) * uint32_t(K) * 2u);
    const uint32_t row_bytes = uint32_t(K) * BITS / 8u;  // (the launcher keeps N * row_bytes below 2^31)
    const __amdgpu_buffer_rsrc_t wr = raw_rsrc(wp, uint32_t(N) * row_bytes);
    const uint32_t p_bytes = uint32_t(N) * uint32_t(G) * PB;
    const __amdgpu_buffer_rsrc_t sr = raw_rsrc(sp, p_bytes);
    const __amdgpu_buffer_rsrc_t br = raw_rsrc(bp ? bp : sp, bp ? p_bytes : 0u);
    // Parameter windows in LDS: [buffer][scale, bias][word][column]; a word is
    // two consecutive groups (the first in the low half).
    constexpr int PWW = !WIN ? 1 : GS == 32 ? 2 * U : GS == 64 ? U : U / 2;  // words per column and window
    constexpr int PPR = PWW > 4 ? 2 : 1, PWD = PWW / PPR;                  // pieces per column, words per piece
    constexpr int PIT = (BN * 2 * PPR + kQmmThreads - 1) / kQmmThreads;     // pieces per lane
    static_assert(!WIN || PWW % PPR == 0, "whole pieces");
    __shared__ uint32_t pbuf[WIN ? 2 : 1][2][PWW][WIN ? BN : 1];

    // Lane offsets (chunk 0); rows past M and columns past N read zero.
    // Activations go straight from memory to LDS: load i of wave w fills the
    // 1 KiB (8 rows of 128 B) at (TM w + i) KiB of the BM x 64 tile, lane l
    // the 16 B at 16 l, i.e. row 8 (TM w + i) + l / 8, slot l % 8.  Slot p of
    // row r holds the row's 16-byte chunk p ^ ((r / 2) & 7), so the lane loads
    // chunk (l % 8) ^ ((row / 2) & 7).  (A 16-lane group of an A-operand read
    // takes rows r .. r + 15 at one chunk; 64 banks of 4 bytes span two rows,
    // so the rows of one parity must land in 8 different 16-byte bank groups.)
    uint32_t a_goff[4];  // (the first TM used; a bound of TM fails clang's host pass when a lambda captures it)
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int row = 8 * (TM * wave + i) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        int src = m0 + row;
        bool live = src < M;
        if (args.groups) {
            // (the routes' rows are read where they are: no gathered copy)
            if (live) src = args.lhs ? args.lhs[first + src] : x_rows == 1 ? 0 : first + src;
            live = live && src >= 0 && src < x_rows;
        }
        a_goff[i] = live ? (uint32_t(src) * uint32_t(K) + uint32_t(8 * c)) * 2u : kOutOfRange;
    }
    // Codes, too, go straight to LDS: per step a row's 128 codes (its chunks of
    // both K-groups, 16 BITS bytes), load q of wave v = 4 kgrp + wave filling the
    // KiB v CL + q, lane l slot l % P of row l / P there.  Slot p of row r holds
    // the row's 16-byte piece p ^ (r / (16 / P) % P), so that the 16 rows of a
    // 16-lane read land in different bank groups.
    constexpr int CL = TN * BITS / 4, P = BITS, PLOG = BITS == 4 ? 2 : 3;  // loads per wave and step; pieces per row
    static_assert(BITS == 4 || BITS == 8, "code widths");
    uint32_t c_goff[4];  // (the first CL used)
#pragma unroll
    for (int q = 0; q < CL; q++) {
        const int row = (64 / P) * ((4 * kgrp + wave) * CL + q) + (lane >> PLOG);
        const int piece = (lane & (P - 1)) ^ ((row >> (4 - PLOG)) & (P - 1));
        c_goff[q] = n0 + row < N ? uint32_t(n0 + row) * row_bytes + uint32_t(16 * piece) : kOutOfRange;
    }
    // Per-step parameter loads (without windows): columns n0 + 32 TN wave + 32 j + l32.
    uint32_t soff[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const uint32_t n = uint32_t(n0 + 32 * TN * wave + 32 * j + l32);
        soff[j] = int(n) < N ? (n * uint32_t(G)) * PB + uint32_t((32 * kb) / GS) * PB : kOutOfRange;
    }
    // (a lane's 32 codes lie in one group when the group size is a multiple of
    // 32 -- chunks start at multiples of 64, so its group is k0 / GS + 32 kb /
    // GS -- and in groups 2 kb, 2 kb + 1 of the chunk at group size 16)

    // Loads of this K-group's chunk i, i.e. chunk 2i + kgrp of the split (past
    // the split's end: the last chunk again, in cache and never used).
    auto chunk_k0 = [&](int i) __attribute__((always_inline)) {
        return (c_begin + min(2 * i + kgrp, nloc - 1)) * kBK;
    };
    // (LDS pointers, so that no access goes through a generic address)
    typedef __attribute__((address_space(3))) char lds_char;
    typedef __attribute__((address_space(3))) const bf16x8 lds_bf16x8;
    typedef __attribute__((address_space(3))) const q_u32x4 lds_u32x4;
    auto abuf = [&](int k) __attribute__((always_inline)) { return k == 0 ? (lds_char*)abuf0 : (lds_char*)abuf1; };
    auto cbuf = [&](int k) __attribute__((always_inline)) {
        return k == 0 ? (lds_char*)cbuf0 : k == 1 ? (lds_char*)cbuf1 : k == 2 ? (lds_char*)cbuf2 : (lds_char*)cbuf3;
    };
    auto load_a = [&](lds_char* buf, uint32_t ks, int q) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            xr, (__attribute__((address_space(3))) void*)(buf + gofs + (TM * wave + q) * 1024), 16, a_goff[q], ks, 0, 0);
    };
    auto a_koff = [&](int i) __attribute__((always_inline)) {
        return __builtin_amdgcn_readfirstlane(uint32_t(chunk_k0(i)) * 2u);
    };
    auto load_c = [&](lds_char* buf, uint32_t ks, int q) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            wr, (__attribute__((address_space(3))) void*)(buf + ((4 * kgrp + wave) * CL + q) * 1024), 16, c_goff[q], ks, 0,
            0);
    };
    auto c_koff = [&](int i) __attribute__((always_inline)) {
        return __builtin_amdgcn_readfirstlane(uint32_t((c_begin + 2 * min(i, steps - 1)) * kBK) * BITS / 8u);
    };
    // One step's parameters of this lane, without windows.
    struct PSlot {
        uint32_t s[TN][NPL], b[TN][NPL];
    };
    // Past the last step the buffers are empty, so that nothing is fetched: a
    // parameter load touches a cache line per row, and in a split of 4 steps the
    // 4 requested ahead would double them (group 16, 1024 x 4096, 4-bit, 8
    // splits: M = 64 13.6 us with those, 13.0 without).
    auto load_p = [&](PSlot& S, int i) __attribute__((always_inline)) {
        const uint32_t kp = __builtin_amdgcn_readfirstlane(uint32_t(chunk_k0(i) / GS) * PB);
        const __amdgpu_buffer_rsrc_t sr = raw_rsrc(sp, i < steps ? p_bytes : 0u);
        const __amdgpu_buffer_rsrc_t br = raw_rsrc(bp ? bp : sp, bp && i < steps ? p_bytes : 0u);
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if constexpr (MX) {
                S.s[j][0] = __builtin_amdgcn_raw_buffer_load_b8(sr, soff[j], kp, 0);
                S.b[j][0] = 0u;
            } else if constexpr (GS == 16 && PW) {
                // the lane's 32 codes span two groups: both parameters in one word
                S.s[j][0] = __builtin_amdgcn_raw_buffer_load_b32(sr, soff[j], kp, 0);
                S.b[j][0] = __builtin_amdgcn_raw_buffer_load_b32(br, soff[j], kp, 0);
            } else {
#pragma unroll
                for (int q = 0; q < NPL; q++) {
                    S.s[j][q] = __builtin_amdgcn_raw_buffer_load_b16(sr, soff[j] + 2 * q, kp, 0);
                    S.b[j][q] = __builtin_amdgcn_raw_buffer_load_b16(br, soff[j] + 2 * q, kp, 0);
                }
            }
        }
    };
    // Parameter window w (steps U w .. U w + U - 1): piece p of the workgroup
    // (thread + it * threads) is (column p % BN, array p / BN % 2, part p / 2 BN).
    typedef uint32_t q_u32x2 __attribute__((ext_vector_type(2)));
    uint32_t pst[PIT][4], poff[PIT];
    int parr[PIT], ppart[PIT], pcol[PIT];
#pragma unroll
    for (int it = 0; it < PIT; it++) {
        const int p = it * kQmmThreads + int(threadIdx.x);
        pcol[it] = p % BN;
        parr[it] = __builtin_amdgcn_readfirstlane(p / BN) % 2;  // (BN is a multiple of 64: wave-uniform)
        ppart[it] = __builtin_amdgcn_readfirstlane(p / (2 * BN));
        poff[it] = n0 + pcol[it] < N && ppart[it] < PPR
                       ? uint32_t(n0 + pcol[it]) * uint32_t(G) * PB + uint32_t(c_begin * kBK / GS) * 2u +
                             uint32_t(ppart[it]) * uint32_t(PWD * 4)
                       : kOutOfRange;
    }
    auto load_pw = [&](int w) __attribute__((always_inline)) {
        const uint32_t kq = __builtin_amdgcn_readfirstlane(uint32_t(w) * uint32_t(PWW * 4));
#pragma unroll
        for (int it = 0; it < PIT; it++) {
            const __amdgpu_buffer_rsrc_t r = parr[it] ? br : sr;
            if constexpr (PWD == 4) {
                const q_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, poff[it], kq, 0);
                for (int e = 0; e < 4; e++) pst[it][e] = v[e];
            } else if constexpr (PWD == 2) {
                const q_u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, poff[it], kq, 0);
                for (int e = 0; e < 2; e++) pst[it][e] = v[e];
            } else {
                pst[it][0] = __builtin_amdgcn_raw_buffer_load_b32(r, poff[it], kq, 0);
            }
        }
    };
    auto store_pw = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < PIT; it++)
            if (ppart[it] < PPR) {
#pragma unroll
                for (int e = 0; e < PWD; e++) pbuf[buf][parr[it]][ppart[it] * PWD + e][pcol[it]] = pst[it][e];
            }
    };
    auto barrier = [&]() __attribute__((always_inline)) { asm volatile("s_barrier" ::: "memory"); };

    // A operand of this lane for k-step t and row block mi: row 32 mi + l32,
    // chunk 4 kb + t in slot (4 kb + t) ^ ((row / 2) & 7) (the same for every mi).
    uint32_t aoff[4];
#pragma unroll
    for (int t = 0; t < 4; t++) aoff[t] = uint32_t(l32 * (kBK * 2) + (((4 * kb + t) ^ ((l32 >> 1) & 7)) << 4));
    auto read_a = [&](lds_char* buf, int t, int mi) __attribute__((always_inline)) -> bf16x8 {
        return *(lds_bf16x8*)(buf + gofs + aoff[t] + mi * 32 * (kBK * 2));
    };

    // This lane's codes of a chunk: row 32 TN wave + 32 j + l32, pieces from
    // (P / 2) kgrp + (P / 4) kb, in the order of the k-steps.
    constexpr int NW = BITS / 4;  // 16-byte pieces per lane and column block
    uint32_t coff[NW];
#pragma unroll
    for (int q = 0; q < NW; q++) {
        const int row = 32 * TN * wave + l32;
        coff[q] = uint32_t(row * (16 * P) + (((P / 2 * kgrp + P / 4 * kb + q) ^ ((row >> (4 - PLOG)) & (P - 1))) << 4));
    }
    q_u32x4 cw[TN][NW];
    auto read_c = [&](lds_char* buf, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < NW; q++) cw[j][q] = *(lds_u32x4*)(buf + coff[q] + j * 32 * (16 * P));
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x16{};

    // Scale and bias of a chunk, per column block (group 16: of the lane's
    // codes 0..15 and 16..31).
    constexpr int NG = GS == 16 ? 2 : 1;
    auto param_words = [&](const PSlot& S, int r, int buf, uint32_t (&sw)[TN], uint32_t (&bw)[TN])
                           __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if constexpr (WIN) {
                const int col = 32 * TN * wave + 32 * j + l32;
                // group 32: the chunk's two groups are one word; 64: the groups
                // of the step's two chunks; 128: those of two steps
                const int w = GS == 32 ? 2 * r + kgrp : GS == 64 ? r : r / 2;
                sw[j] = pbuf[buf][0][w][col], bw[j] = pbuf[buf][1][w][col];
            } else {
                sw[j] = S.s[j][0], bw[j] = S.b[j][0];
                if constexpr (NPL == 2) sw[j] |= S.s[j][1] << 16, bw[j] |= S.b[j][1] << 16;
            }
        }
    };
    auto params = [&](int r, const uint32_t (&sw)[TN], const uint32_t (&bw)[TN], float (&s)[TN][NG],
                      float (&b)[TN][NG]) __attribute__((always_inline)) {
        const int sh = !WIN ? 0 : GS == 32 ? 16 * kb : GS == 64 ? 16 * kgrp : 16 * (r & 1);
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if constexpr (MX) {
                s[j][0] = e8m0_to_f32(sw[j]);
                b[j][0] = 0.f;
            } else {
                s[j][0] = qmm_param<ST>(sw[j] >> sh), b[j][0] = qmm_param<ST>(bw[j] >> sh);
                if constexpr (NG == 2) s[j][1] = qmm_param<ST>(sw[j] >> 16), b[j][1] = qmm_param<ST>(bw[j] >> 16);
            }
        }
    };
    // Codes -> B operand words: word k (pair 2k, 2k + 1) of column block j at
    // k-step t.  4-bit codes are split once per (j, t) into even and odd codes.
    uint32_t lo[TN], hi[TN];
    float odd0[TN], odd1[TN];  // the second pair of a conversion
    auto split_codes = [&](int j, int t) __attribute__((always_inline)) {
        if constexpr (BITS == 4 && !MX) {
            const uint32_t w = cw[j][0][t];
            lo[j] = w & 0x0f0f0f0fu, hi[j] = (w >> 4) & 0x0f0f0f0fu;
            // (opaque to the optimiser, so that each code converts with one
            // instruction instead of a bit-field extract plus a convert)
            asm volatile("" : "+v"(lo[j]), "+v"(hi[j]));
        }
    };
    auto dequant_pair = [&](const float (&s)[TN][NG], const float (&b)[TN][NG], int j, int t, int k)
                            __attribute__((always_inline)) -> uint32_t {
        if constexpr (MX) {
            const uint32_t w = cw[j][0][t];
            if (k == 0) return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s[j][0], 0));
            if (k == 1) return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s[j][0], 1));
            if (k == 2) return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s[j][0], 2));
            return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, s[j][0], 3));
        } else {
            const int g = t < 2 ? 0 : NG - 1;
            float c0, c1;
            if constexpr (BITS == 4) {
                // A byte 0..15 read as E4M3 is code * 2^-9 (subnormals below 8, the first
                // normal binade from 8 on), so one conversion gives the f32 values of two
                // codes, exactly: half the conversions of v_cvt_f32_ubyte (4 % of the launch).
                // Words 2a and 2a + 1 come from the halves a of the two code words.
                if (k % 2 == 0) {
                    const auto l = k == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo[j], 512.f, 0)
                                          : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(lo[j], 512.f, 1);
                    const auto h = k == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi[j], 512.f, 0)
                                          : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(hi[j], 512.f, 1);
                    c0 = l[0], c1 = h[0];
                    odd0[j] = l[1], odd1[j] = h[1];
                } else {
                    c0 = odd0[j], c1 = odd1[j];
                }
            } else {
                const uint32_t w = cw[j][t / 2][2 * (t % 2) + k / 2];
                c0 = float((w >> (16 * (k % 2))) & 0xffu), c1 = float((w >> (16 * (k % 2) + 8)) & 0xffu);
            }
            return QmmAct<XT>::pack(fmaf(s[j][g], c0, b[j][g]), fmaf(s[j][g], c1, b[j][g]));
        }
    };

    PSlot pring[WIN ? 1 : U];
    uint32_t sw[TN], bw[TN];                    // the next chunk's parameter words
    float ps[TN][NG], pb[TN][NG];               // parameters of the chunk being dequantized
    q_u32x4 bq[2][TN];                          // B operands of the current and the next k-step
    bf16x8 aop[2][TM];                          // A operands, likewise
    auto dequant_step = [&](auto tc, auto pc) __attribute__((always_inline)) {  // pair p % 4 of column block p / 4
        constexpr int t = decltype(tc)::value, p = decltype(pc)::value;
        if constexpr (p % 4 == 0) split_codes(p / 4, t);
        bq[t & 1][p / 4][p % 4] = dequant_pair(ps, pb, p / 4, t, p % 4);
    };

    // Prologue: the first parameter window, the codes of steps 0 .. U - 1 and
    // the activations of steps 0 and 1 requested; the window stored to LDS,
    // step 0's loads awaited, its first operands prepared.
    if constexpr (WIN) load_pw(0);
    else
#pragma unroll
        for (int c = 0; c < U; c++) load_p(pring[c], c);
    __builtin_amdgcn_sched_barrier(0);  // (the waits below count on this order)
#pragma unroll
    for (int q = 0; q < CL; q++) load_c(cbuf(0), c_koff(0), q);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
        for (int q = 0; q < TM; q++) load_a(abuf(c), a_koff(c), q);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int c = 1; c < U; c++)
#pragma unroll
        for (int q = 0; q < CL; q++) load_c(cbuf(c), c_koff(c), q);
    if constexpr (WIN) store_pw(0);
    __builtin_amdgcn_sched_barrier(0);
    wait_lds_and_vmcnt<TM + (U - 1) * CL>();
    barrier();

    if (mine > 0) {
#pragma unroll
        for (int j = 0; j < TN; j++) read_c(cbuf(0), j);
        param_words(pring[0], 0, 0, sw, bw);
        params(0, sw, bw, ps, pb);
        unrolled<4 * TN>([&](auto pc) __attribute__((always_inline)) { dequant_step(std::integral_constant<int, 0>{}, pc); });
#pragma unroll
        for (int mi = 0; mi < TM; mi++) aop[0][mi] = read_a(abuf(0), 0, mi);
        bool more = true;
        for (int i0 = 0; more; i0 += U) {
            const int pw_cur = (i0 / U) & 1;  // this iteration's parameter window buffer
            unrolled<U>([&](auto rc) __attribute__((always_inline)) {
                constexpr int r = decltype(rc)::value;
                if (!more) return;
                const int i = i0 + r;
                const uint32_t ka = a_koff(i + 2), kc = c_koff(i + U);
                unrolled<4>([&](auto tc) __attribute__((always_inline)) {
                    constexpr int t = decltype(tc)::value;
                    if constexpr (t == 3) {
                        // Every wave has read this step's activations and codes: their buffers
                        // are free; the next step's have landed.
                        // (memory operations complete in order, and the newest CL are the
                        // codes requested in the last step, which U = 4 leaves in flight)
                        if constexpr (WIN && r == U - 1) store_pw(pw_cur ^ 1);
                        __builtin_amdgcn_sched_barrier(0);
                        wait_lds_and_vmcnt<U == 4 ? CL : 0>();
                        barrier();
                    }
                    // k-step t's MFMAs; between them the next k-step's A reads and dequantization
                    // and, in the last k-step, the loads of the steps ahead
                    constexpr int MF = TM * TN, NP = 4 * TN, LD = TM + CL;
                    unrolled<MF>([&](auto kc_) __attribute__((always_inline)) {
                        constexpr int k = decltype(kc_)::value, mi = k / TN, j = k % TN;
                        acc[mi][j] = QmmAct<XT>::mfma(bq[t & 1][j], aop[t & 1][mi], acc[mi][j]);
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr (t == 3 && k == 0) {
#pragma unroll
                            for (int jj = 0; jj < TN; jj++) read_c(cbuf((r + 1) % U), jj);
                            param_words(pring[WIN ? 0 : (r + 1) % U], (r + 1) % U, r + 1 < U ? pw_cur : pw_cur ^ 1, sw, bw);
                        }
                        if constexpr (k < TM) aop[(t + 1) & 1][k] = read_a(abuf(t < 3 ? r & 1 : (r + 1) & 1), (t + 1) & 3, k);
                        // (the last k-step's dequantization waits for the codes just read)
                        constexpr int K0 = t == 3 ? (MF >= 4 ? MF / 4 : MF - 1) : 0;
                        if constexpr (t == 3 && k == K0) params((r + 1) % U, sw, bw, ps, pb);
                        if constexpr (k >= K0) {
                            constexpr int p0 = (k - K0) * NP / (MF - K0), p1 = (k - K0 + 1) * NP / (MF - K0);
                            unrolled<p1 - p0>([&](auto pc) __attribute__((always_inline)) {
                                dequant_step(std::integral_constant<int, (t + 1) & 3>{},
                                             std::integral_constant<int, p0 + decltype(pc)::value>{});
                            });
                        }
                        if constexpr (t == 3) {
                            if constexpr (k == 0) {
                                if constexpr (!WIN) load_p(pring[r], i + U);
                                else if constexpr (r == 0) load_pw(i0 / U + 1);
                                __builtin_amdgcn_sched_barrier(0);
                            }
                            constexpr int q0 = k * LD / MF, q1 = (k + 1) * LD / MF;
                            unrolled<q1 - q0>([&](auto qc) __attribute__((always_inline)) {
                                constexpr int q = q0 + decltype(qc)::value;
                                if constexpr (q < TM) load_a(abuf(r & 1), ka, q);
                                else load_c(cbuf(r), kc, q - TM);
                                if constexpr (q == TM - 1) __builtin_amdgcn_sched_barrier(0);
                            });
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    });
                });
                more = i + 1 < mine;
            });
        }
    }
    for (int i = mine; i < steps; i++) barrier();  // (the other K-group's last step)
    // Every load has landed (the ring buffers are reused below).
    __builtin_amdgcn_s_waitcnt(0);
    // The second K-group's sums go to LDS, one row block (16 TN KiB, at most
    // a buffer's 2 LBUF bytes) at a time through alternating buffers, and the
    // first adds them.  Layout: [wave][j][q][lane] x 16 B, q = the run of 4
    // accumulator registers.
    static_assert(4 * TN * 4 * 64 * 16 <= 2 * LBUF, "a row block's sums fit one buffer");
    __syncthreads();
#pragma unroll
    for (int mi = 0; mi < TM; mi++) {
        f32x4* red = reinterpret_cast<f32x4*>(mi & 1 ? abuf1 : abuf0);
        if (kgrp == 1) {
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    red[((wave * TN + j) * 4 + q) * 64 + lane] =
                        f32x4{acc[mi][j][4 * q], acc[mi][j][4 * q + 1], acc[mi][j][4 * q + 2], acc[mi][j][4 * q + 3]};
        }
        __syncthreads();
        if (kgrp == 0) {
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const f32x4 v = red[((wave * TN + j) * 4 + q) * 64 + lane];
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[mi][j][4 * q + e] += v[e];
                }
        }
    }
    if (kgrp == 1) return;

    // The MFMA computed y^T blocks (weights as the first operand): register r
    // of lane l holds row m = 32 mi + l % 32 and column n = 32 j + 8 (r / 4) +
    // 4 (l / 32) + r % 4, so each run of 4 registers is 4 adjacent columns of
    // one row.  Columns past N are whole waves (N % 128 == 0).
    if (n0 + 32 * TN * wave >= N) return;
#pragma unroll
    for (int mi = 0; mi < TM; mi++) {
        const int m = m0 + 32 * mi + l32;
        if (m < M) {
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int n = n0 + 32 * TN * wave + 32 * j + 8 * q + 4 * kb;
                    const f32x4 v = {acc[mi][j][4 * q], acc[mi][j][4 * q + 1], acc[mi][j][4 * q + 2], acc[mi][j][4 * q + 3]};
                    if (args.ws) {
                        *reinterpret_cast<f32x4*>(args.ws + (int64_t(split) * M + m) * N + n) = v;
                    } else {
                        const uint32_t lo = QmmAct<XT>::pack(v[0], v[1]), hi = QmmAct<XT>::pack(v[2], v[3]);
                        *reinterpret_cast<uint2*>(yp + int64_t(m) * args.ldy + n) = make_uint2(lo, hi);
                    }
                }
        }
    }
}

// Scale, activation, group-size and parameter-load (pw) dispatch of one tile
// shape; MXFP4 reads its scales a byte at a time.
template <int TM, int TN>
static bool qmm_run_tile(int bits, int gs, int scale_dtype, int x_dtype, bool pw, const QmmArgs& a, int workgroups,
                         hipStream_t st) {
    const dim3 grid{unsigned(workgroups)}, block{unsigned(kQmmThreads)};
    auto by_gs = [&](auto bc, auto stt, auto xt) -> bool {
        constexpr int B = decltype(bc)::value;
        typedef decltype(stt) ST;
        typedef decltype(xt) XT;
        if (gs == 16 && pw) qmm_mfma_kernel<B, 16, ST, true, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else if (gs == 16) qmm_mfma_kernel<B, 16, ST, false, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else if (gs == 32 && pw) qmm_mfma_kernel<B, 32, ST, true, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else if (gs == 32) qmm_mfma_kernel<B, 32, ST, false, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else if (gs == 64 && pw) qmm_mfma_kernel<B, 64, ST, true, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else if (gs == 64) qmm_mfma_kernel<B, 64, ST, false, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else if (gs == 128 && pw) qmm_mfma_kernel<B, 128, ST, true, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else if (gs == 128) qmm_mfma_kernel<B, 128, ST, false, XT, TM, TN><<<grid, block, 0, st>>>(a);
        else return false;
        return true;
    };
    auto by_x = [&](auto bc, auto stt) -> bool {
        if (x_dtype == EQ_DTYPE_BF16) return by_gs(bc, stt, BF16T{});
        if (x_dtype == EQ_DTYPE_F16) return by_gs(bc, stt, F16T{});
        return false;
    };
    auto by_scale = [&](auto bc) -> bool {
        if (scale_dtype == EQ_DTYPE_BF16) return by_x(bc, BF16T{});
        if (scale_dtype == EQ_DTYPE_F16) return by_x(bc, F16T{});
        return false;
    };
    if (scale_dtype == EQ_DTYPE_U8) {
        if (bits != 4 || gs != 32 || x_dtype != EQ_DTYPE_BF16) return false;
        qmm_mfma_kernel<4, 32, E8M0T, false, BF16T, TM, TN><<<grid, block, 0, st>>>(a);
        return true;
    }
    if (bits == 4) return by_scale(std::integral_constant<int, 4>{});
    if (bits == 8) return by_scale(std::integral_constant<int, 8>{});
    return false;
}

// The tile shapes (rows x columns): 128 x 256, 128 x 128, 96 x 128, 64 x 128.
// False: no variant for these types.
bool qmm_run_t42(int bits, int gs, int scale_dtype, int x_dtype, bool pw, const QmmArgs& a, int workgroups, hipStream_t st);
bool qmm_run_t41(int bits, int gs, int scale_dtype, int x_dtype, bool pw, const QmmArgs& a, int workgroups, hipStream_t st);
bool qmm_run_t31(int bits, int gs, int scale_dtype, int x_dtype, bool pw, const QmmArgs& a, int workgroups, hipStream_t st);
bool qmm_run_t21(int bits, int gs, int scale_dtype, int x_dtype, bool pw, const QmmArgs& a, int workgroups, hipStream_t st);

}  // namespace eq
