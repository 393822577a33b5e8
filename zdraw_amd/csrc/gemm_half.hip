// gfx950 GEMM for the projections either side of attention:
//   C[m][n] = A[m][k] x W[n][k]^T, 16-bit MFMA, fp32 accumulation.
//
// What it replaces in the reference: the half-mode simdgroup GEMMs behind
// zdraw_metal_run_gemm_enc / _off_enc / _ours16_enc / _f16a_enc
// (metal/mgemm_shader.zig, metal_api.m) that produce Q, K, V from the block
// input and drain the attention output (klein/zflux2_resident.zig:1473-1513,
// 1986-1998). Both operands are K-major (activation rows and weight rows are
// contiguous in k), which is exactly the register layout of the 16-bit MFMAs
// (v_mfma_f32_16x16x32): a lane supplies 8 consecutive k of one row.
//
// Two kernels share the tile walk, the operand layout and the schedule (four waves, one per SIMD,
// slabs of 64 k fetched from global memory straight into swizzled, unpadded LDS rows):
//   * gemm_ring_kernel: 256 x 256 tiles, each wave 128 x 128 of C; an eight-wave build of that tile
//     is kept behind a knob;
//   * gemm_pipe_kernel: nine tiles from 64 x 64 to 256 x 160 with three or four slabs in LDS, for
//     problems that do not fill the chip with 256-tiles, and for any k that is not a multiple of 64;
//   * f32 activations are rounded to the weight's type by a launch of their own;
//   * gemm_unstaged_kernel: what neither can take (no rounded copy under capture, rows of 4 GiB);
//   * two or three products of one A with equal shapes (q/k/v, gate/up) run as one launch
//     whose tiles cover all of them;
//   * fixed summation order and no atomics (a thinly filled last round is cut along k and
//     merged in part order): bit-identical run to run.
#include "attn_device.hpp"
#include "gemm_kernel.h"

#include <cmath>

namespace zdraw {

namespace gemm {

constexpr int BM = 256, BN = 256, BK = 64;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// v_mfma_f32_16x16x32: a lane supplies 8 consecutive k (chunk lane / 16 of the 32) of row lane % 16
// and receives, of the 16 x 16 result, row lane % 16 of the second operand against rows
// 4 (lane / 16) .. + 3 of the first. Per FLOP it moves half the accumulator bytes of the 32 x 32
// form through the register file, and at the board's power limit that is worth clock.
// Written as assembly with the accumulator tied to the result: given the builtin, the compiler
// picks the three-address form for these 64 four-register accumulators and then moves them
// around the accumulation file inside the loop (several copies per MFMA). The compiler inserts
// no hazard waits around assembly: the caller keeps dependent MFMAs apart (here at least four MFMAs) and
// calls mfma16_drain() in the same basic block as the last MFMA, before control can reach code
// the compiler may have placed on its own (copies or spills of the accumulators at a join): a
// result read within the MFMA's four passes is the old value.
template <bool F16>
__device__ __forceinline__ void mfma16(const u32x4& a, const u32x4& b, f32x4& c) {
    if constexpr (F16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma16_drain() {
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
}

// A wave's (16 TI) x (16 TJ) block of C from 16 x 16 x 32 MFMAs. They take the W fragment as
// their first operand, so a lane (c = lane % 16, q = lane / 16) holds row row0 + 16 i + c of C
// and, in tile (i, j), columns col0 + 16 j + 4 q .. + 3: a store instruction covers 16 rows x 64
// contiguous bytes of f32.
template <bool F16, typename TC, int TI, int TJ>
__device__ __forceinline__ void store_tile16(const GemmArgs& g, void* c, const f32x4 (&acc)[TI][TJ], int row0, int col0, int lane) {
    const int c16 = lane & 15, q = lane >> 4;
    const bool vec = (g.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(c) % (4 * sizeof(TC))) == 0);
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const int row = row0 + 16 * i + c16;
        if (row >= g.m) continue;
        TC* const crow = reinterpret_cast<TC*>(c) + (int64_t)row * g.ldc;
#pragma unroll
        for (int j = 0; j < TJ; j++) {
            const int col = col0 + 16 * j + 4 * q;
            const f32x4 v = acc[i][j];
            if (vec && col + 4 <= g.n) {
                if constexpr (std::is_same<TC, float>::value) *reinterpret_cast<f32x4*>(crow + col) = v;
                else if constexpr (F16) *reinterpret_cast<u32x2*>(crow + col) = __builtin_bit_cast(u32x2, __builtin_convertvector(v, f16x4));
                else *reinterpret_cast<u32x2*>(crow + col) = __builtin_bit_cast(u32x2, __builtin_convertvector(v, bf16x4));
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    if (col + e >= g.n) break;
                    if constexpr (std::is_same<TC, float>::value) crow[col + e] = v[e];
                    else if constexpr (F16) { const _Float16 x = (_Float16)v[e]; crow[col + e] = __builtin_bit_cast(unsigned short, x); }
                    else { const bf16_t x = (bf16_t)v[e]; crow[col + e] = __builtin_bit_cast(unsigned short, x); }
                }
            }
        }
    }
}

// A 128-column block of a 16-bit C, as whole rows of the block (256 bytes): the wave turns 32 rows
// at a time (two rows of tiles) through 8 KB of LDS of its own at lds_wave, so it needs no barrier
// of its own; the caller sees to it that nobody else uses that LDS any more. Staged rows are
// unpadded; the 16-byte chunk c of row r sits at c ^ (r & 15), which spreads both the 8-byte writes (16 rows x 2 halves per half wave) and the row-wise reads over
// all banks. A wave's LDS operations complete in order, so the reads of one pass see its
// writes and the next pass's writes follow its reads. Rows of C that do not start on 16 bytes,
// and the columns past n, are stored element by element.
template <bool F16, typename TC, int TI>
__device__ __forceinline__ void store_tile_lds16(const GemmArgs& g, void* c, const f32x4 (&acc)[TI][8], unsigned lds_wave, int row0, int col0, int lane) {
    static_assert(sizeof(TC) == 2, "16-bit C only");
    static_assert(TI % 2 == 0, "rows in pairs of tiles");
    constexpr int TJ = 8;
    constexpr int ROWB = 32 * TJ;   // bytes per staged row
    constexpr int NCH = 2 * TJ;     // 16-byte chunks per row
    constexpr int RPI = 64 / NCH;   // rows per read-back instruction
    typedef __attribute__((address_space(3))) u32x2* lds_u32x2_t;
    typedef const __attribute__((address_space(3))) u32x4* lds_u32x4_t;
    auto swz = [](int r) { return r & 15; };
    const int c16 = lane & 15, q = lane >> 4;
    // write: row 16 (i & 1) + c16, bytes 32 j + 8 q .. + 8 = chunk 2 j + q / 2, half q & 1
    const unsigned wbase = lds_wave + (unsigned)(c16 * ROWB + (q & 1) * 8);
    const unsigned wsw = (unsigned)(swz(c16) ^ (q >> 1)); // (2 j + q / 2) ^ s = (2 j) ^ (s ^ (q / 2))
    // read: row RPI p + lane / NCH (p < 32 / RPI), chunk lane % NCH
    const int rr = lane / NCH, ch = lane % NCH;
    const int col = col0 + 8 * ch;
    // (uniform over the launch: rows of C start on 16 bytes; otherwise element by element)
    const bool whole = col + 8 <= g.n && (g.ldc % 8 == 0) && (reinterpret_cast<uintptr_t>(c) % 16 == 0);
    unsigned short* const cbase = reinterpret_cast<unsigned short*>(c) + (int64_t)(row0 + rr) * g.ldc + col;
#pragma unroll
    for (int ip = 0; ip < TI / 2; ip++) {
#pragma unroll
        for (int ii = 0; ii < 2; ii++)
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                const f32x4 v = acc[2 * ip + ii][j];
                u32x2 pk;
                if constexpr (F16) pk = __builtin_bit_cast(u32x2, __builtin_convertvector(v, f16x4));
                else pk = __builtin_bit_cast(u32x2, __builtin_convertvector(v, bf16x4));
                // (rows 16 .. 31 swizzle as rows 0 .. 15 do)
                *(lds_u32x2_t)(wbase + (unsigned)(ii * 16 * ROWB) + (((unsigned)(2 * j) ^ wsw) * 16u)) = pk;
            }
        __builtin_amdgcn_sched_barrier(0); // (keeps the scheduler from reading every accumulator out at once)
        u32x4 v[32 / RPI];
#pragma unroll
        for (int p2 = 0; p2 < 32 / RPI; p2++) {
            const int r = RPI * p2 + rr;
            v[p2] = *(lds_u32x4_t)(lds_wave + (unsigned)(r * ROWB) + (unsigned)((ch ^ swz(r)) * 16));
        }
#pragma unroll
        for (int p2 = 0; p2 < 32 / RPI; p2++) {
            const int row = row0 + 32 * ip + RPI * p2 + rr;
            if (row >= g.m) continue;
            unsigned short* const dst = cbase + (int64_t)(32 * ip + RPI * p2) * g.ldc;
            if (whole) {
                *reinterpret_cast<u32x4*>(dst) = v[p2];
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (col + e < g.n) dst[e] = (unsigned short)(v[p2][e >> 1] >> (16 * (e & 1)));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// A 128-column block of f32 C in the same way: 16 rows (8 KB) at a time, the 16-byte chunk c of
// row r at c ^ (r & 7) (eight rows written at once hit eight different chunks; the swizzle stays
// inside 128 bytes, so an instruction still stores two whole 512-byte rows).
template <int TI>
__device__ __forceinline__ void store_tile_lds32(const GemmArgs& g, void* c, const f32x4 (&acc)[TI][8], unsigned lds_wave, int row0, int col0, int lane) {
    typedef __attribute__((address_space(3))) f32x4* lds_f32x4_t;
    const int c16 = lane & 15, q = lane >> 4;
    const bool vec = (g.ldc % 4 == 0) && (reinterpret_cast<uintptr_t>(c) % 16 == 0);
#pragma unroll
    for (int i = 0; i < TI; i++) {
#pragma unroll
        for (int j = 0; j < 8; j++)
            *(lds_f32x4_t)(lds_wave + (unsigned)(c16 * 512) + (unsigned)(((4 * j + q) ^ (c16 & 7)) * 16)) = acc[i][j];
        __builtin_amdgcn_sched_barrier(0);
        f32x4 v[8];
#pragma unroll
        for (int p = 0; p < 8; p++) v[p] = *(lds_f32x4_t)(lds_wave + (unsigned)(p * 1024 + lane * 16));
#pragma unroll
        for (int p = 0; p < 8; p++) {
            const int r = 2 * p + (lane >> 5);
            const int row = row0 + 16 * i + r, col = col0 + (((lane & 31) ^ (r & 7)) * 4);
            if (row >= g.m || col >= g.n) continue;
            float* const dst = reinterpret_cast<float*>(c) + (int64_t)row * g.ldc + col;
            if (vec && col + 4 <= g.n) {
                *reinterpret_cast<f32x4*>(dst) = v[p];
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (col + e < g.n) dst[e] = v[p][e];
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The same for either type of C and any TJ, with padded rows instead of a swizzle: two rows of
// tiles at a time go through 32 x (16 TJ sizeof(TC) + 16) bytes of LDS of the wave's own at
// lds_wave and leave as whole rows of the block, 16 bytes per lane. (Stored from the registers a
// lane's four columns make every instruction 16 separate pieces of 32 or 64 bytes, which the
// CU's address unit takes one by one: a 256 x 160 tile of bf16 took 6 us that way.)
template <typename TC, int TJ>
constexpr int rows_wave_bytes() { return 32 * (16 * TJ * (int)sizeof(TC) + 16); }
template <bool F16, typename TC, int TI, int TJ, bool RAG>
__device__ __forceinline__ void store_rows_lds(const GemmArgs& g, void* c, const f32x4 (&acc)[TI][TJ], unsigned lds_wave, int row0, int col0, int lane) {
    constexpr int ES = (int)sizeof(TC);
    constexpr int PITCH = 16 * TJ * ES + 16; // bytes per staged row
    constexpr int CPR = TJ * ES;             // 16-byte chunks per row
    constexpr int PER = 16 / ES;             // elements per chunk
    static_assert(TI % 2 == 0, "rows of tiles in pairs");
    // From 96 columns of 128 rows a tile on, rows leave through the L2 (store_through): all tiles of a launch of one
    // round end together, and their rows are then in memory when the last wave ends. Calls, us: q/k/v and output
    // products of 1024 and 512 f32 rows, hidden 3072, 180.6 -> 175.9; a segment of 1632 tokens, 30 heads, f32, two layers
    // 524.6 -> 517.1; 643 tokens 255.4 -> 249.9. Smaller tiles carry so little that the stores' own way shows: 139 and 108
    // rows of bf16 96.0 -> 96.5. (A wave's part of a row need not be whole cache lines for that, it is 160 or 320 bytes in
    // the 160-column tiles: segments of bf16 C, 30 heads, two layers, 1536 tokens 450.7 -> 444.8, 672 tokens 232.7 -> 229.0.)
    // 16-bit rows of a length that lines do not divide lose: hidden 2568, through -> ordinary, 1675 and 512 rows 223.9 -> 220.8,
    // 315 and 512 140.8 -> 139.4; f32 rows of that width gain, 2023 and 512 rows 283.2 -> 281.5. Such a C belongs to a
    // product of as ragged a k, and that is what tells: a test of the address, with both stores behind it, costs the others
    // up to 0.9 %.
    constexpr bool THROUGH = TI * TJ >= 12 && (ES == 4 || !RAG);
    typedef __attribute__((address_space(3))) u32x2* lds_u32x2_t;
    typedef __attribute__((address_space(3))) f32x4* lds_f32x4_t;
    typedef const __attribute__((address_space(3))) u32x4* lds_u32x4_t;
    const int c16 = lane & 15, q = lane >> 4;
    const unsigned wbase = lds_wave + (unsigned)(c16 * PITCH + 4 * q * ES);
    // (uniform over the launch: rows of C start on 16 bytes; otherwise element by element)
    const bool vec = ((g.ldc * ES) % 16 == 0) && (reinterpret_cast<uintptr_t>(c) % 16 == 0);
#pragma unroll
    for (int ip = 0; ip < TI / 2; ip++) {
#pragma unroll
        for (int ii = 0; ii < 2; ii++)
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                const f32x4 v = acc[2 * ip + ii][j];
                const unsigned at = wbase + (unsigned)(ii * 16 * PITCH + j * 16 * ES);
                if constexpr (ES == 4) *(lds_f32x4_t)at = v;
                else if constexpr (F16) *(lds_u32x2_t)at = __builtin_bit_cast(u32x2, __builtin_convertvector(v, f16x4));
                else *(lds_u32x2_t)at = __builtin_bit_cast(u32x2, __builtin_convertvector(v, bf16x4));
            }
        __builtin_amdgcn_sched_barrier(0); // (keeps the scheduler from reading every accumulator out at once)
        u32x4 v[CPR / 2];
#pragma unroll
        for (int p = 0; p < CPR / 2; p++) {
            const int x = 64 * p + lane;
            v[p] = *(lds_u32x4_t)(lds_wave + (unsigned)((x / CPR) * PITCH + (x % CPR) * 16));
        }
#pragma unroll
        for (int p = 0; p < CPR / 2; p++) {
            const int x = 64 * p + lane;
            const int row = row0 + 32 * ip + x / CPR, col = col0 + (x % CPR) * PER;
            if (row >= g.m || col >= g.n) continue;
            TC* const dst = reinterpret_cast<TC*>(c) + (int64_t)row * g.ldc + col;
            if (vec && col + PER <= g.n) {
                if constexpr (THROUGH) store_through(dst, v[p]);
                else *reinterpret_cast<u32x4*>(dst) = v[p];
            } else {
#pragma unroll
                for (int e = 0; e < PER; e++) {
                    if (col + e >= g.n) break;
                    if constexpr (ES == 4) reinterpret_cast<unsigned*>(dst)[e] = v[p][e];
                    else reinterpret_cast<unsigned short*>(dst)[e] = (unsigned short)(v[p][e >> 1] >> (16 * (e & 1)));
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// XCD-aware tile id: workgroups go to the XCDs in turn, so each XCD gets one contiguous
// run of the tile sequence
__device__ __forceinline__ int logical_tile(int wg, int nwg) {
    const int xcd = wg & 7;
    const int idx = wg >> 3;
    const int base = nwg >> 3;
    const int rem = nwg & 7;
    return idx + xcd * base + (xcd < rem ? xcd : rem);
}

// Order of the tiles within that sequence: strips of kStrip tile columns (the groups lie side
// by side along n), walked row by row. The 32 tiles an XCD works on at one time then cover
// about 4 x 8 tiles of C and share 12 row panels of A and W in its L2; in row-major order
// they are 1 x 32 and share 33 (measured on a 4608 x 3072 x 9216 product: 1.08 GB of L2
// misses per launch against 0.50 GB). The last strip takes the columns that are left.
constexpr int kStrip = 8;
__device__ __forceinline__ void tile_coords(int logical, int tiles_m, int tiles_row, int& tm, int& tn) {
    const int per_strip = kStrip * tiles_m;
    const int nfull = tiles_row / kStrip;
    int strip = logical / per_strip;
    int width = kStrip;
    if (strip >= nfull) {
        strip = nfull;
        width = tiles_row - nfull * kStrip;
    }
    const int r = logical - strip * per_strip;
    tm = r / width;
    tn = strip * kStrip + (r - tm * width);
}

// The eight-wave build (k a multiple of 64; kept behind a knob). Both slabs go from global
// memory straight into LDS (buffer_load ... lds), no staging registers and no LDS store
// instructions; the other kernels use the same layout. Such a load writes lane i's 16 bytes
// at (LDS base) + 16 i, so rows are 128 bytes with no padding and bank conflicts
// are avoided by a swizzle instead: the 16-byte chunk c of row r lives at chunk
// position c ^ ((r >> 1) & 7); the lane that fills position p of row r fetches
// logical chunk p ^ ((r >> 1) & 7) from memory. A 16-lane fragment read of one
// logical chunk over 16 consecutive rows then touches 16 distinct bank groups.
constexpr int DMA_STAGE_BYTES = (BM + BN) * BK * 2; // 64 KB
constexpr size_t kDmaLdsBytes = 2 * (size_t)DMA_STAGE_BYTES;

// 256 x 256 tile of C, 4 x 2 waves (two per SIMD, 64 x 128 each).
template <bool F16, typename TC, int WM, int WN>
__global__ void __launch_bounds__(WM * WN * 64, 2) gemm_dma_kernel(const GemmArgs g) {
    constexpr int TB = 256;
    constexpr int STAGE_BYTES = 2 * TB * BK * 2; // A rows then W rows
    constexpr int NW = WM * WN;
    constexpr int TM = TB / WM / 16, TN = TB / WN / 16; // 16 x 16 MFMA tiles per wave
    constexpr int RW = TB / NW;                           // slab rows a wave fetches, of A and of W
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    typedef __attribute__((address_space(3))) void* lds_ptr_t;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int c16 = lane & 15;
    const int q4 = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;
    const int logical = logical_tile((int)blockIdx.x, (int)gridDim.x);
    const int tiles_row = g.tiles_n * g.groups;
    int tm, tn;
    tile_coords(logical, (g.m + TB - 1) / TB, tiles_row, tm, tn);
    const int grp = tn / g.tiles_n;
    tn -= grp * g.tiles_n;
    const void* const wp = grp == 0 ? g.w : g.w_more[grp - 1];
    void* const cp = grp == 0 ? g.c : g.c_more[grp - 1];
    const int m0 = tm * TB, n0 = tn * TB;

    const unsigned a_span = ((unsigned)(g.m - 1) * (unsigned)g.lda + (unsigned)g.k) * 2u;
    const unsigned w_span = ((unsigned)(g.n - 1) * (unsigned)g.ldw + (unsigned)g.k) * 2u;
    const rsrc_t a_rsrc = make_rsrc(g.a, a_span);
    const rsrc_t w_rsrc = make_rsrc(wp, w_span);
    // wave w fills rows RW w + 8 j + lane / 8 (j < RW / 8) of the A slab and of the W slab
    unsigned a_off[RW / 8], w_off[RW / 8];
#pragma unroll
    for (int j = 0; j < RW / 8; j++) {
        const int r = wave * RW + j * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int ar = min(m0 + r, g.m - 1); // rows past the edge re-read the last row; never stored
        const int wr = min(n0 + r, g.n - 1);
        a_off[j] = ((unsigned)ar * (unsigned)g.lda + (unsigned)(c * 8)) * 2u;
        w_off[j] = ((unsigned)wr * (unsigned)g.ldw + (unsigned)(c * 8)) * 2u;
    }
    const int nslab = g.k / BK;
    auto fetch_slab = [&](int s) __attribute__((always_inline)) {
        unsigned char* st = smem + (s & 1) * STAGE_BYTES + wave * (RW * BK * 2);
#pragma unroll
        for (int j = 0; j < RW / 8; j++) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(st + j * (8 * BK * 2)), 16, (int)a_off[j],
                                                     (int)((unsigned)s * (BK * 2u)), 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_ptr_t)(st + TB * BK * 2 + j * (8 * BK * 2)), 16,
                                                     (int)w_off[j], (int)((unsigned)s * (BK * 2u)), 0, 0);
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // fragment addresses: row (.. + c16), logical chunk 4 ks + q4 at position (4 ks + q4) ^ ((c16 >> 1) & 7)
    const int sw = (c16 >> 1) & 7;
    const int a_row = (wm * (16 * TM) + c16) * (BK * 2);
    const int w_row = TB * BK * 2 + (wn * (16 * TN) + c16) * (BK * 2);
    struct Frag { u32x4 a[TM], w[TN]; };
    auto read_frag = [&](Frag& f, int s, int ks) __attribute__((always_inline)) {
        const unsigned char* st = smem + (s & 1) * STAGE_BYTES;
        const int pos = ((4 * ks + q4) ^ sw) * 16;
#pragma unroll
        for (int i = 0; i < TM; i++) f.a[i] = *reinterpret_cast<const u32x4*>(st + a_row + i * 16 * (BK * 2) + pos);
#pragma unroll
        for (int j = 0; j < TN; j++) f.w[j] = *reinterpret_cast<const u32x4*>(st + w_row + j * 16 * (BK * 2) + pos);
    };
    // (The builtin form: with this few accumulators the compiler keeps them in place, and it
    // adds the wait states itself.)
    auto mfma_frag = [&](const Frag& f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                if constexpr (F16)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, f.w[j]), __builtin_bit_cast(f16x8, f.a[i]), acc[i][j], 0, 0, 0);
                else
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.w[j]), __builtin_bit_cast(bf16x8, f.a[i]), acc[i][j], 0, 0, 0);
            }
    };

    fetch_slab(0);
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): this wave's part of slab 0 is in LDS
    __syncthreads();
    for (int s = 0; s < nslab; s++) {
        // slab s+1 into the other stage: its readers (iteration s-1) are behind the last barrier.
        // (Spreading these loads over the four steps measured 9 % slower here: the compiler
        // then makes the fragment reads that follow each load wait for it.)
        if (s + 1 < nslab) fetch_slab(s + 1);
#pragma unroll
        for (int ks = 0; ks < BK / 32; ks++) {
            Frag f;
            read_frag(f, s, ks);
            mfma_frag(f);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): slab s+1 has landed
        __syncthreads();
    }
    store_tile16<F16, TC, TM, TN>(g, cp, acc, m0 + wm * (16 * TM), n0 + wn * (16 * TN), lane);
}

// ---------------------------------------------------------------------------
// Four-wave build: one wave per SIMD, each owning 128 x 128 of C as 8 x 8 tiles of
// v_mfma_f32_16x16x32 (256 accumulation registers; 16 fragment reads per 64 MFMAs, a third
// fewer LDS bytes per MFMA than the 8-wave build). One wave per SIMD has no neighbour to hide
// its waits, so the schedule leaves none. A 64-wide slab is two 32-wide steps of 64 MFMAs; the
// 16 fragments of the next step are read one per two MFMAs under the first half of the current
// one. The slab's one barrier sits in its FIRST step, after the 40th MFMA, when the slab's last
// fragments are in registers: it both frees the slab's LDS slots and makes slab s + 1 visible,
// whose first fragments are read under the second step. The 16 loads into the freed slots follow
// the barrier one per four MFMAs (the CU's address unit takes 16 cycles per 1 KB load and the
// four waves issue in the same phase: 64 cycles per round of loads).
// The LDS is five slots of one operand's slab (32 KB), W and A of the slabs going round in turn:
// into the two slots slab s frees go A of slab s + 2, which has 96 MFMAs (0.6-0.8 us) to arrive,
// and W of slab s + 3, which has 224 (weights come from memory, 0.6 us away when it is idle).
// With two whole stages, where all loads of slab s + 2 went out after the barrier and the last had
// 64 MFMAs, cold weights cost 8-16 % (same shapes with weights in the last-level cache: 204 / 246 us
// against 221 / 285 for 4608 x 3072 x 9216 and 4608 x 12288 x 3072); now 4-10 % (195 / 234, 204 / 259).
// The loop is unrolled over the five slots, so every LDS address is a pointer plus a constant. Same
// 128-byte swizzled rows as the direct-to-LDS build above.
constexpr int SLOT = BM * BK * 2; // one operand's half of a slab: 32 KB
constexpr size_t kRingLdsBytes = 5 * (size_t)SLOT; // 160 KB
template <bool F16, typename TC>
__global__ void __launch_bounds__(256, 1) gemm_ring_kernel(const GemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int c16 = lane & 15;
    const int q4 = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    // a tile of the split last round: workgroup = (tile, part), the part is a range of slabs
    int logical, part_id = 0, splits = 1;
    const int tiles_row = g.tiles_n * g.groups;
    const int tiles_m = (g.m + BM - 1) / BM;
    if ((int)blockIdx.x < g.part_wgs) {
        const int t = (int)blockIdx.x / g.splits;
        if (t >= tiles_m * tiles_row - g.tile_base) return; // padding up to a multiple of 8
        part_id = (int)blockIdx.x - t * g.splits;
        splits = g.splits;
        logical = g.tile_base + t;
    } else {
        // (part_wgs is a multiple of 8, so a workgroup's XCD is its id's low bits here too)
        logical = logical_tile((int)blockIdx.x - g.part_wgs, (int)gridDim.x - g.part_wgs);
    }
    int tm, tn;
    tile_coords(logical, tiles_m, tiles_row, tm, tn);
    const int grp = tn / g.tiles_n;
    tn -= grp * g.tiles_n;
    const void* const wp = grp == 0 ? g.w : g.w_more[grp - 1];
    void* const cp = grp == 0 ? g.c : g.c_more[grp - 1];
    const int m0 = tm * BM, n0 = tn * BN;

    const unsigned a_span = ((unsigned)(g.m - 1) * (unsigned)g.lda + (unsigned)g.k) * 2u;
    const unsigned w_span = ((unsigned)(g.n - 1) * (unsigned)g.ldw + (unsigned)g.k) * 2u;
    // The 16 loads of a slab go as four runs of four whose LDS targets lie 1 KB apart: M0 is set
    // once per run and the other three use the instruction's offset field, which also moves the
    // address in memory; that is taken off the lane's offset, and the descriptors start 3 KB
    // below the operands so that the offset stays positive.
    constexpr unsigned kBias = kGemmDescBias;
    const u32x4 a_rsrc = make_rsrc_words(reinterpret_cast<const unsigned char*>(g.a) - kBias, a_span + kBias);
    const u32x4 w_rsrc = make_rsrc_words(reinterpret_cast<const unsigned char*>(wp) - kBias, w_span + kBias);
    const unsigned lds0 = lds_address(smem);
    // wave w fills rows 64 w + 8 j + lane / 8 (j < 8) of the A slab and of the W slab
    unsigned a_off[8], w_off[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int r = wave * 64 + j * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int ar = min(m0 + r, g.m - 1); // rows past the edge re-read the last row; never stored
        const int wr = min(n0 + r, g.n - 1);
        a_off[j] = ((unsigned)ar * (unsigned)g.lda + (unsigned)(c * 8)) * 2u + kBias - (unsigned)(j & 3) * 1024u;
        w_off[j] = ((unsigned)wr * (unsigned)g.ldw + (unsigned)(c * 8)) * 2u + kBias - (unsigned)(j & 3) * 1024u;
    }
    int nslab = g.k / BK, slab0 = 0;
    if (splits > 1) {
        const int per = (nslab + splits - 1) / splits;
        slab0 = part_id * per;
        // (uniform, but the division runs on the vector unit)
        nslab = __builtin_amdgcn_readfirstlane(max(min(nslab - slab0, per), 0));
        slab0 = __builtin_amdgcn_readfirstlane(slab0);
    }
    const unsigned fetch_lds = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * (64 * BK * 2));
    // the i-th (i < 8) of the loads that bring this wave's rows of an operand's slab s into slot `slot`
    // (eight rows a load), in order: the first of every four sets M0 for the rest. Slabs past the end
    // re-fetch the last one into a slot nobody reads any more.
    auto fetch_one = [&](bool is_w, int s, int slot, int i) __attribute__((always_inline)) {
        // (uniform, but the compiler may have formed it in a vector register)
        const unsigned uo = __builtin_amdgcn_readfirstlane((unsigned)min(slab0 + max(s < nslab ? s : nslab - 1, 0), g.k / BK - 1) * (BK * 2u));
        if ((i & 3) == 0) lds_dma_base(fetch_lds + (unsigned)(slot * SLOT + (i >> 2) * (32 * BK * 2)));
        const u32x4& rsrc = is_w ? w_rsrc : a_rsrc;
        const unsigned off = is_w ? w_off[i] : a_off[i];
        if ((i & 3) == 0) load_to_lds_16_at<0>(rsrc, off, uo);
        if ((i & 3) == 1) load_to_lds_16_at<1024>(rsrc, off, uo);
        if ((i & 3) == 2) load_to_lds_16_at<2048>(rsrc, off, uo);
        if ((i & 3) == 3) load_to_lds_16_at<3072>(rsrc, off, uo);
    };

    f32x4 acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // fragment addresses: row (.. + c16), logical chunk 4 ks + q4 (ks < 2) at c ^ ((row >> 1) & 7);
    // a tile row adds 16 rows = 2 KB. (Pointers, so that the constant parts go into the
    // instruction's offset field; that field reaches 64 KB: one pointer per two slots.)
    typedef const __attribute__((address_space(3))) unsigned char* lds_byte_t;
    typedef const __attribute__((address_space(3))) u32x4* lds_u32x4_t;
    const lds_byte_t lds_base = (lds_byte_t)smem;
    const int sw = (c16 >> 1) & 7;
    lds_byte_t fa[3][2], fw[3][2]; // [slot / 2][ks]
#pragma unroll
    for (int sp = 0; sp < 3; sp++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const int pos = ((4 * ks + q4) ^ sw) * 16;
            fa[sp][ks] = lds_base + (2 * sp * SLOT + (wm * 128 + c16) * (BK * 2) + pos);
            fw[sp][ks] = lds_base + (2 * sp * SLOT + (wn * 128 + c16) * (BK * 2) + pos);
        }
    struct Frag { u32x4 a[8], w[8]; };
    // the r-th of the 16 reads of a fragment set; W and A of slab s are in slots 2 s and 2 s + 1 (mod 5)
    auto read_one = [&](Frag& f, int a_slot, int w_slot, int ks, int r) __attribute__((always_inline)) {
        if (r < 8) f.a[r] = *(lds_u32x4_t)(fa[a_slot >> 1][ks] + ((a_slot & 1) * SLOT + r * 16 * (BK * 2)));
        else f.w[r - 8] = *(lds_u32x4_t)(fw[w_slot >> 1][ks] + ((w_slot & 1) * SLOT + (r - 8) * 16 * (BK * 2)));
    };
    // One 32-wide step of slab s (P = s mod 5): 64 MFMAs on `cur`, the 16 reads of `nxt` under the
    // first 32 of them. FIRST (the slab's first step): the barrier after the 40th MFMA, then the first
    // 6 of the 16 loads that go into the slab's two slots, one per four MFMAs; the second step sends
    // the other 10.
    auto mfma_step = [&](auto first_c, auto p_c, const Frag& cur, Frag& nxt, int s) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value;
        constexpr int P = decltype(p_c)::value;
        constexpr int NP = FIRST ? P : (P + 1) % 5; // the slab nxt belongs to
        auto send = [&](int i) __attribute__((always_inline)) {
            if (i < 8) fetch_one(false, s + 2, (2 * P) % 5, i);
            else fetch_one(true, s + 3, (2 * P + 1) % 5, i - 8);
        };
#pragma unroll
        for (int t = 0; t < 64; t++) {
            if (FIRST && t >= 40 && (t & 3) == 0) send((t - 40) >> 2);
            if (!FIRST && (t & 3) == 1 && t < 40) send(6 + (t >> 2));
            if ((t & 1) == 0 && t < 32) read_one(nxt, (2 * NP + 1) % 5, (2 * NP) % 5, FIRST ? 1 : 0, t >> 1);
            mfma16<F16>(cur.w[t & 7], cur.a[t >> 3], acc[t >> 3][t & 7]);
            __builtin_amdgcn_sched_barrier(0);
            if (FIRST && t == 39) {
                __builtin_amdgcn_s_waitcnt(0x0078); // vmcnt(8) lgkmcnt(0): all but W of slab s + 2 has landed
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

#pragma unroll
    for (int i = 0; i < 8; i++) fetch_one(true, 0, 0, i);
#pragma unroll
    for (int i = 0; i < 8; i++) fetch_one(false, 0, 1, i);
#pragma unroll
    for (int i = 0; i < 8; i++) fetch_one(true, 1, 2, i);
#pragma unroll
    for (int i = 0; i < 8; i++) fetch_one(false, 1, 3, i);
#pragma unroll
    for (int i = 0; i < 8; i++) fetch_one(true, 2, 4, i);
    __builtin_amdgcn_s_waitcnt(0x4F78); // vmcnt(24): slab 0 has landed
    __syncthreads();
    Frag f0, f1;
#pragma unroll
    for (int r = 0; r < 16; r++) read_one(f0, 1, 0, 0, r);
    auto slab = [&](auto p_c, int s) __attribute__((always_inline)) {
        mfma_step(std::true_type{}, p_c, f0, f1, s);
        mfma_step(std::false_type{}, p_c, f1, f0, s);
    };
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 2> I2;
    typedef std::integral_constant<int, 3> I3;
    typedef std::integral_constant<int, 4> I4;
    int s = 0;
    for (; s + 5 <= nslab; s += 5) {
        slab(I0{}, s);
        slab(I1{}, s + 1);
        slab(I2{}, s + 2);
        slab(I3{}, s + 3);
        slab(I4{}, s + 4);
        mfma16_drain(); // (24 cycles per five slabs: whatever follows the loop body may read the accumulators)
    }
    if (s < nslab) { slab(I0{}, s); mfma16_drain(); }
    if (s + 1 < nslab) { slab(I1{}, s + 1); mfma16_drain(); }
    if (s + 2 < nslab) { slab(I2{}, s + 2); mfma16_drain(); }
    if (s + 3 < nslab) { slab(I3{}, s + 3); mfma16_drain(); }
    __builtin_amdgcn_s_waitcnt(0x0F70); // no direct load may outlive the workgroup's LDS
    if (splits > 1) {
        // partial tile in the accumulation layout: [tile][part][wave][i][j][lane] x 16 bytes,
        // every store instruction 1 KB in a row; the merge kernel reads it the same way
        f32x4* dst = reinterpret_cast<f32x4*>(g.part) +
                     ((((int64_t)(logical - g.tile_base) * g.splits + part_id) * 4 + wave) * 64) * 64 + lane;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) dst[(i * 8 + j) * 64] = acc[i][j];
        return;
    }
    // (this wave's 8 KB of the slot that A of slab `nslab` went to: only this wave's loads write them,
    // they have landed, and nobody needs what is there)
    const unsigned epi_lds = fetch_lds + (unsigned)(((2 * nslab + 1) % 5) * SLOT);
    if constexpr (sizeof(TC) == 2) store_tile_lds16<F16, TC, 8>(g, cp, acc, epi_lds, m0 + wm * 128, n0 + wn * 128, lane);
    else store_tile_lds32<8>(g, cp, acc, epi_lds, m0 + wm * 128, n0 + wn * 128, lane);
}

// ---------------------------------------------------------------------------
// Problems with too few 256-tiles to fill the chip: the four-wave schedule of gemm_ring_kernel
// for any tile of (32 TI) x (32 TJ), one workgroup per CU, each wave (16 TI) x (16 TJ) of C. A
// smaller tile spends fewer cycles on a slab than the slab takes to arrive, so the LDS holds ST
// slabs and ST - 1 of them are on their way while one is worked on.
//   slab s, first step: the MFMAs of its k 0..31 on f0; its k 32..63 fragments are read into f1;
//     after the last of those reads the slab's one barrier (this wave's part of slab s + 1 has
//     landed, everybody has slab s in registers: its stage is free);
//   second step: the MFMAs on f1, the k 0..31 fragments of slab s + 1 are read into f0;
//   from the barrier on, one load of slab s + ST per five MFMAs (fewer where a slab has fewer to a load);
//     what is left of them goes out in the next slab's first step, ahead of its barrier.
constexpr int vm_lgkm0(int vm) { return (vm & 15) | 0x70 | ((vm >> 4) << 14); }           // vmcnt(vm) lgkmcnt(0)
constexpr int vm_only(int vm) { return (vm & 15) | 0xF70 | ((vm >> 4) << 14); }           // vmcnt(vm)
constexpr size_t pipe_lds_bytes(int ti, int tj, int st) { return (size_t)st * (size_t)(ti + tj) * 32 * BK * 2; }

template <bool F16, typename TC, int TI, int TJ, int ST, bool RAG>
__global__ void __launch_bounds__(256, 1) gemm_pipe_kernel(const GemmArgs g) {
    constexpr int TBM = 32 * TI, TBN = 32 * TJ;
    constexpr int STAGE = (TBM + TBN) * BK * 2; // bytes: A rows then W rows
    constexpr int NM = TI * TJ;                 // MFMAs of a step
    constexpr int NR = TI + TJ;                 // fragment reads of a step
    constexpr int NL = TI + TJ;                 // loads of a wave per slab
    constexpr int RS = NM >= 32 ? 2 : 1;        // MFMAs per fragment read
    constexpr int TB = (NR - 1) * RS + 5 < NM - 1 ? (NR - 1) * RS + 5 : NM - 1; // the barrier follows this MFMA of the first step
    // MFMAs per load: five where a slab has that many (192 x 192 and 256 x 160 tiles), so that the loads spread over all of it;
    // closer, they hold the waves at the memory queue. Launches, us, at 2, 3, 4, 5 and 6: 1024 x 3072 x 9216 65.0, 61.3, 57.1,
    // 54.1-55.5, 54.4; 1632 x 3840 x 11520 140, 133, 132, 130, 130; 1632 x 3840 x 3840 60.8, 58.2, 56.4, 55.9, 56.0. Four against
    // five over twelve products of 900 to 3000 rows: 0 to 4 % (3000 x 10272 x 2568 164.4 -> 158.4), none slower.
    constexpr int LS = 2 * NM / NL < 5 ? 2 * NM / NL : 5;
    // load i goes out ahead of MFMA TB + 1 + LS i, counted from the start of the slab that frees its stage
    constexpr int IW = (2 * NM - (TB + 1) + LS - 1) / LS < NL ? (2 * NM - (TB + 1) + LS - 1) / LS : NL; // loads that go out within that slab
    static_assert(LS >= 1 && TB + 1 + LS * (NL - 1) <= 2 * NM + TB, "all loads of a slab are out by the next barrier");
    static_assert((ST - 1) * NL <= 63, "vmcnt counts to 63");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int c16 = lane & 15;
    const int q4 = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    const int tiles_row = g.tiles_n * g.groups;
    const int tiles_m = (g.m + TBM - 1) / TBM;
    int tm, tn;
    tile_coords(logical_tile((int)blockIdx.x, (int)gridDim.x), tiles_m, tiles_row, tm, tn);
    const int grp = tn / g.tiles_n;
    tn -= grp * g.tiles_n;
    const void* const wp = grp == 0 ? g.w : g.w_more[grp - 1];
    void* const cp = grp == 0 ? g.c : g.c_more[grp - 1];
    const int m0 = tm * TBM, n0 = tn * TBN;

    const unsigned a_span = ((unsigned)(g.m - 1) * (unsigned)g.lda + (unsigned)g.k) * 2u;
    const unsigned w_span = ((unsigned)(g.n - 1) * (unsigned)g.ldw + (unsigned)g.k) * 2u;
    // loads in runs of four under one M0, as in gemm_ring_kernel
    constexpr unsigned kBias = kGemmDescBias;
    const u32x4 a_rsrc = make_rsrc_words(reinterpret_cast<const unsigned char*>(g.a) - kBias, a_span + kBias);
    const u32x4 w_rsrc = make_rsrc_words(reinterpret_cast<const unsigned char*>(wp) - kBias, w_span + kBias);
    const unsigned lds0 = lds_address(smem);
    // wave w fills rows 8 TI w + 8 j + lane / 8 (j < TI) of the A slab and rows 8 TJ w + .. of the W slab
    unsigned a_off[TI], w_off[TJ];
#pragma unroll
    for (int j = 0; j < TI; j++) {
        const int r = wave * (8 * TI) + j * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int ar = min(m0 + r, g.m - 1); // rows past the edge re-read the last row; never stored
        a_off[j] = ((unsigned)ar * (unsigned)g.lda + (unsigned)(c * 8)) * 2u + kBias - (unsigned)(j & 3) * 1024u;
    }
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        const int r = wave * (8 * TJ) + j * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int wr = min(n0 + r, g.n - 1);
        w_off[j] = ((unsigned)wr * (unsigned)g.ldw + (unsigned)(c * 8)) * 2u + kBias - (unsigned)(j & 3) * 1024u;
    }
    const int nslab = (g.k + BK - 1) / BK;
    const unsigned a_lds = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * (8 * TI * BK * 2));
    const unsigned w_lds = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)(TBM * BK * 2) + (unsigned)wave * (8 * TJ * BK * 2));
    // the i-th (i < NL) load of this wave's part of slab s into stage st: A rows, then W rows; within an
    // operand in order, the first of every four sets M0 for the rest. Slabs past the end re-fetch the
    // last one into a stage nobody reads any more.
    auto fetch_one = [&](int s, int st, int i) __attribute__((always_inline)) {
        const unsigned uo = (unsigned)(s < nslab ? s : nslab - 1) * (BK * 2u);
        const bool is_w = i >= TI;
        const int j = is_w ? i - TI : i;
        if ((j & 3) == 0) lds_dma_base((is_w ? w_lds : a_lds) + (unsigned)(st * STAGE + (j >> 2) * 4096));
        const u32x4& rsrc = is_w ? w_rsrc : a_rsrc;
        const unsigned off = is_w ? w_off[is_w ? j : 0] : a_off[is_w ? 0 : j];
        if ((j & 3) == 0) load_to_lds_16_at<0>(rsrc, off, uo);
        if ((j & 3) == 1) load_to_lds_16_at<1024>(rsrc, off, uo);
        if ((j & 3) == 2) load_to_lds_16_at<2048>(rsrc, off, uo);
        if ((j & 3) == 3) load_to_lds_16_at<3072>(rsrc, off, uo);
    };

    f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    typedef const __attribute__((address_space(3))) unsigned char* lds_byte_t;
    typedef const __attribute__((address_space(3))) u32x4* lds_u32x4_t;
    const lds_byte_t lds_base = (lds_byte_t)smem;
    const int sw = (c16 >> 1) & 7;
    lds_byte_t fa[ST][2], fw[ST][2]; // [stage][ks]: row (.. + c16), logical chunk 4 ks + q4 at c ^ ((row >> 1) & 7)
#pragma unroll
    for (int st = 0; st < ST; st++)
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const int pos = ((4 * ks + q4) ^ sw) * 16;
            fa[st][ks] = lds_base + (st * STAGE + (wm * (16 * TI) + c16) * (BK * 2) + pos);
            fw[st][ks] = lds_base + (st * STAGE + TBM * BK * 2 + (wn * (16 * TJ) + c16) * (BK * 2) + pos);
        }
    struct Frag { u32x4 a[TI], w[TJ]; };
    auto read_one = [&](Frag& f, int st, int ks, int r) __attribute__((always_inline)) {
        if (r < TI) f.a[r] = *(lds_u32x4_t)(fa[st][ks] + r * 16 * (BK * 2));
        else f.w[r - TI] = *(lds_u32x4_t)(fw[st][ks] + (r - TI) * 16 * (BK * 2));
    };
    Frag f0, f1;
    // one step of slab s (in stage S0): FIRST = the MFMAs on its k 0..31
    auto step = [&](auto first_c, auto st_c, Frag& cur, Frag& nxt, int s) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value;
        if constexpr (RAG) {
            // the last slab of a k that is not a multiple of 64: what lies past k in a row (the next
            // row, or what the descriptor's bound made of it) must not count
            if (s == nslab - 1) {
                const bool keep = s * BK + (FIRST ? 0 : 32) + 8 * q4 < g.k;
#pragma unroll
                for (int i = 0; i < TI; i++) cur.a[i] = keep ? cur.a[i] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int j = 0; j < TJ; j++) cur.w[j] = keep ? cur.w[j] : u32x4{0u, 0u, 0u, 0u};
            }
        }
        constexpr int S0 = decltype(st_c)::value;
        constexpr int SN = (S0 + 1) % ST;           // stage of slab s + 1
        constexpr int SP = (S0 + ST - 1) % ST;      // of slab s - 1, which slab s - 1 + ST takes
#pragma unroll
        for (int t = 0; t < NM; t++) {
            const int late = 2 * NM + t - (TB + 1); // loads of slab s - 1 + ST that are still to go out
            if (FIRST && t <= TB && late % LS == 0 && late / LS >= IW && late / LS < NL) fetch_one(s - 1 + ST, SP, late / LS);
            const int own = (FIRST ? t : NM + t) - (TB + 1);
            if (own >= 0 && own % LS == 0 && own / LS < IW) fetch_one(s + ST, S0, own / LS);
            if (t % RS == 0 && t / RS < NR) read_one(nxt, FIRST ? S0 : SN, FIRST ? 1 : 0, t / RS);
            mfma16<F16>(cur.w[t % TJ], cur.a[t / TJ], acc[t / TJ][t % TJ]);
            __builtin_amdgcn_sched_barrier(0);
            if (FIRST && t == TB) {
                __builtin_amdgcn_s_waitcnt(vm_lgkm0((ST - 2) * NL));
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    auto slab = [&](auto st_c, int s) __attribute__((always_inline)) {
        step(std::true_type{}, st_c, f0, f1, s);
        step(std::false_type{}, st_c, f1, f0, s);
    };

#pragma unroll
    for (int st = 0; st < ST; st++)
#pragma unroll
        for (int i = 0; i < (st < ST - 1 ? NL : IW); i++) fetch_one(st, st, i); // (the rest of the last one goes out in slab 0)
    __builtin_amdgcn_s_waitcnt(vm_only((ST - 2) * NL + IW)); // slab 0 has landed
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NR; r++) read_one(f0, 0, 0, r);
    int s = 0;
    for (; s + ST <= nslab; s += ST) {
        slab(std::integral_constant<int, 0>{}, s);
        slab(std::integral_constant<int, 1>{}, s + 1);
        if constexpr (ST > 2) slab(std::integral_constant<int, 2 % ST>{}, s + 2);
        if constexpr (ST > 3) slab(std::integral_constant<int, 3 % ST>{}, s + 3);
        static_assert(ST >= 2 && ST <= 4, "two to four stages");
        mfma16_drain(); // whatever follows the loop body may read the accumulators
    }
    if (s < nslab) { slab(std::integral_constant<int, 0>{}, s); mfma16_drain(); }
    if constexpr (ST > 2) if (s + 1 < nslab) { slab(std::integral_constant<int, 1>{}, s + 1); mfma16_drain(); }
    if constexpr (ST > 3) if (s + 2 < nslab) { slab(std::integral_constant<int, 2 % ST>{}, s + 2); mfma16_drain(); }
    __builtin_amdgcn_s_waitcnt(0x0F70); // this wave's direct loads (re-fetches past the end) have landed
    __syncthreads();                    // and everybody's: the stages are idle
    static_assert(4 * rows_wave_bytes<TC, TJ>() <= ST * STAGE, "the epilogue's rows fit the stages");
    store_rows_lds<F16, TC, TI, TJ, RAG>(g, cp, acc, lds0 + (unsigned)(wave * rows_wave_bytes<TC, TJ>()), m0 + wm * (16 * TI), n0 + wn * (16 * TJ), lane);
}

// Adds the parts of the k-split tiles in part order and writes C. A workgroup takes the 32 x
// 128 block (tile, wave, i) of the four-wave build's accumulation layout: its wave j owns the
// 16 x 16 tiles (2 i + r / 2, 2 j + r % 2), r < 4; a lane holds row lane % 16 and columns
// 4 (lane / 16) .. + 4 of each. Every part's load (4 x splits of 16 bytes per lane) is sent
// before the first is used; the sums are turned through LDS so that C is stored as whole rows
// of the block.
constexpr int kMaxKSplits = 8;
template <bool F16, typename TC>
__global__ void __launch_bounds__(256) gemm_merge_kernel(const GemmArgs g) {
    constexpr int ES = (int)sizeof(TC);
    constexpr int PITCH = 128 * ES + 16; // bytes per staged row
    __shared__ __attribute__((aligned(16))) unsigned char stage[32 * PITCH];
    const int t = (int)blockIdx.x >> 4;
    const int wave = ((int)blockIdx.x >> 2) & 3, i = (int)blockIdx.x & 3;
    const int j = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    // quad (tile row 2 i + (r >> 1), tile column 2 j + (r & 1)) for r < 4
    const f32x4* src = reinterpret_cast<const f32x4*>(g.part) +
                       ((((int64_t)t * g.splits) * 4 + wave) * 64 + (16 * i + 2 * j)) * 64 + lane;
    f32x4 v[kMaxKSplits][4];
#pragma unroll
    for (int z = 0; z < kMaxKSplits; z++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            v[z][r] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (z < g.splits) v[z][r] = src[(int64_t)z * (4 * 64 * 64) + ((r >> 1) * 8 + (r & 1)) * 64];
        }
    const int c16 = lane & 15, q4 = lane >> 4;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        f32x4 sum = v[0][r];
#pragma unroll
        for (int z = 1; z < kMaxKSplits; z++)
            if (z < g.splits) sum += v[z][r];
        unsigned char* dst = stage + (16 * (r >> 1) + c16) * PITCH + (32 * j + 16 * (r & 1) + 4 * q4) * ES;
        if constexpr (ES == 4) {
            *reinterpret_cast<f32x4*>(dst) = sum;
        } else {
            if constexpr (F16) *reinterpret_cast<u32x2*>(dst) = __builtin_bit_cast(u32x2, __builtin_convertvector(sum, f16x4));
            else *reinterpret_cast<u32x2*>(dst) = __builtin_bit_cast(u32x2, __builtin_convertvector(sum, bf16x4));
        }
    }
    __syncthreads();

    const int tiles_row = g.tiles_n * g.groups;
    int tm, tn;
    tile_coords(g.tile_base + t, (g.m + BM - 1) / BM, tiles_row, tm, tn);
    const int grp = tn / g.tiles_n;
    tn -= grp * g.tiles_n;
    void* const cp = grp == 0 ? g.c : g.c_more[grp - 1];
    const int row0 = tm * BM + (wave >> 1) * 128 + 32 * i;
    const int col0 = tn * BN + (wave & 1) * 128;
    constexpr int PER = 16 / ES;       // elements per 16-byte chunk
    constexpr int CH = 128 / PER;      // chunks per row of the block
    const bool vec = (g.ldc % PER == 0) && (reinterpret_cast<uintptr_t>(cp) % 16 == 0);
#pragma unroll
    for (int q = 0; q < 32 * CH / 256; q++) {
        const int c = (int)threadIdx.x + 256 * q;
        const int rr = c / CH, cc = c % CH;
        const int row = row0 + rr, col = col0 + PER * cc;
        if (row >= g.m || col >= g.n) continue;
        const u32x4 x = *reinterpret_cast<const u32x4*>(stage + rr * PITCH + cc * 16);
        TC* dst = reinterpret_cast<TC*>(cp) + (int64_t)row * g.ldc + col;
        if (vec && col + PER <= g.n) {
            *reinterpret_cast<u32x4*>(dst) = x;
        } else {
#pragma unroll
            for (int e = 0; e < PER; e++) {
                if (col + e >= g.n) break;
                if constexpr (ES == 4) reinterpret_cast<unsigned*>(dst)[e] = x[e];
                else reinterpret_cast<unsigned short*>(dst)[e] = (unsigned short)(x[e >> 1] >> (16 * (e & 1)));
            }
        }
    }
}

// f32 activations rounded to the weight's 16-bit type, once, into dense [m][k] rows: the
// products that follow then move their A slabs straight into LDS like 16-bit activations
// instead of rounding every slab of every tile (each row of A is read by every column tile).
template <bool F16>
__global__ void __launch_bounds__(256) gemm_round_kernel(const float* a, int64_t lda, unsigned short* out, int m, int k) {
    // grid x = row, grid y = 4096-element stretch of the row; a thread rounds two groups of 8
    const int row = (int)blockIdx.x;
    const int c0 = (int)blockIdx.y * 4096 + (int)threadIdx.x * 8;
    const float* src = a + (int64_t)row * lda;
    unsigned short* dst = out + (int64_t)row * k;
    f32x4 lo[2], hi[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int c = min(c0 + u * 2048, k - 8); // past the end: re-read the last group, not stored
        lo[u] = *reinterpret_cast<const f32x4*>(src + c);
        hi[u] = *reinterpret_cast<const f32x4*>(src + c + 4);
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int c = c0 + u * 2048;
        if (c >= k) continue;
        f32x8 v;
#pragma unroll
        for (int i = 0; i < 4; i++) { v[i] = lo[u][i]; v[4 + i] = hi[u][i]; }
        u32x4 r;
        if constexpr (F16) r = __builtin_bit_cast(u32x4, __builtin_convertvector(v, f16x8));
        else r = __builtin_bit_cast(u32x4, __builtin_convertvector(v, bf16x8));
        store_through(dst + c, r);
    }
}

// f32 activations where there is no room for their rounded copy or none may be taken (a queue under
// capture), and rows so long that a descriptor does not reach their end: each (32 TI) x (32 TI)
// tile reads its rows through pointers and rounds them on their way into LDS, the next
// 64-wide slab on its way in registers. Bound by that slab's wait for memory, or (many tiles) by what the
// tiles read from L2: the way out and never the choice (f32 A, us: 77 x 3072 x 3 x 3072 39, 600 x 3000 x 3 x
// 3000 91, 4096 x 3000 x 3000 146). The MFMAs add k in the order of the other kernels: same bits.
template <typename TA, bool F16, typename TC, int TI>
__global__ void __launch_bounds__(256) gemm_unstaged_kernel(const GemmArgs g) {
    constexpr bool F32 = std::is_same<TA, float>::value;
    constexpr int T = 32 * TI, PITCH = BK * 2 + 16; // bytes per LDS row
    constexpr int CPT = T * BK / (256 * 8);         // 8-element chunks of a slab per thread and operand
    __shared__ __attribute__((aligned(16))) unsigned char sa[T * PITCH], sw[T * PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c16 = lane & 15, q4 = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    int tm, tn;
    tile_coords(logical_tile((int)blockIdx.x, (int)gridDim.x), (g.m + T - 1) / T, g.tiles_n * g.groups, tm, tn);
    const int grp = tn / g.tiles_n;
    tn -= grp * g.tiles_n;
    const void* const wp = grp == 0 ? g.w : g.w_more[grp - 1];
    void* const cp = grp == 0 ? g.c : g.c_more[grp - 1];
    const int m0 = tm * T, n0 = tn * T;
    // thread = chunk c of rows r, r + 32, .. of either operand; rows past the edge re-read the last one, never stored
    const int r = tid >> 3, c = (tid & 7) * 8;
    const TA* arow[CPT];
    const unsigned short* wrow[CPT];
#pragma unroll
    for (int u = 0; u < CPT; u++) {
        arow[u] = static_cast<const TA*>(g.a) + (int64_t)min(m0 + r + 32 * u, g.m - 1) * g.lda;
        wrow[u] = static_cast<const unsigned short*>(wp) + (int64_t)min(n0 + r + 32 * u, g.n - 1) * g.ldw;
    }
    f32x4 acc[TI][TI];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TI; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const unsigned k = (unsigned)g.k; // (may be just short of 2^31)
    constexpr int AV = F32 ? 2 : 1;   // 16-byte loads per chunk of A
    u32x4 av[CPT * AV], wv[CPT];
    auto load = [&](unsigned k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < CPT; u++) {
            const unsigned at = k0 + c < k ? k0 + c : 0; // (k is a multiple of 8: a chunk is whole or past the end)
#pragma unroll
            for (int x = 0; x < AV; x++) av[u * AV + x] = *reinterpret_cast<const u32x4*>(arow[u] + at + 4 * x);
            wv[u] = *reinterpret_cast<const u32x4*>(wrow[u] + at);
        }
    };
    load(0);
    for (unsigned k0 = 0; k0 < k; k0 += BK) {
        u32x4 ah[CPT], wh[CPT];
#pragma unroll
        for (int u = 0; u < CPT; u++) {
            if constexpr (F32) {
                f32x8 v;
#pragma unroll
                for (int i = 0; i < 8; i++) v[i] = __uint_as_float(av[2 * u + (i >> 2)][i & 3]);
                if constexpr (F16) ah[u] = __builtin_bit_cast(u32x4, __builtin_convertvector(v, f16x8));
                else ah[u] = __builtin_bit_cast(u32x4, __builtin_convertvector(v, bf16x8));
            } else {
                ah[u] = av[u];
            }
            wh[u] = wv[u];
            if (k0 + c >= k) ah[u] = wh[u] = u32x4{0u, 0u, 0u, 0u};
        }
        __syncthreads(); // the last slab's fragments have been read
#pragma unroll
        for (int u = 0; u < CPT; u++) {
            *reinterpret_cast<u32x4*>(sa + (r + 32 * u) * PITCH + c * 2) = ah[u];
            *reinterpret_cast<u32x4*>(sw + (r + 32 * u) * PITCH + c * 2) = wh[u];
        }
        __syncthreads();
        if (k - k0 > BK) load(k0 + BK);
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            u32x4 fa[TI], fw[TI];
#pragma unroll
            for (int i = 0; i < TI; i++) {
                fa[i] = *reinterpret_cast<const u32x4*>(sa + ((wm * TI + i) * 16 + c16) * PITCH + ks * 64 + q4 * 16);
                fw[i] = *reinterpret_cast<const u32x4*>(sw + ((wn * TI + i) * 16 + c16) * PITCH + ks * 64 + q4 * 16);
            }
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TI; j++) mfma16<F16>(fw[j], fa[i], acc[i][j]);
            mfma16_drain();
        }
    }
    store_tile16<F16, TC, TI, TI>(g, cp, acc, m0 + wm * (16 * TI), n0 + wn * (16 * TI), lane);
}
// From this many 128-tiles on they are taken instead of 64-tiles (us, 64 against 128: 192 tiles 46 / 65, 240
// 71 / 72, 360 111 / 91, 768 215 / 146).
constexpr int kUnstagedLargeTiles = 240;
template <typename TA, bool F16, typename TC>
static hipError_t launch_unstaged(GemmArgs g, hipStream_t stream) {
    auto count = [&](int t) { return (int64_t)((g.m + t - 1) / t) * ((g.n + t - 1) / t) * g.groups; };
    const int t = count(128) >= kUnstagedLargeTiles ? 128 : 64;
    g.tiles_n = (g.n + t - 1) / t;
    const int64_t nwg = count(t);
    if (nwg <= 0 || nwg > 0x7fffffff) return hipErrorInvalidValue;
    if (t == 128) gemm_unstaged_kernel<TA, F16, TC, 4><<<dim3((unsigned)nwg), dim3(256), 0, stream>>>(g);
    else gemm_unstaged_kernel<TA, F16, TC, 2><<<dim3((unsigned)nwg), dim3(256), 0, stream>>>(g);
    return hipGetLastError();
}

// Measured on the Klein projections, same box, all with row-by-row stores and row-major tile
// order: eight waves (two per SIMD, 64 x 128 each) 1048-1217 TFLOP/s; four waves with the
// schedule above 1047-1248; four waves with the simple loop of the eight-wave build 960-1120.
constexpr int DMA_WM = 4, DMA_WN = 2;

static int g_gemm_build = 1; // measurement knob (gemm_set_build)

// The tiles gemm_pipe_kernel is built for: (32 ti) x (32 tj) with st slabs in LDS, what one slab of
// it takes when weights come from memory (us, every CU busy) and what a tile costs beside its slabs.
// A slab's time is its bytes (A and W rows of 128 bytes) at 55 to 66 GB/s: a CU has at most 32 KB of
// loads in flight, in order, and memory answers after 600 ns, 55 GB/s (350 ns from the last-level
// cache, 190 ns from L2: 93 and 173 GB/s; part of A comes from there). So a tile's bytes per FLOP decide, and they fall with its
// size, until there are fewer tiles than CUs. (The last two were timed with a load every four MFMAs; every five
// takes 0 to 4 % off a launch of theirs.)
struct PipeShape { int ti, tj, st; float slab_us, fix_us; };
constexpr PipeShape kPipe[] = {
    {2, 2, 4, 0.30f, 4.0f}, {2, 3, 4, 0.31f, 4.0f}, {4, 2, 4, 0.385f, 4.5f}, {4, 3, 4, 0.446f, 4.5f}, {4, 4, 4, 0.54f, 5.0f},
    {4, 5, 4, 0.66f, 5.0f}, {4, 6, 3, 0.74f, 5.5f}, {6, 6, 3, 0.83f, 6.0f}, {8, 5, 3, 0.88f, 6.5f},
};
constexpr int kPipeShapes = (int)(sizeof(kPipe) / sizeof(kPipe[0]));
constexpr int kRingShape = -1;
// The same for the 256-tiles of gemm_ring_kernel; a last round split along k also pays for its
// partial tiles' way through memory and for the merge.
constexpr float kRingSlabUs = 1.28f, kRingFixUs = 8.0f, kRingSplitUs = 28.0f;

// A ragged k (RAG) is built for every tile too: its products have the rows and columns of the others (a
// hidden width of 2568 is 40 slabs and an eighth), and the estimates hold for them.
template <bool F16, typename TC, int I, bool RAG>
static const void* pipe_entry() {
    return reinterpret_cast<const void*>(&gemm_pipe_kernel<F16, TC, kPipe[I].ti, kPipe[I].tj, kPipe[I].st, RAG>);
}

template <bool F16, typename TC, bool RAG>
static hipError_t launch_pipe(GemmArgs g, hipStream_t stream) {
    const PipeShape& p = kPipe[g.shape];
    g.tiles_n = (g.n + 32 * p.tj - 1) / (32 * p.tj);
    const int64_t nwg = (int64_t)((g.m + 32 * p.ti - 1) / (32 * p.ti)) * g.tiles_n * g.groups;
    if (nwg <= 0 || nwg > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)nwg), block(256);
    const size_t lds = pipe_lds_bytes(p.ti, p.tj, p.st);
    switch (g.shape) {
#define ZD_PIPE(I) \
    case I: gemm_pipe_kernel<F16, TC, kPipe[I].ti, kPipe[I].tj, kPipe[I].st, RAG><<<grid, block, lds, stream>>>(g); break;
    ZD_PIPE(0) ZD_PIPE(1) ZD_PIPE(2) ZD_PIPE(3) ZD_PIPE(4) ZD_PIPE(5) ZD_PIPE(6) ZD_PIPE(7) ZD_PIPE(8)
#undef ZD_PIPE
    default: return hipErrorInvalidValue;
    }
    static_assert(kPipeShapes == 9, "one case per shape");
    return hipGetLastError();
}

template <bool F16, typename TC>
static hipError_t launch_one(const GemmArgs& g0, hipStream_t stream) {
    GemmArgs g = g0;
    if (g.k % BK != 0) return launch_pipe<F16, TC, true>(g, stream);
    if (g.shape != kRingShape) return launch_pipe<F16, TC, false>(g, stream);
    g.tiles_n = (g.n + BN - 1) / BN;
    const int64_t nwg = (int64_t)((g.m + BM - 1) / BM) * g.tiles_n * g.groups;
    if (nwg <= 0 || nwg > 0x7fffffff) return hipErrorInvalidValue;
    if (g_gemm_build != 1) {
        gemm_dma_kernel<F16, TC, DMA_WM, DMA_WN><<<dim3((unsigned)nwg), dim3(DMA_WM * DMA_WN * 64), kDmaLdsBytes, stream>>>(g);
        return hipGetLastError();
    }
    // one launch: (splits > 1) the tiles of the last round in parts, the whole tiles behind them; then the merge
    const int tail = g0.splits > 1 ? g0.tile_base : 0; // the planner leaves the tail size in tile_base
    if (tail < 0 || tail > nwg || g0.splits > kMaxKSplits || (tail > 0 && g0.part == nullptr)) return hipErrorInvalidValue;
    const int64_t whole = nwg - tail;
    g.tile_base = (int32_t)whole;
    g.splits = tail > 0 ? g0.splits : 1;
    g.part_wgs = tail > 0 ? (int32_t)(((int64_t)tail * g0.splits + 7) & ~(int64_t)7) : 0;
    if (whole + g.part_wgs > 0x7fffffff) return hipErrorInvalidValue;
    gemm_ring_kernel<F16, TC><<<dim3((unsigned)(whole + g.part_wgs)), dim3(256), kRingLdsBytes, stream>>>(g);
    if (tail > 0) {
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        gemm_merge_kernel<F16, TC><<<dim3((unsigned)tail * 16u), dim3(256), 0, stream>>>(g);
    }
    return hipGetLastError();
}

template <bool F16, typename TC, int I>
static hipError_t raise_pipe() {
    const int lds = (int)pipe_lds_bytes(kPipe[I].ti, kPipe[I].tj, kPipe[I].st);
    hipError_t e = hipFuncSetAttribute(pipe_entry<F16, TC, I, false>(), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e == hipSuccess) e = hipFuncSetAttribute(pipe_entry<F16, TC, I, true>(), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if constexpr (I + 1 < kPipeShapes) return e == hipSuccess ? raise_pipe<F16, TC, I + 1>() : e;
    return e;
}
template <bool F16, typename TC>
static hipError_t raise_lds() {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_dma_kernel<F16, TC, DMA_WM, DMA_WN>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDmaLdsBytes);
    if (e != hipSuccess) return e;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_ring_kernel<F16, TC>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)kRingLdsBytes);
    return e == hipSuccess ? raise_pipe<F16, TC, 0>() : e;
}

} // namespace gemm

int gemm_tile_rows() { return gemm::BM; }
int gemm_tile_cols() { return gemm::BN; }

// Only the four-wave build splits (whole slabs, enough tiles for 256-tiles).
// A last round that fills at most half the CUs is cut along k so that it fills them: the round
// then costs 1 / splits of a tile's time plus the partial tiles' trip through memory (256 KB
// per part, which is why the number of parts is kept small and a fuller round is left whole).
void gemm_tail_plan(const GemmArgs& g, int cus, int* tail_tiles, int* splits) {
    *tail_tiles = 0;
    *splits = 1;
    if (gemm::g_gemm_build != 1 || g.k % gemm::BK != 0 || cus <= 0) return;
    const int64_t tiles = (int64_t)((g.m + 255) / 256) * ((g.n + 255) / 256) * g.groups;
    if (tiles < 160 || tiles > 0x7fffffff) return;
    const int tail = (int)(tiles % cus);
    if (tail == 0 || tail * 2 > cus) return;
    int s = cus / tail;
    if (s > gemm::kMaxKSplits) s = gemm::kMaxKSplits;
    const int nslab = g.k / gemm::BK;
    if (s > nslab / 4) s = nslab / 4; // at least four slabs per part
    if (s < 2) return;
    *tail_tiles = tail;
    *splits = s;
}
size_t gemm_part_bytes(int tail_tiles, int splits) {
    return (size_t)tail_tiles * splits * gemm::BM * gemm::BN * sizeof(float);
}

// The tile whose estimate (rounds of tiles over the CUs, each its slabs and its fixed part) is the
// smallest. The estimates are within 10 % of what was measured for 77 to 4608 rows, 3072 and 3840
// columns once and three times, k 3072 to 12288, and put the measured best first or within 3 % of it
// (us, cold weights, bf16; the 128-tiles with one slab in flight that did all of these before, or the
// 256-tiles, in brackets): 512 x 3072 x 3 x 3072 128 x 160 tiles 40 (51), 512 x 3072 x 3072 64 x 96
// 20 (47), 1024 x 3072 x 3 x 3072 256 x 160 56 (86), 1024 x 3072 x 3072 128 x 96 28 (47), 77 x 3072 x
// 3 x 3072 64 x 96 20 (48), 2816 x 12288 x 3072 192 x 192 164 (238), 2304 x 3840 x 3840 192 x 192 61 (95).
int gemm_shape(const GemmArgs& g, int cus) {
    using namespace gemm;
    if (g_gemm_build == 2) return kGemmUnstaged;
    if (cus <= 0) return 0;
    auto count = [&](int rows, int cols) { return (int64_t)((g.m + rows - 1) / rows) * ((g.n + cols - 1) / cols) * g.groups; };
    const int nslab = (g.k + BK - 1) / BK;
    const int64_t tiles256 = count(BM, BN);
    int best = kRingShape;
    float best_us = INFINITY;
    if (g.k % BK == 0) {
        if (g_gemm_build != 1 && tiles256 >= 160) return kRingShape;
        int tail = 0, splits = 1;
        gemm_tail_plan(g, cus, &tail, &splits);
        const float round_us = (float)nslab * kRingSlabUs + kRingFixUs;
        best_us = splits > 1 ? (float)(tiles256 / cus) * round_us + (float)((nslab + splits - 1) / splits) * kRingSlabUs + kRingSplitUs
                             : (float)((tiles256 + cus - 1) / cus) * round_us;
    }
    for (int i = 0; i < kPipeShapes; i++) {
        const int64_t rounds = (count(32 * kPipe[i].ti, 32 * kPipe[i].tj) + cus - 1) / cus;
        const float us = (float)rounds * ((float)nslab * kPipe[i].slab_us + kPipe[i].fix_us);
        if (us < best_us) { best_us = us; best = i; }
    }
    return best;
}
void gemm_shape_tile(int shape, int* rows, int* cols) {
    *rows = shape == kGemmUnstaged ? 64 : shape < 0 ? gemm::BM : 32 * gemm::kPipe[shape].ti;
    *cols = shape == kGemmUnstaged ? 64 : shape < 0 ? gemm::BN : 32 * gemm::kPipe[shape].tj;
}

int32_t gemm_launch_rows(int32_t rows, int64_t ld, int32_t k) {
    const uint64_t most = kGemmSpanLimit / 2; // elements
    if ((uint64_t)k > most) return 0;
    if (rows == 1 || (uint64_t)(rows - 1) * (uint64_t)ld + (uint64_t)k <= most) return rows;
    const uint64_t fit = (most - (uint64_t)k) / (uint64_t)ld + 1; // < rows
    return (int32_t)(fit >= 256 ? fit & ~uint64_t{255} : fit);
}

// f32 activations are rounded to the weight's type once, ahead of the product.
size_t gemm_round_bytes(const GemmArgs& g, int a_dtype) { return a_dtype == kF32 ? (size_t)g.m * (size_t)g.k * 2 : 0; }

// Products of less than a 256-tile either way, or of a ragged k, must not fail for want of that copy's
// room; larger ones report the failed allocation rather than run several times slower.
bool gemm_rounds_in_place(const GemmArgs& g) { return g.k % gemm::BK != 0 || g.m < gemm::BM || g.n < gemm::BN; }

hipError_t launch_gemm(const GemmArgs& g0, int a_dtype, int w_dtype, int c_dtype, hipStream_t stream) {
    using namespace gemm;
    typedef unsigned short h16; // a 16-bit operand in the compute type (bf16 or f16 per the weight)
    GemmArgs g = g0;
    if (a_dtype != kF32 && a_dtype != w_dtype) return hipErrorInvalidValue;
    if (g.shape == kGemmUnstaged) {
#define ZD_UNSTAGED(TA) \
    (w_dtype == kBF16 ? (c_dtype == kF32 ? launch_unstaged<TA, false, float>(g, stream) : launch_unstaged<TA, false, h16>(g, stream)) \
                      : (c_dtype == kF32 ? launch_unstaged<TA, true, float>(g, stream) : launch_unstaged<TA, true, h16>(g, stream)))
        return a_dtype == kF32 ? ZD_UNSTAGED(float) : ZD_UNSTAGED(h16);
#undef ZD_UNSTAGED
    }
    if (a_dtype == kF32) {
        if (g.a16 == nullptr) return hipErrorInvalidValue;
        const dim3 grid((unsigned)g.m, (unsigned)((g.k + 4095) / 4096));
        if (w_dtype == kF16)
            gemm_round_kernel<true><<<grid, dim3(256), 0, stream>>>(static_cast<const float*>(g.a), g.lda, static_cast<h16*>(g.a16), g.m, g.k);
        else
            gemm_round_kernel<false><<<grid, dim3(256), 0, stream>>>(static_cast<const float*>(g.a), g.lda, static_cast<h16*>(g.a16), g.m, g.k);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        g.a = g.a16;
        g.lda = g.k;
    }
    if (w_dtype == kBF16) {
        if (c_dtype == kF32) return launch_one<false, float>(g, stream);
        if (c_dtype == kBF16) return launch_one<false, h16>(g, stream);
    } else if (w_dtype == kF16) {
        if (c_dtype == kF32) return launch_one<true, float>(g, stream);
        if (c_dtype == kF16) return launch_one<true, h16>(g, stream);
    }
    return hipErrorInvalidValue;
}

void gemm_set_build(int build) { gemm::g_gemm_build = build == 1 || build == 2 ? build : 0; }

hipError_t gemm_setup() {
    using namespace gemm;
    typedef unsigned short h16;
    hipError_t e;
    if ((e = raise_lds<false, float>()) != hipSuccess) return e;
    if ((e = raise_lds<false, h16>()) != hipSuccess) return e;
    if ((e = raise_lds<true, float>()) != hipSuccess) return e;
    if ((e = raise_lds<true, h16>()) != hipSuccess) return e;
    return hipSuccess;
}

} // namespace zdraw
