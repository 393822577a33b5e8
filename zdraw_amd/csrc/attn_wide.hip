// gfx950 attention for one wide head (heads = 1, head_dim = 512): the VAE
// mid-block shape, 16384 tokens at 1024 px.
//
// What it replaces in the reference: attention_wide_mma
// (metal/mattn_shader.zig:225-390), reached through zdraw_metal_run_attention
// with kernel = wide (metal/mattn.zig:152-173, 261-275). The contract is the
// reference's: f32 token-major q, k, v, out [tokens][512], tokens % 64 == 0, no
// mask, not causal; anything else is refused on the host.
//
// Shape of the computation on this machine:
//   * a pre-pass rounds Q (times log2(e)/sqrt(512)), K and V to bf16 once, so the
//     main kernel moves half the bytes and fetches blocks straight into LDS;
//   * a workgroup is four waves, one per SIMD (512 registers each), and owns 128 query rows
//     and ALL 512 output dims over a range of the keys. A wave forms the scores of 32 of the rows
//     (its Q fragments are half the ordinary registers), runs their softmax, and hands the exponentiated
//     block (2 KB) to its partner through LDS: the two waves of a pair own 64 rows together, each over one
//     half of the dims, so a V fragment read from LDS feeds four MFMAs instead of two (with all 512 dims of
//     its own rows a wave read 32 KB of V a block, now 16). O^T is 64 tiles of 16 x 16, the whole accumulation
//     file. No score is formed twice;
//   * all MFMAs are v_mfma_f32_16x16x32: half the accumulator bytes per FLOP through the register file of the
//     32 x 32 form, and in its transposed scores (S^T = K Q^T) a lane holds the eight keys of one query that the
//     product's B operand wants (16 t + 4 (lane / 16) .. + 3, t = 0, 1): no lane exchange. They are assembly
//     statements with the accumulator tied to the result, which keeps the 256 accumulation
//     registers where they are (given the builtin the compiler moves such tuples about and
//     spills); nothing else may touch those registers between such an MFMA and the wait that
//     ends the step (zdraw_amd.build.tied_mfma_hazards checks the compiled code);
//   * a query tile's keys are split over up to eight workgroups (two at 16384 tokens: 256
//     workgroups, one per CU; wide_splits), each leaving its unnormalised O and its (reference
//     point, row sum) in scratch; wide_merge_kernel combines the ranges in range order;
//   * per 32-key block a wave forms S^T (64 MFMAs) and adds V^T P^T to O^T (64 MFMAs), with the exponentials of
//     the next block between the latter;
//   * K blocks and V blocks (32 KB) cycle through two LDS slots each, P through two of 8 KB,
//     filled by buffer_load ... lds in a swizzled 256-byte-row layout. A wave's 16 loads per block go one per
//     four MFMAs of the product, into what its barrier has just freed: the CU's address unit takes 16 cycles per
//     load, and a burst from four waves at once holds them at the memory queue;
//   * one barrier per block, placed after the 56th of the 64 S MFMAs, when the last K
//     fragments are in registers: P and the V fragments of the product are read under the rest;
//   * fixed block order and fixed summation order: bit-identical from run to run.
#include "attn_device.hpp"

#include <cmath>
#include <utility>

namespace zdraw {

namespace wide {

constexpr int WD = 512;           // head_dim
constexpr int SL = 128;           // dims per LDS tile ("slice")
constexpr int NSL = WD / SL;
constexpr int KB = 32;            // keys per block
constexpr int NW = 4;
constexpr int NT = NW * 64;
constexpr int BQ = 128;           // query rows per workgroup
constexpr int TILE_BYTES = KB * SL * 2;        // 8 KB
constexpr int K_SLOT = NSL * TILE_BYTES;       // a K block: 32 KB
constexpr int V_SLOT = NSL * TILE_BYTES;       // a V block: 32 KB
constexpr int NSK = 2;                         // slots of the K ring
constexpr int NSV = 2;                         // slots of the V ring
constexpr int V_RING = NSK * K_SLOT;
constexpr int P_RING = V_RING + NSV * V_SLOT;  // two slots of the exponentiated blocks
constexpr int P_SLOT = NW * 2 * 1024;          // 2 KB a wave
constexpr size_t kLdsBytes = (size_t)P_RING + 2 * P_SLOT + 16384; // 160 KB: the last 16 KB hold query rows only
constexpr float kTau = 8.0f;      // log2 headroom of the lazy softmax maximum (safe::form_again)
constexpr float kRowSumLimit = 0x1p90f; // a row sum past this has its tile's range formed again: a P beyond 2^90 may be on its way to overflow
constexpr int RA = 6;             // K fragments read ahead of their MFMA
constexpr int VA = 3;             // V fragment pairs read ahead
constexpr int kMaxSplits = 8;     // key ranges per query tile

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// f32 -> bf16 with a scale, 8 elements per thread; blockIdx.y selects the operand.
__global__ void __launch_bounds__(256) wide_round_kernel(const WidePrepArgs p) {
    const int op = (int)blockIdx.y;
    // the launch that precedes every attention launch also clears its redo flags
    if (op == 0 && blockIdx.x == 0)
        for (int i = threadIdx.x; i < p.redo_tiles; i += blockDim.x) p.redo[i] = 0;
    const float* src = op == 0 ? p.q : op == 1 ? p.k : p.v;
    bf16_t* dst = reinterpret_cast<bf16_t*>(op == 0 ? p.qo : op == 1 ? p.ko : p.vo);
    const float scale = op == 0 ? p.q_scale : 1.0f;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < p.chunks; i += stride) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(src + 8 * i);
        const f32x4 b = *reinterpret_cast<const f32x4*>(src + 8 * i + 4);
        const float x[8] = {a[0] * scale, a[1] * scale, a[2] * scale, a[3] * scale,
                            b[0] * scale, b[1] * scale, b[2] * scale, b[3] * scale};
        // (through the L2: the attention launch starts 0.8 us sooner behind this one, calls of 6208 tokens 111.8 -> 110.9 us,
        // of 16384 430.4 -> 429.6)
        store_through(dst + 8 * i, pack_bf16x8(x));
    }
}

template <int N> using IC = std::integral_constant<int, N>;
// f(IC<0>), f(IC<1>), ..: a loop whose counter is a constant to the front end. (A phase of 64 MFMAs is past the
// size up to which `#pragma unroll` works, and a phase that stays a loop spills.)
template <typename F, int... I>
__device__ __forceinline__ void unrolled_seq(F&& f, std::integer_sequence<int, I...>) { (f(IC<I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void unrolled(F&& f) { unrolled_seq(f, std::make_integer_sequence<int, N>{}); }

__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int j = 0; j < 16; j++) z[j] = 0.f;
    return z;
}

// O^T += A B on the accumulation file, the accumulator tied to the result. The compiler adds no
// hazard waits around assembly: consecutive MFMAs on one accumulator are 64 MFMAs apart in the
// product's order, and acc_drain() ends every step in the basic block of its last MFMA, before
// anything else (the epilogue, a copy the compiler placed at a join) can read the
// accumulation registers.
__device__ __forceinline__ void mfma_acc(f32x4& c, const bf16x8& x, const bf16x8& y) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
}
// The same for the scores, in ordinary registers (the accumulation file is full): `FIRST` starts
// the chain from zero. A tile's MFMAs are four apart; in the key loop the scores are first read by other
// instructions behind the third product MFMA after the chains' last, ahead of it through a wait whose operands they are. The
// hardware needs eight wait states there, and zdraw_amd.build.early_mfma_result_uses holds the compiled code to them.
template <bool FIRST>
__device__ __forceinline__ void mfma_score(f32x4& c, const bf16x8& x, const bf16x8& y) {
    if constexpr (FIRST) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(x), "v"(y));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(x), "v"(y));
}
__device__ __forceinline__ void mfma_score_from(f32x4& c, const bf16x8& x, const bf16x8& y, const f32x4& start) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %3" : "=&v"(c) : "v"(x), "v"(y), "v"(start));
}
// Largest value / sum over the pair of lane rows (16 lanes) 2 i, 2 i + 1.
__device__ __forceinline__ float row_pair_max(float x) {
    const u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float row_pair_sum(float x) {
    const u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// c = 0 as an MFMA of zeros: the tuple is defined whole, never element by element. (An MFMA may
// not read a register in the two issue slots after an ordinary vector instruction wrote it; the
// compiler keeps that distance for its own MFMAs, not around assembly: z may just have been set.)
__device__ __forceinline__ void mfma_zero(f32x4& c, const bf16x8& z) {
    asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %1, 0" : "=&a"(c) : "v"(z));
}
__device__ __forceinline__ void acc_drain() {
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
}

// ---------------------------------------------------------------------------------------------
// The rows of a workgroup of attn_wide_kernel one of whose scores lies some 90 (log2) above its row's first block,
// over the same key range, formed again with a lazy running maximum: one half of the 512 output dims at a time (the scores
// of the range are formed for each), so that O^T takes 128 accumulation registers per wave and the compiler has
// room to rescale it in place when a reference point moves. K blocks (32 KB) and V half-blocks (16 KB) cycle through three
// LDS slots each. It runs behind the kernel's own epilogue, by the workgroup that found the row sum, where nothing of the
// fast path is live any more: a kernel of its own behind every call, which this was, costs ordinary data its launch.
// Calls, us, as a launch of its own -> here: 256 tokens 38.5 -> 37.2, 1024 43.7 -> 42.4, 2560 59.0 -> 57.7, 6208 111.3 -> 109.9,
// 16384 438.1 -> 435.6. With every row formed again: 256 59.6 -> 57.9, 512 68.9 -> 60.0, 1024 89 -> 65 (two workgroups take
// a half each, wide_halves), 6208 330 -> 252, 16384 1224 -> 1134 (a launch of its own went over all keys, this over the range that
// needs it; where the keys are one range and the tiles more than 64, as with 32768 tokens, a lone such tile takes twice as long).
namespace safe {
constexpr int HALF = WD / 2;      // output dims per workgroup
constexpr int V_SLOT = (NSL / 2) * TILE_BYTES; // half the dims of a V block: 16 KB
constexpr int NS = 3;                          // slots per ring
constexpr int V_RING = NS * K_SLOT;
static_assert((size_t)NS * (K_SLOT + V_SLOT) <= wide::kLdsBytes, "144 of the kernel's 160 KB");

// Output dims HALF dh .. of query tile `tile` over key blocks blk0 .. blk0 + nblk - 1, written as key range `part` of nsp
// (nsp 1: the result). Every wave of the workgroup calls it, behind a barrier that ends all use of the LDS.
__device__ __forceinline__ void form_again(const WideArgs& a, unsigned char* smem, int wave, int tile, int part, int nsp, int blk0, int nblk, int dh) {
    int lane; // (formed here: kept from the kernel's start it would cost the key loop a register)
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    const int l32 = lane & 31;
    const int h = lane >> 5;
    blk0 = __builtin_amdgcn_readfirstlane(blk0); // (uniform, and formed on the scalar unit from here on)
    nblk = __builtin_amdgcn_readfirstlane(nblk);
    const int q0 = tile * BQ + 32 * wave; // this wave's query rows

    const unsigned lds0 = lds_address(smem);

    // ---- Q fragments (B operand of S^T = K Q^T): query q0 + l32, dims 16 kk + 8 h .. +7
    bf16x8 qf[32];
    {
        // rows past the end read the last row and are never stored
        const bf16_t* qp = reinterpret_cast<const bf16_t*>(a.q) + (int64_t)min(q0 + l32, a.tokens - 1) * WD + 8 * h;
#pragma unroll
        for (int kk = 0; kk < 32; kk++) qf[kk] = *reinterpret_cast<const bf16x8*>(qp + 16 * kk);
    }

    // ---- block fetch. K: wave w fills tile w (dims 128 w .. +127) of the block, four rows per
    // instruction. V: wave w fills rows 16 (w >> 1) .. +15 of tile (w & 1) of this workgroup's
    // half. The lane that fills chunk position p of row r fetches the chunk the swizzle places
    // there: K chunk c of row r sits at c ^ (r & 15), V chunk c at c ^ ((r & 3) << 2).
    const unsigned span = (unsigned)a.tokens * (unsigned)(WD * 2);
    const u32x4 k_rsrc = make_rsrc_words(a.k, span);
    const u32x4 v_rsrc = make_rsrc_words(a.v, span);
    unsigned fk_off[4], fv_off[4]; // K rows 4 j + 16 take the same chunks 16 rows further on
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = 4 * j + (lane >> 4);
        const unsigned kc = (unsigned)((lane & 15) ^ (row & 15));
        fk_off[j] = (unsigned)row * (WD * 2) + (unsigned)wave * (SL * 2) + kc * 16u;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = 16 * (wave >> 1) + 4 * j + (lane >> 4);
        const unsigned vc = (unsigned)((lane & 15) ^ ((row & 3) << 2));
        fv_off[j] = (unsigned)row * (WD * 2) + (unsigned)(2 * dh + (wave & 1)) * (SL * 2) + vc * 16u;
    }
    const unsigned fetch_k_lds = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * TILE_BYTES);
    const unsigned fetch_v_lds = __builtin_amdgcn_readfirstlane(lds0 + V_RING + (unsigned)(wave & 1) * TILE_BYTES + (unsigned)(16 * (wave >> 1)) * (SL * 2));
    // the i-th (i < 12) load of the group that brings K block kb into K slot ks and V block vb into V slot vs
    auto fetch_one = [&](int kb, int ks, int vb, int vs, int i) __attribute__((always_inline)) {
        if (i < 8) {
            const unsigned uo = (unsigned)(blk0 + (kb < nblk ? kb : nblk - 1)) * (unsigned)(KB * WD * 2) + (unsigned)(i >> 2) * (16 * WD * 2);
            load_to_lds_16(k_rsrc, fetch_k_lds + (unsigned)ks * K_SLOT + (unsigned)(4 * i) * (SL * 2), fk_off[i & 3], uo);
        } else {
            const unsigned uo = (unsigned)(blk0 + (vb < nblk ? vb : nblk - 1)) * (unsigned)(KB * WD * 2);
            load_to_lds_16(v_rsrc, fetch_v_lds + (unsigned)vs * V_SLOT + (unsigned)(4 * (i - 8)) * (SL * 2), fv_off[i - 8], uo);
        }
    };

    // ---- fragment addresses in slot 0 (a tile and a slot add constants)
    const int tr_row = (lane & 15) >> 2;
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    // (pointers, so that the constant parts of an address go into the instruction's offset field)
    typedef __attribute__((address_space(3))) unsigned char* lds_byte_t;
    typedef const __attribute__((address_space(3))) bf16x8* lds_bf16x8_t;
    typedef __attribute__((address_space(3))) s16x4* lds_s16x4_t;
    const lds_byte_t lds_base = (lds_byte_t)smem;
    lds_byte_t kfo[8], vfo[4];
#pragma unroll
    for (int kk = 0; kk < 8; kk++) kfo[kk] = lds_base + ((l32 * SL + (((2 * kk + h) ^ (l32 & 15)) * 8)) * 2);
#pragma unroll
    for (int blk = 0; blk < 4; blk++)
        vfo[blk] = lds_base + V_RING + (((4 * h + tr_row) * SL + ((blk ^ tr_row) * 32) + tr_col) * 2);
    auto k_read = [&](int slot, int kk) __attribute__((always_inline)) {
        return *(lds_bf16x8_t)(kfo[kk & 7] + (slot * K_SLOT + (kk >> 3) * TILE_BYTES));
    };

    f32x16 oacc[8]; // O^T: lane = query l32, dims 256 dh + 32 blk + 8 i + 4 h + j
#pragma unroll
    for (int blk = 0; blk < 8; blk++)
#pragma unroll
        for (int j = 0; j < 16; j++) oacc[blk][j] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    // ---- prologue: K(0..2), V(0..1) in; S(0); then K(3) requested
#pragma unroll
    for (int i = 0; i < 12; i++) fetch_one(0, 0, 0, 0, i);
#pragma unroll
    for (int i = 0; i < 12; i++) fetch_one(1, 1, 1, 1, i);
#pragma unroll
    for (int i = 0; i < 8; i++) fetch_one(2, 2, 0, 0, i);
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
    __syncthreads();
    f32x16 sv; // scores of the block the next step exponentiates: lane = query l32, element 4 i + j = key 8 i + 4 h + j
    {
        f32x16 s = zero16();
#pragma unroll
        for (int kk = 0; kk < 32; kk++) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k_read(0, kk), qf[kk], s, 0, 0, 0);
        sv = s;
    }
    __syncthreads(); // K(0) has no reader left
#pragma unroll
    for (int i = 0; i < 4; i++) fetch_one(3, 0, 0, 0, i); // the first step sends the other eight of this group
    bf16x8 kf[RA + 1]; // ring of fragments in flight
#pragma unroll
    for (int kk = 0; kk < RA; kk++) kf[kk] = k_read(1, kk);

    // The running maximum moved (rare after the first blocks): O^T *= alpha, in place in the
    // accumulation file. Written out by hand: left to the compiler, the two versions of O that
    // meet after the branch cost more registers than there are.
    auto rescale = [&](float alpha) __attribute__((always_inline)) {
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); // MFMA results are read next
#pragma unroll
        for (int blk = 0; blk < 8; blk++)
#pragma unroll
            for (int j = 0; j < 16; j++) {
                float x = oacc[blk][j], t;
                asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\ts_nop 0\n\tv_accvgpr_write_b32 %0, %1" : "+a"(x), "=&v"(t) : "v"(alpha));
                oacc[blk][j] = x;
            }
        asm volatile("s_nop 7" ::: "memory"); // and feed the next MFMAs
    };

    // One step b with K(b+1) in K slot KS = (b + 1) % 3 and V(b) in V slot VS = b % 3:
    //   S phase: the 32 MFMAs of S(b+1) = K(b+1) Q^T with the softmax of block b in their shadow;
    //   barrier: K(b+2) and V(b) have landed (requested two steps ago), K(b+1) and V(b-1) have no
    //            reader left;
    //   PV phase: O += V(b)^T P(b)^T (16 MFMAs), the first fragments of K(b+2) read under them.
    // The 12 loads that bring K(b+4) and V(b+2) into the two freed slots follow the barrier, 4
    // under the PV phase and 8 under the next S phase.
    auto step = [&](auto ks_c, auto vs_c, int b) __attribute__((always_inline)) {
        constexpr int KS = decltype(ks_c)::value;       // slot of K(b+1); K(b+2) is in (KS + 1) % 3
        constexpr int VS = decltype(vs_c)::value;       // slot of V(b); V(b-1) was in (VS + 2) % 3
        constexpr int KN = (KS + 1) % 3;
        f32x16 s;
        float mloc = 0.f, mc = 0.f, alpha = 1.f, psum = 0.f, e_even = 0.f;
        bool up = false;
        unsigned pc[8];
        s16x4 vlo[VA + 1], vhi[VA + 1];
        // idx < 16: tile idx >> 3 of the half, key half (idx >> 2) & 1, 32-dim block idx & 3
        auto v_read = [&](int idx) __attribute__((always_inline)) {
            const lds_byte_t va = vfo[idx & 3] + (VS * V_SLOT + (idx >> 3) * TILE_BYTES + (16 * ((idx >> 2) & 1)) * (SL * 2));
            vlo[idx % (VA + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)va);
            vhi[idx % (VA + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(va + 8 * (SL * 2)));
        };
        __builtin_amdgcn_sched_barrier(0);
        unrolled<32>([&](auto t_c) __attribute__((always_inline)) {
            constexpr int t = decltype(t_c)::value;
            // the previous barrier's group: K(b+3) into the slot K(b) left, V(b+1) into V(b-2)'s
            if constexpr ((t & 3) == 0) fetch_one(b + 3, (KS + 2) % 3, b + 1, (VS + 1) % 3, 4 + (t >> 2));
            if constexpr (t + RA < 32) kf[(t + RA) % (RA + 1)] = k_read(KS, t + RA);
            if constexpr (t >= 28 && t - 28 < VA) v_read(t - 28);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[t % (RA + 1)], qf[t], t == 0 ? zero16() : s, 0, 0, 0);
            // softmax of block b in the exp2 domain (the scale rides on Q) with a lazy maximum: the
            // reference point moves only when this block's maximum exceeds it by more than kTau
            if constexpr (t == 0) {
                mloc = fmaxf(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])), fmaxf(fmaxf(sv[4], sv[5]), fmaxf(sv[6], sv[7])));
            } else if constexpr (t == 1) {
                mloc = fmaxf(mloc, fmaxf(fmaxf(fmaxf(sv[8], sv[9]), fmaxf(sv[10], sv[11])), fmaxf(fmaxf(sv[12], sv[13]), fmaxf(sv[14], sv[15]))));
                const float mlc = pair_max(mloc);
                up = mlc > m_run + kTau;
                const float m_new = up ? mlc : m_run;
                mc = (m_new == -INFINITY) ? 0.f : m_new;
                alpha = __builtin_amdgcn_exp2f(m_run - mc);
                m_run = m_new;
            } else if constexpr (t >= 3 && t < 19) {
                constexpr int e = t - 3; // one exponential per MFMA
                const float x = __builtin_amdgcn_exp2f(sv[e] - mc);
                psum += x;
                if constexpr (e & 1) {
                    f32x2 pp = {e_even, x};
                    pc[e >> 1] = __builtin_bit_cast(unsigned, __builtin_convertvector(pp, bf16x2));
                } else {
                    e_even = x;
                }
            } else if constexpr (t == 19) {
                l_run = l_run * alpha + psum;
                if (__any(up)) rescale(alpha);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (t == 27) {
                // every fragment of K(b+1) is in registers; K(b+2), V(b) have landed: everything but
                // the 12 loads sent since the last barrier
                __builtin_amdgcn_s_waitcnt(0x007C); // vmcnt(12) lgkmcnt(0)
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        const bf16x8 p0 = __builtin_bit_cast(bf16x8, u32x4{pc[0], pc[1], pc[2], pc[3]});
        const bf16x8 p1 = __builtin_bit_cast(bf16x8, u32x4{pc[4], pc[5], pc[6], pc[7]});
        unrolled<16>([&](auto i_c) __attribute__((always_inline)) {
            constexpr int idx = decltype(i_c)::value;
            if constexpr ((idx & 3) == 1) fetch_one(b + 4, KS, b + 2, (VS + 2) % 3, idx >> 2);
            if constexpr (idx + VA < 16) v_read(idx + VA);
            if constexpr (idx >= 16 - RA) kf[(idx - (16 - RA)) % (RA + 1)] = k_read(KN, idx - (16 - RA));
            const bf16x8 vf = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(vlo[idx % (VA + 1)], vhi[idx % (VA + 1)], 0, 1, 2, 3, 4, 5, 6, 7));
            constexpr int ob = (idx >> 3) * 4 + (idx & 3);
            oacc[ob] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, ((idx >> 2) & 1) ? p1 : p0, oacc[ob], 0, 0, 0);
            if constexpr (idx == 4) sv = s; // the S MFMAs have drained by now
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    int b = 0;
    for (; b + 2 < nblk; b += 3) {
        step(IC<1>{}, IC<0>{}, b);
        step(IC<2>{}, IC<1>{}, b + 1);
        step(IC<0>{}, IC<2>{}, b + 2);
    }
    if (b < nblk) step(IC<1>{}, IC<0>{}, b);
    if (b + 1 < nblk) step(IC<2>{}, IC<1>{}, b + 1);
    __builtin_amdgcn_s_waitcnt(0x0F70); // no direct load may outlive the workgroup's LDS

    // ---- epilogue: O = O^T / l, or the range's share as it stands
    const float l_tot = pair_sum(l_run);
    if (q0 + l32 >= a.tokens) return; // (the lane joins the next half's barrier all the same: this is inlined)
    const float scale = nsp > 1 ? 1.0f : l_tot > 0.f ? 1.0f / l_tot : 0.f;
    float* op = (nsp > 1 ? a.part_o + ((int64_t)part * a.tokens + q0 + l32) * WD : a.o + (int64_t)(q0 + l32) * WD) + HALF * dh;
    if (nsp > 1 && dh == 0 && h == 0) *reinterpret_cast<f32x2*>(a.part_ml + ((int64_t)part * a.tokens + q0 + l32) * 2) = f32x2{m_run, l_tot};
#pragma unroll
    for (int blk = 0; blk < 8; blk++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = oacc[blk][4 * i + j] * scale;
            *reinterpret_cast<f32x4*>(op + 32 * blk + 8 * i + 4 * h) = v;
        }
}

} // namespace safe

__global__ void __launch_bounds__(NT, 1) attn_wide_kernel(const WideArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15;
    const int g4 = lane >> 4;
    // workgroup = (key range, query tile), range-major, and each XCD takes one contiguous run of
    // that order (workgroups go to the XCDs in turn): the workgroups behind one L2 walk the same
    // range, so a K/V block comes in once per XCD, not once per range as well. With a.halves, two workgroups in a row form
    // the same and each stores, and where need be forms again, one half of the output dims (wide_halves).
    const int nsp = a.splits > 1 ? a.splits : 1;
    const int tiles = ((int)gridDim.x >> a.halves) / nsp;
    const int xcd = (int)blockIdx.x & 7, xrem = (int)gridDim.x & 7;
    const int wg = ((int)blockIdx.x >> 3) + xcd * ((int)gridDim.x >> 3) + min(xcd, xrem);
    const int logical = wg >> a.halves;
    // (uniform, but the divisions run on the vector unit)
    const int part = __builtin_amdgcn_readfirstlane(logical / tiles);
    const int tile = logical - part * tiles;
    const int q0 = tile * BQ + 32 * wave;                           // the query rows whose scores this wave forms
    const int dh = wave & 1;                                       // the half of the output dims it owns, for its rows and its partner's
    const int per = __builtin_amdgcn_readfirstlane((a.tokens / KB + nsp - 1) / nsp);
    const int blk0 = part * per;                                    // this range's first key block
    const int nblk = max(min(a.tokens / KB - blk0, per), 1);        // and how many it has (the host gives every range some)

    const unsigned lds0 = lds_address(smem);

    // ---- block fetch. Wave w fills tile w (dims 128 w .. +127) of a K block and of a V block, four rows
    // (1 KB) an instruction, four instructions to a run whose LDS targets lie 1 KB apart: the run's first
    // sets M0, the others use the instruction's offset field, which also moves the address in memory; that
    // is taken off the lane's offset, and the descriptors start 3 KB below the operands so that it stays
    // positive. The lane that fills chunk position p of row r fetches the chunk the swizzle places there: K
    // chunk c of row r sits at c ^ (r & 15), V chunk c at c ^ ((r & 3) << 2) ^ (((r >> 2) & 1) << 1).
    constexpr unsigned kBias = 3 * 1024;
    const unsigned span = (unsigned)a.tokens * (unsigned)(WD * 2);
    const u32x4 k_rsrc = make_rsrc_words(static_cast<const unsigned char*>(a.k) - kBias, span + kBias);
    const u32x4 v_rsrc = make_rsrc_words(static_cast<const unsigned char*>(a.v) - kBias, span + kBias);
    unsigned fk_off[4], fv_off[2]; // the second run of a block takes the same chunks 16 rows further on (V: eight rows)
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int r = 4 * j + (lane >> 4);
        const unsigned at = (unsigned)r * (WD * 2) + (unsigned)wave * (SL * 2) + kBias - (unsigned)j * 1024u;
        fk_off[j] = at + (unsigned)((lane & 15) ^ r) * 16u;
        if (j < 2) fv_off[j] = at + (unsigned)((lane & 15) ^ ((lane >> 4) << 2) ^ ((j & 1) << 1)) * 16u;
    }
    const unsigned fetch_k_lds = __builtin_amdgcn_readfirstlane(lds0 + (unsigned)wave * TILE_BYTES);
    const unsigned fetch_v_lds = __builtin_amdgcn_readfirstlane(lds0 + V_RING + (unsigned)wave * TILE_BYTES);
    // byte offset of key block kb; positions past the range re-fetch its last block into a slot nobody reads any more
    auto block_at = [&](int kb) __attribute__((always_inline)) -> unsigned { return (unsigned)(blk0 + min(kb, nblk - 1)) * (unsigned)(KB * WD * 2); };
    // the i-th (i < 8) load of the K block at `at` into K slot ks / of the V block at `at` into V slot vs
    auto fetch_k = [&](unsigned at, int ks, auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if constexpr ((i & 3) == 0) lds_dma_base(fetch_k_lds + (unsigned)(ks * K_SLOT + (i >> 2) * (16 * SL * 2)));
        load_to_lds_16_at<1024 * (i & 3)>(k_rsrc, fk_off[i & 3], at + (unsigned)(i >> 2) * (16 * WD * 2));
    };
    auto fetch_v = [&](unsigned at, int vs, auto i_c) __attribute__((always_inline)) {
        constexpr int i = decltype(i_c)::value;
        if constexpr ((i & 3) == 0) lds_dma_base(fetch_v_lds + (unsigned)(vs * V_SLOT + (i >> 2) * (16 * SL * 2)));
        load_to_lds_16_at<1024 * (i & 3)>(v_rsrc, fv_off[i & 1], at + (unsigned)((i >> 2) * (16 * WD * 2) + ((i >> 1) & 1) * (8 * WD * 2 - 2048)));
    };

    // ---- fragment addresses in slot 0 (a tile and a slot add constants)
    // K: row c16 (+ 16), logical chunk 4 x + g4 of a tile's row (x < 4). V: the 4 x 16 patch of the
    // transposing read, rows 4 g4 + tr_row (+ 16), dims 16 x .. + 15 of a tile (x < 8).
    // (pointers, so that the constant parts of an address go into the instruction's offset field)
    const int tr_row = (lane & 15) >> 2;
    typedef __attribute__((address_space(3))) unsigned char* lds_byte_t;
    typedef const __attribute__((address_space(3))) bf16x8* lds_bf16x8_t;
    typedef __attribute__((address_space(3))) u32x4* lds_u32x4_t;
    typedef __attribute__((address_space(3))) f32x2* lds_f32x2_t;
    typedef __attribute__((address_space(3))) f32x4* lds_f32x4_t;
    typedef __attribute__((address_space(3))) s16x4* lds_s16x4_t;
    const lds_byte_t lds_base = (lds_byte_t)smem;
    lds_byte_t kfo[4], vfo[8];
#pragma unroll
    for (int x = 0; x < 4; x++) kfo[x] = lds_base + ((c16 * SL + (((4 * x + g4) ^ c16) * 8)) * 2);
#pragma unroll
    for (int x = 0; x < 8; x++)
        vfo[x] = lds_base + V_RING + 2 * dh * TILE_BYTES +
                 (((4 * g4 + tr_row) * SL + (((2 * x) ^ (tr_row << 2) ^ ((g4 & 1) << 1)) * 8) + 4 * (lane & 3)) * 2);
    // fragment f < 32 of a K block: dims 32 (f >> 1) .. + 31, keys 16 (f & 1) .. + 15
    auto k_read = [&](int slot, int f) __attribute__((always_inline)) {
        return *(lds_bf16x8_t)(kfo[(f >> 1) & 3] + (slot * K_SLOT + (f >> 3) * TILE_BYTES + (f & 1) * (16 * SL * 2)));
    };
    lds_byte_t p_own = lds_base + (P_RING + wave * (2 * 1024) + lane * 16);
    lds_byte_t p_other = lds_base + (P_RING + (wave ^ 1) * (2 * 1024) + lane * 16);

    // O^T, 16 tiles of 16 dims (256 dh + 16 dt ..) by 4 of 16 queries (this wave's two, then its
    // partner's): lane = query c16, dims 16 dt + 4 g4 + j.
    f32x4 oacc[16][4];
    const bf16x8 zero_frag = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
    f32x4 sv[2][2]; // scores of the block the next step exponentiates: [r][t] = query 16 r + c16, keys 16 t + 4 g4 + j
    float l_run[2] = {0.f, 0.f};

    // ---- prologue: K(0) and the query rows in; then K(1) and V(0) on their way under S(0); K(2)
    // The rows come whole (1 KB a load, chunk c of row r at c ^ (r & 15)) into 32 KB per wave of what the
    // rings do not hold yet: V's two slots, K's second one, what lies behind the V ring. (Fragments read from
    // memory as they lie, 16 pieces of 64 bytes a load, and K(1) and V(0) waited for ahead of S(0): 16 k cycles to the
    // first step instead of 12.4 k at 6208 tokens, 15.5 k instead of 7.7 k with few workgroups; what is left there is
    // the rate at which 160 KB per CU arrive.)
    unrolled<8>([&](auto i) __attribute__((always_inline)) { fetch_k(block_at(0), 0, i); });
    bf16x8 qf[16][2]; // (B operand of S^T = K Q^T): queries q0 + 16 r + c16, dims 32 kk + 8 g4 .. +7
    {
        const unsigned q_at = (unsigned)(wave < 2 ? V_RING + wave * V_SLOT : wave == 2 ? K_SLOT : P_RING);
        const unsigned q_lds = __builtin_amdgcn_readfirstlane(lds0 + q_at);
        const u32x4 q_rsrc = make_rsrc_words(a.q, span);
#pragma unroll
        for (int i = 0; i < 32; i++) {
            // rows past the end read the last row and are never stored
            const unsigned uo = __builtin_amdgcn_readfirstlane((unsigned)min(q0 + i, a.tokens - 1) * (unsigned)(WD * 2));
            load_to_lds_16(q_rsrc, q_lds + (unsigned)(i * WD * 2), (unsigned)(lane ^ (i & 15)) * 16u, uo);
        }
#pragma unroll
        for (int dt = 0; dt < 16; dt++)
#pragma unroll
            for (int o = 0; o < 4; o++) mfma_zero(oacc[dt][o], zero_frag);
        acc_drain();
        __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
        asm volatile("" ::: "memory");
        const lds_byte_t qp = lds_base + q_at + c16 * (WD * 2);
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int kk = 0; kk < 16; kk++) qf[kk][r] = *(lds_bf16x8_t)(qp + r * (16 * WD * 2) + (((4 * kk + g4) ^ c16) * 16));
    }
    __syncthreads(); // K(0) is in, the query rows are in registers
    unrolled<8>([&](auto i) __attribute__((always_inline)) { fetch_k(block_at(1), 1, i); });
    unrolled<8>([&](auto i) __attribute__((always_inline)) { fetch_v(block_at(0), 0, i); });
    bf16x8 kf[RA + 1]; // ring of fragments in flight
#pragma unroll
    for (int f = 0; f < RA; f++) kf[f] = k_read(0, f);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < 32; f++) {
        if (f + RA < 32) kf[(f + RA) % (RA + 1)] = k_read(0, f + RA);
#pragma unroll
        for (int r = 0; r < 2; r++) {
            if (f < 2) mfma_score<true>(sv[r][f & 1], kf[f % (RA + 1)], qf[f >> 1][r]);
            else mfma_score<false>(sv[r][f & 1], kf[f % (RA + 1)], qf[f >> 1][r]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // The scores are read next: they go through the wait, or the compiler, for which they are ready, reads them ahead of it.
    asm volatile("s_nop 15" : "+v"(sv[0][0]), "+v"(sv[0][1]), "+v"(sv[1][0]), "+v"(sv[1][1]));
    __builtin_amdgcn_sched_barrier(0);
    // Softmax in the exp2 domain (the scale rides on Q) against ONE reference point per row: the
    // largest score of the range's first block. It never moves, so nothing is ever rescaled
    // (any branch that touches the 256 accumulation registers inside the loop costs hundreds of
    // spills). fp32 and bf16 share one exponent
    // range, so a later score may lie far above the reference (P up to 2^90)
    // or far below it without any loss; only a row whose scores climb some 90 (log2) above
    // its first block's is out of reach. Such a row shows in its row sum, and the workgroup then
    // forms its rows again with a running maximum (safe::form_again).
    float mc[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        float m = sv[r][0][0];
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) m = fmaxf(m, sv[r][t][j]);
        mc[r] = pair_max(row_pair_max(m)); // over the four lane rows that share the query
    }
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): K(1) and V(0)
    __syncthreads(); // K(0) has no reader left
    unrolled<8>([&](auto i) __attribute__((always_inline)) { fetch_k(block_at(2), 0, i); });
#pragma unroll
    for (int f = 0; f < RA; f++) kf[f] = k_read(1, f);

    // Block 0's probabilities; from here on a step forms the next block's under its product.
    // P of 16 queries by 32 keys as the product's B operand: [r][k] packs keys 16 (k / 2) + 4 g4 + 2 (k % 2) .. + 1
    // what the scores start from: minus the reference point (which is not kept beside it: the pins hide that they are one)
    f32x4 neg[2];
#pragma unroll
    for (int r = 0; r < 2; r++) {
        neg[r] = f32x4{-mc[r], -mc[r], -mc[r], -mc[r]};
        asm volatile("" : "+v"(neg[r]));
    }
    u32x4 p_cur[2], p_alt[2];
    float block_sum[2] = {0.f, 0.f}; // their row sums, this lane's keys: part of l_run once the block counts
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const f32x4 v = sv[e >> 3][(e >> 2) & 1];
        const f32x2 y = {__builtin_amdgcn_exp2f(v[e & 3] - mc[e >> 3]), __builtin_amdgcn_exp2f(v[(e & 3) + 1] - mc[e >> 3])};
        block_sum[e >> 3] += y[0];
        block_sum[e >> 3] += y[1];
        p_cur[e >> 3][(e & 7) >> 1] = __builtin_bit_cast(unsigned, __builtin_convertvector(y, bf16x2));
    }

    // One step b with K(b+1) in K slot KS = (b + 1) % 2 and V(b) in V slot VS = b % 2:
    //   S phase: the 64 MFMAs of S(b+1) = K(b+1) Q^T; P(b), formed in the previous step, also goes
    //            into LDS for the partner;
    //   barrier: everything requested in the previous step's PV phase (V(b), K(b+2)) has landed;
    //            K(b+1) and V(b-1) have no reader left; both waves of a pair have their P(b) in LDS;
    //   PV phase: O += V(b)^T P(b)^T (64 MFMAs: 16 dim tiles by the four query tiles of the pair),
    //            the 8 loads each of V(b+1) and K(b+3) into the slots V(b-1) and K(b+1) left,
    //            the exponentials of block b+1, the first fragments of K(b+2).
    // Bound by what a lone wave can issue: 128 MFMAs of 16 cycles are 2048 cycles a step, and the step
    // takes 2730 (6208 and 16384 tokens; 2950 with the exponentials bunched in the S phase, M0 and the
    // offsets formed per load and the reference point subtracted from every score). Timing builds without
    // the loads -280, without the exchange of P -200, without K's or V's fragment reads -120 each, all of
    // them 2254. Fragments read further ahead change nothing; slots of half a K block, which spread the
    // loads over both phases, cost more in addresses than they gave (3130). At 16384 tokens the clock is
    // 1.86 GHz (1.59 GHz for the 32 x 32 x 16 form).
    auto step = [&](auto ks_c, int b, const u32x4 (&pc)[2], u32x4 (&pn)[2]) __attribute__((always_inline)) {
        constexpr int KS = decltype(ks_c)::value;       // slot of K(b+1); K(b+2) is in the other
        constexpr int VS = KS ^ 1;                      // slot of V(b); V(b+1) goes to the other
        constexpr int PS = VS;                          // P(b)'s slot: the one before was read before the last barrier
        f32x4 s[2][2];
        u32x4 pp[2];
        s16x4 vlo[VA + 1], vhi[VA + 1];
        // dim tile dt < 16 of this wave's half
        auto v_read = [&](int dt) __attribute__((always_inline)) {
            const lds_byte_t va = vfo[dt & 7] + (VS * V_SLOT + (dt >> 3) * TILE_BYTES);
            vlo[dt % (VA + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)va);
            vhi[dt % (VA + 1)] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(va + 16 * (SL * 2)));
        };
        // (what the last step exponentiates is past the range and never added)
#pragma unroll
        for (int r = 0; r < 2; r++) {
            l_run[r] += block_sum[r];
            block_sum[r] = 0.f;
        }
        // (the addresses are "redefined" here, or base + constant is formed again and again from one of them)
#pragma unroll
        for (int i = 0; i < 4; i++) asm volatile("" : "+v"(kfo[i]));
#pragma unroll
        for (int i = 0; i < 8; i++) asm volatile("" : "+v"(vfo[i]));
        asm volatile("" : "+v"(p_own));
        asm volatile("" : "+v"(p_other));
        __builtin_amdgcn_sched_barrier(0);
        unrolled<64>([&](auto t_c) __attribute__((always_inline)) {
            constexpr int t = decltype(t_c)::value, f = t >> 1, r = t & 1;
            if constexpr (r == 0 && f + RA < 32) kf[(f + RA) % (RA + 1)] = k_read(KS, f + RA);
            if constexpr (t >= 64 - 2 * VA && (t & 1) == 0) v_read((t - (64 - 2 * VA)) / 2);
            if constexpr (f < 2) mfma_score_from(s[r][f & 1], kf[f % (RA + 1)], qf[f >> 1][r], neg[r]);
            else mfma_score<false>(s[r][f & 1], kf[f % (RA + 1)], qf[f >> 1][r]);
            if constexpr (t == 3) *(lds_u32x4_t)(p_own + (PS * P_SLOT)) = pc[0];
            if constexpr (t == 7) *(lds_u32x4_t)(p_own + (PS * P_SLOT + 1024)) = pc[1];
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (t == 55) {
                __builtin_amdgcn_s_waitcnt(0x0070); // vmcnt(0) lgkmcnt(0)
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (t == 55) pp[0] = *(lds_u32x4_t)(p_other + (PS * P_SLOT));
            if constexpr (t == 57) pp[1] = *(lds_u32x4_t)(p_other + (PS * P_SLOT + 1024));
        });
        float x = 0.f, y = 0.f, even = 0.f;
        const unsigned at_v = block_at(b + 1), at_k = block_at(b + 3);
        unrolled<64>([&](auto m_c) __attribute__((always_inline)) {
            constexpr int m = decltype(m_c)::value, dt = m >> 2, o = m & 3;
            if constexpr (o == 1) { // 16 loads, V first
                if constexpr (dt < 8) fetch_v(at_v, VS ^ 1, IC<dt>{});
                else fetch_k(at_k, KS, IC<dt - 8>{});
            }
            if constexpr (o == 0 && dt + VA < 16) v_read(dt + VA);
            if constexpr ((m & 1) == 0 && m >= 64 - 2 * RA) kf[(m - (64 - 2 * RA)) / 2] = k_read(KS ^ 1, (m - (64 - 2 * RA)) / 2);
            const bf16x8 vf = __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(vlo[dt % (VA + 1)], vhi[dt % (VA + 1)], 0, 1, 2, 3, 4, 5, 6, 7));
            mfma_acc(oacc[dt][o], vf, __builtin_bit_cast(bf16x8, o < 2 ? pc[o & 1] : pp[o & 1]));
            // the exponential of score dt of block b + 1 (its MFMAs have drained: three more stand in between)
            if constexpr (o == 2) x = s[dt >> 3][(dt >> 2) & 1][dt & 3];
            if constexpr (o == 3) y = __builtin_amdgcn_exp2f(x);
            if constexpr (o == 0 && dt > 0) { // what is left to do of the one before
                block_sum[(dt - 1) >> 3] += y;
                if constexpr ((dt - 1) & 1) pn[(dt - 1) >> 3][((dt - 1) & 7) >> 1] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{even, y}), bf16x2));
                else even = y;
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        block_sum[1] += y;
        pn[1][3] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{even, y}), bf16x2));
        acc_drain();
    };
    int b = 0;
    for (; b + 1 < nblk; b += 2) {
        step(IC<1>{}, b, p_cur, p_alt);
        step(IC<0>{}, b + 1, p_alt, p_cur);
    }
    if (b < nblk) step(IC<1>{}, b, p_cur, p_alt);
    __builtin_amdgcn_s_waitcnt(0x0F70); // no direct load may outlive the workgroup's LDS

    // ---- epilogue: O = O^T / l, or the range's share as it stands
    // (the lane's coordinates are formed again: kept across the loop they would cost it registers)
    int el;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(el));
    const int ec = el & 15, eg = el >> 4;
    float l_tot[2];
    bool out_of_reach = false;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        l_tot[r] = pair_sum(row_pair_sum(l_run[r]));
        out_of_reach |= !(l_tot[r] <= kRowSumLimit);
    }
    // a row sum past kRowSumLimit (or not a number): some score left the reach of the fixed reference
    const bool mine_out = __any(out_of_reach);
    if (mine_out && el == 0) a.redo[tile] = 1;
    // the partner's reference points and row sums, through P's first slot (every wave is done with it)
    typedef __attribute__((address_space(3))) int* lds_int_t;
    __syncthreads();
    if (el == 0) *(lds_int_t)(lds_base + (P_RING + BQ * 8 + wave * 4)) = mine_out ? 1 : 0;
    if (eg == 0) {
#pragma unroll
        for (int r = 0; r < 2; r++) *(lds_f32x2_t)(lds_base + (P_RING + (wave * 32 + 16 * r + ec) * 8)) = f32x2{-neg[r][0], l_tot[r]};
    }
    __syncthreads();
    // A lane's four dims would leave as pieces of 64 bytes, which the CU's address unit takes one by
    // one (19 k cycles, 8 us of every launch): 16 rows at a time are turned through 16 KB of the
    // wave's own (chunk c of row r at c ^ r) and stored 1 KB an instruction (12 k).
    const lds_byte_t turn = lds_base + wave * (16 * 1024);
#pragma unroll
    for (int o = 0; o < 4; o++) {
        const int w = o < 2 ? wave : wave ^ 1;
        const int row0 = tile * BQ + 32 * w + 16 * (o & 1);
        if (row0 >= a.tokens) continue; // (whole groups of 16 rows: tokens % 64 == 0)
        const f32x2 ml = *(lds_f32x2_t)(lds_base + (P_RING + (w * 32 + 16 * (o & 1) + ec) * 8));
        // (one workgroup of two writes them, the one that would write them again)
        if (nsp > 1 && o < 2 && eg == 0 && (wg & a.halves) == 0) *reinterpret_cast<f32x2*>(a.part_ml + ((int64_t)part * a.tokens + row0 + ec) * 2) = ml;
        if (a.halves && dh != (wg & 1)) continue;
        const float scale = nsp > 1 ? 1.0f : ml[1] > 0.f ? 1.0f / ml[1] : 0.f;
#pragma unroll
        for (int dt = 0; dt < 16; dt++) *(lds_f32x4_t)(turn + ec * 1024 + (((4 * dt + eg) ^ ec) * 16)) = oacc[dt][o] * scale;
        float* op = (nsp > 1 ? a.part_o + ((int64_t)part * a.tokens + row0) * WD : a.o + (int64_t)row0 * WD) + 256 * dh;
#pragma unroll
        for (int r = 0; r < 16; r++)
            store_through(op + (int64_t)r * WD + ((el ^ r) * 4), (f32x4)*(lds_f32x4_t)(turn + r * 1024 + el * 16));
    }
    // what any wave of the workgroup found, read by all of them (nothing has been written there since the barrier)
    int again = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) again |= *(lds_int_t)(lds_base + (P_RING + BQ * 8 + w * 4));
    if (__builtin_amdgcn_readfirstlane(again) == 0) return;
    __builtin_amdgcn_s_waitcnt(0x0F70); // the rows above are in memory before they are written again
    for (int half = wg & a.halves; half < 2; half += 1 + a.halves) {
        __syncthreads(); // and nobody reads what is in the LDS
        int dh2 = half;
        asm volatile("" : "+s"(dh2)); // (nothing of a half is to be kept for the other)
        safe::form_again(a, smem, wave, tile, part, nsp, blk0, nblk, dh2);
    }
}

// Combines the key ranges of a split launch, in range order: with reference points m_p and row
// sums l_p, O = sum_p 2^(m_p - m) O_p / sum_p 2^(m_p - m) l_p, m = max_p m_p. A thread owns four
// dims of one row; NP = the number of ranges is the build's, so that every range's load is sent
// before the first is used, with no branch between them.
template <int NP>
__global__ void __launch_bounds__(256) wide_merge_kernel(const WideArgs a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; // (row, dim / 4)
    const int64_t row = i / (WD / 4);
    if (row >= a.tokens) return;
    const int c4 = (int)(i - row * (WD / 4));
    f32x2 ml[NP];
    f32x4 o[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) ml[p] = *reinterpret_cast<const f32x2*>(a.part_ml + ((int64_t)p * a.tokens + row) * 2);
#pragma unroll
    for (int p = 0; p < NP; p++) o[p] = *reinterpret_cast<const f32x4*>(a.part_o + ((int64_t)p * a.tokens + row) * WD + 4 * c4);
    float mm = -INFINITY;
#pragma unroll
    for (int p = 0; p < NP; p++) mm = fmaxf(mm, ml[p][0]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    float lt = 0.f;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const float w = (ml[p][0] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(ml[p][0] - mm);
        acc += o[p] * w;
        lt += ml[p][1] * w;
    }
    const float inv = lt > 0.f ? 1.0f / lt : 0.f;
    store_through(a.o + row * WD + 4 * c4, acc * inv);
}

} // namespace wide

int wide_head_dim() { return wide::WD; }
int wide_block_rows() { return 64; } // the reference's tokens % 64 == 0; a last tile may be half full

hipError_t launch_wide_round(const WidePrepArgs& p, hipStream_t stream) {
    if (p.chunks <= 0) return hipErrorInvalidValue;
    const int64_t want = (p.chunks + 255) / 256;
    const unsigned blocks = (unsigned)(want < 4096 ? want : 4096);
    wide::wide_round_kernel<<<dim3(blocks, 3), dim3(256), 0, stream>>>(p);
    return hipGetLastError();
}

size_t wide_part_bytes(int tokens, int splits) {
    return splits > 1 ? (size_t)splits * (size_t)tokens * (wide::WD + 2) * sizeof(float) : 0;
}
// Key ranges per query tile (one workgroup each, of equal length but for the last, at least eight
// blocks): the number whose estimate is the smallest. A full round over the CUs takes kFullUs per
// block of a range (the power limit), one that fills up to kThinFill of them kThinUs (a wave's own chain), in between
// in proportion; every range's share of O goes to memory and back once. The constants are a fit to
// 1 to 8 ranges of 37 lengths from 256 to 18432 tokens, every number of ranges timed: the pick is the best or within 4 % of it, 0.6 %
// in the mean (but at 1280 tokens: 48.9 us with five for 45.8 with four; a rule that rose in proportion to the fill from the
// start took the widest split too late: us per call 1408 tokens 53.2 -> 47.5, 2560 57.0 -> 54.6,
// 5248 93.9 -> 90.5, 7424 141.7 -> 131.6, 8192 157.2 -> 150.4, 21248 850.3 -> 730.1; of 49 lengths up to 35072 that the new
// constants moved, none slower). 6208 tokens stay at four, 110.9 for 107.6 with five, whose shares take a quarter more. Estimates
// leave out a call's other 25 us, so
// ranges that save less than 3 % are not worth their shares (1019904 tokens would take five ranges and 10 GB
// for 1.6 %), and neither are shares of more than kMaxShareBytes, which the queue keeps (33024 tokens: six
// ranges, 389 MiB, 29 % of the time by the estimate; 18432: three, 108 MiB, 13 %).
// (A power of two that divides the blocks, which this was at first, left 6208 tokens, 194 blocks, at
// two ranges and 98 workgroups: call 152 us against 119 with four; 18432 tokens at one range:
// 678 against 610 with three.)
int wide_splits(int tokens, int cus) {
    constexpr size_t kMaxShareBytes = (size_t)512 << 20;
    constexpr float kMinGain = 0.03f;
    constexpr float kFullUs = 1.55f, kThinUs = 1.13f, kThinFill = 0.66f, kRoundUs = 5.5f, kMergeUs = 4.0f, kShareBytesPerUs = 3.3e6f;
    if (cus <= 0) return 1;
    const int tiles = (tokens + wide::BQ - 1) / wide::BQ;
    const int nblk = tokens / wide::KB;
    int best = 1;
    float best_us = INFINITY, whole_us = INFINITY;
    for (int s = 1; s <= wide::kMaxSplits; s++) {
        if (wide_part_bytes(tokens, s) > kMaxShareBytes) break;
        const int per = (nblk + s - 1) / s;
        if (s > 1 && (per < 8 || (s - 1) * per >= nblk)) continue; // (no empty range)
        const int rounds = tiles * s / cus, last = tiles * s % cus;
        float us = (float)rounds * ((float)per * kFullUs + kRoundUs);
        const float past = fmaxf((float)last / (float)cus - kThinFill, 0.f) / (1.f - kThinFill);
        if (last) us += (float)per * (kThinUs + (kFullUs - kThinUs) * past) + kRoundUs;
        if (s > 1) us += kMergeUs + (float)s * (float)tokens * (float)(wide::WD * sizeof(float)) / kShareBytesPerUs;
        if (s == 1) whole_us = us;
        if (us < best_us) { best_us = us; best = s; }
    }
    return best_us < whole_us * (1.f - kMinGain) ? best : 1;
}
// Whether two workgroups take each tile and range, each for one half of the output dims: where both together fill
// no more than half of the CUs. Rows that are formed again are formed once per half, which one workgroup does in turn; two at
// once lose nothing meanwhile, and each has half of the rows to store. us per call, one -> two, every row formed again: 64
// tokens 53.4 -> 42.0, 256 77.1 -> 57.9, 512 79.5 -> 60.0, 1152 (45 workgroups) 86.4 -> 67.4, 8192 in one range (64) 851 -> 604;
// ordinary data 256 38.2 -> 38.2, 512 40.8 -> 40.3, 960 43.0 -> 42.1, 1152 47.3 -> 46.8, 8192 in one range 353.6 -> 353.1. Past the line both read K and V too often: ordinary 1664 tokens (91) 46.1 -> 46.4,
// 2048 (128) 48.3 -> 49.3, 2560 (160) 53 -> 73.
int wide_halves(int tokens, int splits, int cus) {
    const int64_t wgs = (int64_t)wide_tiles(tokens) * (splits > 1 ? splits : 1);
    return 4 * wgs <= cus ? 1 : 0;
}

hipError_t launch_wide_attention(const WideArgs& a, hipStream_t stream) {
    if (a.tokens <= 0 || a.tokens % wide_block_rows() != 0) return hipErrorInvalidValue;
    const int nsp = a.splits > 1 ? a.splits : 1;
    const int nblk = a.tokens / wide::KB;
    if (nsp > wide::kMaxSplits || (nsp - 1) * ((nblk + nsp - 1) / nsp) >= nblk) return hipErrorInvalidValue; // every range has a block
    if (nsp > 1 && (a.part_o == nullptr || a.part_ml == nullptr)) return hipErrorInvalidValue;
    const unsigned tiles = (unsigned)((a.tokens + wide::BQ - 1) / wide::BQ);
    if (a.redo == nullptr || (a.halves != 0 && a.halves != 1)) return hipErrorInvalidValue;
    wide::attn_wide_kernel<<<dim3((tiles * (unsigned)nsp) << a.halves), dim3(wide::NT), wide::kLdsBytes, stream>>>(a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (nsp > 1) {
        const int64_t threads = (int64_t)a.tokens * (wide::WD / 4);
        const dim3 mgrid((unsigned)((threads + 255) / 256));
        switch (nsp) {
#define ZD_MERGE(N) case N: wide::wide_merge_kernel<N><<<mgrid, dim3(256), 0, stream>>>(a); break;
        ZD_MERGE(2) ZD_MERGE(3) ZD_MERGE(4) ZD_MERGE(5) ZD_MERGE(6) ZD_MERGE(7) ZD_MERGE(8)
#undef ZD_MERGE
        }
        static_assert(wide::kMaxSplits == 8, "one case per number of ranges");
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t wide_setup() {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&wide::attn_wide_kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)wide::kLdsBytes);
}
int wide_tiles(int tokens) { return (tokens + wide::BQ - 1) / wide::BQ; }

} // namespace zdraw
