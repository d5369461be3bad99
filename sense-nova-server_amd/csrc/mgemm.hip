// Matrix-core block-quantised GEMM for chunked prefill (M up to 512 token rows), gfx950.
//
// y[m, n] = sum_b s[n, b] * sum_{i<32} q[n, 32b + i] * x[m, 32b + i]
//
// The reference runs its tiled matmul for more than 8 rows (src/shaders/matmul.wgsl:200-318,
// MatKind::Tiled in src/gpu.rs:191-218).  Here every product runs on v_mfma_f32_32x32x16_f16
// with exact operands, as in the decode GEMV: quants become f16 exactly, and each token row is
// split into f16 hi + lo parts (22 significant bits) under a per-token power of two.  Four MFMAs
// (two halves of K, hi and lo) cover exactly one quant block, so the 32x32 block result of each
// (token tile, row tile) is scaled by its 32 block scales and accumulated in f32.
//
// The scale FMAs (16 per lane and block result) and the dequantisation run beside the MFMAs.  On
// this part a 32x32x16 MFMA takes 13.9 ns per SIMD alone and 14.6 with 6 vector instructions
// between it and the next; a 16x16x32 one, half the work, takes 8.9 ns alone, 10.3 with 3 and 13.3
// with 4.  So the larger shape does the same block results in 0.7 of the time.
//
// Panel order of the weights (a second copy beside the decode GEMV's tile order, kept for the
// prefill path only).  A stage is two quant blocks (64 elements of K):
//   row tile R    rows 32R..32R+31 (rows past N are zero, scale 0)
//   Q8 pieces     (R, stage, block): 64 lanes x 16 bytes; lane l = 32g + j holds row 32R + j's bytes
//                 [8g, 8g+8) and [16+8g, 16+8g+8) of the block, in offset binary (q + 128)
//   Q4 piece      (R, stage): lane l holds words g and 2 + g of the stage's first block, then of the second
//   scales        [R][stage][32 rows][2 blocks] f32
// Row tile R's pieces are contiguous, so a wave streams its rows in 1 KiB loads.
//
// Token fragments (written by launch_rows_to_frags): for token tile T (32 rows), block b and half
// h of the block, the hi then the lo MFMA A fragment, 64 lanes x 8 f16, lane 32g + t holding token
// 32T + t's elements 32b + 16h + 8g + (0..7) (Q4: in the order 0, 4, 1, 5, 2, 6, 3, 7 that the
// nibble dequant produces), scaled by 2^-e(token); xs[m] = 2^e(m) restores the scale.
//
// Each output element's arithmetic is fixed by its row and column, whatever M or the tile it falls
// in, so a token's result does not depend on the chunk that carries it.  K is cut into slices by a
// rule on (N, K) alone (slices_of), the slices into groups; a slice's blocks are summed in order from
// zero, a group's slices in order and the groups in order, whether one block runs them all or each
// slice, or each group, is a block of its own.
#include <algorithm>

#include "common.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace snl {

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));


__device__ __forceinline__ half2_t as_h2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }

// 8 quants of one block as exact f16 (Q8: offset-binary bytes of two words; Q4: the 8 nibbles of one word, in
// the order 0, 4, 1, 5, 2, 6, 3, 7).
__device__ __forceinline__ half8_t q8_to_h8(uint32_t w0, uint32_t w1) {
    const half2_t bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const half2_t p0 = as_h2(__builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u)) - bias;
    const half2_t p1 = as_h2(__builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u)) - bias;
    const half2_t p2 = as_h2(__builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u)) - bias;
    const half2_t p3 = as_h2(__builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u)) - bias;
    return half8_t{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

__device__ __forceinline__ half8_t q4_to_h8(uint32_t v) {
    const half2_t bias = {(_Float16)1032.0f, (_Float16)1032.0f};
    const half2_t p0 = as_h2((v & 0x000F000Fu) | 0x64006400u) - bias;
    const half2_t p1 = as_h2(((v >> 4) & 0x000F000Fu) | 0x64006400u) - bias;
    const half2_t p2 = as_h2(((v >> 8) & 0x000F000Fu) | 0x64006400u) - bias;
    const half2_t p3 = as_h2(((v >> 12) & 0x000F000Fu) | 0x64006400u) - bias;
    return half8_t{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

// ---- reference layout -> panel order ----
// one thread per (piece, lane)
__global__ __launch_bounds__(256) void panel_pack_q_kernel(int quant, int N, int K, const uint8_t* q, uint8_t* qp,
                                                           size_t n_items) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= n_items) return;
    const int lane = (int)(idx & 63);
    const size_t pc = idx >> 6;
    const int npc = quant == 0 ? K / 32 : K / 64;  // pieces per row tile
    const int R = (int)(pc / npc), p = (int)(pc % npc);
    const int j = lane & 31, g = lane >> 5;
    const int row = 32 * R + j;
    uint4 out = quant == 0 ? make_uint4(0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u) : make_uint4(0u, 0u, 0u, 0u);
    if (row < N) {
        if (quant == 0) {
            const uint32_t* s4 = reinterpret_cast<const uint32_t*>(q + (size_t)row * K + (size_t)p * 32 + 8 * g);
            out = make_uint4(s4[0] ^ 0x80808080u, s4[1] ^ 0x80808080u, s4[4] ^ 0x80808080u, s4[5] ^ 0x80808080u);
        } else {
            const uint32_t* s4 = reinterpret_cast<const uint32_t*>(q + (size_t)row * (K / 2) + (size_t)p * 32 + 4 * g);
            out = make_uint4(s4[0], s4[2], s4[4], s4[6]);
        }
    }
    reinterpret_cast<uint4*>(qp)[idx] = out;
}

// one thread per (row tile, stage, row)
__global__ __launch_bounds__(256) void panel_pack_s_kernel(int N, int K, const float* s, float* sp, size_t n_items) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= n_items) return;
    const int j = (int)(idx & 31);
    const size_t rq = idx >> 5;
    const int nst = K / 64;
    const int R = (int)(rq / nst), p = (int)(rq % nst);
    const int row = 32 * R + j;
    float2 v = make_float2(0.f, 0.f);
    if (row < N) {
        const float* sr = s + (size_t)row * (K / 32) + 2 * p;
        v = make_float2(sr[0], sr[1]);
    }
    reinterpret_cast<float2*>(sp)[idx] = v;
}

// ---- token rows -> MFMA A fragments (hi, lo) ----
constexpr int kRowThreads = 256;

__device__ __forceinline__ float block_max256(float v, float* red) {
    v = wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// the hi fragment entry of 8-element group u of token 32T + t (the lo entry is 64 further)
__device__ __forceinline__ size_t frag_index(int T, int nb, int u, int t) {
    return (((size_t)T * nb + (u >> 2)) * 4 + (u & 2)) * 64 + 32 * (u & 1) + t;
}

// One block per token row: the row's 8-element groups are held in registers (GPT per thread),
// the branch input is formed (RMSNorm (1 + w) of stream 0 or of the mHC pre-mix, the DeltaNet head
// factor, one per group, or SwiGLU of a gate and up row), then the row's largest magnitude sets the power of two and each
// group is written as its hi and lo halves of the MFMA A fragments.
template <int GPT>
__global__ __launch_bounds__(kRowThreads) void rows_to_frags_kernel(RowsArgs a) {
    __shared__ float red[4];
    __shared__ float rs[4];
    // Block b runs on XCD b % 8; each XCD takes an eighth of the rows in a run, so the 16-byte pieces of
    // neighbouring rows that share a fragment's cache lines meet in one L2.  (The grid is whole tiles of
    // 32 rows.)
    const int m = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const int tid = threadIdx.x, K = a.K, nb = K / 32, ngr = K / 8;
    const int T = m >> 5, t = m & 31;
    half8_t* xf = reinterpret_cast<half8_t*>(a.frags);
    if (m >= a.M) {  // padding rows of the last token tile
        const half8_t z = {};
        for (int u = tid; u < ngr; u += kRowThreads) {
            const size_t f = frag_index(T, nb, u, t);
            xf[f] = z;
            xf[f + 64] = z;
        }
        if (tid == 0) a.xs[m] = 0.0f;
        return;
    }
    const float* xr = a.x + (size_t)m * a.x_stride;
    float f0 = 1.0f, f1 = 0.0f;
    if (a.mode == ROWS_NORM_MHC) {
        f0 = a.coef[m * 8];
        f1 = a.coef[m * 8 + 1];
    }
    float v[GPT][8];
    float ss = 0.0f;
#pragma unroll
    for (int gi = 0; gi < GPT; ++gi) {
        const int u = tid + kRowThreads * gi;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[gi][e] = 0.0f;
        if (u < ngr) {
            const float4* p = reinterpret_cast<const float4*>(xr + 8 * u);
            const float4 p0 = p[0], p1 = p[1];
            float w8[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
            if (a.mode == ROWS_NORM_MHC) {
                const float4* q = reinterpret_cast<const float4*>(xr + a.h + 8 * u);
                const float4 q0 = q[0], q1 = q[1];
                const float u8[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) w8[e] = f0 * w8[e] + f1 * u8[e];
            } else if (a.mode == ROWS_SWIGLU) {  // layers.wgsl:164-175: silu(gate) * up
                const float4* q = reinterpret_cast<const float4*>(xr + a.h + 8 * u);
                const float4 q0 = q[0], q1 = q[1];
                const float u8[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) w8[e] = silu(w8[e]) * u8[e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[gi][e] = w8[e];
                ss = fmaf(w8[e], w8[e], ss);
            }
        }
    }
    if (a.mode == ROWS_NORM || a.mode == ROWS_NORM_MHC) {
        // layers.wgsl:46-73: RMSNorm of the (pre-mixed) stream-0 row
        const float tot = block_sum<kRowThreads>(ss, rs);
        const float rinv = 1.0f / sqrtf(tot / (float)K + a.eps);
#pragma unroll
        for (int gi = 0; gi < GPT; ++gi) {
            const int u = tid + kRowThreads * gi;
            if (u < ngr)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[gi][e] = (v[gi][e] * rinv) * (1.0f + a.w[8 * u + e]);
        }
    } else if (a.mode == ROWS_GNORM) {  // head factor of the gated RMS norm of 128-wide heads
#pragma unroll
        for (int gi = 0; gi < GPT; ++gi) {
            const int u = tid + kRowThreads * gi;
            if (u < ngr) {
                const float* ps = a.ssq + ((size_t)m * (K / 128) + u / 16) * kDeltaPrefillGroups;
                float t = ps[0];
#pragma unroll
                for (int gi = 1; gi < kDeltaPrefillGroups; ++gi) t = t + ps[gi];
                const float var_o = t / 128.0f;
                const float f = 1.0f / sqrtf(var_o + a.eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[gi][e] = v[gi][e] * f;
            }
        }
    }
    float amax = 0.0f;
#pragma unroll
    for (int gi = 0; gi < GPT; ++gi)
#pragma unroll
        for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[gi][e]));
    amax = block_max256(amax, red);
    // hi = f16(v * 2^-e) with the largest magnitude in [2^14, 2^15)
    int ex = 0;
    if (amax > 0.0f) ex = max(ilogbf(amax) - 14, -110);
    const float down = ldexpf(1.0f, -ex);
    const int q4 = a.perm4;
#pragma unroll
    for (int gi = 0; gi < GPT; ++gi) {
        const int u = tid + kRowThreads * gi;
        if (u >= ngr) continue;
        half8_t hi, lo;
#pragma unroll
        for (int pp = 0; pp < 8; ++pp) {
            // Q4 fragments take the element order 0, 4, 1, 5, 2, 6, 3, 7 of the nibble dequant
            const float x = (q4 ? v[gi][(pp & 1) ? 4 + (pp >> 1) : (pp >> 1)] : v[gi][pp]) * down;
            const _Float16 hv = (_Float16)x;
            hi[pp] = hv;
            lo[pp] = (_Float16)(x - (float)hv);
        }
        const size_t f = frag_index(T, nb, u, t);
        xf[f] = hi;
        xf[f + 64] = lo;
    }
    if (tid == 0) a.xs[m] = ldexpf(1.0f, ex);
}

// ---- the GEMM ----
// Block: WT waves along the tokens x WR along the rows; wave (wt, wr) takes TTW token tiles x RT
// row tiles of 32.  A stage's token fragments, weight pieces and scales are copied global -> LDS by
// global_load_lds (16 bytes per lane, lane i at base + 16i) into a ring of D buffers.  Every copy of
// a wave keeps one scalar base address; the stages advance through one vector offset per operand, so
// issuing a stage costs three instructions a copy (forming the addresses anew in a loop took longer
// than the stage's products: 64 x 128 blocks 0.98 -> 0.80 us a stage).  The fragments of a block are
// read from LDS while the block before it is multiplied.
//
// What bounds it.  The same MFMAs and FMAs in a bare loop run at 2160 TFLOP/s on constant operands and at
// 1500 on random ones (no instruction waits for another in either), the matrix cores' rate on real
// data.  The hi / lo split doubles the useful flops, so 750 TFLOP/s of a 512-row product is the ceiling
// of this form.  gate_up at 512 rows reaches 460.  Its products alone, with no copy, LDS read or barrier
// in the loop, took 211 of 257 us in 128 x 256 blocks, 489 TFLOP/s: 384 blocks are 1.5 rounds of the
// CUs, and the rest of the distance to 750 is not explained by what was measured.
//
// The whole launch, before -> now, Q8 / Q4 (us, N x K, M 512): 24576 x 4096 316 / 301 -> 224 / 223,
// 12352 x 4096 167 / 196 -> 124 / 126, 4096 x 4096 72 / 65 -> 50 / 51, 4096 x 12288 201 / 183 ->
// 127 / 127 by group (145 / 141 in whole blocks); M 45: 24576 x 4096 69 / 62 -> 44 / 46, 4096 x 4096
// 64 / 57 -> 16 / 15 and 4096 x 12288 182 / 163 -> 25 / 25, by slice.
// Slices of K for matrices whose 128-row panels alone leave most CUs idle.  At 4096 x 12288, 45 rows,
// one block per panel takes 182 us and 8 slices 25.  The line at 46 panels is laid for 512 rows (K 4096:
// 45 panels in two slices 85 us, 46 in one 73); as a rule on the shape alone it also keeps few rows from a
// cut that they would gain from (45 rows: 45 panels 17.5 us, 46 39).  Slices of 512 elements are 8 stages,
// about as long as a block's first copies take.
constexpr int kSliceMin = 512;
// 64 x 128 panels up to which a launch splits its slices over blocks (4096 x 4096: 192 rows, split, 39 us,
// 193, whole, 44; 4096 x 12288: 72 and, by group, 100; 2048 x 4096: 384 rows 42, 385 44.  More panels were
// not tried: of 256 rows, 128 panels, the partial sums would be 33 MB)
constexpr int kSplitPanels = 96;

// WT x WR waves along tokens and rows, TTW x RT 32x32 tiles per wave
template <int QT, int WT_, int WR_, int TTW, int RT>
struct GemmStage {
    static constexpr int WT = WT_, WR = WR_, NW = WT * WR;
    static constexpr int TT = WT * TTW;  // token tiles per block
    static constexpr int BR = WR * RT;   // row tiles per block
    // 1 KiB copies per stage: token fragments (two blocks, two halves, hi and lo per token tile),
    // weight pieces, scales of 4 row tiles each
    static constexpr int PB = QT == 0 ? 2 : 1;  // weight pieces per row tile
    static constexpr int NA = TT * 8, NB = BR * PB, NS = (BR + 3) / 4;
    static constexpr int NC = NA + NB + NS;
    static constexpr int U4 = NC * 64;  // uint4 per stage
    // copies of a wave: the remainder of the weight pieces goes to the first waves, the scales to the last
    static constexpr int WA = NA / NW, WB = NB / NW, XB = NB % NW;
    static constexpr int WC = WA + WB;  // a wave's copies, one more for wave < XB or >= NW - NS
    static_assert(NA % NW == 0 && XB + NS <= NW, "at most one more copy for some waves");
    // stage buffers; where there is room for six, stages are published in pairs (PS), one barrier each
    static constexpr int D_MAX = 160 * 1024 / (U4 * 16);
    static constexpr int D = D_MAX >= 8 ? 8 : D_MAX >= 6 ? 6 : D_MAX;
    static constexpr int PS = D >= 6 ? 2 : 1;
    static constexpr size_t BYTES = D * (size_t)U4 * 16;
    static_assert(D >= 3 && BYTES <= 160 * 1024, "at least three stages fit the LDS");
};

// s_waitcnt immediate (gfx9 layout): vector memory count vm, LDS count 0, export count untouched
constexpr int wait_vm_lgkm0(int vm) { return (vm & 15) | ((vm >> 4) << 14) | (7 << 4); }

// Wait until at most `n` (a uniform value up to MAX, or more) stages of C copies each are outstanding.
template <int C, int MAX, int STEP>
__device__ __forceinline__ void wait_stages(int n) {
    if constexpr (MAX > 0) {
        if (n >= MAX) {
            __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(MAX * C));
            return;
        }
        wait_stages<C, MAX - STEP, STEP>(n);
    } else {
        __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(0));
    }
}

// 1 KiB global -> LDS copy of one wave: lane i moves 16 bytes from base + voff(i) to LDS
// dst + 16 i.  Issued as inline assembly, so the compiler's wait insertion does not see it and
// does not hold every LDS read until all copies in flight have landed; the kernel orders the
// copies itself (s_waitcnt on the vector memory count before the barrier that publishes a stage).
// The compiler's own waits stay correct: loads it does not know about can only make them wait
// longer.
__device__ __forceinline__ void copy16_to_lds(const char* base, unsigned voff, unsigned dst) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(voff), "s"(base)
                 : "memory", "m0");
}

// What one block runs of its outputs' sums (struct Slices): all of K, or one slice or one group of
// slices, whose sum it leaves in a.part.
enum Split { WHOLE = 0, BY_SLICE = 1, BY_GROUP = 2 };
struct Slices {
    int n, st;         // slices, stages of each (the last takes the rest)
    int groups, per;   // groups, slices of each
    int run_st(int split) const { return split == BY_SLICE ? st : st * per; }
    int runs(int split) const { return split == BY_SLICE ? n : groups; }
};
template <int QT, int WT, int WR, int TTW, int RT, int SPLIT>
__global__ __launch_bounds__(WT * WR * 64) void mgemm_kernel(GemmArgs a, int r_first, int rpanels, int tpanels,
                                                             Slices sl) {
    using G = GemmStage<QT, WT, WR, TTW, RT>;
    extern __shared__ __align__(16) uint4 lds[];  // D stage buffers of G::U4
    // the wave index in a scalar register: the copies' addresses then form in scalar code
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wt = wave / G::WR, wr = wave % G::WR;
    // XCD-aware numbering: block b runs on XCD b % 8; give each XCD whole row panels (SPLIT: whole
    // slices of row panels), whose weights its L2 then serves to every token panel
    const int runs = SPLIT == BY_SLICE ? sl.n : SPLIT == BY_GROUP ? sl.groups : 1;
    const int units = rpanels * runs;
    const int bid = blockIdx.x;
    const int xcd = bid & 7, idx = bid >> 3;
    const int per_xcd = (units + 7) / 8;
    const int unit = xcd * per_xcd + idx / tpanels;
    const int tp = idx % tpanels;
    if (unit >= units) return;
    const int rp = SPLIT ? unit / runs : unit, z = SPLIT ? unit % runs : 0;
    const int nb = a.K / 32, nst_all = a.K / 64;
    const int run_st = SPLIT == BY_SLICE ? sl.st : sl.st * sl.per;
    const int st0 = SPLIT ? z * run_st : 0;
    const int nst = SPLIT ? min(run_st, nst_all - st0) : nst_all;
    const int j = lane & 31, g = lane >> 5;
    const int R0 = r_first + rp * G::BR, T0 = tp * G::TT;

    // The panel copies and the token fragments are allocated in whole block panels (gemm_q_bytes,
    // gemm_s_floats, frags_bytes), so no copy needs a clamp.  Rows and tokens past the matrix only
    // feed outputs that are not stored.
    const char* xf_b = reinterpret_cast<const char*>(a.frags);
    const char* wq_b = reinterpret_cast<const char*>(a.wq);
    const char* ws_b = reinterpret_cast<const char*>(a.ws);
    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
    const char *srcA[G::WA], *srcB[G::WB + 1];
#pragma unroll
    for (int i = 0; i < G::WA; ++i) {  // token tile c / 8, block c / 4 % 2, half c / 2 % 2, hi / lo c % 2
        const int c = wave + G::NW * i;
        srcA[i] = xf_b + ((((size_t)(T0 + c / 8) * nb + 2 * st0) * 4 + c % 8) << 10);
    }
    auto piece = [&](int c) {  // weight piece c of the block
        return wq_b + ((((size_t)(R0 + c / G::PB) * nst_all + st0) * G::PB + c % G::PB) << 10);
    };
#pragma unroll
    for (int i = 0; i < G::WB; ++i) srcB[i] = piece(wave + G::NW * i);
    // the extra copy: a weight piece, the scales of 4 row tiles, or none
    const bool xb = wave < G::XB, xs_copy = wave >= G::NW - G::NS;
    const int sc = wave - (G::NW - G::NS);
    srcB[G::WB] = xs_copy ? ws_b + ((size_t)(R0 + 4 * sc) * nst_all + st0) * 256 : piece(G::NW * G::WB + wave);
    const unsigned dst_x = (unsigned)(xs_copy ? G::NA + G::NB + sc : G::NA + G::NW * G::WB + wave) * 1024u;
    const bool extra = xb || xs_copy;
    // lane offsets, advanced stage by stage (copies are issued in stage order)
    unsigned offA = (unsigned)lane * 16u, offB = (unsigned)lane * 16u;
    // scales: lane l -> row tile l / 16 of the copy's 4, 16 of its stage's 256 bytes
    unsigned offX = xs_copy ? (unsigned)(lane >> 4) * (unsigned)nst_all * 256u + (unsigned)(lane & 15) * 16u : offB;
    const unsigned stepX = xs_copy ? 256u : 1024u * G::PB;
    auto issue = [&](unsigned dst0) {
#pragma unroll
        for (int i = 0; i < G::WA; ++i) copy16_to_lds(srcA[i], offA, dst0 + (unsigned)(wave + G::NW * i) * 1024u);
#pragma unroll
        for (int i = 0; i < G::WB; ++i)
            copy16_to_lds(srcB[i], offB, dst0 + (unsigned)(G::NA + wave + G::NW * i) * 1024u);
        if (extra) copy16_to_lds(srcB[G::WB], offX, dst0 + dst_x);
        offA += 8192u;
        offB += 1024u * G::PB;
        offX += stepX;
    };
    // at most n stages outstanding (the first wait, which could leave more, leaves as many as the
    // others: it costs one latency per block), every LDS read complete
    auto wait_copies = [&](int n) {
        if (extra) wait_stages<G::WC + 1, G::D - 2 * G::PS, G::PS>(n);
        else wait_stages<G::WC, G::D - 2 * G::PS, G::PS>(n);
    };

    // the running sums of the slice, of the group and of all groups
    f32x16_t acc[RT][TTW], grp[RT][TTW], tot[RT][TTW];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < TTW; ++t) acc[r][t] = grp[r][t] = tot[r][t] = f32x16_t{};

    half8_t x[2][TTW][4];  // [block of the stage][token tile][2 * half + (0 hi, 1 lo)]
    uint4 wv[2][RT][G::PB];  // [stage % 2]; Q8: the two blocks' bytes; Q4: both blocks' words
    float2 sv[2][RT];
    auto read_block = [&](int b, const uint4* la) {
#pragma unroll
        for (int t = 0; t < TTW; ++t)
#pragma unroll
            for (int f = 0; f < 4; ++f)
                x[b][t][f] = __builtin_bit_cast(half8_t, la[(((wt * TTW + t) * 2 + b) * 4 + f) * 64 + lane]);
    };
    auto read_weights = [&](int p, const uint4* la) {
        const uint4* lb = la + G::NA * 64;
        const float2* ls = reinterpret_cast<const float2*>(lb + G::NB * 64);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
#pragma unroll
            for (int c = 0; c < G::PB; ++c) wv[p][r][c] = lb[((wr * RT + r) * G::PB + c) * 64 + lane];
            sv[p][r] = ls[(wr * RT + r) * 32 + j];
        }
    };
    // A step is one 32x32 result of one block: its four MFMAs, beside the scale FMAs of the step
    // before and a share of the next row tile's dequantisation.  The group barriers interleave them
    // behind each MFMA, so both pipes run at once.
    f32x16_t d[2];
    half8_t wh[2][2];  // [row tile step parity][half]
    float dsc = 0.0f;
    auto dequant = [&](int p, int b, int r, int h) {
        if constexpr (QT == 0) {
            const uint4 v = wv[p][r][b];
            return h ? q8_to_h8(v.z, v.w) : q8_to_h8(v.x, v.y);
        } else {
            const uint4 v = wv[p][r][0];
            return q4_to_h8(b ? (h ? v.w : v.z) : (h ? v.y : v.x));
        }
    };
    auto scale = [&](int k, int r, int t) {  // the result of step parity k, tile (r, t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][t][i] = fmaf(dsc, d[k][i], acc[r][t][i]);
        // (opaque here and below, or the compiler moves the work of a step past the stage's branches)
        asm volatile("" : "+v"(acc[r][t]));
    };
    auto multiply = [&](int p, int b) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int kw = (b * RT + r) & 1;
#pragma unroll
            for (int t = 0; t < TTW; ++t) {
                const int k = ((b * RT + r) * TTW + t) & 1;
                f32x16_t v = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[b][t][0], wh[kw][0], f32x16_t{}, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[b][t][2], wh[kw][1], v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[b][t][1], wh[kw][0], v, 0, 0, 0);
                d[k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[b][t][3], wh[kw][1], v, 0, 0, 0);
                if (t > 0) scale(k ^ 1, r, t - 1);
                else scale(k ^ 1, r ? r - 1 : RT - 1, TTW - 1);
                dsc = b ? sv[p][r].y : sv[p][r].x;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (t == (h ? TTW - 1 : 0)) {
                        wh[kw ^ 1][h] = r + 1 < RT ? dequant(p, b, r + 1, h) : b ? dequant(p ^ 1, 0, 0, h) : dequant(p, 1, 0, h);
                        asm volatile("" : "+v"(wh[kw ^ 1][h]));
                    }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, TTW > 1 ? 6 : 8, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    for (int st = 0; st < G::D && st < nst; ++st) issue(lds_base + (unsigned)(st * G::U4) * 16u);
    // Entering stage st (and, published in pairs, st + 1): its copies of this wave have landed when at
    // most the younger stages' are outstanding, and every LDS read of this wave is complete; past the
    // barrier that holds for every wave, so the buffers of the PS stages before st take those D
    // further.  No LDS access moves across.
    constexpr int PS = G::PS, D = G::D;
    auto enter = [&](int st) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        wait_copies(nst - PS - st);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    enter(0);
    int buf = 0, left = sl.st, left_g = sl.per;
    read_weights(0, lds);
    read_block(0, lds);
    wh[0][0] = dequant(0, 0, 0, 0);
    wh[0][1] = dequant(0, 0, 0, 1);
    d[1] = f32x16_t{};
    auto stage = [&](int st, int p) {  // p = st % 2, a constant where it is called
        read_block(1, lds + buf * G::U4);
        __builtin_amdgcn_sched_barrier(0);
        multiply(p, 0);
        // the reads above complete here, on every path: behind the branches the compiler would else
        // wait for them again, and with them for the reads issued meanwhile
        __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0(63));
        if (st + 1 < nst) {
            const int next = buf + 1 == D ? 0 : buf + 1;
            const bool publish = PS == 1 || p == 1;
            if (publish) enter(st + 1);
            const uint4* la = lds + next * G::U4;
            read_weights(p ^ 1, la);
            read_block(0, la);
            if (publish && st + D < nst) {
#pragma unroll
                for (int i = 0; i < PS; ++i) issue(lds_base + (unsigned)((buf - (PS - 1 - i)) * G::U4) * 16u);
            }
            buf = next;
            __builtin_amdgcn_sched_barrier(0);
        }
        multiply(p, 1);
        if constexpr (SPLIT != BY_SLICE && RT * TTW <= 2) {
            if (--left == 0) {
                left = sl.st;
                scale(1, RT - 1, TTW - 1);
                dsc = 0.0f;
                d[1] = f32x16_t{};
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int t = 0; t < TTW; ++t) {
                        grp[r][t] = grp[r][t] + acc[r][t];
                        acc[r][t] = f32x16_t{};
                    }
                if (SPLIT == WHOLE && --left_g == 0) {
                    left_g = sl.per;
#pragma unroll
                    for (int r = 0; r < RT; ++r)
#pragma unroll
                        for (int t = 0; t < TTW; ++t) {
                            tot[r][t] = tot[r][t] + grp[r][t];
                            grp[r][t] = f32x16_t{};
                        }
                }
            }
        }
    };
    for (int st = 0; st < nst; st += 2) {  // nst is even (K % 128 == 0)
        stage(st, 0);
        stage(st + 1, 1);
    }
    scale(1, RT - 1, TTW - 1);
    // lane (n = j, g) holds tokens 8u + 4g + (0..3), u < 4, of each token tile
#pragma unroll
    for (int t = 0; t < TTW; ++t) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int m = 32 * (T0 + wt * TTW + t) + 8 * (i / 4) + 4 * g + i % 4;
            if (m >= a.M) continue;
            const float xs = a.xs[m];
            float* yr = SPLIT ? a.part + ((size_t)z * a.M + m) * a.N : a.y + (size_t)m * a.y_stride + a.n_off;
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const int n = 32 * (R0 + wr * RT + r) + j;
                if (n >= a.N) continue;
                const float sum = SPLIT == BY_SLICE ? acc[r][t][i] : grp[r][t][i] + acc[r][t][i];
                yr[n] = SPLIT ? sum : (tot[r][t][i] + sum) * xs;
            }
        }
    }
}

// y[m, n] = xs[m] * the sum over groups, in order, of each group's n partials summed in order
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmArgs a, int n_part, int per) {
    const int m = blockIdx.y, n = blockIdx.x * 256 + threadIdx.x;
    if (n >= a.N) return;
    const float* p = a.part + (size_t)m * a.N + n;
    const size_t step = (size_t)a.M * a.N;
    float t = 0.0f;
    for (int z = 0; z < n_part;) {
        float g = 0.0f;
        for (int e = min(n_part, z + per); z < e; ++z) g = g + p[z * step];
        t = t + g;
    }
    a.y[(size_t)m * a.y_stride + a.n_off + n] = t * a.xs[m];
}

// Row tiles [r_first, r_first + r_count) of the matrix.
template <int QT, int WT, int WR, int TTW, int RT, int SPLIT>
int gemm_launch(const GemmArgs& a, int r_first, int r_count, const Slices& sl, hipStream_t s) {
    using G = GemmStage<QT, WT, WR, TTW, RT>;
    const auto kernel = &mgemm_kernel<QT, WT, WR, TTW, RT, SPLIT>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::BYTES);
    if (attr != hipSuccess) return -2;
    const int mtiles = (a.M + 31) / 32;
    const int rpanels = (r_count + G::BR - 1) / G::BR, tpanels = (mtiles + G::TT - 1) / G::TT;
    const int units = SPLIT ? rpanels * sl.runs(SPLIT) : rpanels;
    const int blocks = 8 * ((units + 7) / 8) * tpanels;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(G::NW * 64), G::BYTES, s, a, r_first, rpanels, tpanels, sl);
    if (SPLIT)
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3((a.N + 255) / 256, a.M), dim3(256), 0, s, a, sl.runs(SPLIT),
                           SPLIT == BY_SLICE ? sl.per : 1);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Rounds that the 32 CUs of an XCD need for `panels` row panels, dealt to the 8 XCDs, times `tpanels`.
int xcd_rounds(int panels, int tpanels) { return ((panels + 7) / 8 * tpanels + 31) / 32; }

// Microseconds of one round of blocks at K = 4096 (Q8, all CUs busy): 128 x 256, 128 x 128 and
// 64 x 128 blocks.  What a launch costs is its rounds times this; only the proportions matter.
constexpr int kRoundWide = 127, kRoundMid = 67, kRoundNarrow = 44;
// and what two groups of slices and the addition of their sums cost beside one of all K (4096 x 4096, 512
// rows: 50 us one block, 51 by group; 4096 x 12288: 145 and 126)
constexpr int kReduce = 14;

// The slices of K, a rule on the matrix's shape alone.  Four or more form two groups.
Slices slices_of(int N, int K) {
    const int p = (N + 127) / 128, q = K / 128;
    const int s = p >= 46 ? 1 : std::max(1, std::min({8, 256 / p, K / kSliceMin}));
    const int len = (q + s - 1) / s;  // slices in units of 128 elements
    const int n = (q + len - 1) / len, per = n >= 4 ? (n + 1) / 2 : n;
    return Slices{n, 2 * len, (n + per - 1) / per, per};
}

// What a block of a launch over several slices runs, where there is scratch for partial sums.
Split split_of(int M, int N, int K, const Slices& sl) {
    const int pn = (N + 127) / 128, mtiles = (M + 31) / 32;
    if (pn * ((mtiles + 1) / 2) <= kSplitPanels) return BY_SLICE;
    // Many rows: 64 x 128 blocks over all of K, or 128 x 128 ones over a group of slices each, which
    // read the LDS half as often per product, and kReduce to add the groups' sums.
    const int whole = xcd_rounds(pn, (mtiles + 1) / 2) * kRoundNarrow * 2;
    const int by_group = xcd_rounds(pn * sl.groups, (mtiles + 3) / 4) * kRoundMid * 2 / sl.groups;
    return sl.groups > 1 && by_group * (K / 128) + 2 * kReduce * 32 < whole * (K / 128) ? BY_GROUP : WHOLE;
}

template <int QT>
int gemm_dispatch(const GemmArgs& a, hipStream_t s) {
    const int rt = (a.N + 31) / 32, mtiles = (a.M + 31) / 32;
    const Slices sl = slices_of(a.N, a.K);
    if (sl.n > 1) {
        const Split split = a.part ? split_of(a.M, a.N, a.K, sl) : WHOLE;
        if (split == BY_SLICE && mtiles <= 1) return gemm_launch<QT, 1, 4, 1, 1, BY_SLICE>(a, 0, rt, sl, s);
        if (split == BY_SLICE) return gemm_launch<QT, 2, 4, 1, 1, BY_SLICE>(a, 0, rt, sl, s);
        if (split == BY_GROUP) return gemm_launch<QT, 2, 4, 2, 1, BY_GROUP>(a, 0, rt, sl, s);
        return gemm_launch<QT, 2, 4, 1, 1, WHOLE>(a, 0, rt, sl, s);
    }
    if (mtiles <= 1) return gemm_launch<QT, 1, 4, 1, 1, WHOLE>(a, 0, rt, sl, s);
    // The block size by the rounds each needs: the last one costs as much as a full one.  Whole rounds
    // of 128 x 256 blocks may leave their remainder to 128 x 128 ones.
    const int tw = (mtiles + 3) / 4, tn = (mtiles + 1) / 2, pw = (rt + 7) / 8, pn = (rt + 3) / 4;
    const int narrow = xcd_rounds(pn, tn) * kRoundNarrow, mid = xcd_rounds(pn, tw) * kRoundMid;
    const int rw = xcd_rounds(pw, tw), wide = rw * kRoundWide;
    const int head = (rw - 1) * 32 / tw * 8;  // panels of the whole rounds
    const int mixed = rw > 1 && head > 0 && head < pw
                          ? xcd_rounds(head, tw) * kRoundWide + xcd_rounds((rt - 8 * head + 3) / 4, tw) * kRoundMid : wide;
    if (narrow <= mid && narrow <= wide && narrow <= mixed) return gemm_launch<QT, 2, 4, 1, 1, WHOLE>(a, 0, rt, sl, s);
    if (mid < wide && mid <= mixed) return gemm_launch<QT, 2, 4, 2, 1, WHOLE>(a, 0, rt, sl, s);
    if (wide <= mixed) return gemm_launch<QT, 2, 4, 2, 2, WHOLE>(a, 0, rt, sl, s);
    const int rc = gemm_launch<QT, 2, 4, 2, 2, WHOLE>(a, 0, 8 * head, sl, s);
    return rc ? rc : gemm_launch<QT, 2, 4, 2, 1, WHOLE>(a, 8 * head, rt - 8 * head, sl, s);
}

}  // namespace

// Row tiles of a panel copy: whole panels of 8 row tiles, so no copy of a block runs past it.
static size_t panel_tiles(int N) { return ((size_t)(N + 31) / 32 + 7) / 8 * 8; }

size_t gemm_q_bytes(int quant, int N, int K) { return panel_tiles(N) * (quant == 0 ? 32 : 16) * K; }

size_t gemm_s_floats(int N, int K) { return panel_tiles(N) * 32 * (K / 32); }

size_t gemm_part_floats(int M, int N, int K) {
    const Slices sl = slices_of(N, K);
    if (sl.n == 1) return 0;
    const int p = (N + 127) / 128;
    return std::max((size_t)sl.n * std::min(M, kSplitPanels / p * 64), (size_t)(sl.groups > 1 ? sl.groups * M : 0)) * N;
}

int gemm_split(int M, int N, int K) {
    const Slices sl = slices_of(N, K);
    return sl.n > 1 ? split_of(M, N, K, sl) : WHOLE;
}

int launch_panel_pack(int quant, int N, int K, const void* q, const float* s, void* qp, float* sp, hipStream_t st) {
    if (K % 128 || N <= 0 || (quant != 0 && quant != 1)) return -1;
    const size_t rt = (size_t)(N + 31) / 32;
    const size_t nq = rt * (quant == 0 ? K / 32 : K / 64) * 64;
    const size_t ns = rt * (K / 64) * 32;
    hipLaunchKernelGGL(panel_pack_q_kernel, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, st, quant, N, K,
                       (const uint8_t*)q, (uint8_t*)qp, nq);
    hipLaunchKernelGGL(panel_pack_s_kernel, dim3((unsigned)((ns + 255) / 256)), dim3(256), 0, st, N, K, s, sp, ns);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// token fragments in whole 128-token panels, the widest token panel of a block
size_t frags_bytes(int M, int K) { return (size_t)((M + 127) / 128) * 128 * K * 4; }

int launch_rows_to_frags(const RowsArgs& a, hipStream_t s) {
    if (a.M <= 0 || a.K % 128 || !a.frags || !a.xs) return -1;
    if (a.mode == ROWS_GNORM && (a.K % 128 || !a.ssq)) return -1;
    const int mpad = (a.M + 31) / 32 * 32;
    const int gpt = (a.K / 8 + kRowThreads - 1) / kRowThreads;
    if (gpt <= 2) hipLaunchKernelGGL(rows_to_frags_kernel<2>, dim3(mpad), dim3(kRowThreads), 0, s, a);
    else if (gpt <= 4) hipLaunchKernelGGL(rows_to_frags_kernel<4>, dim3(mpad), dim3(kRowThreads), 0, s, a);
    else if (gpt <= 6) hipLaunchKernelGGL(rows_to_frags_kernel<6>, dim3(mpad), dim3(kRowThreads), 0, s, a);
    else if (gpt <= 8) hipLaunchKernelGGL(rows_to_frags_kernel<8>, dim3(mpad), dim3(kRowThreads), 0, s, a);
    else return -1;  // rows longer than 16384
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_mgemm(const GemmArgs& a, int quant, hipStream_t s) {
    if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.K % 128 || !a.wq || !a.ws || !a.frags || !a.xs || !a.y) return -1;
    return quant == 0 ? gemm_dispatch<0>(a, s) : gemm_dispatch<1>(a, s);
}

}  // namespace snl
