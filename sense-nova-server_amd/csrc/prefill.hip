// Per-token kernels of the chunked prefill pass (up to 512 token rows per launch): the embedding
// gather, the mHC token coefficients, and the Gated DeltaNet over a chunk.
//
// DeltaNet (src/shaders/linear.wgsl:38-140).  The causal conv, SiLU, q/k L2 normalisation and the
// per-token gates do not depend on the recurrent state, so they run for every token of the chunk
// at once (dn_conv_kernel, one block per (token, head)); the conv state then takes the chunk's
// last three inputs (dn_conv_state_kernel).  The recurrence itself takes 16 tokens at a time in the
// blocked form of the delta rule, as f32 matrix products: dn_block_kernel forms each block's
// state-independent matrices, dn_recur_kernel runs the blocks in order, 8 blocks of 4 waves per value
// head, each owning 16 state columns in registers.  The state is updated in place in the current slot
// (a prefill pass has no checkpoint).
#include "common.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace snl {

namespace {

constexpr int DK = 128, DV = 128;
// the recurrence: 8 blocks of 16 state columns per value head, 4 waves each (one wave per SIMD
// on every CU for the 32 value heads of the 9B shape)
constexpr int kCG = kDeltaPrefillGroups, kCols = DV / kCG;
constexpr int kThreads = 256, kWaves = kThreads / 64;
static_assert(kCols == 16 && kWaves * 32 == DK, "a wave's rows are two 16 x 16 MFMA tiles");

// x[m, 0:h] = dequant(embed[tokens[m]]), x[m, h:2h] = 0 (src/engine.rs:777-790)
__global__ __launch_bounds__(256) void pf_embed_kernel(const uint32_t* tokens, const int8_t* eq, const float* es,
                                                        int vocab, int h, float* x) {
    const int m = blockIdx.x;
    uint32_t tok = tokens[m];
    if (tok >= (uint32_t)vocab) tok = 0;  // the host rejects out-of-range ids before launching
    const int8_t* q = eq + (size_t)tok * h;
    const float* s = es + (size_t)tok * (h / 32);
    float* xr = x + (size_t)m * 2 * h;
    for (int i = threadIdx.x; i < h; i += 256) {
        xr[i] = (float)q[i] * s[i >> 5];
        xr[h + i] = 0.0f;
    }
}

// coef[m] = mhc_coefficients of the token's router sums part[m][0..8] (layers.wgsl:94-126)
__global__ __launch_bounds__(64) void mhc_coef_kernel(const float* part, const float* w, int d, int iterations,
                                                       float* coef, int M) {
    const int m = blockIdx.x * 64 + threadIdx.x;
    if (m >= M) return;
    mhc_coefficients(part + (size_t)m * 9, w, d, iterations, coef + (size_t)m * 8);
}

// Block (token m, slot): slots [0, n_k) the q heads, [n_k, 2n_k) the k heads, then the v heads.
// 128 threads, one channel each (linear.wgsl:38-66, :104-117).
__global__ __launch_bounds__(128) void dn_conv_kernel(DnPrefillArgs a) {
    __shared__ float red[2];
    const int m = blockIdx.x, slot = blockIdx.y, tid = threadIdx.x;
    const int n_k = a.n_k, n_v = a.n_v, cd = a.conv_dim, key_dim = n_k * DK;
    const int kind = slot < n_k ? 0 : slot < 2 * n_k ? 1 : 2;
    const int head = kind == 0 ? slot : kind == 1 ? slot - n_k : slot - 2 * n_k;
    const int ch = kind == 0 ? head * DK + tid : kind == 1 ? key_dim + head * DK + tid : 2 * key_dim + head * DV + tid;
    const float4 w = *reinterpret_cast<const float4*>(a.lw + (size_t)ch * 4);
    // input t of the chunk: proj row t, or conv state row 3 + t for t < 0 (oldest first)
    float in[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = m - 3 + i;
        in[i] = t >= 0 ? a.proj[(size_t)t * a.proj_stride + ch] : a.conv_state[(size_t)(3 + t) * cd + ch];
    }
    const float o = ((w.x * in[0] + w.y * in[1]) + w.z * in[2]) + w.w * in[3];
    const float v = o / (1.0f + expf(-o));
    if (kind == 2) {
        a.v[((size_t)m * n_v + head) * DV + tid] = v;
        const float z = a.proj[(size_t)m * a.proj_stride + cd + head * DV + tid];
        a.gz[((size_t)m * n_v + head) * DV + tid] = z / (1.0f + expf(-z));
        if (tid == 0) {  // linear.wgsl:113-117
            const float* lwp = a.lw + (size_t)cd * 4;
            const float* prow = a.proj + (size_t)m * a.proj_stride;
            const int b_off = cd + n_v * DV, a_off = b_off + n_v;
            a.beta[(size_t)m * n_v + head] = 1.0f / (1.0f + expf(-prow[b_off + head]));
            const float araw = prow[a_off + head] + lwp[n_v + head];
            const float sp = araw <= 20.0f ? logf(1.0f + expf(araw)) : araw;
            a.decay[(size_t)m * n_v + head] = expf(-expf(lwp[head]) * sp);
        }
        return;
    }
    // L2 normalisation over the head's 128 channels (two wave sums, added in wave order)
    const float s = wave_sum(v * v);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (kind == 0) {
        const float qs = (1.0f / sqrtf((red[0] + red[1]) + 1e-6f)) * (1.0f / sqrtf((float)DK));
        a.q[((size_t)m * n_k + head) * DK + tid] = v * qs;
    } else {
        const float ks = 1.0f / sqrtf((red[0] + red[1]) + 1e-6f);
        a.k[((size_t)m * n_k + head) * DK + tid] = v * ks;
    }
}

// Blocked recurrence: the chunk's tokens go through the state kBlk = 16 at a time.  With decays g_b,
// G_b = g_0 ... g_b and P_bc = g_{c+1} ... g_b inside a block, token b sees the state
// G_b S + sum_{c<b} P_bc k_c u_c^T, so the deltas (linear.wgsl:118-136) solve
//   u_b + beta_b sum_{c<b} P_bc (k_c . k_b) u_c = beta_b (v_b - G_b S^T k_b),
// a unit lower triangular system whose inverse T does not depend on the state or on the column:
//   U = T diag(beta) (V - diag(G) K S),
//   O = diag(G) Q S + A U with A_bc = P_bc (k_c . q_b), c <= b,
//   S := G_last S + sum_c P_last,c k_c u_c^T.
// dn_block_kernel forms T diag(beta), A, G and P_last for every block of the chunk at once, one
// block of 64 threads per (16 tokens, key head); the recurrence is then matrix products.
constexpr int kBlk = 16;
struct DnBlock {  // of one (block, value head)
    float tb[kBlk][kBlk], a[kBlk][kBlk];
    float g[kBlk], pl[kBlk];
};
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef double f64x4_t __attribute__((ext_vector_type(4)));

// acc += X Y^T over 16 columns of both: xv / yv hold columns 4g .. 4g + 3 of the lane's row l % 16
// (v_mfma_f32_16x16x4_f32, the 4 lane groups' g as its K); acc row 4g + i, column l % 16
__device__ __forceinline__ f32x4_t mfma16(const float4& xv, const float4& yv, f32x4_t acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv.x, yv.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv.y, yv.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv.z, yv.z, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(xv.w, yv.w, acc, 0, 0, 0);
}
__device__ __forceinline__ float4 as_float4(f32x4_t v) { return make_float4(v[0], v[1], v[2], v[3]); }

// L X of a lower triangular L (lv: columns 4g .. 4g + 3 of row l % 16) and X in accumulator layout
// (row 4g + i).  The product adds 0 x the rows past a row's own, which is NaN where such a row is not
// finite: then each row is formed again with those rows taken as 0, so a token never sees a later one.
// (The check runs beside the product's MFMAs: 512 tokens of 32 heads, the conv included, 94 us without it,
// 104 with it made before them and the 16 rows unrolled, 93 so.)
__device__ __forceinline__ f32x4_t lower16(const float4& lv, f32x4_t x, int g) {
    f32x4_t out = mfma16(lv, as_float4(x), f32x4_t{});
    const float mag = (fabsf(x[0]) + fabsf(x[1])) + (fabsf(x[2]) + fabsf(x[3]));
    if (__any(!(mag < INFINITY))) {
#pragma unroll 1
        for (int b = 0; b < 16; ++b) {
            f32x4_t xb;
#pragma unroll
            for (int i = 0; i < 4; ++i) xb[i] = 4 * g + i <= b ? x[i] : 0.0f;
            const f32x4_t y = mfma16(lv, as_float4(xb), f32x4_t{});
#pragma unroll
            for (int i = 0; i < 4; ++i) out[i] = 4 * g + i == b ? y[i] : out[i];
        }
    }
    return out;
}

__global__ __launch_bounds__(64) void dn_block_kernel(DnPrefillArgs a, int M) {
    __shared__ float kk[kBlk][kBlk + 1], kq[kBlk][kBlk + 1], lw[4][kBlk][kBlk + 1];
    const int blk = blockIdx.x, kh = blockIdx.y, lane = threadIdx.x, n_k = a.n_k, n_v = a.n_v, group = n_v / n_k;
    const int c = lane & 15, g = lane >> 4;
    const int t = blk * kBlk + c;
    const float4* kp = reinterpret_cast<const float4*>(a.k + ((size_t)min(t, M - 1) * n_k + kh) * DK) + g;
    const float4* qp = reinterpret_cast<const float4*>(a.q + ((size_t)min(t, M - 1) * n_k + kh) * DK) + g;
    // In 64 bits: the deltas take differences of rows that are alike, so what rounding leaves in k . k and
    // q . k comes back enlarged (v_mfma_f64_16x16x4_f64: row 4i + g, column l % 16; see dn_recur_kernel)
    f64x4_t dk = {}, dq = {};
#pragma unroll
    for (int s = 0; s < DK / 16; ++s) {
        const float4 k4 = kp[4 * s], q4 = qp[4 * s];
        const float kv[4] = {k4.x, k4.y, k4.z, k4.w}, qv[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            dk = __builtin_amdgcn_mfma_f64_16x16x4f64((double)kv[i], (double)kv[i], dk, 0, 0, 0);
            dq = __builtin_amdgcn_mfma_f64_16x16x4f64((double)qv[i], (double)kv[i], dq, 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        kk[4 * i + g][c] = (float)dk[i];  // k_b . k_c
        kq[4 * i + g][c] = (float)dq[i];  // q_b . k_c
    }
    __syncthreads();
    // lane group g takes value heads g, g + 4, ... of the key head, lane c column c of its matrices
    // (tokens past the chunk: decay 1, beta 0, so their columns of T diag(beta) are 0)
    for (int h0 = 0; h0 < group; h0 += 4) {
        const bool live = h0 + g < group;
        const int h = kh * group + min(h0 + g, group - 1);
        float tcol[kBlk];
        const float beta_c = t < M ? a.beta[(size_t)t * n_v + h] : 0.0f;
        const float dec_c = t < M ? a.decay[(size_t)t * n_v + h] : 1.0f;
        DnBlock* out = reinterpret_cast<DnBlock*>(a.blocks) + (size_t)blk * n_v + h;
        float p = 1.0f, gp = 1.0f;
#pragma unroll
        for (int b = 0; b < kBlk; ++b) {
            const float gb = __shfl(dec_c, (lane & 48) + b), bb = __shfl(beta_c, (lane & 48) + b);
            p = b > c ? p * gb : 1.0f;  // P_bc
            gp = b <= c ? gp * gb : gp;
            lw[g][b][c] = b > c ? bb * (p * kk[b][c]) : 0.0f;
            if (live) out->a[b][c] = b >= c ? p * kq[b][c] : 0.0f;
        }
        if (live) {
            out->g[c] = gp;
            out->pl[c] = p;
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < kBlk; ++b) {
            float v = b == c ? 1.0f : 0.0f;
#pragma unroll
            for (int j = 0; j < b; ++j) v = fmaf(-lw[g][b][j], tcol[j], v);
            tcol[b] = v;
            if (live) out->tb[b][c] = b >= c ? v * beta_c : 0.0f;  // (0 also where a later token's beta is NaN)
        }
        __syncthreads();
    }
}

// conv state := the chunk's last three inputs (from the old state when the chunk is shorter)
__global__ __launch_bounds__(256) void dn_conv_state_kernel(DnPrefillArgs a, int M) {
    const int ch = blockIdx.x * 256 + threadIdx.x;
    const int cd = a.conv_dim;
    if (ch >= cd) return;
    float r[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int t = M - 3 + i;
        r[i] = t >= 0 ? a.proj[(size_t)t * a.proj_stride + ch] : a.conv_state[(size_t)(3 + t) * cd + ch];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) a.conv_state[(size_t)i * cd + ch] = r[i];
}

// The recurrence over the chunk, kCG blocks of 16 state columns per value head.  Wave w holds rows
// 32w .. 32w + 31 of the block's columns as two MFMA accumulators (row 4g + i, column l % 16), which
// are also the B operands of K S and Q S (K index g, one MFMA per i).  Per 16 tokens: each wave's
// share of K S and Q S, their sum over the waves through LDS, U by every wave, the output by one
// wave, the state update.  All products run on v_mfma_f32_16x16x4_f32.  A wave reads its own inputs,
// two blocks ahead of the one computed.
// What bounds it: the chain through a block (two products, an exchange between the waves and another
// product, 1.6 us per 16 tokens).  512 tokens of 32 heads take 55 us + 8 in dn_block_kernel; on the
// vector ALUs, 4 tokens at a time with every row sum reduced across lanes, they took 154 + 5.
// Rounding: each wave's products are sums of 16 from zero, added in pairs, then to the decayed state or the
// value in one fma.  Against 64 bits (17 / 512 tokens, error of the outputs, decays near 1): 1.1e-7 / 2.0e-7;
// with k . k as one f32 sum of 128 and the state as accumulator of its products 1.7e-7 / 2.9e-7, and
// 2.7e-7 / 3.1e-7 against 1.3e-7 / 1.6e-7 where keys are alike; token by token in blocks of 4 on the vector
// ALUs 1.3e-7 / 2.8e-7 and 1.0e-7 / 1.5e-7.  The time is the same.
struct RecurIn {
    float4 k[2], q[2];   // token l % 16, rows 32w + 16t + 4g ..
    float kt[2][4];      // token 4g + i, row 32w + 16t + l % 16
    float v[4], gz[4];   // token 4g + i, column l % 16
    float4 tb, a, g, pl; // row l % 16, columns 4g ..; tokens 4g ..
    float glast;
};

__global__ __launch_bounds__(kThreads) void dn_recur_kernel(DnPrefillArgs a, int M) {
    __shared__ f32x4_t part[2][2][kWaves][64];  // [block parity][K S, Q S][wave][lane]
    const int h = blockIdx.x / kCG, cg = blockIdx.x % kCG;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int n_k = a.n_k, n_v = a.n_v, kh = h / (n_v / n_k);
    const int col = cg * kCols + c, r0 = 32 * wave;
    float* S = a.state + (size_t)h * DK * DV + col;
    f32x4_t s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[t][i] = S[(size_t)(r0 + 16 * t + 4 * g + i) * DV];
    const float norm_w = a.lw[(size_t)a.conv_dim * 4 + 2 * n_v + col];
    const int nblk = (M + kBlk - 1) / kBlk;

    // Tokens past the chunk read the last one's rows: their columns of T diag(beta) are 0, so they
    // leave the state as it is, and their outputs are not stored.
    auto load = [&](int blk, RecurIn& d) {
        if (blk >= nblk) return;
        const int tc = min(blk * kBlk + c, M - 1);
        const float4* kp = reinterpret_cast<const float4*>(a.k + ((size_t)tc * n_k + kh) * DK + r0) + g;
        const float4* qp = reinterpret_cast<const float4*>(a.q + ((size_t)tc * n_k + kh) * DK + r0) + g;
        const DnBlock* b = reinterpret_cast<const DnBlock*>(a.blocks) + (size_t)blk * n_v + h;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            d.k[t] = kp[4 * t];
            d.q[t] = qp[4 * t];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tr = min(blk * kBlk + 4 * g + i, M - 1);
            const float* kr = a.k + ((size_t)tr * n_k + kh) * DK + r0 + c;
            d.kt[0][i] = kr[0];
            d.kt[1][i] = kr[16];
            d.v[i] = a.v[((size_t)tr * n_v + h) * DV + col];
            d.gz[i] = a.gz[((size_t)tr * n_v + h) * DV + col];
        }
        d.tb = reinterpret_cast<const float4*>(b->tb[c])[g];
        d.a = reinterpret_cast<const float4*>(b->a[c])[g];
        d.g = reinterpret_cast<const float4*>(b->g)[g];
        d.pl = reinterpret_cast<const float4*>(b->pl)[g];
        d.glast = b->g[kBlk - 1];
    };
    auto wave_parts = [&](int par, int which) {  // the waves' shares of a product, added in pairs
        const auto& p = part[par][which];
        return (p[0][lane] + p[1][lane]) + (p[2][lane] + p[3][lane]);
    };
    auto step = [&](int blk, const RecurIn& d) {
        const int par = blk & 1;
        f32x4_t ks[2], qs[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) ks[t] = mfma16(d.k[t], as_float4(s[t]), f32x4_t{});
#pragma unroll
        for (int t = 0; t < 2; ++t) qs[t] = mfma16(d.q[t], as_float4(s[t]), f32x4_t{});
        part[par][0][wave][lane] = ks[0] + ks[1];
        part[par][1][wave][lane] = qs[0] + qs[1];
        // (one barrier a block: the other parity's sums are read before the next one)
        __syncthreads();
        f32x4_t z = wave_parts(par, 0);
        const float gv[4] = {d.g.x, d.g.y, d.g.z, d.g.w}, pl[4] = {d.pl.x, d.pl.y, d.pl.z, d.pl.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) z[i] = fmaf(-gv[i], z[i], d.v[i]);
        const f32x4_t u = lower16(d.tb, z, g);
        f32x4_t pu;
#pragma unroll
        for (int i = 0; i < 4; ++i) pu[i] = pl[i] * u[i];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const f32x4_t ku = mfma16(make_float4(d.kt[t][0], d.kt[t][1], d.kt[t][2], d.kt[t][3]), as_float4(pu), f32x4_t{});
#pragma unroll
            for (int i = 0; i < 4; ++i) s[t][i] = fmaf(d.glast, s[t][i], ku[i]);
        }
        if (wave == (blk & (kWaves - 1))) {  // the outputs: the waves take turns
            f32x4_t o = wave_parts(par, 1);
            const f32x4_t au = lower16(d.a, u, g);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = fmaf(gv[i], o[i], au[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = blk * kBlk + 4 * g + i;
                float q2 = o[i] * o[i];
                q2 = xor_sum<1>(q2);
                q2 = xor_sum<2>(q2);
                q2 = xor_sum<4>(q2);
                q2 = xor_sum<8>(q2);
                if (m >= M) continue;
                a.out[(size_t)m * n_v * DV + h * DV + col] = (o[i] * norm_w) * d.gz[i];
                if (c == 0) a.ssq[((size_t)m * n_v + h) * kCG + cg] = q2;
            }
        }
    };
    RecurIn d0, d1, d2;
    load(0, d0);
    load(1, d1);
    for (int blk = 0; blk < nblk; blk += 3) {
        load(blk + 2, d2);
        step(blk, d0);
        if (blk + 1 >= nblk) break;
        load(blk + 3, d0);
        step(blk + 1, d1);
        if (blk + 2 >= nblk) break;
        load(blk + 4, d1);
        step(blk + 2, d2);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[(size_t)(r0 + 16 * t + 4 * g + i) * DV] = s[t][i];
}

}  // namespace

int launch_embed_tokens(const uint32_t* tokens, const int8_t* eq, const float* es, int vocab, int h, float* x, int M,
                        hipStream_t s) {
    if (M < 1) return -1;
    hipLaunchKernelGGL(pf_embed_kernel, dim3(M), dim3(256), 0, s, tokens, eq, es, vocab, h, x);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_mhc_coef(const float* part, const float* w, int h, int iterations, float* coef, int M, hipStream_t s) {
    if (M < 1) return -1;
    hipLaunchKernelGGL(mhc_coef_kernel, dim3((M + 63) / 64), dim3(64), 0, s, part, w, 2 * h, iterations, coef, M);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

size_t dn_block_floats(int M, int n_v) { return (size_t)((M + kBlk - 1) / kBlk) * n_v * (sizeof(DnBlock) / sizeof(float)); }

int launch_deltanet_prefill(const DnPrefillArgs& a, int M, hipStream_t s) {
    if (M < 1 || M > SNL_PF_M || a.n_k < 1 || a.n_v % a.n_k || !a.blocks) return -1;
    hipLaunchKernelGGL(dn_conv_kernel, dim3(M, 2 * a.n_k + a.n_v), dim3(128), 0, s, a);
    hipLaunchKernelGGL(dn_conv_state_kernel, dim3((a.conv_dim + 255) / 256), dim3(256), 0, s, a, M);
    hipLaunchKernelGGL(dn_block_kernel, dim3((M + kBlk - 1) / kBlk, a.n_k), dim3(64), 0, s, a, M);
    hipLaunchKernelGGL(dn_recur_kernel, dim3(a.n_v * kCG), dim3(kThreads), 0, s, a, M);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace snl
