// Gated GQA attention over a prefill chunk (src/shaders/attention.wgsl: prep :59-127, attend
// :129-246, combine :248-269), on the matrix cores.
//
// prep: block (slot, token) as in the decode kernel: RMSNorm (1 + w) of each q / k head, partial
// rotate-half RoPE at the token's rotary position, q rows to qbuf (f32), k / v rows into the f16
// cache at the token's cache position.
//
// attend: block (kv head, 16 queries, key part), wave w = query head 4*kv + w of the GQA group;
// the block streams its part of the keys [0, last query's position] in steps of 32 through LDS (K rows and V rows, each staged with 16-byte copies; the V^T fragments come
// back from the V rows through the transposing LDS read, two 8-byte reads per fragment),
// shared by the group's 4 heads.
//   scores  S^T = K Q^T on v_mfma_f32_16x16x32_f16: A = 16 keys x 32 dims of K (exact f16),
//           B = the query's dims split into f16 hi + lo under a per-query power of two, so the
//           f32 score carries the decode kernel's precision; lane (query j, group g) ends with
//           keys 4g..4g+3 of each 16-key half;
//   softmax online per query (running max, rescaled partial sums), keys past the query's own
//           position weigh 0;
//   values  O^T += V^T P^T: B = the lane's own 8 probabilities as f16 hi + lo (keys 4g..4g+3 and
//           16+4g..16+4g+3, the same order in the V^T fragment), A = 16 dims x those keys.
//
// A query's keys are summed the same way whatever shares its pass: every leaf of 256 keys (128 within the
// cache's first 1024) from zero, the leaves of 1024 keys to a node, two nodes to a top and the tops one
// after the other, each time merged in order (merge()).  A part is a leaf, a node or a top (part_level),
// so a block merges what lies inside its part and pf_combine_kernel the rest, by the same steps; a leaf
// past a query's position weighs 0 and changes nothing.  Each part leaves (unnormalised output, running max,
// sum); with one part the output is divided by the softmax sum and multiplied by the sigmoid gate at
// once, as in combine.
#include <float.h>

#include <algorithm>
#include <hip/hip_fp16.h>

#include "common.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace snl {

namespace {

constexpr int HD = 256, G = 4;
constexpr int QTILE = 16, KB = 32;
// Keys summed from zero, and merged.  The first 1024 keys have shorter leaves, for the short contexts whose
// blocks are few: 45 rows over 260 keys 32 us a call in leaves of 256, 25 in leaves of 128, over 1045 keys 35
// and 29.  Throughout they would double the merges of long parts (512 rows over 12800 keys 355 us, 381).
constexpr int LEAF = 256, FINE = 128, FINE_KEYS = 1024, NODE = 1024, TOP = 2 * NODE;
constexpr int kNodeLeaves = NODE / LEAF, kFirstLeaves = kNodeLeaves + FINE_KEYS / FINE - FINE_KEYS / LEAF;
constexpr int PSTRIDE = HD + 4;  // floats of a part's partial: output, running max, sum (16-byte rows)
constexpr int KROW = HD + 8;  // K tile row (halfs): 528 bytes keeps the 16 rows of a read on distinct banks
constexpr int VROW = HD + 16;  // V row (halfs): 544 bytes, so the 4 rows of a transposed read hit distinct banks

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// the weights of two partials with running maxima ma and mb in their merge (one of them is 1); ma becomes
// the merge's
__device__ __forceinline__ void merge_weights(float& ma, float mb, float& fa, float& fb) {
    const float e = expf(-fabsf(ma - mb));
    fa = ma >= mb ? 1.0f : e;
    fb = ma >= mb ? e : 1.0f;
    ma = fmaxf(ma, mb);
}
__device__ __forceinline__ float merge(float a, float fa, float b, float fb) { return fmaf(b, fb, a * fa); }
__device__ __forceinline__ f32x4_t merge4(f32x4_t a, float fa, f32x4_t b, float fb) {
    return f32x4_t{merge(a[0], fa, b[0], fb), merge(a[1], fa, b[1], fb), merge(a[2], fa, b[2], fb),
                   merge(a[3], fa, b[3], fb)};
}

// the first key of part p, and the parts of `keys` keys, where a part is a leaf, a node or a top
__host__ __device__ constexpr int part_key(int level, int p) {
    if (level) return p * (level > 1 ? TOP : NODE);
    return p < FINE_KEYS / FINE ? p * FINE : FINE_KEYS + (p - FINE_KEYS / FINE) * LEAF;
}
__host__ __device__ constexpr int part_count(int level, int keys) {
    if (level) return (keys + (level > 1 ? TOP : NODE) - 1) / (level > 1 ? TOP : NODE);
    return keys <= FINE_KEYS ? (keys + FINE - 1) / FINE : FINE_KEYS / FINE + (keys - FINE_KEYS + LEAF - 1) / LEAF;
}
__device__ __forceinline__ int leaf_end(int key) { return key + (key < FINE_KEYS ? FINE : LEAF); }

__global__ __launch_bounds__(256) void pf_prep_kernel(AttnArgs a, const PrefillDev* st) {
    __shared__ float sh[HD];
    __shared__ float red[4];
    const int slot = blockIdx.x, m = blockIdx.y, d = threadIdx.x;
    const int pos = st->pos0 + m;
    const int q_dim = a.n_heads * HD, kv_dim = a.n_kv * HD;
    const float* row = a.proj + (size_t)m * a.proj_stride;
    if (slot >= a.n_heads + a.n_kv) {
        const int kh = slot - a.n_heads - a.n_kv;
        const float v = row[2 * q_dim + kv_dim + kh * HD + d];
        a.vcache[(size_t)pos * kv_dim + kh * HD + d] = __half_as_ushort(__float2half_rn(v));
        return;
    }
    const bool is_q = slot < a.n_heads;
    float v = is_q ? row[slot * 2 * HD + d] : row[2 * q_dim + (slot - a.n_heads) * HD + d];
    const float total = block_sum<256>(v * v, red);
    v = (v * (1.0f / sqrtf(total / (float)HD + a.eps))) * (1.0f + a.norms[(is_q ? 0 : HD) + d]);
    sh[d] = v;
    __syncthreads();
    const int half = a.rot_dim / 2;
    if (d < a.rot_dim) {
        const int fi = d % half;
        const float inv_freq = powf(a.rope_theta, -(float)(2 * fi) / (float)a.rot_dim);
        const uint32_t* rp = st->rpos[m];
        uint32_t rot_pos = rp[0];
        if (fi % 3 == 1 && (uint32_t)fi < (a.mrope >> 16)) rot_pos = rp[1];
        else if (fi % 3 == 2 && (uint32_t)fi < (a.mrope & 0xFFFFu)) rot_pos = rp[2];
        const float ang = (float)rot_pos * inv_freq;
        const float cs = cosf(ang), sn = sinf(ang);
        v = d < half ? sh[d] * cs - sh[d + half] * sn : sh[d] * cs + sh[d - half] * sn;
    }
    if (is_q) {
        a.qbuf[(size_t)m * q_dim + slot * HD + d] = v;
    } else {
        const int kh = slot - a.n_heads;
        a.kcache[(size_t)pos * kv_dim + kh * HD + d] = __half_as_ushort(__float2half_rn(v));
    }
}

// A node's sums stay beside the leaf's: NR of its 16 output tiles in registers, the others in LDS, as much
// of each as two blocks on a CU have.  A top's first node waits in the block's own partial.
template <int LEVEL>
__global__ __launch_bounds__(256, 2) void pf_attend_kernel(AttnArgs a, const PrefillDev* st, int M, int row0, float* part,
                                                           int parts) {
    constexpr int NR = LEVEL ? 5 : 0;
    __shared__ __align__(16) f32x4_t node_lds[LEVEL ? 16 - NR : 1][LEVEL ? 256 : 1];
    __shared__ __align__(16) _Float16 ks[KB * KROW];
    __shared__ __align__(16) _Float16 vs[KB * VROW];
    const int kh = blockIdx.x, q0 = row0 + blockIdx.y * QTILE;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hh = kh * G + w;
    const int pos0 = st->pos0;
    const int qn = min(QTILE, M - q0);
    const int kend = pos0 + q0 + qn;  // keys of the block's last query
    const int p = blockIdx.z;
    const int kfirst = part_key(LEVEL, p), kstop = min(kend, part_key(LEVEL, p + 1));
    if (kfirst >= kend) return;
    const int q_dim = a.n_heads * HD, kv_dim = a.n_kv * HD;
    const int j = lane & 15, g = lane >> 4;
    const int mq = q0 + j;
    const bool qvalid = j < qn;
    const int qlim = pos0 + mq;  // the last key this lane's query sees

    // ---- the query as B fragments (dims 32s + 8g + i), hi + lo under a power of two ----
    float qv[8][8];
    float amax = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const float4* qp = reinterpret_cast<const float4*>(a.qbuf + (size_t)(qvalid ? mq : q0) * q_dim + hh * HD + 32 * s + 8 * g);
        const float4 u0 = qp[0], u1 = qp[1];
        qv[s][0] = u0.x, qv[s][1] = u0.y, qv[s][2] = u0.z, qv[s][3] = u0.w;
        qv[s][4] = u1.x, qv[s][5] = u1.y, qv[s][6] = u1.z, qv[s][7] = u1.w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (!qvalid) qv[s][i] = 0.0f;
            amax = fmaxf(amax, fabsf(qv[s][i]));
        }
    }
    amax = xor_max<32>(xor_max<16>(amax));
    const int e = amax > 0.0f ? max(ilogbf(amax) - 14, -110) : 0;
    const float down = ldexpf(1.0f, -e), up = ldexpf(1.0f, e) * a.scale;
    half8_t qh[8], ql[8];
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float v = qv[s][i] * down;
            const _Float16 hv = (_Float16)v;
            qh[s][i] = hv;
            ql[s][i] = (_Float16)(v - (float)hv);
        }

    f32x4_t o[16];
    float mrun, lpart, l;
    f32x4_t node[NR ? NR : 1];
    float node_m = 0.0f, node_l = 0.0f, top_m = 0.0f, top_l = 0.0f;
    // (lanes past the pass's rows read the first row's partial and write none)
    float* pp = part + (((size_t)((qvalid ? mq : q0) - row0) * a.n_heads + hh) * parts + p) * PSTRIDE;
    f32x4_t* prow = reinterpret_cast<f32x4_t*>(pp + 4 * g);  // this lane's 16 bytes of output tile dt at prow[4 dt]
    const uint16_t* kc = a.kcache + kh * HD;
    const uint16_t* vc = a.vcache + kh * HD;

    // K and V rows of a step: thread (key t >> 3, 32 dims), the next step's loaded while this one's
    // values are multiplied
    uint4 kr[4], vr[4];
    auto load_rows = [&](int kb) {
        const int kk = kb + (tid >> 3), seg = tid & 7;
#pragma unroll
        for (int i = 0; i < 4; ++i) kr[i] = vr[i] = make_uint4(0u, 0u, 0u, 0u);
        if (kk < kstop) {
            const uint4* ksrc = reinterpret_cast<const uint4*>(kc + (size_t)kk * kv_dim + seg * 32);
            const uint4* vsrc = reinterpret_cast<const uint4*>(vc + (size_t)kk * kv_dim + seg * 32);
#pragma unroll
            for (int i = 0; i < 4; ++i) kr[i] = ksrc[i];
#pragma unroll
            for (int i = 0; i < 4; ++i) vr[i] = vsrc[i];
        }
    };
    load_rows(kfirst);
    auto step = [&](int kb) {
        __syncthreads();  // the previous step's tiles are consumed
        {
            const int key = tid >> 3, seg = tid & 7;
            uint4* kdst = reinterpret_cast<uint4*>(ks + key * KROW + seg * 32);
            uint4* vdst = reinterpret_cast<uint4*>(vs + key * VROW + seg * 32);
#pragma unroll
            for (int i = 0; i < 4; ++i) kdst[i] = kr[i];
#pragma unroll
            for (int i = 0; i < 4; ++i) vdst[i] = vr[i];
        }
        __syncthreads();

        // ---- scores: two 16-key halves ----
        f32x4_t sc[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            f32x4_t c = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const half8_t kf = *reinterpret_cast<const half8_t*>(ks + (16 * kt + j) * KROW + 32 * s + 8 * g);
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qh[s], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, ql[s], c, 0, 0, 0);
            }
            sc[kt] = c;
        }
        // ---- online softmax for this lane's query ----
        float val[8];
        bool ok[8];
        float bmax = -1e30f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int kk = kb + 16 * kt + 4 * g + r;
                const int i = 4 * kt + r;
                ok[i] = qvalid && kk <= qlim && kk < kstop;
                val[i] = sc[kt][r] * up;
                if (ok[i]) bmax = fmaxf(bmax, val[i]);
            }
        bmax = xor_max<32>(xor_max<16>(bmax));
        const float mnew = fmaxf(mrun, bmax);
        const float factor = expf(mrun - mnew);
        half8_t ph, pl;
        float psum = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float p = ok[i] ? expf(val[i] - mnew) : 0.0f;
            psum = psum + p;
            const _Float16 hv = (_Float16)p;
            ph[i] = hv;
            pl[i] = (_Float16)(p - (float)hv);
        }
        lpart = lpart * factor + psum;
        mrun = mnew;
        // ---- values ----
        load_rows(kb + KB);
#pragma unroll
        for (int dt = 0; dt < 16; ++dt) {
            o[dt] = o[dt] * factor;
            // transposed reads (ds_read_b64_tr_b16): in each 16-lane group, lane 4a + b receives
            // element b of the 8 bytes addressed by lanes a, a + 4, a + 8, a + 12; lane s
            // addresses key 4g + s / 4 (then 16 + 4g + s / 4), dims 16 dt + 4 (s % 4), so lane j
            // receives dim 16 dt + j of keys 4g .. 4g + 3 (then 16 + 4g ..)
            const _Float16* pa = vs + (4 * g + (j >> 2)) * VROW + 16 * dt + 4 * (j & 3);
            const half4_t va = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) short4_t*)(pa)));
            const half4_t vb = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) short4_t*)(pa + 16 * VROW)));
            const half8_t vf = half8_t{va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, ph, o[dt], 0, 0, 0);
            o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl, o[dt], 0, 0, 0);
        }
    };
    for (int kn = kfirst; kn < kstop; kn += NODE) {
        const int nstop = min(kstop, kn + NODE);
        for (int kl = kn; kl < nstop; kl = leaf_end(kl)) {
#pragma unroll
            for (int dt = 0; dt < 16; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            mrun = -1e30f;
            lpart = 0.0f;
            for (int kb = kl; kb < min(nstop, leaf_end(kl)); kb += KB) step(kb);
            l = xor_sum<32>(xor_sum<16>(lpart));
            if constexpr (LEVEL > 0) {  // o, mrun, l: the node's sums up to this leaf
                if (kl > kn) {
                    float fa, fb;
                    merge_weights(node_m, mrun, fa, fb);
                    mrun = node_m;
                    l = merge(node_l, fa, l, fb);
#pragma unroll
                    for (int dt = 0; dt < 16; ++dt)
                        o[dt] = merge4(dt < NR ? node[dt < NR ? dt : 0] : node_lds[dt < NR ? 0 : dt - NR][tid], fa, o[dt], fb);
                }
                if (leaf_end(kl) < nstop) {
                    node_m = mrun;
                    node_l = l;
#pragma unroll
                    for (int dt = 0; dt < 16; ++dt) {
                        if (dt < NR) node[dt < NR ? dt : 0] = o[dt];
                        else node_lds[dt < NR ? 0 : dt - NR][tid] = o[dt];
                    }
                }
            }
        }
        if constexpr (LEVEL > 1) {
            if (kn > kfirst) {
                float fa, fb;
                merge_weights(top_m, mrun, fa, fb);
                mrun = top_m;
                l = merge(top_l, fa, l, fb);
#pragma unroll
                for (int dt = 0; dt < 16; ++dt) o[dt] = merge4(prow[4 * dt], fa, o[dt], fb);
            } else if (nstop < kstop) {
                top_m = mrun;
                top_l = l;
                if (qvalid)
#pragma unroll
                    for (int dt = 0; dt < 16; ++dt) prow[4 * dt] = o[dt];
            }
        }
    }
    // ---- normalise, gate, store: lane (query j) holds dims 16dt + 4g + r ----
    if (!qvalid) return;
    if (parts > 1) {  // this part's unnormalised output, running max and sum for the combine
#pragma unroll
        for (int dt = 0; dt < 16; ++dt) prow[4 * dt] = o[dt];
        if (g == 0) {
            pp[HD] = mrun;
            pp[HD + 1] = l;
        }
        return;
    }
    const float* grow = a.proj + (size_t)mq * a.proj_stride + hh * 2 * HD + HD;
    float* orow = a.out + (size_t)mq * q_dim + hh * HD;
#pragma unroll
    for (int dt = 0; dt < 16; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 16 * dt + 4 * g + r;
            orow[d] = o[dt][r] / l / (1.0f + expf(-grow[d]));
        }
}

// Merge the key parts of one (query, head): block (4 heads, query), a wave per head, lane = 4 dims.  Parts
// of a node, nodes of a top, then the tops, each in order; then the division by the softmax sum and the
// sigmoid gate.
struct Partial {
    f32x4_t o;
    float m, l;
    __device__ __forceinline__ void add(const Partial& b, bool first) {
        if (first) {
            *this = b;
            return;
        }
        float fa, fb;
        merge_weights(m, b.m, fa, fb);
        o = merge4(o, fa, b.o, fb);
        l = merge(l, fa, b.l, fb);
    }
};

template <int LEVEL>
__global__ __launch_bounds__(256) void pf_combine_kernel(AttnArgs a, const PrefillDev* st, int M, int row0,
                                                         const float* part, int parts) {
    const int hh = blockIdx.x * G + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int m = row0 + blockIdx.y, q0 = m / QTILE * QTILE, qn = min(QTILE, M - q0);
    const int nparts = part_count(LEVEL, st->pos0 + q0 + qn);
    const float* pp = part + ((size_t)blockIdx.y * a.n_heads + hh) * parts * PSTRIDE + 4 * lane;
    const float* ml = pp - 4 * lane + HD;
    Partial tot = {}, top = {};
    for (int p = 0, n = 0; p < nparts; ++n) {
        // node n's partial: of its parts (leaves, the first node's first ones shorter), or itself
        Partial node = {};
        if constexpr (LEVEL == 0) {
            Partial in[kFirstLeaves];
            const int count = min(n ? kNodeLeaves : kFirstLeaves, nparts - p);
#pragma unroll
            for (int i = 0; i < kFirstLeaves; ++i) {
                const size_t at = (size_t)min(p + i, nparts - 1) * PSTRIDE;
                in[i] = Partial{*reinterpret_cast<const f32x4_t*>(pp + at), ml[at], ml[at + 1]};
            }
#pragma unroll
            for (int i = 0; i < kFirstLeaves; ++i)
                if (i < count) node.add(in[i], i == 0);
            p += count;
        } else {
            const size_t at = (size_t)p * PSTRIDE;
            node = Partial{*reinterpret_cast<const f32x4_t*>(pp + at), ml[at], ml[at + 1]};
            ++p;
        }
        const bool top_first = LEVEL > 1 || n % (TOP / NODE) == 0;
        top.add(node, top_first);
        if (LEVEL > 1 || n % (TOP / NODE) == TOP / NODE - 1 || p >= nparts) tot.add(top, n < TOP / NODE && (LEVEL < 2 || n == 0));
    }
    const float* grow = a.proj + (size_t)m * a.proj_stride + hh * 2 * HD + HD + 4 * lane;
    float* orow = a.out + ((size_t)m * a.n_heads + hh) * HD + 4 * lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) orow[r] = tot.o[r] / tot.l / (1.0f + expf(-grow[r]));
}

}  // namespace

static int cdiv(int a, int b) { return (a + b - 1) / b; }

// The level of the parts of a pass over `keys` keys.  A step of 32 keys is a chain of loads, LDS and dependent
// MFMAs that one block alone takes 3.3 us for, so few blocks of many steps leave the chip idle (two fit a CU);
// past two rounds of leaves their partials cost more than longer blocks do.  us a call in parts of a leaf /
// node / top, 16 heads, leaves of 256: 512 rows over 2048 keys 98 / 101 / 175 (1024 blocks of a leaf), 4600 200 / 157 / 176,
// 12800 495 / 342 / 355 (1664 blocks of a node), 32768 1336 / 837 / 796; 100 rows over 7000 keys 74 / 88 / 156,
// 9500 102 / 94 / 157; 45 rows over 12800 keys 76 / 88 / 156.
// Parts of any length, cut by the blocks that a pass gives, were faster where rows are many (512 rows over
// 1045 keys 69 us, 72 so; 2048 91 and 104; 12800 322 and 352) and slower where they are few (3 over 12800 keys
// 74 and 48) or the keys (512 rows over 520 55 and 49, 200 over 1045 47 and 42), but a token's sums then changed
// with the tokens that shared its pass.
// A launch takes as many query tiles as keep its partials within kMaxBlocks blocks' (136 MB, 16 heads at any
// context).
constexpr int kLeafBlocks = 1280, kMaxBlocks = 2048;
static int part_level(int tiles, int n_kv, int keys) {
    if (keys <= FINE || n_kv * tiles * part_count(0, keys) <= kLeafBlocks) return 0;
    return keys <= NODE || n_kv * tiles * part_count(1, keys) <= kMaxBlocks ? 1 : 2;
}
static int launch_tiles(int tiles, int n_kv, int parts) {
    const int most = std::max(1, kMaxBlocks / (n_kv * parts));
    return cdiv(tiles, cdiv(tiles, most));
}

size_t attention_prefill_part_floats(int ctx, int n_heads) {
    if (ctx <= FINE || n_heads < G) return 0;  // one part, or a model without attention
    const int n_kv = n_heads / G;
    size_t most = 0;
    for (int tiles = 1; tiles <= SNL_PF_M / QTILE; ++tiles) {
        // of any pass up to ctx positions: as many parts as each level's blocks, or its keys, allow
        const int base = n_kv * tiles;
        const int parts[3] = {std::min(part_count(0, ctx), kLeafBlocks / base),
                              std::min(part_count(1, ctx), std::max(1, kMaxBlocks / base)), part_count(2, ctx)};
        for (int n : parts)
            most = std::max(most, std::min((size_t)base * n, (size_t)std::max(kMaxBlocks, n_kv * n)));
    }
    return most * QTILE * G * PSTRIDE;
}

template <int LEVEL>
static void launch_parts(const AttnArgs& a, const PrefillDev* pstep, int M, float* part, int parts, int tiles,
                         hipStream_t s) {
    for (int row0 = 0; row0 < M; row0 += tiles * QTILE) {
        const int rows = std::min(M - row0, tiles * QTILE);
        hipLaunchKernelGGL(pf_attend_kernel<LEVEL>, dim3(a.n_kv, cdiv(rows, QTILE), parts), dim3(256), 0, s, a, pstep, M,
                           row0, part, parts);
        if (parts > 1)
            hipLaunchKernelGGL(pf_combine_kernel<LEVEL>, dim3(a.n_kv, rows), dim3(256), 0, s, a, pstep, M, row0, part,
                               parts);
    }
}

int launch_attention_prefill(const AttnArgs& a, const PrefillDev* pstep, int M, int keys, float* part,
                             size_t part_floats, hipStream_t s) {
    if (M < 1 || M > SNL_PF_M || a.n_kv < 1 || a.n_heads != G * a.n_kv || a.rot_dim > HD || a.rot_dim % 2 || !pstep) return -1;
    const int tiles = cdiv(M, QTILE), level = part_level(tiles, a.n_kv, keys);
    const int parts = part_count(level, keys);  // parts of the pass's longest key range
    const int step = launch_tiles(tiles, a.n_kv, parts);
    if ((parts > 1 || level > 1) && (!part || (size_t)step * QTILE * a.n_heads * parts * PSTRIDE > part_floats)) return -1;
    hipLaunchKernelGGL(pf_prep_kernel, dim3(a.n_heads + 2 * a.n_kv, M), dim3(256), 0, s, a, pstep);
    if (level == 0) launch_parts<0>(a, pstep, M, part, parts, step, s);
    else if (level == 1) launch_parts<1>(a, pstep, M, part, parts, step, s);
    else launch_parts<2>(a, pstep, M, part, parts, step, s);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace snl
