// The device half of the reference's sampler (src/sampler.rs:98-141): the repetition / presence /
// frequency penalties on a logits row, then its k largest entries in the order top_k_small
// produces (value descending, index ascending among equal values), so that only k (token,
// logit) pairs leave the device.  Temperature, softmax, min-p, top-p and the draw run on the host
// over those pairs.
//
// Top-k: every entry becomes a 64-bit key (order-preserving bits of the value << 32 | ~index), so
// one descending sort of keys gives the reference's order.  Chunks of 4096 keys keep their first k,
// and the survivors go through chunks again until one remains.  For k up to 64 a chunk keeps a sorted
// list of one key per lane in each wave (below); for more it is sorted in LDS (bitonic, 1024 threads).
// Keys differ, so whatever the network, the result is the same.
#include "common.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace snl {

namespace {

constexpr int kChunk = 4096, kSortThreads = 1024;

__device__ __forceinline__ uint32_t order_bits(float v) {
    const uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// src/sampler.rs:99-106, applied to the row in place
__global__ __launch_bounds__(256) void penalty_kernel(float* logits, const uint32_t* tok, const uint32_t* cnt, int n,
                                                      int V, float rep, float presence, float frequency) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n || tok[i] >= (uint32_t)V) return;
    float l = logits[tok[i]];
    if (rep != 1.0f) l = l > 0.0f ? l / rep : l * rep;
    l = l - (presence + frequency * (float)cnt[i]);
    logits[tok[i]] = l;
}

__device__ __forceinline__ void bitonic_desc(unsigned long long* s) {
    const int tid = threadIdx.x;
    for (int size = 2; size <= kChunk; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kChunk / 2 / kSortThreads; ++q) {
                const int p = tid + q * kSortThreads;               // pair index
                const int i = 2 * p - (p & (stride - 1));            // lower element of the pair
                const int j = i + stride;
                const bool desc = (i & size) == 0;                   // direction of this run
                const unsigned long long a = s[i], b = s[j];
                if ((a < b) == desc) {
                    s[i] = b;
                    s[j] = a;
                }
            }
        }
    }
    __syncthreads();
}

// ---- k <= 64: a wave's 64 largest keys, one per lane, descending ----
// A chunk of 4096 keys sorted whole took 78 barriers of 1024 threads, whose latency bound both launches
// (248320 logits, k 20: 72 us a call, 31 as here).  In registers a sort of 64 keys is 21 exchanges
// and a merge 6, with no barrier, and a batch with no key above the k-th so far is skipped.
typedef unsigned long long u64;

template <int O>
__device__ __forceinline__ u64 lane_xor64(u64 v) {
    return ((u64)lane_xor_bits<O>((uint32_t)(v >> 32)) << 32) | lane_xor_bits<O>((uint32_t)v);
}
// compare-exchange with lane l ^ O; `upper`: this lane keeps the larger key
template <int O>
__device__ __forceinline__ u64 exchange(u64 v, bool upper) {
    const u64 o = lane_xor64<O>(v);
    return (v > o) == upper ? v : o;
}
// a bitonic sequence of 64 (of each SIZE lanes) -> descending where desc, else ascending
template <int SIZE>
__device__ __forceinline__ u64 bitonic_merge(u64 v, int lane, bool desc) {
    if constexpr (SIZE >= 64) v = exchange<32>(v, ((lane & 32) == 0) == desc);
    if constexpr (SIZE >= 32) v = exchange<16>(v, ((lane & 16) == 0) == desc);
    if constexpr (SIZE >= 16) v = exchange<8>(v, ((lane & 8) == 0) == desc);
    if constexpr (SIZE >= 8) v = exchange<4>(v, ((lane & 4) == 0) == desc);
    if constexpr (SIZE >= 4) v = exchange<2>(v, ((lane & 2) == 0) == desc);
    return exchange<1>(v, ((lane & 1) == 0) == desc);
}
__device__ __forceinline__ u64 wave_sort(u64 v, int lane, bool desc) {
    v = bitonic_merge<2>(v, lane, (lane & 2) == 0);
    v = bitonic_merge<4>(v, lane, (lane & 4) == 0);
    v = bitonic_merge<8>(v, lane, (lane & 8) == 0);
    v = bitonic_merge<16>(v, lane, (lane & 16) == 0);
    v = bitonic_merge<32>(v, lane, (lane & 32) == 0);
    return bitonic_merge<64>(v, lane, desc);
}
// the 64 largest of a (descending) and b (ascending), descending
__device__ __forceinline__ u64 merge_top(u64 a, u64 b, int lane) { return bitonic_merge<64>(a > b ? a : b, lane, true); }

// The k largest of the block's chunk to out: each wave 4 batches of 64 keys, then the 16 lists in pairs.
template <class Key>
__device__ __forceinline__ void block_top64(Key key, int k, u64* out) {
    constexpr int kW = kSortThreads / 64;
    __shared__ u64 list[kW][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    u64 b[kChunk / kSortThreads];
#pragma unroll
    for (int i = 0; i < kChunk / kSortThreads; ++i) b[i] = key((w * (kChunk / kSortThreads) + i) * 64 + lane);
    u64 a = wave_sort(b[0], lane, true);
#pragma unroll
    for (int i = 1; i < kChunk / kSortThreads; ++i)
        if (__any(b[i] > __shfl(a, k - 1))) a = merge_top(a, wave_sort(b[i], lane, false), lane);
    list[w][lane] = a;
    for (int n = kW / 2; n > 0; n >>= 1) {
        __syncthreads();
        if (w < n) {
            a = merge_top(a, list[w + n][63 - lane], lane);
            list[w][lane] = a;
        }
    }
    if (w == 0 && lane < k) out[lane] = a;
}

__global__ __launch_bounds__(kSortThreads) void top64_logits_kernel(const float* logits, int V, int k, u64* out) {
    const int first = blockIdx.x * kChunk;
    block_top64(
        [&](int e) {
            const int i = first + e;
            return i < V ? ((u64)order_bits(logits[i]) << 32) | (0xFFFFFFFFu - (uint32_t)i) : 0ull;
        },
        k, out + (size_t)blockIdx.x * k);
}

__global__ __launch_bounds__(kSortThreads) void top64_keys_kernel(const u64* in, int n, int k, u64* out) {
    const int first = blockIdx.x * kChunk;
    block_top64([&](int e) { return first + e < n ? in[first + e] : 0ull; }, k, out + (size_t)blockIdx.x * k);
}

// ---- k > 64 ----
// level 0: keys of logits[c*kChunk ..] sorted, the first k kept per chunk
__global__ __launch_bounds__(kSortThreads) void topk_logits_kernel(const float* logits, int V, int k,
                                                                   unsigned long long* out) {
    __shared__ unsigned long long s[kChunk];
    const int c = blockIdx.x, tid = threadIdx.x;
    for (int e = tid; e < kChunk; e += kSortThreads) {
        const int i = c * kChunk + e;
        s[e] = i < V ? ((unsigned long long)order_bits(logits[i]) << 32) | (0xFFFFFFFFu - (uint32_t)i) : 0ull;
    }
    bitonic_desc(s);
    for (int e = tid; e < k; e += kSortThreads) out[(size_t)c * k + e] = s[e];
}

// later levels: n keys in chunks, the first k of each chunk kept
__global__ __launch_bounds__(kSortThreads) void topk_keys_kernel(const unsigned long long* in, int n, int k,
                                                                 unsigned long long* out) {
    __shared__ unsigned long long s[kChunk];
    const int c = blockIdx.x, tid = threadIdx.x;
    for (int e = tid; e < kChunk; e += kSortThreads) {
        const int i = c * kChunk + e;
        s[e] = i < n ? in[i] : 0ull;
    }
    bitonic_desc(s);
    for (int e = tid; e < k; e += kSortThreads) out[(size_t)c * k + e] = s[e];
}

}  // namespace

size_t topk_scratch_keys(int V, int k) { return 2 * (size_t)((V + kChunk - 1) / kChunk) * k + kChunk; }

int launch_penalties(float* logits, int V, const uint32_t* tok, const uint32_t* cnt, int n, float rep, float presence,
                     float frequency, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(penalty_kernel, dim3((n + 255) / 256), dim3(256), 0, s, logits, tok, cnt, n, V, rep, presence,
                       frequency);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int launch_topk(const float* logits, int V, int k, unsigned long long* scratch, unsigned long long** result,
                hipStream_t s) {
    if (k < 1 || k > kChunk / 2 || V < 1) return -1;
    unsigned long long* a = scratch;
    unsigned long long* b = scratch + (size_t)((V + kChunk - 1) / kChunk) * k;
    int chunks = (V + kChunk - 1) / kChunk;
    const bool small = k <= 64;
    if (small) hipLaunchKernelGGL(top64_logits_kernel, dim3(chunks), dim3(kSortThreads), 0, s, logits, V, k, a);
    else hipLaunchKernelGGL(topk_logits_kernel, dim3(chunks), dim3(kSortThreads), 0, s, logits, V, k, a);
    int n = chunks * k;
    while (chunks > 1) {
        chunks = (n + kChunk - 1) / kChunk;
        if (small) hipLaunchKernelGGL(top64_keys_kernel, dim3(chunks), dim3(kSortThreads), 0, s, a, n, k, b);
        else hipLaunchKernelGGL(topk_keys_kernel, dim3(chunks), dim3(kSortThreads), 0, s, a, n, k, b);
        n = chunks * k;
        unsigned long long* t = a;
        a = b;
        b = t;
    }
    *result = a;
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace snl
