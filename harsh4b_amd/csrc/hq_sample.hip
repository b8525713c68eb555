// hq_sample.hip - the stochastic sampler of the reference's CPU runner
// (sample_logits, cpu_lightspark.py:706-726 in the reference repository) on
// gfx950: repetition penalty, temperature, top-k, softmax, top-p and the
// inverse-cdf draw of numpy's Generator.choice, given the uniform draw u.
//
//   1. block b loads logits[b*S, (b+1)*S) into LDS and applies the penalty
//      there: v[id] = logits[id] > 0 ? logits[id] / rp : logits[id] * rp for
//      every id of `generated` in its slice (a repeated id writes the same
//      value again)
//   2. it turns v_i / temperature into 64-bit sort keys (value descending,
//      NaN last, index ascending; the value is recoverable from the key)
//      and radix-selects its k smallest keys, 11 bits per pass from the
//      highest bit in which the keys differ, into a candidate list in
//      global memory
//   3. the lists are merged in a tree: as many lists a node as the LDS array
//      holds (all of them up to k = 107 of 151936 logits; two at k = 2048,
//      where one block merging 38 lists of 2048 took most of 535 us), the
//      node's last block to finish (a ticket counter) selecting the k
//      smallest
//   4. the root sorts its k keys and runs softmax / top-p / cdf in the
//      reference's order with the repo's exp and numpy's float32 summation
//      order: the pairwise sums' leaves side by side, the cumulative sums
//      on thread 0 (up to k = 64 all of it in one wave)
// Bound by latency: a merge is a ticket and a round trip (about 3 us) and
// its passes' block barriers.
// The result equals the oracle's or_sample_token bit for bit (ids,
// probabilities, token).  One launch per token.
#include <algorithm>

#include "hq_device.h"
#include "hq_internal.h"

namespace hq {

constexpr int kSampleThreads = 1024;
constexpr int kSampleSlice = 4096;               // logits per block; keys the LDS array holds
constexpr int kSampleMaxK = kSampleSlice / 2;    // the last block's chunks add at least k keys

// Sort key: ascending key order = value descending (NaN last), then index
// ascending.  -0 ranks (and is recovered) as +0.
__device__ __forceinline__ uint64_t sample_key(float v, int i)
{
    uint32_t hi;
    if (v != v) {
        hi = 0xFFFFFFFFu;
    } else {
        uint32_t u = f32_bits(v);
        if (u == 0x80000000u) u = 0;
        const uint32_t asc = (u & 0x80000000u) ? ~u : (u | 0x80000000u);   // ascending with the value
        hi = ~asc;
    }
    return (uint64_t(hi) << 32) | uint32_t(i);
}

// Past the end of the logits: after every real key (NaN keys included,
// whose indices are < n) and distinct, as the radix select needs.
__device__ __forceinline__ uint64_t pad_key(int i) { return (uint64_t(0xFFFFFFFFu) << 32) | uint32_t(i); }

__device__ __forceinline__ float key_value(uint64_t key)
{
    const uint32_t asc = ~uint32_t(key >> 32);
    return __uint_as_float((asc & 0x80000000u) ? (asc & 0x7FFFFFFFu) : ~asc);
}

__device__ __forceinline__ int key_index(uint64_t key) { return int(uint32_t(key)); }

__device__ __forceinline__ void publish_u64(uint64_t* p, uint64_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t read_u64(const uint64_t* p)
{
    return __hip_atomic_load(const_cast<uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr int kSampleBins = 2048;                // radix digits of 11 bits
constexpr int kSampleWaves = kSampleThreads / kWave;

struct SampleShared {
    uint64_t key[kSampleSlice];
    union {
        float v[kSampleSlice];                          // the slice's values (phase 1)
        struct {
            alignas(16) uint64_t win[kSampleMaxK];                  // selected keys
            float p[kSampleMaxK];
            float drop[kSampleMaxK];
        } f;
    } u;
    int hist[kSampleBins];
    uint64_t wave_min[kSampleWaves], wave_max[kSampleWaves];
    int wave_sum[kSampleWaves];
    int digit, before, done, count, ticket;
    float total;
    float leaf_sum[64];   // the pairwise sum's leaves by path
};

// The k smallest of the `count` keys S.key[0..count) (1 <= k <= count; the
// keys must be distinct, or the last bin could hand out more than k), written
// unordered to out[0..k).  Radix select: each pass histograms the keys that
// share the digits chosen so far and picks the digit bin holding the k-th
// key; when that bin is taken whole the selection stops early.  (Of 8-bit
// digits a slice's logits fill a handful, and the histogram's atomics queue on
// them.)  Every thread of the block calls it; out may be
// global memory (published with agent scope).
template <bool GLOBAL>
__device__ void select_k(SampleShared& S, int count, int k, uint64_t* out)
{
    constexpr int KPT = kSampleSlice / kSampleThreads;
    const int t = threadIdx.x;
    const int lane = t & (kWave - 1), wave = t / kWave;
    uint64_t x[KPT];
    bool in[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        in[i] = t + kSampleThreads * i < count;
        x[i] = in[i] ? S.key[t + kSampleThreads * i] : 0;
    }
    if (t == 0) S.count = 0;
    uint64_t mask = 0, prefix = 0;
    int shift = 64 - 11;
    if (!GLOBAL || k == 1) {
        // a merge's keys share their high bits: from the highest in which
        // two differ
        uint64_t lo = ~uint64_t(0), hi = 0;
#pragma unroll
        for (int i = 0; i < KPT; ++i) {
            lo = in[i] && x[i] < lo ? x[i] : lo;
            hi = in[i] && x[i] > hi ? x[i] : hi;
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            const uint64_t a = __shfl_xor((unsigned long long)lo, o, kWave);
            const uint64_t b = __shfl_xor((unsigned long long)hi, o, kWave);
            lo = a < lo ? a : lo;
            hi = b > hi ? b : hi;
        }
        if (lane == 0) {
            S.wave_min[wave] = lo;
            S.wave_max[wave] = hi;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kSampleWaves; ++w) {
            lo = S.wave_min[w] < lo ? S.wave_min[w] : lo;
            hi = S.wave_max[w] > hi ? S.wave_max[w] : hi;
        }
        if (k == 1) {                          // (block-uniform)
            if (t == 0) {
                if (GLOBAL) publish_u64(out, lo);
                else out[0] = lo;
            }
            __syncthreads();
            return;
        }
        const int top = lo == hi ? 0 : 63 - __clzll((long long)(lo ^ hi));
        shift = top > 10 ? top - 10 : 0;
        mask = shift + 11 < 64 ? ~uint64_t(0) << (shift + 11) : 0;
        prefix = lo & mask;
    }
    int need = k;
    while (true) {
        for (int b = t; b < kSampleBins; b += kSampleThreads) S.hist[b] = 0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < KPT; ++i)
            if (in[i] && (x[i] & mask) == prefix) atomicAdd(&S.hist[int(x[i] >> shift) & (kSampleBins - 1)], 1);
        __syncthreads();
        // the bin in which the running count reaches need: two bins a thread
        const int c0 = S.hist[2 * t], c1 = S.hist[2 * t + 1];
        int incl = c0 + c1;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int y = __shfl_up(incl, o, kWave);
            if (lane >= o) incl += y;
        }
        if (lane == kWave - 1) S.wave_sum[wave] = incl;
        __syncthreads();
        int below = lane < wave ? S.wave_sum[lane & (kSampleWaves - 1)] : 0;   // (16 waves: lanes 0-15)
        below = wave_isum64(below);
        const int before0 = __builtin_amdgcn_readfirstlane(below) + incl - c0 - c1;
        if (before0 < need && need <= before0 + c0 + c1) {
            const bool second = need > before0 + c0;
            const int before = second ? before0 + c0 : before0;
            S.digit = 2 * t + (second ? 1 : 0);
            S.before = before;
            S.done = need - before == (second ? c1 : c0);
        }
        __syncthreads();
        need -= S.before;
        prefix |= uint64_t(S.digit) << shift;
        mask |= uint64_t(kSampleBins - 1) << shift;
        if (S.done || shift == 0) break;       // (block-uniform)
        // the last digit may overlap the one before it: its high bits are
        // then fixed by the prefix
        shift = shift > 11 ? shift - 11 : 0;
    }
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const bool take = in[i] && (x[i] & mask) <= prefix;
        const uint64_t votes = __ballot(take);
        int base = 0;
        if (lane == 0 && votes) base = atomicAdd(&S.count, __popcll(votes));
        base = __builtin_amdgcn_readfirstlane(base);
        if (take) {
            const int pos = base + __popcll(votes & ((uint64_t(1) << lane) - 1));
            if (GLOBAL) publish_u64(out + pos, x[i]);
            else out[pos] = x[i];
        }
    }
    __syncthreads();
}

// S.key[0..k) ascending: by rank (the keys are distinct) up to 256 keys, four
// threads or more a key and no barrier between the comparisons (1024 keys by
// rank: 38 us of comparisons); else a bitonic sort padded with the largest
// key, whose steps of distance below 64 stay within a wave and need no block
// barrier.
__device__ void sort_keys(SampleShared& S, int k)
{
    const int t = threadIdx.x;
    if (k <= kSampleThreads / 4) {
        int per = 1;                           // threads per key, within a wave
        while (per < 32 && 2 * per * k <= kSampleThreads) per <<= 1;
        const int i = t / per, part = t % per;
        int rank = 0;
        uint64_t mine = 0;
        if (i < k) {
            mine = S.key[i];
            for (int j = part; j < k; j += per) rank += S.key[j] < mine;
        }
        for (int o = per >> 1; o >= 1; o >>= 1) rank += __shfl_xor(rank, o, kWave);
        __syncthreads();
        if (i < k && part == 0) S.key[rank] = mine;
        __syncthreads();
        return;
    }
    int n = 1;
    while (n < k) n <<= 1;
    for (int j = k + t; j < n; j += kSampleThreads) S.key[j] = ~uint64_t(0);
    __syncthreads();
    for (int b = 2; b <= n; b <<= 1) {
        for (int j = b >> 1; j > 0; j >>= 1) {
            for (int i = t; i < n; i += kSampleThreads) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const uint64_t x = S.key[i], y = S.key[ixj];
                    if ((x > y) == ((i & b) == 0)) {
                        S.key[i] = y;
                        S.key[ixj] = x;
                    }
                }
            }
            const int next = j > 1 ? j >> 1 : b;
            if (j >= kWave || next >= kWave || (j == 1 && b == n)) __syncthreads();
            else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    }
}

// numpy's float32 add.reduce order (pairwise_sum of umath's loops_utils):
// < 8 values in order, <= 128 in eight running sums, larger halves split at
// a multiple of 8 below n/2 and summed left + right.  A leaf is named by its
// path from the root (bit 5 - d: right at depth d; zeros below the leaf; n <=
// kSampleMaxK splits at most 5 times): eight threads a path run the leaf's
// running sums, then lane `path` of wave 0 adds left + right, level by level.
// Every thread calls it; the sum is in S.total after it.
constexpr int kPaths = 64;
struct PairwisePath {
    int off, len, splits;     // the leaf's values, its depth
    bool leaf;                // false: another path names it
    __device__ __forceinline__ PairwisePath(int path, int n) : off(0), len(n), splits(0)
    {
#pragma unroll
        for (int d = 0; d < 6; ++d) {
            if (len > 128) {
                int n2 = len / 2;
                n2 -= n2 % 8;
                const bool right = (path >> (5 - d)) & 1;
                off += right ? n2 : 0;
                len = right ? len - n2 : n2;
                splits = d + 1;
            }
        }
        leaf = (path & ((kPaths >> splits) - 1)) == 0;
    }
};
__device__ void pairwise_sum_f32(SampleShared& S, const float* a, int n)
{
    const int t = threadIdx.x;
    if (t < 8 * kPaths) {
        const int r8 = t & 7;
        const PairwisePath w(t >> 3, n);
        float r = 0.0f;
        if (w.leaf) {
            const float* b = a + w.off;
            const int l = w.len;
            if (l >= 8) {
                r = b[r8];
                for (int i = 8 + r8; i < l - l % 8; i += 8) r += b[i];
            }
            // ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7))
            r = r + __shfl_xor(r, 1, kWave);
            r = r + __shfl_xor(r, 2, kWave);
            r = r + __shfl_xor(r, 4, kWave);
            if (r8 == 0) {
                for (int i = l < 8 ? 0 : l - l % 8; i < l; ++i) r += b[i];
                S.leaf_sum[t >> 3] = r;
            }
        }
    }
    __syncthreads();
    if (t < kPaths) {
        const PairwisePath w(t, n);
        float v = w.leaf ? S.leaf_sum[t] : 0.0f;
#pragma unroll
        for (int d = 5; d >= 0; --d) {
            const float right = __shfl_xor(v, 32 >> d, kWave);
            if (w.splits > d) v = v + right;   // (right children's lanes hold sums no one reads)
        }
        if (t == 0) S.total = v;
    }
    __syncthreads();
}

struct SampleParams {
    const float* logits;
    const int32_t* generated;
    const double* u;
    int32_t* out_token;
    int32_t* ids_out;
    float* probs_out;
    uint64_t* cand;       // gridDim.x * k candidate keys
    int* counter;         // one per merge node, zero between calls (a node's last block resets its own)
    int n, n_generated, k;
    int arity;            // lists a merge node takes
    float rp, temperature, top_p;
};

// sample_finish for k <= 64, by one wave: lane i holds probability i, the sums
// run over lanes in the same orders, without block barriers (k = 40: 24.6 -> 19.7 us).
__device__ __forceinline__ float wave_pairwise(float p, int k)
{
    const int lane = threadIdx.x & (kWave - 1);
    float r = 0.0f;
    const int whole = k < 8 ? 0 : k - k % 8;
    if (k >= 8) {
        r = __shfl(p, lane & 7, kWave);
        for (int i = 8; i < whole; i += 8) r += __shfl(p, i + (lane & 7), kWave);
        r = r + __shfl_xor(r, 1, kWave);
        r = r + __shfl_xor(r, 2, kWave);
        r = r + __shfl_xor(r, 4, kWave);
    }
    for (int i = whole; i < k; ++i) r += __shfl(p, i, kWave);
    return r;
}
__device__ void sample_finish_wave(SampleShared& S, const SampleParams& p)
{
    const int i = threadIdx.x;
    const int k = p.k;
    const bool mine = i < k;
    const uint64_t key = S.key[mine ? i : 0];
    float prob = mine ? spec_expf(key_value(key) - key_value(S.key[0])) : 0.0f;
    prob = prob / wave_pairwise(prob, k);
    if (p.top_p < 1.0f) {
        float c = 0.0f, drop = 0.0f;
        for (int j = 0; j < k; ++j) {
            const float x = bits_f32(__builtin_amdgcn_readlane(f32_bits(prob), j));
            c = c + x;
            drop = i == j ? c - x : drop;
        }
        if (drop >= p.top_p) prob = 0.0f;
        prob = prob / wave_pairwise(prob, k);
    }
    double c = 0.0, cdf = 0.0;
    for (int j = 0; j < k; ++j) {
        c = c + double(bits_f32(__builtin_amdgcn_readlane(f32_bits(prob), j)));
        cdf = i == j ? c : cdf;
    }
    const uint64_t below = __ballot(mine && cdf / c <= *p.u);
    const int index = min(below ? 64 - __clzll((long long)below) : 0, k - 1);
    if (i == index) *p.out_token = key_index(key);
    if (mine && p.ids_out) p.ids_out[i] = key_index(key);
    if (mine && p.probs_out) p.probs_out[i] = prob;
}

__device__ __forceinline__ void load8(const float* a, float (&x)[8])
{
    const float4 u = *reinterpret_cast<const float4*>(a), v = *reinterpret_cast<const float4*>(a + 4);
    x[0] = u.x; x[1] = u.y; x[2] = u.z; x[3] = u.w;
    x[4] = v.x; x[5] = v.y; x[6] = v.z; x[7] = v.w;
}
__device__ __forceinline__ void store8(float* a, const float (&x)[8])
{
    *reinterpret_cast<float4*>(a) = make_float4(x[0], x[1], x[2], x[3]);
    *reinterpret_cast<float4*>(a + 4) = make_float4(x[4], x[5], x[6], x[7]);
}

// softmax / top-p / Generator.choice over the k sorted keys S.key[0..k).
__device__ void sample_finish(SampleShared& S, const SampleParams& p)
{
    const int t = threadIdx.x;
    const int k = p.k;
    float* prob = S.u.f.p;
    float* drop = S.u.f.drop;
    const float top = key_value(S.key[0]);
    for (int i = t; i < (k + 7 & ~7); i += kSampleThreads)   // (zeros up to whole groups of eight)
        prob[i] = i < k ? spec_expf(key_value(S.key[i]) - top) : 0.0f;
    __syncthreads();
    pairwise_sum_f32(S, prob, k);
    for (int i = t; i < k; i += kSampleThreads) prob[i] = prob[i] / S.total;
    __syncthreads();
    if (p.top_p < 1.0f) {
        if (t == 0) {
            // (the next eight probabilities load under this eight's sums, whose
            // order is theirs).  Once the sum is clearly past top_p every
            // later value is dropped: the probabilities are not negative, so
            // the sum does not fall, and drop[i] is the sum before i to
            // within two roundings of a value near 1.
            float c = 0.0f, x[8], y[8];
            const float past = p.top_p + 1e-5f;
            int i = 0;
            load8(prob, x);
            for (; i < k; i += 8) {
                load8(prob + min(i + 8, kSampleMaxK - 8), y);
                float d[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    c = c + x[j];
                    d[j] = c - x[j];
                    x[j] = y[j];
                }
                store8(drop + i, d);
                if (c >= past) break;
            }
            S.count = min(i + 8, k);           // drop is written up to here
        }
        __syncthreads();
        for (int i = t; i < k; i += kSampleThreads)
            if (i >= S.count || drop[i] >= p.top_p) prob[i] = 0.0f;
        __syncthreads();
        pairwise_sum_f32(S, prob, k);
        for (int i = t; i < k; i += kSampleThreads) prob[i] = prob[i] / S.total;
        __syncthreads();
    }
    // Generator.choice: cdf = cumsum(double(p)) / its last entry; the token is
    // ids[#{i : cdf_i <= u}].  The sum stops at the last nonzero probability
    // (adding 0.0 changes nothing).
    double* cdf = reinterpret_cast<double*>(S.key + kSampleMaxK);
    if (t == 0) {
        S.count = 0;
        S.digit = 0;
    }
    __syncthreads();
    for (int i = t; i < k; i += kSampleThreads)
        if (!(prob[i] == 0.0f)) atomicMax(&S.count, i + 1);
    __syncthreads();
    const int last_i = S.count;
    if (t == 0) {
        double c = 0.0;
        float x[8], y[8];
        load8(prob, x);
        for (int i = 0; i < last_i; i += 8) {
            load8(prob + min(i + 8, kSampleMaxK - 8), y);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                c = c + double(x[j]);
                cdf[i + j] = c;
                x[j] = y[j];
            }
        }
    }
    __syncthreads();
    const double last = last_i > 0 ? cdf[last_i - 1] : 0.0;
    const double draw = *p.u;
    for (int i = t; i < k; i += kSampleThreads)
        if ((i < last_i ? cdf[i] : last) / last <= draw) atomicMax(&S.digit, i + 1);
    __syncthreads();
    if (t == 0) *p.out_token = key_index(S.key[S.digit >= k ? k - 1 : S.digit]);
    if (p.ids_out)
        for (int i = t; i < k; i += kSampleThreads) p.ids_out[i] = key_index(S.key[i]);
    if (p.probs_out)
        for (int i = t; i < k; i += kSampleThreads) p.probs_out[i] = prob[i];
}

// S.key[0..count) reduced to its k smallest, in S.key[0..k).
__device__ void keep_k(SampleShared& S, int count, int k)
{
    if (count <= k) return;
    select_k<false>(S, count, k, S.u.f.win);
    for (int j = threadIdx.x; j < k; j += kSampleThreads) S.key[j] = S.u.f.win[j];
    __syncthreads();
}

__global__ __launch_bounds__(kSampleThreads) void sample_kernel(SampleParams p)
{
    __shared__ SampleShared S;
    const int t = threadIdx.x;
    const int k = p.k;
    const int base = blockIdx.x * kSampleSlice;
    // 1. the slice's values, penalised
    for (int j = t; j < kSampleSlice; j += kSampleThreads) {
        const int i = base + j;
        S.u.v[j] = i < p.n ? p.logits[i] : 0.0f;
    }
    __syncthreads();
    if (p.rp != 1.0f) {
        for (int g = t; g < p.n_generated; g += kSampleThreads) {
            const int id = p.generated[g];
            if (id < base || id >= base + kSampleSlice || id >= p.n) continue;
            const float x = p.logits[id];
            S.u.v[id - base] = x > 0.0f ? x / p.rp : x * p.rp;
        }
        __syncthreads();
    }
    // 2. keys, and this slice's k smallest
    for (int j = t; j < kSampleSlice; j += kSampleThreads) {
        const int i = base + j;
        S.key[j] = i < p.n ? sample_key(S.u.v[j] / p.temperature, i) : pad_key(i);
    }
    __syncthreads();
    // 3. up the merge tree: the list of a node lies in the place of its first
    // slice's list, `span` slices apart on a level
    int lists = gridDim.x, span = 1, node0 = 0;
    int slot = blockIdx.x;
    int count = kSampleSlice;                  // keys of this block's list, in S.key
    while (lists > 1) {
        const int node = slot / span / p.arity;
        const int children = min(p.arity, lists - node * p.arity);
        if (children > 1) {
            if (count > k) {
                select_k<true>(S, count, k, p.cand + size_t(slot) * k);
            } else {
                for (int j = t; j < k; j += kSampleThreads) publish_u64(p.cand + size_t(slot) * k + j, S.key[j]);
            }
            wait_all_memory();                 // this thread's candidate stores have completed
            __syncthreads();
            if (t == 0) S.ticket = atomicAdd(p.counter + node0 + node, 1);
            __syncthreads();
            if (S.ticket != children - 1) return;
            if (t == 0) publish_i(p.counter + node0 + node, 0);
            // the node's last block: its children's lists, in as many rounds
            // as the LDS array needs (one, but for huge vocabularies)
            slot = node * p.arity * span;
            const int total = children * k;
            count = 0;
            for (int off = 0; off < total;) {
                const int chunk = min(total - off, kSampleSlice - count);
                for (int j = t; j < chunk; j += kSampleThreads) {
                    const int child = (off + j) / k;
                    S.key[count + j] = read_u64(p.cand + size_t(slot + child * span) * k + (off + j - child * k));
                }
                off += chunk;
                count += chunk;
                __syncthreads();
                if (off < total) {
                    keep_k(S, count, k);
                    count = min(count, k);
                }
            }
        }
        const int groups = (lists + p.arity - 1) / p.arity;
        node0 += groups;
        span *= p.arity;
        lists = groups;
    }
    // 4. the root
    keep_k(S, count, k);
    sort_keys(S, k);
    if (k > kWave) sample_finish(S, p);
    else if (t < kWave) sample_finish_wave(S, p);
}

static size_t al256s(size_t v) { return (v + 255) & ~size_t(255); }

static int sample_slices(int n) { return (n + kSampleSlice - 1) / kSampleSlice; }

// The counters' fixed place at the workspace's start: calls with any n and k
// share them.  A tree over up to kSampleNodes slices has at most 1023 nodes
// (lone children can make them more than its slices: 521 over 513); more
// slices (4.2M logits) merge in one node.
constexpr int kSampleNodes = 1024;
constexpr size_t kSampleHead = kSampleNodes * 4;

}  // namespace hq

using namespace hq;

extern "C" size_t hq_sample_workspace_bytes(int n, int top_k)
{
    if (n <= 0 || top_k <= 0) return 0;
    const int k = top_k < n ? top_k : n;
    return kSampleHead + al256s(size_t(sample_slices(n)) * size_t(k) * 8);   // counters, then candidates
}

extern "C" int hq_sample_token(const float* logits, int n, const int32_t* generated, int n_generated,
                               float repetition_penalty, float temperature, int top_k, float top_p,
                               const double* u, int32_t* out_token, int32_t* ids_out, float* probs_out,
                               void* workspace, void* stream)
{
    if (!logits || !u || !out_token || !workspace || n <= 0 || n_generated < 0) return HQ_ERR_ARG;
    if (n_generated > 0 && !generated) return HQ_ERR_ARG;
    if (top_k < 1 || top_k > kSampleMaxK) return HQ_ERR_ARG;
    if (!(temperature > 0.0f) || !(repetition_penalty > 0.0f) || !(top_p > 0.0f)) return HQ_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(workspace) & 255u) return HQ_ERR_ALIGN;
    SampleParams p;
    p.logits = logits;
    p.generated = generated;
    p.u = u;
    p.out_token = out_token;
    p.ids_out = ids_out;
    p.probs_out = probs_out;
    p.n = n;
    p.n_generated = n_generated;
    p.k = top_k < n ? top_k : n;
    p.rp = repetition_penalty;
    p.temperature = temperature;
    p.top_p = top_p;
    const int blocks = sample_slices(n);
    p.arity = blocks > kSampleNodes ? blocks : std::max(2, kSampleSlice / p.k);
    char* ws = static_cast<char*>(workspace);
    p.counter = reinterpret_cast<int*>(ws);
    p.cand = reinterpret_cast<uint64_t*>(ws + kSampleHead);
    hipLaunchKernelGGL(sample_kernel, dim3(blocks), dim3(kSampleThreads), 0, static_cast<hipStream_t>(stream), p);
    return hipGetLastError() == hipSuccess ? HQ_OK : HQ_ERR_LAUNCH;
}
