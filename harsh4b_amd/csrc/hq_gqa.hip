// hq_gqa.hip - the drop-in GQA decode (hq_gqa_decode): single-token attention
// over an fp16 KV cache, with the mathematics of litespark_gqa_decode
// (cpu_kernels/litespark_int4.cpp:160-259 in the reference repository) in the
// spec order of the oracle's or_gqa_decode_split:
//   score   16 partial fmaf chains of D/16 consecutive dims, halving tree
//           over the 16, times 1/sqrt(D);
//   chunk   m = max, e_t = exp(s_t - m), l = halving tree over 64 slots,
//           o[d] = fmaf chain of e_t * v_t[d] over ascending t;
//   combine M = max m_c; a_c = exp(m_c - M); L and O[d] as fmaf chains over
//           ascending c; out = O * (1 / L).
// Short contexts run in one latency-bound launch (gqa_flash_kernel; the rule
// is one_launch's); longer ones as a memory-bound launch over the chunks
// and a combine (gqa_items_kernel, gqa_combine_kernel).
#include <algorithm>
#include <mutex>

#include "hq_device.h"
#include "hq_internal.h"

namespace hq {

// ---- short contexts: one launch ------------------------------------------
//
// Block i < nc * kv is chunk item (chunk c = i / kv,
// kv head g = i % kv); the launch's last blocks combine.  An item block
// copies its chunk's K and V rows (64 rows of 2D bytes each) straight into
// LDS with global->LDS loads (no register round trip), loads its kv head's
// G query heads into registers meanwhile, and computes, in the spec order
// of or_gqa_decode_split: the scores (16 partial fmaf chains of D/16 dims,
// the 16-lane halving tree, times 1 / sqrt(D)), the chunk's max m, e_t =
// exp(s_t - m) and l = the 64-slot tree, and o[d] = the fmaf chain of e_t *
// v_t[d] over ascending t.  A one-chunk context finishes there (out = o *
// (1 / l) through the combine's operations); otherwise the item publishes
// (m, l, o[0..D-1]) per query head as 32-bit words holding the value's bits
// XOR kGqaKey (a signalling-NaN pattern no arithmetic result carries, so a
// published word is never 0) with agent-scope stores.  A combine block
// (256 / D query heads, one thread per (head, dim) chain) waits for those
// words -- one lane per head first watches the last chunk's last word (the
// last items start last), then every thread polls its own words -- and runs
// the spec's combine over ascending chunks: M = max m_c, a_c = exp(m_c - M),
// L = fmaf(a_c, l_c, L), O = fmaf(a_c, o_c[d], O), out = O * (1 / L); it
// then stores 0 over every word it read.  The words therefore start and end
// every call at zero: the workspace must be zero-filled before its first
// use, and calls that share a workspace must not overlap.  Every wait is
// bounded (kGqaSpinLimit rounds), so the launch always ends.
constexpr uint32_t kGqaKey = 0x7FA5A5A5u;
constexpr unsigned kGqaSpinLimit = 1u << 22;

__device__ __forceinline__ void gqa_word_store(uint32_t* p, float v)
{
    __hip_atomic_store(p, f32_bits(v) ^ kGqaKey, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t gqa_word_load(const uint32_t* p)
{
    return __hip_atomic_load(const_cast<uint32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void gqa_word_clear(uint32_t* p)
{
    __hip_atomic_store(p, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The value of word *p once it is published (bounded wait).
__device__ __forceinline__ float gqa_word_wait(const uint32_t* p, unsigned& budget)
{
    uint32_t w = gqa_word_load(p);
    while (w == 0u && budget != 0u) {
        __builtin_amdgcn_s_sleep(1);
        if (--budget == 0u) break;
        w = gqa_word_load(p);
    }
    return bits_f32(w ^ kGqaKey);
}

constexpr int kFlashThreads = 512;   // threads of a gqa_flash_kernel block (8 waves)

template <int D, int GMAX>
struct FlashLds {
    alignas(16) uint16_t k[kAttnChunk * D];   // the chunk's K rows [t][d]
    alignas(16) uint16_t v[kAttnChunk * D];   // and V rows
    alignas(16) float e[GMAX][kAttnChunk];    // scores, then exp terms
    alignas(16) float q[GMAX * D];            // the kv head's query rows
    float m[GMAX], l[GMAX];
};

struct FlashParams {
    const float* q;           // [kv * G, D]
    const uint16_t* keys;     // [context, kv, D] fp16
    const uint16_t* values;
    uint32_t* words;          // published partials (zero between calls), nc4 = nc rounded up to 4,
                              // U = combine units per head: o [kv * G][nc4 / 4][D][4], then
                              // m [kv * G][U][nc4], then l [kv * G][U][nc4] (one copy per unit)
    float* out;               // [kv * G, D]
    long long time_stride;    // elements per position (kv * D)
    int n, nc, kv, G;
};

// DPL consecutive halves of an LDS row as fp32.
template <int DPL>
__device__ __forceinline__ void lds_halves(const uint16_t* p, float (&k)[DPL])
{
    if constexpr (DPL == 8) {
        const uint4 v = *reinterpret_cast<const uint4*>(p);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) { k[2 * j] = f16_to_f32(uint16_t(w[j])); k[2 * j + 1] = f16_to_f32(uint16_t(w[j] >> 16)); }
    } else if constexpr (DPL == 4) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        k[0] = f16_to_f32(uint16_t(v.x)); k[1] = f16_to_f32(uint16_t(v.x >> 16));
        k[2] = f16_to_f32(uint16_t(v.y)); k[3] = f16_to_f32(uint16_t(v.y >> 16));
    } else if constexpr (DPL == 2) {
        const uint32_t v = *reinterpret_cast<const uint32_t*>(p);
        k[0] = f16_to_f32(uint16_t(v)); k[1] = f16_to_f32(uint16_t(v >> 16));
    } else {
        k[0] = f16_to_f32(*p);
    }
}

template <int D>
constexpr int flash_units_per_head() { return D == 128 ? 2 : 1; }

template <int D, int GMAX>
__device__ void flash_item(const FlashParams& a, FlashLds<D, GMAX>& S, int c, int g)
{
    constexpr int C = kAttnChunk;
    constexpr int T = kFlashThreads;
    constexpr int NW = T / kWave;                        // waves
    constexpr int DPL = D / 16;                          // dims per score lane
    constexpr int HSTEP = T / D;                         // heads between a thread's V chains
    constexpr int PAIRS = (GMAX * D + T - 1) / T;
    constexpr int REPS = C / (T / 16);                   // score positions per 16-lane group
    constexpr int RPI = 1024 / (2 * D);                  // K rows per 1 KB copy instruction
    constexpr int LPR = 2 * D / 16;                      // lanes per row in a copy
    constexpr int NINS = C / RPI;                        // copy instructions per matrix
    const int tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid & (kWave - 1);
    const int G = a.G;
    const int t0 = c * C;
    const int tn = min(C, a.n - t0);
    // The kv head's G query rows, then K rows, then V rows, straight into
    // LDS, all by global->LDS copies (a wave's loads complete in issue
    // order, and the compiler tracks none of these, so its own waits do not
    // hold the scores back for V).  K/V instruction `ins` moves rows RPI*ins
    // .. +RPI-1, lane i row RPI*ins + i/LPR, bytes 16(i%LPR)..; rows past the
    // context re-read the last one (never used).  The scores run once K is
    // in, while V is still arriving.
    {
        const int qbytes = G * D * 4;
        const float* qb = a.q + size_t(g) * G * D;
        for (int ins = wave; ins * 1024 < qbytes; ins += NW)
            dma16(qb, uint32_t(min(ins * 1024 + lane * 16, qbytes - 16)), lds_addr(S.q) + uint32_t(ins) * 1024u);
    }
    const int nq = wave * 1024 < G * D * 4 ? 1 : 0;   // this wave's q copies (G * D * 4 <= 4 KB < NW KB)
    const uint16_t* kb = a.keys + size_t(t0) * size_t(a.time_stride) + size_t(g) * D;
    const uint16_t* vb = a.values + size_t(t0) * size_t(a.time_stride) + size_t(g) * D;
    auto copy_off = [&](int ins) {
        const int row = min(RPI * ins + lane / LPR, tn - 1);
        return uint32_t(size_t(row) * size_t(a.time_stride) * 2u) + uint32_t(lane % LPR) * 16u;
    };
    for (int ins = wave; ins < NINS; ins += NW) dma16(kb, copy_off(ins), lds_addr(S.k) + uint32_t(ins) * 1024u);
    for (int ins = wave; ins < NINS; ins += NW) dma16(vb, copy_off(ins), lds_addr(S.v) + uint32_t(ins) * 1024u);
    // this wave's q and K copies are done when at most its V copies are
    // outstanding (memory operations complete in issue order)
    constexpr int VMAX = (NINS + NW - 1) / NW;
    static_assert(VMAX <= 2, "wait_vm_le covers up to two outstanding copies");
    static_assert(GMAX * D * 4 <= NW * 1024, "one q copy per wave at most");
    (void)nq;
    wait_vm_le(wave < NINS ? (NINS - 1 - wave) / NW + 1 : 0);
    lds_sync();
    // this lane's DPL dims of every query head (a head past G repeats G - 1)
    const int l16 = tid & 15, grp = tid >> 4;
    float qr[GMAX][DPL];
#pragma unroll
    for (int h = 0; h < GMAX; ++h)
#pragma unroll
        for (int j = 0; j < DPL; ++j) qr[h][j] = S.q[min(h, G - 1) * D + l16 * DPL + j];
    // scores, 16 lanes per position.  Every lane computes every head and
    // row (a head past G repeats head G - 1, a row past the context repeats
    // the last one; neither is stored), so no branch splits the REPS x GMAX
    // independent fmaf chains and trees; lane 0 of each row stores.
    const float scale = 1.0f / __builtin_sqrtf(float(D));
    float dot[REPS][GMAX];
#pragma unroll
    for (int rep = 0; rep < REPS; ++rep) {
        float k[DPL];
        lds_halves<DPL>(S.k + (grp + (T / 16) * rep) * D + l16 * DPL, k);
#pragma unroll
        for (int h = 0; h < GMAX; ++h) {
            float pp = 0.0f;
#pragma unroll
            for (int j = 0; j < DPL; ++j) pp = __builtin_fmaf(qr[h][j], k[j], pp);
            dot[rep][h] = pp;
        }
    }
#pragma unroll
    for (int rep = 0; rep < REPS; ++rep)
#pragma unroll
        for (int h = 0; h < GMAX; ++h) dot[rep][h] = row_tree_sum16(dot[rep][h]);
    if (l16 == 0) {
#pragma unroll
        for (int rep = 0; rep < REPS; ++rep) {
            const int i = grp + (T / 16) * rep;
#pragma unroll
            for (int h = 0; h < GMAX; ++h) S.e[h][i] = i < tn ? dot[rep][h] * scale : -__builtin_inff();
        }
    }
    lds_sync();
    // chunk statistics, one wave per head
    for (int h = wave; h < G; h += NW) {
        const float sc = S.e[h][lane];
        const float m = wave_max64_all(sc);
        const float e = lane < tn ? spec_expf(sc - m) : 0.0f;
        const float l = wave_tree_sum64(e);
        S.e[h][lane] = e;
        if (lane == 0) { S.m[h] = m; S.l[h] = l; }
    }
    wait_all_memory();   // this wave's V copies have landed
    lds_sync();
    // V: thread (h0, d) runs the chains of heads h0, h0 + HSTEP, ...; the
    // exp terms are read four positions at a time
    const int d = tid % D, h0 = tid / D;
    float o[PAIRS];
#pragma unroll
    for (int r = 0; r < PAIRS; ++r) o[r] = 0.0f;
    int i = 0;
    for (; i + 8 <= tn; i += 8) {
        float v[8];
        float4 e[PAIRS][2];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = f16_to_f32(S.v[(i + j) * D + d]);
#pragma unroll
        for (int r = 0; r < PAIRS; ++r) {
            const float* er = &S.e[min(h0 + HSTEP * r, GMAX - 1)][i];
            e[r][0] = *reinterpret_cast<const float4*>(er);
            e[r][1] = *reinterpret_cast<const float4*>(er + 4);
        }
#pragma unroll
        for (int r = 0; r < PAIRS; ++r) {
            o[r] = __builtin_fmaf(e[r][0].x, v[0], o[r]);
            o[r] = __builtin_fmaf(e[r][0].y, v[1], o[r]);
            o[r] = __builtin_fmaf(e[r][0].z, v[2], o[r]);
            o[r] = __builtin_fmaf(e[r][0].w, v[3], o[r]);
            o[r] = __builtin_fmaf(e[r][1].x, v[4], o[r]);
            o[r] = __builtin_fmaf(e[r][1].y, v[5], o[r]);
            o[r] = __builtin_fmaf(e[r][1].z, v[6], o[r]);
            o[r] = __builtin_fmaf(e[r][1].w, v[7], o[r]);
        }
    }
    for (; i < tn; ++i) {
        const float v = f16_to_f32(S.v[i * D + d]);
#pragma unroll
        for (int r = 0; r < PAIRS; ++r) o[r] = __builtin_fmaf(S.e[min(h0 + HSTEP * r, GMAX - 1)][i], v, o[r]);
    }
#pragma unroll
    for (int r = 0; r < PAIRS; ++r) {
        const int h = h0 + HSTEP * r;
        if (h >= G) continue;
        const int qh = g * G + h;
        if (a.nc == 1) {
            // the combine's operations over the one chunk
            const float al = spec_expf(S.m[h] - S.m[h]);
            const float L = __builtin_fmaf(al, S.l[h], 0.0f);
            const float O = __builtin_fmaf(al, o[r], 0.0f);
            a.out[size_t(qh) * D + d] = O * (1.0f / L);
        } else {
            const size_t nc4 = size_t((a.nc + 3) & ~3), H = size_t(a.kv) * G;
            uint32_t* ow = a.words + (size_t(qh) * nc4 + (c & ~3)) * D + size_t(d) * 4;
            gqa_word_store(ow + (c & 3), o[r]);
            // the last chunk also publishes 0.0 into its group's padding slots
            if (c == a.nc - 1)
                for (int p = (c & 3) + 1; p < 4; ++p) gqa_word_store(ow + p, 0.0f);
            // m and l once per combine unit of the head: each unit clears
            // the copy it reads
            constexpr int U = flash_units_per_head<D>();
            if (d < U) {
                gqa_word_store(a.words + H * nc4 * D + (size_t(qh) * U + d) * nc4 + c, S.m[h]);
                gqa_word_store(a.words + H * nc4 * (D + U) + (size_t(qh) * U + d) * nc4 + c, S.l[h]);
            }
        }
    }
}

// Combine blocks: wave 0 of each runs one unit -- (query head, half of its
// dims) for D = 128, a query head for D <= 64 (lanes past D run the chunk
// roles only); the other waves leave at once, so the units' loads and
// clears issue from as many CUs as there are units.  Per batch of 64
// chunks, lane c holds chunk c's m_c and l_c, so M is one wave max and a_c
// = exp(m_c - M) is computed in lane c; the chain reads a_c and l_c from
// lane c (readlane), with no LDS and no barrier.  A batch's words are
// fetched in one burst (the lane's o_c[d] and its m_c, l_c), the
// unpublished ones polled again, and cleared once held.  Chunks past the
// context enter the chain as a_c = 0, l_c = 0, o_c = 0: fmaf(0, 0, x)
// returns x, and neither L nor O is ever -0 (their terms' zeros are +0
// sums), so the padding leaves the bits unchanged.  With more than one
// batch M comes from a first pass over every m_c.
constexpr int kFlashCB = 64;   // chunks per batch: one per lane


template <int D>
__device__ void flash_combine(const FlashParams& a, int unit)
{
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    constexpr int NG = kFlashCB / 4;          // chunk groups per batch
    const int lane = threadIdx.x & (kWave - 1);
    const int hraw = unit / flash_units_per_head<D>();
    const int half = unit % flash_units_per_head<D>();
    const int d = half * kWave + lane;        // this lane's dim (a chain when d < D)
    const bool chain = d < D;
    const int nc = a.nc;
    const size_t nc4 = size_t((nc + 3) & ~3), H = size_t(a.kv) * a.G;
    uint32_t* obase = a.words + size_t(hraw) * nc4 * D;              // [nc4 / 4][D][4]
    constexpr int U = flash_units_per_head<D>();
    uint32_t* mbase = a.words + H * nc4 * D + size_t(unit) * nc4;    // this unit's copy [nc4]
    uint32_t* lbase = a.words + H * nc4 * (D + U) + size_t(unit) * nc4;
    unsigned budget = kGqaSpinLimit;
    float M = -__builtin_inff();
    if (nc > kFlashCB) {
        float mm = -__builtin_inff();
        for (int c = lane; c < nc; c += kWave) mm = fmaxf(mm, gqa_word_wait(mbase + c, budget));
        M = wave_max64_all(mm);
    }
    float L = 0.0f, O = 0.0f;
    for (int c0 = 0; c0 < nc; c0 += kFlashCB) {
        const int nb = min(kFlashCB, nc - c0);
        const int ngrp = (nb + 3) >> 2;          // chunk groups of the batch
        // every load unconditional, through buffer descriptors that end at
        // the batch's last chunk (group): a load past one returns 0 without
        // touching memory and a store there is dropped.  Group g4's four
        // chunks of dim d are one 16-byte word of the lane, at a constant
        // scalar offset; a group's padding slots past the context hold a
        // published 0.0 (written by the last chunk's item), groups past the
        // batch are set to 0.0 here, and lanes past D (D < 64) read dim 0's
        // words and discard them.
        const __amdgpu_buffer_rsrc_t ro = raw_rsrc(obase + size_t(c0) * D, ngrp * D * 16);
        const __amdgpu_buffer_rsrc_t rm = raw_rsrc(mbase + c0, nb * 4);
        const __amdgpu_buffer_rsrc_t rl = raw_rsrc(lbase + c0, nb * 4);
        const uint32_t vo = uint32_t(chain ? d : 0) * 16u;
        // first the batch's m_c and l_c, one chunk per lane (two loads per
        // round): an item publishes them with its o words, so once every
        // chunk's are in, the o burst below rarely meets an empty word
        const bool mine = lane < nb;             // lane c's chunk
        uint32_t mw = 0u, lw = 0u;
        while (true) {
            mw = mw != 0u ? mw : __builtin_amdgcn_raw_buffer_load_b32(rm, lane * 4, 0, kAgentSC1);
            lw = lw != 0u ? lw : __builtin_amdgcn_raw_buffer_load_b32(rl, lane * 4, 0, kAgentSC1);
            mw = mine ? mw : f32_bits(-__builtin_inff()) ^ kGqaKey;
            lw = mine ? lw : kGqaKey;
            if (!__builtin_amdgcn_ballot_w64((mw == 0u) | (lw == 0u)) || budget == 0u) break;   // (wave-uniform)
            __builtin_amdgcn_s_sleep(1);
            --budget;
        }
        v4u ow[NG];
#pragma unroll
        for (int g4 = 0; g4 < NG; ++g4) ow[g4] = __builtin_amdgcn_raw_buffer_load_b128(ro, vo, g4 * D * 16, kAgentSC1);
#pragma unroll
        for (int g4 = 0; g4 < NG; ++g4)
            if (g4 >= ngrp) ow[g4] = v4u{kGqaKey, kGqaKey, kGqaKey, kGqaKey};   // (wave-uniform)
        // poll what was not published yet (a published word keeps its value
        // for the rest of the call, so the whole burst is simply re-read;
        // the padding entries set above are nonzero and stay so)
        while (budget != 0u) {
            bool pending = false;
#pragma unroll
            for (int g4 = 0; g4 < NG; ++g4)
                pending |= (ow[g4][0] == 0u) | (ow[g4][1] == 0u) | (ow[g4][2] == 0u) | (ow[g4][3] == 0u);
            if (!pending) break;
            __builtin_amdgcn_s_sleep(1);
            --budget;
#pragma unroll
            for (int g4 = 0; g4 < NG; ++g4) {
                const v4u w = __builtin_amdgcn_raw_buffer_load_b128(ro, vo, g4 * D * 16, kAgentSC1);
#pragma unroll
                for (int j = 0; j < 4; ++j) ow[g4][j] = ow[g4][j] != 0u ? ow[g4][j] : w[j];
            }
        }
        const float mc = bits_f32(mw ^ kGqaKey);
        if (nc <= kFlashCB) M = wave_max64_all(mc);
        const float ac = mine ? spec_expf(mc - M) : 0.0f;
        const float lc = bits_f32(lw ^ kGqaKey);
#pragma unroll
        for (int c = 0; c < kFlashCB; ++c) {
            const float al = bits_f32(__builtin_amdgcn_readlane(f32_bits(ac), c));
            L = __builtin_fmaf(al, bits_f32(__builtin_amdgcn_readlane(f32_bits(lc), c)), L);
            O = __builtin_fmaf(al, bits_f32(ow[c >> 2][c & 3] ^ kGqaKey), O);
            // (the broadcasts stay next to their use: hoisted, 128 of them
            // would not fit the scalar registers)
            if ((c & 7) == 7) __builtin_amdgcn_sched_barrier(0);
        }
        // the words go back to 0 (each is read by this lane alone -- m_c and
        // l_c are this unit's own copies -- and the first pass over m_c
        // above is done)
        if (chain) {
#pragma unroll
            for (int g4 = 0; g4 < NG; ++g4)
                __builtin_amdgcn_raw_buffer_store_b128(v4u{0u, 0u, 0u, 0u}, ro, vo, g4 * D * 16, kAgentSC1);
        }
        if (mine) {
            __builtin_amdgcn_raw_buffer_store_b32(0u, rm, lane * 4, 0, kAgentSC1);
            __builtin_amdgcn_raw_buffer_store_b32(0u, rl, lane * 4, 0, kAgentSC1);
        }
    }
    if (chain) a.out[size_t(hraw) * D + d] = O * (1.0f / L);
}

template <int D, int GMAX>
__global__ __launch_bounds__(kFlashThreads) void gqa_flash_kernel(FlashParams a)
{
    __shared__ FlashLds<D, GMAX> lds;
    const int items = a.nc * a.kv;
    const int b = blockIdx.x;
    if (b < items) flash_item<D, GMAX>(a, lds, b / a.kv, b % a.kv);   // (block-uniform)
    else if (threadIdx.x < kWave) flash_combine<D>(a, b - items);
}

template <int D, int GMAX>
static void launch_flash(const FlashParams& a, hipStream_t s)
{
    const int H = a.kv * a.G;
    const int blocks = a.nc * a.kv + (a.nc > 1 ? H * flash_units_per_head<D>() : 0);
    hipLaunchKernelGGL((gqa_flash_kernel<D, GMAX>), dim3(blocks), dim3(kFlashThreads), 0, s, a);
}

// ---- longer contexts: items, then the combine --------------------------------------
//
// One wave takes one item: a 64-position chunk of one kv head, for all its
// query heads.  v_mfma_f32_4x4x1_16b is one fmaf per output (as the 16x16x1
// form: hq_prefill_attn.hip), and its 16 blocks fit the shape: four query heads
// (A rows, one block of A broadcast by CBSZ / ABID) x 64 keys, then x 64
// dims.  So a score chain is D/16 instructions for four heads and 64 keys, a
// position of the V chain D/64, and nothing crosses lanes but the softmax
// statistics and one 4 x 4 transpose of the exp terms.  K goes to LDS
// (global_load_lds; a lane then reads its key's row), V straight to
// registers, half of it behind K and half once K has arrived (a wave counts
// at most 63 loads).  No wave waits for another, so the chip's waves drift
// apart and keep the memory busy: 32767 positions of 8 x 4 heads take 29.7 us
// (4.5 TB/s; a bare read of the cache 23.7) and the combine 11.
//
// Four waves a block, two blocks a CU.  The partials are plain floats in the
// workspace; the combine, a launch of its own (polled from within the items'
// launch, its agent-scope reads of 8 MB by 32 blocks took 18 us), leaves
// every word it read at zero, as the one-launch kernel needs it.
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kItemWaves = 4;
template <int D>
constexpr int gqa_units() { return D == 128 ? 2 : 1; }   // U: combine blocks per head

struct GqaParams {
    const float* q;           // [kv * G, D]
    const uint16_t* keys;     // [context, kv, D] fp16
    const uint16_t* values;
    float* part;              // partials (zero between calls)
    float* out;               // [kv * G, D]
    long long time_stride;    // elements per position (kv * D)
    int n, nc, kv, G;
};

// Element j of the quad's four lanes, in every lane.
template <int J>
__device__ __forceinline__ float quad_bcast(float v)
{
    return dpp_f<J * 0x55>(v);
}

// Item: chunk c of kv head g, by one wave; ks: its LDS.  GS: sets of four
// query heads.
template <int D, int GS>
__device__ __forceinline__ void gqa_item(const GqaParams& a, uint16_t* ks, int c, int g)
{
    constexpr int DPL = D / 16;                 // dims per score chain
    constexpr int P = D / 8;                    // 16-byte pieces of a K row
    constexpr int RPI = 64 / P;                 // K rows per copy instruction (1 KB)
    constexpr int DV = D == 128 ? 2 : 1;        // V dims per lane (lanes past D repeat the last)
    constexpr int SH = P == 16 ? 0 : P == 8 ? 1 : P == 4 ? 2 : 3;
    const int lane = threadIdx.x & (kWave - 1);
    const int G = a.G;
    const int t0 = c * kAttnChunk;
    const int tn = min(kAttnChunk, a.n - t0);

    // queries: lane 4 j + h, element i = dim DPL j + i of head h of the set
    float q[GS][DPL];
#pragma unroll
    for (int s = 0; s < GS; ++s) {
        const float* qp = a.q + size_t(g * G + min(4 * s + (lane & 3), G - 1)) * D + DPL * (lane >> 2);
#pragma unroll
        for (int i = 0; i < DPL; ++i) q[s][i] = qp[i];
    }
    // K rows: piece p of row r at slot p ^ ((r >> SH) & (P - 1)), so that the
    // 16 lanes of a read phase cover every bank once; rows past the context
    // re-read the last one (masked)
    const uint16_t* kb = a.keys + size_t(t0) * size_t(a.time_stride) + size_t(g) * D;
    const uint16_t* vb = a.values + size_t(t0) * size_t(a.time_stride) + size_t(g) * D;
    const uint32_t row_bytes = uint32_t(a.time_stride) * 2u;
#pragma unroll
    for (int ins = 0; ins < P; ++ins) {
        const int r = RPI * ins + lane / P;
        const int piece = (lane % P) ^ ((r >> SH) & (P - 1));
        dma16(kb, uint32_t(min(r, tn - 1)) * row_bytes + uint32_t(piece) * 16u, lds_addr(ks) + uint32_t(ins) * 1024u);
    }
    // V rows: a load at or past the chunk's last byte returns 0 and touches no
    // memory, so positions past the context add fmaf(0, 0, o) = o (o is never
    // -0)
    uint32_t v[kAttnChunk];
    const __amdgpu_buffer_rsrc_t rv = raw_rsrc(vb, (tn - 1) * int(row_bytes) + D * 2);
    const int vd = min(lane * DV, D - DV) * 2;
    auto load_v = [&](int t) {
        if constexpr (DV == 2) return uint32_t(__builtin_amdgcn_raw_buffer_load_b32(rv, vd, t * int(row_bytes), 0));
        else return uint32_t(__builtin_amdgcn_raw_buffer_load_b16(rv, vd, t * int(row_bytes), 0));
    };
#pragma unroll
    for (int t = 0; t < 32; ++t) v[t] = load_v(t);
    __builtin_amdgcn_sched_barrier(0);
    // the K rows (and the queries) are in: the 32 V loads above are the only
    // ones issued since (no load crosses the block's memory clobber, nor the
    // scheduling barriers)
    asm volatile("s_waitcnt vmcnt(32)" ::: "memory");
#pragma unroll
    for (int t = 32; t < 64; ++t) v[t] = load_v(t);
    __builtin_amdgcn_sched_barrier(0);

    // scores: lane = key, element = head.  The lane's K row first (one burst
    // of LDS reads), then the chains in the tree's order, four at a time:
    // (0 8 4 12) (2 10 6 14) (1 9 5 13) (3 11 7 15)
    uint4 raw[P];
    const int swz = (lane >> SH) & (P - 1);
#pragma unroll
    for (int i = 0; i < P; ++i) raw[i] = *reinterpret_cast<const uint4*>(ks + lane * D + (i ^ swz) * 8);
    auto k_at = [&](auto dim) {
        constexpr int w = dim % 8 / 2;
        const uint4& r = raw[dim / 8];
        const uint32_t u = w == 0 ? r.x : w == 1 ? r.y : w == 2 ? r.z : r.w;
        return f16_to_f32(uint16_t(dim % 2 ? u >> 16 : u));
    };
    f32x4 quad[4][GS];
    unrolled<4>([&](auto n) {
        constexpr int first = n == 0 ? 0 : n == 1 ? 2 : n == 2 ? 1 : 3;
        f32x4 x[4][GS] = {};
        unrolled<DPL>([&](auto i) {
            unrolled<4>([&](auto y) {
                constexpr int chain = first + (y == 0 ? 0 : y == 1 ? 8 : y == 2 ? 4 : 12);
                const float k = k_at(std::integral_constant<int, chain * DPL + i>{});
#pragma unroll
                for (int s = 0; s < GS; ++s)
                    x[y][s] = __builtin_amdgcn_mfma_f32_4x4x1f32(q[s][i], k, x[y][s], 4, chain, 0);
            });
        });
#pragma unroll
        for (int s = 0; s < GS; ++s) quad[n][s] = (x[0][s] + x[1][s]) + (x[2][s] + x[3][s]);
    });
    f32x4 dot[GS];
#pragma unroll
    for (int s = 0; s < GS; ++s) dot[s] = (quad[0][s] + quad[1][s]) + (quad[2][s] + quad[3][s]);

    // softmax statistics per head, and the exp terms transposed within quads:
    // e[s][i] of lane 4 x + h = term of head h, position 4 x + i
    const float scale = 1.0f / __builtin_sqrtf(float(D));
    float m[GS][4], l[GS][4], e[GS][4];
#pragma unroll
    for (int s = 0; s < GS; ++s) {
        float t[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const float sc = lane < tn ? dot[s][h] * scale : -__builtin_inff();
            m[s][h] = wave_max64_all(sc);
            const float x = spec_expf_neg(sc - m[s][h]);
            t[h] = lane < tn ? x : 0.0f;
            l[s][h] = wave_tree_sum64_all(t[h]);
        }
        const int h = lane & 3;
        unrolled<4>([&](auto i) {
            const float b0 = quad_bcast<i>(t[0]), b1 = quad_bcast<i>(t[1]);
            const float b2 = quad_bcast<i>(t[2]), b3 = quad_bcast<i>(t[3]);
            e[s][i] = h & 2 ? (h & 1 ? b3 : b2) : (h & 1 ? b1 : b0);
        });
    }

    // V chains: lane = dim (dims 2 lane and 2 lane + 1 for D = 128)
    f32x4 o[GS][DV];
#pragma unroll
    for (int s = 0; s < GS; ++s)
#pragma unroll
        for (int x = 0; x < DV; ++x) o[s][x] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto position = [&](auto t) {
        const float v0 = f16_to_f32(uint16_t(v[t]));
        const float v1 = f16_to_f32(uint16_t(v[t] >> 16));
#pragma unroll
        for (int s = 0; s < GS; ++s) {
            o[s][0] = __builtin_amdgcn_mfma_f32_4x4x1f32(e[s][t % 4], v0, o[s][0], 4, t / 4, 0);
            if constexpr (DV == 2) o[s][1] = __builtin_amdgcn_mfma_f32_4x4x1f32(e[s][t % 4], v1, o[s][1], 4, t / 4, 0);
        }
    };
    unrolled<kAttnChunk>([&](auto t) { position(t); });

    // partials: o [kv * G][nc][D], then U copies of m [kv * G][nc], then U of l
    const size_t H = size_t(a.kv) * G, nc = size_t(a.nc);
#pragma unroll
    for (int s = 0; s < GS; ++s) {
#pragma unroll
        for (int h4 = 0; h4 < 4; ++h4) {
            if (4 * s + h4 >= G) break;
            const size_t at = size_t(g * G + 4 * s + h4) * nc + c;
            float* ow = a.part + at * D + lane * DV;
            if constexpr (DV == 2) *reinterpret_cast<float2*>(ow) = make_float2(o[s][0][h4], o[s][1][h4]);
            else if (D >= kWave || lane < D) *ow = o[s][0][h4];
            // m and l once per combine block of the head (each clears the copy it reads)
            if (lane < 2 * gqa_units<D>())
                a.part[H * nc * (D + lane) + at] = lane < gqa_units<D>() ? m[s][h4] : l[s][h4];
        }
    }
}

template <int D, int GS>
__global__ __launch_bounds__(kItemWaves* kWave, 2) void gqa_items_kernel(GqaParams a)
{
    __shared__ uint4 k_s[kItemWaves][kAttnChunk * D / 8];
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int item = int(blockIdx.x) * kItemWaves + wave;
    if (item >= a.nc * a.kv) return;
    gqa_item<D, GS>(a, reinterpret_cast<uint16_t*>(k_s[wave]), item / a.kv, item % a.kv);
}

// Block (head, 64 dims): lane d holds the O chain of dim d, and a wave takes
// 64 chunks at a time: lane c holds chunk c's m_c and l_c, so a_c = exp(m_c -
// M) is computed in lane c and the chains read a_c and l_c from lane c
// (readlane).  The eight waves fetch their chunks side by side and run their
// links of the O chains in turn, the state passing through LDS, each wave's
// link of the L chain (needed only at the end) beside the next wave's O link.
// Chunks past the context enter the chains as a_c = 0, l_c = 0, o_c = 0:
// fmaf(0, 0, x) returns x, and neither L nor O is ever -0 (their terms' zeros
// are +0 sums), so the padding leaves the bits unchanged.
constexpr int kCombWaves = 8;
template <int D>
__global__ __launch_bounds__(kCombWaves* kWave) void gqa_combine_kernel(GqaParams a)
{
    constexpr int U = gqa_units<D>();
    __shared__ float max_s[kCombWaves];
    __shared__ float o_s[kWave];
    __shared__ float l_s;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int head = blockIdx.x / U;
    const int d = (blockIdx.x % U) * kWave + lane;   // (lanes past D, for D < 64, follow dim 0 and discard it)
    const bool chain = d < D;
    const int nc = a.nc;
    const int batches = (nc + kWave - 1) / kWave;
    const size_t H = size_t(a.kv) * a.G;
    float* o = a.part + size_t(head) * nc * D;
    float* mw = a.part + H * nc * (D + blockIdx.x % U) + size_t(head) * nc;   // this block's copies
    float* lw = mw + H * nc * U;
    float mm = -__builtin_inff();
    for (int c = wave * kWave + lane; c < nc; c += kCombWaves * kWave) mm = fmaxf(mm, mw[c]);
    mm = wave_max64_all(mm);
    if (lane == 0) max_s[wave] = mm;
    float L = 0.0f, O = 0.0f, M = -__builtin_inff();
    for (int b0 = 0; b0 < batches; b0 += kCombWaves) {
        const int c0 = min((b0 + wave) * kWave, nc);
        const int nb = min(kWave, nc - c0);
        // loads past the batch return 0 and touch no memory
        const __amdgpu_buffer_rsrc_t ro = raw_rsrc(o + size_t(c0) * D, nb * D * 4);
        const int vo = chain ? d * 4 : 0;
        float ov[kWave];
#pragma unroll
        for (int c = 0; c < kWave; ++c)
            ov[c] = bits_f32(__builtin_amdgcn_raw_buffer_load_b32(ro, vo, c * D * 4, 0));
        const bool mine = lane < nb;
        const float mc = mine ? mw[c0 + lane] : 0.0f;
        const float lc = mine ? lw[c0 + lane] : 0.0f;
        if (b0 == 0) {
            lds_sync();
            for (int w = 0; w < kCombWaves; ++w) M = fmaxf(M, max_s[w]);
        }
        const float ac = mine ? spec_expf(mc - M) : 0.0f;
        auto links = [&](bool o_chain) {
#pragma unroll
            for (int c = 0; c < kWave; ++c) {
                const float al = bits_f32(__builtin_amdgcn_readlane(f32_bits(ac), c));
                if (o_chain) O = __builtin_fmaf(al, ov[c], O);
                else L = __builtin_fmaf(al, bits_f32(__builtin_amdgcn_readlane(f32_bits(lc), c)), L);
                // (the broadcasts stay next to their use: hoisted, they
                // would not fit the scalar registers)
                if ((c & 7) == 7) __builtin_amdgcn_sched_barrier(0);
            }
        };
        const int turns = min(kCombWaves, batches - b0);
        for (int turn = 0; turn <= turns; ++turn) {
            if (turn == wave && turn < turns) {
                if (b0 + turn > 0) O = o_s[lane];
                links(true);
                o_s[lane] = O;
            }
            if (turn == wave + 1) {
                if (b0 + wave > 0) L = l_s;
                links(false);
                if (lane == 0) l_s = L;
            }
            lds_sync();
        }
        if (wave == turns - 1 && b0 + turns == batches && chain) a.out[size_t(head) * D + d] = O * (1.0f / L);
        // the partials back to zero (each o is read by this lane alone, and
        // every wave passed the barriers after its first pass over m)
        if (chain) {
#pragma unroll
            for (int c = 0; c < kWave; ++c) __builtin_amdgcn_raw_buffer_store_b32(0u, ro, vo, c * D * 4, 0);
        }
        if (mine) {
            mw[c0 + lane] = 0.0f;
            lw[c0 + lane] = 0.0f;
        }
    }
}

template <int D, int GS>
static hipError_t launch_items(const GqaParams& a, hipStream_t s)
{
    const int items = a.nc * a.kv;
    hipLaunchKernelGGL((gqa_items_kernel<D, GS>), dim3((items + kItemWaves - 1) / kItemWaves),
                       dim3(kItemWaves * kWave), 0, s, a);
    hipLaunchKernelGGL(gqa_combine_kernel<D>, dim3(a.kv * a.G * gqa_units<D>()), dim3(kCombWaves * kWave), 0, s,
                       a);
    return hipGetLastError();
}

// The one-launch kernel while one combine batch holds every chunk (4096
// positions of 8 x 4 heads of 128: 11.6 us against 13).  Up to two batches
// with more than four query heads per kv head (4 x 8 heads, 8192: 17.2
// against 18.1, 16384: 31 against 22), and for heads of 128 where the items'
// launch gains little from its waves: up to 512 of them (2 x 4 heads, 8192:
// 13.3 against 14.9; 4 x 4, 4097: 13.1 against 15.1; 8192, 512 items: 15.1
// against 15.4; but 8 x 4, 4608, 576 items: 16.5 against 15.9), and just past
// one block of four a CU, where some CUs take two (16 x 4 heads, 4097, 1040
// items: 20.8 against 22.2; 5120, 1280: 22.9 against 23.6; 8192, 2048: 30.2
// against 27.4; 8 x 4, 8192, 1024: 20.8 against 18.4).  Heads of 16 to 64 gain
// nothing from it (of 64, 4097 positions: 2 x 4 12.6 against 13.0, 4 x 4 even,
// 8 x 4 15.4 against 13.3).
static bool one_launch(int nc, int kv_heads, int groups, int head_dim)
{
    if (nc <= kFlashCB || nc > 2 * kFlashCB) return nc <= kFlashCB;
    const int items = nc * kv_heads;
    return groups > 4 || (head_dim == 128 && (items <= 512 || (items > 1024 && items <= 1280)));
}

// head_dim 16/32/64/128, groups <= 8 (checked by the caller)
static hipError_t launch_gqa_decode(const float* query, const uint16_t* keys, const uint16_t* values, uint32_t* words,
                                    float* output, int context, int kv_heads, int groups, int head_dim, hipStream_t s)
{
    const int nc = (context + kAttnChunk - 1) / kAttnChunk;
    if (one_launch(nc, kv_heads, groups, head_dim)) {
        FlashParams a{};
        a.q = query;
        a.keys = keys;
        a.values = values;
        a.words = words;
        a.out = output;
        a.time_stride = (long long)kv_heads * head_dim;
        a.n = context;
        a.nc = nc;
        a.kv = kv_heads;
        a.G = groups;
        switch (head_dim) {
        case 16: launch_flash<16, 8>(a, s); break;
        case 32: launch_flash<32, 8>(a, s); break;
        case 64: launch_flash<64, 8>(a, s); break;
        default:
            if (groups <= 4) launch_flash<128, 4>(a, s);
            else launch_flash<128, 8>(a, s);
        }
        return hipGetLastError();
    }
    GqaParams a{};
    a.q = query;
    a.keys = keys;
    a.values = values;
    a.part = reinterpret_cast<float*>(words);
    a.out = output;
    a.time_stride = (long long)kv_heads * head_dim;
    a.n = context;
    a.nc = nc;
    a.kv = kv_heads;
    a.G = groups;
    switch (head_dim) {
    case 16: return groups <= 4 ? launch_items<16, 1>(a, s) : launch_items<16, 2>(a, s);
    case 32: return groups <= 4 ? launch_items<32, 1>(a, s) : launch_items<32, 2>(a, s);
    case 64: return groups <= 4 ? launch_items<64, 1>(a, s) : launch_items<64, 2>(a, s);
    default: return groups <= 4 ? launch_items<128, 1>(a, s) : launch_items<128, 2>(a, s);
    }
}

}  // namespace hq

using namespace hq;

extern "C" size_t hq_gqa_workspace_bytes(int score_stride, int kv_heads, int groups, int head_dim)
{
    if (score_stride <= 0 || kv_heads <= 0 || groups <= 0 || head_dim <= 0) return 0;
    const int nc = (score_stride + kAttnChunk - 1) / kAttnChunk;
    // a 256-byte header (reserved), then the chunk partials of whole groups
    // of four chunks (D + 2 words per query head and chunk, and up to two
    // more for the combine units' own copies of m and l): one workspace
    // serves every context up to score_stride
    return 256 + attention_workspace_floats(kv_heads * groups, (nc + 3) & ~3, head_dim + 2) * 4;
}

// Checks and launch shared by hq_gqa_decode and hq_gqa_decode_noalloc.
static int gqa_check(const float* query, const uint16_t* keys, const uint16_t* values, const float* output,
                     int context, int kv_heads, int groups, int head_dim, int score_stride)
{
    if (!query || !keys || !values || !output) return HQ_ERR_ARG;
    if (context <= 0 || kv_heads <= 0 || groups <= 0 || groups > 8) return HQ_ERR_ARG;
    if (score_stride < context) return HQ_ERR_ARG;
    if (head_dim != 16 && head_dim != 32 && head_dim != 64 && head_dim != 128) return HQ_ERR_ARG;
    if (kv_heads > 64) return HQ_ERR_ARG;
    if ((reinterpret_cast<uintptr_t>(keys) & 15u) != 0 || (reinterpret_cast<uintptr_t>(values) & 15u) != 0)
        return HQ_ERR_ALIGN;
    return HQ_OK;
}

static int gqa_launch(const float* query, const uint16_t* keys, const uint16_t* values, void* workspace,
                      float* output, int context, int kv_heads, int groups, int head_dim, hipStream_t stream)
{
    uint32_t* words = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace) + 256);
    const hipError_t e = launch_gqa_decode(query, keys, values, words, output, context, kv_heads, groups, head_dim,
                                          stream);
    return e == hipSuccess ? HQ_OK : HQ_ERR_LAUNCH;
}

// The reference's argument list (litespark_int4.cpp:160-171): the K/V time
// stride is kv_heads * head_dim (:172), and score_stride is the row stride of
// its `scores` scratch, i.e. the context capacity that scratch was sized for
// (cpu_lightspark.py:405 passes state.capacity).  Here the workspace takes
// the scratch's place and is sized by the same number.
extern "C" int hq_gqa_decode(const float* query, const uint16_t* keys, const uint16_t* values,
                             void* workspace, float* output, int context, int kv_heads,
                             int groups, int head_dim, int score_stride, void* stream)
{
    const int st = gqa_check(query, keys, values, output, context, kv_heads, groups, head_dim, score_stride);
    if (st != HQ_OK) return st;
    if (!workspace) return HQ_ERR_ARG;
    if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return HQ_ERR_ALIGN;
    return gqa_launch(query, keys, values, workspace, output, context, kv_heads, groups, head_dim,
                      static_cast<hipStream_t>(stream));
}

// ---- the variant that allocates nothing ----------------------------------------
//
// For callers that cannot allocate device memory (code under HIP graph
// capture, serving loops that forbid hipMalloc): hq_gqa_decode with its
// workspace in a file-scope device array instead of a caller buffer.  Each
// GPU holds its own copy of `scratch` until the process ends.  The array's
// name is only a host-side stand-in: its device address is taken with
// hipGetSymbolAddress once per device, with that device current, and that
// address is what the kernels receive.  Every call on a device shares the
// device's array, so calls that overlap on one GPU race.
constexpr size_t kNoAllocScratchBytes = size_t(4) << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices];
static std::mutex g_scratch_mutex;

// The device address of this device's `scratch` (nullptr on failure).
static void* scratch_address(int dev)
{
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) return nullptr;
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

extern "C" int hq_gqa_decode_noalloc(const float* query, const uint16_t* keys, const uint16_t* values,
                                     float* output, int context, int kv_heads, int groups, int head_dim,
                                     int score_stride, void* stream)
{
    const int st = gqa_check(query, keys, values, output, context, kv_heads, groups, head_dim, score_stride);
    if (st != HQ_OK) return st;
    // the bytes this call uses (its context's chunk partials), not the
    // score_stride sizing of the caller-workspace form
    if (hq_gqa_workspace_bytes(context, kv_heads, groups, head_dim) > kNoAllocScratchBytes) return HQ_ERR_ARG;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return HQ_ERR_DEVICE;
    void* ws = scratch_address(dev);
    if (ws == nullptr) return HQ_ERR_DEVICE;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    return gqa_launch(query, keys, values, ws, output, context, kv_heads, groups, head_dim, s);
}
