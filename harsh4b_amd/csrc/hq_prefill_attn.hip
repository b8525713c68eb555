// hq_prefill_attn.hip - causal attention of a batch of prompt tokens over
// the fp16 KV cache (head_dim 128), with the bits of the single-token
// attention (hq_attention.hip), on the fp32 matrix cores.
//
// The spec's two contractions are fmaf chains, and v_mfma_f32_16x16x1_4b
// (one product per output and instruction) is exactly one fmaf per output:
// checked against fmaf over normal, subnormal, infinite and signed-zero
// operands, bit for bit.  So the chains run on the matrix cores at twice the
// rate of scalar fp32 code:
//   score   16 chains of 8 dims (8 instructions each), whose 64 keys x 16
//           queries tiles are added in the spec's halving tree;
//   V       one chain over the chunk's positions in ascending order.
// A wave owns 16 queries of one head.  Scores come out transposed (lane =
// query, registers = keys), so an exp term is already where the V product
// reads it: the instruction's B operand broadcasts one 16-lane group (BLGP),
// with no shuffle or LDS round trip between the two products.  The query
// tiles are aligned to 16 absolute positions: every query of a tile then has
// the same number of 64-position chunks.
//
// The combine needs the maximum over all chunks first, so the scores of a
// tile go to the workspace and come back for the V pass (storing each
// chunk's 128 partial sums instead would move 1 KB per query, head and
// chunk).  Batches too small to fill the chip give each block a few chunks,
// write the chunk partials and let attention_combine_kernel combine them;
// contexts whose scores exceed the workspace compute them twice.
//
// Bound by fp32 arithmetic.  Of the SIMDs' cycles in prefill_attention_kernel
// the matrix instructions (256 of 32 cycles per 16 queries, 64 keys and head)
// take 48 % and the other vector instructions (about 1000 of 4 cycles:
// conversions, tree sums, exponentials) 25 %, by counters; LDS reads conflict
// in no bank, and memory moves 0.6 GB a layer.  Three waves a SIMD is what the
// registers allow (168, nine more spilled and reloaded at a chunk's ends, not
// among its products).
// 2000 tokens of 32 heads: 440 to 480 us a layer by GPU, 68 to 75 TFLOP/s (1890 us
// with one query per block on the vector unit, 672 us with the scores computed
// twice).
#include <algorithm>

#include "hq_device.h"
#include "hq_internal.h"
#include "hq_prefill_place.h"

namespace hq {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kPaD = 128;
static_assert(kPaChunk == kAttnChunk, "the placement counts the spec's chunks");

template <int GROUP>
__device__ __forceinline__ f32x16 mfma1(float a, float b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 4 + GROUP);
}

// Stage I of the scores: chains I and I + 8 (dims 8 I .. and 8 I + 64 ..),
// whose sum is the first level of the halving tree.  The K pieces arrive in
// `raw` and leave as the pieces of stage NEXT, so a stage's LDS reads and the
// previous stage's tree sums run under its matrix instructions.  q[j] of lane
// group g = dim 32 g + j.
struct PaPair { f32x16 a, b; };
template <int I, int NEXT>
__device__ __forceinline__ PaPair pa_stage(const uint16_t* row, int swz, uint4 (&raw)[2], const float (&q)[32])
{
    float k0[8], k1[8];
    const uint32_t w0[4] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w};
    const uint32_t w1[4] = {raw[1].x, raw[1].y, raw[1].z, raw[1].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        k0[2 * j] = f16_to_f32(uint16_t(w0[j]));
        k0[2 * j + 1] = f16_to_f32(uint16_t(w0[j] >> 16));
        k1[2 * j] = f16_to_f32(uint16_t(w1[j]));
        k1[2 * j + 1] = f16_to_f32(uint16_t(w1[j] >> 16));
    }
    if constexpr (NEXT >= 0) {
        raw[0] = *reinterpret_cast<const uint4*>(row + (NEXT ^ swz) * 8);
        raw[1] = *reinterpret_cast<const uint4*>(row + ((NEXT + 8) ^ swz) * 8);
    }
    PaPair t{};
    unrolled<8>([&](auto j) {
        t.a = mfma1<I / 4>(k0[j], q[8 * (I % 4) + j], t.a);
        t.b = mfma1<I / 4 + 2>(k1[j], q[8 * (I % 4) + j], t.b);
    });
    return t;
}

// Scaled scores of the wave's queries and the chunk's keys: lane 16 g + c,
// element 4 b + r = query c, key 16 b + 4 g + r.  The stages run in the
// order of the tree (0 4 2 6 1 5 3 7: at most two partial sums wait), each
// stage's sums placed under the next one's instructions.
__device__ __forceinline__ f32x16 pa_scores(const uint16_t* k, const float (&q)[32])
{
    const int lane = threadIdx.x & (kWave - 1);
    const uint16_t* row = k + lane * kPaD;
    const int swz = lane & 15;
    uint4 raw[2];
    raw[0] = *reinterpret_cast<const uint4*>(row + (0 ^ swz) * 8);
    raw[1] = *reinterpret_cast<const uint4*>(row + (8 ^ swz) * 8);
#define PA_FENCE __builtin_amdgcn_sched_barrier(0)
    const PaPair s0 = pa_stage<0, 4>(row, swz, raw, q);
    PA_FENCE;
    const PaPair s4 = pa_stage<4, 2>(row, swz, raw, q);
    const f32x16 t0 = s0.a + s0.b;
    PA_FENCE;
    const PaPair s2 = pa_stage<2, 6>(row, swz, raw, q);
    const f32x16 t04 = t0 + (s4.a + s4.b);
    PA_FENCE;
    const PaPair s6 = pa_stage<6, 1>(row, swz, raw, q);
    const f32x16 t2 = s2.a + s2.b;
    PA_FENCE;
    const PaPair s1 = pa_stage<1, 5>(row, swz, raw, q);
    const f32x16 t0426 = t04 + (t2 + (s6.a + s6.b));
    PA_FENCE;
    const PaPair s5 = pa_stage<5, 3>(row, swz, raw, q);
    const f32x16 t1 = s1.a + s1.b;
    PA_FENCE;
    const PaPair s3 = pa_stage<3, 7>(row, swz, raw, q);
    const f32x16 t15 = t1 + (s5.a + s5.b);
    PA_FENCE;
    const PaPair s7 = pa_stage<7, -1>(row, swz, raw, q);
    const f32x16 t3 = s3.a + s3.b;
    PA_FENCE;
#undef PA_FENCE
    return (t0426 + (t15 + (t3 + (s7.a + s7.b)))) * (1.0f / __builtin_sqrtf(float(kPaD)));
}

// Maximum / sum over the four lane groups (lanes c, c + 16, c + 32, c + 48),
// in every lane; the sum adds group pairs (g, g + 2), then (0, 1).
__device__ __forceinline__ float groups_max(float v)
{
    unsigned x = f32_bits(v), y = x;
    swap32(x, y);
    v = fmaxf(bits_f32(x), bits_f32(y));
    x = f32_bits(v);
    y = x;
    swap16(x, y);
    return fmaxf(bits_f32(x), bits_f32(y));
}
__device__ __forceinline__ float groups_sum(float v)
{
    unsigned x = f32_bits(v), y = x;
    swap32(x, y);
    v = bits_f32(x) + bits_f32(y);
    x = f32_bits(v);
    y = x;
    swap16(x, y);
    return bits_f32(x) + bits_f32(y);
}

// The chunk's scores with the keys past each query's position at -inf
// (masked: the tile's last chunk; query c sees the first tn keys).
__device__ __forceinline__ void pa_mask(f32x16& s, bool masked, int tn)
{
    if (masked) {
        const int g = (threadIdx.x & (kWave - 1)) >> 4;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 16 * (i >> 2) + 4 * g + (i & 3) < tn ? s[i] : -__builtin_inff();
    }
}

__device__ __forceinline__ float pa_lane_max(const f32x16& s)
{
    float m = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) m = fmaxf(m, s[i]);
    return m;
}

// The chunk's partial results from its (masked) scores: s becomes the exp
// terms, m their reference maximum and l their sum (the 64-slot halving
// tree: levels 32 and 16 over the elements, 8 and 4 over the lane groups, 2
// and 1 over the elements again), ae / ao the V chains of dims 2 (16 b + 4 g +
// r) and the next (element 4 b + r).  full: 16-key blocks every query of the
// tile sees whole (4: the chunk is not the tile's last).
__device__ __forceinline__ void pa_values(const uint16_t* v, f32x16& s, int full, float& m, float& l, f32x16& ae,
                                          f32x16& ao)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int c16 = lane & 15, g = lane >> 4;
    m = groups_max(pa_lane_max(s));
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = spec_expf_neg(s[i] - m);
    if (full < 4) {   // (a masked slot is 0 also where m is -inf)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 16 * (i >> 2) + 4 * g + (i & 3) <= 16 * full + c16 ? s[i] : 0.0f;
    }
    float t4[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) t4[r] = groups_sum((s[r] + s[8 + r]) + (s[4 + r] + s[12 + r]));
    l = (t4[0] + t4[2]) + (t4[1] + t4[3]);
    ae = f32x16{};
    ao = f32x16{};
    const uint16_t* vrow = v + 2 * lane;
    if (full == 4) {
        unrolled<16>([&](auto tq) {                      // positions 4 tq .. 4 tq + 3
            uint32_t w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = *reinterpret_cast<const uint32_t*>(vrow + (4 * tq + r) * kPaD);
            unrolled<4>([&](auto r) {
                ae = mfma1<tq % 4>(f16_to_f32(uint16_t(w[r])), s[4 * (tq / 4) + r], ae);
                ao = mfma1<tq % 4>(f16_to_f32(uint16_t(w[r] >> 16)), s[4 * (tq / 4) + r], ao);
            });
        });
        return;
    }
    // the tile's last chunk: whole blocks, then the tile's own 16 positions,
    // of which query c sees the first c + 1.  A masked query's chain keeps
    // its value (its exp term is 0, but the row may hold infinities).
    auto terms = [&](int b, float (&e)[4]) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float e01 = b & 1 ? s[4 + r] : s[r], e23 = b & 1 ? s[12 + r] : s[8 + r];
            e[r] = b & 2 ? e23 : e01;
        }
    };
    float e[4];
#pragma unroll 1
    for (int b = 0; b < full; ++b) {
        terms(b, e);
        unrolled<16>([&](auto t) {
            const uint32_t w = *reinterpret_cast<const uint32_t*>(vrow + (16 * b + t) * kPaD);
            ae = mfma1<t / 4>(f16_to_f32(uint16_t(w)), e[t % 4], ae);
            ao = mfma1<t / 4>(f16_to_f32(uint16_t(w >> 16)), e[t % 4], ao);
        });
    }
    terms(full, e);
    unrolled<16>([&](auto t) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(vrow + (16 * full + t) * kPaD);
        const f32x16 ne = mfma1<t / 4>(f16_to_f32(uint16_t(w)), e[t % 4], ae);
        const f32x16 no = mfma1<t / 4>(f16_to_f32(uint16_t(w >> 16)), e[t % 4], ao);
        const bool ok = t <= c16;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            ae[i] = ok ? ne[i] : ae[i];
            ao[i] = ok ? no[i] : ao[i];
        }
    });
}

// One step of the combine over ascending chunks.
__device__ __forceinline__ void pa_combine(float M, float m, float l, const f32x16& ae, const f32x16& ao, float& L,
                                           f32x16& oe, f32x16& oo)
{
    const float al = spec_expf_neg(m - M);
    L = __builtin_fmaf(al, l, L);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        oe[i] = __builtin_fmaf(al, ae[i], oe[i]);
        oo[i] = __builtin_fmaf(al, ao[i], oo[i]);
    }
}

__host__ __device__ constexpr PaBatch pa_batch(const PrefillAttnParams& p)
{
    return PaBatch{p.p0, p.rows, p.kv_heads, p.groups};
}

// A wave's slot (wave-uniform), and this lane's query in it.
struct PaPlace : PaSlot {
    int pos, z;                       // this lane's query position and row (clamped into the batch)
    bool store;

    __device__ __forceinline__ explicit PaPlace(const PrefillAttnParams& p)
        : PaSlot(pa_slot(pa_batch(p), int(blockIdx.x), __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave)))
    {
        pos = tile * kPaTile + int(threadIdx.x & 15);
        z = min(max(pos - p.p0, 0), p.rows - 1);
        store = live && pos >= p.p0 && pos < p.p0 + p.rows;
    }
    // 16-key blocks of chunk c that every query of the tile sees whole
    __device__ __forceinline__ int full(int c) const { return min(4, tile - c * (kAttnChunk / kPaTile)); }
};

// This wave's quarter of chunk c's rows straight into LDS, 1 KB (four rows)
// per instruction; K: 16-byte piece q of row r at slot q ^ (r & 15).  Rows
// past the batch's last position re-read it (they are masked).
template <bool K>
__device__ __forceinline__ void pa_copy(const PrefillAttnParams& p, const PaPlace& w, int c, uint16_t* lds)
{
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave);
    const int lane = threadIdx.x & (kWave - 1);
    const uint16_t* base = (K ? p.keys : p.values) + size_t(w.kvh) * kPaD + size_t(c) * kAttnChunk * size_t(p.time_stride);
    const int last = p.p0 + p.rows - 1 - c * kAttnChunk;
#pragma unroll
    for (int i = 0; i < kAttnChunk / 4 / kPaWaves; ++i) {
        const int ins = wave + kPaWaves * i;
        const int r = 4 * ins + (lane >> 4);
        const int piece = K ? (lane & 15) ^ (r & 15) : lane & 15;
        dma16(base, uint32_t(min(r, last)) * uint32_t(p.time_stride) * 2u + uint32_t(piece) * 16u,
              lds_addr(lds) + uint32_t(ins) * 1024u);
    }
}

// The wave's query rows: q[j] of lane group g = dim 32 g + j of query lane % 16.
__device__ __forceinline__ void pa_load_q(const PrefillAttnParams& p, const PaPlace& w, float (&q)[32])
{
    const int g = (threadIdx.x & (kWave - 1)) >> 4;
    const float4* src = reinterpret_cast<const float4*>(p.q + (size_t(w.z) * p.heads + w.h) * kPaD + 32 * g);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float4 v = src[i];
        q[4 * i] = v.x;
        q[4 * i + 1] = v.y;
        q[4 * i + 2] = v.z;
        q[4 * i + 3] = v.w;
    }
}

__device__ __forceinline__ void pa_store_out(const PrefillAttnParams& p, const PaPlace& w, float L, const f32x16& oe,
                                             const f32x16& oo)
{
    const int g = (threadIdx.x & (kWave - 1)) >> 4;
    const float inv = 1.0f / L;
    float* out = p.out + (size_t(w.z) * p.heads + w.h) * kPaD + 8 * g;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        float4* dst = reinterpret_cast<float4*>(out + 32 * b);
        dst[0] = make_float4(oe[4 * b] * inv, oo[4 * b] * inv, oe[4 * b + 1] * inv, oo[4 * b + 1] * inv);
        dst[1] = make_float4(oe[4 * b + 2] * inv, oo[4 * b + 2] * inv, oe[4 * b + 3] * inv, oo[4 * b + 3] * inv);
    }
}

constexpr int kPaScoreVecs = kAttnChunk * kPaTile / 4;   // float4s of a tile's scores for one chunk and head

// A pass over the keys that writes each chunk's masked scores to the
// workspace and keeps their maximum, then a pass over the values that reads
// them back (one chunk ahead).  Per (tile, head, chunk) 256 matrix
// instructions and 8 KB of traffic, where a second score pass costs 128
// more instructions and their tree sums.
__global__ __launch_bounds__(kPaWaves * kWave, 3) void prefill_attention_kernel(PrefillAttnParams p)
{
    __shared__ alignas(16) uint16_t lds[2][kAttnChunk * kPaD];
    const PaPlace w(p);
    const int lane = threadIdx.x & (kWave - 1);
    const int nb = w.nc_block;
    pa_copy<true>(p, w, 0, lds[0]);
    float4* sc = reinterpret_cast<float4*>(p.part) +
                 (size_t(pa_chunks_before(w.tile) - pa_chunks_before(p.p0 / kPaTile)) * size_t(p.heads) +
                  size_t(w.h) * size_t(w.nc)) * kPaScoreVecs + lane;
    float M = -__builtin_inff();
    {
        float q[32];
        pa_load_q(p, w, q);
#pragma unroll 1
        for (int c = 0; c < nb; ++c) {
            wait_all_memory();      // this step's copies
            lds_sync();
            if (c + 1 < nb) pa_copy<true>(p, w, c + 1, lds[(c + 1) & 1]);
            else pa_copy<false>(p, w, 0, lds[nb & 1]);
            if (c >= w.nc || !w.live) continue;          // (wave-uniform)
            f32x16 s = pa_scores(lds[c & 1], q);
            pa_mask(s, w.full(c) < 4, w.pos - c * kAttnChunk + 1);
            M = fmaxf(M, pa_lane_max(s));
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sc[(4 * c + i) * kWave] = make_float4(s[4 * i], s[4 * i + 1], s[4 * i + 2], s[4 * i + 3]);
        }
    }
    M = groups_max(M);
    auto load = [&](int c, f32x16& s) {                  // (this lane wrote them)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = sc[(4 * c + i) * kWave];
            s[4 * i] = v.x;
            s[4 * i + 1] = v.y;
            s[4 * i + 2] = v.z;
            s[4 * i + 3] = v.w;
        }
    };
    float L = 0.0f;
    f32x16 oe = {}, oo = {}, next = {};
    if (w.live) load(0, next);
#pragma unroll 1
    for (int c = 0; c < nb; ++c) {
        wait_all_memory();
        lds_sync();
        if (c + 1 < nb) pa_copy<false>(p, w, c + 1, lds[(nb + c + 1) & 1]);
        if (c >= w.nc || !w.live) continue;
        f32x16 s = next;
        if (c + 1 < w.nc) load(c + 1, next);
        float m, l;
        f32x16 ae, ao;
        pa_values(lds[(nb + c) & 1], s, w.full(c), m, l, ae, ao);
        pa_combine(M, m, l, ae, ao, L, oe, oo);
    }
    if (w.store) pa_store_out(p, w, L, oe, oo);
}

struct PaShared {
    alignas(16) uint16_t k[2][kAttnChunk * kPaD];
    alignas(16) uint16_t v[2][kAttnChunk * kPaD];
};

// Without stored scores.  PART: block (x, y) takes chunks [y * cpb, y * cpb +
// cpb) and writes chunk partials (one-chunk tiles their outputs); otherwise
// a block walks all chunks of its tiles twice, the first time for the
// scores' maximum alone.
template <bool PART>
__global__ __launch_bounds__(kPaWaves * kWave, 2) void prefill_attention_walk_kernel(PrefillAttnParams p)
{
    __shared__ PaShared S;
    const PaPlace w(p);
    const int g = (threadIdx.x & (kWave - 1)) >> 4;
    const int c_begin = PART ? int(blockIdx.y) * p.cpb : 0;
    const int c_end = PART ? min(w.nc_block, c_begin + p.cpb) : w.nc_block;
    if (c_begin >= c_end) return;                        // (block-uniform)
    const int first = PART ? 0 : w.nc_block;             // steps of the maximum pass
    const int steps = first + (c_end - c_begin);
    pa_copy<true>(p, w, c_begin, S.k[0]);
    if (first == 0) pa_copy<false>(p, w, c_begin, S.v[0]);
    float q[32];
    pa_load_q(p, w, q);
    float M = -__builtin_inff(), L = 0.0f;
    f32x16 oe = {}, oo = {};
#pragma unroll 1
    for (int st = 0; st < steps; ++st) {
        wait_all_memory();      // this step's copies
        lds_sync();
        if (st + 1 < steps) {
            const int nx = st + 1, c = nx < first ? nx : c_begin + nx - first;
            pa_copy<true>(p, w, c, S.k[nx & 1]);
            if (nx >= first) pa_copy<false>(p, w, c, S.v[nx & 1]);
        }
        const int c = st < first ? st : c_begin + st - first;
        if (c >= w.nc || !w.live) continue;              // (wave-uniform)
        f32x16 s = pa_scores(S.k[st & 1], q);
        pa_mask(s, w.full(c) < 4, w.pos - c * kAttnChunk + 1);
        if (st < first) {
            M = fmaxf(M, groups_max(pa_lane_max(s)));
            continue;
        }
        float m, l;
        f32x16 ae, ao;
        pa_values(S.v[st & 1], s, w.full(c), m, l, ae, ao);
        if (PART && w.nc > 1) {
            if (w.store) {
                float* pp = p.part + ((size_t(w.z) * p.heads + w.h) * p.part_chunks + c) * (kPaD + 2);
                if (g == 0) {
                    pp[0] = m;
                    pp[1] = l;
                }
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    *reinterpret_cast<float2*>(pp + 2 + 2 * (16 * (i >> 2) + 4 * g + (i & 3))) =
                        make_float2(ae[i], ao[i]);
            }
            continue;
        }
        if (PART) M = m;                                 // one chunk
        pa_combine(M, m, l, ae, ao, L, oe, oo);
    }
    if (w.store && pa_stores_output(PART, w.nc, c_begin)) pa_store_out(p, w, L, oe, oo);
}

// Workspace limit: batches whose scores exceed it take the two-pass form,
// which needs none (2048 tokens of 32 heads up to position 4096 store 805 MB;
// in two halves of half the blocks they took 1.16 times as long, and more in
// smaller pieces).
constexpr size_t kPaPartBytes = size_t(1) << 30;

constexpr size_t kPaPartialBytes = size_t(kPaD + 2) * 4;          // a query, head and chunk
constexpr size_t kPaScoreBytes = size_t(kPaScoreVecs) * 16;       // a tile, head and chunk

static size_t pa_part_bytes(const PrefillAttnParams& p)
{
    return size_t(pa_partials(pa_batch(p))) * size_t(p.heads) * kPaPartialBytes;
}
static size_t pa_score_bytes(const PrefillAttnParams& p)
{
    return size_t(pa_tile_chunks(pa_batch(p))) * size_t(p.heads) * kPaScoreBytes;
}

size_t prefill_attention_part_bytes(int rows, int heads, int capacity)
{
    const size_t partials = size_t(pa_max_partials(rows, heads, capacity)) * size_t(heads) * kPaPartialBytes;
    const size_t scores = size_t(pa_max_tile_chunks(rows, capacity)) * size_t(heads) * kPaScoreBytes;
    return std::min(std::max(partials, scores), kPaPartBytes);
}

hipError_t launch_prefill_attention(const PrefillAttnParams& a, hipStream_t s)
{
    if (a.rows < 1 || a.p0 < 0 || a.groups < 1 || a.groups > 8) return hipErrorInvalidValue;
    PrefillAttnParams p = a;
    p.heads = a.kv_heads * a.groups;
    const int nc = (p.p0 + p.rows - 1) / kAttnChunk + 1;
    AttnParams c{};
    c.q = p.q;
    c.keys = p.keys;
    c.values = p.values;
    c.time_stride = p.time_stride;
    c.context = p.p0 + 1;
    c.batch = p.rows;
    c.kv_heads = p.kv_heads;
    c.groups = p.groups;
    c.head_dim = kPaD;
    c.max_chunks = nc;
    c.part = p.part;
    c.out = p.out;
    // One query per block where tiles of 16 leave the chip idle or compute for
    // absent queries: one chunk (64 tokens: 8.8 us against 14.0), and one or
    // two queries (hq_prefill over 6 layers of 32 / 8 heads at position 24000:
    // one query 475 us against 714, two 575 against 719; three are even, four
    // take 773 against 725).
    if (nc == 1 || (p.rows <= 2 && pa_part_bytes(p) <= p.part_bytes))
        return launch_query_attention(c, s);
    // fewer blocks than CUs: chunk partials from several blocks per tile, as
    // many as fill two blocks per CU
    if (pa_takes_partials(pa_batch(p)) && pa_part_bytes(p) <= p.part_bytes) {
        const PaPartGrid g = pa_part_grid(pa_batch(p));
        p.cpb = g.cpb;
        p.part_chunks = nc;
        hipLaunchKernelGGL(prefill_attention_walk_kernel<true>, dim3(g.blocks, g.splits), dim3(kPaWaves * kWave), 0, s,
                           p);
        return launch_attention_combine(c, s);
    }
    const int blocks = pa_blocks_per_kv(pa_batch(p)) * p.kv_heads;
    if (pa_score_bytes(p) <= p.part_bytes)
        hipLaunchKernelGGL(prefill_attention_kernel, dim3(blocks), dim3(kPaWaves * kWave), 0, s, p);
    else
        hipLaunchKernelGGL(prefill_attention_walk_kernel<false>, dim3(blocks), dim3(kPaWaves * kWave), 0, s, p);
    return hipGetLastError();
}

}  // namespace hq
