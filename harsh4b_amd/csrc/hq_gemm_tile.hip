// hq_gemm_tile.hip - packed-int4 weights x int8 activation rows for batches
// of more than 32 rows (prompts; hq_gemm.hip's two_passes says which of 33 to
// 64 rows take its kernels twice instead): output tiles on v_mfma_i32_32x32x32_i8, the
// same integers as hq_gemm.hip's kernels.
//
// Activation rows go on the A side (output rows), weight rows on the B side
// (output columns), so a lane holds 16 rows of one output column and a store
// writes 128 contiguous bytes of two rows.  A block computes BM x BN outputs
// in steps of 128 columns of K, both operands copied straight to LDS
// (global_load_lds, no register round trip) a step ahead: the activations in
// the MFMA order they are stored in (bq_pos), the weights still packed, 64
// bytes per row, 16-byte pieces swizzled so that the 16 rows of a read phase
// cover every bank once.  The nibbles become bytes in registers (x 16, exact:
// hq_gemm.hip), once per wave that owns their columns.  A wave's 64 x 128
// tile reads 16 KB of LDS per 1024 MFMA cycles, half of what the LDS
// delivers beside four SIMDs.
#include <algorithm>

#include "hq_gemm_block.h"

namespace hq {

typedef int i32x16 __attribute__((ext_vector_type(16)));

enum TileEpi { TILE_OUT = 0, TILE_SWIGLU = 1, TILE_PART = 2 };

struct TileParams {
    const int8_t* x;          // activation tiles (bq_pos), row stride kp
    const float* act;         // [m]
    const uint8_t* w;         // [n, k/2] (SWIGLU: [2 n, k/2], gate rows then up rows)
    const float* ws;          // [n] ([2 n])
    float* out;               // [m, n]
    int32_t* acc_out;         // OUT: nullable [m, n]
    int32_t* part;            // PART: [splits, m, n], 16 x the partial sums
    int m, n, k, kp;
    int tiles_m, tiles_n, per_xcd, splits;
};

template <int N>
__device__ __forceinline__ void wait_vm()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// TM x TN tiles of 32 x 32 per wave, WM x WN waves, KG groups of them that
// take every KG-th step of K and add their integer sums in LDS.
template <int TM, int TN, int WM, int WN, int KG, int ST, int EPI, bool RAGGED>
__global__ __launch_bounds__(WM* WN* KG* kWave, 2) void gemm_tile_kernel(TileParams p)
{
    constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
    constexpr int W = WM * WN;
    constexpr int ABYTES = BM * 128, WBYTES = BN * 64;
    constexpr uint32_t STEP = ABYTES + WBYTES;
    constexpr int AI = ABYTES / 1024 / W, WI = WBYTES / 1024 / W;   // copies per wave and step
    static_assert(AI * W * 1024 == ABYTES && WI * W * 1024 == WBYTES, "whole copies per wave");
    static_assert(EPI != TILE_SWIGLU || TN % 2 == 0, "a wave holds gate and up columns of the same outputs");
    __shared__ alignas(16) uint8_t lds[KG * ST * (ABYTES + WBYTES)];
    static_assert(KG == 1 || (KG + 1) / 2 * BM * BN * 4 <= KG * ST * (ABYTES + WBYTES), "the sums alias the copies");
    __shared__ alignas(16) float act_s[BM];
    const int tid = threadIdx.x;
    const int wave_all = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid & (kWave - 1);
    const int wave = wave_all % W, kg = wave_all / W;   // wave of its K group
    const int r32 = lane & 31, g = lane >> 5;
    // consecutive tiles of an XCD (blocks go round robin over the 8) share
    // their weight columns in its L2
    const int t = (int(blockIdx.x) & 7) * p.per_xcd + (int(blockIdx.x) >> 3);
    if (t >= p.tiles_m * p.tiles_n) return;
    const int m0 = (t % p.tiles_m) * BM;
    const int tn = t / p.tiles_m;
    const int half = p.k >> 1;
    const int steps = (p.k + 127) >> 7;
    const int b0 = EPI == TILE_PART ? steps * int(blockIdx.y) / p.splits : 0;
    const int b1 = EPI == TILE_PART ? steps * (int(blockIdx.y) + 1) / p.splits : steps;
    const int rounds = (b1 - b0 + KG - 1) / KG;          // steps b0 + kg + KG * round

    // weight row of tile column c (rows past the matrix re-read its last)
    auto wrow = [&](int c) {
        if constexpr (EPI == TILE_SWIGLU) {
            const int j = c >> 5;   // 32-column blocks alternate gate, up
            return (j & 1 ? p.n : 0) + min(tn * (BN / 2) + (j >> 1) * 32 + (c & 31), p.n - 1);
        } else {
            return min(tn * BN + c, p.n - 1);
        }
    };
    const int last_tile = (p.m - 1) >> 4;
    const uint8_t* xbase = reinterpret_cast<const uint8_t*>(p.x);
    uint32_t aoff[AI], woff[WI], wpiece[WI];
#pragma unroll
    for (int i = 0; i < AI; ++i) {
        const int ins = wave + W * i;             // 1 KB: half of a 16-row tile's step
        aoff[i] = uint32_t(min(m0 / 16 + (ins >> 1), last_tile)) * 16u * uint32_t(p.kp) + uint32_t(ins & 1) * 1024u +
                  uint32_t(lane) * 16u;
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int c = 16 * (wave + W * i) + (lane >> 2);   // 1 KB: 16 rows x 64 bytes
        wpiece[i] = uint32_t((lane & 3) ^ ((c >> 2) & 3)) * 16u;
        woff[i] = uint32_t(wrow(c)) * uint32_t(half) + wpiece[i];
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds)) + uint32_t(wave) * 1024u;
    auto copy = [&](int round, uint32_t buf) {   // buf: byte offset of the step's buffer
        const int s = min(b0 + kg + KG * round, steps - 1);
#pragma unroll
        for (int i = 0; i < AI; ++i)
            dma16(xbase + size_t(s) * 2048, aoff[i], lds0 + buf + uint32_t(W * i) * 1024u);
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            uint32_t off = woff[i];
            if constexpr (RAGGED)   // pieces past the row re-read its last one (zeroed below)
                off -= uint32_t(max(0, s * 64 + int(wpiece[i]) - (half - 16)));
            dma16(p.w + size_t(s) * 64, off, lds0 + buf + uint32_t(ABYTES) + uint32_t(W * i) * 1024u);
        }
    };

    i32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = i32x16{};
    const int wm = wave % WM, wn = wave / WM;
    constexpr uint32_t m4 = 0xF0F0F0F0u;
    if constexpr (EPI != TILE_PART) {
        for (int i = tid; i < BM; i += W * KG * kWave) act_s[i] = p.act[min(m0 + i, p.m - 1)];
    }
    wait_all_memory();   // (the copies are counted from here)
    uint32_t buf = uint32_t(kg) * ST * STEP;   // this round's buffer, and the one freed by the last
    const uint32_t buf_first = buf, buf_last = buf + (ST - 1) * STEP;
    uint32_t next = buf_last;
#pragma unroll
    for (int i = 0; i < ST - 1; ++i)
        if (i < rounds) copy(i, buf + uint32_t(i) * STEP);
#pragma unroll 1
    for (int r = 0; r < rounds; ++r) {
        // this round's copies: all but those of the next ST - 2 rounds
        if (r + ST - 2 < rounds) wait_vm<(ST - 2) * (AI + WI)>();
        else wait_vm<0>();
        lds_sync();
        if (r + ST - 1 < rounds) copy(r + ST - 1, next);
        const uint8_t* a_s = lds + buf + wm * TM * 32 * 128;
        const uint8_t* w_s = lds + buf + ABYTES + wn * TN * 32 * 64;
        next = buf;
        buf = buf == buf_last ? buf_first : buf + STEP;
        const int s = b0 + kg + KG * r;
        if (KG > 1 && s >= b1) continue;                 // (wave-uniform; the last round)
        // every operand read of the step first, then its products
        i32x4 a[2][TM][2], w[2][TN];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            // lane group g: the 16-byte packed piece q = 2 u + g, i.e. columns
            // 32 q .. 32 q + 31 of the step, as two operands of 16 columns
            const int q = 2 * u + g;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    a[u][i][h] = *reinterpret_cast<const i32x4*>(a_s + (2 * i + (r32 >> 4)) * 2048 + h * 1024 +
                                                                 q * 256 + (r32 & 15) * 16);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int c = 32 * j + r32;
                w[u][j] = *reinterpret_cast<const i32x4*>(w_s + c * 64 + (q ^ ((c >> 2) & 3)) * 16);
                if constexpr (RAGGED) {
                    if (s * 64 + q * 16 >= half) w[u][j] = i32x4{0, 0, 0, 0};
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const i32x4 v = w[u][j];
                const i32x4 b0 = {int((uint32_t(v[0]) << 4) & m4), int(uint32_t(v[0]) & m4),
                                  int((uint32_t(v[1]) << 4) & m4), int(uint32_t(v[1]) & m4)};
                const i32x4 b1 = {int((uint32_t(v[2]) << 4) & m4), int(uint32_t(v[2]) & m4),
                                  int((uint32_t(v[3]) << 4) & m4), int(uint32_t(v[3]) & m4)};
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u][i][0], b0, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[u][i][1], b1, acc[i][j], 0, 0, 0);
                }
            }
    }

    // the K groups' sums: the upper half of the groups to the lower, until one
    // holds them all
    if constexpr (KG > 1) {
        i32x4* sums = reinterpret_cast<i32x4*>(lds);
#pragma unroll
        for (int half_g = KG / 2; half_g >= 1; half_g /= 2) {
            lds_sync();
            i32x4* mine = sums + size_t((kg % half_g) * W + wave) * (TM * TN * 4 * kWave) + lane;
            if (kg >= half_g && kg < 2 * half_g) {
#pragma unroll
                for (int i = 0; i < TM * TN * 4; ++i) {
                    const i32x16& c = acc[i / 4 / TN][i / 4 % TN];
                    mine[i * kWave] = i32x4{c[4 * (i % 4)], c[4 * (i % 4) + 1], c[4 * (i % 4) + 2], c[4 * (i % 4) + 3]};
                }
            }
            lds_sync();
            if (kg < half_g) {
#pragma unroll
                for (int i = 0; i < TM * TN * 4; ++i) {
                    const i32x4 v = mine[i * kWave];
                    i32x16& c = acc[i / 4 / TN][i / 4 % TN];
#pragma unroll
                    for (int e = 0; e < 4; ++e) c[4 * (i % 4) + e] += v[e];
                }
            }
        }
        if (kg != 0) return;
    }

    // element e of a 32 x 32 tile: row 8 (e / 4) + 4 g + e % 4, column r32
    const int mw = wm * TM * 32 + 4 * g;
    float ws_c[TN];
    if constexpr (EPI != TILE_PART) {
#pragma unroll
        for (int j = 0; j < TN; ++j) ws_c[j] = p.ws[wrow((wn * TN + j) * 32 + r32)];
    }
    constexpr int NB = EPI == TILE_SWIGLU ? BN / 2 : BN;   // output columns of the block
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int e4 = 0; e4 < 4; ++e4) {
            float4 am = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if constexpr (EPI != TILE_PART) am = *reinterpret_cast<const float4*>(act_s + mw + 32 * i + 8 * e4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int mm = m0 + mw + 32 * i + 8 * e4 + e;
                const float a = e == 0 ? am.x : e == 1 ? am.y : e == 2 ? am.z : am.w;
                const size_t row = size_t(mm) * p.n;
#pragma unroll
                for (int j = 0; j < TN; j += (EPI == TILE_SWIGLU ? 2 : 1)) {
                    const int col = EPI == TILE_SWIGLU ? (wn * TN + j) * 16 : (wn * TN + j) * 32;
                    const int n = tn * NB + col + r32;
                    const bool ok = mm < p.m && n < p.n;
                    const int v = acc[i][j][4 * e4 + e];
                    if constexpr (EPI == TILE_PART) {
                        if (ok) p.part[size_t(blockIdx.y) * size_t(p.m) * p.n + row + n] = v;
                    } else if constexpr (EPI == TILE_SWIGLU) {
                        const float gv = (float(v >> 4) * a) * ws_c[j];
                        const float uv = (float(acc[i][j + 1][4 * e4 + e] >> 4) * a) * ws_c[j + 1];
                        const float t1 = 1.0f + spec_expf_sel(-gv);
                        if (ok) p.out[row + n] = (gv / t1) * uv;
                    } else {
                        if (ok) p.out[row + n] = (float(v >> 4) * a) * ws_c[j];
                        if (ok && p.acc_out) p.acc_out[row + n] = v >> 4;
                    }
                }
            }
        }
    }
}

template <int TM, int TN, int WM, int WN, int KG, int ST, int EPI>
static hipError_t launch_tile(TileParams p, hipStream_t s)
{
    constexpr int BM = 32 * TM * WM, BN = EPI == TILE_SWIGLU ? 16 * TN * WN : 32 * TN * WN;
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = (p.n + BN - 1) / BN;
    p.per_xcd = (p.tiles_m * p.tiles_n + 7) / 8;
    const dim3 grid(8 * p.per_xcd, EPI == TILE_PART ? p.splits : 1), block(WM * WN * KG * kWave);
    if (p.k & 127)
        hipLaunchKernelGGL((gemm_tile_kernel<TM, TN, WM, WN, KG, ST, EPI, true>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((gemm_tile_kernel<TM, TN, WM, WN, KG, ST, EPI, false>), grid, block, 0, s, p);
    return hipGetLastError();
}

// 64 x 64 tiles of an output (n: weight rows).
static long long tiles64(int m, long long n) { return ((m + 63LL) / 64) * ((n + 63) / 64); }

// By the number of 64 x 64 tiles (times in us over weights that come from
// HBM, M rows of the 2560 x 4096, 6144 x 2560, 2560 x 9728 and 19456 x 2560
// matrices): up to 200, 64 x 64 blocks of two K groups (128 x 6144 10.7,
// where 64 x 128 blocks take 12.8); up to 960, 64 x 128 blocks
// with four steps in flight (501 x 6144 18.9, against 22.2 and, of 128 x 128,
// 21.9; 160 x 19456 18.6, 24.7, 24.4); beyond, 128 x 128 blocks, three per CU
// (700 x 6144 23.8 against 26.7; 2000 x 19456 113 against 169: 1.8 POP/s,
// the library's int8 product reaches 1.7 here on 8192 cubed).
constexpr long long kSmallTiles = 200, kMidTiles = 960;
template <int EPI>
static hipError_t run_tile(const TileParams& p, hipStream_t s)
{
    const long long t = tiles64(p.m, EPI == TILE_SWIGLU ? 2LL * p.n : p.n);
    if constexpr (EPI != TILE_SWIGLU) {   // (SwiGLU of so few tiles follows K parts)
        if (t <= kSmallTiles) return launch_tile<1, 2, 2, 1, 2, 3, EPI>(p, s);
    }
    if (t <= kMidTiles) return launch_tile<1, 2, 2, 2, 1, 4, EPI>(p, s);
    return launch_tile<2, 2, 2, 2, 1, 2, EPI>(p, s);
}

static TileParams tile_params(const int8_t* x, const float* act, const uint8_t* w, const float* ws, float* out, int m,
                              int n, int k)
{
    TileParams p{};
    p.x = x;
    p.act = act;
    p.w = w;
    p.ws = ws;
    p.out = out;
    p.m = m;
    p.n = n;
    p.k = k;
    p.kp = gemm_padded_k(k);
    return p;
}

// K parts of a GEMM whose consumer adds them: 4 up to 80 tiles of 64 x 64
// (64 x 2560 x 9728: 9.4 us against 21.9 whole and 11.9 in two parts), 2 up
// to kSmallTiles (320 x 2560 x 9728: 19.2 against 22.1 and 21.8), 0 beyond.
int gemm_part_splits(int m, int n, int k)
{
    const long long t = tiles64(m, n);
    if (t > kSmallTiles || !gemm_tile_fits(m, n, k)) return 0;
    return t <= 80 ? 4 : 2;
}
size_t gemm_part_bytes() { return 2 * kSmallTiles * 64 * 64 * 4; }
static_assert(2 * kSmallTiles >= 4 * 80, "both part counts fit");

hipError_t gemm_tile_part(const int8_t* x, const uint8_t* w, int32_t* part, int splits, int m, int n, int k,
                          hipStream_t s)
{
    if (splits < 1 || splits != gemm_part_splits(m, n, k)) return hipErrorInvalidValue;
    TileParams p = tile_params(x, nullptr, w, nullptr, nullptr, m, n, k);
    p.part = part;
    p.splits = splits;
    return launch_tile<1, 2, 2, 1, 2, 3, TILE_PART>(p, s);
}

bool gemm_tile_fits(int m, int n, int k)
{
    // 32-bit operand offsets
    return m > 0 && size_t(gemm_padded_m(m)) * size_t(gemm_padded_k(k)) < (size_t(1) << 32) &&
           size_t(n) * size_t(k >> 1) < (size_t(1) << 32);
}

hipError_t gemm_tile_run(const int8_t* x, const float* act, const uint8_t* w, const float* ws, float* out, int m,
                         int n, int k, int32_t* acc_out, hipStream_t s)
{
    if (!gemm_tile_fits(m, n, k)) return hipErrorInvalidValue;
    TileParams p = tile_params(x, act, w, ws, out, m, n, k);
    p.acc_out = acc_out;
    return run_tile<TILE_OUT>(p, s);
}

hipError_t gemm_tile_swiglu(const int8_t* x, const float* act, const uint8_t* w, const float* ws, float* out, int m,
                            int n, int k, hipStream_t s)
{
    if (!gemm_tile_fits(m, 2 * n, k) || gemm_part_splits(m, 2 * n, k) != 0) return hipErrorInvalidValue;
    return run_tile<TILE_SWIGLU>(tile_params(x, act, w, ws, out, m, n, k), s);
}

}  // namespace hq
