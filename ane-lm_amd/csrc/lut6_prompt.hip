// LUT6 projections of many inputs at once (prompt prefill): Y[b][r] (+)= sum_c
// W[r][c] X[b][c] for batches past what the register-window kernel of
// lut6_mfma.hip takes in one or two passes of 32.
//
// That kernel decodes every weight once per 32 inputs, and the decode (two
// weights per LDS lookup) bounds it: a 4096-token prompt decoded each weight
// 128 times, 5.1 ms for the 2560 -> 2 x 9216 -> 2560 FFN block.  Here the
// weights are decoded once into fp16 (exactly: a LUT entry is an fp16 value),
// the inputs are rounded to fp16 once (as every LUT6 path takes them), and one
// fp16 MFMA product with fp32 accumulation follows: that block takes 795 us
// (the two products with their preparation 410 + 235).
// Reference math: matvec (core/cpu_ops.cpp:77-80) on the dequantised weights,
// per input.
//
// Operand layout.  Both operands are stored in blocks of 32 columns,
// [column block][row][32 halves], so one pipeline stage of a tile is one
// contiguous piece of memory and goes to LDS in 1 KiB wave loads without any
// address arithmetic.  Within a row's 64 bytes the four 16-byte chunks are
// permuted by (row / 2) % 4, so the 8 lanes that read 8 consecutive rows'
// chunk c in one LDS cycle fall on distinct banks.  Rows are padded to whole
// tiles: a tile's loads stay inside the buffers, and what they read past the
// last row only reaches outputs that are not stored.
#include "anelm_internal.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace anelm {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kKB = 32;            // columns per block (one pipeline stage)
constexpr int kRowB = kKB * 2;     // bytes of one row in one block
constexpr int kChain = 8;          // column blocks per accumulation chain (256 columns)

// Byte offset of 16-byte chunk c of row r in its column block.
__device__ __forceinline__ int chunk_off(int r, int c) { return r * kRowB + ((c ^ (r >> 1)) & 3) * 16; }

struct PrepArgs {
    char* xb;              // out: X blocks [nk][mp] rows
    char* wb;              // out: W blocks [nk][np] rows
    const float* x;        // [batch][in_dim]
    const uint8_t* w;      // [out_dim][in_dim * 3 / 4]
    const uint16_t* lut;   // [out_dim / 32][64]
    int batch, out_dim, in_dim, mp, np, nk;
    int groups, wy, passes;   // W part: out_dim / 32 groups x wy ranges of `passes` column passes
};

// X rows of one workgroup: 64 rows x one column block, fp32 -> fp16, zeros
// past in_dim.  Thread = (row, chunk): 32 bytes read, 16 written; a wave
// covers 16 rows x 64 bytes.
__device__ __forceinline__ void convert_x(const PrepArgs& a, int id) {
    const int kb = id % a.nk, r = (id / a.nk) * 64 + (threadIdx.x >> 2), c = threadIdx.x & 3;
    if (r >= a.batch) return;
    const int c0 = kb * kKB + c * 8;
    half8 h = half8{};
    if (c0 < a.in_dim) {   // in_dim is a multiple of 16
        const float4 u = *reinterpret_cast<const float4*>(a.x + (size_t)r * a.in_dim + c0);
        const float4 v = *reinterpret_cast<const float4*>(a.x + (size_t)r * a.in_dim + c0 + 4);
        h = half8{(_Float16)u.x, (_Float16)u.y, (_Float16)u.z, (_Float16)u.w,
                  (_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
    }
    *reinterpret_cast<half8*>(a.xb + (size_t)kb * a.mp * kRowB + chunk_off(r, c)) = h;
}

// W rows of one LUT group (32 rows) x a range of columns -> blocks of fp16.
// Per pass of 512 columns the packed rows go to LDS with 16-byte loads (the
// next pass's in flight meanwhile); then a thread takes one 16-byte output
// chunk (8 columns = 6 packed bytes) at a time, 16 rows x 4 chunks per wave,
// so every store instruction writes 1 KiB of consecutive memory.  The pair
// table T[(i1 << 6) | i0] = (lut[i0], lut[i1]) turns 12 bits into two weights
// per LDS read.
constexpr int kDecCols = 512;
constexpr int kDecRow = kDecCols * 3 / 4 + 16;   // staged row pitch (bytes): rows start 4 banks apart
typedef uint32_t u32x4_dw __attribute__((ext_vector_type(4), aligned(4)));   // rows start at multiples of 12 bytes
__device__ __forceinline__ void decode_w(const PrepArgs& a, uint32_t* tab, char* raw, int g, int range) {
    const int tid = threadIdx.x, lane = tid & 63, in_dim = a.in_dim;
    const uint32_t mine = a.lut[(size_t)g * 64 + lane];
    for (int i1 = tid >> 6; i1 < 64; i1 += 4)
        tab[i1 * 64 + lane] = mine | ((uint32_t)__builtin_amdgcn_readlane((int)mine, i1) << 16);
    const int row_bytes = in_dim * 3 / 4;   // a multiple of 12
    const uint8_t* base = a.w + (size_t)g * 32 * row_bytes;
    constexpr int CH = kDecCols * 3 / 4 / 16;   // 16-byte chunks per staged row
    constexpr int NC = 32 * CH / 256;           // per thread
    auto fetch = [&](int p, u32x4 (&v)[NC]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int e = tid + 256 * i, r = e / CH, o = p * (kDecCols * 3 / 4) + (e % CH) * 16;
            const uint8_t* src = base + (size_t)r * row_bytes + o;
            v[i] = u32x4{0u, 0u, 0u, 0u};
            if (o + 16 <= row_bytes) {
                v[i] = *reinterpret_cast<const u32x4_dw*>(src);
            } else if (o < row_bytes) {   // 4, 8 or 12 bytes left
                v[i].x = *reinterpret_cast<const uint32_t*>(src);
                if (o + 4 < row_bytes) v[i].y = *reinterpret_cast<const uint32_t*>(src + 4);
                if (o + 8 < row_bytes) v[i].z = *reinterpret_cast<const uint32_t*>(src + 8);
            }
        }
    };
    const int p0 = range * a.passes, p1 = min(p0 + a.passes, (in_dim + kDecCols - 1) / kDecCols);
    u32x4 v[NC];
    if (p0 < p1) fetch(p0, v);
    for (int p = p0; p < p1; p++) {
        __syncthreads();   // (the first one covers the table)
#pragma unroll
        for (int i = 0; i < NC; i++) {
            const int e = tid + 256 * i;
            *reinterpret_cast<u32x4*>(raw + (e / CH) * kDecRow + (e % CH) * 16) = v[i];
        }
        __syncthreads();
        if (p + 1 < p1) fetch(p + 1, v);
        const int r = (tid >> 2) & 31, c = tid & 3, kb0 = tid >> 7;
#pragma unroll
        for (int i = 0; i < kDecCols / kKB / 2; i++) {
            const int kl = 2 * i + kb0, kb = p * (kDecCols / kKB) + kl;
            const char* src = raw + r * kDecRow + kl * 24 + c * 6;
            // 6 bytes from a 2-byte aligned address: two dwords, shifted by 0 or 16
            const uint32_t* s4 = reinterpret_cast<const uint32_t*>(src - 2 * (c & 1));
            const uint32_t lo = s4[0], hi = s4[1];
            const int sh = 16 * (c & 1);
            const uint32_t f0 = __builtin_amdgcn_alignbit(hi, lo, sh), f1 = hi >> sh;
            u32x4 o;
            o.x = tab[f0 & 4095u];
            o.y = tab[(f0 >> 12) & 4095u];
            o.z = tab[__builtin_amdgcn_alignbit(f1, f0, 24) & 4095u];
            o.w = tab[(f1 >> 4) & 4095u];
            const int col = kb * kKB + c * 8;
            if (col >= in_dim) o = u32x4{0u, 0u, 0u, 0u};
            if (kb < a.nk)
                *reinterpret_cast<u32x4*>(a.wb + (size_t)kb * a.np * kRowB + chunk_off(g * 32 + r, c)) = o;
        }
    }
}

// One launch prepares both operands: the W workgroups first (they take
// longer), then the X ones.
__global__ __launch_bounds__(256) void prompt_prep_kernel(const PrepArgs a) {
    __shared__ uint32_t tab[4096];
    __shared__ __attribute__((aligned(16))) char raw[32 * kDecRow];
    const int id = blockIdx.x, nw = a.groups * a.wy;
    if (id < nw) decode_w(a, tab, raw, id % a.groups, id / a.groups);
    else convert_x(a, id - nw);
}

struct PromptArgs {
    float* y;              // [m][ldy]
    const char* x;         // blocks of [mp] rows
    const char* w;         // blocks of [np] rows
    int m, n;              // valid rows of x, of w
    int mp, np;            // padded rows
    int nk;                // column blocks
    int ksplit;            // gridDim.y slices of the column blocks; slice s writes y + s * sy
    long sy;
    long ldy;
    int accumulate;
};

template <int... S, class F>
__device__ __forceinline__ void for_each_stage(std::integer_sequence<int, S...>, F f) {
    (f(std::integral_constant<int, S>{}), ...);
}

// Tile of BM inputs x BN weight rows, WM x WN waves; wave tile (BM / WM) x
// (BN / WN) in 32x32 blocks of v_mfma_f32_32x32x16_f16 (A = inputs, B = weight
// rows, so 32 lanes hold 32 consecutive outputs of one input).  NS stages of
// 32 columns in LDS, NS - 1 ahead in flight; the operands of the second half
// of a stage are read while the first half is multiplied, those of the next
// stage's first half (behind the one barrier per stage) while the second is.
// The products accumulate in chains of kChain stages, each added to a sum in
// fp32: one chain over all columns rounds at the size of the whole sum every
// time, 3.2e-7 off 64 bits at 2560 columns and 6.1e-7 at 9216, where the passes
// of 32 inputs and these chains are 1.2e-7 and 1.3 to 1.5e-7 off.  A wave's
// blocks end their chains in different stages, so the additions hide behind the
// other blocks' products (all at once they cost 5 % of the FFN block).
// Bound: the matrix units' power (whole call with the preparation, us: 4096 x
// 18432 x 2560 410, 4096 x 2560 x 9216 235; the library's 8192^3 product runs
// at 1.19 PFLOP/s on the same card; with 160 of 256 CUs busy each CU runs 1.6
// times faster).
template <int BM, int BN, int WM, int WN, int NS>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(WM * WN / 4, WM * WN / 4)))
void prompt_gemm_kernel(const PromptArgs a) {
    constexpr int NW = WM * WN, MI = BM / WM / 32, NI = BN / WN / 32;
    constexpr int STAGE = (BM + BN) * kRowB, PIECES = STAGE / 1024, LPW = (PIECES + NW - 1) / NW;
    static_assert(PIECES * 1024 == STAGE && BM * kRowB % 1024 == 0, "whole wave loads");
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w % WM, wn = w / WM;
    // tile of this workgroup: XCD-contiguous, 4 row tiles x column tiles
    const int tm = (a.m + BM - 1) / BM, tn = (a.n + BN - 1) / BN, nt = tm * tn;
    int id = blockIdx.x;
    {
        const int per = nt / 8, rem = nt % 8, xcd = id & 7, k = id >> 3;
        id = xcd * per + min(xcd, rem) + k;
    }
    constexpr int GM = 4;
    const int grp = id / (GM * tn), first = grp * GM, gm = min(GM, tm - first), in = id - grp * GM * tn;
    const int m0 = (first + in % gm) * BM, n0 = (in / gm) * BN;

    // piece c of a stage: X pieces first, then W pieces
    constexpr int XP = BM * kRowB / 1024;
    const size_t xstep = (size_t)a.mp * kRowB, wstep = (size_t)a.np * kRowB;
    const int k0 = a.nk * (int)blockIdx.y / a.ksplit, nk = a.nk * ((int)blockIdx.y + 1) / a.ksplit - k0;
    const char* xs = a.x + (size_t)m0 * kRowB + k0 * xstep;
    const char* ws = a.w + (size_t)n0 * kRowB - (size_t)BM * kRowB + k0 * wstep;
    const uint32_t lane16 = lane * 16;
    auto issue = [&](int i) __attribute__((always_inline)) {
        const int k = min(i, nk - 1);   // past the end: the last block again, into a buffer nobody reads
        char* dst = lds + (i % NS) * STAGE;
        const char *xk = xs + k * xstep, *wk = ws + k * wstep;
#pragma unroll
        for (int j = 0; j < LPW; j++) {
            const int c = min(w * LPW + j, PIECES - 1);
            const char* src = (c < XP ? xk : wk) + c * 1024;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + lane16),
                                             (__attribute__((address_space(3))) void*)(dst + c * 1024), 16, 0, 0);
        }
    };
    const int lr = lane & 31, lh = lane >> 5;
    // chunk 2 ks + lh of row lr (+ 32 j) of the wave's rows; rows 32 apart keep the permutation
    const int a_off = (wm * (BM / WM) + lr) * kRowB, b_off = BM * kRowB + (wn * (BN / WN) + lr) * kRowB;
    const int sw = (lr >> 1) & 3;
    float16_t acc[MI][NI], sum[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++) acc[i][j] = sum[i][j] = float16_t{};
    half8 fa[2][MI], fb[2][NI];
    auto read = [&](int i, int ks) __attribute__((always_inline)) {
        const char* base = lds + (i % NS) * STAGE + (((2 * ks + lh) ^ sw) & 3) * 16;
#pragma unroll
        for (int j = 0; j < MI; j++) fa[ks][j] = *reinterpret_cast<const half8*>(base + a_off + j * 32 * kRowB);
#pragma unroll
        for (int j = 0; j < NI; j++) fb[ks][j] = *reinterpret_cast<const half8*>(base + b_off + j * 32 * kRowB);
    };
    constexpr int NB = MI * NI;
    static_assert(NB <= kChain, "a stage of the chain for every block");
    // `last`: the block multiplied last, `fresh`: it starts a new chain
    auto mul = [&](int ks, int last, bool fresh) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int e = (last + 1 + b) % NB, i = e / NI, j = e % NI;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[ks][i], fb[ks][j],
                                                              fresh && e == last ? float16_t{} : acc[i][j], 0, 0, 0);
        }
    };
    constexpr int VM = (NS - 2) * LPW;   // loads that may stay in flight while the next stage is used
    constexpr int kWait = 0x0070 | (VM & 15) | ((VM >> 4) << 14);   // vmcnt(VM), lgkmcnt(0)
    for (int i = 0; i < NS - 1; i++) issue(i);
    __builtin_amdgcn_s_waitcnt(kWait);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0);
    // Stage i.  FL in 0 .. NB - 1: block FL of the wave's ends its chain of
    // kChain stages here: it is added to the sum while the other blocks' products run.
    auto stage = [&](int i, auto fl) __attribute__((always_inline)) {
        constexpr int FL = decltype(fl)::value;
        constexpr bool flush = FL >= 0 && FL < NB;
        issue(i + NS - 1);
        read(i, 1);
        if constexpr (flush) sum[FL / NI][FL % NI] += acc[FL / NI][FL % NI];
        mul(0, flush ? FL : NB - 1, flush);
        // interleave: one load or read between the products
#pragma unroll
        for (int s = 0; s < NB; s++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(kWait);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read(i + 1, 0);
        mul(1, NB - 1, false);
#pragma unroll
        for (int s = 0; s < NB; s++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
    };
    int i = 0;
    for (; i + kChain <= nk; i += kChain)
        for_each_stage(std::make_integer_sequence<int, kChain>{}, [&](auto s) __attribute__((always_inline)) {
            stage(i + decltype(s)::value, s);
        });
    auto end_chains = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < MI; x++)
#pragma unroll
            for (int y = 0; y < NI; y++) {
                sum[x][y] += acc[x][y];
                acc[x][y] = float16_t{};
            }
    };
    end_chains();
    if (i < nk) {   // (fewer than kChain stages left)
        for (; i < nk; i++) stage(i, std::integral_constant<int, -1>{});
        end_chains();
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);   // no load into LDS outlives the workgroup
    float* y = a.y + blockIdx.y * a.sy;
    // C layout: element e of lane l is input row 8 (e / 4) + 4 (l / 32) + e % 4,
    // weight row l % 32: 32 lanes write 128 consecutive bytes
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int row = m0 + wm * (BM / WM) + i * 32 + 8 * (e >> 2) + 4 * lh + (e & 3);
            if (row >= a.m) continue;
            float* yr = y + (size_t)row * a.ldy;
#pragma unroll
            for (int j = 0; j < NI; j++) {
                const int col = n0 + wn * (BN / WN) + j * 32 + lr;
                if (col >= a.n) continue;
                yr[col] = a.accumulate ? yr[col] + sum[i][j][e] : sum[i][j][e];
            }
        }
}

// Which tile and how many column slices: estimated time of each pair.  `one`:
// a lone tile's 32-column stage; `full`: a stage of 256 tiles running at once,
// where the chip's throughput bounds it; a partly filled round lies between.
// Column slices (partial sums added by split_sum in a fixed order) fill the
// chip when there are few tiles; they cost their traffic, which mostly stays in
// the last-level cache.  The constants are a fit of the order of the pairs'
// whole-call times (their unit is near a microsecond) over 77 shapes (65..4096
// inputs of seven projections) x 16 pairs: what the model picks is within 0.3 %
// of the best pair on average and 4 % at most.  256 x 192 is the largest tile
// whose accumulators and sums fit a wave's 256 registers.
struct Tile {
    int bm, bn;
    float one, full;
};
constexpr Tile kTiles[] = {{256, 192, 0.774f, 0.898f},
                           {256, 128, 0.476f, 0.711f},
                           {128, 128, 0.447f, 0.454f},
                           {64, 128, 0.249f, 0.285f}};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kSplits[] = {1, 2, 4, 8};

struct Plan {
    int m, n, nk, tile, splits;
    int mp, np;
    size_t xb, wb, bytes;   // operand blocks of X and W; with the slices' partial sums
};

Plan make_plan(int m, int n, int nk, bool may_split, int cus) {
    Plan p{m, n, nk, -1, 1, 0, 0, 0, 0, 0};
    float best = 0.f;
    for (int t = 0; t < kNumTiles; t++)
        for (int s : kSplits) {
            if (s > 1 && (!may_split || nk / s < 8)) continue;
            const Tile& k = kTiles[t];
            const long units = (long)((m + k.bm - 1) / k.bm) * ((n + k.bn - 1) / k.bn) * s;
            const long rounds = units / cus, rem = units % cus;
            const float stage = (float)rounds * k.full + (rem ? std::max(k.one, k.full * (float)rem / (float)cus) : 0.f);
            float us = stage * (float)nk / (float)s;
            if (s > 1) us += 2.63f + (float)(2 * s + 1) * (float)m * (float)n * 4.f / 5.37e6f;
            if (p.tile < 0 || us < best) best = us, p.tile = t, p.splits = s;
        }
    const Tile& k = kTiles[p.tile];
    p.mp = (m + k.bm - 1) / k.bm * k.bm;
    p.np = (n + k.bn - 1) / k.bn * k.bn;
    p.xb = (size_t)nk * p.mp * kRowB;
    p.wb = (size_t)nk * p.np * kRowB;
    p.bytes = p.xb + p.wb + (p.splits > 1 ? (size_t)p.splits * m * n * sizeof(float) : 0);
    return p;
}

template <int BM, int BN, int WM, int WN>
int gemm_launch(const PromptArgs& a, hipStream_t st) {
    constexpr int NS = 4, kLds = NS * (BM + BN) * kRowB;
    static_assert(kLds <= 160 * 1024, "LDS of a CU");
    ANELM_REQUIRE(a.mp % BM == 0 && a.np % BN == 0 && a.mp >= a.m && a.np >= a.n && a.nk >= a.ksplit,
                  "prompt_gemm: rows %d of %d, %d of %d, %d stages in %d", a.m, a.mp, a.n, a.np, a.nk, a.ksplit);
    auto kern = prompt_gemm_kernel<BM, BN, WM, WN, NS>;
    static DeviceOnce lds;
    const int rc = allow_lds(lds, reinterpret_cast<const void*>(kern), kLds);
    if (rc) return rc;
    hipLaunchKernelGGL(kern, dim3((a.mp / BM) * (a.np / BN), a.ksplit), dim3(WM * WN * 64), kLds, st, a);
    ANELM_LAUNCHED("prompt_gemm_kernel");
    return ANELM_OK;
}

// Bounds of one preparation: 8192 inputs (176 MiB at the longest rows, 11264)
// and 256 MiB of decoded weights at a time, both far past where the chip is
// full, rounded up to whole tiles.  Partial sums of column slices come on top:
// slices are chosen only where the tiles are fewer than the compute units.
constexpr int kMaxRows = 8192;
constexpr size_t kMaxW16 = (size_t)256 << 20;

}  // namespace

// From 65 inputs on the one-time decode always wins (128 inputs, us: 18432 x
// 2560 72 -> 50, 2560 x 9216 75 -> 37, 2560 x 4096 80 -> 25, 7168 x 1024 117 ->
// 22); 33..64 inputs take two passes of the register-window kernel, which the
// one-time decode beats except for the largest matrices (64 inputs: 2560 x
// 9216 36 -> 31, 7168 x 1024 58 -> 23, but 12352 x 2560 37 -> 38 and 18432 x
// 2560 37 -> 47).  Streams under capture keep the register-window kernel: a
// captured launch would hold this path's workspace, which a later call may
// replace.  w needs dword loads, x 16-byte ones.
bool lut6_prompt_fits(const uint8_t* w, const float* x, int batch, int out_dim, int in_dim, hipStream_t st) {
    if (batch <= 32 || (batch <= 64 && (long)out_dim * in_dim > 24L << 20)) return false;
    if ((reinterpret_cast<uintptr_t>(w) & 3) || (reinterpret_cast<uintptr_t>(x) & 15)) return false;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return cs == hipStreamCaptureStatusNone;
}

// Y[b][r] (+)= W X[b], b < batch; out_dim % 32 == 0, in_dim % 16 == 0 (the
// caller checks).  ANELM_ENOMEM, with nothing launched, when the workspace
// cannot be had.
int lut6_prompt_gemm(float* y, const uint8_t* w, const uint16_t* lut, const float* x, int batch, int out_dim, int in_dim,
                     int accumulate, hipStream_t st) {
    Device* dev = device();
    if (!dev) return ANELM_EHIP;
    const int nk = (in_dim + kKB - 1) / kKB;
    const int n_max = (int)std::min<size_t>((size_t)out_dim, std::max<size_t>(256, kMaxW16 / ((size_t)nk * kRowB) / 256 * 256));
    // column slices write packed partial rows: only for whole output rows
    const bool whole = n_max == out_dim;
    auto plan = [&](int b0, int n0) {
        return make_plan(std::min(kMaxRows, batch - b0), std::min(n_max, out_dim - n0), nk, whole, dev->num_cus);
    };
    size_t bytes = 0;
    for (int b0 = 0; b0 < batch; b0 += kMaxRows)
        for (int n0 = 0; n0 < out_dim; n0 += n_max) bytes = std::max(bytes, plan(b0, n0).bytes);
    void* buf = nullptr;
    const int got = prompt_workspace(&buf, bytes, st);
    if (got) return got;
    char* ws = static_cast<char*>(buf);
    for (int b0 = 0; b0 < batch; b0 += kMaxRows)
        for (int n0 = 0; n0 < out_dim; n0 += n_max) {
            const Plan p = plan(b0, n0);
            float* yb = y + (size_t)b0 * out_dim + n0;
            float* parts = reinterpret_cast<float*>(ws + p.xb + p.wb);
            // W workgroups: about four per CU, each with as many column passes
            // as that leaves (the pair table is built per workgroup)
            const int steps = (in_dim + kDecCols - 1) / kDecCols, groups = p.n / 32;
            const int passes = std::max(1, std::min(steps, steps * groups / (4 * dev->num_cus)));
            PrepArgs pa{ws, ws + p.xb, x + (size_t)b0 * in_dim, w + (size_t)n0 * (in_dim * 3 / 4),
                        lut + (size_t)(n0 / 32) * 64, p.m, p.n, in_dim, p.mp, p.np, nk, groups,
                        (steps + passes - 1) / passes, passes};
            const unsigned blocks = (unsigned)(groups * pa.wy) + (unsigned)((p.m + 63) / 64) * (unsigned)nk;
            hipLaunchKernelGGL(prompt_prep_kernel, dim3(blocks), dim3(256), 0, st, pa);
            ANELM_LAUNCHED("prompt_prep_kernel");
            const bool sum = p.splits > 1;
            PromptArgs a{sum ? parts : yb, ws, ws + p.xb, p.m, p.n, p.mp, p.np, nk, p.splits, (long)p.m * p.n, out_dim,
                         sum ? 0 : accumulate};
            int rc;
            switch (p.tile) {
                case 0: rc = gemm_launch<256, 192, 4, 2>(a, st); break;
                case 1: rc = gemm_launch<256, 128, 4, 2>(a, st); break;
                case 2: rc = gemm_launch<128, 128, 2, 2>(a, st); break;
                default: rc = gemm_launch<64, 128, 1, 4>(a, st); break;
            }
            if (rc == ANELM_OK && sum) rc = lut6_split_sum(yb, parts, (long)p.m * p.n, p.splits, accumulate, st);
            if (rc) return rc;
        }
    return ANELM_OK;
}

}  // namespace anelm
