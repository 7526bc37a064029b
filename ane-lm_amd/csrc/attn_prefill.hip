// Causal GQA prefill attention on fp16 MFMA (v_mfma_f32_32x32x16_f16) with
// fp32 accumulation and an online softmax.
//
// Reference semantics: the reference has no batched prefill; generate.cpp:76-84
// runs the decode core once per prompt token, so output row t is
// gqa_attention (core/cpu_ops.cpp:148-204) over keys 0..t.
//
// Formulation: each wave owns 32 query rows of one head and computes the
// transposed score tile S^T = K Q^T (32 keys x 32 rows), so that in the MFMA
// accumulator layout every lane holds 16 scores of ONE query row.  The row's
// softmax statistics therefore need one cross-half exchange only, the output
// rescale is a per-lane scalar, and P^T is already in the B-operand layout of
// the second product O^T += V^T P^T (the contraction order over keys is
// permuted identically in both operands).  K and V tiles of 32 keys are
// staged in LDS once per workgroup and shared by all waves (the query heads of
// one KV head and several row blocks).
#include "anelm_internal.hpp"

#include <math.h>

#include <type_traits>

namespace anelm {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kBN = 32;  // keys per tile

// A ring of `cap` rows [Hkv][D] (k, v): key i of the sequence is row
// (start + i) mod cap.  A plain array of L keys is the ring (0, L).
struct KeyRing {
    const _Float16* k;
    const _Float16* v;
    int start, cap;
};

// Query row r is key qoff + r of the L keys in k / v (the keys before qoff
// are a cached prefix) and attends keys (qoff + r - win, qoff + r] (win 0: no
// lower bound).  With gate, the output row is multiplied by sigmoid of
// gate[r * gtok + h * ghead + d] (the reference's output gate).
template <int D, int HB, int RB, bool OUT16>
__global__ __launch_bounds__(HB * RB * 64) void prefill_kernel(void* out, const _Float16* q,
                                                               const KeyRing rg,
                                                               int S, int L, int qoff, int win, int Hq, int Hkv,
                                                               const float* gate, int gtok, int ghead) {
    constexpr int NW = HB * RB;
    constexpr int NT = NW * 64;
    constexpr int KS = D / 16;   // QK k-steps
    constexpr int DB = D / 32;   // PV dim blocks
    constexpr int KP = D + 8;    // K tile row pitch (halfs): 16-byte aligned rows, conflict-free reads
    constexpr int VP = kBN + 4;  // V^T row pitch (halfs)
    __shared__ __attribute__((aligned(16))) _Float16 Ks[kBN][KP];
    __shared__ __attribute__((aligned(16))) _Float16 Vt[D][VP];

    const int G = Hq / Hkv;
    const int qt = gridDim.x - 1 - blockIdx.x;  // longest causal ranges first
    const int h0 = blockIdx.y * HB;
    const int kvh = h0 / G;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int h = h0 + (w % HB);
    const int q0 = (qt * RB + w / HB) * 32;
    const int row_end = min(S, (qt + 1) * RB * 32);
    const int r = lane & 31, hh = lane >> 5;
    const int qrow = q0 + r;

    half8 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        if (qrow < S) qf[ks] = *reinterpret_cast<const half8*>(q + ((size_t)qrow * Hq + h) * D + 16 * ks + 8 * hh);
        else qf[ks] = half8{};
    }

    float16_t o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++) o[db] = float16_t{};
    float m = -INFINITY, l = 0.f;
    const float sl2 = (1.0f / sqrtf((float)D)) * 1.4426950408889634f;

    const int nkt = (qoff + row_end + kBN - 1) / kBN;
    // first tile any row of the workgroup sees
    const int kt0 = win > 0 ? max(0, qoff + qt * RB * 32 + 1 - win) / kBN : 0;
    for (int kt = kt0; kt < nkt; kt++) {
        const int j0 = kt * kBN;
        __syncthreads();
        for (int c = tid; c < kBN * D / 8; c += NT) {
            const int kr = c / (D / 8), kc = (c % (D / 8)) * 8;
            const int key = j0 + kr;
            uint4 kv4 = make_uint4(0, 0, 0, 0), vv4 = make_uint4(0, 0, 0, 0);
            if (key < L) {
                const int at = key + rg.start;
                const size_t row = at - (at >= rg.cap ? rg.cap : 0);
                kv4 = *reinterpret_cast<const uint4*>(rg.k + (row * Hkv + kvh) * D + kc);
                vv4 = *reinterpret_cast<const uint4*>(rg.v + (row * Hkv + kvh) * D + kc);
            }
            *reinterpret_cast<uint4*>(&Ks[kr][kc]) = kv4;
            const _Float16* vh = reinterpret_cast<const _Float16*>(&vv4);
#pragma unroll
            for (int i = 0; i < 8; i++) Vt[kc + i][kr] = vh[i];
        }
        __syncthreads();
        // wave-uniform: every key of the tile after the wave's rows, or (with
        // a window) before the window of its first row
        if (q0 >= S || j0 > qoff + q0 + 31 || (win > 0 && j0 + kBN <= qoff + q0 + 1 - win)) continue;

        float16_t s = float16_t{};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const half8 a = *reinterpret_cast<const half8*>(&Ks[r][16 * ks + 8 * hh]);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[ks], s, 0, 0, 0);
        }
        // s[e] = score of key j0 + 8*(e/4) + 4*hh + e%4 for query row qrow
        float mx = -INFINITY;
        const int kmax = qoff + qrow, kmin = win > 0 ? qoff + qrow - win : -1;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int key = j0 + 8 * (e / 4) + 4 * hh + (e % 4);
            const float val = (key <= kmax && key > kmin) ? s[e] * sl2 : -INFINITY;
            s[e] = val;
            mx = fmaxf(mx, val);
        }
        mx = fmaxf(mx, shfl_xor(mx, 32));
        // a row that has seen no key yet (below its window) keeps m = -inf:
        // its terms are exp2(-inf) = 0 against a finite reference
        const float m_new = fmaxf(m, mx);
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = exp2f(m - m_ref);
        float ps = 0.f;
        half8 pf[2];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const float pe = exp2f(s[e] - m_ref);
            ps += pe;
            pf[e / 8][e % 8] = (_Float16)pe;
        }
        l = l * alpha + ps;
        m = m_new;
#pragma unroll
        for (int db = 0; db < DB; db++) {
#pragma unroll
            for (int e = 0; e < 16; e++) o[db][e] *= alpha;
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const half4 lo = *reinterpret_cast<const half4*>(&Vt[32 * db + r][16 * kk + 4 * hh]);
                const half4 hi = *reinterpret_cast<const half4*>(&Vt[32 * db + r][16 * kk + 8 + 4 * hh]);
                const half8 a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pf[kk], o[db], 0, 0, 0);
            }
        }
    }
    if (q0 >= S) return;
    l += shfl_xor(l, 32);
    if (qrow >= S) return;
    const float inv = 1.0f / l;
    // o[db][e] = output dim 32*db + 8*(e/4) + 4*hh + e%4 of row qrow
#pragma unroll
    for (int db = 0; db < DB; db++) {
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
            const int d = 32 * db + 8 * g4 + 4 * hh;
            const size_t off = ((size_t)qrow * Hq + h) * D + d;
            float a0 = o[db][4 * g4] * inv, a1 = o[db][4 * g4 + 1] * inv;
            float a2 = o[db][4 * g4 + 2] * inv, a3 = o[db][4 * g4 + 3] * inv;
            if (gate) {
                const float* gr = gate + (size_t)qrow * gtok + (size_t)h * ghead + d;
                a0 = a0 / (1.0f + expf(-gr[0]));
                a1 = a1 / (1.0f + expf(-gr[1]));
                a2 = a2 / (1.0f + expf(-gr[2]));
                a3 = a3 / (1.0f + expf(-gr[3]));
            }
            if (OUT16) {
                half4 hv = {(_Float16)a0, (_Float16)a1, (_Float16)a2, (_Float16)a3};
                *reinterpret_cast<half4*>(static_cast<_Float16*>(out) + off) = hv;
            } else {
                *reinterpret_cast<float4*>(static_cast<float*>(out) + off) = make_float4(a0, a1, a2, a3);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Pipelined kernel for head_dim 256 and 4 query heads per KV head (the Qwen3.5
// shapes), any prompt length and cached history.
//
// * A wave's 32 columns are 8 tokens x the 4 query heads of the KV head; a
//   workgroup's 8 waves are 8 / KP column groups x KP key parts: a step stages
//   KP consecutive 32-key tiles and each wave takes the one of its part, so
//   the KP waves of a column group merge their (m, l, O) through LDS at the
//   end (each ends with 256 / KP of the dims).
// * A group of 64 / KP tokens whose steps exceed `sps` is cut into parts of
//   sps steps, one workgroup each; parts write (m, l, unnormalised O) records
//   and prefill_split_combine merges them.  The rule stands at plan_split.
// * K and V tiles (32 keys x 256) go straight to LDS with buffer loads (1 KiB
//   per wave instruction: rows c and c+16 of a tile share a chunk).  K chunks
//   are 1040 bytes (16 of padding) so the MFMA operand reads are conflict-free
//   with immediate offsets; V chunks are 1088 bytes, so the four key rows a
//   16-lane group reads with ds_read_b64_tr_b16 (4 keys x 16 dims, delivered
//   transposed: lane n gets dim n of the 4 keys) fall on distinct banks.  That
//   transposing read builds the V^T operand of O^T += V^T P^T from the V rows
//   as stored.  KP 1 and 2: four and two steps of tiles in LDS, the loads of
//   the step three and one ahead behind the one barrier of a step.  KP 4: one
//   step in LDS; the next step's K tiles are requested once the scores are
//   formed, its V tiles once the outputs are (four barriers per step).
// * Scores S^T = K Q^T (v_mfma_f32_32x32x16_f16).  The A-operand lane i reads
//   key row pi(i) (bits 2 and 3 of i swapped): lane (r, h) of the accumulator
//   then holds the scores of column r for keys 8h..8h+7 and 16+8h..16+8h+7,
//   exactly the B-operand keys of O^T += V^T P^T.
// * Softmax in the log2 domain; the running maximum only moves when it grows
//   by more than 8, so probabilities stay below 2^8 (fp16-exact range) and the
//   128-register output rescale is rare.
// Bound: the matrix units and LDS in turn (a step's 32 products per wave are
// 1 us of the CU's matrix time and its operand reads 1 us of its LDS; a step
// takes 1.9 us, 2.8 us with every CU under load).  Whole layer call, before
// (64-row blocks in causal pairs, two workgroups per pair, which left the chip
// to 2 Hkv ceil(S / 128) workgroups) and now: 4096 tokens 16q/4kv 230 -> 202
// us, 1000 tokens 86 -> 45, 777 tokens 8q/2kv behind 1500 keys 150 -> 42.5.
constexpr int kGKeys = 32;                       // keys per tile
constexpr int kGKBytes = 16 * 1040;              // K tile: chunk c = rows c, c + 16
constexpr int kGVChunk = 1088;                   // V tile chunk: rows c, c + 16 + 64 bytes of bank offset
constexpr int kGTile = kGKBytes + 16 * kGVChunk; // + V tile (32 x 256 fp16)
constexpr int kGNT = 512;
// Running maximum of a column that has seen no key yet: far below any score
// and finite, so a tile that is wholly masked for the column adds
// exp2(-inf - kNoKey) = 0 (from -inf it would add NaN).
constexpr float kNoKey = -1e30f;

__device__ __forceinline__ int key_perm(int i) { return (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1); }

// One 32-key tile (staged at `base`) against a wave's 32 query columns, in
// three parts.  S^T = K Q^T:
__device__ __forceinline__ float16_t tile_scores(const char* base, int ln, const half8 (&qf)[16]) {
    constexpr int KS = 16;
    float16_t sc = float16_t{};
    {
        const int krow = key_perm(ln & 31);
        const char* kb = base + (krow & 15) * 1040 + (krow >> 4) * 512 + (ln >> 5) * 16;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
            sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8*>(kb + 32 * ks), qf[ks], sc,
                                                        0, 0, 0);
        // K fragment ks + 1 is read while the product of fragment ks runs
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
        for (int ks = 0; ks < KS - 2; ks++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
    return sc;
}

// The online softmax: running maximum m, this lane half's sum l, O rescaled
// when the maximum moves; P^T in pf.  The tile's keys are j0 .. j0 + 31,
// element e of the scores being key j0 + (e < 8 ? 8 h + e : 16 + 8 h + e - 8);
// masked: some column stops before the last of them, qr being the last key of
// this lane's column.
__device__ __forceinline__ void tile_softmax(float16_t sc, half8 (&pf)[2], float16_t (&o)[8], float& m, float& l,
                                             float sl2, int ln, int j0, bool masked, int qr) {
    constexpr int DB = 8;
    if (masked) {
        const int h2 = ln >> 5;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int key = j0 + (e < 8 ? 8 * h2 + e : 16 + 8 * h2 + (e - 8));
            sc[e] = key <= qr ? sc[e] : -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; e++) mx = fmaxf(mx, sc[e]);
    mx = fmaxf(mx, shfl_xor(mx, 32)) * sl2;
    if (__builtin_amdgcn_ballot_w64(mx > m + 8.0f) != 0) {
        const float m_new = fmaxf(m, mx);
        const float alpha = __builtin_amdgcn_exp2f(m - m_new);
        l *= alpha;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[db][e] *= alpha;
        m = m_new;
    }
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const float pe = __builtin_amdgcn_exp2f(fmaf(sc[e], sl2, -m));
        l += pe;
        pf[e / 8][e % 8] = (_Float16)pe;
    }
}

// O^T += V^T P^T.  The A operand of lane (m, h2) for keys 16u + 8 h2 .. +8
// and dim 32 db + m comes from two transposing reads: 16-lane group i (m =
// 16 (i & 1) + n, h2 = i >> 1) has its lane n address key 16u + 8 (i >> 1) +
// 4r + n / 4, dims 32 db + 16 (i & 1) + 4 (n % 4) .. +4 of the V rows (key t
// at chunk t % 16, half t / 16).
__device__ __forceinline__ void tile_values(const char* base, int ln, const half8 (&pf)[2], float16_t (&o)[8]) {
    constexpr int DB = 8;
    {
        const int gi = ln >> 4, nn = ln & 15;
        const char* vbase = base + kGKBytes + (8 * (gi >> 1) + (nn >> 2)) * kGVChunk +
                            (16 * (gi & 1) + 4 * (nn & 3)) * 2;
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        static_assert(4 * kGVChunk == 4352, "offset of the second read");
        const uint32_t va = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const char*)vbase);
        // product k = 2 db + u; the reads of product k + 1 are issued
        // before product k (each asm statement waits only for the
        // older pair, which it passes through to the product)
        s16x4 lo[2], hi[2];
        asm volatile("ds_read_b64_tr_b16 %0, %2\n\tds_read_b64_tr_b16 %1, %2 offset:4352"
                     : "=&v"(lo[0]), "=&v"(hi[0])
                     : "v"(va)
                     : "memory");
#pragma unroll
        for (int kk = 0; kk < 2 * DB; kk++) {
            const int db = kk >> 1, u = kk & 1, c = kk & 1, n = c ^ 1;
            if (kk + 1 < 2 * DB) {
                const int u1 = (kk + 1) & 1, db1 = (kk + 1) >> 1;
                asm volatile(
                    "ds_read_b64_tr_b16 %0, %4\n\tds_read_b64_tr_b16 %1, %4 offset:4352\n\ts_waitcnt lgkmcnt(2)"
                    : "=&v"(lo[n]), "=&v"(hi[n]), "+v"(lo[c]), "+v"(hi[c])
                    : "v"(va + (uint32_t)(u1 * 512 + 64 * db1))
                    : "memory");
            } else {
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(lo[c]), "+v"(hi[c]) : : "memory");
            }
            const half8 av =
                __builtin_bit_cast(half8, __builtin_shufflevector(lo[c], hi[c], 0, 1, 2, 3, 4, 5, 6, 7));
            o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, pf[u], o[db], 0, 0, 0);
        }
    }
}

// Byte offset, in its ring, of 16-byte chunk `ch` of key `key` (kv head kvh);
// keys past the last one (L) are out of the buffers' range and read zeros.
__device__ __forceinline__ int ring_off(const KeyRing& rg, int L, int Hkv, int kvh, int key, int ch) {
    const int at = key + rg.start, row = at - (at >= rg.cap ? rg.cap : 0);
    return key < L ? ((row * Hkv + kvh) * 256 + 8 * ch) * 2 : 0x7fffffff;
}

// LDS: four tiles, then m and l of the 8 waves.
template <int KP>
constexpr int split_lds() { return 4 * kGTile + 2 * 8 * 64 * (int)sizeof(float); }

// Steps of KP tiles that group grp (64 / KP tokens) needs.
__host__ __device__ inline int split_steps(int KP, int grp, int S, int qoff) {
    const int tok = 64 / KP, end = (grp + 1) * tok < S ? (grp + 1) * tok : S;
    return (qoff + end + 32 * KP - 1) / (32 * KP);
}

// Four output values (dims d .. d + 3 of row (tok, h)), gated by g, and the
// gate logits of such a place (rows of any stride: dword aligned).
typedef float f4_dw __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f4_dw split_gate(const float* gate, int gtok, int ghead, int tok, int h, int d) {
    return *reinterpret_cast<const f4_dw*>(gate + (size_t)tok * gtok + (size_t)h * ghead + d);
}
template <bool OUT16, bool GATE>
__device__ __forceinline__ void split_store(void* out, int tok, int h, int Hq, int d, float4 x, f4_dw g) {
    if constexpr (GATE)
        x = make_float4(x.x / (1.0f + expf(-g[0])), x.y / (1.0f + expf(-g[1])), x.z / (1.0f + expf(-g[2])),
                        x.w / (1.0f + expf(-g[3])));
    const size_t off = ((size_t)tok * Hq + h) * 256 + d;
    if constexpr (OUT16)
        *reinterpret_cast<half4*>(static_cast<_Float16*>(out) + off) =
            half4{(_Float16)x.x, (_Float16)x.y, (_Float16)x.z, (_Float16)x.w};
    else
        *reinterpret_cast<float4*>(static_cast<float*>(out) + off) = x;
}

struct SplitArgs {
    void* out;
    const _Float16* q;
    KeyRing rg;
    float* rec;            // [Hkv][ngrp][parts] records
    const float* gate;
    int S, L, qoff, Hq, Hkv, gtok, ghead;
    int ngrp, parts, sps;  // groups per kv head, most parts of a group, steps per part
};

// Record of one part: O in accumulator order ([wave][8 / KP blocks of 32
// dims][4][64 lanes] float4), then m and l of [8 / KP column groups][32].
template <int KP>
constexpr int split_rec_floats() { return 8 * (8 / KP) * 4 * 256 + 2 * (8 / KP) * 32; }

template <int KP, bool OUT16, bool GATE>
__global__ __launch_bounds__(kGNT) void prefill_split_kernel(const SplitArgs a) {
    constexpr int KS = 16, DB = 8, CG = 8 / KP, QB = 8 / KP;   // column groups; dim blocks a wave ends with
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cg = w % CG, kp = w / CG;
    // workgroup -> (kv head, group, part): an XCD (workgroup id mod 8) serves
    // one kv head where 8 is a multiple of their number; last groups (the
    // longest) first
    const int bpk = a.ngrp * a.parts;
    int kvh, idx;
    if (8 % a.Hkv == 0) {
        const int spx = 8 / a.Hkv, xcd = blockIdx.x & 7;
        kvh = xcd / spx;
        idx = (int)(blockIdx.x >> 3) * spx + xcd % spx;
    } else {
        kvh = blockIdx.x % a.Hkv;
        idx = blockIdx.x / a.Hkv;
    }
    if (idx >= bpk) return;
    const int grp = a.ngrp - 1 - idx % a.ngrp, part = idx / a.ngrp;
    const int steps = split_steps(KP, grp, a.S, a.qoff);
    const int s0 = part * a.sps, s1 = min(steps, s0 + a.sps);
    if (s0 >= s1) return;
    const int tok0 = grp * (64 / KP) + 8 * cg;

    const __amdgpu_buffer_rsrc_t rk =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(a.rg.k), 0, a.rg.cap * a.Hkv * 512, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16*>(a.rg.v), 0, a.rg.cap * a.Hkv * 512, 0x00020000);
    constexpr int PERW = 16 / CG;   // chunks of its part's K (and V) tile that a wave loads
    char* const mine = lds + kp * kGTile;
    constexpr int NST = 4 / KP, kStage = KP * kGTile;   // step s in stage s % NST
    // the K or V part of step s's tiles, to the stage of step `to`
    auto issue = [&](int s, auto is_v, int to) __attribute__((always_inline)) {
        constexpr bool values = decltype(is_v)::value;
        char* base = mine + (to & (NST - 1)) * kStage + (values ? kGKBytes : 0);
        const int j0 = (s * KP + kp) * kGKeys, at = j0 + a.rg.start, row = at - (at >= a.rg.cap ? a.rg.cap : 0);
        int ln = threadIdx.x & 63;
        asm volatile("" : "+v"(ln));   // lane offsets are recomputed here, not held across the loop
        if (j0 + kGKeys <= a.L && row + kGKeys <= a.rg.cap) {
            // (wave-uniform) the whole tile is consecutive rows: one lane offset, the chunk's in a scalar
            const int voff = (ln >> 5) * 16 * a.Hkv * 512 + (ln & 31) * 16;
#pragma unroll
            for (int x = 0; x < PERW; x++) {
                const int c = PERW * cg + x;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    values ? rv : rk, (__attribute__((address_space(3))) void*)(base + c * (values ? kGVChunk : 1040)),
                    16, voff, ((row + c) * a.Hkv + kvh) * 512, 0, 0);
            }
            return;
        }
#pragma unroll
        for (int x = 0; x < PERW; x++) {
            const int c = PERW * cg + x, key = j0 + c + 16 * (ln >> 5);
            const int off = ring_off(a.rg, a.L, a.Hkv, kvh, key, ln & 31);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                values ? rv : rk, (__attribute__((address_space(3))) void*)(base + c * (values ? kGVChunk : 1040)), 16, off,
                0, 0, 0);
        }
    };
    constexpr std::integral_constant<bool, false> K{};
    constexpr std::integral_constant<bool, true> V{};
    // (KP 1: past the last step its tiles again, so that as many loads are in flight at every wait)
    auto request = [&](int s) __attribute__((always_inline)) {
        issue(KP == 1 ? min(s, s1 - 1) : s, K, s);
        issue(KP == 1 ? min(s, s1 - 1) : s, V, s);
    };
    request(s0);
    if constexpr (KP == 1) {
        request(s0 + 1);
        request(s0 + 2);
    }
    half8 qf[KS];
    {
        const int lane = threadIdx.x & 63, tok = min(tok0 + ((lane & 31) >> 2), a.S - 1);
        const _Float16* qr = a.q + ((size_t)tok * a.Hq + kvh * 4 + (lane & 3)) * 256 + 8 * (lane >> 5);
#pragma unroll
        for (int ks = 0; ks < KS; ks++) qf[ks] = *reinterpret_cast<const half8*>(qr + 16 * ks);
    }
    float16_t o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++) o[db] = float16_t{};
    float m = kNoKey, l = 0.f;
    const float sl2 = (1.0f / 16.0f) * 1.4426950408889634f;   // 1/sqrt(256) * log2(e)
    const int first = a.qoff + tok0, last = a.qoff + min(tok0 + 7, a.S - 1);   // last keys of the wave's tokens
    if constexpr (KP <= 2) {
        for (int s = s0; s < s1; s++) {
            // this wave's loads of step s have landed (KP 1: those of the next two may be in flight)
            __builtin_amdgcn_s_waitcnt(0x0F70 | (KP == 1 ? 4 * PERW : 0));
            lds_barrier();                      // every wave's; the stage of step s - 1 is free
            if (KP == 1 || s + 1 < s1) request(s + NST - 1);
            const int j0 = (s * KP + kp) * kGKeys;
            int ln = threadIdx.x & 63;
            asm volatile("" : "+v"(ln));
            // (wave-uniform) a tile past the wave's last token has nothing for it
            if (tok0 < a.S && j0 <= last) {
                const char* base = mine + (s & (NST - 1)) * kStage;
                half8 pf[2];
                tile_softmax(tile_scores(base, ln, qf), pf, o, m, l, sl2, ln, j0, j0 + 31 > first,
                             a.qoff + tok0 + ((ln & 31) >> 2));
                tile_values(base, ln, pf, o);
            }
        }
    } else {
        constexpr int kHalf = 0x0F70 | PERW;   // vmcnt(PERW): all but the newest PERW loads
        for (int s = s0; s < s1; s++) {
            const bool next = s + 1 < s1;
            const int j0 = (s * KP + kp) * kGKeys;
            const bool live = tok0 < a.S && j0 <= last;   // (wave-uniform)
            int ln = threadIdx.x & 63;
            asm volatile("" : "+v"(ln));
            __builtin_amdgcn_s_waitcnt(kHalf);   // K of step s (V of step s behind it)
            lds_barrier();
            float16_t sc = float16_t{};
            half8 pf[2] = {};
            if (live) sc = tile_scores(mine, ln, qf);
            lds_barrier();   // K is free
            if (next) issue(s + 1, K, s + 1);
            if (live)
                tile_softmax(sc, pf, o, m, l, sl2, ln, j0, j0 + 31 > first, a.qoff + tok0 + ((ln & 31) >> 2));
            if (next) __builtin_amdgcn_s_waitcnt(kHalf);   // V of step s (K of step s + 1 behind it)
            else __builtin_amdgcn_s_waitcnt(0x0F70);
            lds_barrier();
            if (live) tile_values(mine, ln, pf, o);
            lds_barrier();   // V is free
            if (next) issue(s + 1, V, s + 1);
        }
    }
    // ---- merge the KP key parts of each column group: every wave scales its O
    // to the group's maximum, then halves are exchanged until each wave holds
    // the sum over the parts of its own QB dim blocks
    l += shfl_xor(l, 32);
    int ln = threadIdx.x & 63;
    asm volatile("" : "+v"(ln));
    float* const ms = reinterpret_cast<float*>(lds + 4 * kGTile);
    if constexpr (KP == 1) __builtin_amdgcn_s_waitcnt(0x0F70);   // the repeated last tiles
    __syncthreads();   // the tiles are no longer read
    ms[w * 64 + ln] = m;
    ms[512 + w * 64 + ln] = l;
    __syncthreads();
    float M = kNoKey, lt = 0.f;
#pragma unroll
    for (int p = 0; p < KP; p++) M = fmaxf(M, ms[(p * CG + cg) * 64 + ln]);
#pragma unroll
    for (int p = 0; p < KP; p++)
        lt += ms[512 + (p * CG + cg) * 64 + ln] * __builtin_amdgcn_exp2f(ms[(p * CG + cg) * 64 + ln] - M);
    const float al = __builtin_amdgcn_exp2f(m - M);
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[db][e] *= al;
    float4* const xch = reinterpret_cast<float4*>(lds);
#pragma unroll
    for (int n = DB / 2, bit = KP / 2; bit >= 1; n /= 2, bit /= 2) {
        // partner: the wave of part kp ^ bit; this wave keeps blocks [0, n) of
        // its current 2n when its bit is clear, [n, 2n) otherwise
        const bool up = (kp & bit) != 0;
        const int mate = (kp ^ bit) * CG + cg;
#pragma unroll
        for (int db = 0; db < n; db++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                float4 snd;
                snd.x = up ? o[db][4 * g4] : o[n + db][4 * g4];
                snd.y = up ? o[db][4 * g4 + 1] : o[n + db][4 * g4 + 1];
                snd.z = up ? o[db][4 * g4 + 2] : o[n + db][4 * g4 + 2];
                snd.w = up ? o[db][4 * g4 + 3] : o[n + db][4 * g4 + 3];
                xch[((w * n + db) * 4 + g4) * 64 + ln] = snd;
            }
        __syncthreads();
#pragma unroll
        for (int db = 0; db < n; db++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                const float4 r = xch[((mate * n + db) * 4 + g4) * 64 + ln];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float rv4 = i == 0 ? r.x : i == 1 ? r.y : i == 2 ? r.z : r.w;
                    const float kept = up ? o[n + db][4 * g4 + i] : o[db][4 * g4 + i];
                    // the sum of two parts is the same whichever wave forms it
                    o[db][4 * g4 + i] = kept + rv4;
                }
            }
        __syncthreads();
    }
    // this wave holds dim blocks QB * b .. + QB - 1 with b = kp (its bits high to low)
    if (steps <= a.sps) {
        // Through the wave's own LDS (the exchange is over), so a store writes
        // 256 consecutive bytes of four rows, and the gate logits are read
        // that way, instead of 32 bytes of 32 rows; 64 dims at a time (4096
        // tokens of 16 heads, fp32 rows without a gate: 165 -> 161 us).
        constexpr int ROW = 64 + 4;   // (rows start 4 banks apart)
        float* const tr = reinterpret_cast<float*>(lds) + w * 32 * ROW;
        const float inv = 1.0f / lt;
        const int d = 4 * (ln & 15), h = kvh * 4 + (ln >> 4);
#pragma unroll
        for (int r = 0; r < QB / 2; r++) {
            const int d0 = 32 * (QB * kp + 2 * r) + d;
            f4_dw g[8];
            if constexpr (GATE) {
#pragma unroll
                for (int i = 0; i < 8; i++)
                    g[i] = split_gate(a.gate, a.gtok, a.ghead, min(tok0 + i, a.S - 1), h, d0);
            }
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int g4 = 0; g4 < 4; g4++) {
                    const float16_t& c = o[2 * r + j];
                    *reinterpret_cast<float4*>(tr + (ln & 31) * ROW + 32 * j + 8 * g4 + 4 * (ln >> 5)) =
                        make_float4(c[4 * g4] * inv, c[4 * g4 + 1] * inv, c[4 * g4 + 2] * inv, c[4 * g4 + 3] * inv);
                }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float4 x = *reinterpret_cast<const float4*>(tr + (4 * i + (ln >> 4)) * ROW + d);
                if (tok0 + i < a.S) split_store<OUT16, GATE>(a.out, tok0 + i, h, a.Hq, d0, x, g[i]);
            }
        }
        return;
    }
    float* rec = a.rec + ((size_t)(kvh * a.ngrp + grp) * a.parts + part) * split_rec_floats<KP>();
#pragma unroll
    for (int j = 0; j < QB; j++)
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++)
            reinterpret_cast<float4*>(rec)[((w * QB + j) * 4 + g4) * 64 + ln] =
                make_float4(o[j][4 * g4], o[j][4 * g4 + 1], o[j][4 * g4 + 2], o[j][4 * g4 + 3]);
    if (kp == 0 && ln < 32) {
        float* ml = rec + 8 * QB * 4 * 256;
        ml[cg * 32 + ln] = M;
        ml[CG * 32 + cg * 32 + ln] = lt;
    }
}

// Merge of a group's part records: workgroup (group of a kv head, float4 slot
// of the wave's 4 QB), thread = (wave, lane) of the kernel above; the parts'
// values are requested kCombineAhead at a time.
constexpr int kCombineAhead = 8;
template <int KP, bool OUT16, bool GATE>
__global__ __launch_bounds__(kGNT) void prefill_split_combine(const SplitArgs a) {
    constexpr int CG = 8 / KP, QB = 8 / KP, REC = split_rec_floats<KP>();
    const int w = threadIdx.x >> 6, ln = threadIdx.x & 63, cg = w % CG, kp = w / CG;
    const int kvh = blockIdx.x / a.ngrp, grp = blockIdx.x % a.ngrp, slot = blockIdx.y;
    const int steps = split_steps(KP, grp, a.S, a.qoff), np = (steps + a.sps - 1) / a.sps;
    const int tok = grp * (64 / KP) + 8 * cg + ((ln & 31) >> 2);
    if (np <= 1 || tok >= a.S) return;
    const float* base = a.rec + (size_t)(kvh * a.ngrp + grp) * a.parts * REC;
    const float* ml = base + 8 * QB * 4 * 256 + cg * 32 + (ln & 31);
    const float4* ov = reinterpret_cast<const float4*>(base) + (w * QB * 4 + slot) * 64 + ln;
    float M = kNoKey, lt = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int p0 = 0; p0 < np; p0 += kCombineAhead) {
        float4 x[kCombineAhead];
        float pm[kCombineAhead], pl[kCombineAhead];
#pragma unroll
        for (int i = 0; i < kCombineAhead; i++) {
            const int p = min(p0 + i, np - 1);
            x[i] = ov[(size_t)p * (REC / 4)];
            pm[i] = ml[(size_t)p * REC];
            pl[i] = p0 + i < np ? ml[(size_t)p * REC + CG * 32] : 0.f;
            if (p0 + i >= np) pm[i] = kNoKey;
        }
        float Mn = M;
#pragma unroll
        for (int i = 0; i < kCombineAhead; i++) Mn = fmaxf(Mn, pm[i]);
        const float sc = __builtin_amdgcn_exp2f(M - Mn);
        lt *= sc;
        acc = make_float4(acc.x * sc, acc.y * sc, acc.z * sc, acc.w * sc);
#pragma unroll
        for (int i = 0; i < kCombineAhead; i++) {
            // (a part without keys for this column: m = kNoKey, l = 0, O = 0)
            const float f = p0 + i < np ? __builtin_amdgcn_exp2f(pm[i] - Mn) : 0.f;
            lt += pl[i] * f;
            acc.x += x[i].x * f;
            acc.y += x[i].y * f;
            acc.z += x[i].z * f;
            acc.w += x[i].w * f;
        }
        M = Mn;
    }
    const float inv = 1.0f / lt;
    const int h = kvh * 4 + (ln & 3), d = 32 * (QB * kp + slot / 4) + 8 * (slot % 4) + 4 * (ln >> 5);
    f4_dw g = {};
    if constexpr (GATE) g = split_gate(a.gate, a.gtok, a.ghead, tok, h, d);
    split_store<OUT16, GATE>(a.out, tok, h, a.Hq, d, make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv), g);
}

// How a prompt is cut: the least estimated time over KP 2 and 4 and 1 .. 16 parts
// of the longest group.  From sweeps of both (us): a step takes 1.9 (KP 2) or
// 2.8 (KP 4, half the tokens over twice the keys), a workgroup 9 besides; more
// workgroups than compute units run one after another (the longest first, so
// half of one is the tail); parts cost a second launch of 4.5 and 0.35 per MB
// of records.  Measured against the model, layer prologue taken off: 777
// tokens behind 1500 keys 2 kv heads, KP 2: 5 parts 38 (38), 2 parts 49 (52);
// 4096 tokens 4 kv heads KP 2 184 (194), KP 4 233 (238); 1000 tokens KP 4 34
// (31), KP 2 43 (39); 2000 tokens KP 2 in 2 parts 77 (77).
//
// KP 1 brings half as many tile bytes to LDS per product as KP 2, but its
// groups are twice as long: it is the faster one where there are enough of
// them to even out, from 1.4 workgroups per compute unit on (whole layer, us,
// KP 1 and KP 2: 16384 tokens of 4 kv heads 2140 and 2306, 8192 603 and 646,
// 6144 (1.5 per unit) 396 and 412, 5000 (1.2) 312 and 299; 12000 of 2 kv heads
// (1.5) 689 and 687).
struct SplitPlan {
    int kp, ngrp, parts, sps;
};

SplitPlan plan_split(int S, int qoff, int Hkv, int cus) {
    const int n1 = (S + 63) / 64;
    if (5L * Hkv * n1 >= 7L * cus) return SplitPlan{1, n1, 1, split_steps(1, n1 - 1, S, qoff)};
    SplitPlan best{0, 0, 0, 0};
    float best_us = 0.f;
    for (int kp = 2; kp <= 4; kp += 2) {
        const int tok = 64 / kp, ngrp = (S + tok - 1) / tok, most = split_steps(kp, ngrp - 1, S, qoff);
        int last = 0;
        for (int p = 1; p <= 16; p++) {
            const int sps = (most + p - 1) / p;
            if (sps == last) continue;
            last = sps;
            const int parts = (most + sps - 1) / sps;
            if (parts > 1 && (long)Hkv * ngrp * parts > 2L * cus) break;   // (records: 64 MB on 256 CUs)
            long wgs = 0, steps = 0, recs = 0;
            for (int g = 0; g < ngrp; g++) {
                const int n = split_steps(kp, g, S, qoff), np = (n + sps - 1) / sps;
                steps += n;
                wgs += np;
                if (np > 1) recs += np;
            }
            const float load = wgs * Hkv <= cus ? (float)sps
                                                : (float)(steps * Hkv) / (float)cus + 0.5f * (float)sps;
            float us = 9.f + load * (kp == 2 ? 1.9f : 2.8f);
            if (parts > 1) us += 4.5f + 0.35f * (float)(recs * Hkv) * (kp == 2 ? 0.131f : 0.066f);
            if (best.kp == 0 || us < best_us) best = SplitPlan{kp, ngrp, parts, sps}, best_us = us;
        }
    }
    return best;
}

template <int KP>
int launch_split(const SplitArgs& a, bool out16, hipStream_t st) {
    using K = void (*)(const SplitArgs);
    static const K kern[2][2] = {{prefill_split_kernel<KP, false, false>, prefill_split_kernel<KP, false, true>},
                                 {prefill_split_kernel<KP, true, false>, prefill_split_kernel<KP, true, true>}};
    static DeviceOnce lds[2][2];
    const int o = out16 ? 1 : 0, g = a.gate != nullptr ? 1 : 0, bpk = a.ngrp * a.parts;
    const int rc = allow_lds(lds[o][g], reinterpret_cast<const void*>(kern[o][g]), split_lds<KP>());
    if (rc) return rc;
    const int spx = 8 % a.Hkv == 0 ? 8 / a.Hkv : 1;
    const dim3 grid(8 % a.Hkv == 0 ? (bpk + spx - 1) / spx * 8 : bpk * a.Hkv);
    hipLaunchKernelGGL(kern[o][g], grid, dim3(kGNT), split_lds<KP>(), st, a);
    ANELM_LAUNCHED("prefill_split_kernel");
    if constexpr (KP > 1) {   // (KP 1 is never cut)
        static const K comb[2][2] = {{prefill_split_combine<KP, false, false>, prefill_split_combine<KP, false, true>},
                                     {prefill_split_combine<KP, true, false>, prefill_split_combine<KP, true, true>}};
        if (a.parts > 1) {
            hipLaunchKernelGGL(comb[o][g], dim3(a.ngrp * a.Hkv, 4 * (8 / KP)), dim3(kGNT), 0, st, a);
            ANELM_LAUNCHED("prefill_split_combine");
        }
    }
    return ANELM_OK;
}

int launch_prefill_split(void* out, bool out16, const void* q, const KeyRing& rg, int S, int L, int qoff, int Hq,
                      int Hkv, const float* gate, int gtok, int ghead, hipStream_t st) {
    ANELM_REQUIRE((size_t)rg.cap * Hkv * 512 < 0x7fffffffu, "prefill: %d keys exceed the 2 GiB buffer range", rg.cap);
    Device* dev = device();
    if (!dev) return ANELM_EHIP;
    const SplitPlan sp = plan_split(S, qoff, Hkv, dev->num_cus);
    SplitArgs a{out, static_cast<const _Float16*>(q), rg, nullptr, gate, S, L, qoff, Hq, Hkv, gtok, ghead,
                sp.ngrp, sp.parts, sp.sps};
    if (sp.parts > 1) {
        const size_t rec = sp.kp == 2 ? split_rec_floats<2>() : split_rec_floats<4>();
        a.rec = static_cast<float*>(record_workspace((size_t)Hkv * sp.ngrp * sp.parts * rec * sizeof(float), st));
        if (!a.rec) return ANELM_ENOMEM;
    }
    switch (sp.kp) {
        case 1: return launch_split<1>(a, out16, st);
        case 2: return launch_split<2>(a, out16, st);
        default: return launch_split<4>(a, out16, st);
    }
}

template <int D, int HB, int RB>
int launch_prefill(void* out, bool out16, const void* q, const KeyRing& rg, int S, int L, int qoff,
                   int win, int Hq, int Hkv, const float* gate, int gtok, int ghead, hipStream_t st) {
    const int rows = 32 * RB;
    dim3 grid((S + rows - 1) / rows, Hq / HB), block(HB * RB * 64);
    const _Float16* qh = static_cast<const _Float16*>(q);
    if (out16)
        hipLaunchKernelGGL((prefill_kernel<D, HB, RB, true>), grid, block, 0, st, out, qh, rg, S, L, qoff, win,
                           Hq, Hkv, gate, gtok, ghead);
    else
        hipLaunchKernelGGL((prefill_kernel<D, HB, RB, false>), grid, block, 0, st, out, qh, rg, S, L, qoff, win,
                           Hq, Hkv, gate, gtok, ghead);
    ANELM_LAUNCHED("prefill_kernel");
    return ANELM_OK;
}

template <int D>
int dispatch_g(void* out, bool out16, const void* q, const KeyRing& rg, int S, int L, int qoff, int win,
               int Hq, int Hkv, const float* gate, int gtok, int ghead, hipStream_t st) {
    switch (Hq / Hkv) {
        case 1: return launch_prefill<D, 1, 8>(out, out16, q, rg, S, L, qoff, win, Hq, Hkv, gate, gtok, ghead, st);
        case 2: return launch_prefill<D, 2, 4>(out, out16, q, rg, S, L, qoff, win, Hq, Hkv, gate, gtok, ghead, st);
        case 4:
            // the pipelined kernel walks every key from 0: no window
            if (D == 256 && win == 0)
                return launch_prefill_split(out, out16, q, rg, S, L, qoff, Hq, Hkv, gate, gtok, ghead, st);
            return launch_prefill<D, 4, 2>(out, out16, q, rg, S, L, qoff, win, Hq, Hkv, gate, gtok, ghead, st);
        case 8: return launch_prefill<D, 4, 2>(out, out16, q, rg, S, L, qoff, win, Hq, Hkv, gate, gtok, ghead, st);
        default: return set_error(ANELM_EINVAL, "prefill: n_heads/n_kv_heads = %d unsupported", Hq / Hkv);
    }
}

}  // namespace

int prefill_core(void* out, bool out16, const uint16_t* q, const uint16_t* k, const uint16_t* v, int start, int cap,
                 int S, int L, int qoff, int win, int Hq, int Hkv, int D, const float* gate, int gtok, int ghead,
                 hipStream_t st) {
    ANELM_REQUIRE(L <= cap && start >= 0 && start < cap, "prefill: %d keys in a ring of %d from %d", L, cap, start);
    const KeyRing rg{reinterpret_cast<const _Float16*>(k), reinterpret_cast<const _Float16*>(v), start, cap};
    switch (D) {
        case 128: return dispatch_g<128>(out, out16, q, rg, S, L, qoff, win, Hq, Hkv, gate, gtok, ghead, st);
        case 256: return dispatch_g<256>(out, out16, q, rg, S, L, qoff, win, Hq, Hkv, gate, gtok, ghead, st);
        default: return set_error(ANELM_EINVAL, "prefill: head_dim %d unsupported (128, 256)", D);
    }
}

}  // namespace anelm

using namespace anelm;

extern "C" int anelm_attn_prefill(void* out, int out_dtype, const uint16_t* q, const uint16_t* k,
                                  const uint16_t* v, int S, int n_heads, int n_kv_heads,
                                  int head_dim, void* stream) {
    ANELM_NONNULL(out);
    ANELM_NONNULL(q);
    ANELM_NONNULL(k);
    ANELM_NONNULL(v);
    ANELM_REQUIRE(S > 0, "prefill: S %d", S);
    ANELM_REQUIRE(n_kv_heads > 0 && n_heads % n_kv_heads == 0, "prefill: heads %d/%d", n_heads,
                  n_kv_heads);
    ANELM_REQUIRE(out_dtype == ANELM_F32 || out_dtype == ANELM_F16, "prefill: out_dtype %d", out_dtype);
    return prefill_core(out, out_dtype == ANELM_F16, q, k, v, 0, S, S, S, 0, 0, n_heads, n_kv_heads, head_dim, nullptr, 0,
                        0, as_stream(stream));
}
