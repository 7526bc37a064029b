// Gated DeltaNet: decode step for all value heads and sequence prefill
// (dk = dv = 128).
//
// Reference: models/llm/qwen3_5.cpp:879-908 calling ssm_step
// (core/cpu_ops.cpp:131-146).  The reference reads each 64 KiB head state five
// times and writes it twice across four BLAS calls; here a workgroup holds a
// slab of state columns in registers and reads and writes it exactly once:
//   Sk[j] = sum_i S[i][j] k[i];  delta[j] = v[j] - Sk[j]
//   S'[i][j] = decay S[i][j] + beta k[i] delta[j];  y[j] = sum_i S'[i][j] q[i]
// Column j depends only on column j, so slabs of a head are independent.  The
// gated RMSNorm epilogue needs a whole head's y, so that variant gives one
// workgroup the whole head instead of combining slabs across workgroups.
#include "anelm_internal.hpp"

#include <math.h>


namespace anelm {
namespace {

constexpr int kDK = 128;
constexpr int kDV = 128;

struct DnParams {
    float* y;
    float* state;
    const float* q;
    const float* k;
    const float* v;
    const float* a;
    const float* b;
    const float* A;
    const float* dt_bias;
    const float* z;
    const float* norm_w;
    int Hk, Hv, flags;
    int w_heads;   // A / dt_bias hold w_heads entries: head h uses entry h % w_heads
    // conv prologue (qwen3_5.cpp:867-874): q, k, v are channels of the raw
    // mixed projection `mix`, passed through the conv ring and SiLU here
    const float* mix;       // [2*Hk*dk + Hv*dv]
    float* conv_state;      // [2*Hk*dk + Hv*dv][conv_k - 1]
    const float* conv_w;    // [2*Hk*dk + Hv*dv][conv_k]
    int conv_pos, conv_k;
    uint32_t* readers_done; // [Hk] zeroed counters: workgroups done reading a key head's ring
    int readers;            // workgroups that read one key head's q/k channels
};

// conv1d_update for one channel (core/cpu_ops.cpp:89-129): the K-1 ring
// entries oldest first from `pos`, then the new input; followed by SiLU
// (silu_vec_inplace, cpu_ops.cpp:6-13: x / (1 + exp(-x))).  The ring write
// of the new input is left to the caller (it may be shared by workgroups).
__device__ __forceinline__ float conv_silu(const DnParams& p, int c, float xc) {
    const int sl = p.conv_k - 1;
    const float* st = p.conv_state + (size_t)c * sl;
    const float* w = p.conv_w + (size_t)c * p.conv_k;
    float sum = 0.f;
    int idx = p.conv_pos;
    for (int j = 0; j < sl; j++) {
        sum += st[idx] * w[j];
        idx = idx + 1 == sl ? 0 : idx + 1;
    }
    const float y = sum + xc * w[sl];
    return y / (expf(-y) + 1.0f);
}

// CB state columns per workgroup of NT threads: thread t owns column
// t % CB for rows [(t / CB) * RPT, +RPT).
// CONV: the inputs come from the raw projection through conv_silu; each
// value channel is read by exactly one workgroup, which also writes its ring
// slot; a key head's q/k channels are read by `readers` workgroups, and the
// last of them to finish reading (counter) writes their ring slots.
template <int CB, int NT, bool GATED, bool CONV = false>
__global__ __launch_bounds__(NT) void deltanet_decode_kernel(const DnParams p) {
    constexpr int RC = NT / CB;       // row chunks
    constexpr int RPT = kDK / RC;     // rows per thread
    static_assert(!GATED || CB == kDV, "the gated epilogue needs the whole head");
    __shared__ float qs[kDK], ks[kDK];
    __shared__ float red_a[RC][CB];
    __shared__ float red[NT / 64];
    __shared__ float vs[CB];
    __shared__ int last_reader;

    const int h = blockIdx.y;
    const int tid = threadIdx.x;
    const int c = tid % CB, rc = tid / CB;
    const int j = blockIdx.x * CB + c;
    const int kh = h / (p.Hv / p.Hk);

    // The state slab is requested first; the prologue below overlaps it.
    float* S = p.state + (size_t)h * kDK * kDV;
    float s[RPT];
#pragma unroll
    for (int r = 0; r < RPT; r++) s[r] = S[(size_t)(rc * RPT + r) * kDV + j];

    // q, k of the key head: optional l2 normalisation (cpu_ops.cpp:82-87) and
    // the 1/sqrt(dk) query scale (qwen3_5.cpp:879-887).
    float qv = 0.f, kv = 0.f, qx = 0.f, kx = 0.f;
    if constexpr (CONV) {
        // channels: Q [Hk][dk] | K [Hk][dk] | V [Hv][dv] (qwen3_5.cpp:872-874)
        const int cq = kh * kDK + tid, ck = p.Hk * kDK + kh * kDK + tid;
        if (tid < kDK) {
            qx = p.mix[cq];
            kx = p.mix[ck];
            qv = conv_silu(p, cq, qx);
            kv = conv_silu(p, ck, kx);
        }
        if (tid < CB) {
            const int cv = 2 * p.Hk * kDK + h * kDV + j;
            const float vx = p.mix[cv];
            vs[tid] = conv_silu(p, cv, vx);
            p.conv_state[(size_t)cv * (p.conv_k - 1) + p.conv_pos] = vx;   // this workgroup is its only reader
        }
        // the key head's q/k ring slots take their new inputs at the end of
        // the kernel, off the path of the recurrence
    } else if (tid < kDK) {
        qv = p.q[(size_t)kh * kDK + tid];
        kv = p.k[(size_t)kh * kDK + tid];
    }
    if (p.flags & ANELM_DN_L2NORM) {
        const float sq = block_sum<NT>(qv * qv, red);
        const float sk = block_sum<NT>(kv * kv, red);
        qv = qv * (1.0f / sqrtf(sq + 1e-12f));
        kv = kv * (1.0f / sqrtf(sk + 1e-12f));
    }
    qv = qv * (1.0f / sqrtf((float)kDK));
    if (tid < kDK) { qs[tid] = qv; ks[tid] = kv; }

    // Gates (qwen3_5.cpp:896-898; cpu_ops.h:13-14).
    const float beta = 1.0f / (1.0f + expf(-p.b[h]));
    const int hw = h % p.w_heads;
    const float sp = logf(1.0f + expf(p.a[h] + p.dt_bias[hw]));
    const float decay = expf(-p.A[hw] * sp);
    const bool tf = (p.flags & ANELM_DN_ORDER_TRANSFORMERS) != 0;
    float vj = 0.f;
    if constexpr (!CONV) vj = p.v[(size_t)h * kDV + j];
    __syncthreads();
    if constexpr (CONV) vj = vs[c];

    float part = 0.f;
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        if (tf) s[r] = decay * s[r];
        part = fmaf(s[r], ks[rc * RPT + r], part);
    }
    red_a[rc][c] = part;
    __syncthreads();
    float sk = 0.f;
#pragma unroll
    for (int i = 0; i < RC; i++) sk += red_a[i][c];
    const float delta = tf ? (vj - sk) * beta : vj - sk;
    __syncthreads();

    float yp = 0.f;
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        const int i = rc * RPT + r;
        const float n = tf ? fmaf(ks[i], delta, s[r]) : fmaf(beta * ks[i], delta, decay * s[r]);
        S[(size_t)i * kDV + j] = n;
        yp = fmaf(n, qs[i], yp);
    }
    red_a[rc][c] = yp;
    __syncthreads();
    float yj = 0.f;
#pragma unroll
    for (int i = 0; i < RC; i++) yj += red_a[i][c];

    if constexpr (!GATED) {
        if (rc == 0) p.y[(size_t)h * kDV + j] = yj;
    } else {
        // rmsnorm_gated (cpu_ops.cpp:32-38): rmsnorm(y, w, 1e-6) * sigmoid(z) * z
        const float ss = block_sum<NT>(rc == 0 ? yj * yj : 0.f, red);
        const float inv = 1.0f / sqrtf(ss / (float)kDV + 1e-6f);
        if (rc == 0) {
            const float zi = p.z[(size_t)h * kDV + j];
            float o = (yj * inv) * p.norm_w[j];
            o = o / (1.0f + expf(-zi));
            p.y[(size_t)h * kDV + j] = o * zi;
        }
    }
    if constexpr (CONV) {
        // Every ring read of this workgroup returned long ago (the values fed
        // the recurrence): count the workgroup as done with its key head; the
        // last of the head's readers stores the new q/k inputs into the ring
        // and re-zeroes the counter.  No data of this workgroup is published
        // through the counter, so it is relaxed.
        __syncthreads();
        if (tid == 0) {
            const uint32_t n = __hip_atomic_fetch_add(p.readers_done + kh, 1u, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
            last_reader = n == (uint32_t)p.readers - 1u;
            if (last_reader) __hip_atomic_store(p.readers_done + kh, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (last_reader && tid < kDK) {
            const int sl = p.conv_k - 1;
            p.conv_state[(size_t)(kh * kDK + tid) * sl + p.conv_pos] = qx;
            p.conv_state[(size_t)(p.Hk * kDK + kh * kDK + tid) * sl + p.conv_pos] = kx;
        }
    }
}

// ---------------------------------------------------------------- prefill
// Pre-pass: per (token, key head) l2-normalise q and k and scale q
// (qwen3_5.cpp:879-887); per (token, value head) beta and decay
// (qwen3_5.cpp:896-898).
// One wave per (token, key head) row, four rows per workgroup; each lane
// holds two adjacent elements and the norms reduce within the wave.
constexpr int kPrepRows = 4;
__global__ __launch_bounds__(64 * kPrepRows) void dn_prep_kernel(float* qn, float* kn, float* beta, float* decay,
                                                                 float* ldecay, const float* q, const float* k,
                                                                 const float* a, const float* b, const float* A,
                                                                 const float* dt_bias, int S, int Hk, int Hv,
                                                                 int flags) {
    const int row = blockIdx.x * kPrepRows + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= S * Hk) return;   // (no barrier in this kernel)
    const int t = row / Hk, kh = row % Hk;
    const size_t off = (size_t)row * kDK + 2 * lane;
    float2 qv = *reinterpret_cast<const float2*>(q + off), kv = *reinterpret_cast<const float2*>(k + off);
    if (flags & ANELM_DN_L2NORM) {
        float sq = qv.x * qv.x + qv.y * qv.y, sk = kv.x * kv.x + kv.y * kv.y;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            sq += __shfl_xor(sq, m, 64);
            sk += __shfl_xor(sk, m, 64);
        }
        const float iq = 1.0f / sqrtf(sq + 1e-12f), ik = 1.0f / sqrtf(sk + 1e-12f);
        qv = make_float2(qv.x * iq, qv.y * iq);
        kv = make_float2(kv.x * ik, kv.y * ik);
    }
    const float qs = 1.0f / sqrtf((float)kDK);
    *reinterpret_cast<float2*>(qn + off) = make_float2(qv.x * qs, qv.y * qs);
    *reinterpret_cast<float2*>(kn + off) = kv;
    const int group = Hv / Hk;
    for (int gi = lane; gi < group; gi += 64) {
        const int h = kh * group + gi;
        const size_t g = (size_t)t * Hv + h;
        beta[g] = 1.0f / (1.0f + expf(-b[g]));
        const float sp = logf(1.0f + expf(a[g] + dt_bias[h]));
        decay[g] = expf(-A[h] * sp);
        if (ldecay) ldecay[g] = -A[h] * sp;   // log of the decay, for the chunked form
    }
}

constexpr int kScanCB = 32;                 // columns per scan workgroup
constexpr int kScanNT = 256;
constexpr int kScanRC = kScanNT / kScanCB;  // 8 row chunks
constexpr int kScanRPT = kDK / kScanRC;     // 16 rows per thread

// Sequential scan over tokens: a workgroup owns a 32-column slab of one
// head's state in registers for the whole sequence (one HBM read and write of
// the state per call); per token it reads q, k, v and the gates and writes y.
__global__ __launch_bounds__(kScanNT) void dn_scan_kernel(float* y, float* state, const float* qn,
                                                          const float* kn, const float* v,
                                                          const float* beta, const float* decay,
                                                          int S, int Hk, int Hv, int flags) {
    __shared__ float red_a[2][kScanRC][kScanCB];
    const int h = blockIdx.y, slab = blockIdx.x, tid = threadIdx.x;
    const int c = tid % kScanCB, rc = tid / kScanCB;
    const int j = slab * kScanCB + c;
    const int kh = h / (Hv / Hk);
    const bool tf = (flags & ANELM_DN_ORDER_TRANSFORMERS) != 0;
    float* Sp = state + (size_t)h * kDK * kDV;
    float s[kScanRPT];
#pragma unroll
    for (int r = 0; r < kScanRPT; r++) s[r] = Sp[(size_t)(rc * kScanRPT + r) * kDV + j];
    for (int t = 0; t < S; t++) {
        const float* kt = kn + ((size_t)t * Hk + kh) * kDK + rc * kScanRPT;
        const float* qt = qn + ((size_t)t * Hk + kh) * kDK + rc * kScanRPT;
        float kr[kScanRPT], qr[kScanRPT];
#pragma unroll
        for (int r = 0; r < kScanRPT; r += 4) {
            const float4 k4 = *reinterpret_cast<const float4*>(kt + r);
            const float4 q4 = *reinterpret_cast<const float4*>(qt + r);
            kr[r] = k4.x; kr[r + 1] = k4.y; kr[r + 2] = k4.z; kr[r + 3] = k4.w;
            qr[r] = q4.x; qr[r + 1] = q4.y; qr[r + 2] = q4.z; qr[r + 3] = q4.w;
        }
        const float bt = beta[(size_t)t * Hv + h], dc = decay[(size_t)t * Hv + h];
        const float vj = v[((size_t)t * Hv + h) * kDV + j];
        const int buf = t & 1;
        float part = 0.f;
#pragma unroll
        for (int r = 0; r < kScanRPT; r++) {
            if (tf) s[r] = dc * s[r];
            part = fmaf(s[r], kr[r], part);
        }
        red_a[buf][rc][c] = part;
        __syncthreads();
        float sk = 0.f;
#pragma unroll
        for (int i = 0; i < kScanRC; i++) sk += red_a[buf][i][c];
        const float delta = tf ? (vj - sk) * bt : vj - sk;
        float yp = 0.f;
#pragma unroll
        for (int r = 0; r < kScanRPT; r++) {
            s[r] = tf ? fmaf(kr[r], delta, s[r]) : fmaf(bt * kr[r], delta, dc * s[r]);
            yp = fmaf(s[r], qr[r], yp);
        }
        __syncthreads();
        red_a[buf][rc][c] = yp;
        __syncthreads();
        if (rc == 0) {
            float yj = 0.f;
#pragma unroll
            for (int i = 0; i < kScanRC; i++) yj += red_a[buf][i][c];
            y[((size_t)t * Hv + h) * kDV + j] = yj;
        }
    }
#pragma unroll
    for (int r = 0; r < kScanRPT; r++) Sp[(size_t)(rc * kScanRPT + r) * kDV + j] = s[r];
}

// ------------------------------------------------------- chunked prefill
// The recurrence over a chunk of C = 64 tokens in closed form (per value head,
// chunk start state S0, lg_t = sum_{j<=t} log g_j inside the chunk):
//   cpu_ops order (core/cpu_ops.cpp:131-146): u_t = beta_t (v_t - S_{t-1}^T k_t)
//     S_t = exp(lg_t) S0 + sum_{i<=t} exp(lg_t - lg_i) k_i u_i^T
//     u_t = beta_t (v_t - exp(lg_{t-1}) S0^T k_t) - sum_{i<t} A_ti u_i,
//     A_ti = beta_t exp(lg_{t-1} - lg_i) (k_t . k_i)
//   decay-first order: the same with lg_{t-1} replaced by lg_t in A and u.
// With T = (I + A)^-1 (unit lower triangular):
//   Ut = T diag(beta) V,  Wm = T diag(beta exp(lg_{t-1 or t})) K,  U = Ut - Wm S0
//   y  = Op + Qh S0,      Op = P Ut,  Qh = diag(exp(lg)) Q - P Wm,
//                         P_ti = exp(lg_t - lg_i) (q_t . k_i), i <= t
//   S_end = gC S0 + Kh^T U,  Kh = diag(exp(lg_L - lg)) K,  gC = exp(lg_L)
// Everything but the products with S0 and U is independent of the state and is
// computed for all chunks at once (dn_chunk_prep_kernel); dn_chunk_scan_kernel
// then carries the state through the chunks.  The scan forms
//   U = Ut - Wm S0,  y = diag(exp(lg)) (Q S0) + P U,
//   S_end = gC S0 + K^T (diag(exp(lg_L - lg)) U),
// so a value head's record holds Ut, Wm, P and the decay factors only, and the
// normalised Q and K rows are stored once per key head (Op, Qh and Kh per value
// head were 160 KB a chunk and half of the preparation's products; now 76 KB
// and 64 KB shared by the key head's value heads).  Decay ratios are formed in
// log space (all exponents <= 0).  Rows past the sequence end are zero (beta
// 0, log decay 0), so they change nothing.
//
// The chunk matrices are stored as the scan's operand fragments: 16x16 tiles
// of 64 lanes x 4 floats, so each of its loads is 1 KiB of consecutive memory
// (row-major records made every load 16 pieces of 64 bytes: the address units
// were busy all through the scan, 270 us for 4096 tokens of 32 heads, 193 with
// the same bytes consecutive).
//   "D" fragment: lane n + 16 k holds rows 4 k + (0..3) of column n, the
//       layout of a product's result;
//   "A" fragment: lane m + 16 k holds columns 4 k + (0..3) of row m, the left
//       operand of four products v_mfma_f32_16x16x4_f32 (the contraction index
//       of product e is 4 k + e in both operands; a D fragment is the right
//       operand of the same).
constexpr int kChunk = 64;
constexpr int kCMat = kChunk * kDK;             // floats per chunk matrix
// record of a (chunk, value head): Ut D[4][8], Wm A[4][8] (row tile, column
// tile), P A[10] (tile (r, x <= r) at r (r + 1) / 2 + x), exp(lg_t) [64],
// exp(lg_L - lg_t) [64], gC
constexpr int kVW = kCMat, kVP = 2 * kCMat, kVE = kVP + 10 * 256, kVRec = kVE + 192;
// record of a (chunk, key head): Q A[4][8], K^T A[8][4] (state row tile, chunk row tile)
constexpr int kKT = kCMat, kKRec = 2 * kCMat;

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// 4x4 transpose within each quad of lanes: lane i's element j <-> lane j's
// element i.
__device__ __forceinline__ v4f quad_transpose(v4f x, int lane) {
    const bool b0 = lane & 1, b1 = lane & 2;
    // exchange with lane ^ 1: (0,1) and (2,3)
    const float s0 = partner<1>(b0 ? x[0] : x[1]), s1 = partner<1>(b0 ? x[2] : x[3]);
    x = v4f{b0 ? s0 : x[0], b0 ? x[1] : s0, b0 ? s1 : x[2], b0 ? x[3] : s1};
    // exchange with lane ^ 2: (0,2) and (1,3)
    const float t0 = partner<2>(b1 ? x[0] : x[2]), t1 = partner<2>(b1 ? x[1] : x[3]);
    return v4f{b1 ? t0 : x[0], b1 ? t1 : x[1], b1 ? x[2] : t0, b1 ? x[3] : t1};
}

// Inputs of the preparation.  CONV: q, k, v are channels of the raw projection
// rows `proj` [S][pd] (mixed qkv | z | a | b) passed through the causal conv1d
// of width 4 over [conv ring | prompt] and SiLU here (cpu_ops.cpp:89-129,
// :6-13); rows and weights 16-byte aligned.
struct ChunkArgs {
    float* vrec;               // [chunks][Hv][kVRec]
    float* krec;               // [chunks][Hk][kKRec]
    const float* q;            // [S][Hk][dk]
    const float* k;
    const float* v;            // [S][Hv][dv]
    const float* a;            // token t, head h at a[t * as + h]
    const float* b;
    const float* A;
    const float* dt_bias;
    const float* proj;
    const float* conv_state;   // [C][3], oldest at slot conv_pos
    const float* conv_w;       // [C][4]
    long as, pd;
    int conv_pos, S, Hk, Hv, flags;
    int per_wg;                // value heads per workgroup (Hv / Hk, or 1)
};

// Input of token tt < 0 of channel c: the ring holds inputs -3 .. -1 oldest
// first from slot conv_pos.
__device__ __forceinline__ float ring_input(const ChunkArgs& p, int c, int tt) {
    int idx = p.conv_pos + tt + 3;
    if (idx >= 3) idx -= 3;
    return p.conv_state[(size_t)c * 3 + idx];
}

// The conv over four consecutive inputs, the oldest three first, then SiLU.
__device__ __forceinline__ float conv_tap4(float x0, float x1, float x2, float x3, float4 w) {
    float sum = 0.0f;
    sum += x0 * w.x;
    sum += x1 * w.y;
    sum += x2 * w.z;
    const float y = sum + x3 * w.w;
    return y / (expf(-y) + 1.0f);
}

// ------------------------------------------- chunk preparation on fp32 MFMA
// The per-chunk matrices above, on v_mfma_f32_16x16x4_f32, from the raw
// inputs: conv and SiLU (CONV), l2 norm and q scale, beta, log decay are
// formed here, so the inputs are read once and nothing is staged through
// memory.  One workgroup (8 waves) per (chunk, key head, per_wg value heads);
// the value heads of a workgroup share its key and query rows: the Gram tiles
// K K^T and Q K^T (the 10 lower 16x16 tiles of each) are computed once and
// kept in registers, transposed (K as the left operand), so four consecutive
// columns of a row are a lane's four elements.
// Per value head:
//   Am = -A (strictly lower, row-major) goes to LDS, P to the record;
//   wave 0 turns the diagonal 16x16 blocks of Am into T_rr = (I + A_rr)^-1
//   by substitution, in place;
//   for B = [beta V | beta exp(lgT) K] (64 x 256) the blocked forward
//   substitution runs per 16-column tile of B (wave w owns V tile w and K tile
//   w; it forms them straight in the accumulator layout, V columns from memory,
//   K columns from LDS):
//     X_r = T_rr (B_r + sum_{s<r} Am_rs X_s),  X = [Ut | Wm]
//   X tiles stay in registers: a result tile is the right operand of the next
//   product.  Ut tiles are stored as they are, Wm tiles transposed in quads.
// LDS matrices are row-major with 16-byte chunks XOR-swizzled by (row & 15);
// 66 KB, so two workgroups share a CU (one's serial phases overlap the other).
// Bound: memory (134 MB read, 224 MB of records written for 4096 tokens of 32
// heads: 65 us at 5.5 TB/s) and the vector units (conv and SiLU): 114 us, where
// conv pass and preparation took 77 + 140 (86 us without the conv).
constexpr int kPmNT = 512;
constexpr int kPmK = 0;                        // K rows [64][128]
constexpr int kPmR = kCMat;                    // Q rows [64][128] for the Gram tiles, then:
constexpr int kPmA = kPmR;                     //   Am [64][64] (T_rr on its diagonal blocks)
constexpr int kPmLg = kPmR + kCMat;            // lg[65] (+3 pad)
constexpr int kPmBt = kPmLg + 68;              // beta[64]
constexpr int kPmEb = kPmBt + kChunk;          // exp(lg[t + 1]) (decay-first) or exp(lg[t]): scales K in B
constexpr int kPmLds = (kPmEb + kChunk) * 4;

__device__ __forceinline__ int sw128(int t, int d) { return t * kDK + 4 * ((d >> 2) ^ (t & 15)) + (d & 3); }
__device__ __forceinline__ int sw64(int r, int c) { return r * kChunk + 4 * ((c >> 2) ^ (r & 15)) + (c & 3); }

template <bool TF, bool CONV>
__global__ __launch_bounds__(kPmNT, 2) void dn_chunk_prep_kernel(const ChunkArgs p) {
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* Ks = sm + kPmK;
    float* Rs = sm + kPmR;
    float* Am = sm + kPmA;
    float* lg = sm + kPmLg;
    float* bt = sm + kPmBt;
    float* eb = sm + kPmEb;
    const int S = p.S, Hk = p.Hk, Hv = p.Hv;
    const int c = blockIdx.x, kh = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 15, lk = lane >> 4;
    const int t0 = c * kChunk, L = min(kChunk, S - t0);
    // ---- key and query rows of the chunk, l2-normalised (qwen3_5.cpp:879-887),
    // q also scaled by 1/sqrt(dk); zero past the sequence end.  A row is 32
    // float4 chunks held by 32 consecutive lanes (half a wave), which take four
    // consecutive tokens
    {
        const int ch = tid & 31, tb = 4 * (tid >> 5);
        float4 kv[4], qv[4];
        if constexpr (CONV) {
            const int cq = kh * kDK + 4 * ch, ck = Hk * kDK + cq;
            float4 qx[7], kx[7];   // inputs of tokens tb - 3 .. tb + 3
#pragma unroll
            for (int i = 0; i < 7; i++) {
                const int tt = t0 + tb + i - 3;
                const float* row = p.proj + (size_t)min(max(tt, 0), S - 1) * p.pd;
                qx[i] = *reinterpret_cast<const float4*>(row + cq);
                kx[i] = *reinterpret_cast<const float4*>(row + ck);
                if (i < 3 && tt < 0) {
                    qx[i] = make_float4(ring_input(p, cq, tt), ring_input(p, cq + 1, tt), ring_input(p, cq + 2, tt),
                                        ring_input(p, cq + 3, tt));
                    kx[i] = make_float4(ring_input(p, ck, tt), ring_input(p, ck + 1, tt), ring_input(p, ck + 2, tt),
                                        ring_input(p, ck + 3, tt));
                }
            }
            float4 wq[4], wk[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                wq[j] = *reinterpret_cast<const float4*>(p.conv_w + (size_t)(cq + j) * 4);
                wk[j] = *reinterpret_cast<const float4*>(p.conv_w + (size_t)(ck + j) * 4);
            }
#pragma unroll
            for (int x = 0; x < 4; x++) {
                qv[x] = make_float4(conv_tap4(qx[x].x, qx[x + 1].x, qx[x + 2].x, qx[x + 3].x, wq[0]),
                                    conv_tap4(qx[x].y, qx[x + 1].y, qx[x + 2].y, qx[x + 3].y, wq[1]),
                                    conv_tap4(qx[x].z, qx[x + 1].z, qx[x + 2].z, qx[x + 3].z, wq[2]),
                                    conv_tap4(qx[x].w, qx[x + 1].w, qx[x + 2].w, qx[x + 3].w, wq[3]));
                kv[x] = make_float4(conv_tap4(kx[x].x, kx[x + 1].x, kx[x + 2].x, kx[x + 3].x, wk[0]),
                                    conv_tap4(kx[x].y, kx[x + 1].y, kx[x + 2].y, kx[x + 3].y, wk[1]),
                                    conv_tap4(kx[x].z, kx[x + 1].z, kx[x + 2].z, kx[x + 3].z, wk[2]),
                                    conv_tap4(kx[x].w, kx[x + 1].w, kx[x + 2].w, kx[x + 3].w, wk[3]));
            }
        } else {
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const size_t off = ((size_t)(t0 + min(tb + x, L - 1)) * Hk + kh) * kDK + 4 * ch;
                kv[x] = *reinterpret_cast<const float4*>(p.k + off);
                qv[x] = *reinterpret_cast<const float4*>(p.q + off);
            }
        }
        const float qk_scale = 1.0f / sqrtf((float)kDK);
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const int t = tb + x;
            float ik = 1.f, iq = 1.f;
            if (p.flags & ANELM_DN_L2NORM) {
                float sk = kv[x].x * kv[x].x + kv[x].y * kv[x].y + kv[x].z * kv[x].z + kv[x].w * kv[x].w;
                float sq = qv[x].x * qv[x].x + qv[x].y * qv[x].y + qv[x].z * qv[x].z + qv[x].w * qv[x].w;
                sk = wave_sum_from<16>(sk);   // over the row's 32 lanes
                sq = wave_sum_from<16>(sq);
                ik = 1.0f / sqrtf(sk + 1e-12f);
                iq = 1.0f / sqrtf(sq + 1e-12f);
            }
            const float mk = t < L ? ik : 0.f, mq = t < L ? iq * qk_scale : 0.f;
            *reinterpret_cast<float4*>(Ks + sw128(t, 4 * ch)) =
                make_float4(kv[x].x * mk, kv[x].y * mk, kv[x].z * mk, kv[x].w * mk);
            *reinterpret_cast<float4*>(Rs + sw128(t, 4 * ch)) =
                make_float4(qv[x].x * mq, qv[x].y * mq, qv[x].z * mq, qv[x].w * mq);
        }
    }
    lds_barrier();
    // ---- the key head's record (one workgroup of the key head): wave w stores
    // Q tiles (w / 2, 4 (w % 2) ..) and K^T row tile w
    if (blockIdx.z == 0) {
        float* kr = p.krec + ((size_t)c * Hk + kh) * kKRec;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const int rt = w >> 1, xt = 4 * (w & 1) + x;
            *reinterpret_cast<v4f*>(kr + ((rt * 8 + xt) * 64 + lane) * 4) =
                *reinterpret_cast<const v4f*>(Rs + sw128(16 * rt + lm, 16 * xt + 4 * lk));
            v4f kt;
#pragma unroll
            for (int j = 0; j < 4; j++) kt[j] = Ks[sw128(16 * x + 4 * lk + j, 16 * w + lm)];
            *reinterpret_cast<v4f*>(kr + kKT + ((w * 4 + x) * 64 + lane) * 4) = kt;
        }
    }
    // A value head's memory operands, requested ahead of the phase before their
    // use: the V rows 16 r + 4 lk + e of the wave's tile (CONV: the inputs of
    // the three tokens before them too), and token `lane`'s gates
    constexpr int NI = CONV ? 7 : 4;
    float vx[4][NI], ga = 0.f, gb = 0.f;
    float4 wv = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load_head = [&](int h) __attribute__((always_inline)) {
        int lt = threadIdx.x & 63;
        asm volatile("" : "+v"(lt));   // (addresses are formed here, not held)
        const int lm = lt & 15, lk = lt >> 4;
        // (rows of a chunk: 32-bit offsets)
        const int last = S - 1 - t0, col = 16 * w + lm;
        const int pd = CONV ? (int)p.pd : Hv * kDV;
        const int cv = CONV ? 2 * Hk * kDK + h * kDV + col : h * kDV + col;
        const float* pv = (CONV ? p.proj : p.v) + (size_t)t0 * pd + cv;
        if constexpr (CONV) wv = *reinterpret_cast<const float4*>(p.conv_w + (size_t)cv * 4);
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int i = 0; i < NI; i++) {
                int t = min(16 * r + 4 * lk + i - (NI - 4), last);
                if (r == 0 && i < NI - 4) t = max(t, -t0);
                vx[r][i] = pv[t * pd];
            }
        if constexpr (CONV) {
            if (t0 == 0 && lk == 0) {
#pragma unroll
                for (int i = 0; i < 3; i++) vx[0][i] = ring_input(p, cv, i - 3);
            }
        }
        if (w == 7) {
            const size_t gi = (size_t)(t0 + min(lt, L - 1)) * p.as + h;
            ga = p.a[gi];
            gb = p.b[gi];
        }
    };
    const int h0 = kh * (Hv / Hk) + blockIdx.z * p.per_wg;
    load_head(h0);
    // ---- Gram tiles: 10 lower tiles of K K^T (ids 0..9) and of Q K^T (10..19);
    // wave w takes ids w, w + 8, w + 16.  Element e of lane (lm, lk) is row
    // 16 ti + lm, column 16 tj + 4 lk + e
    v4f gram[3];
#pragma unroll
    for (int u = 0; u < 3; u++) {
        const int id = w + 8 * u;
        gram[u] = v4f{0.f, 0.f, 0.f, 0.f};
        if (id >= 20) continue;
        const int pi = id % 10, ti = (pi >= 1) + (pi >= 3) + (pi >= 6), tj = pi - ti * (ti + 1) / 2;
        const float* src = id < 10 ? Ks : Rs;
        v4f a0 = gram[u], a1 = gram[u];
#pragma unroll
        for (int x = 0; x < 8; x++) {
            const float4 a4 = *reinterpret_cast<const float4*>(Ks + sw128(16 * tj + lm, 16 * x + 4 * lk));
            const float4 b4 = *reinterpret_cast<const float4*>(src + sw128(16 * ti + lm, 16 * x + 4 * lk));
            a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.x, b4.x, a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.y, b4.y, a1, 0, 0, 0);
            a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.z, b4.z, a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a4.w, b4.w, a1, 0, 0, 0);
        }
        gram[u] = a0 + a1;
        __builtin_amdgcn_sched_barrier(0);   // one tile's operands live at a time
    }
    lds_barrier();   // the query rows are no longer read: their space takes Am
    for (int g = 0; g < p.per_wg; g++) {
        const int h = h0 + g;
        float* out = p.vrec + ((size_t)c * Hv + h) * kVRec;
        // lane-derived addresses are recomputed per value head, not held across the loop
        int ltid = tid;
        asm volatile("" : "+v"(ltid));
        const int lane = ltid & 63, lm = lane & 15, lk = lane >> 4;
        // this head's V rows 16 r + 4 lk + e, column lm of the wave's tile
        float pre[4][4];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float y;
                if constexpr (CONV) y = conv_tap4(vx[r][e], vx[r][e + 1], vx[r][e + 2], vx[r][e + 3], wv);
                else y = vx[r][e];
                pre[r][e] = 16 * r + 4 * lk + e < L ? y : 0.f;
            }
        // ---- beta = sigmoid(b) and log decay = -A softplus(a + dt_bias)
        // (qwen3_5.cpp:896-898); lg[t + 1] = sum_{j <= t} log decay_j (wave 7)
        if (w == 7) {
            float x = 0.f, bv = 0.f;
            if (lane < L) {
                bv = 1.0f / (1.0f + expf(-gb));
                x = -p.A[h] * logf(1.0f + expf(ga + p.dt_bias[h]));
            }
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const float y = __shfl_up(x, d, 64);
                if (lane >= d) x += y;
            }
            lg[lane + 1] = x;
            if (lane == 0) lg[0] = 0.f;
            bt[lane] = bv;
            // the per-row decay factors, evaluated once per row
            const float xs = __shfl_up(x, 1, 64);   // (every lane takes part in the shuffles)
            const float xl = __shfl(x, 63, 64);     // lg_L
            const float xp = lane == 0 ? 0.f : xs;  // lg[t]
            const float e1 = expf(x);
            eb[lane] = TF ? e1 : expf(xp);
            out[kVE + lane] = e1;
            out[kVE + 64 + lane] = expf(xl - x);
            if (lane == 63) out[kVE + 128] = e1;    // gC
        }
        lds_barrier();
        // ---- Am = -A and P from the Gram tiles
#pragma unroll
        for (int u = 0; u < 3; u++) {
            const int id = w + 8 * u;
            if (id >= 20) continue;
            const int pi = id % 10, ti = (pi >= 1) + (pi >= 3) + (pi >= 6), tj = pi - ti * (ti + 1) / 2;
            const int t = 16 * ti + lm, i0 = 16 * tj + 4 * lk;
            const bool isA = id < 10;
            const float lgt = isA && !TF ? lg[t] : lg[t + 1], bs = -bt[t];
            v4f o4;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int i = i0 + e;
                const float f = expf(lgt - lg[i + 1]);
                if (isA) o4[e] = i < t ? bs * f * gram[u][e] : 0.f;
                else o4[e] = i <= t ? f * gram[u][e] : 0.f;
            }
            if (isA) *reinterpret_cast<v4f*>(Am + sw64(t, i0)) = o4;
            else *reinterpret_cast<v4f*>(out + kVP + (pi * 64 + lane) * 4) = o4;
        }
        lds_barrier();
        if (w == 0) {
            // ---- T_rr = (I + A_rr)^-1 for the 4 diagonal blocks: lane 16 b + j
            // computes column j of block b by substitution, then writes it over A_rr
            const int b = lk, j = lm;
            float x[16];
#pragma unroll
            for (int t = 0; t < 16; t++) {
                float acc = t == j ? 1.f : 0.f;
#pragma unroll
                for (int i4 = 0; i4 < t; i4 += 4) {
                    const float4 a4 = *reinterpret_cast<const float4*>(Am + sw64(16 * b + t, 16 * b + i4));
                    acc = fmaf(a4.x, x[i4], acc);
                    if (i4 + 1 < t) acc = fmaf(a4.y, x[i4 + 1], acc);
                    if (i4 + 2 < t) acc = fmaf(a4.z, x[i4 + 2], acc);
                    if (i4 + 3 < t) acc = fmaf(a4.w, x[i4 + 3], acc);
                }
                x[t] = acc;
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = 0; t < 16; t++) Am[sw64(16 * b + t, 16 * b + j)] = x[t];
        }
        lds_barrier();
        if (g + 1 < p.per_wg) load_head(h + 1);
        // ---- X of this wave's two tiles (u 0: V, u 1: K), block row by block row
        v4f X[2][4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            // B_r in the accumulator layout: rows 16 r + 4 lk + e, column lm
            v4f acc[2], xr[2];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = 16 * r + 4 * lk + e;
                const float bv = bt[t];
                acc[0][e] = bv * pre[r][e];
                acc[1][e] = bv * (Ks[sw128(t, 16 * w + lm)] * eb[t]);
            }
#pragma unroll
            for (int s2 = 0; s2 < r; s2++) {
                const v4f a4 = *reinterpret_cast<const v4f*>(Am + sw64(16 * r + lm, 16 * s2 + 4 * lk));
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[e], X[u][s2][e], acc[u], 0, 0, 0);
            }
            const v4f t4 = *reinterpret_cast<const v4f*>(Am + sw64(16 * r + lm, 16 * r + 4 * lk));
            xr[0] = xr[1] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int u = 0; u < 2; u++)
                    xr[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(t4[e], acc[u][e], xr[u], 0, 0, 0);
            X[0][r] = xr[0];
            X[1][r] = xr[1];
            // Ut: the D fragment; Wm: transposed in quads, lane (4 c + i, k)
            // then holds row 4 k + i, columns 4 c .. 4 c + 3 of its A fragment
            *reinterpret_cast<v4f*>(out + ((r * 8 + w) * 64 + lane) * 4) = xr[0];
            *reinterpret_cast<v4f*>(out + kVW + ((r * 8 + w) * 64 + 4 * lk + (lm & 3) + 16 * (lm >> 2)) * 4) =
                quad_transpose(xr[1], lane);
            __builtin_amdgcn_sched_barrier(0);   // bounds the loads hoisted ahead of this row
        }
        lds_barrier();   // Am, lg and beta are rewritten for the next value head
    }
}

// The state is carried through the chunks in slabs of 16 columns (8 per head).
constexpr int kSeqCB = 16;
constexpr int kSlabs = kDV / kSeqCB;

// ------------------------------------------------ chunk scan on fp32 MFMA
// The state products per chunk on v_mfma_f32_16x16x4_f32 (fp32 inputs, fp32
// accumulation).  A workgroup (8 waves, two per SIMD) owns a 16-column slab of
// one head's state.  Only X = Wm S0 -> U -> S_end stands between one chunk and
// the next, so the waves split by role:
//   waves 0-3 (one per SIMD, raised priority) carry the state: X of chunk rows
//     [16 w, 16 w + 16), U = Ut - X and its decayed copy to LDS | barrier |
//     S = gC S + K^T (decayed U) of state rows [32 w, 32 w + 32), kept in
//     registers and published to the other of two LDS slabs | barrier;
//   waves 4-7 form the outputs of chunk rows [16 (w - 4), ...) in their wake:
//     the first half of Q S0 beside the state update, the second half and
//     diag(exp(lg)) (.) + P U beside the next chunk's X (the slab and U of a
//     chunk stay in LDS until then).
// Every operand but the slab and U is read by one wave only, so it goes from
// memory straight into registers (1 KiB fragments), the next chunk's loads
// spread over this chunk's products: issued all at once they fill the CU's
// memory queue and the waves stall at their next memory instruction.
// Bound: the fp32 matrix units and the chain above: a chunk takes 5300 clocks
// of which 3400 are the two waves' products; 4096 tokens of 32 heads 158 us
// (195 with all waves on both roles, 270 with row-major records too).
constexpr int kMsNT = 512;
constexpr int kScP = kDK + 4;        // slab column pitch (floats): 16-byte reads of 16 lanes hit distinct banks
constexpr int kUlP = kChunk + 4;     // U column pitch, likewise
constexpr int kMsLds = kSeqCB * (2 * kScP + 3 * kUlP) * 4;

struct ScanArgs {
    float* y;              // [S][Hv][dv]
    float* state;
    const float* vrec;
    const float* krec;
    int S, Hk, Hv, n_chunks;
    // the conv ring after the prompt (null: none): input t sits at slot
    // (conv_pos + t) mod 3, so the last 3 inputs overwrite their slots
    float* conv_state;     // [C][3]
    const float* proj;     // [S][pd]
    long pd;
    int C, conv_pos;
};

// The two records of chunk ch for head h, as buffer resources (offsets stay
// small for any sequence length).
struct ScanSrc {
    __amdgpu_buffer_rsrc_t rv, rk;
};
__device__ __forceinline__ ScanSrc scan_src(const ScanArgs& a, int ch, int h) {
    ch = min(ch, a.n_chunks - 1);   // (past the last chunk: its operands again, unused)
    ScanSrc s;
    s.rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.vrec) + ((size_t)ch * a.Hv + h) * kVRec, 0, kVRec * 4,
                                             0x00020000);
    s.rk = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.krec) + ((size_t)ch * a.Hk + h / (a.Hv / a.Hk)) * kKRec, 0, kKRec * 4, 0x00020000);
    return s;
}
__device__ __forceinline__ v4f scan_ld(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// Operands of one chunk: a state wave's, an output wave's.
struct StateOps {
    v4f m[8];       // Wm row tile w
    v4f kt[2][4];   // K^T row tiles 2w, 2w + 1
    v4f u, ev;      // Ut (row tile w, this slab's columns); exp(lg_L - lg) of its rows
    float gc;
};
struct OutOps {
    v4f q[8];       // Q row tile mt
    v4f p[4];       // P tiles (mt, x <= mt)
    v4f ev;         // exp(lg) of its rows
};

// Wave 4 + MT of the scan: the outputs of chunk rows [16 MT, 16 MT + 16).
template <int MT>
__device__ __forceinline__ void scan_outputs(const ScanArgs& a, float (*Sc)[kScP], float (*Ul)[kUlP], int h, int c0,
                                             int lane) {
    const int lr = lane & 15, lq = lane >> 4, Hv = a.Hv, n_chunks = a.n_chunks;
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    const __amdgpu_buffer_rsrc_t ry =
        __builtin_amdgcn_make_buffer_rsrc(a.y, 0, (int)((size_t)a.S * Hv * kDV * 4), 0x00020000);
    const int qo = (MT * 8 * 64 + lane) * 16, po = (kVP + (MT * (MT + 1) / 2 * 64 + lane) * 4) * 4;
    const int eo = (kVE + 16 * MT + 4 * lq) * 4;
    OutOps opA, opB;
    v4f Z[4];
    // part x (0..3) of a chunk's second loads (the first four Q tiles are loaded a step earlier)
    auto load2 = [&](OutOps& o, const ScanSrc& s, int x) __attribute__((always_inline)) {
        o.q[4 + x] = scan_ld(s.rk, qo + (4 + x) * 1024);
        if (x <= MT) o.p[x] = scan_ld(s.rv, po + x * 1024);
        if (x == 0) o.ev = scan_ld(s.rv, eo);
    };
    // Q S0 of chunk ch, state rows 0..63, the first operands of chunk ch + 1 requested
    auto first = [&](const OutOps& cur, OutOps& nxt, int ch, int par) __attribute__((always_inline)) {
        const ScanSrc src = scan_src(a, ch + 1, h);
        float (*sc)[kScP] = Sc + par * kSeqCB;
        v4f sb[4];
#pragma unroll
        for (int x = 0; x < 4; x++) sb[x] = *reinterpret_cast<const v4f*>(&sc[lr][16 * x + 4 * lq]);
#pragma unroll
        for (int e = 0; e < 4; e++) Z[e] = zero;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            nxt.q[x] = scan_ld(src.rk, qo + x * 1024);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; e++)
                Z[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.q[x][e], sb[x][e], Z[e], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the rest of chunk ch's outputs, the other operands of chunk ch + 1 requested
    auto finish = [&](const OutOps& cur, OutOps& nxt, int ch, int par) __attribute__((always_inline)) {
        const ScanSrc src = scan_src(a, ch + 1, h);
        float (*sc)[kScP] = Sc + par * kSeqCB;
        float (*ul)[kUlP] = Ul + par * kSeqCB;
        v4f uv[MT + 1], sb[4], T[4];
#pragma unroll
        for (int x = 0; x <= MT; x++) uv[x] = *reinterpret_cast<const v4f*>(&ul[lr][16 * x + 4 * lq]);
#pragma unroll
        for (int x = 0; x < 4; x++) sb[x] = *reinterpret_cast<const v4f*>(&sc[lr][64 + 16 * x + 4 * lq]);
#pragma unroll
        for (int e = 0; e < 4; e++) T[e] = zero;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            load2(nxt, src, x);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (x <= MT) T[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.p[x][e], uv[x][e], T[e], 0, 0, 0);
                Z[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.q[4 + x][e], sb[x][e], Z[e], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const v4f y = ((Z[0] + Z[1]) + (Z[2] + Z[3])) * cur.ev + ((T[0] + T[1]) + (T[2] + T[3]));
        // rows past S fall out of the buffer range and are dropped
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float yv = y[j];   // (a bit_cast of a vector element is lowered as element 0)
            const int off = (((ch * kChunk + 16 * MT + 4 * lq + j) * Hv + h) * kDV + c0 + lr) * 4;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, yv), ry, off, 0, 0);
        }
    };
    {
        const ScanSrc s = scan_src(a, 0, h);
#pragma unroll
        for (int x = 0; x < 4; x++) opA.q[x] = scan_ld(s.rk, qo + x * 1024);
#pragma unroll
        for (int x = 0; x < 4; x++) load2(opA, s, x);
    }
    __syncthreads();
    lds_barrier();
    first(opA, opB, 0, 0);
    lds_barrier();
    // (beside the state waves' chunk ch: finish ch - 1 | barrier | first half of ch | barrier)
    int ch = 1;
    for (; ch + 1 < n_chunks; ch += 2) {
        finish(opA, opB, ch - 1, 0);
        lds_barrier();
        first(opB, opA, ch, 1);
        lds_barrier();
        finish(opB, opA, ch, 1);
        lds_barrier();
        first(opA, opB, ch + 1, 0);
        lds_barrier();
    }
    if (ch < n_chunks) {
        finish(opA, opB, ch - 1, 0);
        lds_barrier();
        first(opB, opA, ch, 1);
        lds_barrier();
        finish(opB, opA, ch, 1);
    } else {
        finish(opA, opB, ch - 1, 0);
    }
}

__global__ __launch_bounds__(kMsNT) __attribute__((amdgpu_waves_per_eu(2, 2))) void dn_chunk_scan_kernel(
    const ScanArgs a) {
    extern __shared__ __attribute__((aligned(16))) float smem[];
    typedef float (*Slab)[kScP];
    typedef float (*Ucols)[kUlP];
    Slab Sc = reinterpret_cast<Slab>(smem);                            // [2 x 16] columns: slab of even / odd chunks
    Ucols Ul = reinterpret_cast<Ucols>(smem + 2 * kSeqCB * kScP);      // [2 x 16] U of even / odd chunks
    Ucols Ud = Ul + 2 * kSeqCB;                                        // decayed U of this chunk
    const int S = a.S, n_chunks = a.n_chunks;
    // XCD-aware: the 8 slabs of a head share its chunk records, so they go to
    // one XCD (workgroup id mod 8 selects the XCD; Hv * 8 workgroups)
    const int nwg = gridDim.x, id = blockIdx.x;
    const int per_xcd = nwg / 8, k8 = id / 8, xcd = id % 8;
    const int h = (xcd * per_xcd + k8) / kSlabs, slab = (xcd * per_xcd + k8) % kSlabs;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lq = lane >> 4;
    const int mt = w & 3;
    const int c0 = slab * kSeqCB;
    float* Sp = a.state + (size_t)h * kDK * kDV;
    for (int e = tid; e < kDK * kSeqCB; e += kMsNT) {
        const int i = e / kSeqCB, c = e % kSeqCB;
        Sc[c][i] = Sp[(size_t)i * kDV + c0 + c];
    }
    if (a.conv_state != nullptr) {
        const int nt = min(S, 3);
        for (int e = id * kMsNT + tid; e < a.C * nt; e += nwg * kMsNT) {
            const int t = S - nt + e / a.C, c = e % a.C;
            a.conv_state[(size_t)c * 3 + (a.conv_pos + t) % 3] = a.proj[(size_t)t * a.pd + c];
        }
    }
    const v4f zero = {0.f, 0.f, 0.f, 0.f};

    if (w < 4) {
        // ------------------------------------------------ state waves
        const int mo = (kVW + (mt * 8 * 64 + lane) * 4) * 4, ko = (kKT + (mt * 8 * 64 + lane) * 4) * 4;
        const int uo = ((mt * 8 + slab) * 64 + lane) * 16, eo = (kVE + 64 + 16 * mt + 4 * lq) * 4;
        // two operand sets: a chunk is computed from one while the next
        // chunk's loads land in the other (no register copies between them)
        StateOps opA, opB;
        {
            const ScanSrc s = scan_src(a, 0, h);
#pragma unroll
            for (int x = 0; x < 8; x++) opA.m[x] = scan_ld(s.rv, mo + x * 1024);
            opA.u = scan_ld(s.rv, uo);
            opA.ev = scan_ld(s.rv, eo);
            opA.gc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(s.rv, (kVE + 128) * 4, 0, 0));
#pragma unroll
            for (int x = 0; x < 8; x++) opA.kt[x >> 2][x & 3] = scan_ld(s.rk, ko + x * 1024);
        }
        __builtin_amdgcn_s_setprio(2);
        __syncthreads();
        v4f Sr[2];   // this wave's state rows: 32 w + 16 t + 4 lq + (0..3), column lr
#pragma unroll
        for (int t = 0; t < 2; t++) Sr[t] = *reinterpret_cast<const v4f*>(&Sc[lr][32 * mt + 16 * t + 4 * lq]);
        auto chunk = [&](const StateOps& cur, StateOps& nxt, int ch, int par) __attribute__((always_inline)) {
            const ScanSrc src = scan_src(a, ch + 1, h);
            Slab sc = Sc + par * kSeqCB;
            v4f sb[8], Z[4];
#pragma unroll
            for (int x = 0; x < 8; x++) sb[x] = *reinterpret_cast<const v4f*>(&sc[lr][16 * x + 4 * lq]);
#pragma unroll
            for (int e = 0; e < 4; e++) Z[e] = zero;
            // ---- X = Wm S0: 32 products in 4 chains
#pragma unroll
            for (int x = 0; x < 8; x++) {
                nxt.m[x] = scan_ld(src.rv, mo + x * 1024);
                if (x == 6) nxt.u = scan_ld(src.rv, uo);
                __builtin_amdgcn_sched_barrier(0);   // the loads are issued here, not hoisted or sunk
#pragma unroll
                for (int e = 0; e < 4; e++)
                    Z[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.m[x][e], sb[x][e], Z[e], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            // element j is chunk row 16 w + 4 lq + j, slab column lr
            const v4f U = cur.u - ((Z[0] + Z[1]) + (Z[2] + Z[3]));
            *reinterpret_cast<v4f*>(&Ud[lr][16 * mt + 4 * lq]) = U * cur.ev;
            *reinterpret_cast<v4f*>(&(Ul + par * kSeqCB)[lr][16 * mt + 4 * lq]) = U;
            lds_barrier();   // U complete
            // ---- S = gC S + K^T Ud: 2 row tiles, 16 products each in 2 chains
            v4f ub[4], T[2][2];
#pragma unroll
            for (int x = 0; x < 4; x++) ub[x] = *reinterpret_cast<const v4f*>(&Ud[lr][16 * x + 4 * lq]);
#pragma unroll
            for (int t = 0; t < 2; t++) {
                T[t][0] = cur.gc * Sr[t];
                T[t][1] = zero;
            }
#pragma unroll
            for (int x = 0; x < 4; x++) {
                nxt.kt[0][x] = scan_ld(src.rk, ko + x * 1024);
                nxt.kt[1][x] = scan_ld(src.rk, ko + (4 + x) * 1024);
                if (x == 2) nxt.ev = scan_ld(src.rv, eo);
                if (x == 3)
                    nxt.gc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src.rv, (kVE + 128) * 4, 0, 0));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int t = 0; t < 2; t++)
                        T[t][e & 1] =
                            __builtin_amdgcn_mfma_f32_16x16x4f32(cur.kt[t][x][e], ub[x][e], T[t][e & 1], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            sc = Sc + (par ^ 1) * kSeqCB;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                Sr[t] = T[t][0] + T[t][1];
                *reinterpret_cast<v4f*>(&sc[lr][32 * mt + 16 * t + 4 * lq]) = Sr[t];
            }
            lds_barrier();   // new state complete
        };
        // pairs of chunks, then an odd last one: inside the loop both halves run
        // unconditionally, so the loads a half issues for the other are not sunk
        // into a conditional block next to their use
        int ch = 0;
        for (; ch + 1 < n_chunks; ch += 2) {
            chunk(opA, opB, ch, 0);
            chunk(opB, opA, ch + 1, 1);
        }
        if (ch < n_chunks) chunk(opA, opB, ch, 0);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) Sp[(size_t)(32 * mt + 16 * t + 4 * lq + j) * kDV + c0 + lr] = Sr[t][j];
    } else {
        switch (mt) {
            case 0: scan_outputs<0>(a, Sc, Ul, h, c0, lane); break;
            case 1: scan_outputs<1>(a, Sc, Ul, h, c0, lane); break;
            case 2: scan_outputs<2>(a, Sc, Ul, h, c0, lane); break;
            default: scan_outputs<3>(a, Sc, Ul, h, c0, lane); break;
        }
    }
}

// Both launches over the inputs of `p` (vrec, krec and per_wg are set here).
int chunk_prefill(ChunkArgs p, ScanArgs s, bool conv, hipStream_t st) {
    Device* dev = device();
    if (!dev) return ANELM_EHIP;
    const int n_chunks = (p.S + kChunk - 1) / kChunk, G = p.Hv / p.Hk;
    const size_t nv = (size_t)n_chunks * p.Hv * kVRec, nk = (size_t)n_chunks * p.Hk * kKRec;
    float* rec = static_cast<float*>(workspace((nv + nk) * sizeof(float), st));
    if (!rec) return ANELM_ENOMEM;
    p.vrec = rec;
    p.krec = rec + nv;
    using K = void (*)(const ChunkArgs);
    static const K kern[2][2] = {{dn_chunk_prep_kernel<false, false>, dn_chunk_prep_kernel<false, true>},
                                 {dn_chunk_prep_kernel<true, false>, dn_chunk_prep_kernel<true, true>}};
    static DeviceOnce lds[2][2];
    const int t = p.flags & ANELM_DN_ORDER_TRANSFORMERS ? 1 : 0, c = conv ? 1 : 0;
    const int rc = allow_lds(lds[t][c], reinterpret_cast<const void*>(kern[t][c]), kPmLds);
    if (rc) return rc;
    // a workgroup takes all value heads of its key head where that fills the
    // chip (two workgroups per CU), else one (the Gram tiles formed again)
    const bool each = G > 1 && (long)n_chunks * p.Hk < 2L * dev->num_cus;
    p.per_wg = each ? 1 : G;
    hipLaunchKernelGGL(kern[t][c], dim3(n_chunks, p.Hk, each ? G : 1), dim3(kPmNT), kPmLds, st, p);
    ANELM_LAUNCHED("dn_chunk_prep_kernel");
    s.vrec = p.vrec;
    s.krec = p.krec;
    s.S = p.S;
    s.Hk = p.Hk;
    s.Hv = p.Hv;
    s.n_chunks = n_chunks;
    // grid = Hv * kSlabs, a multiple of 8 (XCD mapping inside the kernel)
    hipLaunchKernelGGL(dn_chunk_scan_kernel, dim3(kSlabs * p.Hv), dim3(kMsNT), kMsLds, st, s);
    ANELM_LAUNCHED("dn_chunk_scan_kernel");
    return ANELM_OK;
}

}  // namespace
}  // namespace anelm

using namespace anelm;

namespace anelm {
namespace {
int deltanet_decode_impl(float* y, float* state, const float* q, const float* k, const float* v, const float* a,
                         const float* b, const float* A, const float* dt_bias, const float* z, const float* norm_w,
                         int n_seqs, int Hk, int Hv, int dk, int dv, int flags, hipStream_t st);
}  // namespace
}  // namespace anelm

extern "C" int anelm_deltanet_decode(float* y, float* state, const float* q, const float* k,
                                     const float* v, const float* a, const float* b,
                                     const float* A, const float* dt_bias, const float* z,
                                     const float* norm_w, int Hk, int Hv, int dk, int dv,
                                     int flags, void* stream) {
    return deltanet_decode_impl(y, state, q, k, v, a, b, A, dt_bias, z, norm_w, 1, Hk, Hv, dk, dv, flags,
                                as_stream(stream));
}

extern "C" int anelm_deltanet_decode_batched(float* y, float* state, const float* q, const float* k,
                                             const float* v, const float* a, const float* b,
                                             const float* A, const float* dt_bias, const float* z,
                                             const float* norm_w, int n_seqs, int Hk, int Hv, int dk,
                                             int dv, int flags, void* stream) {
    return deltanet_decode_impl(y, state, q, k, v, a, b, A, dt_bias, z, norm_w, n_seqs, Hk, Hv, dk, dv, flags,
                                as_stream(stream));
}

namespace anelm {
namespace {
// n_seqs sequences of Hk key / Hv value heads as one launch over n_seqs * Hv
// heads: sequence s's value head j is head s*Hv + j, its key head
// s*Hk + j/(Hv/Hk) -- the same h / (Hv/Hk) mapping over the stacked heads --
// and A / dt_bias (layer weights) are shared by the sequences.
int deltanet_decode_impl(float* y, float* state, const float* q, const float* k, const float* v, const float* a,
                         const float* b, const float* A, const float* dt_bias, const float* z, const float* norm_w,
                         int n_seqs, int Hk, int Hv, int dk, int dv, int flags, hipStream_t st) {
    ANELM_NONNULL(y);
    ANELM_NONNULL(state);
    ANELM_NONNULL(q);
    ANELM_NONNULL(k);
    ANELM_NONNULL(v);
    ANELM_NONNULL(a);
    ANELM_NONNULL(b);
    ANELM_NONNULL(A);
    ANELM_NONNULL(dt_bias);
    ANELM_REQUIRE(dk == kDK && dv == kDV, "deltanet_decode: dk=%d dv=%d (only 128x128)", dk, dv);
    ANELM_REQUIRE(Hk > 0 && Hv > 0 && Hv % Hk == 0, "deltanet_decode: Hv %d not a multiple of Hk %d",
                  Hv, Hk);
    ANELM_REQUIRE((flags & ~7) == 0, "deltanet_decode: unknown flags 0x%x", flags);
    ANELM_REQUIRE(n_seqs > 0 && (long)n_seqs * Hv <= 65535, "deltanet_decode: %d sequences x %d value heads "
                  "(at most 65535 heads per launch)", n_seqs, Hv);
    DnParams p{};
    p.y = y;
    p.state = state;
    p.q = q;
    p.k = k;
    p.v = v;
    p.a = a;
    p.b = b;
    p.A = A;
    p.dt_bias = dt_bias;
    p.Hk = Hk * n_seqs;
    p.Hv = Hv * n_seqs;
    p.w_heads = Hv;
    p.flags = flags;
    if (flags & ANELM_DN_GATED_NORM) {
        ANELM_NONNULL(z);
        ANELM_NONNULL(norm_w);
        p.z = z;
        p.norm_w = norm_w;
        hipLaunchKernelGGL((deltanet_decode_kernel<128, 512, true>), dim3(1, p.Hv), dim3(512), 0, st, p);
    } else {
        hipLaunchKernelGGL((deltanet_decode_kernel<32, 256, false>), dim3(kDV / 32, p.Hv), dim3(256), 0,
                           st, p);
    }
    ANELM_LAUNCHED("deltanet_decode_kernel");
    return ANELM_OK;
}
}  // namespace
}  // namespace anelm

extern "C" int anelm_deltanet_decode_from_proj(float* y, float* state, float* conv_state, int* conv_pos,
                                               const float* proj, const float* conv_w, const float* A,
                                               const float* dt_bias, const float* norm_w, int Hk, int Hv,
                                               int dk, int dv, int conv_kernel, int flags, void* stream) {
    ANELM_NONNULL(y);
    ANELM_NONNULL(state);
    ANELM_NONNULL(conv_state);
    ANELM_NONNULL(conv_pos);
    ANELM_NONNULL(proj);
    ANELM_NONNULL(conv_w);
    ANELM_NONNULL(A);
    ANELM_NONNULL(dt_bias);
    ANELM_REQUIRE(dk == kDK && dv == kDV, "deltanet_decode_from_proj: dk=%d dv=%d (only 128x128)", dk, dv);
    ANELM_REQUIRE(Hk > 0 && Hv > 0 && Hv % Hk == 0 && Hv <= 65535,
                  "deltanet_decode_from_proj: Hv %d not a multiple of Hk %d", Hv, Hk);
    ANELM_REQUIRE(conv_kernel >= 2 && conv_kernel <= 16, "deltanet_decode_from_proj: conv kernel %d",
                  conv_kernel);
    ANELM_REQUIRE(*conv_pos >= 0 && *conv_pos < conv_kernel - 1, "deltanet_decode_from_proj: conv_pos %d",
                  *conv_pos);
    ANELM_REQUIRE((flags & ~7) == 0, "deltanet_decode_from_proj: unknown flags 0x%x", flags);
    const bool gated = (flags & ANELM_DN_GATED_NORM) != 0;
    ANELM_REQUIRE(!gated || norm_w != nullptr, "deltanet_decode_from_proj: GATED_NORM needs norm_w");
    hipStream_t st = as_stream(stream);
    uint32_t* ctr = counters((size_t)Hk, kCtrDeltaNetConv, st);
    if (!ctr) return ANELM_ERANGE;
    const long qkv = 2L * Hk * kDK + (long)Hv * kDV;
    DnParams p{};
    p.y = y;
    p.state = state;
    p.z = proj + qkv;                       // [Hv][dv]
    p.a = p.z + (long)Hv * kDV;             // [Hv]
    p.b = p.a + Hv;                         // [Hv]
    p.A = A;
    p.dt_bias = dt_bias;
    p.norm_w = norm_w;
    p.Hk = Hk;
    p.Hv = Hv;
    p.w_heads = Hv;
    p.flags = flags;
    p.mix = proj;
    p.conv_state = conv_state;
    p.conv_w = conv_w;
    p.conv_pos = *conv_pos;
    p.conv_k = conv_kernel;
    p.readers_done = ctr;
    if (gated) {
        p.readers = Hv / Hk;
        hipLaunchKernelGGL((deltanet_decode_kernel<128, 512, true, true>), dim3(1, Hv), dim3(512), 0, st, p);
    } else {
        p.readers = (Hv / Hk) * (kDV / 32);
        hipLaunchKernelGGL((deltanet_decode_kernel<32, 256, false, true>), dim3(kDV / 32, Hv), dim3(256), 0, st,
                           p);
    }
    ANELM_LAUNCHED("deltanet_decode_kernel (conv prologue)");
    int np = *conv_pos + 1;
    if (np == conv_kernel - 1) np = 0;
    *conv_pos = np;
    return ANELM_OK;
}

extern "C" int anelm_deltanet_prefill(float* y, float* state, const float* q, const float* k,
                                      const float* v, const float* a, const float* b,
                                      const float* A, const float* dt_bias, int S, int Hk, int Hv,
                                      int dk, int dv, int chunk, int flags, void* stream) {
    ANELM_NONNULL(y);
    ANELM_NONNULL(state);
    ANELM_NONNULL(q);
    ANELM_NONNULL(k);
    ANELM_NONNULL(v);
    ANELM_NONNULL(a);
    ANELM_NONNULL(b);
    ANELM_NONNULL(A);
    ANELM_NONNULL(dt_bias);
    ANELM_REQUIRE(dk == kDK && dv == kDV, "deltanet_prefill: dk=%d dv=%d (only 128x128)", dk, dv);
    ANELM_REQUIRE(Hk > 0 && Hv > 0 && Hv % Hk == 0 && Hv / Hk <= kDK,
                  "deltanet_prefill: Hv %d not a multiple of Hk %d", Hv, Hk);
    ANELM_REQUIRE(S >= 0, "deltanet_prefill: S %d", S);
    ANELM_REQUIRE(chunk == kChunk || chunk == 1,
                  "deltanet_prefill: chunk %d (64: chunked form; 1: token-by-token scan)", chunk);
    ANELM_REQUIRE((size_t)(S + kChunk) * Hv * kDV * sizeof(float) < 0x7fffffffu,
                  "deltanet_prefill: %d tokens x %d heads exceed the 2 GiB output range", S, Hv);
    ANELM_REQUIRE((flags & ~3) == 0, "deltanet_prefill: flags 0x%x (GATED_NORM is decode-only)", flags);
    if (S == 0) return ANELM_OK;
    hipStream_t st = as_stream(stream);
    if (chunk == 1) {
        const size_t nqk = (size_t)S * Hk * kDK, ng = (size_t)S * Hv;
        float* ws = static_cast<float*>(workspace((2 * nqk + 3 * ng) * sizeof(float), st));
        if (!ws) return ANELM_ENOMEM;
        float* qn = ws;
        float* kn = qn + nqk;
        float* beta = kn + nqk;
        float* decay = beta + ng;
        float* ldecay = decay + ng;
        hipLaunchKernelGGL(dn_prep_kernel, dim3((S * Hk + kPrepRows - 1) / kPrepRows), dim3(64 * kPrepRows), 0, st,
                           qn, kn, beta, decay, ldecay, q, k, a, b, A, dt_bias, S, Hk, Hv, flags);
        ANELM_LAUNCHED("dn_prep_kernel");
        hipLaunchKernelGGL(dn_scan_kernel, dim3(kDV / kScanCB, Hv), dim3(kScanNT), 0, st, y, state, qn,
                           kn, v, beta, decay, S, Hk, Hv, flags);
        ANELM_LAUNCHED("dn_scan_kernel");
        return ANELM_OK;
    }
    ChunkArgs p{};
    p.q = q;
    p.k = k;
    p.v = v;
    p.a = a;
    p.b = b;
    p.as = Hv;
    p.A = A;
    p.dt_bias = dt_bias;
    p.S = S;
    p.Hk = Hk;
    p.Hv = Hv;
    p.flags = flags;
    ScanArgs s{};
    s.y = y;
    s.state = state;
    return chunk_prefill(p, s, false, st);
}

namespace anelm {
// Chunked prefill straight from the projection rows (conv width 4).
bool deltanet_prefill_proj_fits(const float* proj, const float* conv_w, int pd, int conv_kernel) {
    return conv_kernel == 4 && pd % 4 == 0 &&
           ((reinterpret_cast<uintptr_t>(proj) | reinterpret_cast<uintptr_t>(conv_w)) & 15) == 0;
}

int deltanet_prefill_proj(float* y, float* state, float* conv_state, int conv_pos, const float* proj,
                          const float* conv_w, const float* A, const float* dt_bias, int S, int Hk, int Hv, int pd,
                          int flags, hipStream_t st) {
    ANELM_REQUIRE(Hv / Hk <= kDK && (size_t)(S + kChunk) * Hv * kDV * sizeof(float) < 0x7fffffffu,
                  "deltanet_prefill: %d tokens x %d heads exceed the 2 GiB output range", S, Hv);
    ChunkArgs p{};
    const int C = 2 * Hk * kDK + Hv * kDV;
    p.proj = proj;
    p.pd = pd;
    p.conv_state = conv_state;
    p.conv_w = conv_w;
    p.conv_pos = conv_pos;
    p.a = proj + C + Hv * kDV;
    p.b = p.a + Hv;
    p.as = pd;
    p.A = A;
    p.dt_bias = dt_bias;
    p.S = S;
    p.Hk = Hk;
    p.Hv = Hv;
    p.flags = flags;
    ScanArgs s{};
    s.y = y;
    s.state = state;
    s.conv_state = conv_state;
    s.proj = proj;
    s.pd = pd;
    s.C = C;
    s.conv_pos = conv_pos;
    return chunk_prefill(p, s, true, st);
}
}  // namespace anelm
