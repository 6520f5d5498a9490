// The recurrences whose state is a matrix S [d keys][dv values] per head -- wkv and gated linear attention (a decay per key channel), the gated delta rule (one decay per head) -- for a
// portion of tokens, in CHUNKS of 16 on the fp32 matrix cores.  What bounded the token-by-token scans (k_seqmix.hip) was a token's chain of LDS reads, sums over a column's lanes and
// the update, 0.6 - 0.8 us a token whatever the number of heads.  With c_t the running sum of a chunk's log decays (each held above CK_LEAST, kept in double: |c| <= 2048, so a
// difference of two is good to 5e-13; exponents are never positive), S the state in front of the chunk and tokens t, s of it:
//   decay per channel   o_t = (r_t exp(c_(t-1))) S + sum_(s < t) A_ts v_s + (r_t . bonus k_t) v_t,  A_ts = sum_i r_ti k_si exp(c_(t-1)i - c_si)      (wkv)
//                       o_t = (q_t exp(c_t)) S + sum_(s <= t) A_ts v_s,  A_ts = sum_i q_ti k_si exp(c_ti - c_si)                                      (gated linear attention)
//                       S   <- diag(exp(c_end)) S + sum_s (k_s exp(c_end - c_s)) v_s^T
//   delta rule          U   = M (V - (K exp(c)) S),  M = (I + L)^-1 diag(beta),  L_ts = beta_t exp(c_t - c_s) (k_t . k_s) for s < t
//                       o_t = (q_t exp(c_t)) S + sum_(s <= t) B_ts u_s,  B_ts = exp(c_t - c_s) (q_t . k_s);   S <- exp(c_end) S + sum_s (k_s exp(c_end - c_s)) u_s^T
// Everything that does not depend on the state -- the scaled q, k rows, the 16 x 16 matrices (M by forward substitution in double) -- is made for all chunks at once by the two
// prep kernels; chunk_scan_kernel walks the chunks with the state in the matrix instructions' accumulators.  Measured, 512 tokens of 16 heads of 128 x 128: wkv 303 -> 19 + 32 us,
// delta rule 391 -> 13 + 45 us (token by token and in chunks, the first form of the scan); 2047 tokens, the scan alone, that form and now, under the profiler: wkv 148 -> 70 us, delta rule 222 -> 115.
#include "ps_attn_dev.h"
#include "ps_seq.h"

#include <cmath>
#include <type_traits>

typedef float ck_f4 __attribute__((ext_vector_type(4)));
typedef float ck_f2 __attribute__((ext_vector_type(2)));
typedef double ck_d2 __attribute__((ext_vector_type(2)));
#define CK_Q 16
#define CK_AHEAD 2 // chunks (3 and 4 are no faster)

// A token's log decay, from below: e^-128 is zero in fp32 as every decay below it is (the scans' exp(-1e30) or exp(-inf)), but beside a -1e13 in the running sum the decays behind it would
// be lost, and -inf - -inf is no number.  (A NaN stays one.)
#define CK_LEAST -128.f
static __device__ __forceinline__ float ck_log_decay(float x) { return x < CK_LEAST ? CK_LEAST : x; }
static __device__ __forceinline__ float ck_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// What a chunk of a head leaves for the scan (floats; d a multiple of 16, so every part is 16-byte aligned)
struct ck_layout {
    int d;
    __host__ __device__ int rows1() const { return 0; }              // [16][d] the rows that meet the state for the output: r / q times exp(c)
    __host__ __device__ int rows2() const { return CK_Q * d; }       // [16][d] delta rule: k times exp(c)
    __host__ __device__ int keys() const { return 2 * CK_Q * d; }    // [d][16] k times exp(c_end - c), a channel's tokens together
    __host__ __device__ int decay() const { return 3 * CK_Q * d; }   // [d] exp(c_end) per channel (delta rule: [0])
    __host__ __device__ int intra() const { return 3 * CK_Q * d + d; } // [16][16] A or B
    __host__ __device__ int solve() const { return intra() + CK_Q * CK_Q; } // [16][16] delta rule: M
    __host__ __device__ int size() const { return solve() + CK_Q * CK_Q; }
};

// block (chunk, head).  dynamic LDS: doubles [16][d + 2], floats 2 x [16][d + 2], 2 x [16][16] (two channels a read; the sixteen rows of a wave's reads lie in banks of their own).  What bounds it is the
// matrix A, an exponential per channel and pair of tokens and the LDS reads for it: the 120 pairs stand in 120 threads for each half of the channels (all 256 pairs in a thread each: the half
// above the diagonal waits; 2047 tokens, 16 heads of 128: 55 us, 40 now).
template <bool GLA>
__global__ __launch_bounds__(256) void chunk_decay_prep_kernel(const float *r, const float *k, const float *z, long long ld, long long ldz, const float *bonus, int d, float qscale,
                                                               float inv_tau, int T, float *scratch) {
    extern __shared__ double ck_lds[];
    const int ldr = d + 2, tid = threadIdx.x, h = blockIdx.y, H = gridDim.y, t0 = blockIdx.x * CK_Q, nt = min(CK_Q, T - t0);
    double *cs = ck_lds;
    float *rs = (float *)(cs + CK_Q * ldr), *ks = rs + CK_Q * ldr, *parts = ks + CK_Q * ldr;
    const ck_layout at{d};
    float *out = scratch + ((long long)blockIdx.x * H + h) * at.size();
    const long long hb = (long long)h * d;
    parts[tid] = parts[CK_Q * CK_Q + tid] = 0.f;
    for (int i = tid; i < d; i += 256) { // running log decays (tokens that are not there: k = r = 0 and no decay)
        float zv[CK_Q];
#pragma unroll
        for (int t = 0; t < CK_Q; t++) zv[t] = z[(long long)(t0 + min(t, nt - 1)) * ldz + hb + i];
        double c = 0.0;
#pragma unroll
        for (int t = 0; t < CK_Q; t++) {
            if (t < nt) c += (double)ck_log_decay(GLA ? -ck_softplus(-zv[t]) * inv_tau : -expf(zv[t]));
            cs[t * ldr + i] = c;
        }
        out[at.decay() + i] = expf((float)c);
    }
    __syncthreads();
    for (int x = tid; x < 2 * d; x += 256) { // a channel's eight tokens
        const int i = x < d ? x : x - d, t8 = x < d ? 0 : 8;
        float rv[8], kv[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const long long row = (long long)(t0 + min(t8 + u, nt - 1)) * ld + hb + i;
            rv[u] = r[row];
            kv[u] = k[row];
        }
        const double cend = cs[(CK_Q - 1) * ldr + i];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int t = t8 + u;
            const bool in = t < nt;
            const double after = cs[t * ldr + i], before = t ? cs[(t ? t - 1 : 0) * ldr + i] : 0.0;
            rv[u] = in ? (GLA ? rv[u] * qscale : rv[u]) : 0.f;
            kv[u] = in ? kv[u] : 0.f;
            rs[t * ldr + i] = rv[u];
            ks[t * ldr + i] = kv[u];
            out[at.rows1() + t * d + i] = rv[u] * la_exp((float)(GLA ? after : before));
            kv[u] *= la_exp((float)(cend - after));
        }
        *(ck_f4 *)(out + at.keys() + i * CK_Q + t8) = ck_f4{kv[0], kv[1], kv[2], kv[3]};
        *(ck_f4 *)(out + at.keys() + i * CK_Q + t8 + 4) = ck_f4{kv[4], kv[5], kv[6], kv[7]};
    }
    __syncthreads();
    const int half = tid >> 7, pair = tid & 127;
    if (pair < 120) { // tokens s < t, t (t - 1) / 2 pairs in front of a t's first
        int t = (int)((1.f + sqrtf(1.f + 8.f * (float)pair)) * 0.5f);
        t -= t * (t - 1) / 2 > pair;
        t += t * (t + 1) / 2 <= pair;
        const int s = pair - t * (t - 1) / 2;
        const double *ct = cs + (GLA ? t : t - 1) * ldr, *cp = cs + s * ldr;
        const float *rt = rs + t * ldr, *kp = ks + s * ldr;
        ck_f2 a = {0.f, 0.f};
        const int to = (half + 1) * (d / 2);
#pragma unroll 4
        for (int i = half * (d / 2); i < to; i += 2) {
            const ck_d2 x = *(const ck_d2 *)(ct + i), y = *(const ck_d2 *)(cp + i);
            const ck_f2 u = *(const ck_f2 *)(rt + i), w = *(const ck_f2 *)(kp + i);
#pragma unroll
            for (int e = 0; e < 2; e++) a[e] = fmaf(u[e] * w[e], la_exp((float)(x[e] - y[e])), a[e]);
        }
        parts[half * CK_Q * CK_Q + t * CK_Q + s] = a[0] + a[1];
    } else { // the diagonal, eight tokens for each half of the threads
        const int t = half * 8 + pair - 120;
        const float *rt = rs + t * ldr, *kp = ks + t * ldr;
        float a = 0.f;
#pragma unroll 4
        for (int i = 0; i < d; i++) a = fmaf(GLA ? rt[i] : rt[i] * bonus[hb + i], kp[i], a);
        parts[t * CK_Q + t] = a;
    }
    __syncthreads();
    out[at.intra() + tid] = parts[tid] + parts[CK_Q * CK_Q + tid];
}

// block (chunk, head).  dynamic LDS: floats 2 x [16][d + 4], 16 x 17 doubles in front
__global__ __launch_bounds__(256) void chunk_delta_prep_kernel(const float *q, const float *k, const float *braw, const float *araw, long long ld, long long ldb, const float *a_log,
                                                               const float *dt_bias, int KH, int d, int T, float *scratch) {
    extern __shared__ double ck_lds[];
    __shared__ double cs[CK_Q];
    __shared__ float beta[CK_Q];
    const int ldr = d + 4, tid = threadIdx.x, h = blockIdx.y, H = gridDim.y, t0 = blockIdx.x * CK_Q, nt = min(CK_Q, T - t0), t = tid >> 4, s = tid & 15;
    double *L = ck_lds; // [16][17]
    float *qs = (float *)(L + CK_Q * 17), *ks = qs + CK_Q * ldr;
    const ck_layout at{d};
    float *out = scratch + ((long long)blockIdx.x * H + h) * at.size();
    const long long qb = (long long)(h / (H / KH)) * d, row = t0 + min(t, nt - 1);
    if (tid < CK_Q) { // running log decays and write strengths (tokens that are not there: no decay, nothing written)
        const bool in = tid < nt;
        const long long rr = t0 + min(tid, nt - 1);
        double c = in ? (double)ck_log_decay(-expf(a_log[h]) * ck_softplus(araw[rr * ldb + h] + dt_bias[h])) : 0.0;
#pragma unroll
        for (int o = 1; o < CK_Q; o <<= 1) {
            const double u = __shfl_up(c, o, 64);
            if (tid >= o) c += u;
        }
        cs[tid] = c;
        beta[tid] = in ? 1.f / (1.f + expf(-braw[rr * ldb + h])) : 0.f;
    }
    // unit vectors: sixteen lanes per token
    float a = 0.f, b = 0.f;
    for (int i = s; i < d; i += CK_Q) {
        const float x = t < nt ? q[row * ld + qb + i] : 0.f, y = t < nt ? k[row * ld + qb + i] : 0.f;
        qs[t * ldr + i] = x;
        ks[t * ldr + i] = y;
        a = fmaf(x, x, a);
        b = fmaf(y, y, b);
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) { a += __shfl_xor(a, o, 64); b += __shfl_xor(b, o, 64); }
    const float iq = 1.f / sqrtf((float)d) / sqrtf(a + 1e-6f), ik = 1.f / sqrtf(b + 1e-6f);
    __syncthreads();
    const float et = expf((float)cs[t]);
    for (int i = s; i < d; i += CK_Q) {
        const float x = qs[t * ldr + i] * iq, y = ks[t * ldr + i] * ik;
        qs[t * ldr + i] = x;
        ks[t * ldr + i] = y;
        out[at.rows1() + t * d + i] = x * et;
        out[at.rows2() + t * d + i] = y * et;
    }
    __syncthreads();
    const double cend = cs[CK_Q - 1];
    for (int i = tid; i < d; i += 256) {
        float kt[CK_Q];
#pragma unroll
        for (int u = 0; u < CK_Q; u++) kt[u] = ks[u * ldr + i] * expf((float)(cend - cs[u]));
#pragma unroll
        for (int u = 0; u < CK_Q; u += 4) *(ck_f4 *)(out + at.keys() + i * CK_Q + u) = ck_f4{kt[u], kt[u + 1], kt[u + 2], kt[u + 3]};
    }
    float kk = 0.f, qk = 0.f;
    for (int i = 0; i < d; i += 4) { // (rows of d + 4 floats: the sixteen s of a wave meet every bank twice at most)
        const ck_f4 kt = *(const ck_f4 *)(ks + t * ldr + i), qt = *(const ck_f4 *)(qs + t * ldr + i), kp = *(const ck_f4 *)(ks + s * ldr + i);
#pragma unroll
        for (int e = 0; e < 4; e++) { kk = fmaf(kt[e], kp[e], kk); qk = fmaf(qt[e], kp[e], qk); }
    }
    const float ed = s <= t ? expf((float)(cs[t] - cs[s])) : 0.f;
    out[at.intra() + tid] = ed * qk;
    L[t * 17 + s] = s < t ? (double)(beta[t] * ed * kk) : 0.0;
    if (tid == 0) out[at.decay()] = expf((float)cend);
    __syncthreads();
    if (tid < CK_Q) { // column tid of (I + L)^-1, times beta of its token
        double x[CK_Q];
#pragma unroll
        for (int u = 0; u < CK_Q; u++) {
            double y = u == tid ? 1.0 : 0.0;
#pragma unroll
            for (int w = 0; w < u; w++) y -= L[u * 17 + w] * x[w];
            x[u] = y;
            out[at.solve() + u * CK_Q + tid] = (float)(y * (double)beta[tid]);
        }
    }
}

// block (16 value columns, head), wave w of the first four keeps the state's row tiles w, w + 4, ... (16 rows each, NT of them) in accumulators: lane (column l % 16, quarter l / 16) holds rows
// 4 (l / 16) + i, which is also what the next product's column operand asks of it when k is taken in that order -- the state never leaves its registers.  A wave's part of the
// products with the state meets the others' in LDS (two buffers, one barrier per chunk); the fifth wave adds them, makes the chunk's outputs and stores them, beside the others' next chunk.
// What bounds it is the chain of a chunk, 16 matrix instructions per state wave (NT 2; delta rule 28, those with q where the wave would wait for the others): 0.55 and 0.9 us a chunk, in proportion to
// them, with eight state waves of half the tiles too (0.54 and 1.06: each makes u).  A chunk's operands are requested CK_AHEAD chunks ahead, at addresses that are a scalar and a constant per
// lane; FULL (d = 64 NT, whole column blocks): no branch between the requests, so a wait counts them and none drains the queue, as each did before.
template <int NT, bool DELTA, bool FULL>
__global__ __launch_bounds__(320) void chunk_scan_kernel(const ps_seq_step *step, long long state_off, const float *scratch, const float *v, long long ld, int d, int dv, int T, float *o,
                                                         long long ldo) {
    __shared__ ck_f4 part[2][DELTA ? 2 : 1][4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lq = lane >> 4, H = gridDim.y, tiles = FULL ? 4 * NT : d / 16;
    const int chunks = (T + CK_Q - 1) / CK_Q, last = chunks - 1;
    int h = blockIdx.y, block = blockIdx.x;
    if (H % 8 == 0) { // a head's column blocks, which read the same operands, on one XCD (work-groups go to the eight in turn)
        const int id = blockIdx.x + gridDim.x * blockIdx.y;
        h = id % 8 + 8 * (id / 8 / (int)gridDim.x);
        block = id / 8 % (int)gridDim.x;
    }
    const int col = block * 16 + lr, colc = FULL ? col : min(col, dv - 1);
    const ck_layout at{d};
    const char *ph = (const char *)(scratch + (long long)h * at.size()), *vh = (const char *)(v + (long long)h * dv);
    const long long per = (long long)H * at.size() * 4;
    struct operands { ck_f4 q[NT], k[DELTA ? NT : 1], kt[NT], dec[DELTA ? 1 : NT], in, m; float v[4]; };
    unsigned at_v[4], at_end[4]; // bytes from a chunk's first row to the lane's four, in a whole chunk and in the last one (rows that are not there repeat the last one: nothing is made of them)
#pragma unroll
    for (int i = 0; i < 4; i++) {
        at_v[i] = (unsigned)(((long long)(4 * lq + i) * ld + colc) * 4);
        at_end[i] = (unsigned)(((long long)min(4 * lq + i, T - 1 - last * CK_Q) * ld + colc) * 4);
    }
    auto fetch_v = [&](int c, operands &a) { // (c: at most the last)
        const char *p = vh + (long long)c * CK_Q * ld * 4;
#pragma unroll
        for (int i = 0; i < 4; i++) a.v[i] = *(const float *)(p + (c < last ? at_v[i] : at_end[i]));
    };
    const unsigned at_m = (unsigned)(at.solve() + lr * CK_Q + 4 * lq) * 4, at_in = (unsigned)(at.intra() + lr * CK_Q + 4 * lq) * 4;
    if (wave == 4) {
        auto fetch = [&](int c, operands &a) {
            c = min(c, last);
            const char *p = ph + c * per;
            if constexpr (DELTA) a.m = *(const ck_f4 *)(p + at_m);
            a.in = *(const ck_f4 *)(p + at_in);
            fetch_v(c, a);
        };
        ck_f4 held_in, held_u; // the delta rule's products with q are there one barrier later
        auto finish = [&](auto whole, int c, const ck_f4 &in, const ck_f4 &u) {
            const int buf = c & 1;
            ck_f4 y = (part[buf][0][0][lane] + part[buf][0][1][lane]) + (part[buf][0][2][lane] + part[buf][0][3][lane]);
#pragma unroll
            for (int i = 0; i < 4; i++) y = __builtin_amdgcn_mfma_f32_16x16x4f32(in[i], u[i], y, 0, 0, 0);
            float *oh = o + (long long)(c * CK_Q + 4 * lq) * ldo + (long long)h * dv + col;
            if constexpr (whole.value) {
#pragma unroll
                for (int i = 0; i < 4; i++) oh[i * ldo] = y[i];
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (c * CK_Q + 4 * lq + i < T && col < dv) oh[i * ldo] = y[i];
            }
        };
        auto chunk = [&](auto whole, int c, const operands &b, operands &later) {
            fetch(c + CK_AHEAD, later);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            ck_f4 u = {b.v[0], b.v[1], b.v[2], b.v[3]};
            if constexpr (DELTA) {
                const int buf = c & 1;
                const ck_f4 w = (part[buf][1][0][lane] + part[buf][1][1][lane]) + (part[buf][1][2][lane] + part[buf][1][3][lane]);
                u = ck_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 4; i++) u = __builtin_amdgcn_mfma_f32_16x16x4f32(b.m[i], b.v[i] - w[i], u, 0, 0, 0);
                if (c) finish(std::integral_constant<bool, FULL>(), c - 1, held_in, held_u); // (not the last chunk: all its rows are there)
                held_in = b.in;
                held_u = u;
            } else finish(whole, c, b.in, u);
        };
        operands a[CK_AHEAD + 1];
#pragma unroll
        for (int i = 0; i < CK_AHEAD; i++) fetch(i, a[i]);
        int c = 0;
        for (; FULL && c + CK_AHEAD < T / CK_Q; c += CK_AHEAD + 1) {
#pragma unroll
            for (int i = 0; i <= CK_AHEAD; i++) chunk(std::true_type(), c + i, a[i], a[(i + CK_AHEAD) % (CK_AHEAD + 1)]);
        }
        for (; c < chunks; c += CK_AHEAD + 1) {
#pragma unroll
            for (int i = 0; i <= CK_AHEAD; i++)
                if (c + i < chunks) chunk(std::false_type(), c + i, a[i], a[(i + CK_AHEAD) % (CK_AHEAD + 1)]); // (uniform)
        }
        if constexpr (DELTA) {
            __syncthreads();
            finish(std::false_type(), last, held_in, held_u);
        }
        return;
    }
    float *S0 = step->state + state_off + (long long)h * d * dv;
    ck_f4 S[NT];
    unsigned at_q[NT], at_kt[NT], at_dec[NT]; // (a tile that is not there repeats the last one; its rows of the state are zero and not stored)
#pragma unroll
    for (int x = 0; x < NT; x++) {
        const int tile = wave + 4 * x, row = 16 * min(tile, tiles - 1);
        at_q[x] = (unsigned)(lr * d + row + 4 * lq) * 4;
        at_kt[x] = (unsigned)(at.keys() + (row + lr) * CK_Q + 4 * lq) * 4;
        at_dec[x] = (unsigned)(at.decay() + row + 4 * lq) * 4;
#pragma unroll
        for (int i = 0; i < 4; i++) S[x][i] = FULL || (tile < tiles && col < dv) ? S0[(long long)(16 * tile + 4 * lq + i) * dv + col] : 0.f;
    }
    auto fetch = [&](int c, operands &a) {
        c = min(c, last);
        const char *p = ph + c * per;
#pragma unroll
        for (int x = 0; x < NT; x++) {
            if constexpr (DELTA) a.k[x] = *(const ck_f4 *)(p + at.rows2() * 4 + at_q[x]);
            a.q[x] = *(const ck_f4 *)(p + at.rows1() * 4 + at_q[x]);
            a.kt[x] = *(const ck_f4 *)(p + at_kt[x]);
            if constexpr (!DELTA) a.dec[x] = *(const ck_f4 *)(p + at_dec[x]);
        }
        if constexpr (DELTA) {
            const float g = *(const float *)(p + at.decay() * 4);
            a.dec[0] = ck_f4{g, g, g, g};
            a.m = *(const ck_f4 *)(p + at_m);
        }
        fetch_v(c, a);
    };
    auto chunk = [&](int c, const operands &b, operands &later) {
        const int buf = c & 1;
        ck_f4 oq = {0.f, 0.f, 0.f, 0.f}, ok = {0.f, 0.f, 0.f, 0.f};
        auto with_q = [&](int from, int to) {
#pragma unroll
            for (int x = from; x < to; x++)
                if (FULL || wave + 4 * x < tiles) { // (uniform per wave)
#pragma unroll
                    for (int i = 0; i < 4; i++) oq = __builtin_amdgcn_mfma_f32_16x16x4f32(b.q[x][i], S[x][i], oq, 0, 0, 0);
                }
        };
        fetch(c + CK_AHEAD, later);
        ck_f4 u = {b.v[0], b.v[1], b.v[2], b.v[3]}; // what the chunk's tokens write
        if constexpr (DELTA) {
#pragma unroll
            for (int x = 0; x < NT; x++)
                if (FULL || wave + 4 * x < tiles) {
#pragma unroll
                    for (int i = 0; i < 4; i++) ok = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[x][i], S[x][i], ok, 0, 0, 0);
                }
            part[buf][1][wave][lane] = ok;
            __builtin_amdgcn_sched_barrier(0);
            with_q(0, NT / 2); // (the products with q where the others' parts are waited for)
            __syncthreads();
            const ck_f4 p0 = part[buf][1][0][lane], p1 = part[buf][1][1][lane], p2 = part[buf][1][2][lane], p3 = part[buf][1][3][lane];
            __builtin_amdgcn_sched_barrier(0);
            with_q(NT / 2, NT);
            const ck_f4 w = (p0 + p1) + (p2 + p3);
            u = ck_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; i++) u = __builtin_amdgcn_mfma_f32_16x16x4f32(b.m[i], b.v[i] - w[i], u, 0, 0, 0);
        } else with_q(0, NT);
        part[buf][0][wave][lane] = oq;
        __builtin_amdgcn_sched_barrier(0); // (the requests have gone out here)
#pragma unroll
        for (int x = 0; x < NT; x++)
            if (FULL || wave + 4 * x < tiles) {
#pragma unroll
                for (int i = 0; i < 4; i++) S[x][i] *= b.dec[DELTA ? 0 : x][i];
            }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int x = 0; x < NT; x++)
                if (FULL || wave + 4 * x < tiles) S[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.kt[x][i], u[i], S[x], 0, 0, 0);
        if constexpr (!DELTA) __syncthreads();
    };
    operands a[CK_AHEAD + 1];
#pragma unroll
    for (int i = 0; i < CK_AHEAD; i++) fetch(i, a[i]);
#pragma unroll
    for (int x = 0; x < NT; x++) asm volatile("" : "+v"(S[x])); // (there before the loop: a wait for them inside would wait for everything, each time around)
    int c = 0;
    for (; c + CK_AHEAD < chunks; c += CK_AHEAD + 1) {
#pragma unroll
        for (int i = 0; i <= CK_AHEAD; i++) chunk(c + i, a[i], a[(i + CK_AHEAD) % (CK_AHEAD + 1)]);
    }
#pragma unroll
    for (int i = 0; i < CK_AHEAD; i++)
        if (c + i < chunks) chunk(c + i, a[i], a[(i + CK_AHEAD) % (CK_AHEAD + 1)]); // (uniform)
    if constexpr (DELTA) __syncthreads();
#pragma unroll
    for (int x = 0; x < NT; x++)
        if (FULL || (wave + 4 * x < tiles && col < dv)) {
#pragma unroll
            for (int i = 0; i < 4; i++) S0[(long long)(16 * (wave + 4 * x) + 4 * lq + i) * dv + col] = S[x][i];
        }
}

bool psk_chunked_ok(int d) { return d % 16 == 0 && d <= 256; }
size_t psk_chunked_scratch(int H, int d, int T) { return (size_t)((T + CK_Q - 1) / CK_Q) * H * ck_layout{d}.size() * 4; }

template <bool DELTA>
static void ck_scan(hipStream_t st, const ps_seq_step *step, int64_t state_off, const float *scratch, const float *v, int64_t ld, int H, int d, int dv, int T, float *o, int64_t ldo) {
    const auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((dv + 15) / 16, H), dim3(320), 0, st, step, (long long)state_off, scratch, v, (long long)ld, d, dv, T, o, (long long)ldo); };
    const int nt = (d + 63) / 64;
    if (d % 64 == 0 && dv % 16 == 0) launch(nt == 1 ? chunk_scan_kernel<1, DELTA, true> : nt == 2 ? chunk_scan_kernel<2, DELTA, true> : nt == 3 ? chunk_scan_kernel<3, DELTA, true> : chunk_scan_kernel<4, DELTA, true>);
    else launch(nt == 1 ? chunk_scan_kernel<1, DELTA, false> : nt == 2 ? chunk_scan_kernel<2, DELTA, false> : nt == 3 ? chunk_scan_kernel<3, DELTA, false> : chunk_scan_kernel<4, DELTA, false>);
}
template <bool GLA>
static void ck_decay(hipStream_t st, const ps_seq_step *step, int64_t state_off, const float *r, const float *k, const float *v, int64_t ld, const float *z, int64_t ldz, const float *bonus,
                     float qscale, float inv_tau, int H, int d, int dv, int T, float *scratch, float *o, int64_t ldo) {
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)chunk_decay_prep_kernel<GLA>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    hipLaunchKernelGGL(chunk_decay_prep_kernel<GLA>, dim3((T + CK_Q - 1) / CK_Q, H), dim3(256), (size_t)CK_Q * (d + 2) * 16 + 2 * CK_Q * CK_Q * 4, st, r, k, z, (long long)ld, (long long)ldz, bonus, d, qscale,
                       inv_tau, T, scratch);
    ck_scan<false>(st, step, state_off, scratch, v, ld, H, d, dv, T, o, ldo);
}
void psk_wkv_chunked(hipStream_t st, const ps_seq_step *step, int64_t state_off, const float *r, const float *k, const float *v, const float *z, int64_t ld, const float *bonus, int H, int d,
                     int T, float *scratch, float *o, int64_t ldo) {
    ck_decay<false>(st, step, state_off, r, k, v, ld, z, ld, bonus, 1.f, 1.f, H, d, d, T, scratch, o, ldo);
}
void psk_gla_chunked(hipStream_t st, const ps_seq_step *step, int64_t state_off, const float *q, const float *k, const float *v, int64_t ld, const float *z, int64_t ldz, float tau, int H,
                     int d, int dv, int T, float *scratch, float *o, int64_t ldo) {
    ck_decay<true>(st, step, state_off, q, k, v, ld, z, ldz, nullptr, 1.f / sqrtf((float)d), 1.f / tau, H, d, dv, T, scratch, o, ldo);
}
void psk_delta_chunked(hipStream_t st, const ps_seq_step *step, int64_t state_off, const float *q, const float *k, const float *v, const float *braw, const float *araw, int64_t ld, int64_t ldb,
                       const float *a_log, const float *dt_bias, int H, int KH, int d, int dv, int T, float *scratch, float *o, int64_t ldo) {
    hipLaunchKernelGGL(chunk_delta_prep_kernel, dim3((T + CK_Q - 1) / CK_Q, H), dim3(256), (size_t)CK_Q * 17 * 8 + (size_t)2 * CK_Q * (d + 4) * 4, st, q, k, braw, araw, (long long)ld,
                       (long long)ldb, a_log, dt_bias, KH, d, T, scratch);
    ck_scan<true>(st, step, state_off, scratch, v, ld, H, d, dv, T, o, ldo);
}
