// Dense (unquantized) matrices of the layer-list models: bfloat16 operands with fp32 accumulation on v_mfma_f32_16x16x32_bf16, or
// fp32 throughout on v_mfma_f32_16x16x4_f32 (one rounding per product, fp32 adds: a true fp32 product, no reduced-precision mode), or on the bf16 instruction with the operand as three bf16 lines
// and the weights as they came (dn_ring_take, PL 3: no product is rounded at all).
//   dense_mm_kernel<WT>   tiled mat-mul, 64 tokens x 64 outputs per work-group of four waves, any T / N / K (edges zero-filled)
//   dense_mm_ring_kernel  rows of K in whole 128-byte blocks, more than one token (fp32: two to four by dn_few_first): tiles of 64 x 64 to 192 x 128 over an operand packed by dense_pack_kernel (fp32: in place where its rows
//                         are plain), split along K where the tiles do not fill the chip (dense_mm_sum_kernel adds the parts)
//   dense_mm_big_kernel   the same operands, bf16, tiles of 128, 192 or 256 rows x 256 columns where they are the faster ones (dn_ring_plan)
//   dense_mm_few_kernel   K up to 32, more than 8 tokens: a thread per output column
//   dense_mm_narrow_kernel bf16, K a multiple of 128 up to 1024, more than one token, few tiles: 32 x 32 tiles, the waves share K
//   dense_mv1_kernel<WT,FORM,RAGGED> a single token, or a few tokens' experts' first product: every wave streams its rows, the requests run ahead of everything else
//   dense_mv2_kernel<WT,U,RAGGED> the second product of a few tokens' experts: the waves of a work-group share a row, the activations in registers
//   dense_mv_kernel<WT,C,RW> a few tokens (C <= 8 columns) of a K the ring does not take, and of fp32 where it is the faster one (dn_few_first): the activation rows live in LDS, a wave streams RW weight rows at a time
// All take the same operand description (ps_seq.h psk_dense_args): ring rows, the token-shift mix and the epilogue
// (bias, activation, scale, a factor from a second table) are part of the launch, so no mixer needs a kernel of its own around its projections.
#include "ps_seq.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

typedef float dn_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 dn_bf8 __attribute__((ext_vector_type(8)));
typedef unsigned short dn_us8 __attribute__((ext_vector_type(8)));
typedef unsigned short dn_us4 __attribute__((ext_vector_type(4)));

static __device__ __forceinline__ unsigned short dn_f2bf(float f) { return __builtin_bit_cast(unsigned short, (__bf16)f); } // round to nearest even (v_cvt_pk_bf16_f32)
static __device__ __forceinline__ float dn_bf2f(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

struct dn_args {
    const void *w;
    const float *a;
    long long lda, a_row0, a_mod;
    const ps_seq_step *a_step;
    int T;
    long long N, K;
    float *out;
    unsigned short *out16; // given: the result rounded to bf16 there instead, in out's arrangement (wide mat-mul)
    long long ldo;
    const float *bias;
    int act;
    float act_p, act_q, alpha;
    const float *mu, *shift0;
    int accum;
    const float *out_scale;
    // grouped products (ps_seq.h): N is one matrix's rows, wstride the elements between matrices
    int groups, g_adiv, g_odiv, g_inner;
    const int32_t *g_sel, *g_seg, *g_list;
    const float *g_scale;
    long long wstride;
    const float *g_ident, *g_ident_w; // grouped mat-vec: a slot without a matrix adds g_ident_w[slot] * g_ident[row][n] to output n
    long long g_ident_ld;
    const void *em_table; // a factor per output from the token's row of a second table (psk_dense_args)
    int em_bf16;
    long long em_ld, em_col;
    const int32_t *em_tokens;
    const ps_seq_step *em_step;
};

// rows of A that exist and where they start (ring rows relative to the step's position)
static __device__ __forceinline__ void dn_rows(const dn_args &g, long long &row0, int &T) {
    row0 = g.a_row0;
    T = g.T;
    if (g.g_seg) { // the slots of matrix blockIdx.z: entries row0 .. row0 + T - 1 of the sorted list
        row0 = g.g_seg[blockIdx.z];
        T = g.g_seg[blockIdx.z + 1] - (int)row0;
        return;
    }
    if (g.a_step) {
        const long long p = g.a_step->pos0 + g.a_row0;
        row0 = p > 0 ? p : 0;
        const long long have = g.a_step->pos0 + g.a_step->n - row0;
        if (have < T) T = (int)have;
    }
}
static __device__ __forceinline__ const float *dn_arow(const dn_args &g, long long row0, int t) {
    long long r = row0 + t;
    if (g.g_list) r = g.g_list[r] / g.g_adiv;
    if (g.a_mod > 0) r %= g.a_mod;
    return g.a + r * g.lda;
}
static __device__ __forceinline__ float dn_aval(const dn_args &g, long long row0, int t, long long k) {
    if (g.g_list) return dn_arow(g, row0, t)[k] * (g.g_scale ? g.g_scale[g.g_list[row0 + t]] : 1.f);
    const float x = dn_arow(g, row0, t)[k];
    if (!g.mu) return x;
    const float p = t ? dn_arow(g, row0, t - 1)[k] : g.shift0[k];
    return x + (p - x) * g.mu[k];
}
static __device__ __forceinline__ float dn_epi(const dn_args &g, float acc, long long n) {
    if (g.bias) acc += g.bias[n];
    if (g.act == PSD_ACT_XIELU) {
        if (acc > 0.f) acc = g.act_p * acc * acc + 0.5f * acc;
        else acc = g.act_q * (expm1f(acc) - acc) + 0.5f * acc;
    } else if (g.act == PSD_ACT_TANH) {
        acc = tanhf(acc);
    } else if (g.act == PSD_ACT_RELU2) {
        acc = acc > 0.f ? acc * acc : 0.f;
    } else if (g.act == PSD_ACT_SOFTCAP) {
        acc = g.act_p * tanhf(acc / g.act_p);
    } else if (g.act == PSD_ACT_GELU_TANH) {
        acc = 0.5f * acc * (1.f + tanhf(0.7978845608028654f * (acc + 0.044715f * acc * acc * acc)));
    }
    return acc * g.alpha;
}
// xIELU of a wide product's results without a branch (expm1f and its rarer cases stood behind 2047 x 8192 x 2048 with half as many clocks as the product: 89 us, so 67).  Below zero, with
// x = r + n ln 2, |r| <= (ln 2) / 2, s = 2^n: expm1(x) - x = s (expm1(r) - r) + (s - 1) r + (s - 1 - n ln 2), so next to zero nothing cancels, as it does in expm1f(x) - x; (expm1(r) - r) / r^2
// by a polynomial fitted to it for the least greatest error, 3e-9.  (One constant for ln 2 in r and beside it: what it lacks drops out but for s.)
// Error against 64 bits over 2.6 million x from -2^-20 to -90, relative to the larger summand: rms 2.8e-8, at most 1.9e-7 (with expm1f 6.3e-8 and 2.0e-7).
static __device__ __forceinline__ float dn_xielu(float x, float p, float q) {
    const float c = fmaxf(x, -64.f), m = fmaf(c, 1.44269504f, 12583039.f), n = m - 12583039.f; // (1.5 x 2^23 and 127: n to the nearest, and below it in m as an exponent; c - x: what lies beyond, and a NaN)
    const float r = fmaf(-n, 0.693147181f, c), s = __uint_as_float(__float_as_uint(m) << 23), t = s - 1.f;
    float y = fmaf(1.98578170966e-4f, r, 1.39336404391e-3f);
    y = fmaf(y, r, 8.33336077631e-3f);
    y = fmaf(y, r, 4.16664667428e-2f);
    y = fmaf(y, r, 1.66666671634e-1f);
    y = fmaf(y, r, 0.5f);
    const float below = fmaf(s, y * (r * r), fmaf(t, r, fmaf(-n, 0.693147181f, t))) + (c - x);
    return fmaf(x > 0.f ? p * x : q, x > 0.f ? x : below, 0.5f * x);
}
static __device__ __forceinline__ float dn_relu2(const dn_args &g, float x) { return g.act == PSD_ACT_RELU2 ? (x > 0.f ? x * x : 0.f) : x; }
static __device__ __forceinline__ float dn_silu(float x) { return x / (1.f + expf(-x)); }
// Result acc of (token t, weight row n) goes to its place.  other: the result of row n ^ 1 (the paired activation needs both; every lane of the wave calls
// this with both values, only the even row stores).  O16: the wide mat-mul's, whose result may go to g.out16 (the test of it for each of a few tokens' results, beside its arguments, cost the
// mat-vec of eight tokens 3 to 6 %)
static __device__ __forceinline__ float dn_row_scale(const dn_args &g, long long t) { // of output row t (wide mat-mul)
    return g.out_scale ? g.out_scale[g.g_list && g.out16 ? g.g_list[t] / g.g_odiv : t] : 1.f;
}
template <bool O16 = false>
static __device__ __forceinline__ void dn_put(const dn_args &g, long long t, long long n, float acc, float other, bool in) {
    const float rs = !in ? 1.f : O16 ? dn_row_scale(g, t) : g.out_scale ? g.out_scale[t] : 1.f;
    if (g.act == PSD_ACT_SILU_PAIR || g.act == PSD_ACT_RELU_PAIR) {
        if (in && !(n & 1)) {
            float *p = g.out + t * g.ldo + (n >> 1);
            if (g.bias) { acc += g.bias[n]; other += g.bias[n + 1]; }
            const float v = (g.act == PSD_ACT_SILU_PAIR ? dn_silu(acc) : fmaxf(acc, 0.f)) * other * g.alpha * rs;
            if (O16 && g.out16) g.out16[p - g.out] = dn_f2bf(v);
            else *p = g.accum ? *p + v : v;
        }
        return;
    }
    if (!in) return;
    float *p = g.out + t * g.ldo + n;
    float v = dn_epi(g, acc, n) * rs;
    if (g.em_table) {
        const long long at = (long long)(g.em_tokens ? g.em_tokens[t] : g.em_step->token0) * g.em_ld + g.em_col + n;
        v *= g.em_bf16 ? dn_bf2f(((const unsigned short *)g.em_table)[at]) : ((const float *)g.em_table)[at];
    }
    if (O16 && g.out16) g.out16[p - g.out] = dn_f2bf(v);
    else *p = g.accum ? *p + v : v;
}
// the output row of local row t (t < T): itself, or where the sorted list sends its slot
static __device__ __forceinline__ long long dn_orow(const dn_args &g, long long row0, int t, int T) {
    if (!g.g_list) return t;
    return t < T ? g.out16 ? row0 + t : g.g_list[row0 + t] / g.g_odiv : 0; // (rounded rows of slots: in the list's order, as the next product takes them)
}

// ---------------------------------------------------------------------------------------------------- tiled mat-mul
template <typename WT> struct dn_tile;
template <> struct dn_tile<unsigned short> { static constexpr int BK = 32, LD = 40; typedef unsigned short S; }; // LDS rows padded to 80 B
template <> struct dn_tile<float> { static constexpr int BK = 16, LD = 20; typedef float S; };

template <typename WT>
__global__ __launch_bounds__(256) void dense_mm_kernel(dn_args g) {
    constexpr int BK = dn_tile<WT>::BK, LD = dn_tile<WT>::LD;
    typedef typename dn_tile<WT>::S S;
    __shared__ __attribute__((aligned(16))) S As[64 * LD];
    __shared__ __attribute__((aligned(16))) S Bs[64 * LD];
    long long row0;
    int T;
    dn_rows(g, row0, T);
    const int t0 = blockIdx.y * 64;
    if (t0 >= T) return; // (uniform per work-group: no barrier is skipped by part of it)
    const long long n0 = (long long)blockIdx.x * 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 15, lq = lane >> 4;
    const WT *W = (const WT *)g.w + (g.g_seg ? (long long)blockIdx.z * g.wstride : 0);
    dn_f4 acc[2][2];
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++) acc[i][j] = dn_f4{0.f, 0.f, 0.f, 0.f};
    constexpr int PER = 64 * BK / 256; // elements of each tile a thread stages: 8 (bf16) or 4 (fp32)
    const int srow = tid / (BK / PER), sk = (tid % (BK / PER)) * PER;
    for (long long k0 = 0; k0 < g.K; k0 += BK) {
        { // A: tokens t0 .. t0+63
            const int t = t0 + srow;
            S tmp[PER];
#pragma unroll
            for (int e = 0; e < PER; e++) {
                const long long k = k0 + sk + e;
                const float v = (t < T && k < g.K) ? dn_aval(g, row0, t, k) : 0.f;
                if constexpr (sizeof(WT) == 2) tmp[e] = dn_f2bf(v);
                else tmp[e] = v;
            }
#pragma unroll
            for (int e = 0; e < PER; e++) As[srow * LD + sk + e] = tmp[e];
        }
        { // B: weight rows n0 .. n0+63
            const long long n = n0 + srow;
            const long long k = k0 + sk;
            S tmp[PER];
            if (n < g.N && k + PER <= g.K && ((g.K * (long long)sizeof(WT)) % 16 == 0)) {
                const dn_f4 raw = *(const dn_f4 *)(W + n * g.K + k); // 16 bytes: 8 bf16 or 4 floats
                __builtin_memcpy(tmp, &raw, 16);
            } else {
#pragma unroll
                for (int e = 0; e < PER; e++) tmp[e] = (n < g.N && k + e < g.K) ? W[n * g.K + k + e] : (S)0;
            }
#pragma unroll
            for (int e = 0; e < PER; e++) Bs[srow * LD + sk + e] = tmp[e];
        }
        __syncthreads();
        if constexpr (sizeof(WT) == 2) {
            dn_bf8 fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                dn_us8 ra = *(const dn_us8 *)&As[(wm * 32 + i * 16 + lr) * LD + lq * 8];
                dn_us8 rb = *(const dn_us8 *)&Bs[(wn * 32 + i * 16 + lr) * LD + lq * 8];
                __builtin_memcpy(&fa[i], &ra, 16);
                __builtin_memcpy(&fb[i], &rb, 16);
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        } else {
#pragma unroll
            for (int kk = 0; kk < BK; kk += 4) {
                float fa[2], fb[2];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    fa[i] = As[(wm * 32 + i * 16 + lr) * LD + kk + lq];
                    fb[i] = Bs[(wn * 32 + i * 16 + lr) * LD + kk + lq];
                }
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = t0 + wm * 32 + i * 16 + lq * 4 + e;
                const long long n = n0 + wn * 32 + j * 16 + lr;
                dn_put(g, dn_orow(g, row0, t, T), n, acc[i][j][e], __shfl_xor(acc[i][j][e], 1, 64), t < T && n < g.N); // (row n ^ 1 is the neighbouring lane's)
            }
}

// ---------------------------------------------------------------------------------------------------- a few tokens: mat-vec
// Dynamic LDS: C rows of K activations, as bf16-rounded fp32 values (bf16 mode: the same operand rounding as the tiled kernel) or fp32.
template <typename WT, int C, int RW> // RW rows per wave at a time
__global__ __launch_bounds__(256) void dense_mv_kernel(dn_args g) {
    extern __shared__ __attribute__((aligned(16))) float xs[]; // [C][Kp]
    long long row0;
    int T;
    dn_rows(g, row0, T);
    const long long K = g.K, Kp = (K + 7) / 8 * 8;
#pragma unroll
    for (int c = 0; c < C; c++) {
        const float *x = c < T ? dn_arow(g, row0, c) : nullptr, *p = g.mu && c < T ? (c ? dn_arow(g, row0, c - 1) : g.shift0) : nullptr;
#pragma unroll 4
        for (int k = threadIdx.x; k < (int)Kp; k += 256) {
            float v = x && k < K ? x[k] : 0.f;
            if (p && k < K) v += (p[k] - v) * g.mu[k]; // (the token-shift mix of dn_aval)
            if constexpr (sizeof(WT) == 2) v = dn_bf2f(dn_f2bf(v));
            xs[(long long)c * Kp + k] = v;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const WT *W = (const WT *)g.w;
    constexpr int VE = 16 / (int)sizeof(WT); // elements per 16-byte load
    const bool vec = (K * (long long)sizeof(WT)) % 16 == 0;
    for (long long nb = ((long long)blockIdx.x * 4 + wave) * RW; nb < g.N; nb += (long long)gridDim.x * 4 * RW) {
        float acc[RW][C];
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
            for (int c = 0; c < C; c++) acc[r][c] = 0.f;
        if (vec) {
            // two 16-byte pieces of each row in flight per lane (four rows: 8 KiB per wave and round)
            for (long long k = (long long)lane * VE; k < K; k += 128 * VE) {
                const long long k2 = k + 64 * VE;
                const bool two = k2 < K;
                dn_f4 raw[2][RW];
#pragma unroll
                for (int r = 0; r < RW; r++) {
                    const long long n = nb + r < g.N ? nb + r : g.N - 1;
                    raw[0][r] = __builtin_nontemporal_load((const dn_f4 *)(W + n * K + k));
                    raw[1][r] = two ? __builtin_nontemporal_load((const dn_f4 *)(W + n * K + k2)) : dn_f4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const long long ku = u ? (two ? k2 : k) : k; // (the second piece is zero where there is none: any valid x offset will do)
#pragma unroll
                    for (int r = 0; r < RW; r++) {
                        float wv[VE];
                        if constexpr (sizeof(WT) == 2) {
                            unsigned short h[8];
                            __builtin_memcpy(h, &raw[u][r], 16);
#pragma unroll
                            for (int e = 0; e < 8; e++) wv[e] = dn_bf2f(h[e]);
                        } else {
                            __builtin_memcpy(wv, &raw[u][r], 16);
                        }
#pragma unroll
                        for (int c = 0; c < C; c++) {
                            const float *x = xs + (long long)c * Kp + ku;
#pragma unroll
                            for (int e = 0; e < VE; e++) acc[r][c] = fmaf(wv[e], x[e], acc[r][c]);
                        }
                    }
                }
            }
        } else {
            for (long long k = lane; k < K; k += 64)
#pragma unroll
                for (int r = 0; r < RW; r++) {
                    const long long n = nb + r < g.N ? nb + r : g.N - 1;
                    float wv;
                    if constexpr (sizeof(WT) == 2) wv = dn_bf2f(((const unsigned short *)W)[n * K + k]);
                    else wv = ((const float *)W)[n * K + k];
#pragma unroll
                    for (int c = 0; c < C; c++) acc[r][c] = fmaf(wv, xs[(long long)c * Kp + k], acc[r][c]);
                }
        }
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
            for (int c = 0; c < C; c++) {
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) acc[r][c] += __shfl_xor(acc[r][c], o, 64);
            }
#pragma unroll
        for (int r = 0; r < RW; r++)
#pragma unroll
            for (int c = 0; c < C; c++) dn_put(g, c, nb + r, acc[r][c], acc[RW > 1 ? (r ^ 1) : r][c], lane == 0 && nb + r < g.N && c < T); // (nb is a multiple of four)
    }
}


// Grouped mat-vec (ps_seq.h, grouped products): block row r = one output row, which adds its g_inner slots; slot s = r g_inner + i reads A row s / g_adiv
// times g_scale[s] and the matrix g_sel[s].  Dynamic LDS: [g_inner][Kp] activations, rounded as in dense_mv_kernel.  A wave streams RW weight rows at a
// time, two 16-byte pieces of each in flight; small matrices take fewer rows per wave so that the launch still has waves for every CU.
template <typename WT, int RW>
__global__ __launch_bounds__(256) void dense_mv_grouped_kernel(dn_args g) {
    extern __shared__ __attribute__((aligned(16))) float xs[]; // [inner][Kp]
    const long long K = g.K, Kp = (K + 7) / 8 * 8;
    const int r = blockIdx.y, inner = g.g_inner;
    for (int c = 0; c < inner; c++) {
        const int s = r * inner + c;
        const float *x = g.a + (long long)(s / g.g_adiv) * g.lda, scale = g.g_scale ? g.g_scale[s] : 1.f;
#pragma unroll 4
        for (int k = threadIdx.x; k < (int)Kp; k += 256) {
            float v = k < K ? x[k] * scale : 0.f;
            if constexpr (sizeof(WT) == 2) v = dn_bf2f(dn_f2bf(v));
            xs[(long long)c * Kp + k] = v;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int VE = 16 / (int)sizeof(WT);
    const bool vec = (K * (long long)sizeof(WT)) % 16 == 0;
    for (long long nb = ((long long)blockIdx.x * 4 + wave) * RW; nb < g.N; nb += (long long)gridDim.x * 4 * RW) {
        float acc[RW];
        float ident = 0.f; // the summed weights of the row's slots that have no matrix (identity experts)
#pragma unroll
        for (int q = 0; q < RW; q++) acc[q] = 0.f;
        for (int c = 0; c < inner; c++) {
            const int sel = g.g_sel[(long long)r * inner + c];
            if (sel >= g.groups) { // (no product for this slot; the same for every lane of the block)
                if (g.g_ident) ident += g.g_ident_w[(long long)r * inner + c];
                continue;
            }
            const WT *W = (const WT *)g.w + (long long)sel * g.wstride;
            const float *x = xs + (long long)c * Kp;
            if (vec) {
                for (long long k = (long long)lane * VE; k < K; k += 128 * VE) {
                    const long long k2 = k + 64 * VE;
                    const bool two = k2 < K;
                    dn_f4 raw[2][RW];
#pragma unroll
                    for (int q = 0; q < RW; q++) {
                        const long long n = nb + q < g.N ? nb + q : g.N - 1;
                        raw[0][q] = __builtin_nontemporal_load((const dn_f4 *)(W + n * K + k));
                        raw[1][q] = two ? __builtin_nontemporal_load((const dn_f4 *)(W + n * K + k2)) : dn_f4{0.f, 0.f, 0.f, 0.f};
                    }
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        const long long ku = u ? (two ? k2 : k) : k; // (the second piece is zero where there is none: any valid x offset will do)
#pragma unroll
                        for (int q = 0; q < RW; q++) {
                            float wv[VE];
                            if constexpr (sizeof(WT) == 2) {
                                unsigned short h[8];
                                __builtin_memcpy(h, &raw[u][q], 16);
#pragma unroll
                                for (int e = 0; e < 8; e++) wv[e] = dn_bf2f(h[e]);
                            } else {
                                __builtin_memcpy(wv, &raw[u][q], 16);
                            }
#pragma unroll
                            for (int e = 0; e < VE; e++) acc[q] = fmaf(wv[e], x[ku + e], acc[q]);
                        }
                    }
                }
            } else {
                for (long long k = lane; k < K; k += 64)
#pragma unroll
                    for (int q = 0; q < RW; q++) {
                        const long long n = nb + q < g.N ? nb + q : g.N - 1;
                        float wv;
                        if constexpr (sizeof(WT) == 2) wv = dn_bf2f(((const unsigned short *)W)[n * K + k]);
                        else wv = ((const float *)W)[n * K + k];
                        acc[q] = fmaf(wv, x[k], acc[q]);
                    }
            }
        }
#pragma unroll
        for (int q = 0; q < RW; q++) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) acc[q] += __shfl_xor(acc[q], o, 64);
        }
        if (ident != 0.f && lane == 0) {
#pragma unroll
            for (int q = 0; q < RW; q++)
                if (nb + q < g.N) acc[q] = fmaf(ident, g.g_ident[(long long)r * g.g_ident_ld + nb + q], acc[q]);
        }
#pragma unroll
        for (int q = 0; q < RW; q++) dn_put(g, r, nb + q, acc[q], acc[RW > 1 ? (q ^ 1) : q], lane == 0 && nb + q < g.N);
    }
}
template <typename WT, int RW>
static void dn_launch_mv_grouped(hipStream_t st, const dn_args &g, int rows, size_t lds) {
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)dense_mv_grouped_kernel<WT, RW>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    long long blocks = (g.N + 4 * RW - 1) / (4 * RW);
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL((dense_mv_grouped_kernel<WT, RW>), dim3((unsigned)blocks, (unsigned)rows), dim3(256), lds, st, g);
}

// ---------------------------------------------------------------------------------------------------- wide mat-mul (bf16: K % 64 == 0, fp32: K % 32 == 0)
// BM x BN (192 x 128, 128 x 128, 64 x 128 or 64 x 64) tokens x outputs per work-group: four waves multiply, four load.  Both operands in blocks of 128 bytes of K per row (64 bf16 or 32 fp32)
// through a ring of four LDS stages that the memory system fills by itself (global_load_lds_dwordx4: no registers, three blocks in flight).  What bounded the form before this one --
// 128 x 128 tiles, one block in flight through registers, two barriers per block -- was the latency of a block: 512 x 2048 x 2048 has 64 such tiles, one wave per SIMD on a quarter
// of the chip.  Hence the ring, smaller tiles or SPLITS of K where the tiles are fewer than the CUs (dn_ring_plan): a split product's partial tiles go to a scratch in register
// order and a second launch adds them in a fixed order and applies the epilogue.  The loading waves are apart because a request holds its wave's issue for 60 - 185 cycles:
// with the same four waves loading and multiplying a block of a 128 x 128 tile took 1650 cycles, 1000 of them requests, where its matrix instructions take 512.
//   * A stage is BM token rows, then BN weight rows, 128 bytes each, unpadded.  A piece = one wave-instruction = 8 rows; the instruction fixes where a lane's 16 bytes land but
//     not which 16 it fetches: slot s of row r holds piece s ^ (r / 2 % 8), so that the sixteen lanes a ds_read_b128 is served in meet every bank once.
//   * One barrier per block: in front of it the loaders' shares of block k have landed (counted: the later blocks' requests stay in flight) and the reads of block k - 1 are done;
//     behind it block k may be read and the stage of block k - 1 refilled.
//   * Operand fragments: 16 bytes per lane.  bf16: the eight k of v_mfma_f32_32x32x16_bf16.  fp32: four k, one per v_mfma_f32_32x32x2_f32 (lanes 0-31 and 32-63 hold different k;
//     both operands use the same assignment, so every k meets itself).
//   * Work-group order: dn_ring_place.
// Rows beyond T and outputs beyond N repeat the last one and are not stored.
// Measured (kernel trace, before -> now, bf16, 512 tokens): 2048 x 2048 45 -> 14 us, 8192 x 2048 72 -> 32 us (7 of them the xIELU of its epilogue), 2048 x 8192 190 -> 25 + 13 us (the
// sum); fp32, 300 tokens: 2048 x 2048 180 -> 30 + 11 us, 2048 x 8192 700 -> 103 + 11 us.  Loading alone takes 1030 cycles a block of 32 KiB, multiplying alone 530.  Tried and not
// faster: five to eight stages, a wave that prefetches the weights into L2, every tile starting at another block of K.
#define DN_STAGES 4
size_t psk_dense_split_bytes() { return (size_t)32 << 20; } // (the parts of at most 512 tiles of 64 KiB)
typedef float dn_f16 __attribute__((ext_vector_type(16)));

struct dn_ring {
    const char *A;      // packed operand rows (bf16 or fp32), or NULL: the rows of g.a themselves (fp32)
    long long lda;      // bytes
    int n_tm, tn, S;    // token tiles (grouped: at most, over all matrices), output tiles, splits of K
    float *part;        // S > 1: [tile][S][register order]
    long long each;     // > 0: the columns are those of several matrices with `each` of them (a multiple of BN), matrix i = w[i] over the operand copy i
    const void *w[1 + psk_dense_args::MORE];
    long long copy;     // bytes between their operand copies
};

// The A operand's rows with everything resolved that is not a plain row -- ring rows, token-shift mix, the slots' order and scale -- and, for bf16, rounded.
// PL 3: fp32 numbers as three of bf16, a row's three lines of K one behind the other -- rounded, the rounded rest, the rest of that: 24 bits, nothing lost.
// `mixes` of them (copies of the operand one behind the other) by a thread from one reading of the rows: 2047 tokens of 2048 in four mixes 23.8 us with a work-group for each, 13.2 so.
template <typename WT, int PL>
__global__ __launch_bounds__(256) void dense_pack_kernel(dn_args g, WT *out, int mixes) { // (blockIdx.y: the next so many mixes)
    if (blockIdx.y) { g.mu += (long long)blockIdx.y * mixes * g.K; out += (long long)blockIdx.y * mixes * g.T * g.K * PL; }
    long long row0 = g.a_row0;
    int T = g.T;
    if (!g.g_list) dn_rows(g, row0, T); // (grouped: all T slots in the order of the sorted list, whatever their matrix)
    else row0 = 0;
    const bool vec = g.lda % 4 == 0 && ((uintptr_t)g.a & 15) == 0, vec_mix = vec && ((uintptr_t)g.mu & 15) == 0 && ((uintptr_t)g.shift0 & 15) == 0;
    const unsigned per_row = (unsigned)(g.K / 8), total = (unsigned)T * per_row; // (the packed operand has fewer than 2^31 pieces of eight)
    auto eight = [](const float *x, bool vec, float *v) {
        if (vec) {
            *(dn_f4 *)v = *(const dn_f4 *)x;
            *(dn_f4 *)(v + 4) = *(const dn_f4 *)(x + 4);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = x[e];
        }
    };
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int t = (int)(i / per_row);
        const long long k = (long long)(i % per_row) * 8;
        float v[8];
        eight(dn_arow(g, row0, t) + k, vec, v);
        WT *o = out + (long long)t * g.K * PL + k;
        auto put = [&](const float *v) {
            if constexpr (PL == 3) {
                dn_us8 r[3];
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    // (a finite number that rounds to infinity is cut off instead; infinity has no rest)
                    unsigned short b = dn_f2bf(v[e]);
                    if ((b & 0x7fff) == 0x7f80) b = (unsigned short)(__float_as_uint(v[e]) >> 16);
                    const float rest = (b & 0x7fff) == 0x7f80 ? 0.f : v[e] - dn_bf2f(b);
                    const unsigned short b2 = dn_f2bf(rest);
                    r[0][e] = b; r[1][e] = b2; r[2][e] = dn_f2bf(rest - dn_bf2f(b2));
                }
#pragma unroll
                for (int x = 0; x < 3; x++) *(dn_us8 *)(o + x * g.K) = r[x];
            } else if constexpr (sizeof(WT) == 2) {
                dn_us8 r;
#pragma unroll
                for (int e = 0; e < 8; e++) r[e] = dn_f2bf(v[e]);
                *(dn_us8 *)o = r;
            } else {
                *(dn_f4 *)o = *(const dn_f4 *)v;
                *(dn_f4 *)(o + 4) = *(const dn_f4 *)(v + 4);
            }
        };
        if (g.g_list) {
            if (g.g_scale) {
                const float sc = g.g_scale[g.g_list[row0 + t]];
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] *= sc;
            }
            put(v);
        } else if (g.mu) {
            float p[8], mu[8], y[8];
            eight((t ? dn_arow(g, row0, t - 1) : g.shift0) + k, vec_mix, p);
#pragma unroll
            for (int e = 0; e < 8; e++) p[e] -= v[e];
            for (int c = 0; c < mixes; c++) {
                eight(g.mu + c * g.K + k, vec_mix, mu);
#pragma unroll
                for (int e = 0; e < 8; e++) y[e] = v[e] + p[e] * mu[e];
                put(y);
                o += (long long)g.T * g.K * PL;
            }
        } else put(v);
    }
}

// Four neighbouring results of output row t, columns n .. n + 3 (n a multiple of four).  The four go through ONE copy of the epilogue's code, the registers turning by one
// each time: code that runs a few times per launch has to be fetched first.  Four copies took 7.0 us in the sums of 512 x 2048, one 6.3; the activations of a wide product the same.
// ODD (dn_odd): rows that no 16-byte store fits, number by number.  A form of the kernels of its own: through the loop 282 x 10173 of K = 2304 took 41.5 us (36.4 in four copies, 33.5 so), and a
// branch for it in the other form costs a prompt of experts 1 %.
template <bool ODD>
static __device__ __forceinline__ void dn_put4(const dn_args &g, long long t, long long n, dn_f4 acc) {
    if (n >= g.N) return;
    if constexpr (ODD) {
        if (g.act == PSD_ACT_NONE && !g.bias && !g.accum && !g.out_scale && !g.out16) { // (uniform)
            float *p = g.out + t * g.ldo + n;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < g.N) p[e] = acc[e] * g.alpha;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) dn_put<true>(g, t, n + e, acc[e], 0.f, n + e < g.N);
        }
        return;
    }
    if (__builtin_expect(g.act == PSD_ACT_SILU_PAIR || g.act == PSD_ACT_RELU_PAIR || g.em_table != nullptr, 0)) { // (uniform; out of the others' way: a prompt of experts 6 255 -> 6 206 us)
#pragma unroll 1
        for (int e = 0; e < 4; e++) {
            dn_put<true>(g, t, n + e, acc[0], acc[1], n + e < g.N); // (a pair is stored by its even row)
            acc = dn_f4{acc[1], acc[2], acc[3], acc[0]};
        }
        return;
    }
    float *p = g.out + t * g.ldo + n;
    dn_f4 v = dn_f4{0.f, 0.f, 0.f, 0.f};
    if (g.accum) v = *(const dn_f4 *)p;
    const float rs = dn_row_scale(g, t);
    if (g.act == PSD_ACT_XIELU && !g.bias) { // (uniform)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] = dn_xielu(acc[e], g.act_p, g.act_q) * g.alpha;
    } else if (g.act != PSD_ACT_NONE || g.bias) {
#pragma unroll 1
        for (int e = 0; e < 4; e++) acc = dn_f4{acc[1], acc[2], acc[3], dn_epi(g, acc[0], n + e)};
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) acc[e] *= g.alpha;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float y = acc[e] * rs;
        v[e] = g.accum ? v[e] + y : y;
    }
    if (g.out16) {
        dn_us4 r;
#pragma unroll
        for (int e = 0; e < 4; e++) r[e] = dn_f2bf(v[e]);
        *(dn_us4 *)(g.out16 + (p - g.out)) = r;
    } else {
        *(dn_f4 *)p = v;
    }
}

static __device__ __forceinline__ void dn_dma(const char *src, unsigned lds_dst) { // one wave-instruction: lane l's 16 bytes at src go to lds_dst + 16 l
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(src), "s"(lds_dst) : "memory");
}

static __device__ __forceinline__ int dn_wave_upto(int v) { // the sum of the lanes up to this one
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true); // one, two, four and eight lanes on in a row of sixteen, then a row's last lane to the next row and the second row's to the upper half
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    return v + __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
}
// 64 matrices' slots at a time, a lane each (lanes behind the last matrix: none).  A loop over them one by one was a chain of loads in front of a work-group's first request, and two of them -- their number in
// dn_ring_place, this tile's here -- were half of the time of many experts: four layers of 2 048 with 256 of them, two a token, 150 tokens 2 726 -> 1 528 us, 1 500 4 831 -> 3 309; 64 of them, 1 500 tokens
// 1 935 -> 1 833.
template <int BM>
static __device__ __forceinline__ int dn_ring_slots(const dn_args &g, int base, int &at, int &next) { // tiles of this lane's matrix
    const int e = base + (int)(threadIdx.x & 63);
    at = g.g_seg[min(e, g.groups)];
    next = g.g_seg[min(e + 1, g.groups)];
    return (next - at + BM - 1) / BM;
}
// which tokens a tile holds: matrix e (grouped), its rows row0 .. row0 + T - 1, first local row t0; false: nothing
template <int BM>
static __device__ __forceinline__ bool dn_ring_rows(const dn_args &g, int tm, int &e, long long &row0, int &T, int &t0) {
    e = 0;
    if (g.g_seg) { // (uniform; tiles are counted matrix by matrix)
        for (int base = 0; base < g.groups; base += 64) {
            int at, next;
            const int c = dn_ring_slots<BM>(g, base, at, next), upto = dn_wave_upto(c), all = __builtin_amdgcn_readlane(upto, 63);
            if (tm < all) { // (uniform)
                const int l = __popcll(__ballot(upto <= tm));
                e = base + l;
                row0 = __builtin_amdgcn_readlane(at, l);
                T = __builtin_amdgcn_readlane(next, l) - (int)row0;
                t0 = (tm - __builtin_amdgcn_readlane(upto - c, l)) * BM;
                return true;
            }
            tm -= all;
        }
        return false;
    }
    dn_rows(g, row0, T);
    t0 = tm * BM;
    return t0 < T;
}

// The tile and split of a work-group.  Work-group b runs on XCD b % 8: an XCD has an eighth of the items there are, neighbours in the order of panels of four output tiles, so its L2 sees few token
// rows and few weights at a time, and no XCD has a column more than another.  With whole columns of tiles per XCD 1500 x 10304 of K = 2048 (41 columns of six tiles: 36 for one XCD, 30 for others) took
// two rounds, 97 us; 67 so.
#define DN_PANEL 4
template <int BM>
static __device__ __forceinline__ bool dn_ring_place(const dn_args &g, const dn_ring &p, int &tm, int &tn, int &s) {
    int n_tm = p.n_tm;
    if (g.g_seg) { // (the host's number is a bound)
        n_tm = 0;
#pragma unroll 4
        for (int base = 0; base < g.groups; base += 64) {
            int at, next;
            n_tm += dn_ring_slots<BM>(g, base, at, next);
        }
        n_tm = __builtin_amdgcn_readlane(dn_wave_upto(n_tm), 63);
    }
    const int tiles = n_tm * p.tn, items = tiles * p.S, each = (items + 7) >> 3, j = (int)blockIdx.x >> 3;
    int i = ((int)blockIdx.x & 7) * each + j;
    if (j >= each || i >= items) return false;
    s = p.S > 1 ? i / tiles : 0;
    i -= s * tiles;
    const int panel = i / (n_tm * DN_PANEL), width = min(DN_PANEL, p.tn - panel * DN_PANEL), r = i - panel * n_tm * DN_PANEL;
    tm = r / width;
    tn = panel * DN_PANEL + r % width;
    return true;
}

template <typename WT, int BM, int BN, bool ODD, int PL>
__global__ __launch_bounds__(512) void dense_mm_ring_kernel(dn_args g, dn_ring p) {
    extern __shared__ __attribute__((aligned(16))) char dn_lds[];
    constexpr int MI = BM / 64, NJ = BN / 64, NI = (BM + BN) / 32, STAGE = (BM + BN) * 128, NS = DN_STAGES; // instruction tiles per wave, pieces a loading wave requests per block
    constexpr int NA = BM / 32, NW = BN / 32, WL = NS * BM * 128; // PL 3: of them of the operand and of the weights; where the weights' two stages begin
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = (wave >> 1) & 1, wn = wave & 1;
    const bool loads = wave >= 4;
    int tm, tn, s, e, T, t0;
    if (!dn_ring_place<BM>(g, p, tm, tn, s)) return; // (uniform per work-group)
    long long row0;
    if (!dn_ring_rows<BM>(g, tm, e, row0, T, t0)) return; // (uniform per work-group)
    const long long n0 = (long long)tn * BN, ldw = g.K * (long long)sizeof(WT);
    const int blocks = (int)(ldw >> 7), kb0 = (int)((long long)blocks * s / p.S), nk = ((int)((long long)blocks * (s + 1) / p.S) - kb0) * PL; // (PL 3: block kb is line kb % 3 of K's block kb / 3)
    const int fr = lane & 31, fh = lane >> 5;
    dn_f16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    if (loads) {
        const int lw = wave - 4, lr = lane >> 3, ls = lane & 7;
        const char *W = (const char *)g.w + (g.g_seg ? e * g.wstride * (long long)sizeof(WT) : 0), *A = p.A, *src[NI];
        long long nw = n0, n_rows = g.N; // first row of W, rows of W
        if (p.each) { // (uniform)
            const int i = (int)(n0 / p.each);
            W = (const char *)(i == 0 ? p.w[0] : i == 1 ? p.w[1] : i == 2 ? p.w[2] : p.w[3]);
            A += i * p.copy;
            nw = n0 - i * p.each;
            n_rows = p.each;
        }
#pragma unroll
        for (int j = 0; j < NI; j++) {
            const int row = PL == 3 ? (j < NW ? BM + 8 * (NW * lw + j) : 8 * (NA * lw + j - NW)) + lr : 8 * (NI * lw + j) + lr, kq = ls ^ ((row >> 1) & 7); // (PL 3: the weights' pieces first)
            const char *q;
            if (row < BM) {
                const int t = min(t0 + row, T - 1);
                q = A ? A + (g.g_seg ? row0 + t : t) * p.lda : (const char *)dn_arow(g, row0, t);
            } else {
                const long long n = nw + row - BM;
                q = W + (n < n_rows ? n : n_rows - 1) * ldw;
            }
            src[j] = q + (long long)kb0 * 128 + kq * 16;
        }
        const unsigned lds0 = (unsigned)(size_t)(const __attribute__((address_space(3))) char *)dn_lds + (unsigned)(NI * lw * 1024);
        auto request = [&](const int kb) {
            if (kb >= nk) return;
            if constexpr (PL == 3) { // a block of the weights serves its three lines of the operand: two stages of it, requested with the first line
                const int kq = kb / 3, line = kb - 3 * kq;
                const unsigned at = lds0 - (unsigned)(NI * lw * 1024);
                if (line == 0) {
#pragma unroll
                    for (int j = 0; j < NW; j++) dn_dma(src[j] + (long long)kq * 128, at + (unsigned)(WL + (kq & 1) * BN * 128 + (NW * lw + j) * 1024));
                }
#pragma unroll
                for (int j = 0; j < NA; j++) dn_dma(src[NW + j] + line * ldw + (long long)kq * 128, at + (unsigned)((kb % NS) * BM * 128 + (NA * lw + j) * 1024));
                return;
            }
#pragma unroll
            for (int j = 0; j < NI; j++) dn_dma(src[j] + (long long)kb * 128, lds0 + (unsigned)((kb % NS) * STAGE + j * 1024));
        };
        request(0);
        request(1);
        request(2);
        for (int kb = 0; kb < nk; kb++) {
            const int later = nk - 1 - kb; // blocks requested behind this one: at most NS - 2
            if (PL == 3) { // (with the weights of the next block of K among them, but behind its first line; whole blocks of three lines)
                if (later >= 3 && kb % 3) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * NA + NW) : "memory");
                else if (later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * NA) : "memory");
                else if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(NA) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            } else if (later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * NI) : "memory");
            else if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(NI) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            request(kb + NS - 1);
        }
    } else {
        const int fx = (fr >> 1) & 7;
        const char *fa0 = dn_lds + (wm * MI * 32 + fr) * 128, *fb0 = dn_lds + (PL == 3 ? WL : BM * 128) + (wn * NJ * 32 + fr) * 128;
        dn_f4 xa[2][2][MI], xb[2][2][NJ]; // the fragments of half a block, two sets: the next half is read while this one is multiplied
        auto read = [&](const int kb, const int half) {
            const char *fa = fa0 + (kb % NS) * (PL == 3 ? BM * 128 : STAGE), *fb = fb0 + (PL == 3 ? (kb / 3 & 1) * BN * 128 : (kb % NS) * STAGE);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int po = ((4 * half + 2 * u + fh) ^ fx) << 4; // (the row bases are multiples of 32: (row / 2) % 8 = (fr / 2) % 8)
#pragma unroll
                for (int i = 0; i < MI; i++) xa[half][u][i] = *(const dn_f4 *)(fa + i * 32 * 128 + po);
#pragma unroll
                for (int j = 0; j < NJ; j++) xb[half][u][j] = *(const dn_f4 *)(fb + j * 32 * 128 + po);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto block = [&]() { // the reads of the block before are done; the next block is there
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        auto multiply = [&](const int half) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                if constexpr (sizeof(WT) == 2) {
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            dn_bf8 za, zb;
                            __builtin_memcpy(&za, &xa[half][u][i], 16);
                            __builtin_memcpy(&zb, &xb[half][u][j], 16);
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(zb, za, acc[i][j], 0, 0, 0);
                        }
                } else {
#pragma unroll
                    for (int x = 0; x < 4; x++)
#pragma unroll
                        for (int i = 0; i < MI; i++)
#pragma unroll
                            for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xb[half][u][j][x], xa[half][u][i][x], acc[i][j], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        block();
        read(0, 0);
        for (int kb = 0; kb < nk; kb++) {
            read(kb, 1);
            multiply(0);
            if (kb + 1 < nk) {
                block();
                read(kb + 1, 0);
            }
            multiply(1);
        }
        if (p.S > 1) {
            float *o = p.part + ((long long)(tm * p.tn + tn) * p.S + s) * (MI * NJ * 4096);
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
#pragma unroll
                    for (int q = 0; q < 4; q++)
                        *(dn_f4 *)(o + (((i * NJ + j) * 4 + q) * 256 + tid) * 4) = dn_f4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        }
    }
    if (p.S > 1) return;
    // The weights are the matrix instructions' first operand, so a lane has four neighbouring outputs of a token in four registers: results that need no epilogue go straight to their
    // places.  Through LDS (two barriers, a loop of eight trips) 512 x 8192 of K = 2048 took 35.0 us with its packing, 31.2 this way, 512 x 2048 18.3 and 17.3.
    // An activation of each of the 64 results of a lane, written out, is code that every CU has to fetch once: 40.6 us against 32.6 for a loop; it goes through LDS
    // (a squared relu is two instructions, a row's factor none: 1500 tokens of Pupidra 2048 x 6, 3514 us through LDS, 3283 so, with rounded rows handed on).
    if ((g.act == PSD_ACT_NONE || g.act == PSD_ACT_RELU2) && !g.bias && !g.accum && !g.em_table && g.N % 4 == 0 && g.ldo % 4 == 0 && ((uintptr_t)g.out & 15) == 0 && ((uintptr_t)g.out16 & 7) == 0) { // (uniform)
        if (loads) return;
#pragma unroll
        for (int i = 0; i < MI; i++) {
            const int t = t0 + wm * MI * 32 + i * 32 + fr;
            if (t >= T) continue;
            const long long to = dn_orow(g, row0, t, T), at = to * g.ldo + n0 + wn * NJ * 32 + 4 * fh;
            const float f = g.out_scale ? g.alpha * dn_row_scale(g, to) : g.alpha;
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (n0 + wn * NJ * 32 + j * 32 + 8 * q + 4 * fh >= g.N) continue;
                    dn_f4 v;
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = dn_relu2(g, acc[i][j][4 * q + e]) * f;
                    if (g.out16) {
                        dn_us4 r;
#pragma unroll
                        for (int e = 0; e < 4; e++) r[e] = dn_f2bf(v[e]);
                        *(dn_us4 *)(g.out16 + at + j * 32 + 8 * q) = r;
                    } else {
                        *(dn_f4 *)(g.out + at + j * 32 + 8 * q) = v;
                    }
                }
        }
        return;
    }
    // the tile through LDS (the stages are done with), so that the loading waves have their part in the epilogue
    constexpr int LD = BN + 4;
    float *tile = (float *)dn_lds;
    __syncthreads();
    if (!loads) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    *(dn_f4 *)&tile[(wm * MI * 32 + i * 32 + fr) * LD + wn * NJ * 32 + j * 32 + 8 * q + 4 * fh] = dn_f4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    }
    __syncthreads();
    const int c = (tid % (BN / 4)) * 4;
    for (int r = tid / (BN / 4); r < BM; r += 512 / (BN / 4)) {
        if (t0 + r >= T) break;
        dn_put4<ODD>(g, dn_orow(g, row0, t0 + r, T), n0 + c, *(const dn_f4 *)&tile[r * LD + c]);
    }
}

// the splits of a tile, added in order: one work-group per 32 x 32 instruction tile ij of a wave, read as it was written (a kilobyte per wave-instruction) and turned in LDS, so that
// eight lanes have 128 bytes of a row of the result: 7.5 us, the mean of a mixture-of-experts prompt's launches.  Eight lanes per row in the reading as well took 10.3 (128-byte pieces),
// a lane's registers straight to the result 10.3 too (32-byte pieces).
// A work-group that took the tiles of all four waves had one wave per SIMD of 256 CUs at work and sixteen columns of a row to write one behind the other: 14 us for
// the splits of 512 x 2048, 16 for those of 512 x 8; 5.7 and 4.8 now.
template <int BM, int BN, bool ODD>
__global__ __launch_bounds__(256) void dense_mm_sum_kernel(dn_args g, dn_ring p) {
    constexpr int MI = BM / 64, NJ = BN / 64, IJ = MI * NJ;
    __shared__ __attribute__((aligned(16))) float turn[32 * 36];
    const int tid = threadIdx.x, lane = tid & 63, q = tid >> 6, wave = (int)blockIdx.x & 3, wm = wave >> 1, wn = wave & 1; // (read: D registers 4 q .. 4 q + 3 of `lane`)
    const int ij = (int)(blockIdx.x >> 2) % IJ, tile = (int)(blockIdx.x >> 2) / IJ, tm = tile / p.tn, tn = tile % p.tn;
    int e, T, t0;
    long long row0;
    if (!dn_ring_rows<BM>(g, tm, e, row0, T, t0)) return;
    const float *src = p.part + (long long)tile * p.S * (IJ * 4096) + ij * 4096 + (q * 256 + wave * 64 + lane) * 4;
    dn_f4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < p.S; s += 8) { // (eight loads in flight)
        dn_f4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = *(const dn_f4 *)(src + (long long)min(s + u, p.S - 1) * (IJ * 4096));
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (s + u < p.S) acc += v[u];
    }
    *(dn_f4 *)&turn[(lane & 31) * 36 + 8 * q + 4 * (lane >> 5)] = acc;
    __syncthreads();
    const int r = tid >> 3, c = (tid & 7) * 4, t = t0 + wm * MI * 32 + (ij / NJ) * 32 + r;
    if (t < T) dn_put4<ODD>(g, dn_orow(g, row0, t, T), (long long)tn * BN + wn * NJ * 32 + (ij % NJ) * 32 + c, *(const dn_f4 *)&turn[r * 36 + c]);
}

// Tiles of 64 MI rows (MI 2, 3 or 4) x 256 columns, bf16.  Eight waves, a wave 16 MI x 32 of each quarter of the tile; K in blocks of 64, two LDS stages in four pieces (half of the tokens' rows or of
// the weights').  A block is two phases, one per half of the tokens' rows, a phase two slots: in one a wave reads fragments and requests pieces, in the other it multiplies (8 MI instructions), and the
// waves 4 - 7 are one slot behind the waves 0 - 3 of the same SIMDs, so that the matrix cores have one wave of a SIMD in every slot while the other's requests and reads hold only that one.  Pieces are
// requested over what all waves have just read (both groups' reads are back at the barrier in front), three phases before they are read themselves; a wait per phase is for all but the requests of the
// youngest two phases.  (Four phases, one per quarter, held a block of any height to 1.1 us, the time of eight slots of reads and requests: 1 090 x 6 208 of K = 4 096 in tiles of 128 rows 80 -> 72 us.)
// What bounded the 128 x 128 tiles here were the bytes from L2 (dn_ring_plan); these take half to three quarters of them per product.  A block takes 1.05 us with 256 rows (the matrix instructions
// alone 1.03, at the 2 GHz they hold), 0.88 with 192, 0.72 with 128.  2047 tokens, bf16, in the 128 x 128 form and here: 8192 x 2048 122 -> 59 us (16 of them the 67 MB of results, behind the last
// product of a CU's only tile); 1000 tokens 14336 x 4096 177 -> 117.  The heights against 256 rows only: 900 x 8192 x 4096 88 -> 74, 1532 x 8192 x 14336 332 -> 292.
#define DN_BIG 256
static constexpr int dn_big_lds(int MI) { return std::max(4 * (32 * MI + 128) * 128, 32 * MI * (DN_BIG + 4) * 4); } // the stages, then half of the tile
static __device__ __forceinline__ void dn_dma_at(const char *base, unsigned off, unsigned lds_dst) { // (as dn_dma, from a uniform base)
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(base), "s"(lds_dst) : "memory");
}
template <bool ODD, int PL, int MI>
__global__ __launch_bounds__(512) void dense_mm_big_kernel(dn_args g, dn_ring p) {
    extern __shared__ __attribute__((aligned(16))) char dn_lds[];
    constexpr int BM = 64 * MI, BN = DN_BIG, HR = 32 * MI, HALF_A = HR * 128, HALF = 128 * 128; // (HR: rows of a half of the tokens)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 2, wn = wave & 3;
    int tm, tn, s, e, T, t0;
    if (!dn_ring_place<BM>(g, p, tm, tn, s)) return; // (uniform per work-group)
    long long row0;
    if (!dn_ring_rows<BM>(g, tm, e, row0, T, t0)) return; // (uniform per work-group)
    const long long n0 = (long long)tn * BN, ldw = g.K * 2;
    const int nk = (int)(ldw >> 7) * PL; // (PL 3: block kb is line kb % 3 of K's block kb / 3; the weights' pieces stay for three of them)
    // this wave's two requests of a piece: rows 16 wave + 8 j + lane / 8, sixteen bytes each
    const char *W = (const char *)g.w + (g.g_seg ? e * g.wstride * 2 : 0), *A = p.A;
    long long nw = n0, n_rows = g.N;
    if (p.each) { // (uniform)
        const int i = (int)(n0 / p.each);
        W = (const char *)(i == 0 ? p.w[0] : i == 1 ? p.w[1] : i == 2 ? p.w[2] : p.w[3]);
        A += i * p.copy;
        nw = n0 - i * p.each;
        n_rows = p.each;
    }
    A += (g.g_seg ? row0 + t0 : t0) * p.lda;
    W += nw * ldw;
    // A piece of HR rows is 4 MI requests: where they are not a multiple of the waves, the waves 0 - 3 have one more of the first half and 4 - 7 of the second
    constexpr int NA = (MI + 1) / 2;
    unsigned oa[2][NA], ob[2][2];
    auto piece = [&](const int h, const int j) { return MI == 3 ? (j ? 8 + (wave & 3) : wave) : NA * wave + j; };
    auto has = [&](const int h, const int j) { return MI != 3 || j == 0 || (wm != 0) == (h != 0); }; // (uniform)
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int j = 0; j < NA; j++) {
            const int r = 8 * piece(h, j) + (lane >> 3), kq = (lane & 7) ^ ((r >> 1) & 7);
            oa[h][j] = (unsigned)min(h * HR + r, T - 1 - t0) * (unsigned)p.lda + kq * 16;
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int r = 16 * wave + 8 * j + (lane >> 3), kq = (lane & 7) ^ ((r >> 1) & 7);
            ob[h][j] = (unsigned)min((long long)(h * 128 + r), n_rows - 1 - nw) * (unsigned)ldw + kq * 16;
        }
    }
    const unsigned lds0 = (unsigned)(size_t)(const __attribute__((address_space(3))) char *)dn_lds;
    auto request_a = [&](const int kb, const int h) {
#pragma unroll
        for (int j = 0; j < NA; j++)
            if (has(h, j)) dn_dma_at(A + (PL == 3 ? kb % 3 * ldw + (long long)(kb / 3) * 128 : (long long)kb * 128), oa[h][j], lds0 + (unsigned)((2 * (kb & 1) + h) * HALF_A + piece(h, j) * 1024));
    };
    auto request_w = [&](const int kb, const int h) { // (PL 3: kb counts blocks of K)
#pragma unroll
        for (int j = 0; j < 2; j++) dn_dma_at(W + (long long)kb * 128, ob[h][j], lds0 + (unsigned)(4 * HALF_A + (2 * (kb & 1) + h) * HALF + wave * 2048 + j * 1024));
    };
    dn_f4 acc[2][2][MI][2], xa[2][MI], xb[2][2][2]; // (tokens' half, weights' half)
#pragma unroll
    for (int mh = 0; mh < 2; mh++)
#pragma unroll
        for (int nh = 0; nh < 2; nh++)
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[mh][nh][i][j] = dn_f4{0.f, 0.f, 0.f, 0.f};
    const int fr = lane & 15, po = (((lane >> 4) ^ (fr >> 1)) << 4); // (row bases are multiples of sixteen; the second half of a block: the piece's number with its third bit turned)
    const char *fa[2] = {dn_lds + (wm * 16 * MI + fr) * 128 + po, dn_lds + (wm * 16 * MI + fr) * 128 + (po ^ 64)};
    const char *fb[2] = {dn_lds + 4 * HALF_A + (wn * 32 + fr) * 128 + po, dn_lds + 4 * HALF_A + (wn * 32 + fr) * 128 + (po ^ 64)};
    auto read_a = [&](const int kb, const int h) {
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < MI; i++) xa[u][i] = *(const dn_f4 *)(fa[u] + (2 * (kb & 1) + h) * HALF_A + i * 2048);
    };
    auto read_w = [&](const int kb, const int h) {
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int j = 0; j < 2; j++) xb[h][u][j] = *(const dn_f4 *)(fb[u] + (2 * ((PL == 3 ? kb / 3 : kb) & 1) + h) * HALF + j * 2048);
    };
    auto multiply = [&](const int mh) { // between two barriers: the other group's slot of reads and requests
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int nh = 0; nh < 2; nh++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        dn_bf8 za, zb;
                        __builtin_memcpy(&za, &xa[u][i], 16);
                        __builtin_memcpy(&zb, &xb[nh][u][j], 16);
                        acc[mh][nh][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(zb, za, acc[mh][nh][i][j], 0, 0, 0);
                    }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // requests behind the piece that is waited for: those of two phases (PL 3: of them the operand's)
    constexpr int LATER = MI + (PL == 3 ? 0 : 4);
    request_w(0, 0); request_w(0, 1); request_a(0, 0); request_a(0, 1);
    if (nk > 1) {
        if (PL == 1) { request_w(1, 0); request_w(1, 1); }
        request_a(1, 0);
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(MI / 2 + (PL == 3 ? 0 : 4)) : "memory");
    } else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (wm) __builtin_amdgcn_s_barrier();
    for (int kb = 0; kb < nk; kb++) {
#define DN_BIG_LANDED(more)                                                    \
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LATER) : "memory");     \
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const bool more = kb + 2 < nk;
        read_w(kb, 0);
        read_w(kb, 1);
        read_a(kb, 0);
        if (kb + 1 < nk) request_a(kb + 1, 1);
        DN_BIG_LANDED(more)
        multiply(0);
        read_a(kb, 1);
        if (more) {
            if (PL == 1) { request_w(kb + 2, 0); request_w(kb + 2, 1); }
            else if ((kb + 2) % 3 == 0) { request_w((kb + 2) / 3, 0); request_w((kb + 2) / 3, 1); }
            request_a(kb + 2, 0);
        }
        DN_BIG_LANDED(more)
        multiply(1);
#undef DN_BIG_LANDED
    }
    if (!wm) __builtin_amdgcn_s_barrier();
    if ((g.act == PSD_ACT_NONE || g.act == PSD_ACT_RELU2) && !g.bias && !g.accum && !g.em_table && g.N % 4 == 0 && g.ldo % 4 == 0 && ((uintptr_t)g.out & 15) == 0 && ((uintptr_t)g.out16 & 7) == 0) { // (uniform)
#pragma unroll
        for (int mh = 0; mh < 2; mh++)
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int t = t0 + mh * HR + wm * 16 * MI + i * 16 + fr;
                if (t >= T) continue;
                const long long to = dn_orow(g, row0, t, T), at = to * g.ldo + n0;
                const float f = g.out_scale ? g.alpha * dn_row_scale(g, to) : g.alpha;
#pragma unroll
                for (int nh = 0; nh < 2; nh++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const int c = nh * 128 + wn * 32 + j * 16 + 4 * (lane >> 4);
                        if (n0 + c >= g.N) continue;
                        dn_f4 v;
#pragma unroll
                        for (int x = 0; x < 4; x++) v[x] = dn_relu2(g, acc[mh][nh][i][j][x]) * f;
                        if (g.out16) {
                            dn_us4 r;
#pragma unroll
                            for (int x = 0; x < 4; x++) r[x] = dn_f2bf(v[x]);
                            *(dn_us4 *)(g.out16 + at + c) = r;
                        } else {
                            *(dn_f4 *)(g.out + at + c) = v;
                        }
                    }
            }
        return;
    }
    // half of the tile at a time through LDS (the stages are done with)
    constexpr int LD = BN + 4;
    float *tile = (float *)dn_lds;
#pragma unroll
    for (int mh = 0; mh < 2; mh++) {
        __syncthreads();
#pragma unroll
        for (int nh = 0; nh < 2; nh++)
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) *(dn_f4 *)&tile[(wm * 16 * MI + i * 16 + fr) * LD + nh * 128 + wn * 32 + j * 16 + 4 * (lane >> 4)] = acc[mh][nh][i][j];
        __syncthreads();
        for (int r = wave; r < HR; r += 8) {
            const int t = t0 + mh * HR + r;
            if (t >= T) break;
            dn_put4<ODD>(g, dn_orow(g, row0, t, T), n0 + 4 * lane, *(const dn_f4 *)&tile[r * LD + 4 * lane]);
        }
    }
}
static bool dn_odd(const dn_args &g) { return g.act != PSD_ACT_SILU_PAIR && g.act != PSD_ACT_RELU_PAIR && !g.em_table && (g.N % 4 || g.ldo % 4 || ((uintptr_t)g.out & 15)); }
// Tile and splits of a product of `rows` tokens (grouped: slots of `groups` matrices).  bf16 and three lines: the least of an estimate in us of what a shape makes of a product -- not of its time, which has more
// in it that all shapes have in common (the launch, packing, the results and what of the weights is not there yet: 2.6 us and up in bf16, 6 in three lines): rounds of 256 work-groups times (blocks of K times what a
// block of the shape costs, its start, what the epilogue adds behind a tile: dn_epilogue), and for a split product its second launch and its parts' way through memory.  64 x 64 stands twice on a CU: two of them
// hide each other's waits, one alone does not.  Fitted to 1 200 products of models (six families at widths 2 048 and 4 096, 2 to 2 047 tokens, K 512 .. 14 336, experts, epilogues; ten shapes and splits each,
// timed where they stand in a portion), to 1 240 alone (N 1 024 .. 24 576, K from 512, weights from memory) and to 260 of K 64 .. 384.  What it picks, against the best of all, on average, and the rule before (one
// cost of 64 x 64, no more for few blocks; fitted from 9 tokens and K of 1 536 on): in models bf16 1.0 % and 1.2 % of their time, three lines 0.4 % and 1.8 % (2 to 64 tokens 0.8 % and 4.4 %); on 480 that it was not
// fitted to bf16 0.7 % and 0.7 %, three lines 0.4 % and 0.8 %; K 64 .. 384 in bf16 0.6 % and 11 %.  Us there and here, alone: 300 x 2 048 x 4 096 20.9 and 18.0, 620 x 1 024 x 4 096 20.7 and 17.8, 300 x 512 x 64 7.4
// and 4.3; in three lines 2 x 4 096 x 4 096 22.7 and 20.1, 8 x 8 192 x 2 048 22.7 and 20.0, 190 x 5 120 x 2 560 38.8 and 32.8.
//   A block costs the bytes it fetches: a CU has about 16 KB of requests outstanding, which the mean way to L2 and beyond makes some 60 bytes a ns, whatever the shape -- 32 KB in 0.5 us of 128 x 128, start
// included, 64 KB in 1.0 of 256 x 256.  So larger tiles do more per byte, and a height that leaves no round nearly empty counts as much.
//   Experts' rows: an expert has rows / groups on average, spread as a random routing and some more; the expected number of its tiles (few slots of many experts: of experts that have one.  Nine
// tokens, two of 64 experts, counted as 22 tiles instead of 16 took shapes of two rounds: 584 us of four layers, 553 so; 300 slots of eight matrices of 2 048 x 2 048, 8.01 tiles of 64
// rows, 34 us in 64 x 128 and 28 in 64 x 64).
// The fp32 instruction (dn_ring_plan_f32): a block of K costs its tile's matrix instructions, or its LDS traffic (fragments read by four waves, the block written), whichever is more.
struct dn_ring_shape { int BM, BN, n_tm, tn, S; };
enum { DN_EPI_DIRECT, DN_EPI_FOURS, DN_EPI_ONES }; // results from the registers; through LDS, four at a time; an activation or bias each
static int dn_epilogue(const dn_args &g) {
    if (g.act == PSD_ACT_SILU_PAIR || g.act == PSD_ACT_RELU_PAIR || g.em_table || g.bias) return DN_EPI_ONES;
    if (g.act == PSD_ACT_XIELU) return DN_EPI_FOURS;
    if (g.act != PSD_ACT_NONE && (g.act != PSD_ACT_RELU2 || g.accum)) return DN_EPI_ONES;
    return g.accum || dn_odd(g) ? DN_EPI_FOURS : DN_EPI_DIRECT;
}
static int dn_row_tiles(int rows, int BM, int groups) { // at most
    return rows / BM + (groups > 0 ? std::min(groups, rows) : rows % BM ? 1 : 0);
}
static double dn_mean_row_tiles(int rows, int BM, int groups) {
    if (!groups) return (rows + BM - 1) / BM;
    const double mean = (double)rows / groups, sd = std::sqrt(mean) + mean / 16;
    double tiles = 0;
    for (int k = 0; k <= rows / BM; k++) { // an expert has its tile k where it has more than k BM rows
        const double p = k ? 0.5 * std::erfc((k * BM + 0.5 - mean) / (sd * 1.41421356)) : 1 - std::exp(-mean); // (one tile at least: a slot at all, few of them too)
        tiles += p;
        if (p < 1e-3) break;
    }
    return std::max(1.0, std::ceil(groups * tiles - 0.3)); // (what most routings have: a second tile that one in a hundred experts needs made two rounds of 256 tiles)
}
static dn_ring_shape dn_ring_plan_f32(int rows, int64_t N, int64_t kbytes, int groups, bool may_split) {
    static const int shapes[3][2] = {{128, 128}, {64, 128}, {64, 64}};
    const int64_t blocks = kbytes / 128;
    dn_ring_shape best{};
    double least = 0;
    for (auto &q : shapes) {
        const int BM = q[0], BN = q[1], n_tm = dn_row_tiles(rows, BM, groups), tn = (int)((N + BN - 1) / BN), full = (rows + BM - 1) / BM;
        const int64_t tiles = (int64_t)(groups > 0 ? std::max(full, std::min(groups, rows)) + (rows > groups * BM ? groups / 2 : 0) : full) * tn; // (grouped: about half of the last tiles start a new one)
        const double lds = 3.0 * (BM + BN), mfma = BM * BN / 64.0 * 16, block = std::max(lds, mfma) + 100;
        for (int64_t S = 1; S <= (may_split ? 16 : 1); S++) {
            if (S > 1 && (blocks / S < 4 || tiles * S > 512 || (size_t)n_tm * tn * S * BM * BN * 4 > psk_dense_split_bytes())) break;
            const double rounds = (double)((tiles * S + 255) / 256), t = rounds * (double)((blocks + S - 1) / S) * block + 4000 + (S > 1 ? 9000 + (double)tiles * S * BM * BN * 4 / 3000 : 0);
            if (!best.BM || t < least) { least = t; best = dn_ring_shape{BM, BN, n_tm, tn, (int)S}; }
        }
    }
    return best;
}
static dn_ring_shape dn_ring_plan(int rows, int64_t N, int64_t kbytes, int lines, int groups, bool may_split, bool big, int epilogue) {
    struct shape { int BM, BN; double block[2], round[2]; }; // (bf16, three lines: a block of 128 x 256 there is 3.2, two of 128 x 128 are 2.9.  64 x 64: of two work-groups of a CU, each)
    static const shape shapes[7] = {{256, 256, {1.010, 4.085}, {0.09, 1.65}}, {192, 256, {0.892, 3.571}, {0, 0.12}}, {128, 256, {0.774, 0}, {0.05, 0}}, {192, 128, {0.518, 1.960}, {2.72, 0}},
                                    {128, 128, {0.383, 1.431}, {2.27, 0}}, {64, 128, {0.285, 0.843}, {1.54, 0.37}}, {64, 64, {0.169, 0.543}, {0.87, 0.11}}};
    static const double alone[2] = {0.191, 0.596};                        // 64 x 64 without a second work-group on the CU
    static const double behind[2][3] = {{0, 0.95, 5.2}, {0, 2.0, 6.25}};  // by 128 x 128 numbers; of tiles of 128 columns and less, of 256
    static const double sums[2] = {2.48, 1.60}, parts[2] = {0.194, 0.289}; // a split product: once, by MB
    static const double few = 4;                                          // what fewer than eight blocks of K don't hide of the start of 256 columns, at none; bf16
    const int64_t blocks = kbytes / 128;
    const int l = lines == 3;
    dn_ring_shape best{};
    double least = 0;
    for (auto &q : shapes) {
        if (q.BN == DN_BIG && (!big || q.block[l] == 0)) continue;
        const int n_tm = dn_row_tiles(rows, q.BM, groups), tn = (int)((N + q.BN - 1) / q.BN);
        const double area = q.BM * q.BN / 16384.0, tiles = dn_mean_row_tiles(rows, q.BM, groups) * tn, start = q.round[l] + (l == 0 && q.BN == DN_BIG && blocks < 8 ? few * (8 - blocks) / 8 : 0);
        for (int64_t S = 1; S <= (may_split && q.BN < DN_BIG ? 16 : 1); S++) {
            if (S > 1 && (blocks / S < 4 || tiles * S > 700 || (size_t)n_tm * tn * S * q.BM * q.BN * 4 > psk_dense_split_bytes())) break;
            const double rounds = std::ceil(tiles * S / 256), single = q.BN == 64 ? std::fmod(rounds, 2) : 0, starts = q.BN == 64 ? (rounds + single) / 2 : rounds; // (two work-groups start together)
            const double t = (double)((blocks + S - 1) / S) * ((rounds - single) * q.block[l] + single * alone[l]) + starts * start + (S == 1 ? rounds * behind[q.BN == DN_BIG][epilogue] * area : 0) +
                             (S > 1 ? sums[l] + parts[l] * tiles * S * area * 0.0655 : 0);
            if (!best.BM || t < least) { least = t; best = dn_ring_shape{q.BM, q.BN, n_tm, tn, (int)S}; }
        }
    }
    return best;
}

template <typename WT, int BM, int BN, bool ODD, int PL>
static void dn_launch_ring(hipStream_t st, const dn_args &g, const dn_ring &p) {
    if constexpr (!ODD)
        if (dn_odd(g)) return dn_launch_ring<WT, BM, BN, true, PL>(st, g, p);
    constexpr int LDS = DN_STAGES * (BM + BN) * 128;
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)dense_mm_ring_kernel<WT, BM, BN, ODD, PL>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    const unsigned grid = (unsigned)(((long long)p.tn * p.S * p.n_tm + 7) / 8 * 8);
    hipLaunchKernelGGL((dense_mm_ring_kernel<WT, BM, BN, ODD, PL>), dim3(grid), dim3(512), LDS, st, g, p);
    if (p.S > 1) hipLaunchKernelGGL((dense_mm_sum_kernel<BM, BN, ODD>), dim3((unsigned)(p.n_tm * p.tn * (BM / 64) * (BN / 64) * 4)), dim3(256), 0, st, g, p);
}

template <bool ODD, int PL, int MI>
static void dn_launch_big(hipStream_t st, const dn_args &g, const dn_ring &p) {
    if constexpr (!ODD)
        if (dn_odd(g)) return dn_launch_big<true, PL, MI>(st, g, p);
    constexpr int LDS = dn_big_lds(MI);
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)dense_mm_big_kernel<ODD, PL, MI>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    hipLaunchKernelGGL((dense_mm_big_kernel<ODD, PL, MI>), dim3((unsigned)(((long long)p.tn * p.n_tm + 7) / 8 * 8)), dim3(512), LDS, st, g, p);
}

// The wide mat-mul, where it takes the product: whole blocks of K, room for what has to be packed.  PL 3 (WT: bf16): an fp32 product on the bf16 instruction -- the weights as they came, which is in
// bf16, the operand as the sum of three bf16 lines (dense_pack_kernel): every product is exact, the sums are fp32.  A block of the weights stays in LDS for its three lines.  What bounded the
// fp32 instruction was its rate, a sixteenth of the other's; 300 tokens, it and this: 8192 x 2048 126 -> 64 us, 2048 x 8192 148 + 5 -> 69 + 5, 2048 x 2048 62 -> 31; whole requests from 9
// tokens on (Ranutar 2048 x 3: 9 tokens 505 -> 465 us, 64: 530 -> 475, 512: 1698 -> 1044; Pupidra 4096 x 3, 200: 3662 -> 2149).  Error against 64 bits, ranutar-f32-prompt: 1.0e-6 -> 6.2e-7.
template <typename WT, int PL>
static bool dn_ring_take(hipStream_t st, const psk_dense_args &a, dn_args g) {
    const int64_t kbytes = g.K * (int64_t)sizeof(WT);
    const int copies = 1 + a.n_more;
    if (copies > 1 && (g.N % 128 || !g.mu)) return false;
    if (a.force_tiled || kbytes % 128 || !a.pack) return false;
    const bool rows = !g.mu && !g.g_list && !g.a_mod && !g.a_step && !g.a_row0;
    const bool handed = sizeof(WT) == 2 && PL == 1 && a.a16 && (rows || (g.g_list && !g.g_scale)); // (the producer has rounded them already; slots: in the list's order)
    const bool plain = handed || (sizeof(WT) == 4 && !g.mu && !g.g_scale && g.lda % 4 == 0 && ((uintptr_t)g.a & 15) == 0);
    if (!plain && (size_t)a.T * kbytes * PL * copies > a.pack_bytes) return false;
    if (PL == 3) {
        for (int i = 0; i < copies; i++)
            if (!(i ? a.more[i - 1] : a.w)->half) return false;
        g.w = a.w->half;
    }
    const int64_t each = g.N;
    g.N *= copies;
    const bool may_split = a.split && a.split_bytes >= psk_dense_split_bytes();
    const dn_ring_shape r = sizeof(WT) == 4 ? dn_ring_plan_f32(a.T, g.N, kbytes, g.groups, may_split)
                                            : dn_ring_plan(a.T, g.N, kbytes, PL, g.groups, may_split, (each % DN_BIG == 0 || copies == 1) && kbytes < (1 << 22), dn_epilogue(g)); // (rows of a tile by 32-bit offsets)
    dn_ring p{handed ? (const char *)a.a16 : plain ? nullptr : (const char *)a.pack, kbytes * PL, r.n_tm, r.tn, r.S, a.split};
    p.each = copies > 1 ? each : 0;
    p.copy = a.T * kbytes * PL;
    for (int i = 0; i < copies; i++) p.w[i] = i ? (PL == 3 ? a.more[i - 1]->half : a.more[i - 1]->data) : g.w;
    if (!plain) {
        const int64_t pb = ((int64_t)a.T * (g.K / 8) + 255) / 256;
        const int mixes = pb >= 256 ? copies : 1; // (few tokens: as many work-groups as there are mixes)
        hipLaunchKernelGGL((dense_pack_kernel<WT, PL>), dim3((unsigned)std::min<int64_t>(pb, 8192), (unsigned)(copies / mixes)), dim3(256), 0, st, g, (WT *)a.pack, mixes);
    }
    if (r.BN == DN_BIG) {
        if constexpr (sizeof(WT) == 2) {
            if (r.BM == 128) {
                if constexpr (PL == 1) dn_launch_big<false, PL, 2>(st, g, p);
            } else if (r.BM == 192) dn_launch_big<false, PL, 3>(st, g, p);
            else dn_launch_big<false, PL, 4>(st, g, p);
        }
    } else if (r.BM == 192) {
        if constexpr (sizeof(WT) == 2) dn_launch_ring<WT, 192, 128, false, PL>(st, g, p);
    } else if (r.BM == 128) dn_launch_ring<WT, 128, 128, false, PL>(st, g, p);
    else if (r.BN == 128) dn_launch_ring<WT, 64, 128, false, PL>(st, g, p);
    else dn_launch_ring<WT, 64, 64, false, PL>(st, g, p);
    return true;
}
static bool dn_wide(hipStream_t st, const psk_dense_args &a, const dn_args &g) {
    if (a.w->dtype == PS_BF16) return dn_ring_take<unsigned short, 1>(st, a, g);
    // (a small matrix and few rows: three lines are a launch more.  us on the fp32 instruction and in three lines, weights from memory: 16 tokens 768 x 2048 11.7 and 13.8, 2048 x 1024 12.0 and 13.9,
    // 2048 x 2048 14.3 and 15.3, 1024 x 4096 14.7 and 16.1, 4096 x 2048 18.5 and 18.5; 64 tokens 768 x 768 9.3 and 11.9, 2048 x 1024 11.9 and 14.1, 2048 x 2048 14.2 and 15.5, 2048 x 4096 18.6 and 19.6;
    // 128 tokens 2048 x 1024 13.4 and 14.8, 2048 x 2048 17.7 and 18.0, 4096 x 2048 29.2 and 22.3; 256 tokens 1024 x 1024 12.6 and 15.5, 2048 x 1024 17.8 and 18.7, 2048 x 2048 27.8 and 22.7)
    const bool small = a.small_f32 && !g.groups && !a.n_more && g.N * g.K <= (1 << 22) && a.T * g.N * g.K <= (1 << 28);
    return (a.w->half && !small && dn_ring_take<unsigned short, 3>(st, a, g)) || dn_ring_take<float, 1>(st, a, g);
}

// Products with an inner size of a few numbers (the second matrix of a low-rank decay): a thread has an output column, its KP weights in registers, and runs over sixteen tokens whose
// activations lie in LDS.  Nothing but the writing of the result counts here: 512 x 2048 of K = 8 took the tiled kernel 23 us (a tile's results leave a lane one number per row), 10.9 now.
template <typename WT, int KP>
__global__ __launch_bounds__(256) void dense_mm_few_kernel(dn_args g) {
    __shared__ float as[16 * KP];
    const int tid = threadIdx.x, t0 = blockIdx.y * 16, K = (int)g.K;
    const long long n = (long long)blockIdx.x * 256 + tid;
    float w[KP];
#pragma unroll
    for (int k = 0; k < KP; k++) {
        w[k] = 0.f;
        if (n < g.N && k < K) {
            if constexpr (sizeof(WT) == 2) w[k] = dn_bf2f(((const unsigned short *)g.w)[n * K + k]);
            else w[k] = ((const float *)g.w)[n * K + k];
        }
    }
    for (int i = tid; i < 16 * KP; i += 256) {
        const int t = t0 + i / KP, k = i % KP;
        float v = t < g.T && k < K ? g.a[t * g.lda + k] : 0.f;
        if constexpr (sizeof(WT) == 2) v = dn_bf2f(dn_f2bf(v));
        as[i] = v;
    }
    __syncthreads();
#pragma unroll 4
    for (int t = 0; t < 16; t++) {
        float a = 0.f;
#pragma unroll
        for (int k = 0; k < KP; k++) a = fmaf(as[t * KP + k], w[k], a);
        dn_put(g, t0 + t, n, a, __shfl_xor(a, 1, 64), t0 + t < g.T && n < g.N);
    }
}

// Products with a short inner size and few tiles (the ring would be all packing and prologue): 32 tokens x 32 outputs per work-group.  Each of the NW waves takes
// its share of K, its operand fragments straight from memory (the activations are rounded to bfloat16 in registers: nothing is packed beforehand), all its STEPS of 32 in flight; the
// partial tiles meet in LDS.  Plain rows only (no ring, no token shift, no groups).
template <int NW, int STEPS> // K = NW STEPS 32
__global__ __launch_bounds__(64 * NW) void dense_mm_narrow_kernel(dn_args g) {
    __shared__ float part[NW][32][33];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 15, lq = lane >> 4, t0 = blockIdx.x * 32; // (rows fastest: the blocks that read the same rows of A sit on one XCD where the row tiles are a multiple of 8)
    const long long n0 = (long long)blockIdx.y * 32, kw = STEPS * 32;
    const float *ap[2];
    const unsigned short *bp[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int t = min(t0 + 16 * i + lr, g.T - 1);
        const long long n = min(n0 + 16 * i + lr, g.N - 1);
        ap[i] = g.a + t * g.lda + wave * kw + lq * 8;
        bp[i] = (const unsigned short *)g.w + n * g.K + wave * kw + lq * 8;
    }
    dn_f4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = dn_f4{0.f, 0.f, 0.f, 0.f};
    dn_f4 xa[STEPS][2][2], xb[STEPS][2];
#pragma unroll
    for (int u = 0; u < STEPS; u++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            xa[u][i][0] = *(const dn_f4 *)(ap[i] + 32 * u);
            xa[u][i][1] = *(const dn_f4 *)(ap[i] + 32 * u + 4);
            xb[u][i] = *(const dn_f4 *)(bp[i] + 32 * u);
        }
#pragma unroll
    for (int u = 0; u < STEPS; u++) {
        dn_bf8 fa[2], fb[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            dn_us8 r;
#pragma unroll
            for (int e = 0; e < 8; e++) r[e] = dn_f2bf(xa[u][i][e >> 2][e & 3]);
            __builtin_memcpy(&fa[i], &r, 16);
            __builtin_memcpy(&fb[i], &xb[u][i], 16);
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) part[wave][16 * i + 4 * lq + e][16 * j + lr] = acc[i][j][e];
    __syncthreads();
#pragma unroll
    for (int x = 0; x < 16 / NW; x++) {
        const int r = (tid + 64 * NW * x) >> 5, c = tid & 31;
        float v = part[0][r][c];
#pragma unroll
        for (int w = 1; w < NW; w++) v += part[w][r][c];
        dn_put(g, t0 + r, n0 + c, v, __shfl_xor(v, 1, 64), t0 + r < g.T && n0 + c < g.N); // (row n ^ 1 is the neighbouring lane's)
    }
}

// ---------------------------------------------------------------------------------------------------- a single token: streaming mat-vec
// A wave walks its rows as ONE stream of 1 KiB units (16 bytes per lane, non-temporal), DN_AHEAD of them in flight, requested before the activations are staged and across row ends, so
// that neither the prologue nor a row's reduction leaves the memory idle.  Rows are dealt to the waves of the whole launch in turn (consecutive waves read consecutive rows; a matrix
// of 2048 rows gives each of 2048 waves one), or in neighbouring pairs for a paired activation.  What bounded dense_mv_kernel here was the number of bytes in flight: four rows per wave,
// two pieces each, 128 work-groups of four waves for 2048 rows.  Measured, bf16, before and now: 2048 x 4096 (16.8 MB) 14.6 and 6.6 us, 8192 x 2048 (33 MB) 15 and 9, 14336 x 4096
// (117 MB) 29 to 38 and 22 us (5.3 TB/s).  The first product of a token's experts (top 2 of 3072 x 2048 and a shared one of twice that, 50 MB), which was two launches, 12.4 + 10.4 and 12.0 us.
//  Four units in flight: a token of Ranutar 4096 x 3, 2048 x 6, Pupidra 2048 x 6, 4096 x 3 in us with two units 349 351 378 405, three 334 340 376 395, four 322 343 376 387, five 331 348 378 392,
//  six 339 352 386 399, eight (as it was) 326 356 390 389, sixteen 326 353 390 397; 768 and 1024 work-groups instead of 512: the same or up to 5 % more; ordinary loads instead of
//  non-temporal ones: 357 383 412 420.  (mv2's in flight: one row per wave, three units of it, 376 against 381 with two rows and 382 with its eight.)
//   FORM 0  one matrix
//   FORM 1  grouped, the first product of an expert: work-groups in equal runs per slot (its own matrix and output row), behind them those of the shared expert (g2)
//   FORM 2  several matrices of one shape, each over its own mix of the token and the one before it (psk_dense_args::more): work-groups in equal runs per matrix.  Four of 4096 x 4096,
//           33 MB each: 10.7 us one by one, 23.7 together (5.7 TB/s)
// dynamic LDS: the activations as bf16-rounded fp32 (fp32 mode: as they are), every vector padded with zeros to whole units
#define DN_AHEAD 4
struct dn_mv1 {
    dn_args g2;  // FORM 1: the shared expert's first product (w NULL: none)
    int slots;   // FORM 1: slots of the launch
    int kp;      // padded length of the vector
    int blocks, blocks2; // FORM 1: work-groups per slot, of the shared expert; FORM 2: per matrix
    const void *w[1 + psk_dense_args::MORE]; // FORM 2: the matrices
    psk_dense_pre pre;
};

// one vector into LDS, by all 512 threads
template <typename WT>
static __device__ __forceinline__ void dn_stage(const dn_args &g, const float *x, const float *prev, float scale, float *xs, int kp) {
    const int K = (int)g.K;
    if (K % 4 == 0 && ((uintptr_t)x & 15) == 0 && (!prev || (((uintptr_t)prev | (uintptr_t)g.mu) & 15) == 0)) {
        for (int k = threadIdx.x * 4; k < kp; k += 512 * 4) {
            dn_f4 v = k < K ? *(const dn_f4 *)(x + k) : dn_f4{0.f, 0.f, 0.f, 0.f};
            if (prev && k < K) { // (the token-shift mix of dn_aval; never with a scale)
                const dn_f4 b = *(const dn_f4 *)(prev + k), m = *(const dn_f4 *)(g.mu + k);
#pragma unroll
                for (int e = 0; e < 4; e++) v[e] += (b[e] - v[e]) * m[e];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] *= scale;
                if constexpr (sizeof(WT) == 2) v[e] = dn_bf2f(dn_f2bf(v[e]));
            }
            *(dn_f4 *)(xs + k) = v;
        }
        return;
    }
#pragma unroll 4
    for (int k = threadIdx.x; k < kp; k += 512) {
        float v = k < K ? x[k] * scale : 0.f;
        if (prev && k < K) v += (prev[k] - v) * g.mu[k];
        if constexpr (sizeof(WT) == 2) v = dn_bf2f(dn_f2bf(v));
        xs[k] = v;
    }
}
// one unit: 16 bytes of weights against the same places of x
template <typename WT>
static __device__ __forceinline__ float dn_unit(float acc, const dn_f4 &raw, const float *x) {
    if constexpr (sizeof(WT) == 2) {
        const dn_f4 x0 = *(const dn_f4 *)x, x1 = *(const dn_f4 *)(x + 4);
        unsigned h[4];
        __builtin_memcpy(h, &raw, 16);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            acc = fmaf(__uint_as_float(h[e] << 16), e < 2 ? x0[2 * e] : x1[2 * e - 4], acc);
            acc = fmaf(__uint_as_float(h[e] & 0xffff0000u), e < 2 ? x0[2 * e + 1] : x1[2 * e - 3], acc);
        }
    } else {
        const dn_f4 x0 = *(const dn_f4 *)x;
#pragma unroll
        for (int e = 0; e < 4; e++) acc = fmaf(raw[e], x0[e], acc);
    }
    return acc;
}
static __device__ __forceinline__ float dn_wave_sum(float v) { // every lane gets it: rotations inside a row of sixteen, then the four rows' sums
    auto ror = [](float x, auto n) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + decltype(n)::value, 0xf, 0xf, true)); };
    v += ror(v, std::integral_constant<int, 8>());
    v += ror(v, std::integral_constant<int, 4>());
    v += ror(v, std::integral_constant<int, 2>());
    v += ror(v, std::integral_constant<int, 1>());
    auto row = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
    return (row(0) + row(16)) + (row(32) + row(48));
}

// One vector into LDS through what stands in front of the product (ps_seq.h psk_dense_pre), by all 512 threads: a thread's up to four runs of four numbers, 2048 apart.  All of it is requested in
// front of the weights (dn_pre_request), whose way from memory covers the sums.  A boundary of 2048 numbers and the first product behind it 4.6 + 10.1 us -> 10.9, 4.6 + 5.9 -> 6.8 (kernel trace).
struct dn_pre_runs { dn_f4 x[4], z[4], w[4]; };
template <int PRE>
static __device__ __forceinline__ void dn_pre_request(const dn_args &g, const psk_dense_pre &r, dn_pre_runs &o) {
    const int K = (int)g.K, tid = threadIdx.x;
    const float *second = PRE == psk_dense_pre::BOUNDARY ? r.y : r.gate;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int k = (tid + 512 * j) * 4;
        const bool in = k < K;
        o.x[j] = in ? *(const dn_f4 *)(g.a + k) : dn_f4{0.f, 0.f, 0.f, 0.f};
        o.z[j] = in ? *(const dn_f4 *)(second + k) : dn_f4{0.f, 0.f, 0.f, 0.f};
        o.w[j] = in ? *(const dn_f4 *)(r.w + (PRE == psk_dense_pre::HEADS ? k / r.part * r.w_stride + k % r.part : k)) : dn_f4{0.f, 0.f, 0.f, 0.f};
    }
}
template <typename WT, int PRE>
static __device__ __forceinline__ void dn_stage_pre(const dn_args &g, const psk_dense_pre &r, dn_pre_runs &o, float *xs) {
    __shared__ float red[32];
    const int K = (int)g.K, tid = threadIdx.x, runs = (K + 2047) / 2048;
    auto &x = o.x;
    auto &z = o.z;
    auto &w = o.w;
    float s[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        s[j] = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float v = PRE == psk_dense_pre::BOUNDARY ? z[j][e] : x[j][e];
            s[j] = fmaf(v, v, s[j]);
        }
    }
    if (PRE == psk_dense_pre::HEADS) { // (a head: part / 4 lanes of a wave)
        for (int o = r.part / 8; o > 0; o >>= 1)
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j < runs) s[j] += __shfl_xor(s[j], o, 64);
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (j < runs) {
                const float t = dn_wave_sum(s[j]);
                if ((tid & 63) == 0) red[8 * j + (tid >> 6)] = t;
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j >= runs) continue;
            s[j] = 0.f;
            for (int q = 0; q < K / 256; q++) s[j] += red[q];
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int k = (tid + 512 * j) * 4;
        if (k >= K) continue;
        const float inv = 1.f / sqrtf(s[j] / (float)(PRE == psk_dense_pre::BOUNDARY ? K : r.part) + r.eps);
        dn_f4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (PRE == psk_dense_pre::HEADS) v[e] = x[j][e] * inv * w[j][e] * dn_silu(z[j][e]);
            else v[e] = x[j][e] + z[j][e] * inv * (r.offset + w[j][e]);
        }
        if (PRE == psk_dense_pre::BOUNDARY && blockIdx.x == 0) *(dn_f4 *)(r.xout + k) = v;
        if constexpr (sizeof(WT) == 2) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = dn_bf2f(dn_f2bf(v[e]));
        }
        *(dn_f4 *)(xs + k) = v;
    }
}
template <typename WT, int FORM, bool RAGGED, int PRE = 0> // RAGGED: a row ends inside a unit; PRE: psk_dense_pre (whole units)
__global__ __launch_bounds__(512, 4) void dense_mv1_kernel(dn_args g0, dn_mv1 p) {
    extern __shared__ __attribute__((aligned(16))) float xs[];
    constexpr int VE = 16 / (int)sizeof(WT), UNIT = 64 * VE; // elements per lane and per unit
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int y = FORM == 1 ? min((int)blockIdx.x / p.blocks, p.slots) : FORM == 2 ? (int)blockIdx.x / p.blocks : 0;
    const bool shared_seg = FORM == 1 && y == p.slots;
    dn_args g = g0;
    int sel = 0;
    if constexpr (FORM == 1) { // (field by field: the same K, activation and addition in both)
        g.w = shared_seg ? p.g2.w : g0.w;
        g.N = shared_seg ? p.g2.N : g0.N;
        g.a = shared_seg ? p.g2.a : g0.a;
        g.out = shared_seg ? p.g2.out : g0.out;
        g.ldo = shared_seg ? p.g2.ldo : g0.ldo;
        g.out_scale = shared_seg ? p.g2.out_scale : g0.out_scale;
        g.bias = shared_seg ? p.g2.bias : g0.bias;
        g.alpha = shared_seg ? p.g2.alpha : g0.alpha;
        sel = shared_seg ? 0 : g.g_sel[y];
    }
    if constexpr (FORM == 2) {
        g.w = y == 0 ? p.w[0] : y == 1 ? p.w[1] : y == 2 ? p.w[2] : p.w[3];
        g.mu += (long long)y * g.K;
        g.out += (long long)y * g.N;
    }
    const bool has = FORM != 1 || shared_seg || sel < g.groups; // (an identity expert has no matrix: its rows are zero)
    const int row_units = has ? p.kp / UNIT : 0, N = (int)g.N, K = (int)g.K;
    const bool pair = g.act == PSD_ACT_SILU_PAIR || g.act == PSD_ACT_RELU_PAIR;
    // this wave's rows: first + k step (pairs: first + (k / 2) step + k % 2), k < rows
    const int bx = FORM ? (int)blockIdx.x - y * p.blocks : (int)blockIdx.x, nb = FORM ? (shared_seg ? p.blocks2 : p.blocks) : (int)gridDim.x;
    const int step = nb * 8 * (pair ? 2 : 1), first = (bx * 8 + wave) * (pair ? 2 : 1);
    const int rows = first >= N ? 0 : pair ? ((N - first + step - 2) / step) * 2 : (N - first + step - 1) / step;
    auto row_of = [&](int k) { return pair ? first + (k >> 1) * step + (k & 1) : first + k * step; };
    // the load side of the stream: row lk, unit lu
    int lk = -1, lu = 0;
    const char *lp = nullptr, *lrow = nullptr;
    // this lane's bytes of a row's last unit lie behind the row's end: it reads the row's first ones and puts them aside (an infinite weight times a zero activation is no number)
    const bool beyond = RAGGED && (row_units - 1) * UNIT + lane * VE >= K;
    const WT *mat = (const WT *)g.w + (FORM != 1 || shared_seg ? 0 : (long long)sel * g.wstride);
    auto open = [&]() {
        if (++lk >= rows) return;
        lrow = (const char *)(mat + (long long)row_of(lk) * K);
        lp = lrow + lane * 16;
        lu = 0;
    };
    auto request = [&](dn_f4 &v) {
        if (lk >= rows) return; // (uniform)
        const char *q = beyond && lu == row_units - 1 ? lrow : lp;
        v = __builtin_nontemporal_load((const dn_f4 *)q);
        lp += 1024;
        if (++lu == row_units) open();
    };
    dn_f4 ring[DN_AHEAD];
    dn_pre_runs pre;
    if constexpr (PRE) {
        dn_pre_request<PRE>(g, p.pre, pre);
        asm volatile("" ::: "memory"); // (in front of the weights)
    }
    if (rows && row_units) {
        open();
#pragma unroll
        for (int u = 0; u < DN_AHEAD; u++) request(ring[u]);
    }
    // the activations
    if constexpr (PRE) {
        dn_stage_pre<WT, PRE>(g, p.pre, pre, xs);
    } else if constexpr (FORM != 1) {
        long long row0;
        int T;
        dn_rows(g, row0, T);
        dn_stage<WT>(g, dn_arow(g, row0, 0), g.mu ? g.shift0 : nullptr, 1.f, xs, p.kp);
    } else {
        if (shared_seg) dn_stage<WT>(g, g.a, nullptr, 1.f, xs, p.kp);
        else dn_stage<WT>(g, g.a + (long long)(y / g.g_adiv) * g.lda, nullptr, g.g_scale ? g.g_scale[y] : 1.f, xs, p.kp);
    }
    __syncthreads();
    // the other side: cu units of the row left; lane k % 64 keeps row k's result until 64 of them are there or the rows are through
    int cu = row_units, done = 0, kept = 0;
    const float *xp = xs + lane * VE;
    float acc = 0.f, res = 0.f;
    auto eat = [&](dn_f4 &v) {
        if (RAGGED && cu == 1) v = beyond ? dn_f4{0.f, 0.f, 0.f, 0.f} : v;
        acc = dn_unit<WT>(acc, v, xp);
        request(v);
        xp += UNIT;
        if (--cu) return;
        const float s = dn_wave_sum(acc);
        res = lane == done - kept ? s : res;
        done++;
        acc = 0.f;
        cu = row_units;
        xp = xs + lane * VE;
    };
    auto put = [&]() { // the results of rows kept .. done - 1
        const int k = kept + lane;
        const float v = res;
        dn_put(g, FORM != 1 || shared_seg ? 0 : y, row_of(k), v, __shfl_xor(v, 1, 64), k < done);
        kept = done;
    };
    if (row_units) {
        int left = rows * row_units;
        for (; left >= DN_AHEAD; left -= DN_AHEAD) {
#pragma unroll
            for (int q = 0; q < DN_AHEAD; q++) eat(ring[q]);
            if (done - kept > 64 - DN_AHEAD - 2) { // (kept stays even for pairs)
                const int odd = (done - kept) & 1;
                if (!pair || !odd) put();
            }
        }
#pragma unroll
        for (int q = 0; q < DN_AHEAD; q++)
            if (q < left) eat(ring[q]);
        put();
    } else {
        for (done = min(rows, 64); kept < rows; done = min(done + 64, rows)) put();
    }
}

// Work-groups of eight waves: enough that every wave has a row, at most two per CU (one where the activations are long: each group stages them for itself).
template <typename WT, int FORM>
static bool dn_launch_mv1(hipStream_t st, const dn_args &g, const dn_args *g2, int slots, const psk_dense_args *a = nullptr) {
    constexpr int UNIT = 64 * 16 / (int)sizeof(WT);
    dn_mv1 p;
    if (g2) p.g2 = *g2;
    else { p.g2 = g; p.g2.w = nullptr; }
    p.slots = slots;
    p.kp = (int)((g.K + UNIT - 1) / UNIT * UNIT);
    const size_t lds = (size_t)p.kp * 4;
    if ((g.K * (int64_t)sizeof(WT)) % 16 != 0 || lds > 128 * 1024 || g.N > (1 << 28) || (g2 && (g2->K != g.K || g2->act != g.act || g2->accum != g.accum || g2->N > (1 << 28)))) return false;
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) {
        (void)hipFuncSetAttribute((const void *)dense_mv1_kernel<WT, FORM, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void *)dense_mv1_kernel<WT, FORM, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    }
    const int per = g.act == PSD_ACT_SILU_PAIR || g.act == PSD_ACT_RELU_PAIR ? 16 : 8; // rows that a work-group takes at once
    const int64_t most = lds <= 72 * 1024 ? 512 : 256;
    int64_t grid = std::min<int64_t>((g.N + per - 1) / per, most);
    if (FORM == 1) { // the same number of rows for every work-group of every matrix
        const int64_t all = g.N * slots + (g2 ? g2->N : 0);
        int64_t rounds = std::max<int64_t>((all + most * per - 1) / (most * per), 1);
        do { // (a round more where the matrices' last ones would add up to a work-group too many)
            p.blocks = (int)((g.N + rounds * per - 1) / (rounds * per));
            p.blocks2 = g2 ? (int)((g2->N + rounds * per - 1) / (rounds * per)) : 0;
            grid = (int64_t)p.blocks * slots + p.blocks2;
            rounds++;
        } while (grid > most && (p.blocks > 1 || p.blocks2 > 1));
    }
    if (FORM == 2) {
        const int n = 1 + a->n_more;
        p.blocks = (int)std::max<int64_t>(std::min<int64_t>((g.N + per - 1) / per, most / n), 1);
        grid = (int64_t)p.blocks * n;
        for (int i = 0; i < n; i++) p.w[i] = i ? a->more[i - 1]->data : g.w;
    }
    const auto kernel = p.kp == g.K ? dense_mv1_kernel<WT, FORM, false> : dense_mv1_kernel<WT, FORM, true>;
    if constexpr (FORM == 0) {
        if (a && a->pre.kind) {
            p.pre = a->pre;
            const auto with = p.pre.kind == psk_dense_pre::HEADS ? dense_mv1_kernel<WT, 0, false, psk_dense_pre::HEADS> : dense_mv1_kernel<WT, 0, false, psk_dense_pre::BOUNDARY>;
            hipLaunchKernelGGL(with, dim3((unsigned)grid), dim3(512), lds, st, g, p); // (at most 32 KB of activations: no attribute)
            return true;
        }
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(512), lds, st, g, p);
    return true;
}

// The second product of a token's experts: an output row is the sum over the token's slots (and the shared expert) of the products with their matrices, so a row runs through all of
// them.  `waves` waves of a work-group share a row, each with the same up to U units of it, so that a wave's part of the activations (up to top + 1 vectors of different experts) stays in
// its registers and nothing waits for a copy of all of them in LDS; a row of each wave is in flight (two units at least), across row ends.  The waves' sums of a row meet in LDS at the end.
// blockIdx.y = token.  Top 2 of 2048 x 3072 and a shared one of twice that (50 MB), one token: 16.6 us and 17.5 us more for the shared expert before, 18.0 as one stream with the activations in LDS
// (as above), 14.3 then; 13.9 since the weights are requested in front of what is done to the activations.  The form above is the better one where there is a single vector: 2048 x 4096 6.6 us there, 9 with this kernel's arrangement.
// dynamic LDS: [8][rows] sums
struct dn_mv2 {
    dn_args g2; // the shared expert's second product (w NULL: none; only w, a, lda, K, out_scale are read)
    int slots;  // per token
    int units, units2; // of a row of a slot's matrix, of the shared expert's
    int waves, share;  // waves per row, units per wave
    int rows;          // the most rows that a group of waves has
};
template <typename WT, int U, bool RAGGED> // RAGGED: a row ends inside a unit
__global__ __launch_bounds__(512, U > 8 ? 2 : 4) void dense_mv2_kernel(dn_args g, dn_mv2 p) {
    extern __shared__ __attribute__((aligned(16))) float sums[];
    constexpr int VE = 16 / (int)sizeof(WT), UNIT = 64 * VE, AHEAD = U >= 3 ? 1 : 4 / U; // elements per lane and per unit; rows in flight
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), y = blockIdx.y;
    const int sel = lane < p.slots ? g.g_sel[(long long)y * p.slots + lane] : 0; // lane c: slot c's matrix
    const int N = (int)g.N, K = (int)g.K, K2 = (int)p.g2.K;
    // this wave's rows: first + k step, k < rows
    const int groups = 8 / p.waves, part = wave % p.waves, step = (int)gridDim.x * groups;
    auto first_of = [&](int gi) { return (int)blockIdx.x * groups + gi; };
    auto rows_of = [&](int gi) { return first_of(gi) >= N ? 0 : (N - first_of(gi) + step - 1) / step; };
    const int first = first_of(wave / p.waves), rows = rows_of(wave / p.waves);
    // this wave's units: where unit u of row 0 starts, its activations (a lane beyond the row's end reads the unit's first bytes and puts
    // them aside: an infinite weight times a zero activation is no number)
    const int all = p.slots * p.units + p.units2, u0 = part * p.share, n_units = max(min(p.share, all - u0), 0);
    const char *base[U];
    bool has[U], second[U]; // (a slot without a matrix -- an identity expert -- has none; second: the shared expert's)
    int lo[U];
    float x[U][VE], f[U];
    bool in[U];
    // (requests only, the weights' behind them: what is done to the activations waits for them alone and runs while the weights are on their way)
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int c = min((u0 + u) / p.units, p.slots), at = u0 + u - c * p.units; // slot, unit of a row of its matrix
        second[u] = c == p.slots;
        has[u] = u < n_units;
        const float *xr = p.g2.a + (long long)y * p.g2.lda;
        const WT *w = (const WT *)p.g2.w;
        f[u] = 1.f;
        if (!second[u]) {
            const int s = y * p.slots + c, m = __builtin_amdgcn_readlane(sel, min(c, 63));
            has[u] = has[u] && m < g.groups;
            xr = g.a + (long long)(s / g.g_adiv) * g.lda;
            w = (const WT *)g.w + (long long)m * g.wstride;
            if (g.g_scale && has[u]) f[u] = g.g_scale[s];
        }
        const int k = at * UNIT + lane * VE, Kc = second[u] ? K2 : K;
        in[u] = has[u] && k < Kc;
        lo[u] = !RAGGED || k < Kc ? lane * 16 : 0;
        base[u] = (const char *)(w + (long long)at * UNIT);
        const float *xk = xr + (in[u] ? k : 0); // (the row's first numbers are there whatever is asked for)
        if (((uintptr_t)xr & 15) == 0) { // (uniform)
#pragma unroll
            for (int e = 0; e < VE; e += 4) {
                const dn_f4 v = *(const dn_f4 *)(xk + (in[u] ? e : 0));
#pragma unroll
                for (int i = 0; i < 4; i++) x[u][e + i] = v[i];
            }
        } else {
#pragma unroll
            for (int e = 0; e < VE; e++) x[u][e] = xk[in[u] ? e : 0];
        }
    }
    float ident = 0.f; // the summed weights of the token's slots that have no matrix
    if (g.g_ident)
        for (int c = 0; c < p.slots; c++)
            if ((int)__builtin_amdgcn_readlane(sel, c) >= g.groups) ident += g.g_ident_w[y * p.slots + c];
    const float shared_scale = p.g2.w && p.g2.out_scale ? p.g2.out_scale[y] : 1.f;
    dn_f4 ring[AHEAD][U];
    auto request = [&](dn_f4 (&v)[U], int k) {
        if (k >= rows) return; // (uniform)
        const long long r = first + (long long)k * step;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (has[u]) v[u] = __builtin_nontemporal_load((const dn_f4 *)(base[u] + r * ((second[u] ? K2 : K) * (int)sizeof(WT)) + lo[u]));
    };
#pragma unroll
    for (int d = 0; d < AHEAD; d++) request(ring[d], d);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
        for (int e = 0; e < VE; e++) {
            x[u][e] = in[u] ? x[u][e] * f[u] : 0.f;
            if constexpr (sizeof(WT) == 2) x[u][e] = dn_bf2f(dn_f2bf(x[u][e]));
        }
    for (int k0 = 0; k0 < rows; k0 += AHEAD) {
#pragma unroll
        for (int d = 0; d < AHEAD; d++) {
            const int k = k0 + d;
            if (k >= rows) break;
            float acc = 0.f, own = 0.f;
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (!has[u]) continue;
                if (RAGGED && lo[u] != lane * 16) ring[d][u] = dn_f4{0.f, 0.f, 0.f, 0.f};
                float a = second[u] ? own : acc;
                if constexpr (sizeof(WT) == 2) {
                    unsigned h[4];
                    __builtin_memcpy(h, &ring[d][u], 16);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        a = fmaf(__uint_as_float(h[e] << 16), x[u][2 * e], a);
                        a = fmaf(__uint_as_float(h[e] & 0xffff0000u), x[u][2 * e + 1], a);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) a = fmaf(ring[d][u][e], x[u][e], a);
                }
                if (second[u]) own = a;
                else acc = a;
            }
            request(ring[d], k + AHEAD);
            acc = dn_wave_sum(fmaf(own, shared_scale, acc));
            if (lane == 0) sums[wave * p.rows + k] = acc;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < groups * p.rows; i += 512) {
        const int gi = i / p.rows, k = i - gi * p.rows, n = first_of(gi) + k * step;
        if (k >= rows_of(gi)) continue;
        float v = 0.f;
        for (int q = 0; q < p.waves; q++) v += sums[(gi * p.waves + q) * p.rows + k];
        if (ident != 0.f) v = fmaf(ident, g.g_ident[(long long)y * g.g_ident_ld + n], v);
        dn_put(g, y, n, v, 0.f, true);
    }
}

// Work-groups of eight waves, at most two per CU.  As few waves per row as keep four units of it per wave or less (fewer sums to make, 32 registers of activations), but as many as it
// takes for 4096 waves to have a row.
template <typename WT>
static bool dn_launch_mv2(hipStream_t st, const dn_args &g, const dn_args *g2, int slots, int tokens) {
    constexpr int UNIT = 64 * 16 / (int)sizeof(WT), MOST = sizeof(WT) == 2 ? 8 : 16;
    dn_mv2 p;
    if (g2) p.g2 = *g2;
    else { p.g2 = g; p.g2.w = nullptr; }
    if ((g.K * (int64_t)sizeof(WT)) % 16 != 0 || (g2 && (g2->K * (int64_t)sizeof(WT)) % 16 != 0) || g.K > (1 << 20) || p.g2.K > (1 << 20) || g.N > (1 << 28) || slots > 63) return false;
    p.slots = slots;
    p.units = (int)((g.K + UNIT - 1) / UNIT);
    p.units2 = g2 ? (int)((g2->K + UNIT - 1) / UNIT) : 0;
    const int units = slots * p.units + p.units2;
    p.waves = 1;
    while (p.waves < 8 && ((units + p.waves - 1) / p.waves > 4 || (g.N * tokens * p.waves < 4096 && p.waves < units))) p.waves *= 2;
    p.share = (units + p.waves - 1) / p.waves;
    if (p.share > MOST) return false;
    const int per = 8 / p.waves; // rows that a work-group takes at once
    const int64_t once = (g.N + per - 1) / per, grid = std::max(std::min<int64_t>(once, std::max(512 / tokens, 64)), (once + 1023) / 1024); // (at most 1024 rounds: 32 KiB of sums)
    p.rows = (int)((once + grid - 1) / grid);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid, (unsigned)tokens), dim3(512), (size_t)8 * p.rows * 4, st, g, p); };
    auto pick = [&](auto ragged) {
        constexpr bool R = decltype(ragged)::value;
        if (p.share == 1) go(dense_mv2_kernel<WT, 1, R>);
        else if (p.share == 2) go(dense_mv2_kernel<WT, 2, R>);
        else if (p.share == 3) go(dense_mv2_kernel<WT, 3, R>);
        else if (p.share <= 4) go(dense_mv2_kernel<WT, 4, R>);
        else if (p.share <= 8) go(dense_mv2_kernel<WT, 8, R>);
        else if constexpr (sizeof(WT) == 4) go(dense_mv2_kernel<WT, 16, R>);
    };
    if (g.K % UNIT || (g2 && g2->K % UNIT)) pick(std::true_type());
    else pick(std::false_type());
    return true;
}

template <typename WT, int C, int RW = 4>
static void dn_launch_mv(hipStream_t st, const dn_args &g) {
    const size_t lds = (size_t)C * ((g.K + 7) / 8 * 8) * 4;
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)dense_mv_kernel<WT, C, RW>, hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024);
    long long blocks = (g.N + 4 * RW - 1) / (4 * RW);
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL((dense_mv_kernel<WT, C, RW>), dim3((unsigned)blocks), dim3(256), lds, st, g);
}

static dn_args dn_make(const psk_dense_args &a) {
    dn_args g;
    g.w = a.w->data; g.a = a.a; g.lda = a.lda; g.a_row0 = a.a_row0; g.a_mod = a.a_mod; g.a_step = a.a_step; g.T = a.T;
    g.N = a.w->N; g.K = a.w->K; g.out = a.out; g.out16 = (unsigned short *)a.out16; g.ldo = a.ldo; g.bias = a.bias; g.act = a.act; g.act_p = a.act_p; g.act_q = a.act_q;
    g.alpha = a.alpha; g.mu = a.mu; g.shift0 = a.shift0; g.accum = a.accum; g.out_scale = a.out_scale;
    g.groups = 0; g.g_adiv = 1; g.g_odiv = 1; g.g_inner = 1; g.g_sel = nullptr; g.g_seg = nullptr; g.g_list = nullptr; g.g_scale = nullptr; g.wstride = 0;
    g.g_ident = a.g_ident; g.g_ident_w = a.g_ident_w; g.g_ident_ld = a.g_ident_ld;
    g.em_table = a.em_table ? a.em_table->data : nullptr; g.em_bf16 = a.em_table && a.em_table->dtype == PS_BF16; g.em_ld = a.em_table ? a.em_table->K : 0;
    g.em_col = a.em_col; g.em_tokens = a.em_tokens; g.em_step = a.em_step;
    return g;
}
// a few slots' grouped product as one streaming mat-vec, the shared expert's with it where there is one and it fits: 0 not taken, 1 the slots alone, 2 both
template <typename WT>
static int dn_grouped_mv1(hipStream_t st, const psk_dense_args &a, const dn_args &g) {
    const bool second = g.act == PSD_ACT_NONE; // an output row per token, the sum over its slots; an expert's first product: one per slot
    if (!second && (a.g_inner != 1 || a.g_ident)) return 0;
    if (a.also && a.also->w->dtype == a.w->dtype && (second || a.also->T == 1)) {
        const dn_args g2 = dn_make(*a.also);
        if (second ? dn_launch_mv2<WT>(st, g, &g2, a.g_inner, a.T) : dn_launch_mv1<WT, 1>(st, g, &g2, a.T)) return 2;
    }
    // Alone, the second product is the grouped kernel's where that walks a row in a few trips (two pieces of each slot's matrix at a time) and a token's matrices are not large: measured for one
    // token and eight, us here and there: 2048 x 1024 of two slots 8.0 / 20.0 and 6.8 / 12.9 (two trips), 2048 x 2048 11.9 / 29.1 and 9.7 / 24.7 (four), 2048 x 3072 12.1 / 29.7 and
    // 12.2 / 32.0 (six), 4096 x 2048 14.3 / 45.9 and 13.2 / 50.3 (four, 33 MB), 1024 x 512 of six slots 8.0 / 13.1 and 10.2 / 12.9 (six).
    constexpr int64_t TRIP = 128 * 16 / (int64_t)sizeof(WT);
    if (second && a.g_inner * ((g.K + TRIP - 1) / TRIP) < 6 && g.N * g.K * a.g_inner * (int64_t)sizeof(WT) < ((int64_t)32 << 20)) return 0;
    return (second ? dn_launch_mv2<WT>(st, g, nullptr, a.g_inner, a.T) : dn_launch_mv1<WT, 1>(st, g, nullptr, a.T)) ? 1 : 0;
}

bool psk_dense_takes_pre(const psk_dense_args &a) {
    auto aligned = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
    if (!a.w || a.T != 1 || a.force_tiled || a.groups || a.mu || a.a_mod || a.a_step || a.a_row0 || a.n_more || a.w->N > (1 << 28)) return false;
    const int64_t K = a.w->K, unit = a.w->dtype == PS_BF16 ? 512 : 256; // (whole units of the stream; four runs a thread)
    const psk_dense_pre &r = a.pre;
    if (K % unit || K > 8192 || !aligned(a.a) || !aligned(r.w)) return false;
    // (heads: a token of six Ranutar layers in us, a launch in front | in the product: 1024 channels 259 | 249, 1536 285 | 277, 2048 343 | 335, 2560 396 | 392, 3072 424 | 421, three of 4096 314 | 312 in one
    // measurement, 335 | 336 in another: 4096 numbers and as many of the gate read by 512 work-groups take what the launch did)
    if (r.kind == psk_dense_pre::HEADS) return K <= 2048 && aligned(r.gate) && r.part >= 4 && r.part <= 256 && (r.part & (r.part - 1)) == 0 && K % r.part == 0 && r.w_stride % 4 == 0;
    return r.kind == psk_dense_pre::BOUNDARY && aligned(r.y) && aligned(r.xout) && r.xout != a.a;
}
bool psk_dense_wide16(const psk_dense_args &a) {
    return a.w && a.w->dtype == PS_BF16 && a.T > PSD_FEW && !a.force_tiled && a.pack && a.groups == 0 && !a.mu && !a.a_mod && !a.a_step && !a.a_row0 && a.w->K > 256 && a.w->K % 64 == 0 &&
           (size_t)a.T * a.w->K * 2 <= a.pack_bytes;
}
bool psk_dense_listed16(const psk_dense_args &a) { // (as dn_ring_take)
    return a.w && a.w->dtype == PS_BF16 && a.groups > 0 && a.g_list && !a.force_tiled && a.pack && a.w->K % 64 == 0 && (size_t)a.T * a.w->K * 2 <= a.pack_bytes;
}
// fp32 products of two to four tokens that the mat-vec takes first, though the wide mat-mul takes them: its launches (packing, product, sum) against a second column of the streamed rows.  us there and
// here, weights from memory (bf16 ones stay there: 4096 x 2048 14.9 and 13.1 alone, but a layer's rows come rounded, and whole requests of two tokens are 1 to 4 % faster with the wide one):
//   two tokens, 2048 x 768 11.0 and 7.9, 4096 x 2048 18.2 and 13.8, 4096 x 4096 30.3 and 24.9, but 512 x 4096 12.7 and 14.5; in three lines 11.8 and 7.9, 18.3 and 13.8, 2048 x 3072 15.7 and 14.6, but
//   4096 x 4096 21.6 and 24.9;  three and four, without the lines, 8192 x 2048 30.7 and 23.7, 30.7 and 24.9, but 2048 x 2048 14.2 and 15.6, 14.2 and 16.7
static bool dn_few_first(const psk_dense_args &a, const dn_args &g) {
    if (a.T < 2 || a.T > 4 || a.a16 || a.out16) return false; // (rounded rows are the wide one's to read and to write)
    if (a.w->dtype == PS_BF16) return false;
    if (a.w->half) return a.T == 2 && g.K <= 3072;
    return a.T == 2 ? g.K <= 2048 || 4 * g.N >= g.K : g.N >= 4 * g.K;
}
int psk_dense(hipStream_t st, const psk_dense_args &a) {
    if (!a.w || a.T <= 0) return 0;
    dn_args g = dn_make(a);
    const bool bf = a.w->dtype == PS_BF16;
    if (a.n_more) { // together where the streaming mat-vec or the wide mat-mul takes them, else one by one.  512 tokens, four of 2048 x 2048: 5.5 + 13.5 us each one by one, 6.0 + 30.0 together
        bool alike = true;
        for (int i = 0; i < a.n_more; i++) alike = alike && a.more[i]->dtype == a.w->dtype && a.more[i]->N == a.w->N && a.more[i]->K == a.w->K;
        if (alike && !a.force_tiled && a.T == 1 && (bf ? dn_launch_mv1<unsigned short, 2>(st, g, nullptr, 0, &a) : dn_launch_mv1<float, 2>(st, g, nullptr, 0, &a))) return 0;
        if (alike && a.T > PSD_FEW && dn_wide(st, a, g)) return 0;
        for (int i = 0; i <= a.n_more; i++) {
            psk_dense_args one = a;
            one.n_more = 0;
            if (i) one.w = a.more[i - 1];
            one.mu = a.mu + i * a.w->K;
            one.out = a.out + i * a.w->N;
            psk_dense(st, one);
        }
        return 0;
    }
    const size_t kp4 = (size_t)((g.K + 7) / 8 * 8) * 4;
    if (a.groups > 0) {
        g.groups = a.groups; g.N = a.w->N / a.groups; g.wstride = g.N * g.K;
        g.g_adiv = a.g_adiv; g.g_odiv = a.g_odiv; g.g_inner = a.g_inner; g.g_sel = a.g_sel; g.g_scale = a.g_scale;
        if (!a.g_list) { // a few slots
            const int took = bf ? dn_grouped_mv1<unsigned short>(st, a, g) : dn_grouped_mv1<float>(st, a, g);
            if (took) return took == 2;
            const int64_t waves4 = (g.N + 3) / 4 * a.T; // four rows per wave only where that still leaves about 1024 waves (a gate / up pair sits in one wave)
            const int RW = waves4 >= 1024 ? 4 : waves4 >= 512 || g.act == PSD_ACT_SILU_PAIR || g.act == PSD_ACT_RELU_PAIR ? 2 : 1;
            const auto launch = bf ? (RW == 4 ? dn_launch_mv_grouped<unsigned short, 4> : RW == 2 ? dn_launch_mv_grouped<unsigned short, 2> : dn_launch_mv_grouped<unsigned short, 1>)
                                   : (RW == 4 ? dn_launch_mv_grouped<float, 4> : RW == 2 ? dn_launch_mv_grouped<float, 2> : dn_launch_mv_grouped<float, 1>);
            launch(st, g, a.T, kp4 * a.g_inner);
            return 0;
        }
        g.g_seg = a.g_seg; g.g_list = a.g_list;
        if (dn_wide(st, a, g)) return 0;
        const dim3 grid((unsigned)((g.N + 63) / 64), (unsigned)((a.T + 63) / 64), (unsigned)a.groups);
        if (bf) hipLaunchKernelGGL(dense_mm_kernel<unsigned short>, grid, dim3(256), 0, st, g);
        else hipLaunchKernelGGL(dense_mm_kernel<float>, grid, dim3(256), 0, st, g);
        return 0;
    }
    auto few = [&]() { // the mat-vecs, where they take the product
        if (a.force_tiled || a.T > 8) return false;
        if (a.T == 1 && (bf ? dn_launch_mv1<unsigned short, 0>(st, g, nullptr, 0, &a) : dn_launch_mv1<float, 0>(st, g, nullptr, 0, &a))) return true;
        const int C = a.T <= 1 ? 1 : a.T <= 2 ? 2 : a.T <= 4 ? 4 : 8;
        if (kp4 * C <= 64 * 1024) {
            // (a token's rows that the stream does not take: four per wave would leave at most 64 blocks.  1004 x 4102 14.2 us, with one per wave 11.9; 512 x 1026 6.7 and 5.3)
            const bool one_row = C == 1 && g.N <= 1024 && g.act != PSD_ACT_SILU_PAIR && g.act != PSD_ACT_RELU_PAIR;
            if (one_row) {
                if (bf) dn_launch_mv<unsigned short, 1, 1>(st, g);
                else dn_launch_mv<float, 1, 1>(st, g);
            } else if (bf) {
                if (C == 1) dn_launch_mv<unsigned short, 1>(st, g);
                else if (C == 2) dn_launch_mv<unsigned short, 2>(st, g);
                else if (C == 4) dn_launch_mv<unsigned short, 4>(st, g);
                else dn_launch_mv<unsigned short, 8>(st, g);
            } else {
                if (C == 1) dn_launch_mv<float, 1>(st, g);
                else if (C == 2) dn_launch_mv<float, 2>(st, g);
                else if (C == 4) dn_launch_mv<float, 4>(st, g);
                else dn_launch_mv<float, 8>(st, g);
            }
            return true;
        }
        return false;
    };
    if (dn_few_first(a, g) && few()) return 0;
    if (!a.force_tiled && a.T > 8 && g.K <= 32 && !g.mu && !g.a_mod && !g.a_step && !g.a_row0) {
        const dim3 grid((unsigned)((g.N + 255) / 256), (unsigned)((a.T + 15) / 16));
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, g); };
        if (g.K <= 8) bf ? go(dense_mm_few_kernel<unsigned short, 8>) : go(dense_mm_few_kernel<float, 8>);
        else bf ? go(dense_mm_few_kernel<unsigned short, 32>) : go(dense_mm_few_kernel<float, 32>);
        return 0;
    }
    // K up to 256, and up to 1024 where the small tiles are not more than one per CU and nobody hands rounded rows on (the ring packs its operand first): us here and there, weights from memory,
    // 2048 x 512: 9 tokens 5.4 and 8.0, 128 tokens 6.7 and 9.0; 1024 x 1024: 9 tokens 7.0 and 9.8, 256 tokens 9.1 and 11.2; 3072 x 1024: 64 tokens (192 tiles) 9.3 and 12.0, 128 tokens
    // (384) 17.1 and 12.0; 2048 x 2048: 16 tokens 13.4 and 13.1, 64 tokens 15.8 and 13.4.
    if (bf && !a.force_tiled && a.T > PSD_FEW && g.K % 128 == 0 && g.lda % 4 == 0 && ((uintptr_t)g.a & 15) == 0 && !g.mu && !g.a_mod && !g.a_step && !g.a_row0 &&
        (g.K <= 256 || (g.K <= 1024 && (int64_t)((a.T + 31) / 32) * ((g.N + 31) / 32) <= 256 && !a.a16 && !a.out16))) {
        const dim3 grid((unsigned)((a.T + 31) / 32), (unsigned)((g.N + 31) / 32));
        auto go = [&](auto kernel, int waves) { hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), 0, st, g); };
        switch (g.K / 128) {
        case 1: go(dense_mm_narrow_kernel<4, 1>, 4); break;
        case 2: go(dense_mm_narrow_kernel<4, 2>, 4); break;
        case 3: go(dense_mm_narrow_kernel<4, 3>, 4); break;
        case 4: go(dense_mm_narrow_kernel<4, 4>, 4); break;
        case 5: go(dense_mm_narrow_kernel<4, 5>, 4); break;
        case 6: go(dense_mm_narrow_kernel<4, 6>, 4); break;
        case 7: go(dense_mm_narrow_kernel<4, 7>, 4); break;
        default: go(dense_mm_narrow_kernel<8, 4>, 8);
        }
        return 0;
    }
    if (a.T > PSD_FEW && dn_wide(st, a, g)) return 0;
    if (few()) return 0;
    dim3 grid((unsigned)((g.N + 63) / 64), (unsigned)((a.T + 63) / 64));
    if (bf) hipLaunchKernelGGL(dense_mm_kernel<unsigned short>, grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL(dense_mm_kernel<float>, grid, dim3(256), 0, st, g);
    return 0;
}

// ---------------------------------------------------------------------------------------------------- upload, embedding, arg-max
__global__ void dense_widen_kernel(const unsigned short *in, long long n, float *out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) out[i] = dn_bf2f(in[i]);
}
__global__ void dense_odd_kernel(const unsigned short *in, long long n, int32_t *odd) { // infinities and NaN
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        if ((in[i] & 0x7f80) == 0x7f80) *odd = 1;
}
void psk_dense_widen(hipStream_t st, const uint16_t *bf16, int64_t n, float *out) {
    long long blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(dense_widen_kernel, dim3((unsigned)blocks), dim3(256), 0, st, bf16, (long long)n, out);
}

static __device__ __forceinline__ float dn_table(const void *table, int is_bf16, long long i) {
    return is_bf16 ? dn_bf2f(((const unsigned short *)table)[i]) : ((const float *)table)[i];
}
// bigram: a second table whose row depends on the previous and the present token (psk_embed)
__global__ void dense_embed_kernel(const void *table, int is_bf16, long long K, const int32_t *tokens, const ps_seq_step *step, float scale, float *out,
                                   long long ldo, const void *bigram, long long buckets, long long mul_prev, long long mul_cur) {
    const int t = blockIdx.x;
    const long long tok = (tokens ? tokens[t] : step->token0);
    long long row = 0;
    if (bigram) {
        const long long prev = t ? tokens[t - 1] : step->prev;
        row = step->pos0 + t == 0 ? buckets : (prev * mul_prev + tok * mul_cur) % buckets;
    }
    for (long long k = threadIdx.x; k < K; k += blockDim.x) {
        const float v = dn_table(table, is_bf16, tok * K + k) * scale;
        out[t * ldo + k] = bigram ? v + dn_table(bigram, is_bf16, row * K + k) : v;
    }
}
void psk_embed(hipStream_t st, const ps_dense *table, const int32_t *tokens, const ps_seq_step *step, int T, float scale, float *out, int64_t ldo, const ps_dense *bigram,
               int64_t buckets, int64_t mul_prev, int64_t mul_cur) {
    hipLaunchKernelGGL(dense_embed_kernel, dim3(T), dim3(T <= 8 && table->K >= 1024 ? 1024 : 256), 0, st, table->data, table->dtype == PS_BF16 ? 1 : 0, (long long)table->K, tokens, step, scale, out,
                       (long long)ldo, bigram ? bigram->data : nullptr, (long long)buckets, (long long)mul_prev, (long long)mul_cur);
}

// index of row's first maximum among `count` numbers (thread 0 has it), by 1024 threads: four numbers per load where the row is aligned (32000 logits: 8.5 us with 256 threads and single numbers, 3.1 now)
static __device__ __forceinline__ int dn_first_max(const float *row, int count, float *bv, int *bi) {
    const int tid = threadIdx.x;
    float best = -INFINITY;
    int at = count;
    auto take = [&](float v, int i) {
        if (v > best || (v == best && i < at)) { best = v; at = i; }
    };
    if (count % 4 == 0 && ((uintptr_t)row & 15) == 0) {
#pragma unroll 4
        for (int i = tid * 4; i < count; i += 4096) {
            const dn_f4 v = *(const dn_f4 *)(row + i);
#pragma unroll
            for (int e = 0; e < 4; e++) take(v[e], i + e);
        }
    } else {
#pragma unroll 4
        for (int i = tid; i < count; i += 1024) take(row[i], i);
    }
    for (int o = 32; o > 0; o >>= 1) take(__shfl_xor(best, o, 64), __shfl_xor(at, o, 64));
    if ((tid & 63) == 0) { bv[tid >> 6] = best; bi[tid >> 6] = at; }
    __syncthreads();
    if (tid < 64) {
        best = tid < 16 ? bv[tid] : -INFINITY;
        at = tid < 16 ? bi[tid] : count;
        for (int o = 8; o > 0; o >>= 1) take(__shfl_xor(best, o, 64), __shfl_xor(at, o, 64));
    }
    return at < count ? at : 0;
}
// A greedy step's end and the next one's beginning in one block (ps_seq.h psk_next_token): the arg-max, the step's numbers and the embedding were three launches of 4 us each, most of it their start.
__global__ __launch_bounds__(1024) void dense_next_kernel(const float *x, long long n, ps_seq_step *step, int32_t *ids, int32_t *prev, const void *table, int is_bf16, long long rows, long long K, float scale, float *out,
                                                          const void *bigram, long long buckets, long long mul_prev, long long mul_cur) {
    __shared__ float bv[16];
    __shared__ int bi[16], id;
    const int before = step->token0, kept = step->_pad; // (thread 0 writes them behind the barrier)
    const int at = dn_first_max(x, (int)n, bv, bi);
    if (threadIdx.x == 0) {
        id = at;
        ids[kept] = at;
        step->prev = before;
        if (prev) *prev = before;
        step->_pad = kept + 1;
        step->token0 = at;
        step->pos0 += 1;
    }
    __syncthreads();
    const long long tok = id, row = bigram ? ((long long)before * mul_prev + tok * mul_cur) % buckets : 0; // (never a sequence's first token)
    for (long long k = threadIdx.x; k < K; k += 1024) {
        const float v = tok < rows ? dn_table(table, is_bf16, tok * K + k) * scale : 0.f; // (the logits may be more than the table's rows)
        out[k] = bigram ? v + dn_table(bigram, is_bf16, row * K + k) : v;
    }
}
void psk_next_token(hipStream_t st, const float *logits, int64_t n, ps_seq_step *step, int32_t *ids, int32_t *prev, const ps_dense *table, float scale, float *out, const ps_dense *bigram,
                    int64_t buckets, int64_t mul_prev, int64_t mul_cur) {
    hipLaunchKernelGGL(dense_next_kernel, dim3(1), dim3(1024), 0, st, logits, (long long)n, step, ids, prev, table->data, table->dtype == PS_BF16 ? 1 : 0, (long long)table->N, (long long)table->K, scale, out,
                       bigram ? bigram->data : nullptr, (long long)buckets, (long long)mul_prev, (long long)mul_cur);
}
// a row's largest logit, the lowest index among equals: a block per row
__global__ __launch_bounds__(1024) void dense_argmax_kernel(const float *x, long long n, int32_t *out) {
    __shared__ float bv[16];
    __shared__ int bi[16];
    const int at = dn_first_max(x + (long long)blockIdx.x * n, (int)n, bv, bi);
    if (threadIdx.x == 0) out[blockIdx.x] = at;
}
void psk_argmax_rows(hipStream_t st, const float *x, int64_t n, int rows, int32_t *out) {
    hipLaunchKernelGGL(dense_argmax_kernel, dim3(rows), dim3(1024), 0, st, x, (long long)n, out);
}

extern "C" {
int ps_hip_dense_upload(ps_hip_ctx *c, const uint16_t *host, int64_t N, int64_t K, int as_f32, ps_dense **out) {
    *out = nullptr;
    if (N <= 0 || K <= 0) PS_FAIL(c, "dense_upload: empty matrix");
    PS_CHECK(c, hipSetDevice(c->device));
    auto w = new ps_dense();
    w->N = N; w->K = K; w->dtype = as_f32 ? PS_F32 : PS_BF16;
    const size_t n = (size_t)N * K;
    uint16_t *raw = nullptr;
    if (hipMalloc((void **)&raw, n * 2 + 64) != hipSuccess) { delete w; PS_FAIL(c, "dense_upload: out of device memory"); }
    if (hipMemcpyAsync(raw, host, n * 2, hipMemcpyHostToDevice, c->stream) != hipSuccess) { (void)hipFree(raw); delete w; PS_FAIL(c, "dense_upload: copy"); }
    // PS_DENSE_F32_LINES keeps the bf16 form for the wide mat-mul (PL 3 there) where all its numbers are finite (an infinite one meets the zeros of the operand's lower lines).
    const bool lines = as_f32 == PS_DENSE_F32_LINES;
    int32_t *odd = (int32_t *)((char *)raw + (n * 2 + 15) / 16 * 16), is_odd = 1;
    if (as_f32) {
        float *f = nullptr;
        if (hipMalloc((void **)&f, n * 4 + 64) != hipSuccess) { (void)hipFree(raw); delete w; PS_FAIL(c, "dense_upload: out of device memory"); }
        psk_dense_widen(c->stream, raw, (int64_t)n, f);
        w->data = f;
        if (lines) {
            psk_fill(c->stream, (float *)odd, 0.f, 1);
            hipLaunchKernelGGL(dense_odd_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096)), dim3(256), 0, c->stream, raw, (long long)n, odd);
        }
    } else {
        w->data = raw;
    }
    hipError_t e = lines ? hipMemcpyAsync(&is_odd, odd, 4, hipMemcpyDeviceToHost, c->stream) : hipSuccess;
    const hipError_t done = hipStreamSynchronize(c->stream); // (whatever came before: the copy reads and writes memory of this call)
    if (e == hipSuccess) e = done;
    if (as_f32) {
        if (e == hipSuccess && !is_odd) w->half = raw;
        else (void)hipFree(raw);
    }
    if (e != hipSuccess) { (void)hipFree(w->data); delete w; PS_FAIL(c, std::string("dense_upload: ") + hipGetErrorString(e)); }
    *out = w;
    return 0;
}
int ps_hip_dense_f32_form(ps_hip_ctx *c, uint64_t numbers) {
    size_t free = 0, all = 0;
    const bool known = hipSetDevice(c->device) == hipSuccess && hipMemGetInfo(&free, &all) == hipSuccess;
    if (!known) (void)hipGetLastError();
    return known && numbers <= all / 16 ? PS_DENSE_F32_LINES : PS_DENSE_F32;
}
int ps_hip_dense_form(const ps_dense *w) { return w->dtype == PS_BF16 ? PS_DENSE_BF16 : w->half ? PS_DENSE_F32_LINES : PS_DENSE_F32; }
void ps_hip_dense_free(ps_hip_ctx *c, ps_dense *w) {
    if (!w) return;
    if (c) (void)hipStreamSynchronize(c->stream);
    (void)hipFree(w->data);
    if (w->half) (void)hipFree(w->half);
    delete w;
}
int ps_hip_dense_matmul(ps_hip_ctx *c, const ps_dense *w, const float *x, int T, float *out, float alpha) {
    if (!w || T <= 0) PS_FAIL(c, "dense_matmul: bad argument");
    // The wide mat-mul's scratch is the context's and stays with it: 64 MiB of packed rows (128 rows, where those are more) and the parts of split products.  More rows go through it piece
    // by piece, and where the device has no room for it the product does without.  Products that the wide mat-mul does not take need none.
    const bool lines = w->half && w->K % 64 == 0; // (fp32 on the bf16 instruction)
    const int64_t row = w->K * (w->dtype == PS_BF16 ? 2 : lines ? 6 : 4);
    const bool wide = T > PSD_FEW && row % 128 == 0, packs = w->dtype == PS_BF16 || lines || ((uintptr_t)x & 15) != 0;
    const int64_t piece = wide && packs ? std::min<int64_t>(T, std::max<int64_t>(((int64_t)64 << 20) / row / 128 * 128, 128)) : T;
    const size_t pack = packs ? (size_t)(piece * row + 255) / 256 * 256 : 0, need = pack + psk_dense_split_bytes();
    if (wide && c->act_cap < need) {
        PS_CHECK(c, hipStreamSynchronize(c->stream));
        if (c->act_buf) (void)hipFree(c->act_buf);
        c->act_buf = nullptr; c->act_cap = 0;
        if (hipMalloc(&c->act_buf, need) == hipSuccess) c->act_cap = need;
        else { c->act_buf = nullptr; (void)hipGetLastError(); }
    }
    for (int64_t t = 0; t < T; t += piece) {
        psk_dense_args a;
        a.w = w; a.a = x + t * w->K; a.lda = w->K; a.T = (int)std::min<int64_t>(piece, T - t); a.out = out + t * w->N; a.ldo = w->N; a.alpha = alpha;
        if (wide && c->act_buf) {
            a.pack = c->act_buf; a.pack_bytes = pack; a.split = (float *)((char *)c->act_buf + pack); a.split_bytes = psk_dense_split_bytes();
        }
        psk_dense(c->stream, a);
    }
    PS_CHECK(c, hipGetLastError());
    return 0;
}
}
