// Batched mat-mul of Q8_0 / Q4_0 weights against Q8_0 activations (prefill chunks, tree verification) on v_mfma_f32_16x16x4_4b_f16, bit-exact
// (ggml_vec_dot_q8_0_q8_0 / q4_0_q8_0, ggml-quants.c:5761-5782, :4205-4228; the chains of k_gemv.hip's header).
//
// What bounds it: the reference's own fp32 chain.  Every four products meet a multiplier of their own (d_w * d_y of their 32-block), so an output element costs
// K / 4 fmas that nothing can merge -- 15.6 G of them for 512 tokens of the 1B layer pair, against which the operands are few bytes.  The kernel is therefore built so
// that those fmas are nearly all that the vector units do:
//   * the matrix instruction delivers the dot products of four ("quad" u of a 32-block) ALREADY AS FLOATS: K = 4 and four independent products per instruction are the
//     reference's shape exactly (block = u, rows = 16 weight rows, columns = 16 tokens), the operands are small whole numbers in fp16 and every sum is below 2^24, so
//     (float)partial is exact and there is no conversion.  (The form with v_mfma_i32_4x4x4_16B_i8 spends one conversion per fma, and a cross-lane move per multiplier.)
//   * a lane then holds all eight u of (four rows, one column): the four multipliers of a block serve 32 fmas, and hsum_float_8 is in-lane.
//     With the products of a step issued ahead of the fmas of the step before, 86 % of a stage's vector instructions are the reference's own (288 fmas and multipliers of ~335).
//   * the weights go from memory straight to the lane that feeds them (the upload's lane-major pieces ARE the operand order: one 16-byte load per lane is four blocks) and
//     become fp16 in registers, 11 instructions per block and 16 rows, shared by the wave's columns; the activations are converted once per work-group into LDS in operand
//     order and read conflict-free, a stage of 128 elements ahead (a ring of three, one barrier per stage, so that no wave waits for what it has just asked for).
// Measured (Llama-3.2-1B's layer, 511 columns): gate + up 422 -> 236 us, down 249 -> 105, O 31, Q / K / V 84 -> 50 (Q4_0); 14336 x 4096, 511 columns: 659 -> 330 (Q4_0),
// 976 -> 336 (Q8_0).  A wave's stage takes 820 ns, of which the vector unit issues for 740 (an fma of 64 lanes takes four cycles of a SIMD, measured, with one wave 5.7).
#include "ps_gemv_dev.h"

namespace {

typedef _Float16 g8_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 g8_h2 __attribute__((ext_vector_type(2)));
typedef float g8_f16v __attribute__((ext_vector_type(16)));

struct G8W {
    const uint8_t *qs, *aux;
    float *out;
    const float *bias;
    int64_t N, ldo;
    int n_groups, n_tiles; // row groups as stored; tiles of 16 rows
};
struct G8Params {
    G8W w[3];
    int n_w, n_tasks, K, bs;
    const float *residual;
    const int8_t *aq;
    const float *ad;
};

__device__ __forceinline__ uint32_t g8_sub(const uint32_t a, const g8_h2 m) { // two halves minus a constant (exact)
    g8_h2 v;
    __builtin_memcpy(&v, &a, 4);
    v = v - m;
    uint32_t r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}
__device__ __forceinline__ g8_h4 g8_pair(const uint32_t a, const uint32_t b) {
    const uint32_t t[2] = {a, b};
    g8_h4 r;
    __builtin_memcpy(&r, t, 8);
    return r;
}
// four signed bytes -> four halves in the order (0, 2, 1, 3): 1024 + (b + 128) is a half's bits with the byte as its mantissa
__device__ __forceinline__ g8_h4 g8_bytes(const uint32_t w) {
    const uint32_t x = w ^ 0x80808080u;
    const g8_h2 m = {(_Float16)1152.f, (_Float16)1152.f};
    return g8_pair(g8_sub(__builtin_amdgcn_perm(0x64646464u, x, 0x04020400u), m), g8_sub(__builtin_amdgcn_perm(0x64646464u, x, 0x04030401u), m));
}
// low nibbles of four bytes minus 8, same order
__device__ __forceinline__ g8_h4 g8_nibbles(const uint32_t w, const uint32_t e) { // e: 0x64006400 in a vector register (v_and_or_b32 takes one constant)
    const g8_h2 m = {(_Float16)1032.f, (_Float16)1032.f};
    return g8_pair(g8_sub((w & 0x000F000Fu) | e, m), g8_sub(((w >> 8) & 0x000F000Fu) | e, m));
}

// d_w (a half of h) * d_y, rounded once: the product plus +0, which only turns a product of -0 into +0 -- and the chains, which start at +0, cannot tell
__device__ __forceinline__ float g8_scale(const uint32_t h, const float y, const bool high) {
    float d;
    if (high) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(y));
    else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(y));
    return d;
}

// NRW waves of a work-group: 16 weight rows each, all over the same 16 CT columns.  EPI as gemv_kernel's (1: gate rows first, then the same rows of up).
template <int WT, int EPI, int CT, int NRW>
__global__ __launch_bounds__(NRW * 64, 2) void gemm8f_kernel(const G8Params p) {
    constexpr int NT = NRW * 64, COLS = CT * 16, RG = WT == PS_Q4_0 ? 16 : 8, NQ = WT == PS_Q4_0 ? 1 : 2;
    constexpr int ITEMS = (COLS * 16 + NT - 1) / NT; // (column, block, u) pieces of a stage per thread
    __shared__ __attribute__((aligned(16))) char act[3][4 * CT * 1024];
    __shared__ __attribute__((aligned(16))) float4 yds[3][COLS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, qu = lane >> 4, l16 = lane & 15;
    const int K = p.K, n_units = K / 128, nblk = K / 32, c0 = blockIdx.y * COLS, last = p.bs - 1;
    const int task = min((int)blockIdx.x * NRW + wave, p.n_tasks - 1); // (a wave without rows works on the last ones and stores nothing)
    const bool live = (int)blockIdx.x * NRW + wave < p.n_tasks;

    // activation pieces of this thread: dwords u and u + 4 of a block of a column
    const int8_t *asrc[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; i++) {
        const int idx = min((int)threadIdx.x + i * NT, COLS * 16 - 1); // [block][column tile][u][column]
        asrc[i] = p.aq + (int64_t)min(c0 + ((idx >> 6) % CT) * 16 + (idx & 15), last) * K + (idx >> 6) / CT * 32 + ((idx >> 4) & 3) * 4;
    }
    const float *dsrc = p.ad + (int64_t)min(c0 + (int)threadIdx.x, last) * nblk;
    uint32_t sa[ITEMS][2];
    float4 sd = {};
    auto request = [&](const int un) {
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            sa[i][0] = *(const uint32_t *)(asrc[i] + un * 128);
            sa[i][1] = *(const uint32_t *)(asrc[i] + un * 128 + 16);
        }
        if (threadIdx.x < COLS) sd = *(const float4 *)(dsrc + un * 4);
    };
    auto put = [&](const int buf) {
#pragma unroll
        for (int i = 0; i < ITEMS; i++) {
            const g8_h4 lo = g8_bytes(sa[i][0]), hi = g8_bytes(sa[i][1]);
            const int idx = (int)threadIdx.x + i * NT;
            if (COLS * 16 % NT == 0 || idx < COLS * 16) {
                *(g8_h4 *)(act[buf] + idx * 16) = lo;
                *(g8_h4 *)(act[buf] + idx * 16 + 8) = hi;
            }
        }
        if (threadIdx.x < COLS) yds[buf][threadIdx.x] = sd;
    };

    float yg[CT][4] = {};
    uint32_t e64 = 0x64006400u;
    asm("" : "+v"(e64));
#pragma unroll 1
    for (int pass = 0; pass < (EPI == 1 ? 2 : 1); pass++) {
        int wi = EPI == 1 ? pass : 0, tile = task;
        if (EPI != 1) {
            if (p.n_w > 1 && tile >= p.w[0].n_tiles) { tile -= p.w[0].n_tiles; wi = 1; }
            if (p.n_w > 2 && wi == 1 && tile >= p.w[1].n_tiles) { tile -= p.w[1].n_tiles; wi = 2; }
        }
        const G8W W = wi == 0 ? p.w[0] : wi == 1 ? p.w[1] : p.w[2];
        // operand row l16 of the tile (its pieces u = qu, and for Q8_0 u = qu + 4 64 bytes on), and the scales of result rows 4 qu .. + 3
        const int ga = WT == PS_Q4_0 ? tile : min(tile * 2 + (l16 >> 3), W.n_groups - 1), gd = WT == PS_Q4_0 ? tile : min(tile * 2 + (qu >> 1), W.n_groups - 1);
        const uint8_t *qp = W.qs + (int64_t)ga * n_units * 1024 + (WT == PS_Q4_0 ? l16 * 4 + qu : (l16 & 7) * 8 + qu) * 16;
        const uint8_t *dp = W.aux + (int64_t)gd * n_units * (RG * 8) + (WT == PS_Q4_0 ? qu * 4 : (qu & 1) * 4) * 8;
        g8_f16v acc[CT][2] = {}; // [column tile][u >> 2][(u & 3) * 4 + row]
        g8_f16v D = {};
        float dd[4] = {0.f, 0.f, 0.f, 0.f};
        auto chain = [&](g8_f16v &c) {
#pragma unroll
            for (int i = 0; i < 16; i++) c[i] = __fmaf_rn(dd[i & 3], D[i], c[i]);
            asm volatile("" : "+v"(c)); // (keeps the fmas in their step: without it all of a stage's products are made first and need 16 registers each)
        };
        uint4 nq[NQ], nd[2];
        auto weights = [&](const int un) {
#pragma unroll
            for (int i = 0; i < NQ; i++) nq[i] = *(const uint4 *)(qp + (int64_t)un * 1024 + i * 64);
            nd[0] = *(const uint4 *)(dp + (int64_t)un * (RG * 8));
            nd[1] = *(const uint4 *)(dp + (int64_t)un * (RG * 8) + 16);
        };
        g8_h4 a[2]; // the operand rows of the block at hand, u and u + 4
        auto operands = [&](const uint32_t qa, const uint32_t qb) {
            a[0] = WT == PS_Q4_0 ? g8_nibbles(qa, e64) : g8_bytes(qa);
            a[1] = WT == PS_Q4_0 ? g8_nibbles(qa >> 4, e64) : g8_bytes(qb);
        };
        weights(0);
        request(0);
        if (pass) __syncthreads(); // (the last stages of the pass before are still being read)
        put(0);
        request(min(1, n_units - 1));
        operands(nq[0].x, nq[NQ - 1].x);
        __syncthreads();
        int buf = 0;
        uint4 y = *(const uint4 *)(act[0] + lane * 16);
        float4 yd[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ct++) yd[ct] = yds[0][ct * 16 + l16];
        for (int un = 0; un < n_units; un++) { // the last round's successor is itself: written and read once more, never used
            const uint32_t qa[4] = {nq[0].x, nq[0].y, nq[0].z, nq[0].w}, qb[4] = {nq[NQ - 1].x, nq[NQ - 1].y, nq[NQ - 1].z, nq[NQ - 1].w};
            const uint32_t h[8] = {nd[0].x, nd[0].y, nd[0].z, nd[0].w, nd[1].x, nd[1].y, nd[1].z, nd[1].w}; // [row][block pair]
            const int nbuf = buf == 2 ? 0 : buf + 1;
            weights(min(un + 1, n_units - 1));
#pragma unroll
            for (int s = 0; s < 4 * CT; s++) { // (block, column tile) s: its products are issued, those of the step before meet their multipliers meanwhile
                const int b = s / CT, ct = s % CT;
                const g8_f16v zero = {};
                const g8_f16v E0 = __builtin_amdgcn_mfma_f32_16x16x4f16(a[0], g8_pair(y.x, y.y), zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                const uint4 ny = s + 1 < 4 * CT ? *(const uint4 *)(act[buf] + ((s + 1) * 64 + lane) * 16) : *(const uint4 *)(act[nbuf] + lane * 16);
                chain(acc[(ct + CT - 1) % CT][1]);
                D = E0;
                const float ydb = b == 0 ? yd[ct].x : b == 1 ? yd[ct].y : b == 2 ? yd[ct].z : yd[ct].w;
#pragma unroll
                for (int r = 0; r < 4; r++) dd[r] = g8_scale(h[2 * r + (b >> 1)], ydb, b & 1);
                if (b == 3) yd[ct] = yds[nbuf][ct * 16 + l16];
                __builtin_amdgcn_sched_barrier(0);
                const g8_f16v E1 = __builtin_amdgcn_mfma_f32_16x16x4f16(a[1], g8_pair(y.z, y.w), zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                chain(acc[ct][0]);
                D = E1;
                y = ny;
                if (ct == CT - 1) operands(b < 3 ? qa[(b + 1) & 3] : nq[0].x, b < 3 ? qb[(b + 1) & 3] : nq[NQ - 1].x);
                if (s == 0) { put(nbuf); request(min(un + 2, n_units - 1)); }
                __builtin_amdgcn_sched_barrier(0);
                if (s == 2 * CT) __syncthreads(); // the next stage is there for all; it overwrote the stage before the present one, which every wave has left behind
            }
            buf = nbuf;
        }
        chain(acc[CT - 1][1]);
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int r = 0; r < 4; r++) { // hsum_float_8: (u + 4) + u, then u + 2, then u + 1
                float s[4];
#pragma unroll
                for (int u = 0; u < 4; u++) s[u] = __fadd_rn(acc[ct][1][u * 4 + r], acc[ct][0][u * 4 + r]);
                const float v = __fadd_rn(__fadd_rn(s[0], s[2]), __fadd_rn(s[1], s[3]));
                if (EPI == 1 && pass == 0) { yg[ct][r] = v; continue; }
                const int row = tile * 16 + qu * 4 + r, col = c0 + ct * 16 + l16;
                if (!live || row >= W.N || col > last) continue;
                if (EPI == 1) {
                    p.w[0].out[(int64_t)col * p.w[0].ldo + row] = ps_silu_mul(yg[ct][r], v);
                } else {
                    float val = v;
                    if (W.bias) val = __fadd_rn(val, W.bias[row]);
                    if (p.residual && wi == 0) val = __fadd_rn(p.residual[(int64_t)col * W.ldo + row], val);
                    W.out[(int64_t)col * W.ldo + row] = val;
                }
            }
    }
}

template <int WT, int EPI, int CT, int NRW>
int g8f(hipStream_t st, const G8Params &p) {
    psk_note_kernel("gemm8f_kernel<%d, %d, %d, %d>", WT, EPI, CT, NRW);
    hipLaunchKernelGGL((gemm8f_kernel<WT, EPI, CT, NRW>), dim3((unsigned)((p.n_tasks + NRW - 1) / NRW), (unsigned)((p.bs + CT * 16 - 1) / (CT * 16))), dim3(NRW * 64), 0, st, p);
    return 0;
}
// Which form: 32 columns per wave do the weight side of a block (11-15 instructions to 72 of the chain) once for two column tiles and are the faster ones where they fill
// the chip's 8 waves per CU -- eight waves to a work-group, or four where the last round of eights would be less than 0.7 full and quarter-size groups spread it better
// (3072 x 2048, 511 columns, Q4_0: 58 -> 50 us).  Below that, 16 columns per wave: four to a work-group, two while those still find a CU each (4096 x 4096, 64 columns:
// 28.5 us with 16, 39 with 32).  Measured over K 896 .. 14336, N 896 .. 14336, 2 .. 511 columns, both types: the form taken is within 9 % of the best of all six.
template <int WT, int EPI>
int g8f_pick(hipStream_t st, int n_cu, const G8Params &p) {
    const int64_t w1 = (int64_t)p.n_tasks * ((p.bs + 15) / 16), w2 = (int64_t)p.n_tasks * ((p.bs + 31) / 32), full = 8 * (int64_t)n_cu;
    if (w2 * 8 < full * 7) return w1 <= 2 * n_cu ? g8f<WT, EPI, 1, 2>(st, p) : g8f<WT, EPI, 1, 4>(st, p);
    const int64_t rest = w2 % full;
    return rest == 0 || rest * 10 > full * 7 || w2 < full ? g8f<WT, EPI, 2, 8>(st, p) : g8f<WT, EPI, 2, 4>(st, p);
}

} // namespace

int psk_gemm8f(hipStream_t st, int n_cu, const psk_gemv_args &a, ps_act act, int64_t K, int64_t bs) {
    const int wt = a.w[0]->dtype;
    if ((wt != PS_Q8_0 && wt != PS_Q4_0) || a.pro || a.rope || K % 128 || K >= (1 << 24) || a.n_w < 1 || a.n_w > 3) return -1;
    G8Params p{};
    p.n_w = a.n_w; p.K = (int)K; p.bs = (int)bs; p.residual = a.residual; p.aq = act.qs; p.ad = act.d;
    const int rg = wt == PS_Q4_0 ? 16 : 8;
    for (int i = 0; i < a.n_w; i++) {
        if (a.w[i]->dtype != wt || a.w[i]->K != K) return -1;
        p.w[i] = G8W{a.w[i]->qs, a.w[i]->aux, a.out[i], a.bias[i], a.w[i]->N, a.ldo[i], (int)((a.w[i]->N + rg - 1) / rg), (int)((a.w[i]->N + 15) / 16)};
        p.n_tasks += p.w[i].n_tiles;
    }
    if (a.silu_pair) {
        if (a.n_w != 2 || a.w[0]->N != a.w[1]->N) return -1;
        p.n_tasks = p.w[0].n_tiles;
        return wt == PS_Q4_0 ? g8f_pick<PS_Q4_0, 1>(st, n_cu, p) : g8f_pick<PS_Q8_0, 1>(st, n_cu, p);
    }
    return wt == PS_Q4_0 ? g8f_pick<PS_Q4_0, 0>(st, n_cu, p) : g8f_pick<PS_Q8_0, 0>(st, n_cu, p);
}
