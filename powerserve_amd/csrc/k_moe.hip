// Mixture-of-experts routing for the layer-list models (PS_FF_MOE_SWIGLU, PS_FF_MOE_RELU2).  The experts' matrix products are grouped launches of the dense kernels
// (k_dense.hip); here is what decides who goes where, all fp32:
//   moe_route_kernel    a block per token: router logits (+ bias), sigmoid or soft-max scores, a correction and a group limit on the choice, the `top` largest
//                       (their scores, or the soft-max over the chosen logits alone, times a constant), the shared expert's gate
//   moe_plan_kernel     the token-expert slots sorted by expert (counts, offsets, list) for the tiled products
//   moe_combine_kernel  a token's `top` per-slot results summed into the residual stream; an identity expert's share is its weight times the input
#include "ps_seq.h"

#include <cmath>

static __device__ __forceinline__ float moe_wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
static __device__ __forceinline__ float moe_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

typedef float moe_f4 __attribute__((ext_vector_type(4)));
struct moe_route_args {
    const float *router, *shared_gate, *bias, *correction;
    int experts, top, norm_top, softmax, n_groups, keep;
    float scale;
    long long K;
    int32_t *sel;
    float *wgt, *sgate;
};
// the largest of token t's scores sc[] (one wave)
static __device__ __forceinline__ void moe_choose(const moe_route_args &r, const int t, const int lane, float *sc) {
    const int experts = r.experts, top = r.top, norm_top = r.norm_top, softmax = r.softmax, n_groups = r.n_groups, keep = r.keep;
    const float *shared_gate = r.shared_gate, *correction = r.correction, scale = r.scale;
    int32_t *sel = r.sel;
    float *wgt = r.wgt, *sgate = r.sgate, *ch = sc + experts + 1, *gs = ch + experts;
    if (shared_gate && lane == 0) sgate[t] = sc[experts];
    if (softmax == 1) {
        float mx = -INFINITY, sum = 0.f;
        for (int e = lane; e < experts; e += 64) mx = fmaxf(mx, sc[e]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        for (int e = lane; e < experts; e += 64) sum += expf(sc[e] - mx);
        sum = moe_wave_sum(sum);
        for (int e = lane; e < experts; e += 64) sc[e] = expf(sc[e] - mx) / sum;
    }
    for (int e = lane; e < experts; e += 64) ch[e] = sc[e] + (correction ? correction[e] : 0.f);
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    // (largest value, lowest index) over the wave's proposals
    auto agree = [&](float &best, int &at) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, 64);
            const int oa = __shfl_xor(at, o, 64);
            if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
        }
    };
    if (n_groups > 0) { // a group's score is its best choice score; the rows of every group outside the `keep` best leave the race
        const int size = experts / n_groups;
        for (int g = lane; g < n_groups; g += 64) {
            float b = -INFINITY;
            for (int e = g * size; e < (g + 1) * size; e++) b = fmaxf(b, ch[e]);
            gs[g] = b;
        }
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (int i = 0; i < keep; i++) {
            float best = -INFINITY;
            int at = 0x7fffffff;
            for (int g = lane; g < n_groups; g += 64)
                if (gs[g] > best) { best = gs[g]; at = g; }
            agree(best, at);
            if (lane == 0 && at != 0x7fffffff) gs[at] = -INFINITY; // (struck out = kept)
            __builtin_amdgcn_wave_barrier();
            __threadfence_block();
        }
        for (int e = lane; e < experts; e += 64)
            if (gs[e / size] != -INFINITY) ch[e] = -INFINITY;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    float total = 0.f;
    for (int i = 0; i < top; i++) {
        float best = -INFINITY;
        int at = 0x7fffffff;
        for (int e = lane; e < experts; e += 64)
            if (ch[e] > best) { best = ch[e]; at = e; }
        agree(best, at);
        const bool any = at != 0x7fffffff; // (nothing left in the race: the slot goes to row 0 with weight 0)
        const float w = any ? sc[at] : softmax == 2 ? -INFINITY : 0.f;
        if (lane == 0) { sel[(long long)t * top + i] = any ? at : 0; wgt[(long long)t * top + i] = norm_top || softmax == 2 ? w : w * scale; if (any) ch[at] = -INFINITY; }
        total += w;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
    if (softmax == 2) { // the soft-max over the chosen logits
        float mx = -INFINITY, sum = 0.f;
        for (int i = lane; i < top; i += 64) mx = fmaxf(mx, wgt[(long long)t * top + i]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        for (int i = lane; i < top; i += 64) sum += expf(wgt[(long long)t * top + i] - mx);
        sum = moe_wave_sum(sum);
        for (int i = lane; i < top; i += 64) wgt[(long long)t * top + i] = expf(wgt[(long long)t * top + i] - mx) / sum * scale;
    } else if (norm_top)
        for (int i = lane; i < top; i += 64) wgt[(long long)t * top + i] = wgt[(long long)t * top + i] / total * scale;
}

// One block per token: four waves, sixteen for a few tokens, where a wave then has a row or two instead of walking through all of them (9 rows of 2048, one token: 6.4 us with four, 5.2 with
// sixteen).  The rows of the router (and the shared gate's row as one more) are dealt to the waves; a row's K numbers are read as 16-byte pieces, eight in flight per lane.  Then wave 0 alone: scores (sigmoid, or soft-max over all rows), the choice scores (score + correction), the
// groups that stay in the race, and `top` rounds of (largest choice score, lowest index); the weights are the SCORES of the chosen.
// dynamic LDS: [rows + 1] scores, [rows] choice scores, [groups] group scores.
__global__ __launch_bounds__(1024) void moe_route_kernel(const float *h, long long ldh, moe_route_args r) {
    extern __shared__ float sc[];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float *x = h + (long long)t * ldh;
    const bool vec = r.K % 4 == 0 && ldh % 4 == 0;
    for (int e = wave; e < r.experts + (r.shared_gate ? 1 : 0); e += (int)(blockDim.x >> 6)) {
        const float *w = e < r.experts ? r.router + (long long)e * r.K : r.shared_gate;
        float a = 0.f;
        if (vec) {
            float a4[4] = {0.f, 0.f, 0.f, 0.f};
            for (long long k0 = 0; k0 < r.K; k0 += 2048) {
                moe_f4 wv[8], xv[8];
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const long long k = k0 + 256 * u + 4 * lane;
                    const bool in = k < r.K;
                    wv[u] = in ? *(const moe_f4 *)(w + k) : moe_f4{0.f, 0.f, 0.f, 0.f};
                    xv[u] = in ? *(const moe_f4 *)(x + k) : moe_f4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int u = 0; u < 8; u++)
#pragma unroll
                    for (int i = 0; i < 4; i++) a4[i] = fmaf(wv[u][i], xv[u][i], a4[i]);
            }
            a = (a4[0] + a4[1]) + (a4[2] + a4[3]);
        } else {
            for (long long k = lane; k < r.K; k += 64) a = fmaf(w[k], x[k], a);
        }
        a = moe_wave_sum(a);
        if (r.bias && e < r.experts) a += r.bias[e];
        if (lane == 0) sc[e] = r.softmax && e < r.experts ? a : moe_sigmoid(a);
    }
    __syncthreads();
    if (wave) return;
    moe_choose(r, t, lane, sc);
}

// A single token's sublayer boundary x += y / rms(y) * (offset + wb) (sq_boundary1_fast_kernel's sums, in its order) and the routing of the result, one block.  Both are chains of latencies
// behind a launch of their own; here the wave's first row of the router is requested with everything else, the normed row goes to LDS, and the dot products start where the boundary ends:
// 2048 wide, 9 rows: 3.9 and 5.2 us in two launches, 5.8 in one.  C: runs of four channels per thread.
template <int C>
__global__ __launch_bounds__(1024) void moe_boundary_route_kernel(float *x, const float *y, const float *wb, float offset, float eps, moe_route_args r) {
    extern __shared__ float sc[];
    __shared__ __attribute__((aligned(16))) float xs[C * 4096];
    __shared__ float red[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = (int)r.K, rows = r.experts + (r.shared_gate ? 1 : 0);
    const moe_f4 zero = {0.f, 0.f, 0.f, 0.f};
    moe_f4 xv[C], yv[C], b4[C], wv[8];
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int i = (tid + c * 1024) * 4;
        const bool in = i < n;
        yv[c] = in ? *(const moe_f4 *)(y + i) : zero;
        xv[c] = in ? *(const moe_f4 *)(x + i) : zero;
        b4[c] = in ? *(const moe_f4 *)(wb + i) : zero;
    }
    auto row = [&](const int e) { return e < r.experts ? r.router + (long long)e * n : r.shared_gate; };
    auto request = [&](const float *w, const int k0) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int k = k0 + 256 * u + 4 * lane;
            wv[u] = k < n ? *(const moe_f4 *)(w + k) : zero;
        }
    };
    if (wave < rows) request(row(wave), 0);
    float s1 = 0.f;
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) s1 += yv[c][e] * yv[c][e];
    s1 = sq_wave_sum(s1);
    if (lane == 0) red[wave] = s1;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < 16; w++) t += red[w];
    const float inv = 1.f / sqrtf(t / (float)n + eps);
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int i = (tid + c * 1024) * 4;
#pragma unroll
        for (int e = 0; e < 4; e++) xv[c][e] = xv[c][e] + yv[c][e] * inv * (offset + b4[c][e]);
        *(moe_f4 *)(xs + i) = i < n ? xv[c] : zero;
        if (i < n) *(moe_f4 *)(x + i) = xv[c];
    }
    __syncthreads();
    for (int e = wave; e < rows; e += 16) {
        float a4[4] = {0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < n; k0 += 2048) {
            if (e != wave || k0) request(row(e), k0);
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const moe_f4 v = *(const moe_f4 *)(xs + min(k0 + 256 * u + 4 * lane, C * 4096 - 4)); // (behind the row: the weights are zero)
#pragma unroll
                for (int i = 0; i < 4; i++) a4[i] = fmaf(wv[u][i], v[i], a4[i]);
            }
        }
        float a = moe_wave_sum((a4[0] + a4[1]) + (a4[2] + a4[3]));
        if (r.bias && e < r.experts) a += r.bias[e];
        if (lane == 0) sc[e] = r.softmax && e < r.experts ? a : moe_sigmoid(a);
    }
    __syncthreads();
    if (wave) return;
    moe_choose(r, 0, lane, sc);
}
void psk_moe_route(hipStream_t st, const float *h, int64_t ldh, const float *router, const float *shared_gate, int experts, int top, int norm_top, int64_t K, int T,
                   int32_t *sel, float *wgt, float *sgate, int softmax, const float *correction, int n_groups, int keep, float scale, const float *bias, const psk_moe_front *front) {
    const moe_route_args r = {router, shared_gate, bias, correction, experts, top, norm_top, softmax, n_groups, keep, scale, (long long)K, sel, wgt, sgate};
    const size_t lds = (size_t)(2 * experts + 1 + (n_groups > 0 ? n_groups : 0)) * 4;
    if (front) { // (psk_moe_front_ok)
        if (K <= 4096) hipLaunchKernelGGL(moe_boundary_route_kernel<1>, dim3(1), dim3(1024), lds, st, front->x, front->y, front->w, front->offset, front->eps, r);
        else hipLaunchKernelGGL(moe_boundary_route_kernel<2>, dim3(1), dim3(1024), lds, st, front->x, front->y, front->w, front->offset, front->eps, r);
        return;
    }
    hipLaunchKernelGGL(moe_route_kernel, dim3(T), dim3(T <= 8 ? 1024 : 256), lds, st, h, (long long)ldh, r);
}
// 16-byte pieces of every row, a thread's runs in registers; up to 64 rows: behind that the one block reads longer than it saves
bool psk_moe_front_ok(const psk_moe_front &f, const float *router, const float *shared_gate, int experts, int64_t K) {
    auto aligned = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
    return K % 4 == 0 && K <= 8192 && experts <= 64 && aligned(f.x) && aligned(f.y) && aligned(f.w) && aligned(router) && aligned(shared_gate);
}

// one block; dynamic LDS: 2 x experts ints.  Counts, offsets, then every slot takes the next free place of its expert.  Which place a slot gets is up to the
// atomics, and it does not matter: a row of a tiled product is summed over k in the same order wherever in a tile it sits.
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int32_t *sel, int S, int experts, int32_t *seg, int32_t *list) {
    extern __shared__ int pl[];
    int *cnt = pl, *cur = pl + experts;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int e = tid; e < experts; e += nt) cnt[e] = 0;
    __syncthreads();
    for (int s = tid; s < S; s += nt) atomicAdd(&cnt[sel[s]], 1);
    __syncthreads();
    if (tid == 0) {
        int at = 0;
        for (int e = 0; e < experts; e++) { seg[e] = at; cur[e] = at; at += cnt[e]; }
        seg[experts] = at;
    }
    __syncthreads();
    for (int s = tid; s < S; s += nt) list[atomicAdd(&cur[sel[s]], 1)] = s;
}
void psk_moe_plan(hipStream_t st, const int32_t *sel, int S, int experts, int32_t *seg, int32_t *list) {
    hipLaunchKernelGGL(moe_plan_kernel, dim3(1), dim3(S >= 1024 ? 1024 : 256), (size_t)experts * 8, st, sel, S, experts, seg, list);
}

// x[t] += alpha * sum_k (slot t top + k: its product's result y[slot], or -- a slot whose choice is an identity expert, sel >= n_real -- wgt[slot] * h[t]);
// y NULL: the products have been added already and only the identity slots are left.  store: x[t] = instead of +=.
__global__ void moe_combine_kernel(float *x, const float *y, int top, float alpha, long long n, const int32_t *sel, const float *wgt, int n_real, const float *h,
                                   long long ldh, int store) {
    const long long t = blockIdx.x;
    for (long long i = threadIdx.x; i < n; i += blockDim.x) {
        float a = 0.f;
        for (int k = 0; k < top; k++) {
            const long long s = t * top + k;
            if (sel && sel[s] >= n_real) a = fmaf(wgt[s], h[t * ldh + i], a);
            else if (y) a += y[s * n + i];
        }
        x[t * n + i] = store ? alpha * a : x[t * n + i] + alpha * a;
    }
}
void psk_moe_combine(hipStream_t st, float *x, const float *y, int top, float alpha, int64_t n, int T, const int32_t *sel, const float *wgt, int n_real, const float *h,
                     int64_t ldh, int store) {
    hipLaunchKernelGGL(moe_combine_kernel, dim3(T), dim3(256), 0, st, x, y, top, alpha, (long long)n, sel, wgt, n_real, h, (long long)ldh, store);
}
