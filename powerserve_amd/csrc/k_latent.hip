// Latent attention of the layer-list models: what a token leaves behind is its normalised key-value latent c (kv_rank numbers) and one rotated
// key part shared by all heads (rot_dim numbers), kept in a per-sequence RING of `cap` rows (row = position mod cap; cap >= window - 1 + the
// widest step, so a step never overwrites a row one of its own tokens still sees).  Scores, soft-max and the weighted sum are fp32.  cos and sin of the
// rotation may carry a common factor (rot_mag: frequency scaling by wavelength stretches both), and a head's output a sigmoid gate.
//   latent_prep_kernel   norms of the two latents, rotation of the shared key part, ring append
//   latent_attn_kernel   one wave per (token, head) over per-head keys / values expanded from the ring rows of the window (the plain form)
//   latent_attn_mfma_kernel / latent_absorbed_kernel (+ fold, combine, unfold): the matrix-core forms for a portion and for a single token, below
#include "ps_attn_dev.h"
#include "ps_seq.h"

#include <cmath>

static __device__ __forceinline__ float la_wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
static __device__ __forceinline__ float la_wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// the two numbers of rotated pair i of a part whose first 2 half numbers turn
static __device__ __forceinline__ void la_pair(int i, int half, int pairing, int &a, int &b) {
    if (pairing == PS_ROT_NEIGHBOURS) { a = 2 * i; b = a + 1; }
    else { a = i; b = i + half; }
}

struct la_token { // psk_latent_row and what else the row's preparation takes
    const float *y, *qnorm, *kvnorm;
    long long ldy, ldcq;
    float eps;
    int q_rank, kv_rank, rot_dim, rot_dims, pairing;
    float *cq;
    const float *freq;
    float rot_mag;
};
static __device__ __forceinline__ void la_prepare(const ps_seq_step *step, long long ring_off, int cap, const la_token &w, int t) { // by 256 threads
    const float *y = w.y, *qnorm = w.qnorm, *kvnorm = w.kvnorm, *freq = w.freq;
    float *cq = w.cq;
    const long long ldy = w.ldy, ldcq = w.ldcq;
    const float eps = w.eps, rot_mag = w.rot_mag;
    const int q_rank = w.q_rank, kv_rank = w.kv_rank, rot_dim = w.rot_dim, rot_dims = w.rot_dims, pairing = w.pairing, tid = threadIdx.x;
    // (a thread's numbers and weights are requested together and held: 8 + 4 of them, what is beyond 2048 and 1024 is read again)
    __shared__ float red[8];
    const float *yt = y + (long long)t * ldy, *ckv = yt + q_rank, *kr = ckv + kv_rank;
    float qv[8], qw[8], kv[4], kw[4], a = 0.f, b = 0.f;
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int i = tid + 256 * u;
        qv[u] = i < q_rank ? yt[i] : 0.f;
        qw[u] = i < q_rank ? qnorm[i] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int i = tid + 256 * u;
        kv[u] = i < kv_rank ? ckv[i] : 0.f;
        kw[u] = i < kv_rank ? kvnorm[i] : 0.f;
    }
    const long long pos = step->pos0 + t;
    float *ring = step->state + ring_off + (pos % cap) * (long long)(kv_rank + rot_dim);
#pragma unroll
    for (int u = 0; u < 8; u++) a += qv[u] * qv[u];
#pragma unroll
    for (int u = 0; u < 4; u++) b += kv[u] * kv[u];
    for (int i = 2048 + tid; i < q_rank; i += 256) a += yt[i] * yt[i];
    for (int i = 1024 + tid; i < kv_rank; i += 256) b += ckv[i] * ckv[i];
    a = la_wave_sum(a);
    b = la_wave_sum(b);
    if ((tid & 63) == 0) { red[tid >> 6] = a; red[4 + (tid >> 6)] = b; }
    __syncthreads();
    const float ia = q_rank > 0 ? 1.f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)q_rank + eps) : 0.f; // (q_rank 0: the queries do not pass a latent)
    const float ib = 1.f / sqrtf((red[4] + red[5] + red[6] + red[7]) / (float)kv_rank + eps);
#pragma unroll
    for (int u = 0; u < 8; u++)
        if (tid + 256 * u < q_rank) cq[(long long)t * ldcq + tid + 256 * u] = qv[u] * ia * qw[u];
#pragma unroll
    for (int u = 0; u < 4; u++)
        if (tid + 256 * u < kv_rank) ring[tid + 256 * u] = kv[u] * ib * kw[u];
    for (int i = 2048 + tid; i < q_rank; i += 256) cq[(long long)t * ldcq + i] = yt[i] * ia * qnorm[i];
    for (int i = 1024 + tid; i < kv_rank; i += 256) ring[i] = ckv[i] * ib * kvnorm[i];
    const int half = rot_dims / 2; // the first rot_dims of the part are rotated; the rest passes unchanged
    for (int i = tid; i < half; i += 256) {
        const float ang = (float)pos * freq[i], c = cosf(ang) * rot_mag, s = sinf(ang) * rot_mag;
        int pa, pb;
        la_pair(i, half, pairing, pa, pb);
        const float u = kr[pa], v = kr[pb];
        ring[kv_rank + pa] = u * c - v * s;
        ring[kv_rank + pb] = v * c + u * s;
    }
    for (int i = 2 * half + tid; i < rot_dim; i += 256) ring[kv_rank + i] = kr[i];
}
__global__ __launch_bounds__(256) void latent_prep_kernel(const ps_seq_step *step, long long ring_off, int cap, la_token w) { la_prepare(step, ring_off, cap, w, blockIdx.x); }
static la_token la_token_of(const psk_latent_row &r, int kv_rank, int rot_dim, int rot_dims, const float *freq, float rot_mag, int pairing) {
    return la_token{r.y, r.qnorm, r.kvnorm, (long long)r.ldy, (long long)r.ldcq, r.eps, r.q_rank, kv_rank, rot_dim, rot_dims, pairing, r.cq, freq, rot_mag};
}
void psk_latent_prep(hipStream_t st, const ps_seq_step *step, int64_t ring_off, int cap, const psk_latent_row &row, int kv_rank, int rot_dim, int rot_dims, const float *freq, int T, float rot_mag,
                     int pairing) {
    hipLaunchKernelGGL(latent_prep_kernel, dim3(T), dim3(256), 0, st, step, (long long)ring_off, cap, la_token_of(row, kv_rank, rot_dim, rot_dims, freq, rot_mag, pairing));
}

// dynamic LDS: qs [d + dr], ps [64]
#define LA_NV 4 // value columns per lane: dv <= 256
__global__ __launch_bounds__(64) void latent_attn_kernel(const ps_seq_step *step, long long ring_off, int cap, const float *q, long long ldq, const float *kv,
                                                         long long ldkv, const float *freq, int H, int d, int dr, int rot_dims, int dv, int kv_rank, int window,
                                                         float scale, float *o, long long ldo, float rot_mag, const float *gate, long long ldg, int pairing) {
    extern __shared__ float lds[];
    float *qs = lds, *ps = lds + d + dr;
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const long long pos0 = step->pos0, p = pos0 + t;
    const long long first = pos0 - window + 1 > 0 ? pos0 - window + 1 : 0; // position of kv row 0
    const long long lo = p - window + 1 > 0 ? p - window + 1 : 0;
    const float *qt = q + (long long)t * ldq + (long long)h * (d + dr);
    const int half = rot_dims / 2;
    for (int i = lane; i < d; i += 64) qs[i] = qt[i];
    for (int i = 2 * half + lane; i < dr; i += 64) qs[d + i] = qt[d + i];
    for (int i = lane; i < half; i += 64) {
        const float ang = (float)p * freq[i], c = cosf(ang) * rot_mag, s = sinf(ang) * rot_mag;
        int pa, pb;
        la_pair(i, half, pairing, pa, pb);
        const float u = qt[d + pa], v = qt[d + pb];
        qs[d + pa] = u * c - v * s;
        qs[d + pb] = v * c + u * s;
    }
    __syncthreads();
    const float *ring = step->state + ring_off;
    const long long rs = kv_rank + dr;
    float m = -INFINITY, l = 0.f, acc[LA_NV];
#pragma unroll
    for (int x = 0; x < LA_NV; x++) acc[x] = 0.f;
    for (long long j0 = lo; j0 <= p; j0 += 64) {
        const long long j = j0 + lane;
        float s = -INFINITY;
        if (j <= p) {
            const float *kn = kv + (j - first) * ldkv + (long long)h * d;
            const float *kr = ring + (j % cap) * rs + kv_rank;
            float a = 0.f;
            for (int i = 0; i < d; i++) a = fmaf(qs[i], kn[i], a);
            for (int i = 0; i < dr; i++) a = fmaf(qs[d + i], kr[i], a);
            s = a * scale;
        }
        const float mn = fmaxf(m, la_wave_max(s));
        const float corr = expf(m - mn), pj = j <= p ? expf(s - mn) : 0.f; // (m = -inf in the first round: corr = 0, acc and l are 0)
        l = l * corr + la_wave_sum(pj);
        m = mn;
        __syncthreads();
        ps[lane] = pj;
        __syncthreads();
        const int nk = (int)min((long long)64, p - j0 + 1);
#pragma unroll
        for (int x = 0; x < LA_NV; x++) acc[x] *= corr;
        for (int kk = 0; kk < nk; kk++) {
            const float *vr = kv + (j0 + kk - first) * ldkv + (long long)H * d + (long long)h * dv;
            const float pk = ps[kk];
#pragma unroll
            for (int x = 0; x < LA_NV; x++)
                if (lane + 64 * x < dv) acc[x] = fmaf(pk, vr[lane + 64 * x], acc[x]);
        }
    }
    const float il = (gate ? 1.f / (1.f + expf(-gate[(long long)t * ldg + h])) : 1.f) / l;
#pragma unroll
    for (int x = 0; x < LA_NV; x++)
        if (lane + 64 * x < dv) o[(long long)t * ldo + (long long)h * dv + lane + 64 * x] = acc[x] * il;
}
void psk_latent_attn(hipStream_t st, const ps_seq_step *step, int64_t ring_off, int cap, const float *q, int64_t ldq, const float *kv, int64_t ldkv,
                     const float *freq, int H, int d, int dr, int rot_dims, int dv, int kv_rank, int window, float scale, int T, float *o, int64_t ldo, float rot_mag,
                     const float *gate, int64_t ldg, int pairing) {
    hipLaunchKernelGGL(latent_attn_kernel, dim3(T, H), dim3(64), (size_t)(d + dr + 64) * 4, st, step, (long long)ring_off, cap, q, (long long)ldq, kv, (long long)ldkv,
                       freq, H, d, dr, rot_dims, dv, kv_rank, window, scale, o, (long long)ldo, rot_mag, gate, (long long)ldg, pairing);
}

// ---------------------------------------------------------------------------------------------------- matrix-core form
// One wave attends 16 rows to tiles of 16 keys, fp32 throughout on v_mfma_f32_16x16x4_f32:
//   scores   S[16 x 16] = Q[16 x DK] K^T: the keys come straight from memory as 16-byte pieces (lane (key l % 16, quarter l / 16) holds 4
//            consecutive dimensions; the row operand is read from LDS in the same order, so the sum runs over a permutation of the dimensions)
//   soft-max online, in the accumulator layout (lane holds rows 4 (l / 16) + i of key column l % 16; a row's 16 lanes reduce by rotations)
//   output   O[16 x DV] += P V: P goes through a 16 x 17 LDS patch into the row-operand layout; V comes as 16-byte pieces of 4 consecutive
//            columns, so accumulator tile jj of a 64-column group holds columns 4 (l % 16) + jj -- undone at the final store.
// A "row" is a (token, head) pair.  Two drivers use it: a prompt's portion over per-head keys / values expanded from the ring (rows = 16
// consecutive tokens of one head), and the single-token step in the ABSORBED form -- rows = heads, every head's query folded through its key
// expansion into latent space (q~_h = W_uk,h^T q_h), keys AND values the ring's latents themselves, the value expansion applied afterwards to
// the attended latent -- where the ring is read once for all heads and nothing is expanded per key.
// A prompt's portion: block = RT x 16 consecutive tokens of one head, keys / values expanded per head in kv (position first + row).  The key tiles are dealt to the block's eight waves,
// each with its own running soft-max, and the eight partial results are merged at the end (la_merge).  What bounded the form before (a wave per 16 tokens over all its keys: 512 waves for
// 512 tokens of 16 heads, one per SIMD on half the chip) was the latency of a key tile -- its keys, its soft-max, its values, one behind the other: 270 us per 512 tokens behind a
// 1024-token window where the matrix instructions need 35.  Now every SIMD has two waves and a key piece serves two row tiles: 80 us.
// dynamic LDS: RT x 16 x qld + 8 x RT x 16 x 17 floats, then the merge's slots over them
template <int NJ, int RT>
__global__ __launch_bounds__(512) void latent_attn_mfma_kernel(const ps_seq_step *step, long long ring_off, int cap, const float *q, long long ldq, const float *kv,
                                                               long long ldkv, const float *freq, int H, int d, int dr, int rot_dims, int dv, int kv_rank, int window,
                                                               float scale, int T, float *o, long long ldo, float rot_mag, const float *gate, long long ldg, int pairing) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4, h = blockIdx.y;
    const int qld = d + dr + 4;
    float *qs = lds, *pt = lds + RT * 16 * qld + wave * RT * 16 * 17;
    const long long pos0 = step->pos0;
    const int t0 = blockIdx.x * 16 * RT;
    const long long first = pos0 - window + 1 > 0 ? pos0 - window + 1 : 0;
    const int half = rot_dims / 2;
    // the block's query rows into LDS (no index division, one sincos per rotated pair and row)
    for (int r = wave; r < 16 * RT; r += 8) {
        const int t = t0 + r;
        const bool in = t < T;
        const float *qt = q + (long long)(in ? t : 0) * ldq + (long long)h * (d + dr);
        float *qr = qs + r * qld;
        for (int c = lane; c < d; c += 64) qr[c] = in ? qt[c] : 0.f;
        for (int c = 2 * half + lane; c < dr; c += 64) qr[d + c] = in ? qt[d + c] : 0.f;
        for (int i = lane; i < half; i += 64) {
            const float ang = (float)(pos0 + t) * freq[i], cs = cosf(ang) * rot_mag, sn = sinf(ang) * rot_mag;
            int pa, pb;
            la_pair(i, half, pairing, pa, pb);
            const float u = in ? qt[d + pa] : 0.f, v = in ? qt[d + pb] : 0.f;
            qr[d + pa] = u * cs - v * sn;
            qr[d + pb] = v * cs + u * sn;
        }
    }
    __syncthreads();
    // keys counted from position `first`
    const la_src k1 = {kv + (long long)h * d, ldkv, 0, 0}, vs = {kv + (long long)H * d + (long long)h * dv, ldkv, 0, 0};
    const la_src k2 = la_ring(step->state + ring_off + kv_rank, kv_rank + dr, first, cap);
    float m[RT][4], l[RT][4];
    la_f4 acc[RT][NJ];
#pragma unroll
    for (int r = 0; r < RT; r++) {
#pragma unroll
        for (int i = 0; i < 4; i++) { m[r][i] = -INFINITY; l[r][i] = 0.f; }
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[r][j] = la_f4{0.f, 0.f, 0.f, 0.f};
    }
    const la_window see{(int)(pos0 - first) + t0, window, T - t0, lq, 0.f};
    const int last = see.q0 + min(16 * RT, T - t0) - 1, lo = see.q0 - window + 1 > 0 ? see.q0 - window + 1 : 0;
    for (int j0 = lo + 16 * wave; j0 <= last; j0 += 128) la_tiles<NJ, RT, false>(qs, qld, pt, k1, k2, vs, d, dr, dv, j0, last + 1, see, scale, m, l, acc);
    la_merge8<NJ, RT>(lds, m, l, acc);
    if (wave) return;
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int J = 0; J < NJ / 4; J++)
#pragma unroll
            for (int i = 0; i < 4; i++) { // a lane's four tiles of a 64-column group are four consecutive columns: one 16-byte store
                const int t = t0 + 16 * r + 4 * lq + i, c = 64 * J + 4 * lr;
                if (t < T && c < dv) {
                    const float il = (gate ? 1.f / (1.f + expf(-gate[(long long)t * ldg + h])) : 1.f) / l[r][i];
                    *(la_f4 *)(o + (long long)t * ldo + (long long)h * dv + c) = la_f4{acc[r][4 * J][i] * il, acc[r][4 * J + 1][i] * il, acc[r][4 * J + 2][i] * il, acc[r][4 * J + 3][i] * il};
                }
            }
}
bool psk_latent_attn_mfma_ok(int d, int dr, int dv) { return d % 16 == 0 && dr % 16 == 0 && dv % 4 == 0 && dv <= 128 && la_portion_lds<8, 1>(d + dr) <= 160 * 1024; }
template <int RT>
static void la_launch_latent(hipStream_t st, const ps_seq_step *step, int64_t ring_off, int cap, const float *q, int64_t ldq, const float *kv, int64_t ldkv, const float *freq, int H, int d,
                             int dr, int rot_dims, int dv, int kv_rank, int window, float scale, int T, float *o, int64_t ldo, float rot_mag, const float *gate, int64_t ldg, int pairing) {
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)latent_attn_mfma_kernel<8, RT>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    hipLaunchKernelGGL((latent_attn_mfma_kernel<8, RT>), dim3((T + 16 * RT - 1) / (16 * RT), H), dim3(512), (la_portion_lds<8, RT>(d + dr)), st, step, (long long)ring_off, cap, q, (long long)ldq, kv,
                       (long long)ldkv, freq, H, d, dr, rot_dims, dv, kv_rank, window, scale, T, o, (long long)ldo, rot_mag, gate, (long long)ldg, pairing);
}
void psk_latent_attn_mfma(hipStream_t st, const ps_seq_step *step, int64_t ring_off, int cap, const float *q, int64_t ldq, const float *kv, int64_t ldkv,
                          const float *freq, int H, int d, int dr, int rot_dims, int dv, int kv_rank, int window, float scale, int T, float *o, int64_t ldo, float rot_mag,
                          const float *gate, int64_t ldg, int pairing) {
    if (la_two_tiles(T, H, la_portion_lds<8, 2>(d + dr)))
        la_launch_latent<2>(st, step, ring_off, cap, q, ldq, kv, ldkv, freq, H, d, dr, rot_dims, dv, kv_rank, window, scale, T, o, ldo, rot_mag, gate, ldg, pairing);
    else
        la_launch_latent<1>(st, step, ring_off, cap, q, ldq, kv, ldkv, freq, H, d, dr, rot_dims, dv, kv_rank, window, scale, T, o, ldo, rot_mag, gate, ldg, pairing);
}

// ---------------------------------------------------------------------------------------------------- single token, absorbed
// qa[h][r] = sum_i q[h][i] Wuk[h * d + i][r]: a head's query folded into latent space, and behind it (a block of its own) its rotated part: qa [H][R + dr].  Where the queries come straight
// from the joint projection (row.y given), one more block prepares the token's ring row, which stood a launch in front: a token of
// Pupidra 2048 x 6 377 -> 371 us (two such layers).
template <typename WT>
__global__ __launch_bounds__(256) void latent_fold_q_kernel(const ps_seq_step *step, const float *q, int qstride, const WT *wuk, int d, int R, int dr, int rot_dims, const float *freq,
                                                            float rot_mag, int pairing, float *qa, long long ring_off, int cap, la_token row) {
    if (row.y) { // (uniform)
        if (blockIdx.y == 0) {
            if (blockIdx.x == 0) la_prepare(step, ring_off, cap, row, 0);
            return;
        }
    }
    const int by = (int)blockIdx.y - (row.y ? 1 : 0);
    __shared__ float part[4][64];
    const int h = blockIdx.x, r = by * 64 + (threadIdx.x & 63), grp = threadIdx.x >> 6; // block: 64 latent indices x 4 slices of the head's rows
    const float *qh = q + (long long)h * qstride;
    qa += (long long)h * (R + dr);
    if (blockIdx.y + 1 == gridDim.y) {
        const int half = rot_dims / 2;
        const float p = (float)step->pos0;
        for (int i = threadIdx.x; i < half; i += 256) {
            const float ang = p * freq[i], cs = cosf(ang) * rot_mag, sn = sinf(ang) * rot_mag;
            int pa, pb;
            la_pair(i, half, pairing, pa, pb);
            const float u = qh[d + pa], v = qh[d + pb];
            qa[R + pa] = u * cs - v * sn;
            qa[R + pb] = v * cs + u * sn;
        }
        for (int i = 2 * half + threadIdx.x; i < dr; i += 256) qa[R + i] = qh[d + i];
        return;
    }
    float a = 0.f;
    if (r < R) {
#pragma unroll 8
        for (int i = grp; i < d; i += 4) {
            float w;
            if constexpr (sizeof(WT) == 2) w = __uint_as_float((unsigned)wuk[((long long)h * d + i) * R + r] << 16);
            else w = wuk[((long long)h * d + i) * R + r];
            a = fmaf(qh[i], w, a);
        }
    }
    part[grp][threadIdx.x & 63] = a;
    __syncthreads();
    if (grp == 0 && r < R) qa[r] = part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x];
}
// o[h][x] = sum_r Wuv[h * dv + x][r] ol[h][r]: the value expansion of the attended latent.  A wave per output row.
template <typename WT>
__global__ __launch_bounds__(256) void latent_unfold_v_kernel(const float *ol, const WT *wuv, int dv, int R, int rows, float *o, const float *gate) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float *x = ol + (long long)(row / dv) * R;
    float a = 0.f;
    for (int r = lane; r < R; r += 64) {
        float w;
        if constexpr (sizeof(WT) == 2) w = __uint_as_float((unsigned)wuv[(long long)row * R + r] << 16);
        else w = wuv[(long long)row * R + r];
        a = fmaf(w, x[r], a);
    }
    a = la_wave_sum(a);
    if (lane == 0) o[row] = gate ? a / (1.f + expf(-gate[row / dv])) : a; // (the head's output gate)
}

// rows = heads (16 per block), keys = the 16 ring rows of block x's tile of the window.  The block's four waves share the tile: each multiplies a quarter of the dimensions, the four
// partial scores meet in LDS, every wave takes the soft-max of all of them (a lane: one head, four keys -- the row operand of the second product as it stands) and then a quarter of
// the value columns (groups of 64 columns, G of them per wave).  Queries, keys and values come straight from memory, requested at the start.  What bounded the form before -- a wave per
// tile, four tiles and a copy of the 16 queries in LDS per block -- was its length (272 matrix instructions in a row behind the staging) on 17 to 65 work-groups: 25 us for 540 keys of
// 512 + 64 dimensions and 32 heads; now 6.7 (and 3.4 instead of 7.2 for the merge below).  Partials: per (key tile, head) R unnormalised outputs, then the maximum and the sum.
#define LA_PIECES 9 // pieces of 16 dimensions that a wave has in flight: all of them up to 576 dimensions
template <int G>
__global__ __launch_bounds__(256) void latent_absorbed_kernel(const ps_seq_step *step, long long ring_off, int cap, const float *qa, int dr, int H, int R, int window, float scale,
                                                              float *part) {
    __shared__ __attribute__((aligned(16))) float sc[4][16 * 20];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4, h0 = blockIdx.y * 16;
    const long long p = step->pos0;
    const long long lo = p - window + 1 > 0 ? p - window + 1 : 0;
    const int j0 = blockIdx.x * 16, n = (int)(p - lo) + 1;
    if (j0 >= n) return;
    const la_src ring = la_ring(step->state + ring_off, R + dr, lo, cap); // keys counted from position lo
    const float *kr = la_row(ring, min(j0 + lr, n - 1)) + 4 * lq, *qr = qa + (long long)min(h0 + lr, H - 1) * (R + dr) + 4 * lq; // (a key or head that is not there: the last, masked below)
    const int pieces = (R + dr) / 16;
    la_f4 s4 = {0.f, 0.f, 0.f, 0.f}, v[G][4];
    for (int u0 = wave; u0 < pieces; u0 += 4 * LA_PIECES) {
        la_f4 a[LA_PIECES], b[LA_PIECES];
#pragma unroll
        for (int u = 0; u < LA_PIECES; u++) {
            const bool in = u0 + 4 * u < pieces; // (uniform)
            a[u] = in ? *(const la_f4 *)(qr + 16 * (u0 + 4 * u)) : la_f4{0.f, 0.f, 0.f, 0.f};
            b[u] = in ? *(const la_f4 *)(kr + 16 * (u0 + 4 * u)) : la_f4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int u = 0; u < LA_PIECES; u++)
            if (u0 + 4 * u < pieces)
#pragma unroll
                for (int e = 0; e < 4; e++) s4 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][e], b[u][e], s4, 0, 0, 0);
    }
#pragma unroll
    for (int kk = 0; kk < 4; kk++) { // the value of key 4 (l / 16) + kk: the order in which the soft-max leaves its weights
        const float *vr = la_row(ring, min(j0 + 4 * lq + kk, n - 1)) + 4 * lr;
#pragma unroll
        for (int g = 0; g < G; g++) v[g][kk] = 64 * (wave + 4 * g) + 4 * lr < R ? *(const la_f4 *)(vr + 64 * (wave + 4 * g)) : la_f4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < 4; i++) sc[wave][(4 * lq + i) * 20 + lr] = s4[i];
    __syncthreads();
    la_f4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; w++) s += *(const la_f4 *)(&sc[w][lr * 20 + 4 * lq]);
    float m = -INFINITY, l = 0.f, pw[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
        s[kk] = j0 + 4 * lq + kk < n ? s[kk] * scale : -INFINITY;
        m = fmaxf(m, s[kk]);
    }
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
        pw[kk] = m == -INFINITY ? 0.f : la_exp(s[kk] - m);
        l += pw[kk];
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    // partial of (tile, head): [o[R], m, l, -, -] (rows of R + 4 floats: 16-byte stores)
    float *pp = part + ((long long)blockIdx.x * H + h0) * (R + 4);
    if (wave == 0 && lq == 0 && h0 + lr < H) { pp[(long long)lr * (R + 4) + R] = m; pp[(long long)lr * (R + 4) + R + 1] = l; }
#pragma unroll
    for (int g = 0; g < G; g++) {
        const int c = 64 * (wave + 4 * g) + 4 * lr;
        if (64 * (wave + 4 * g) >= R) break; // (uniform)
        la_f4 acc[4];
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            acc[jj] = la_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < 4; kk++) acc[jj] = __builtin_amdgcn_mfma_f32_16x16x4f32(pw[kk], v[g][kk][jj], acc[jj], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (h0 + 4 * lq + i < H && c < R) *(la_f4 *)(pp + (long long)(4 * lq + i) * (R + 4) + c) = la_f4{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
    }
}
// ol[h][c] = sum_tiles exp(m_t - M) o_t[c] / sum_tiles exp(m_t - M) l_t: block = 64 columns of a head, each wave a quarter of the tiles.  The weights are kept in LDS for as many tiles as
// LA_HELD; of a longer window's every wave makes them again where it needs them (LDS for them all ended at a window of 651 000, where the launch aborted).
#define LA_HELD 16384
__global__ __launch_bounds__(256) void latent_combine_kernel(const ps_seq_step *step, const float *part, int H, int R, int window, int max_tiles, float *ol) {
    extern __shared__ float wts[]; // [max_tiles] weights exp(m_t - M), where max_tiles <= LA_HELD
    __shared__ float red[8], sum[4][64];
    const int h = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = blockIdx.y * 64 + lane;
    const long long p = step->pos0, lo = p - window + 1 > 0 ? p - window + 1 : 0;
    int nt = (int)((p - lo) / 16 + 1);
    if (nt > max_tiles) nt = max_tiles;
    const float *ph = part + (long long)h * (R + 4);
    const long long ts = (long long)H * (R + 4);
    float mx = -INFINITY;
    for (int t = tid; t < nt; t += 256) mx = fmaxf(mx, ph[t * ts + R]);
    mx = la_wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    const float M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const bool held = max_tiles <= LA_HELD;
    auto weight = [&](int t) {
        const float m = ph[t * ts + R];
        return m == -INFINITY ? 0.f : expf(m - M);
    };
    float ls = 0.f;
    for (int t = tid; t < nt; t += 256) {
        const float w = weight(t);
        if (held) wts[t] = w;
        ls = fmaf(w, ph[t * ts + R + 1], ls);
    }
    ls = la_wave_sum(ls);
    if (lane == 0) red[4 + wave] = ls;
    __syncthreads();
    float a = 0.f;
    if (c < R && held) {
#pragma unroll 8
        for (int t = wave; t < nt; t += 4) a = fmaf(wts[t], ph[t * ts + c], a);
    } else if (c < R) {
        for (int t = wave; t < nt; t += 4) a = fmaf(weight(t), ph[t * ts + c], a);
    }
    sum[wave][lane] = a;
    __syncthreads();
    if (wave == 0 && c < R) ol[(long long)h * R + c] = ((sum[0][lane] + sum[1][lane]) + (sum[2][lane] + sum[3][lane])) / (red[4] + red[5] + red[6] + red[7]);
}

bool psk_latent_absorbed_ok(int d, int dr, int dv, int R) { return R % 16 == 0 && dr % 16 == 0 && R <= 512 && R + dr <= 2480; }
size_t psk_latent_absorbed_scratch(int H, int R, int dr, int window) { return ((size_t)((window + 15) / 16 + 1) * H * (R + 4) + (size_t)H * (2 * R + dr)) * 4; }
// q [H][d + dr] (row stride qstride) -> o [H * dv]; ukv: rows uk | uv of the expansion matrix [H d + H dv][R]; scratch from psk_latent_absorbed_scratch
void psk_latent_absorbed(hipStream_t st, const ps_seq_step *step, int64_t ring_off, int cap, const float *q, int qstride, const ps_dense *ukv, const float *freq,
                         int H, int d, int dr, int rot_dims, int dv, int R, int window, float scale, float *scratch, float *o, float rot_mag, const float *gate, int pairing,
                         const psk_latent_row *row) {
    const int max_tiles = (window + 15) / 16 + 1; // (a window that does not start on a tile's edge touches one tile more)
    float *qa = scratch, *ol = qa + (size_t)H * (R + dr), *part = ol + (size_t)H * R;
    const bool bf = ukv->dtype == PS_BF16;
    const la_token prep = row ? la_token_of(*row, R, dr, rot_dims, freq, rot_mag, pairing) : la_token{};
    const dim3 fold(H, (R + 63) / 64 + 1 + (row ? 1 : 0)), grid(max_tiles, (H + 15) / 16);
    if (bf) hipLaunchKernelGGL(latent_fold_q_kernel<unsigned short>, fold, dim3(256), 0, st, step, q, qstride, (const unsigned short *)ukv->data, d, R, dr, rot_dims, freq, rot_mag, pairing, qa, (long long)ring_off, cap, prep);
    else hipLaunchKernelGGL(latent_fold_q_kernel<float>, fold, dim3(256), 0, st, step, q, qstride, (const float *)ukv->data, d, R, dr, rot_dims, freq, rot_mag, pairing, qa, (long long)ring_off, cap, prep);
    const auto attend = R <= 256 ? latent_absorbed_kernel<1> : latent_absorbed_kernel<2>;
    hipLaunchKernelGGL(attend, grid, dim3(256), 0, st, step, (long long)ring_off, cap, qa, dr, H, R, window, scale, part);
    hipLaunchKernelGGL(latent_combine_kernel, dim3(H, (R + 63) / 64), dim3(256), max_tiles <= LA_HELD ? (size_t)max_tiles * 4 : 0, st, step, part, H, R, window, max_tiles, ol);
    const int rows = H * dv;
    if (bf) hipLaunchKernelGGL(latent_unfold_v_kernel<unsigned short>, dim3((rows + 3) / 4), dim3(256), 0, st, ol, (const unsigned short *)ukv->data + (size_t)H * d * R, dv, R, rows, o, gate);
    else hipLaunchKernelGGL(latent_unfold_v_kernel<float>, dim3((rows + 3) / 4), dim3(256), 0, st, ol, (const float *)ukv->data + (size_t)H * d * R, dv, R, rows, o, gate);
}
