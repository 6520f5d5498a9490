// One 16-row x 16-key step of soft-max attention on the fp32 matrix cores (v_mfma_f32_16x16x4_f32), shared by the attention kernels of the
// layer-list models (k_latent.hip, k_winattn.hip):
//   scores   S[16 x 16] = Q[16 x DK] K^T: the keys come straight from memory as 16-byte pieces (lane (key l % 16, quarter l / 16) holds 4
//            consecutive dimensions; the row operand is read from LDS in the same order, so the sum runs over a permutation of the dimensions)
//   soft-max online, in the accumulator layout (lane holds rows 4 (l / 16) + i of key column l % 16; a row's 16 lanes reduce by rotations)
//   output   O[16 x DV] += P V: P goes through a 16 x 17 LDS patch into the row-operand layout; V comes as 16-byte pieces of 4 consecutive
//            columns, so accumulator tile jj of a 64-column group holds columns 4 (l % 16) + jj -- undone at the final store.
// A "row" is a (token, head) pair.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

typedef float la_f4 __attribute__((ext_vector_type(4)));

struct la_src { // where key j (counted from the first visible one) lives: row j + off of base, wrapped once at `mod` (0: no wrap); la_ring: the rows of a ring from position `first` on
    const float *base;
    long long ld;
    int mod, off;
};
static __device__ __forceinline__ la_src la_ring(const float *base, long long ld, long long first, int cap) { return {base, ld, cap, (int)(first % cap)}; }
static __device__ __forceinline__ const float *la_row(const la_src &s, int j) {
    int r = j + s.off;
    if (s.mod > 0 && r >= s.mod) r -= s.mod; // (fewer than mod keys are ever visible)
    return s.base + r * s.ld;
}
// reductions over the 16 lanes of a row, every lane gets the result (rotations inside the row: VALU moves, no trip through LDS)
template <int R>
static __device__ __forceinline__ float la_ror(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + R, 0xf, 0xf, true)); }
static __device__ __forceinline__ float la_max16(float v) {
    v = fmaxf(v, la_ror<8>(v)); v = fmaxf(v, la_ror<4>(v)); v = fmaxf(v, la_ror<2>(v));
    return fmaxf(v, la_ror<1>(v));
}
static __device__ __forceinline__ float la_sum16(float v) {
    v += la_ror<8>(v); v += la_ror<4>(v); v += la_ror<2>(v);
    return v + la_ror<1>(v);
}
// e^x for x <= 0: the hardware's 2^y on y = x log2 e, what y lost in rounding put back (both parts of log2 e): as exact as expf here
static __device__ __forceinline__ float la_exp(float x) {
    const float y = x * 1.44269504f, lo = fmaf(x, 1.44269504f, -y) + x * 1.92596299e-8f;
    const float e = __builtin_amdgcn_exp2f(y);
    return x < -104.f ? 0.f : fmaf(e, lo * 0.693147181f, e);
}

// RT x 16 rows against the 16 keys j0 .. j0 + 15 of those the sources hold, jend of them.  qs: the rows in LDS, row stride qld floats, [DK1 | DK2]; pt: the wave's RT patches of
// 16 x 17.  see: see.sees(r, i, j) -- does accumulator row i of tile r of this lane (row 16 r + 4 (l / 16) + i) see key j (asked for j < jend; false for a row that does not exist);
// DIST: see.minus(r, i, j) is taken off the score behind scale and soft cap.  NJ: accumulator tiles (DV <= 16 NJ).
// The tiles share every key and value piece.  The value pieces of the first 128 columns are requested in front of the soft-max.
template <int NJ, int RT, bool DIST, class SEE>
static __device__ __forceinline__ void la_tiles(const float *qs, int qld, float *pt, const la_src &k1, const la_src &k2, const la_src &vs, int DK1, int DK2, int DV,
                                                int j0, int jend, const SEE &see, float scale, float (&m)[RT][4], float (&l)[RT][4], la_f4 (&acc)[RT][NJ],
                                                float softcap = 0.f) { // softcap > 0: score <- softcap tanh(score / softcap) behind the scale
    const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
    const int jk = j0 + lr < jend ? j0 + lr : jend - 1; // (a key row that exists; masked below)
    la_f4 s4[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) s4[r] = la_f4{0.f, 0.f, 0.f, 0.f};
    const float *kr1 = la_row(k1, jk) + 4 * lq, *kr2 = la_row(k2, jk) + 4 * lq, *qr = qs + lr * qld + 4 * lq;
    // eight 16-byte key pieces in flight per lane ahead of their matrix instructions
    for (int g0 = 0; g0 < DK1 + DK2; g0 += 128) {
        la_f4 b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int g = g0 + 16 * u;
            b[u] = g < DK1 ? *(const la_f4 *)(kr1 + g) : (g < DK1 + DK2 ? *(const la_f4 *)(kr2 + (g - DK1)) : la_f4{0.f, 0.f, 0.f, 0.f});
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int g = g0 + 16 * u;
            if (g < DK1 + DK2) {
                la_f4 a[RT];
#pragma unroll
                for (int r = 0; r < RT; r++) a[r] = *(const la_f4 *)(qr + r * 16 * qld + g);
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int r = 0; r < RT; r++) s4[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r][e], b[u][e], s4[r], 0, 0, 0);
            }
        }
    }
    const float *vr[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int jv = j0 + 4 * s + lq < jend ? j0 + 4 * s + lq : jend - 1; // (weight 0 beyond the end)
        vr[s] = la_row(vs, jv) + 4 * lr;
    }
    constexpr int AHEAD = NJ >= 8 ? 2 : 1;
    la_f4 bn[AHEAD][4];
#pragma unroll
    for (int x = 0; x < AHEAD; x++)
#pragma unroll
        for (int s = 0; s < 4; s++) bn[x][s] = 64 * x + 4 * lr < DV ? *(const la_f4 *)(vr[s] + 64 * x) : la_f4{0.f, 0.f, 0.f, 0.f};
    const int j = j0 + lr;
    float corr[RT][4], pa[RT][4];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool vis = j < jend && see.sees(r, i, j);
            float sv = s4[r][i] * scale;
            if (softcap > 0.f) sv = softcap * tanhf(sv / softcap);
            if constexpr (DIST) sv -= see.minus(r, i, j);
            const float s = vis ? sv : -INFINITY;
            const float mn = fmaxf(m[r][i], la_max16(s));
            corr[r][i] = mn == -INFINITY ? 1.f : la_exp(m[r][i] - mn);
            p[i] = mn == -INFINITY ? 0.f : la_exp(s - mn);
            l[r][i] = l[r][i] * corr[r][i] + la_sum16(p[i]);
            m[r][i] = mn;
        }
        float *pr = pt + r * 16 * 17;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 4; i++) pr[(4 * lq + i) * 17 + lr] = p[i];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < 4; s++) pa[r][s] = pr[lr * 17 + 4 * s + lq];
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int J = 0; J < NJ / 4; J++) {
        if (64 * J < DV) { // (uniform)
            la_f4 b[4];
#pragma unroll
            for (int s = 0; s < 4; s++) b[s] = bn[J % AHEAD][s];
            if (J + AHEAD < NJ / 4 && 64 * (J + AHEAD) < DV) { // the pieces AHEAD groups of 64 columns on are requested before this group's matrix instructions
                const bool in = 64 * (J + AHEAD) + 4 * lr < DV;
#pragma unroll
                for (int s = 0; s < 4; s++) bn[J % AHEAD][s] = in ? *(const la_f4 *)(vr[s] + 64 * (J + AHEAD)) : la_f4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int jj = 0; jj < 4; jj++) {
                    la_f4 a = acc[r][4 * J + jj];
#pragma unroll
                    for (int i = 0; i < 4; i++) a[i] *= corr[r][i];
#pragma unroll
                    for (int s = 0; s < 4; s++) a = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[r][s], b[s][jj], a, 0, 0, 0);
                    acc[r][4 * J + jj] = a;
                }
        }
    }
}

// What wave `from` of a block has gathered over its keys joins what wave `to` has (both hold the same rows): rescaled to the larger maximum, added.  Through LDS, [value][lane], a slot of
// la_merge_floats per pair; every wave of the block calls this, `give` / `take` say what it does (slot: which pair's).
template <int NJ, int RT>
constexpr int la_merge_floats() { return RT * (NJ + 2) * 4 * 64; }
template <int NJ, int RT>
static __device__ __forceinline__ void la_merge(float *lds, int slot, bool give, bool take, float (&m)[RT][4], float (&l)[RT][4], la_f4 (&acc)[RT][NJ]) {
    float *at = lds + slot * la_merge_floats<NJ, RT>() + (threadIdx.x & 63) * 4;
    __syncthreads();
    if (give) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            float *q = at + r * (NJ + 2) * 256;
            *(la_f4 *)q = la_f4{m[r][0], m[r][1], m[r][2], m[r][3]};
            *(la_f4 *)(q + 256) = la_f4{l[r][0], l[r][1], l[r][2], l[r][3]};
#pragma unroll
            for (int j = 0; j < NJ; j++) *(la_f4 *)(q + (2 + j) * 256) = acc[r][j];
        }
    }
    __syncthreads();
    if (take) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            const float *q = at + r * (NJ + 2) * 256;
            const la_f4 mo = *(const la_f4 *)q, lo = *(const la_f4 *)(q + 256);
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float mn = fmaxf(m[r][i], mo[i]);
                a[i] = mn == -INFINITY ? 1.f : la_exp(m[r][i] - mn);
                b[i] = mn == -INFINITY ? 0.f : la_exp(mo[i] - mn);
                l[r][i] = l[r][i] * a[i] + lo[i] * b[i];
                m[r][i] = mn;
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const la_f4 v = *(const la_f4 *)(q + (2 + j) * 256);
#pragma unroll
                for (int i = 0; i < 4; i++) acc[r][j][i] = acc[r][j][i] * a[i] + v[i] * b[i];
            }
        }
    }
}
// eight waves' results into wave 0's
template <int NJ, int RT>
static __device__ __forceinline__ void la_merge8(float *lds, float (&m)[RT][4], float (&l)[RT][4], la_f4 (&acc)[RT][NJ]) {
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int n = 4; n > 0; n >>= 1) la_merge<NJ, RT>(lds, wave & (n - 1), wave >= n && wave < 2 * n, wave < n, m, l, acc);
}
// dynamic LDS of a portion's block: query rows and patches, or the merge's four slots, whichever is more
template <int NJ, int RT>
static constexpr size_t la_portion_lds(int dk) {
    const size_t rows = (size_t)RT * 16 * (dk + 4) + 8 * RT * 16 * 17, merge = 4 * (size_t)la_merge_floats<NJ, RT>();
    return (rows > merge ? rows : merge) * 4;
}
// what the rows of a portion's block see of a window's keys: row n is the token at `q0 + n` in the keys' counting, it sees itself and the window - 1 in front of it (rows: how many exist)
struct la_window {
    int q0, window, rows, lq;
    float slope;
    __device__ __forceinline__ bool sees(int r, int i, int j) const {
        const int n = 16 * r + 4 * lq + i, gap = q0 + n - j;
        return n < rows && gap >= 0 && gap < window;
    }
    __device__ __forceinline__ float minus(int r, int i, int j) const { return slope * (float)(q0 + 16 * r + 4 * lq + i - j); }
};
// Two row tiles per block where that still leaves half the chip's CUs a block (a key piece then serves both); one for a few tokens, or where two do not fit LDS.
static inline bool la_two_tiles(int T, int H, size_t lds) { return T > 16 && (long long)((T + 31) / 32) * H >= 128 && lds <= 160 * 1024; }
