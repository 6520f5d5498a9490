// Soft-max attention of a portion's many rows with fp32 operands on the bf16 matrix instruction (v_mfma_f32_16x16x32_bf16): every operand is the sum of three bf16 numbers -- rounded, the
// rounded rest, the rest of that, 24 bits together -- and a product the six of the nine partial products that are not below 2^-24 of it, accumulated in fp32 (the leading ones and the others
// apart).  Each of those is exact, and a sum of 192 passes 36 roundings where v_mfma_f32_16x16x4_f32 has one for each of its 48 steps; six of the fast instructions cost 96 clocks where the
// fp32 one's eight steps cost 256.  The serving layers' forms (k_latent.hip, k_winattn.hip: portions of any size, and what this does not take) run on the fp32 instruction.
//   split_keys_kernel   the keys and values a portion sees, in blocks of 32 and split, as the images the attention's stages are filled with: 1 KB per instruction operand in lane order
//   split_attn_kernel   128 rows (consecutive tokens) of one head per work-group, a wave 16 of them against all keys; blocks of 32 keys through two LDS stages
// S^T = K Q^T, so that a lane has one row: maximum and sum run over its own registers, two lane moves join the four lanes of a row.  D's rows are the keys 4 (l / 16) + i of two tiles, and the
// second product, O^T = V^T P^T, takes its 32 keys in any order that both operands share: a lane's eight weights are its piece of the operand as they are, and the value images are laid out so.
// What bounded the fp32 form: 2560 clocks of matrix instructions per 16 x 16 scores beside as much again of soft-max in its accumulator layout (four moves per row reduction, weights turned
// in LDS), keys straight from the L2s for 32 rows at a time.  2047 tokens of 16 heads, keys of 192, a window of 1024: 318 -> 141 us, 17 of them the images; 3 us a block of 32 keys and
// work-group, 1.9 of it matrix instructions; without its reads, its requests or its soft-max it is 0.7, 0.3 and 0.5 less.  (The second wave of every SIMD a block behind with its second product, so
// that its soft-max runs beside the others' products: 137 us without the images against 126.)  Error against 64 bits over four seeds: keys of 192 5.6e-7 -> 5.4e-7, 128 with slopes 6.4e-7 -> 4.1e-7.
#include "ps_seq.h"

#include <cmath>

typedef float sa_f4 __attribute__((ext_vector_type(4)));
typedef float sa_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 sa_b2 __attribute__((ext_vector_type(2)));
typedef __bf16 sa_b8 __attribute__((ext_vector_type(8)));
typedef unsigned sa_u4 __attribute__((ext_vector_type(4)));

static __device__ __forceinline__ unsigned sa_round2(float a, float b) { // two numbers to bf16, to nearest even
    const sa_b2 r = __builtin_convertvector((sa_f2){a, b}, sa_b2);
    unsigned u;
    __builtin_memcpy(&u, &r, 4);
    return u;
}
static __device__ __forceinline__ bool sa_finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }
// Two numbers as three pairs.  WIDE: any numbers -- one that rounds to infinity is cut off instead, infinity has no rest (weights of a soft-max are at most 1).
template <bool WIDE>
static __device__ __forceinline__ void sa_split2(float a, float b, unsigned &u1, unsigned &u2, unsigned &u3) {
    u1 = sa_round2(a, b);
    float a1 = __uint_as_float(u1 << 16), b1 = __uint_as_float(u1 & 0xffff0000u);
    if constexpr (WIDE) {
        if (__builtin_isinf(a1)) { u1 = (u1 & 0xffff0000u) | (__float_as_uint(a) >> 16); a1 = __uint_as_float(u1 << 16); }
        if (__builtin_isinf(b1)) { u1 = (u1 & 0xffffu) | (__float_as_uint(b) & 0xffff0000u); b1 = __uint_as_float(u1 & 0xffff0000u); }
    }
    float ra = a - a1, rb = b - b1;
    if constexpr (WIDE) {
        if (__builtin_isinf(a1)) ra = 0.f;
        if (__builtin_isinf(b1)) rb = 0.f;
    }
    u2 = sa_round2(ra, rb);
    u3 = sa_round2(ra - __uint_as_float(u2 << 16), rb - __uint_as_float(u2 & 0xffff0000u));
}
template <bool WIDE>
static __device__ __forceinline__ void sa_split8(const float (&v)[8], sa_u4 (&p)[3]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
        unsigned a, b, c;
        sa_split2<WIDE>(v[2 * e], v[2 * e + 1], a, b, c);
        p[0][e] = a; p[1][e] = b; p[2][e] = c;
    }
}
static __device__ __forceinline__ void sa_join8(const sa_u4 (&p)[3], float (&v)[8]) { // back (the sum is exact)
#pragma unroll
    for (int e = 0; e < 8; e++) {
        auto line = [&](const int x) { return __uint_as_float(e & 1 ? p[x][e >> 1] & 0xffff0000u : p[x][e >> 1] << 16); };
        v[e] = line(0) + (line(1) + line(2));
    }
}
static __device__ __forceinline__ sa_f4 sa_mfma(const sa_u4 &a, const sa_u4 &b, const sa_f4 &c) {
    sa_b8 x, y;
    __builtin_memcpy(&x, &a, 16);
    __builtin_memcpy(&y, &b, 16);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
}
// e^x for x <= 0 (ps_attn_dev.h la_exp)
static __device__ __forceinline__ float sa_exp(float x) {
    const float y = x * 1.44269504f, lo = fmaf(x, 1.44269504f, -y) + x * 1.92596299e-8f;
    const float e = __builtin_amdgcn_exp2f(y);
    return x < -104.f ? 0.f : fmaf(e, lo * 0.693147181f, e);
}
static __device__ __forceinline__ float sa_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

// ---------------------------------------------------------------------------------------------------- images
// Block b of head (or key / value group) g: rows 32 b .. of the front store for b < nbf, else window rows 32 (b - nbf) ..; rows beyond the last are zeros.  The image: [k step][plane][16 keys][lane]
// 16 bytes, then [16 value columns][plane][lane].  blockIdx.y == G: the key parts that all heads share, an image of their own.
struct sa_rows { // window row j (counted from the portion's first visible position) = row j + off of base, wrapped once at mod (0: no wrap)
    const float *base;
    long long ld;
    int mod, off;
};
struct sa_keys {
    sa_rows k, v, shared;  // of group g: base + g * k_step / v_step; shared: the same for all
    long long k_step, v_step;
    const float *front_k, *front_v;
    long long front_ld;
    int n_front, n_window, nbf, nb; // rows; blocks of the front store, blocks in all
    int ks_own, ks_shared, nj;      // k steps of 32 numbers of a head's own key part and of the shared one, value tiles of 16 columns
    int G;
    char *img, *img_shared;
};
static __device__ __forceinline__ const float *sa_row(const sa_rows &r, long long step, int j) {
    int n = j + r.off;
    if (r.mod > 0 && n >= r.mod) n -= r.mod;
    return r.base + step + n * r.ld;
}
__global__ __launch_bounds__(256) void split_keys_kernel(sa_keys a) {
    const int b = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
    const bool shared = g == a.G, front = b < a.nbf;
    const int i0 = 32 * (front ? b : b - a.nbf), n = front ? a.n_front : a.n_window; // rows i0 .. i0 + 31 of those that exist
    const int ks = shared ? a.ks_shared : a.ks_own, nk = ks * 128, nv = shared ? 0 : a.nj * 64; // sixteen-byte pieces per plane
    char *out = shared ? a.img_shared + (size_t)b * a.ks_shared * 6144 : a.img + ((size_t)g * a.nb + b) * (a.ks_own * 6144 + a.nj * 3072);
    for (int x = tid; x < nk + nv; x += 256) {
        float v[8];
        sa_u4 p[3];
        const int lane = x & 63;
        if (x < nk) {
            const int tile = (x >> 6) & 1, s = x >> 7, i = i0 + 16 * tile + (lane & 15);
            const float *row = front ? a.front_k + g * a.k_step + i * a.front_ld : shared ? sa_row(a.shared, 0, i) : sa_row(a.k, g * a.k_step, i);
            if (i < n) {
                *(sa_f4 *)v = *(const sa_f4 *)(row + 32 * s + 8 * (lane >> 4));
                *(sa_f4 *)(v + 4) = *(const sa_f4 *)(row + 32 * s + 8 * (lane >> 4) + 4);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = 0.f;
            }
            sa_split8<true>(v, p);
#pragma unroll
            for (int q = 0; q < 3; q++) *(sa_u4 *)(out + ((s * 3 + q) * 2 + tile) * 1024 + lane * 16) = p[q];
        } else {
            const int ct = (x - nk) >> 6, c = 16 * ct + (lane & 15);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int i = i0 + 16 * (e >> 2) + 4 * (lane >> 4) + (e & 3);
                v[e] = i < n ? (front ? a.front_v + g * a.v_step + i * a.front_ld : sa_row(a.v, g * a.v_step, i))[c] : 0.f;
            }
            sa_split8<true>(v, p);
#pragma unroll
            for (int q = 0; q < 3; q++) *(sa_u4 *)(out + ks * 6144 + (ct * 3 + q) * 1024 + lane * 16) = p[q];
        }
    }
}

// ---------------------------------------------------------------------------------------------------- attention
struct sa_attn {
    const char *img, *img_shared;
    int nbf, nb, ks_own, hpg;      // (heads per image)
    int pos0, first, T, window, pool, keep; // position of row 0, of window row 0
    const float *q;
    long long ldq;
    int d, rot_at, rot_dims, pairing; // numbers of a head's query; its rotated part begins at rot_at (rot_dims 0: it comes rotated)
    const float *freq;
    float rot_mag, scale, softcap;
    const float *temp, *slope, *sink, *gate;
    long long ldg;
    int gate_elem;
    float *o;
    long long ldo;
};
static __device__ __forceinline__ void sa_dma(const char *base, unsigned off, unsigned lds_dst) { // one wave-instruction: lane l's 16 bytes at base + off go to lds_dst + 16 l
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(base), "s"(lds_dst) : "memory");
}
#define SA_ROWS 128
template <int KS, int NJ>
static constexpr int sa_lds() { // two stages; before the second one is filled the queries lie there
    const int q = SA_ROWS * (KS * 32 + 4) * 4, s = KS * 6144 + NJ * 3072;
    return s + (q > s ? q : s);
}
template <int KS, int NJ, bool DIST>
__global__ __launch_bounds__(512) void split_attn_kernel(sa_attn a) {
    extern __shared__ __attribute__((aligned(16))) char sa_smem[];
    constexpr int STAGE = KS * 6144 + NJ * 3072, PIECES = KS * 6 + NJ * 3, QLD = KS * 32 + 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lq = lane >> 4;
    const int h = blockIdx.x, t0 = SA_ROWS * ((int)gridDim.y - 1 - (int)blockIdx.y), g = h / a.hpg; // (the rows with the most keys first)
    const int rows = min(SA_ROWS, a.T - t0), n = 16 * wave + lr, p = a.pos0 + t0 + n;               // this lane's row and its position
    // blocks of this work-group: those of the front store that its last row sees, then the window's from the first row's first key to the last row's own
    const int plast = a.pos0 + t0 + rows - 1, pfirst = a.pos0 + t0;
    int nf = plast - a.window + 1;
    nf = nf <= 0 ? 0 : a.pool > 0 ? nf / a.pool : min(nf, a.keep);
    const int nfb = (nf + 31) / 32, wlo = max(pfirst - a.window + 1, 0) - a.first, wb0 = wlo / 32, nwb = (plast - a.first) / 32 - wb0 + 1, blocks = nfb + nwb;
    const int own = a.ks_own * 6, image = own + NJ * 3; // pieces of a head's own key part, of its image
    const unsigned lds0 = (unsigned)(size_t)(const __attribute__((address_space(3))) char *)sa_smem;
    auto block_of = [&](const int it) { return it < nfb ? it : a.nbf + wb0 + it - nfb; };
    auto request = [&](const int it) {
        const int b = block_of(it);
        const char *im = a.img + ((size_t)g * a.nb + b) * (image * 1024), *sh = a.img_shared + (size_t)b * ((KS * 6 - own) * 1024);
#pragma unroll
        for (int x = 0; x < (PIECES + 7) / 8; x++) {
            const int pc = x * 8 + wave;
            if (pc < PIECES) sa_dma(pc < own ? im + pc * 1024 : pc < KS * 6 ? sh + (pc - own) * 1024 : im + (pc - KS * 6 + own) * 1024, lane * 16, lds0 + (unsigned)((it & 1) * STAGE + pc * 1024));
        }
    };
    request(0);
    // this wave's query rows, rotated, through LDS (behind the first stage) into its operand registers
    float *qs = (float *)(sa_smem + STAGE) + 16 * wave * QLD;
    const int half = a.rot_dims / 2;
    // (sixteen rows' numbers requested at a time; rows that do not exist repeat the last one)
    const float *qw = a.q + (long long)h * a.d;
    auto row_at = [&](const int r) { return qw + (long long)min(t0 + 16 * wave + r, a.T - 1) * a.ldq; };
    for (int c = lane; c < a.d; c += 64) {
        float x[16];
#pragma unroll
        for (int r = 0; r < 16; r++) x[r] = row_at(r)[c];
#pragma unroll
        for (int r = 0; r < 16; r++) qs[r * QLD + c] = x[r];
    }
    for (int x = lane; x < 16 * half; x += 64) { // (a wave's rows are its own: no barrier)
        const int r = x / half, i = x - r * half;
        float *pa = qs + r * QLD + a.rot_at + (a.pairing == PS_ROT_NEIGHBOURS ? 2 * i : i), *pb = pa + (a.pairing == PS_ROT_NEIGHBOURS ? 1 : half);
        const float ang = (float)(a.pos0 + t0 + 16 * wave + r) * a.freq[i], cs = cosf(ang) * a.rot_mag, sn = sinf(ang) * a.rot_mag, u = *pa, v = *pb;
        *pa = u * cs - v * sn;
        *pb = v * cs + u * sn;
    }
    __syncthreads();
    sa_u4 q[KS][3];
#pragma unroll
    for (int s = 0; s < KS; s++) {
        float v[8];
        *(sa_f4 *)v = *(const sa_f4 *)(qs + lr * QLD + 32 * s + 8 * lq);
        *(sa_f4 *)(v + 4) = *(const sa_f4 *)(qs + lr * QLD + 32 * s + 8 * lq + 4);
        sa_split8<true>(v, q[s]);
    }
    const float sc = a.scale * (a.temp ? a.temp[h] : 1.f), slope = DIST ? a.slope[h] : 0.f;
    float m = -INFINITY, l = 0.f; // (l: of this lane's own keys)
    sa_f4 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[j] = sa_f4{0.f, 0.f, 0.f, 0.f};
    const int w0 = pfirst + 16 * wave, w1 = w0 + 15; // positions of the wave's rows
    const bool alive = 16 * wave < rows;
    struct place { bool front, none, all; int j0, kp0; }; // of a block: nothing of it visible to the wave, or all of it to every row of it (uniform)
    auto place_of = [&](const int it) {
        place b;
        b.front = it < nfb;
        b.j0 = b.front ? 32 * it : 32 * (wb0 + it - nfb); // first row of the block, in the front store or behind `first`
        b.kp0 = b.front ? b.j0 : a.first + b.j0;          // (kept first tokens: their positions)
        if (b.front) {
            const int o0 = w0 - a.window + 1, o1 = w1 - a.window + 1; // positions in front of the first and the last row's window
            b.none = a.pool > 0 ? (b.j0 + 1) * a.pool > o1 : b.j0 >= o1;
            b.all = a.pool > 0 ? (b.j0 + 32) * a.pool <= o0 : b.j0 + 31 < o0 && b.j0 + 31 < a.keep;
        } else {
            b.none = b.kp0 > w1 || b.kp0 + 31 <= w0 - a.window;
            b.all = b.kp0 + 31 <= w0 && b.kp0 > w1 - a.window;
        }
        return b;
    };
    auto sees = [&](const place &b, const int i) { // this lane's row the block's key i
        const int out = p - a.window + 1;
        return b.front ? (a.pool > 0 ? (b.j0 + i + 1) * a.pool <= out : b.j0 + i < out && b.j0 + i < a.keep) : b.kp0 + i <= p && b.kp0 + i >= out;
    };
    // a block's products -> its weights; what was gathered in front of it is rescaled to the new maximum
    auto soften = [&](const place &b, float (&e)[8]) {
#pragma unroll
        for (int x = 0; x < 8; x++) {
            float v = e[x] * sc;
            if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
            const int kp = b.kp0 + 16 * (x >> 2) + 4 * lq + (x & 3);
            if constexpr (DIST) v -= slope * (float)(p - kp);
            e[x] = v;
        }
        if (!b.all) {
#pragma unroll
            for (int x = 0; x < 8; x++)
                if (!sees(b, 16 * (x >> 2) + 4 * lq + (x & 3))) e[x] = -INFINITY;
        }
        float mx = e[0];
#pragma unroll
        for (int x = 1; x < 8; x++) mx = fmaxf(mx, e[x]);
        {
            auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
            auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(r2[0]), __uint_as_float(r2[1]));
        }
        const float mn = fmaxf(m, mx);
        if (__any(mn > m)) { // (uniform)
            const float corr = mn == -INFINITY ? 1.f : sa_exp(m - mn);
            l *= corr;
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[j][i] *= corr;
            m = mn;
        }
        const float off = m == -INFINITY ? 0.f : m; // (a row that has seen nothing yet: its weights are e^-inf)
#pragma unroll
        for (int x = 0; x < 8; x++) { e[x] = sa_exp(e[x] - off); l += e[x]; }
    };
    for (int it = 0; it < blocks; it++) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); // the block has landed (this wave's share); the reads of the one before are back
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (it + 1 < blocks) request(it + 1);
        const place b = place_of(it);
        if (!alive || b.none) continue;
        const char *st = sa_smem + (it & 1) * STAGE + lane * 16;
        sa_f4 s1[2], s2[2], s3[2]; // (chains of their own)
#pragma unroll
        for (int u = 0; u < 2; u++) s1[u] = s2[u] = s3[u] = sa_f4{0.f, 0.f, 0.f, 0.f};
        sa_u4 kf[2][3][2];
        auto read_k = [&](const int s) {
#pragma unroll
            for (int x = 0; x < 3; x++)
#pragma unroll
                for (int u = 0; u < 2; u++) kf[s & 1][x][u] = *(const sa_u4 *)(st + ((s * 3 + x) * 2 + u) * 1024);
            __builtin_amdgcn_sched_barrier(0);
        };
        read_k(0);
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (s + 1 < KS) read_k(s + 1);
            const sa_u4 (&k)[3][2] = kf[s & 1];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                s1[u] = sa_mfma(k[0][u], q[s][0], s1[u]);
                s2[u] = sa_mfma(k[2][u], q[s][0], s2[u]);
                s3[u] = sa_mfma(k[1][u], q[s][1], s3[u]);
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                s2[u] = sa_mfma(k[0][u], q[s][2], s2[u]);
                s3[u] = sa_mfma(k[1][u], q[s][0], s3[u]);
            }
#pragma unroll
            for (int u = 0; u < 2; u++) s2[u] = sa_mfma(k[0][u], q[s][1], s2[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
        float e[8];
#pragma unroll
        for (int x = 0; x < 8; x++) e[x] = s1[x >> 2][x & 3] + (s2[x >> 2][x & 3] + s3[x >> 2][x & 3]);
        soften(b, e);
        sa_u4 w[3], vf[2][2][3]; // (two column tiles side by side, the next two's pieces read in front of their products)
        sa_split8<false>(e, w);
        auto read_v = [&](const int j) {
#pragma unroll
            for (int y = 0; y < 2; y++)
#pragma unroll
                for (int x = 0; x < 3; x++) vf[(j >> 1) & 1][y][x] = *(const sa_u4 *)(st + KS * 6144 + ((j + y) * 3 + x) * 1024);
            __builtin_amdgcn_sched_barrier(0);
        };
        read_v(0);
#pragma unroll
        for (int j = 0; j < NJ; j += 2) {
            if (j + 2 < NJ) read_v(j + 2);
            const sa_u4 (&v)[2][3] = vf[(j >> 1) & 1];
#pragma unroll
            for (int z = 0; z < 6; z++) // (the small ones first)
#pragma unroll
                for (int y = 0; y < 2; y++) {
                    constexpr int vi[6] = {2, 1, 0, 1, 0, 0}, wi[6] = {0, 1, 2, 0, 1, 0};
                    acc[j + y] = sa_mfma(v[y][vi[z]], w[wi[z]], acc[j + y]);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (!alive) return;
    // An infinite number's lower lines are zeros that the other operand's leading line meets, and it meets the other's lower lines, whose signs are their own: the infinite number that fp32 arithmetic
    // has, or no number; and one of a key that a row does not see meets its weight's zeros.  No number among the scores ends in the sum of the weights, among the products in the results: where a row
    // of the wave has one there, or an infinite one, the wave does it all again with the lines joined, on the fp32 instruction, the images straight from memory.
    float odd = l * 0.f;
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) odd = fmaf(acc[j][i], 0.f, odd);
    if (__builtin_expect(__any(!sa_finite(odd)), 0)) { // (uniform)
        m = -INFINITY;
        l = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[j] = sa_f4{0.f, 0.f, 0.f, 0.f};
        for (int it = 0; it < blocks; it++) {
            const place b = place_of(it);
            if (b.none) continue;
            const char *im = a.img + ((size_t)g * a.nb + block_of(it)) * (image * 1024) + lane * 16, *sh = a.img_shared + (size_t)block_of(it) * ((KS * 6 - own) * 1024) + lane * 16;
            sa_u4 lines[3];
            float v[8], y[8], e[8];
            sa_f4 s1[2] = {sa_f4{0.f, 0.f, 0.f, 0.f}, sa_f4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const char *ks = 6 * s < own ? im + s * 6144 : sh + (6 * s - own) * 1024;
                sa_join8(q[s], y);
#pragma unroll
                for (int u = 0; u < 2; u++) {
#pragma unroll
                    for (int x = 0; x < 3; x++) lines[x] = *(const sa_u4 *)(ks + (2 * x + u) * 1024);
                    sa_join8(lines, v);
#pragma unroll
                    for (int i = 0; i < 8; i++) s1[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[i], y[i], s1[u], 0, 0, 0);
                }
            }
#pragma unroll
            for (int x = 0; x < 8; x++) e[x] = s1[x >> 2][x & 3];
            soften(b, e);
#pragma unroll 1
            for (int j = 0; j < NJ; j++) {
#pragma unroll
                for (int x = 0; x < 3; x++) lines[x] = *(const sa_u4 *)(im + (own + j * 3 + x) * 1024);
                sa_join8(lines, v);
                sa_f4 t = sa_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int x = 0; x < 8; x++) {
                    t = __builtin_amdgcn_mfma_f32_16x16x4f32(sa_finite(v[x]) ? v[x] : 0.f, e[x], t, 0, 0, 0);
                    if (__all(sa_finite(v[x]))) continue; // (uniform)
                    for (int z = 0; z < 4; z++) { // a value that is not finite: for the rows that see its key, and no others
                        const float wz = __shfl(e[x], lr + 16 * z, 64);
                        const bool seen = sees(b, 16 * (x >> 2) + 4 * z + (x & 3));
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const float vz = __shfl(v[x], 4 * lq + i + 16 * z, 64);
                            if (seen && !sa_finite(vz)) t[i] += vz * wz;
                        }
                    }
                }
#pragma unroll
                for (int y = 0; y < NJ; y++) // (registers)
                    if (y == j) acc[y] += t;
            }
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const int t = t0 + n;
    if (n >= rows) return;
    float f;
    if (a.sink) { // (k_winattn.hip wa_finish)
        const float sk = a.sink[h], M = fmaxf(m, sk), c = expf(m - M);
        f = c / (l * c + expf(sk - M));
    } else {
        f = 1.f / l;
    }
    if (a.gate && !a.gate_elem) f *= sa_sigmoid(a.gate[(long long)t * a.ldg + h]);
    float *o = a.o + (long long)t * a.ldo + (long long)h * (16 * NJ) + 4 * lq;
    const float *ge = a.gate && a.gate_elem ? a.gate + (long long)t * a.ldg + (long long)h * (16 * NJ) + 4 * lq : nullptr;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        sa_f4 v = sa_f4{acc[j][0] * f, acc[j][1] * f, acc[j][2] * f, acc[j][3] * f};
        if (ge) {
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] *= sa_sigmoid(ge[16 * j + i]);
        }
        *(sa_f4 *)(o + 16 * j) = v;
    }
}

// ---------------------------------------------------------------------------------------------------- host
bool psk_split_attn_ok(int own, int shared, int dv) { return dv == 128 && own % 32 == 0 && shared % 32 == 0 && (own + shared == 128 || own + shared == 192); }
// From 80 work-groups on: below, the fp32 form's eight waves per 32 rows hide more than the faster instruction saves.  Attention of a layer in us, fp32 form | this one with its images (keys of
// 192; behind nothing and behind 1024 tokens): 64 work-groups (512 tokens of 16 heads) 50 | 68, 84 | 132; 96 (768 of 16; 384 of 32) 110 | 95, 162 | 135; 70 | 57, 160 | 141; 128 156 | 120,
// 166 | 137; 256 (2047 of 16, 1000 of 32) 318 | 142; 302 | 128, 319 | 160; keys of 128 with slopes: 1500 of 16 198 | 110.
// And from where 16 rows and a head make more than 512: as many the fp32 form has at once on the chip, so fewer take it one pass however many heads there are, while this form splits the window's
// numbers first for rows that fill little of a work-group.  A request of one layer in us, fp32 form | this one, behind 64 and behind 1000 tokens (windows, keys of 128): 80 heads, 1 row 59 | 67,
// 64 | 117; 96 rows 107 | 109, 160 | 176; 112 rows 131 | 110, 224 | 181; 40 heads, 192 rows 99 | 103, 149 | 168; 224 rows 123 | 109, 219 | 173; 64 heads, 128 rows 102 | 108, 152 | 176;
// 129 rows 126 | 113, 221 | 182; 128 heads, 64 rows 117 | 119, 173 | 188; 80 rows 139 | 127, 231 | 210.
bool psk_split_attn_takes(int T, int H) { return (int64_t)((T + SA_ROWS - 1) / SA_ROWS) * H >= 80 && (int64_t)((T + 15) / 16) * H > 512; }
static size_t sa_images(int G, int own, int shared, int dv, int64_t blocks) { return (size_t)blocks * ((size_t)G * (own / 32 * 6144 + dv / 16 * 3072) + (size_t)shared / 32 * 6144); }
size_t psk_split_attn_scratch(int G, int own, int shared, int dv, int64_t n_front, int64_t n_window) { return sa_images(G, own, shared, dv, (n_front + 31) / 32 + (n_window + 31) / 32); }

template <int KS, int NJ, bool DIST>
static void sa_launch(hipStream_t st, const sa_attn &a, int H) {
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)split_attn_kernel<KS, NJ, DIST>, hipFuncAttributeMaxDynamicSharedMemorySize, sa_lds<KS, NJ>());
    hipLaunchKernelGGL((split_attn_kernel<KS, NJ, DIST>), dim3(H, (a.T + SA_ROWS - 1) / SA_ROWS), dim3(512), (sa_lds<KS, NJ>()), st, a);
}
void psk_split_attn(hipStream_t st, const psk_split_attn_args &x) {
    sa_keys k{};
    k.k = {x.k, x.ldk, x.mod, x.off};
    k.v = {x.v, x.ldk, x.mod, x.off};
    k.shared = {x.shared, x.ld_shared, x.shared_mod, x.shared_off};
    k.k_step = x.own; k.v_step = 128;
    k.front_k = x.front_k; k.front_v = x.front_v; k.front_ld = x.ldk;
    k.n_front = x.n_front; k.n_window = x.n_window; k.nbf = (x.n_front + 31) / 32; k.nb = k.nbf + (x.n_window + 31) / 32;
    k.ks_own = x.own / 32; k.ks_shared = x.n_shared / 32; k.nj = 8; k.G = x.G;
    k.img = (char *)x.scratch;
    k.img_shared = k.img + (size_t)x.G * k.nb * (k.ks_own * 6144 + k.nj * 3072);
    hipLaunchKernelGGL(split_keys_kernel, dim3(k.nb, x.G + (x.n_shared > 0)), dim3(256), 0, st, k);
    sa_attn a{k.img, k.img_shared, k.nbf, k.nb, k.ks_own, x.H / x.G, (int)x.pos0, (int)x.first, x.T, x.window, x.pool, x.keep, x.q, x.ldq, x.own + x.n_shared, x.own, x.rot_dims, x.pairing, x.freq,
              x.rot_mag, x.scale, x.softcap, x.temp, x.slope, x.sink, x.gate, x.ldg, x.gate_elem, x.o, x.ldo};
    if (x.own + x.n_shared == 192) x.slope ? sa_launch<6, 8, true>(st, a, x.H) : sa_launch<6, 8, false>(st, a, x.H);
    else x.slope ? sa_launch<4, 8, true>(st, a, x.H) : sa_launch<4, 8, false>(st, a, x.H);
}
