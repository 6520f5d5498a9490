// Soft-max attention of a portion's many rows with fp32 operands on the bf16 matrix instruction (v_mfma_f32_16x16x32_bf16): every operand is the sum of three bf16 numbers -- rounded, the
// rounded rest, the rest of that, 24 bits together -- and a product the six of the nine partial products that are not below 2^-24 of it, accumulated in fp32 (the leading ones and the others
// apart).  Each of those is exact, and a sum of 192 passes 36 roundings where v_mfma_f32_16x16x4_f32 has one for each of its 48 steps; six of the fast instructions cost 96 clocks where the
// fp32 one's eight steps cost 256.  The serving layers' forms (k_latent.hip, k_winattn.hip: portions of any size, and what this does not take) run on the fp32 instruction.
//   split_keys_kernel   the keys and values a portion sees, in blocks of 32 and split, as the images the attention's stages are filled with: 1 KB per instruction operand in lane order
//   split_attn_kernel   128 rows (consecutive tokens) of one head per work-group, a wave 16 of them against all keys, or a part of them; blocks of 32 keys through two LDS stages
//   split_join_kernel   the parts of such rows together (sa_plan_of)
// S^T = K Q^T, so that a lane has one row: maximum and sum run over its own registers, two lane moves join the four lanes of a row.  D's rows are the keys 4 (l / 16) + i of two tiles, and the
// second product, O^T = V^T P^T, takes its 32 keys in any order that both operands share: a lane's eight weights are its piece of the operand as they are, and the value images are laid out so.
// What bounded the fp32 form: 2560 clocks of matrix instructions per 16 x 16 scores beside as much again of soft-max in its accumulator layout (four moves per row reduction, weights turned
// in LDS), keys straight from the L2s for 32 rows at a time.  2047 tokens of 16 heads, keys of 192, a window of 1024: 318 -> 141 us, 17 of them the images; 3 us a block of 32 keys and
// work-group, 1.9 of it matrix instructions; without its reads, its requests or its soft-max it is 0.7, 0.3 and 0.5 less.  (The queries are turned by split_keys_kernel and come straight into the operand registers: through LDS, turned by every head's work-groups,
// a work-group's first product stood 9 us behind its start.)  (The second wave of every SIMD a block behind with its second product, so
// that its soft-max runs beside the others' products: 137 us without the images against 126.)  Error against 64 bits over four seeds: keys of 192 5.6e-7 -> 5.4e-7, 128 with slopes 6.4e-7 -> 4.1e-7.
#include "ps_seq.h"

#include <algorithm>
#include <cmath>
#include <vector>

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
// 16 bytes, then [16 value columns][plane][lane].  The last of blockIdx.y: the key parts that all heads share, an image of their own; the first
// `turners`: the turned part of the queries of rows 32 b .. (behind the images they were the launch's tail: 28 us for 2047 tokens of 16 heads, 21 without them)
#define SA_TURNERS 8 // work-groups that share the heads of 32 rows
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
    const float *q, *freq; // the queries, whose part of the shared numbers is turned (rot_dims > 0; a group is a head): q_turned [T][G][32 ks_shared]
    long long ldq;
    float rot_mag, *q_turned;
    int rot_dims, pairing, pos0, T, turners;
};
static __device__ __forceinline__ const float *sa_row(const sa_rows &r, long long step, int j) {
    int n = j + r.off;
    if (r.mod > 0 && n >= r.mod) n -= r.mod;
    return r.base + step + n * r.ld;
}
__global__ __launch_bounds__(256) void split_keys_kernel(sa_keys a) {
    const int b = blockIdx.x, g = (int)blockIdx.y - a.turners, tid = threadIdx.x;
    if (g < 0) {
        const int dr = 32 * a.ks_shared, half = a.rot_dims / 2;
        for (int x = tid; x < 32 * (dr - half); x += 256) {
            const int t = 32 * b + x / (dr - half), i = x % (dr - half); // pair i, or a number that is not turned
            if (t >= a.T) break;
            const bool pair = i < half, near = a.pairing == PS_ROT_NEIGHBOURS;
            const int c = !pair ? half + i : near ? 2 * i : i, d = near ? 1 : half;
            const float ang = pair ? (float)(a.pos0 + t) * a.freq[i] : 0.f, cs = cosf(ang) * a.rot_mag, sn = sinf(ang) * a.rot_mag;
            const long long own = 32 * a.ks_own + dr;
            const float *q = a.q + t * a.ldq + 32 * a.ks_own + c;
            float *o = a.q_turned + (long long)t * a.G * dr + c;
#pragma unroll 4
            for (int h = g + a.turners; h < a.G; h += a.turners) {
                const float u = q[h * own], v = q[h * own + (pair ? d : 0)];
                o[h * dr] = pair ? u * cs - v * sn : u;
                if (pair) o[h * dr + d] = v * cs + u * sn;
            }
        }
        return;
    }
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
    const float *q_turned; // [T][H][numbers of the shared key part], or NULL: those of q as they are
    float scale, softcap;
    const float *temp, *slope, *sink, *gate;
    long long ldg;
    int gate_elem;
    float *o;
    long long ldo;
    int q16;               // rows of q by sixteen bytes
    int H, most;           // blocks of a part at most: a tile with more of them is worked on by several work-groups, whose results split_join_kernel adds
    float *part, *part_ml; // [work-groups] results of 128 rows not yet divided, their maxima and sums
};
// the blocks of keys of the 128 rows from t0 on: those of the front store that the last row sees, then the window's from the first row's first key to the last row's own
struct sa_span { int nfb, wb0, blocks; };
static __host__ __device__ __forceinline__ int sa_parts(int blocks, int most) { return (blocks + most - 1) / most; }
static __host__ __device__ __forceinline__ sa_span sa_span_of(int t0, int pos0, int first, int T, int window, int pool, int keep) {
    const int plast = pos0 + (t0 + 128 < T ? t0 + 128 : T) - 1, pfirst = pos0 + t0, lo = pfirst - window + 1;
    int nf = plast - window + 1;
    nf = nf <= 0 ? 0 : pool > 0 ? nf / pool : nf < keep ? nf : keep;
    const int nfb = (nf + 31) / 32, wb0 = ((lo > 0 ? lo : 0) - first) / 32;
    return sa_span{nfb, wb0, nfb + (plast - first) / 32 - wb0 + 1};
}
static __device__ __forceinline__ void sa_dma(const char *base, unsigned off, unsigned lds_dst) { // one wave-instruction: lane l's 16 bytes at base + off go to lds_dst + 16 l
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0" : "=&s"(keep) : "v"(off), "s"(base), "s"(lds_dst) : "memory");
}
// a row's results from its maximum, the sum of its weights and their products (a lane: columns 16 j + 4 lq ..)
template <int NJ>
static __device__ __forceinline__ void sa_finish(const sa_attn &a, int h, int t, int lq, float m, float l, const sa_f4 (&acc)[NJ]) {
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
#define SA_ROWS 128
#define SA_CUS 256
#define SA_PART (SA_ROWS * (128 + 2) * 4) // bytes of a part of a tile
template <int KS, int NJ>
static constexpr int sa_lds() { return 2 * (KS * 6144 + NJ * 3072); } // two stages
template <int KS, int NJ, bool DIST>
__global__ __launch_bounds__(512) void split_attn_kernel(sa_attn a) {
    extern __shared__ __attribute__((aligned(16))) char sa_smem[];
    constexpr int STAGE = KS * 6144 + NJ * 3072, PIECES = KS * 6 + NJ * 3;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lq = lane >> 4;
    const unsigned lds0 = (unsigned)(size_t)(const __attribute__((address_space(3))) char *)sa_smem;
    // a part of a tile's blocks (the rows with the most keys first)
    const int h = (int)blockIdx.x % a.H, slot = (int)blockIdx.x;
    int t0 = (a.T - 1) / SA_ROWS * SA_ROWS, part = slot / a.H, parts;
    sa_span span;
    for (;; t0 -= SA_ROWS) { // (uniform; there are as many work-groups as parts)
        span = sa_span_of(t0, a.pos0, a.first, a.T, a.window, a.pool, a.keep);
        parts = sa_parts(span.blocks, a.most);
        if (part < parts || t0 == 0) break;
        part -= parts;
    }
    const int nfb = span.nfb, wb0 = span.wb0, it0 = span.blocks * part / parts, it1 = span.blocks * (part + 1) / parts, g = h / a.hpg;
    const int rows = min(SA_ROWS, a.T - t0), n = 16 * wave + lr, p = a.pos0 + t0 + n, pfirst = a.pos0 + t0; // this lane's row and its position
    const int own = a.ks_own * 6, image = own + NJ * 3; // pieces of a head's own key part, of its image
    auto block_of = [&](const int it) { return it < nfb ? it : a.nbf + wb0 + it - nfb; };
    auto request = [&](const int it) {
        const int b = block_of(it);
        const char *im = a.img + ((size_t)g * a.nb + b) * (image * 1024), *sh = a.img_shared + (size_t)b * ((KS * 6 - own) * 1024);
#pragma unroll
        for (int x = 0; x < (PIECES + 7) / 8; x++) {
            const int pc = x * 8 + wave;
            if (pc < PIECES) sa_dma(pc < own ? im + pc * 1024 : pc < KS * 6 ? sh + (pc - own) * 1024 : im + (pc - KS * 6 + own) * 1024, lane * 16, lds0 + (unsigned)(((it - it0) & 1) * STAGE + pc * 1024));
        }
    };
    request(it0);
    // this lane's share of its query row (rows that do not exist repeat the last one)
    sa_u4 q[KS][3];
    {
        const int t = min(t0 + n, a.T - 1);
        const float *qr = a.q + (long long)t * a.ldq + (long long)h * (32 * KS) + 8 * lq, *qt = a.q_turned ? a.q_turned + ((long long)t * a.H + h) * (32 * (KS - a.ks_own)) + 8 * lq - 32 * a.ks_own : qr;
        float v[KS][8];
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const float *x = (s < a.ks_own ? qr : qt) + 32 * s;
            if (a.q16) { // (uniform)
                *(sa_f4 *)v[s] = *(const sa_f4 *)x;
                *(sa_f4 *)(v[s] + 4) = *(const sa_f4 *)(x + 4);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) v[s][e] = x[e];
            }
        }
#pragma unroll
        for (int s = 0; s < KS; s++) sa_split8<true>(v[s], q[s]);
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
    for (int it = it0; it < it1; it++) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); // the block has landed (this wave's share); the reads of the one before are back
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (it + 1 < it1) request(it + 1);
        const place b = place_of(it);
        if (!alive || b.none) continue;
        const char *st = sa_smem + ((it - it0) & 1) * STAGE + lane * 16;
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
        for (int it = it0; it < it1; it++) {
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
    if (parts == 1) {
        if (n < rows) sa_finish<NJ>(a, h, t0 + n, lq, m, l, acc);
        return;
    }
    // as they are, for split_join_kernel
    float *o = a.part + (size_t)slot * (SA_ROWS * 16 * NJ) + (wave * NJ * 64 + lane) * 4;
#pragma unroll
    for (int j = 0; j < NJ; j++) *(sa_f4 *)(o + j * 256) = acc[j];
    if (lq == 0) *(sa_f2 *)(a.part_ml + (size_t)slot * (2 * SA_ROWS) + 2 * n) = sa_f2{m, l};
}
// The parts of a tile, brought to their common maximum, added in order and finished: a wave has sixteen rows of it.
template <int NJ>
__global__ __launch_bounds__(256) void split_join_kernel(sa_attn a) {
    const int lane = threadIdx.x & 63, wave = 4 * (int)blockIdx.y + (int)(threadIdx.x >> 6), lr = lane & 15, lq = lane >> 4, h = (int)blockIdx.x % a.H, n = 16 * wave + lr;
    int t0 = (a.T - 1) / SA_ROWS * SA_ROWS, tile = (int)blockIdx.x / a.H, first = 0, parts; // (tiles in the same order)
    for (;; t0 -= SA_ROWS, tile--) {
        parts = sa_parts(sa_span_of(t0, a.pos0, a.first, a.T, a.window, a.pool, a.keep).blocks, a.most);
        if (tile == 0 || t0 == 0) break;
        first += parts;
    }
    if (parts == 1 || t0 + 16 * wave >= a.T) return;
    auto slot = [&](const int x) { return (size_t)((first + x) * a.H + h); };
    float m = -INFINITY;
    for (int x = 0; x < parts; x++) m = fmaxf(m, a.part_ml[slot(x) * (2 * SA_ROWS) + 2 * n]);
    float l = 0.f;
    sa_f4 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[j] = sa_f4{0.f, 0.f, 0.f, 0.f};
    for (int x = 0; x < parts; x++) {
        const sa_f2 ml = *(const sa_f2 *)(a.part_ml + slot(x) * (2 * SA_ROWS) + 2 * n);
        const float *o = a.part + slot(x) * (SA_ROWS * 16 * NJ) + (wave * NJ * 64 + lane) * 4;
        if (ml[0] == -INFINITY && ml[1] == 0.f) continue; // (the row sees no key of this part)
        const float f = ml[0] == m ? 1.f : sa_exp(ml[0] - m);
        l += ml[1] * f;
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[j] += *(const sa_f4 *)(o + j * 256) * f;
    }
    if (t0 + n < a.T) sa_finish<NJ>(a, h, t0 + n, lq, m, l, acc);
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
static size_t sa_images(int G, int own, int shared, int dv, int64_t blocks) { return (size_t)blocks * ((size_t)G * (own / 32 * 6144 + dv / 16 * 3072) + (size_t)shared / 32 * 6144 + (size_t)G * shared * 128); }
size_t psk_split_attn_scratch(int G, int own, int shared, int dv, int64_t n_front, int64_t n_window) { return sa_images(G, own, shared, dv, (n_front + 31) / 32 + (n_window + 31) / 32); }

struct sa_plan { int most, wgs; bool join; };
// How many blocks a work-group has at most.  The rows of a tile have up to a window of keys, and where the tiles are fewer than the CUs, or some have many more keys than others, the chip waits for the
// longest: 1500 tokens of 16 heads behind a window of 1024 are 192 tiles of 4 to 36 blocks.  A tile in parts costs each of them a start (the queries, the first block: as much as four blocks) and a launch that
// joins them.  So the host follows the CUs through the work-groups, in the order they are dispatched, for whole tiles and for parts of at most 15 / 16, 14 / 16, .. of the longest, and takes the shortest time; whole
// tiles where that is within 6 % (a tile more of one to its time is what the model is off by).  us, whole and so, with the joining: those 1500 tokens, keys of 192 136 and 92, keys of 128 with slopes and means of
// blocks in front (up to 47 blocks) 104 and 82.
static sa_plan sa_plan_of(const sa_attn &a, size_t part_bytes) {
    const int tiles = (a.T + SA_ROWS - 1) / SA_ROWS;
    const sa_plan whole{1 << 30, tiles * a.H, false};
    if (tiles > 64 || tiles * a.H > 4 * SA_CUS) return whole;
    int blocks[64], longest = 0;
    for (int i = 0; i < tiles; i++) longest = std::max(longest, blocks[i] = sa_span_of(SA_ROWS * (tiles - 1 - i), a.pos0, a.first, a.T, a.window, a.pool, a.keep).blocks);
    constexpr int START = 4;
    std::vector<int> idle;
    auto end_of = [&](const sa_plan &p) { // in blocks
        idle.assign((size_t)(p.wgs / SA_CUS + 2) * (std::min(longest, p.most) + START) + 1, 0); // CUs that become idle at a time
        idle[0] = SA_CUS;
        int now = 0, end = 0;
        for (int i = 0; i < tiles; i++) {
            const int parts = sa_parts(blocks[i], p.most);
            for (int x = 0; x < parts; x++) {
                const int time = blocks[i] * (x + 1) / parts - blocks[i] * x / parts + START;
                for (int n = a.H; n > 0;) {
                    while (!idle[now]) now++;
                    const int k = std::min(n, idle[now]);
                    idle[now] -= k;
                    idle[now + time] += k;
                    end = std::max(end, now + time);
                    n -= k;
                }
            }
        }
        return end;
    };
    sa_plan best = whole;
    double least = 0.94 * end_of(whole);
    for (int s = 15; s >= 2; s--) {
        sa_plan p{(longest * s + 15) / 16, 0, true};
        if (p.most < 4) break;
        for (int i = 0; i < tiles; i++) p.wgs += sa_parts(blocks[i], p.most) * a.H;
        if ((size_t)p.wgs * SA_PART > part_bytes) break;
        const double t = end_of(p) + 1.3 + 0.0044 * p.wgs;
        if (t < least) { least = t; best = p; }
    }
    return best;
}
template <int KS, int NJ, bool DIST>
static void sa_launch(hipStream_t st, const sa_attn &a, const sa_plan &p, int H) {
    static unsigned long long mask = 0;
    if (ps_first_on_device(&mask)) (void)hipFuncSetAttribute((const void *)split_attn_kernel<KS, NJ, DIST>, hipFuncAttributeMaxDynamicSharedMemorySize, sa_lds<KS, NJ>());
    hipLaunchKernelGGL((split_attn_kernel<KS, NJ, DIST>), dim3(p.wgs), dim3(512), (sa_lds<KS, NJ>()), st, a);
    if (p.join) hipLaunchKernelGGL((split_join_kernel<NJ>), dim3(H * ((a.T + SA_ROWS - 1) / SA_ROWS), 2), dim3(256), 0, st, a);
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
    k.q = x.q; k.ldq = x.ldq; k.freq = x.freq; k.rot_mag = x.rot_mag; k.rot_dims = x.rot_dims; k.pairing = x.pairing; k.pos0 = (int)x.pos0; k.T = x.T; k.turners = x.rot_dims > 0 ? SA_TURNERS : 0;
    k.q_turned = x.rot_dims > 0 ? (float *)(k.img_shared + (size_t)k.nb * k.ks_shared * 6144) : nullptr;
    hipLaunchKernelGGL(split_keys_kernel, dim3(k.nb, k.turners + x.G + (x.n_shared > 0)), dim3(256), 0, st, k);
    sa_attn a{k.img, k.img_shared, k.nbf, k.nb, k.ks_own, x.H / x.G, (int)x.pos0, (int)x.first, x.T, x.window, x.pool, x.keep, x.q, x.ldq, k.q_turned, x.scale, x.softcap,
               x.temp, x.slope, x.sink, x.gate, x.ldg, x.gate_elem, x.o, x.ldo, x.ldq % 4 == 0 && ((uintptr_t)x.q & 15) == 0, x.H};
    const sa_plan p = sa_plan_of(a, x.part_bytes);
    a.most = p.most;
    a.part = x.part;
    a.part_ml = x.part + (size_t)p.wgs * (SA_ROWS * 128);
    if (x.own + x.n_shared == 192) x.slope ? sa_launch<6, 8, true>(st, a, p, x.H) : sa_launch<6, 8, false>(st, a, p, x.H);
    else x.slope ? sa_launch<4, 8, true>(st, a, p, x.H) : sa_launch<4, 8, false>(st, a, p, x.H);
}
