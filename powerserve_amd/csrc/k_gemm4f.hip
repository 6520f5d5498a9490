// Q4_K batched mat-mul of many columns on v_mfma_f32_16x16x32_f16, bit-exact with ggml_vec_dot_q4_K_q8_K (ggml-quants.c:7809-7873; the arithmetic, the operand layout and the
// prepared activations are those of k_gemm4k.hip's header).
//
// What bounds it: the issue of a SIMD.  Per super-block, 16 rows and 16 columns the reference's order costs 8 products (16.5 cycles each), one for the mins (32.6: K = 4, four
// independent sums, the mins lanes' shape) and 48 fp32 fmas of 2.4; beside them stand 8 scalings, and the 16 rows' weights as fp16 operands (411 cycles, once per wave and
// super-block).  Matrix and vector instructions hardly overlap here (measured, two and four waves per SIMD: their times add up but for a tenth), LDS reads cost next to nothing
// beside them (256 bytes a cycle and CU).  So:
//   * a wave owns 16 rows and CT column tiles WHOLE -- all eight accumulator lanes and the four mins lanes, 48 CT chains per lane.  Its weights become operands in its own
//     registers (nine instructions per accumulator lane) and meet CT column tiles; no wave waits for another's, and the sums over the lanes at the end are in-lane;
//   * eight waves share the columns: 128 rows x 16 CT columns per work-group, one work-group per CU, persistent.  Activations, weights, headers and column metadata come by
//     global_load_lds_dwordx4 into a ring of three stages of one super-block.  One barrier a quarter into a stage says both that the next stage is there and that the one
//     before has been left, so that its place is asked for at once -- piece by piece: asked for in one go, the wave stands still while the memory pipe takes them (a stage of
//     CT = 3 on an eighth of the chip: 1.60 us, 1.44 with a piece every other step; the barrier in the middle of the stage leaves the last pieces too little time: 3 % more);
//   * the operands of the activations are read NY steps ahead, across the stages; the next stage's scales and metadata at the end of this one (there 1.60 us against 2.0 read when
//     needed).  CT = 4 would need 30 registers more than two waves per SIMD have.
// Measured (with the activations' quantizer in front, k_gemm4k.hip's wide kernel -> this): 4096 x 28672, 512 columns 360 -> 247 us, 203 columns 180 -> 125, 32 columns 57 -> 27;
// 14336 x 4096, 512 columns 190 -> 150; 4096 x 6144 95 -> 70; 4096 x 4096 68 -> 51.  A stage on a full chip takes 1.26 us with two column tiles and 1.63 with three in a single
// round of work-groups, 1.17 and 1.37 over several.
#include "ps_gemv_dev.h"

namespace {

typedef _Float16 g4f_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 g4f_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 g4f_h2 __attribute__((ext_vector_type(2)));
typedef float g4f_f4 __attribute__((ext_vector_type(4)));
typedef float g4f_f16 __attribute__((ext_vector_type(16)));

struct G4FMat {
    const uint8_t *qs, *aux;
    float *out;
    const float *bias;
    int64_t ldo;
    int n_tiles;
};
struct G4FParams {
    G4FMat w[3];
    int n_w, nsb, bs, n_tiles, n_rb, n_cb, n_items; // items = (block of NRW row tiles, block of CT column tiles)
    const float *residual;
    const char *qf;
    const uint8_t *mf;
};

constexpr int G4F_NRW = 8, G4F_NST = 3;
// One LDS stage = one super-block: the activations as ps_act::qf holds them [column tile][u][lane] 16 B; the weights [wave][u][row] 16 B; and per wave its rows' headers
// [row] 16 B with, behind those of wave ct, column tile ct's metadata as ps_act::mf holds it (one request brings both).
constexpr int g4f_w0(const int ct) { return ct * 8192; }
constexpr int g4f_h0(const int ct) { return g4f_w0(ct) + G4F_NRW * 2048; }
constexpr int g4f_hm(const int ct, const int w) { return g4f_h0(ct) + w * 256 + (w < ct ? w : ct) * 576; } // headers of wave w; + 256: the metadata of column tile w
constexpr int g4f_stage(const int ct) { return g4f_hm(ct, G4F_NRW); }
constexpr int g4f_lds(const int ct) { return G4F_NST * g4f_stage(ct) + PS_EXP2F_N * 8; }

__device__ __forceinline__ void g4f_dma(const char *base, const uint32_t off, const unsigned lds_dst) { // lane l's 16 bytes at base + off go to lds_dst + 16 l
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_dst) : "memory", "m0");
}
__device__ __forceinline__ void g4f_dma64(const uint8_t *src, const unsigned lds_dst) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_dst) : "memory", "m0");
}
// y * (a half of h), rounded once: the product plus +0, which only turns a product of -0 into +0 -- and the chains, which start at +0, cannot tell
__device__ __forceinline__ float g4f_scale_lo(const uint32_t h, const float y) {
    float d;
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(y));
    return d;
}
__device__ __forceinline__ float g4f_nscale_hi(const uint32_t h, const float y) {
    float d;
    asm("v_fma_mix_f32 %0, %1, -%2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(h), "v"(y));
    return d;
}
__device__ __forceinline__ g4f_h2 g4f_h2of(const uint32_t v) {
    g4f_h2 r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}
__device__ __forceinline__ uint32_t g4f_u32of(const g4f_h2 v) {
    uint32_t r;
    __builtin_memcpy(&r, &v, 4);
    return r;
}

struct G4FItem { int rb, cb; };
// item -> (row block, column block): panels of four column blocks, so that consecutive items share weights four ways and activations eight
__device__ __forceinline__ G4FItem g4f_item(const G4FParams &p, const int i) {
    const int panel = i / (p.n_rb * 4), width = min(4, p.n_cb - panel * 4), j = i - panel * p.n_rb * 4;
    return G4FItem{j / width, panel * 4 + j % width};
}

template <int EPI, int CT>
__global__ __launch_bounds__(G4F_NRW * 64, G4F_NRW / 4) void gemm4f_kernel(const G4FParams p) {
    constexpr int STAGE = g4f_stage(CT), W0 = g4f_w0(CT);
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int m = lane & 15, kb = lane >> 4, nsb = p.nsb;
    const uint64_t *const tab = (const uint64_t *)(lds + G4F_NST * STAGE);
    if (EPI == 1 && threadIdx.x < PS_EXP2F_N) ((uint64_t *)(lds + G4F_NST * STAGE))[threadIdx.x] = ps_exp2f_tab[threadIdx.x];
    // blocks b, b + 8, .. run on one XCD: they take neighbouring items
    const int per = (int)gridDim.x >> 3, first = (gridDim.x & 7) ? (int)blockIdx.x : (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    const int wave_hm = g4f_h0(CT) + wave * 256 + min(wave, CT) * 576;
    const unsigned lds0 = (unsigned)(size_t)(const __attribute__((address_space(3))) char *)lds;

    // ---- the requests: a stage of the stream (items of this work-group one behind the other)
    int r_item = first, r_sb = 0;
    const uint8_t *r_w = nullptr;                     // per lane: this wave's rows
    constexpr int NB = (8 * CT + G4F_NRW - 1) / G4F_NRW;
    uint32_t r_b[NB] = {};                            // its share of the activations: pieces (column tile, u) = wave + NRW i
    const uint8_t *r_hm = nullptr;                    // per lane: headers (lanes 0..15), metadata (lanes 16..51 of waves below CT)
        const int n_hm = wave < CT ? 52 : 16;
    const uint32_t hm_step = lane < 16 ? 128u : 576u;
    auto tile_of = [&](const int rb, int &wi) { // this wave's row tile (clamped: a wave without rows works on the last ones and stores nothing)
        wi = 0;
        if (EPI == 1) { wi = wave >= G4F_NRW / 2; return min(rb * (G4F_NRW / 2) + wave % (G4F_NRW / 2), p.w[0].n_tiles - 1); }
        int t = min(rb * G4F_NRW + wave, p.n_tiles - 1);
        if (p.n_w > 1 && t >= p.w[0].n_tiles) { t -= p.w[0].n_tiles; wi = 1; }
        if (p.n_w > 2 && wi == 1 && t >= p.w[1].n_tiles) { t -= p.w[1].n_tiles; wi = 2; }
        return t;
    };
    auto point = [&](const int item) {
        const G4FItem I = g4f_item(p, item);
        int wi;
        const int t = tile_of(I.rb, wi);
        const G4FMat &W = wi == 0 ? p.w[0] : wi == 1 ? p.w[1] : p.w[2];
        const int last = (p.bs - 1) / 16;
        r_w = W.qs + ((size_t)(2 * t + (m >> 3)) * nsb << 10) + (m & 7) * 128 + kb * 16;
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int q = min(wave + G4F_NRW * i, 8 * CT - 1);
            r_b[i] = (uint32_t)((min(I.cb * CT + (q >> 3), last) * nsb << 13) + (q & 7) * 1024 + lane * 16);
        }
        r_hm = lane < 16 ? W.aux + ((size_t)(2 * t + (m >> 3)) * nsb) * 128 + (m & 7) * 16
                         : p.mf + (size_t)min(I.cb * CT + min(wave, CT - 1), last) * nsb * 576 + (lane - 16) * 16;
    };
    constexpr int NP = NB + 3; // pieces of a stage per wave
    static_assert(2 * CT + 2 * NP <= 8 * CT, "asked for within the stage");
    auto request_piece = [&](const unsigned st, const int i) {
        if (i < 2) g4f_dma64(r_w + 64 * i, st + (unsigned)(W0 + wave * 2048 + i * 1024));
        else if (i == 2) { if (lane < n_hm) g4f_dma64(r_hm, st + (unsigned)wave_hm); }
        else if (8 * CT % G4F_NRW == 0 || wave + G4F_NRW * (i - 3) < 8 * CT) g4f_dma(p.qf, r_b[i - 3], st + (unsigned)((wave + G4F_NRW * (i - 3)) * 1024));
    };
    auto advance = [&]() { // to the stream's next stage; past the last item's end: its last stage again, never used
        if (++r_sb < nsb) {
            r_w += 1024;
            r_hm += hm_step;
#pragma unroll
            for (int i = 0; i < NB; i++) r_b[i] += 8192;
        } else if (r_item + (int)gridDim.x < p.n_items) {
            r_item += (int)gridDim.x;
            r_sb = 0;
            point(r_item);
        } else {
            r_sb = nsb - 1;
        }
    };
    auto request = [&](const int buf) {
#pragma unroll
        for (int i = 0; i < NP; i++) request_piece(lds0 + (unsigned)(buf * STAGE), i);
        advance();
    };
    point(first);
    request(0);
    request(1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    uint32_t e64 = 0x64006400u, e54 = 0x54005400u;
    asm("" : "+v"(e64), "+v"(e54));
    const g4f_h2 k1024 = {(_Float16)1024.f, (_Float16)1024.f}, km1024 = {(_Float16)-1024.f, (_Float16)-1024.f}, km64 = {(_Float16)-64.f, (_Float16)-64.f};
    const bool hi_half = kb >= 2;
    const uint32_t sel0 = 0x04000400u | (uint32_t)((kb & 1) * 2) * 0x00010001u, sel1 = sel0 + 0x00010001u; // byte pairs (v, 0x64) of this k-group's two sub-blocks

    constexpr int NY = CT == 2 ? 8 : 4; // operands of the activations on their way from LDS (8 CT % NY == 0)
    int buf = 0;
    const char *st = lds;
    // what a stage needs at its start is read at the end of the one before
    ps_u32x4 y[NY], h;
    uint32_t w[2], dd[4];
    float yd[CT];
    uint2 b2[CT];
    auto read_y = [&](const char *sp, const int s) { y[s % NY] = *(const ps_u32x4 *)(sp + lane * 16 + (s % CT) * 8192 + s / CT * 1024); };
    auto read_w = [&](const char *sp, const int u) { w[u & 1] = *(const uint32_t *)(sp + W0 + wave * 2048 + m * 16 + kb * 4 + u * 256); };
    auto read_head = [&](const char *sp) {
        h = *(const ps_u32x4 *)(sp + wave_hm + m * 16);
#pragma unroll
        for (int r = 0; r < 4; r++) dd[r] = *(const uint32_t *)(sp + wave_hm + (4 * kb + r) * 16); // (d, dmin) of the result rows
    };
    auto read_meta = [&](const char *sp, const int ct) {
        yd[ct] = *(const float *)(sp + g4f_hm(CT, ct) + 256 + m * 4);
        b2[ct] = *(const uint2 *)(sp + g4f_hm(CT, ct) + 256 + 64 + m * 32 + kb * 8);
    };
    read_head(st);
#pragma unroll
    for (int ct = 0; ct < CT; ct++) read_meta(st, ct);
    read_w(st, 0);
    read_w(st, 1);
#pragma unroll
    for (int s = 0; s < NY; s++) read_y(st, s);

    for (int item = first; item < p.n_items; item += (int)gridDim.x) {
        g4f_f4 acc[CT][8] = {}, accm[CT][4] = {}; // [column tile][accumulator lane][row 4 kb + r]
#pragma unroll 1
        for (int sb = 0; sb < nsb; sb++) {
            const int nbuf = buf == 2 ? 0 : buf + 1;
            const char *const ns = lds + nbuf * STAGE;
            const unsigned r_st = lds0 + (unsigned)((buf == 0 ? 2 : buf - 1) * STAGE);
            // the operand row's scales and mins (get_scale_min_k4) of sub-blocks 2 kb, 2 kb + 1
            const uint32_t scb = hi_half ? ((h.w & 0x0f0f0f0fu) | (((h.y >> 6) & 0x03030303u) << 4)) : (h.y & 0x3f3f3f3fu);
            const uint32_t mnb = hi_half ? (((h.w >> 4) & 0x0f0f0f0fu) | (((h.z >> 6) & 0x03030303u) << 4)) : (h.z & 0x3f3f3f3fu);
            const g4f_h2 s0 = g4f_h2of(__builtin_amdgcn_perm(0x64646464u, scb, sel0)) - k1024, s1 = g4f_h2of(__builtin_amdgcn_perm(0x64646464u, scb, sel1)) - k1024; // exact
            const g4f_h2 n0 = s0 * km1024, n1 = s1 * km64;
            const g4f_h2 m0 = g4f_h2of(__builtin_amdgcn_perm(0x64646464u, mnb, sel0)) - k1024, m1 = g4f_h2of(__builtin_amdgcn_perm(0x64646464u, mnb, sel1)) - k1024;
            const g4f_h4 am = {m0[0], m0[1], m1[0], m1[1]};
            auto operand = [&](const uint32_t q) { // nibbles as fp16 1024 + n and, from the upper ones in place, 64 + n;  fma(1024 + n, s, -1024 s) = n s, exact
                const uint32_t q8 = q >> 8;
                const uint32_t t[4] = {(q & 0x000F000Fu) | e64, (q8 & 0x000F000Fu) | e64, (q & 0x00F000F0u) | e54, (q8 & 0x00F000F0u) | e54};
                uint32_t o[4];
#pragma unroll
                for (int k = 0; k < 4; k++) o[k] = g4f_u32of(__builtin_elementwise_fma(g4f_h2of(t[k]), k < 2 ? s0 : s1, k < 2 ? n0 : n1));
                g4f_h8 r;
                __builtin_memcpy(&r, o, 16);
                return r;
            };
            g4f_h8 a = operand(w[0]);
            read_w(st, 2);
            float dr[CT][4];
            g4f_f4 D = {};
            g4f_f16 E = {};
#pragma unroll
            for (int s = 0; s < 8 * CT; s++) { // (accumulator lane, column tile) s: its product is issued, that of the step before meets its multipliers meanwhile
                const int u = s / CT, ct = s % CT, pu = s ? (s - 1) / CT : 0, pc = s ? (s - 1) % CT : 0;
                g4f_h8 bv;
                __builtin_memcpy(&bv, &y[s % NY], 16);
                const g4f_f4 zf = {0.f, 0.f, 0.f, 0.f};
                const g4f_f4 P = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bv, zf, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (s + NY < 8 * CT) read_y(st, s + NY);
                else read_y(ns, s + NY - 8 * CT);
                if (ct == CT - 1 && u < 7) {
                    a = operand(w[(u + 1) & 1]);
                    if (u < 5) read_w(st, u + 3);
                    else if (u == 5) read_w(ns, 0);
                    else read_w(ns, 1);
                }
                if (s < CT) {
#pragma unroll
                    for (int r = 0; r < 4; r++) dr[ct][r] = g4f_scale_lo(dd[r], yd[ct]);
                }
                if (s) {
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[pc][pu][r] = __fmaf_rn(dr[pc][r], D[r], acc[pc][pu][r]);
                    asm volatile("" : "+v"(acc[pc][pu])); // (keeps a step's fmas in it: results are not left to wait for theirs in four registers each)
                }
                if (s && s <= CT) { // the mins lanes of column tile s - 1
                    float dm[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) dm[r] = g4f_nscale_hi(dd[r], yd[pc]);
#pragma unroll
                    for (int v = 0; v < 4; v++)
#pragma unroll
                        for (int r = 0; r < 4; r++) accm[pc][v][r] = __fmaf_rn(dm[r], E[4 * v + r], accm[pc][v][r]);
                    asm volatile("" : "+v"(accm[pc][0]), "+v"(accm[pc][1]), "+v"(accm[pc][2]), "+v"(accm[pc][3]));
                }
                if (s < CT) {
                    const g4f_f16 zero = {};
                    g4f_h4 bm;
                    __builtin_memcpy(&bm, &b2[ct], 8);
                    E = __builtin_amdgcn_mfma_f32_16x16x4f16(am, bm, zero, 0, 0, 0);
                }
                D = P;
                __builtin_amdgcn_sched_barrier(0);
                if (s == 2 * CT - 1) { // the next stage is there for all; every wave has left the one before the present one behind, whose place the stage after next takes
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                }
                if (EPI != 1 || sb + 1 < nsb) { // ... which it is asked for piece by piece (all at once, the wave stands still while the memory pipe takes them: 0.28 us of a stage)
                    if (s >= 2 * CT && (s - 2 * CT) % 2 == 0 && (s - 2 * CT) / 2 < NP) request_piece(r_st, (s - 2 * CT) / 2);
                    if (s == 8 * CT - 1) advance();
                }
                if (s == 5 * CT) read_head(ns);
                if (s >= 6 * CT && s < 7 * CT) read_meta(ns, s - 6 * CT);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) acc[CT - 1][7][r] = __fmaf_rn(dr[CT - 1][r], D[r], acc[CT - 1][7][r]);
            buf = nbuf;
            st = ns;
        }
        // ---- hsum_float_8: (u + 4) + u, then u + 2, then u + 1; the mins lanes likewise (v + 2, v + 1)
        const G4FItem I = g4f_item(p, item);
        int wi;
        const int tile = tile_of(I.rb, wi);
        float4 v[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float s[4];
#pragma unroll
                for (int u = 0; u < 4; u++) s[u] = __fadd_rn(acc[ct][u][r], acc[ct][u + 4][r]);
                const float mm = __fadd_rn(__fadd_rn(accm[ct][0][r], accm[ct][2][r]), __fadd_rn(accm[ct][1][r], accm[ct][3][r]));
                o[r] = __fadd_rn(__fadd_rn(__fadd_rn(s[0], s[2]), __fadd_rn(s[1], s[3])), mm);
            }
            v[ct] = make_float4(o[0], o[1], o[2], o[3]);
        }
        if (EPI == 1) { // gate rows (waves 0 - 3) and up rows (4 - 7) meet in the place that the stage after next will take: each half finishes half of the columns
            const int xb = buf == 0 ? 1 : buf == 1 ? 2 : 0; // (buf: the next stage, buf + 1: the one behind it; xb = buf + 1 has not been asked for yet)
            float4 *const x = (float4 *)(lds + xb * STAGE);
            const bool up = wave >= G4F_NRW / 2;
            constexpr int HALF = (CT + 1) / 2;
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
                if (up ? ct < HALF : ct >= HALF) x[((wave % (G4F_NRW / 2)) * CT + ct) * 64 + lane] = v[ct];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            float4 o[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ct++) o[ct] = x[((wave % (G4F_NRW / 2)) * CT + ct) * 64 + lane];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            request(xb);
            if (I.rb * (G4F_NRW / 2) + (wave % (G4F_NRW / 2)) < p.w[0].n_tiles) {
#pragma unroll
                for (int ct = 0; ct < CT; ct++) {
                    const int col = (I.cb * CT + ct) * 16 + m;
                    if ((up ? ct < HALF : ct >= HALF) || col >= p.bs) continue;
                    const float4 g4 = up ? o[ct] : v[ct], u4 = up ? v[ct] : o[ct];
                    const float g[4] = {g4.x, g4.y, g4.z, g4.w}, uu[4] = {u4.x, u4.y, u4.z, u4.w};
                    float q[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) q[r] = __fmul_rn(__fmul_rn(g[r], __fdiv_rn(1.0f, __fadd_rn(1.0f, ps_expf_glibc(-g[r], tab)))), uu[r]); // ps_silu_mul with the table in LDS
                    *(float4 *)(p.w[0].out + (int64_t)col * p.w[0].ldo + tile * 16 + 4 * kb) = make_float4(q[0], q[1], q[2], q[3]);
                }
            }
        } else if (I.rb * G4F_NRW + wave < p.n_tiles) {
            const G4FMat &W = wi == 0 ? p.w[0] : wi == 1 ? p.w[1] : p.w[2];
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const int col = (I.cb * CT + ct) * 16 + m, row = tile * 16 + 4 * kb;
                if (col >= p.bs) continue;
                float4 y = v[ct];
                if (W.bias) {
                    const float4 b = *(const float4 *)(W.bias + row);
                    y = make_float4(__fadd_rn(y.x, b.x), __fadd_rn(y.y, b.y), __fadd_rn(y.z, b.z), __fadd_rn(y.w, b.w));
                }
                if (p.residual && wi == 0) {
                    const float4 b = *(const float4 *)(p.residual + (int64_t)col * W.ldo + row);
                    y = make_float4(__fadd_rn(b.x, y.x), __fadd_rn(b.y, y.y), __fadd_rn(b.z, y.z), __fadd_rn(b.w, y.w));
                }
                *(float4 *)(W.out + (int64_t)col * W.ldo + row) = y;
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (nothing may land in LDS that is no longer this work-group's)
}

int64_t g4f_rounds(const int n_cu, const int64_t row_blocks, const int64_t bs, const int cols) { return (row_blocks * ((bs + cols - 1) / cols) + n_cu - 1) / n_cu; }

template <int EPI, int CT>
int g4f_launch(hipStream_t st, const int n_cu, G4FParams &p) {
    constexpr int LDS = g4f_lds(CT);
    static_assert(LDS <= 160 * 1024, "one work-group per CU");
    static unsigned long long attr = 0;
    if (ps_first_on_device(&attr)) (void)hipFuncSetAttribute((const void *)gemm4f_kernel<EPI, CT>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    p.n_cb = (p.bs + CT * 16 - 1) / (CT * 16);
    p.n_items = p.n_rb * p.n_cb;
    psk_note_kernel("gemm4f_kernel<%d, %d>", EPI, CT);
    hipLaunchKernelGGL((gemm4f_kernel<EPI, CT>), dim3((unsigned)(p.n_items < n_cu ? p.n_items : n_cu)), dim3(G4F_NRW * 64), LDS, st, p);
    return 0;
}

} // namespace

int psk_gemm4f(hipStream_t st, int n_cu, const psk_gemv_args &a, ps_act act, int64_t K, int64_t bs) {
    if (a.pro || a.rope || !act.qf || K % 1024 || bs <= 16 || a.n_w < 1 || a.n_w > 3 || (bs + 15) / 16 * K * 32 >= (int64_t)1 << 31) return -1; // (psk_quantize_act writes act.qf for rows of K % 1024 == 0)
    G4FParams p{};
    p.n_w = a.n_w; p.nsb = (int)(K / 256); p.bs = (int)bs; p.residual = a.residual; p.qf = (const char *)act.qf; p.mf = act.mf;
    auto odd16 = [](const void *q) { return ((uintptr_t)q & 15) != 0; };
    int64_t tiles = 0;
    for (int i = 0; i < a.n_w; i++) {
        if (a.w[i]->dtype != PS_Q4_K || a.w[i]->K != K || a.w[i]->N % 16 || a.ldo[i] % 4 || odd16(a.out[i]) || odd16(a.bias[i])) return -1;
        p.w[i] = G4FMat{a.w[i]->qs, a.w[i]->aux, a.out[i], a.bias[i], a.ldo[i], (int)(a.w[i]->N / 16)};
        tiles += a.w[i]->N / 16;
    }
    if (odd16(a.residual) || tiles >= 1 << 24) return -1;
    if (a.silu_pair && (a.n_w != 2 || a.w[0]->N != a.w[1]->N || a.bias[0] || a.bias[1] || a.residual)) return -1;
    const int64_t pairs = a.silu_pair ? tiles / 2 : tiles;
    p.n_tiles = (int)tiles;
    p.n_rb = (int)(a.silu_pair ? (pairs + G4F_NRW / 2 - 1) / (G4F_NRW / 2) : (tiles + G4F_NRW - 1) / G4F_NRW);
    // By the time of a super-block step times the rounds of work-groups: 1.30 us with two column tiles per wave, 1.63 with three (8 row tiles per work-group in both), 0.92 of
    // k_gemm4k.hip's wide kernel, whose work-groups hold two row tiles and 64 columns and therefore fill the chip first.  What this picks is within 6 % of the best of the three over
    // K 1024, 4096 and 14336, N 1024 .. 28672 and 17 .. 512 columns (fourteen of each); the three themselves are up to 2.2 x apart
    const int64_t r2 = g4f_rounds(n_cu, p.n_rb, bs, 32), r3 = g4f_rounds(n_cu, p.n_rb, bs, 48), old = g4f_rounds(n_cu, (tiles / 2 + 7) / 8 * 8, bs, 64);
    if (min(r2 * 130, r3 * 163) >= old * 92) return -1;
    const bool two = r2 * 130 <= r3 * 163;
    if (a.silu_pair) return two ? g4f_launch<1, 2>(st, n_cu, p) : g4f_launch<1, 3>(st, n_cu, p);
    return two ? g4f_launch<0, 2>(st, n_cu, p) : g4f_launch<0, 3>(st, n_cu, p);
}
