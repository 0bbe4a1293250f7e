// tile.hip — the many-column quantised mat-mat for gfx950 at prefill widths:
// Y[c] = W·x_c for tens to hundreds of activation columns, in 32×32 tiles on
// the int8 matrix cores, bit for bit what the one-column GEMV gives each
// column (gemm.hip states the reference's order for each format).
//
// What bounds a full product of this shape is VALU issue, not the matrix cores
// (counters: Q4_K 89% of the SIMD cycles against 13%, Q8_0 78% against 21%;
// Q6_K, which folds its scales at staging, 49% against 25% on the CUs with a
// tile):
// the integer sub-block sums become f32 through arithmetic that the
// reference's order fixes per output. Measured here: an f32 multiply, add or
// fma issues in 2.5 cycles with two waves on a SIMD (5 with one), a
// conversion, shift, pack or integer multiply in 4.3, and an int8 MFMA
// (32 cycles) holds VALU issue back for about 20 of its cycles. So the
// exact integer work is put into cheap f32 steps or into the matrix cores:
//  - The accumulators start at the bit pattern of 1.5·2^23, so a sum reads
//    as the float 1.5·2^23 + sum (|sum| ≤ 2^22 here) and one exact f32
//    subtraction converts it.
//  - Q4_K: Σ sc·dot over the 8 sub-blocks runs as exact f32 fmas, four
//    sub-blocks a chain (4·63·15·32·128 < 2^24), the two chains meeting in
//    one add whose rounding is the reference's int → f32 conversion's.
//    Σ mn·bsum is one f16 MFMA over 16 elements: the eight bsums split into
//    bsum & 63 and bsum >> 6 against mn and 64·mn, all exact in f16, their
//    sum below 2^24.
//  - Q6_K: the sub-block scales are multiplied into the codes when a block
//    is staged; the products (−4096..4096) are split into two int8 planes,
//    v = sc·(q − 32) + 128: v >> 8 (signed) and (v & 255) − 128, whose sums
//    over the 256 elements add up in the accumulators and meet in one fma
//    (16 scale steps an output in f32 would cost more).
//
// Tiling: 8 waves own 64 weight rows × 128 columns, a wave one 32×32 tile,
// two waves a SIMD. A K step is a 256-element block; the next block's
// operands arrive in a second LDS buffer meanwhile, one barrier a step.
//
// MFMA 32x32x32 int8 lane layout (checked on the part): lane l supplies row
// l % 32 of either operand, elements k = 16·(l / 32) .. +15, and receives
// D[8·(i / 4) + 4·(l / 32) + i % 4][l % 32], i < 16. The activations are the
// first operand, so a lane's 16 results are 16 columns of one weight row.
//
// Measured (MI355X, 512 columns, us): Q4_K 4096×14336 253 → 102, 28672×4096
// 233; Q8_0 14336×4096 169 → 131.5, 4096×4096 52 → 33; Q6_K 4096×14336 at
// 203 columns 283 → 89. A step (Q4_K, cycles, clock stamps of a wave): the
// sub-blocks' products and folds 1,800–2,100 — the two waves' VALU issue
// time — the block's fold 650, the table 200; the rest is the barrier and
// the copies' issue, which two waves a SIMD do not cover.
#include "common.h"

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#define MT_ROWS 64
#define MT_COLS 128
#define MT_MAGIC 0x4B400000        // 1.5·2^23
#define MT_MAGICF 12582912.0f

DEV i32x16 mt_dot(i32x4 a, i32x4 b, i32x16 c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
DEV i32x16 mt_magic() {
    i32x16 c;
#pragma unroll
    for (int i = 0; i < 16; i++) c[i] = MT_MAGIC;
    return c;
}
DEV float mt_sum(int d) { return __fsub_rn(__int_as_float(d), MT_MAGICF); }
// The tile of this workgroup. Column tiles of one row tile run on one XCD
// (workgroups are dealt to the eight XCDs by id), whose L2 then holds the
// rows' weights once, where there are at least 8 row tiles to deal.
DEV bool mt_tile(const cj_gemv_args &a, int64_t &r0, int64_t &c0) {
    const int gx = (a.batch + MT_COLS - 1) / MT_COLS;
    const int gy = (int)((a.rows + MT_ROWS - 1) / MT_ROWS);
    const int id = (int)blockIdx.x;
    int rt = id / gx, ct = id % gx;
    if (gy >= 8) {
        const int k = id >> 3;
        rt = k / gx * 8 + (id & 7);
        ct = k % gx;
    }
    r0 = (int64_t)rt * MT_ROWS;
    c0 = (int64_t)ct * MT_COLS;
    return rt < gy;
}

DEV void mt_write(const cj_gemv_args &a, int64_t r, int64_t c, const f32x16 &acc) {
    if (r >= a.rows) return;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int64_t cc = c + 8 * (i / 4) + i % 4;
        if (cc < a.batch) {
            float *y = a.y + cc * a.y_stride + a.y_off + r;
            *y = a.epi == CJ_EPI_ACCUM ? __fadd_rn(*y, acc[i]) : acc[i];
        }
    }
}

// 16 bytes a lane from global memory straight into LDS: lane l's lands 16·l
// bytes past `dst`, which is the wave's.
DEV void mt_dma(const uint8_t *src, uint8_t *dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                     (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}
// The end of a step: the wave's own copies have landed, then every wave's.
DEV void mt_sync() {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    lds_barrier();
}

// ------------------------------------------------------------------- Q4_K

// The copies go straight from global memory into LDS (no registers, no VALU
// work). Weights: the chunk-major row's pieces of four consecutive blocks at
// a time, 64 bytes a (piece, row) pair (a block at a time would touch every
// 128-byte line eight times for 16 bytes), block k of row r in the pair's
// slot k ^ (r / 4 % 4). Columns: word w of column c at w ^ (c % 16). Either
// way 16 lanes' 16-byte reads of 16 rows or columns fall on all banks once.
// The small operands pass through registers into a table a block: waves 0–3
// split the columns' bsums, wave 4 decodes the rows' headers.
#define MN_A 0                                        // [2][8 pieces][64 rows][4 blocks][16]
#define MN_B (2 * 32768)                              // [2][128 columns][256]
#define MN_T (MN_B + 2 * 32768)                       // two blocks' tables:
#define MN_SC 0                                       //   f32 [64 rows][8]
#define MN_MN (MN_SC + MT_ROWS * 32)                  //   f16 [64 rows][16]: mn, 64·mn
#define MN_BS (MN_MN + MT_ROWS * 32)                  //   f16 [128 columns][16]: bsum & 63, bsum >> 6
#define MN_D (MN_BS + MT_COLS * 32)                   //   f32 [2][64]: d, dmin
#define MN_XS (MN_D + 2 * MT_ROWS * 4)                //   f32 [128]
#define MN_TAB (MN_XS + MT_COLS * 4)
#define MN_LDS (MN_T + 2 * MN_TAB)

struct MnQ4 {
    const uint8_t *asrc, *bsrc[4], *esrc, *hsrc;
    uint8_t *lds;
    int64_t nb;
    int t, wave, m, hf, wr, wc, ablk;
    u32x4 e;
    float xs;
    f32x16 acc;

    DEV void init(const cj_gemv_args &a, uint8_t *l, int64_t r0, int64_t c0) {
        lds = l;
        t = threadIdx.x;
        wave = __builtin_amdgcn_readfirstlane(t >> 6);
        m = t & 31;
        hf = (t >> 5) & 1;
        wr = wave >> 2;
        wc = wave & 3;
        nb = a.cols / 256;
        const int lane = t & 63;
        // weight copies: 16 rows of one piece a wave, lane / 4 the row, lane % 4 the slot
        const int row = 16 * (wave & 3) + (lane >> 2);
        ablk = (lane & 3) ^ ((row >> 2) & 3);
        asrc = a.w + min(r0 + row, a.rows - 1) * a.row_bytes;
        // columns 16·wave + 4·i + lane / 16
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = 16 * wave + 4 * i + (lane >> 4);
            bsrc[i] = a.xp + min(c0 + c, (int64_t)a.batch - 1) * a.xp_stride + 16 * ((lane & 15) ^ (c & 15));
        }
        // threads 0..255: half a column's sums; 256..319: a row's header
        if (t < 256) esrc = a.xp + min(c0 + (t >> 1), (int64_t)a.batch - 1) * a.xp_stride + 256;
        else esrc = a.w + min(r0 + (t & 63), a.rows - 1) * a.row_bytes + nb * 128;
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] = 0.0f;
    }
    // copy k of superblock s: pieces 2k and 2k + 1 (waves 0..3 and 4..7) of four blocks
    DEV void copy_a(int64_t s, int k) {
        const int pc = 2 * k + (wave >> 2);
        mt_dma(asrc + (pc * nb + min(4 * s + ablk, nb - 1)) * 16, lds + MN_A + (s & 1) * 32768 + pc * 4096 + (wave & 3) * 1024);
    }
    DEV void copy_b(int64_t b, int buf, int i) { mt_dma(bsrc[i] + b * 320, lds + MN_B + buf * 32768 + wave * 4096 + i * 1024); }
    DEV void fetch(int64_t b) {
        if (t < 256) {
            e = *(const u32x4 *)(esrc + b * 320 + 16 * (t & 1));
            xs = *(const float *)(esrc + b * 320 + 32);
        } else if (wave == 4) {
            e = *(const u32x4 *)(esrc + b * 16);
        }
    }
    // the fetched block's tables
    DEV void table(int buf) {
        uint8_t *T = lds + MN_T + buf * MN_TAB;
        if (t < 256) {
            const int c = t >> 1, half = t & 1;
            _Float16 lo[4], hi[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int s = (int)e[i];
                lo[i] = (_Float16)(short)(s & 63);
                hi[i] = (_Float16)(short)(s >> 6);
            }
            __builtin_memcpy(T + MN_BS + c * 32 + 8 * half, lo, 8);
            __builtin_memcpy(T + MN_BS + c * 32 + 16 + 8 * half, hi, 8);
            *(float *)(T + MN_XS + c * 4) = xs;
        } else if (wave == 4) {
            const int r = t & 63;
            const uint32_t X = e.y, Y = e.z, Z = e.w;
            const uint32_t s4[2] = {X & 0x3F3F3F3Fu, (Z & 0x0F0F0F0Fu) | ((X >> 2) & 0x30303030u)};
            const uint32_t m4[2] = {Y & 0x3F3F3F3Fu, ((Z >> 4) & 0x0F0F0F0Fu) | ((Y >> 2) & 0x30303030u)};
            f32x4 s0, s1;
            f16x8 mn, mh;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                s0[k] = (float)((s4[0] >> (8 * k)) & 255);
                s1[k] = (float)((s4[1] >> (8 * k)) & 255);
            }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int v = (int)((m4[k >> 2] >> (8 * (k & 3))) & 255);
                mn[k] = (_Float16)(short)v;
                mh[k] = (_Float16)(short)(64 * v);
            }
            *(f32x4 *)(T + MN_SC + r * 32) = s0;
            *(f32x4 *)(T + MN_SC + r * 32 + 16) = s1;
            *(f16x8 *)(T + MN_MN + r * 32) = mn;
            *(f16x8 *)(T + MN_MN + r * 32 + 16) = mh;
            *(float *)(T + MN_D + r * 4) = h2f(e.x);
            *(float *)(T + MN_D + (MT_ROWS + r) * 4) = h2f(e.x >> 16);
        }
    }
    // block K of superblock s; mid(j) runs after sub-block j's fold
    template <int K, class Mid>
    DEV void block(int64_t s, Mid &&mid) {
        const int row = 32 * wr + m, col = 32 * wc + m;
        const uint8_t *ap = lds + MN_A + (s & 1) * 32768 + hf * 4096 + row * 64 + 16 * (K ^ ((row >> 2) & 3));
        const uint8_t *T = lds + MN_T + (K & 1) * MN_TAB;
        const uint8_t *bp = lds + MN_B + (K & 1) * 32768 + col * 256;
        const int sw = (m & 15) ^ hf;
        i32x4 x[8];
        u32x4 q[4];
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
            q[g4] = *(const u32x4 *)(ap + 8192 * g4);
            x[2 * g4] = *(const i32x4 *)(bp + 16 * (sw ^ (4 * g4)));
            x[2 * g4 + 1] = *(const i32x4 *)(bp + 16 * (sw ^ (4 * g4 + 2)));
        }
        const f32x4 sc0 = *(const f32x4 *)(T + MN_SC + row * 32), sc1 = *(const f32x4 *)(T + MN_SC + row * 32 + 16);
        const float sc[8] = {sc0[0], sc0[1], sc0[2], sc0[3], sc1[0], sc1[1], sc1[2], sc1[3]};
        const f16x8 bs = *(const f16x8 *)(T + MN_BS + col * 32 + 16 * hf), mn = *(const f16x8 *)(T + MN_MN + row * 32 + 16 * hf);
        const i32x16 M = mt_magic();
        auto frag = [&](int j) {
            i32x4 w;
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = (int)(((j & 1) ? q[j >> 1][i] >> 4 : q[j >> 1][i]) & 0x0F0F0F0Fu);
            return w;
        };
        f32x16 S0, S1;
        i32x16 P[2];
        P[0] = mt_dot(x[0], frag(0), M);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (j < 7) P[(j + 1) & 1] = mt_dot(x[j + 1], frag(j + 1), M);
            f32x16 &S = j < 4 ? S0 : S1;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const float v = mt_sum(P[j & 1][i]);
                S[i] = (j & 3) ? __fmaf_rn(sc[j], v, S[i]) : __fmul_rn(sc[j], v);
            }
            // the product after next waits for this fold (left free, the
            // compiler issues all eight first and spills their results)
            if (j < 6) asm volatile("" : "+v"(x[j + 2]), "+v"(S));
            mid(j);
        }
        f32x16 Dm;
#pragma unroll
        for (int i = 0; i < 16; i++) Dm[i] = 0.0f;
        Dm = __builtin_amdgcn_mfma_f32_32x32x16_f16(bs, mn, Dm, 0, 0, 0);
        const float d = *(const float *)(T + MN_D + row * 4), dm = *(const float *)(T + MN_D + (MT_ROWS + row) * 4);
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            const f32x4 xv = *(const f32x4 *)(T + MN_XS + (32 * wc + 8 * q4 + 4 * hf) * 4);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int i = 4 * q4 + k;
                const float sumi = __fadd_rn(S0[i], S1[i]);
                acc[i] = __fsub_rn(__fadd_rn(acc[i], __fmul_rn(__fmul_rn(d, xv[k]), sumi)), __fmul_rn(__fmul_rn(dm, xv[k]), Dm[i]));
            }
        }
    }
    template <int K>
    DEV bool step(int64_t s) {
        const int64_t b = 4 * s + K;
        if (b >= nb) return true;
        const int64_t n = min(b + 1, nb - 1);
        // the copies spread over the first sub-blocks: issued together, the
        // waves queue on the address unit (Q8_0 14336×4096 × 512: 138 → 131.5 us,
        // Q4_K 4096×14336 × 512: 104.6 → 102.2; spread to the step's end they
        // come late: 152, 113)
        block<K>(s, [&](int j) {
            if (j < 2) {
                copy_b(n, (K + 1) & 1, 2 * j);
                copy_b(n, (K + 1) & 1, 2 * j + 1);
            }
            if (j == 2) copy_a(s + 1, K);
        });
        table((K + 1) & 1);
        mt_sync();
        fetch(min(b + 2, nb - 1));
        return false;
    }
};

extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) cj_gemm_t_q4k(cj_gemv_args a) {
    __shared__ __align__(16) uint8_t mt_lds[MN_LDS];
    int64_t r0, c0;
    if (!mt_tile(a, r0, c0)) return;
    MnQ4 W;
    W.init(a, mt_lds, r0, c0);
    W.fetch(0);
#pragma unroll
    for (int k = 0; k < 4; k++) W.copy_a(0, k);
#pragma unroll
    for (int i = 0; i < 4; i++) W.copy_b(0, 0, i);
    W.table(0);
    mt_sync();
    W.fetch(min((int64_t)1, W.nb - 1));
    for (int64_t s = 0;; s++) {
        if (W.step<0>(s)) break;
        if (W.step<1>(s)) break;
        if (W.step<2>(s)) break;
        if (W.step<3>(s)) break;
    }
    mt_write(a, r0 + 32 * W.wr + W.m, c0 + 32 * W.wc + 4 * W.hf, W.acc);
}

// ------------------------------------------------------------------- Q6_K

// Rows and columns lie 272 bytes apart in LDS: 16 lanes' 16-byte reads fall
// on all 64 banks once.
#define MT_TS 272
#define MT_Q6_B (2 * MT_ROWS * MT_TS)
#define MT_Q6_D (MT_Q6_B + MT_COLS * MT_TS)           // f32 [64]
#define MT_Q6_XS (MT_Q6_D + MT_ROWS * 4)              // f32 [128]
#define MT_Q6_BUF (MT_Q6_XS + MT_COLS * 4)

// The columns' codes, 16 words a column, and their scales.
struct MtB {
    const uint8_t *src[4];
    const uint8_t *esrc;
    u32x4 v[4];
    float xs;
    DEV void init(const cj_gemv_args &a, int64_t c0, int t) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t c = min(c0 + (t >> 4) + 32 * i, (int64_t)a.batch - 1);
            src[i] = a.xp + c * a.xp_stride + 16 * (t & 15);
        }
        esrc = a.xp + min(c0 + ((t & 255) >> 1), (int64_t)a.batch - 1) * a.xp_stride + 288;
    }
    DEV void fetch(int64_t b) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = *(const u32x4 *)(src[i] + b * 320);
        xs = *(const float *)(esrc + b * 320);
    }
    DEV void store(uint8_t *lds, int t) const {
#pragma unroll
        for (int i = 0; i < 4; i++) *(u32x4 *)(lds + ((t >> 4) + 32 * i) * MT_TS + 16 * (t & 15)) = v[i];
    }
};

// Prepared row: [ql nb·128][qh nb·64][scales nb·16][d nb·2]. In half h of a
// block, word 2·kk + l16 of its ql (16 bytes) holds the elements 32·kk +
// 16·l16 .. +15 of the half in its low nibbles and those 64 further on in
// its high nibbles; qh bits 2·kk and 2·kk + 4 of word l16 are their top two.
// Thread (row t / 8, h, l16, kk) forms both runs of 16.
struct MtQ6A {
    const uint8_t *ql, *qh, *sc, *d;
    uint4 vl, vh;
    uint2 vs;
    uint32_t vd;
    DEV void init(const cj_gemv_args &a, int64_t r0, int t) {
        const int64_t nb = a.cols / 256;
        const int h = (t >> 2) & 1, l16 = (t >> 1) & 1, kk = t & 1;
        const uint8_t *row = a.w + min(r0 + (t >> 3), a.rows - 1) * a.row_bytes;
        ql = row + 64 * h + 32 * kk + 16 * l16;
        qh = row + nb * 128 + 32 * h + 16 * l16;
        sc = row + nb * 192 + 8 * h;
        d = row + nb * 208;
    }
    DEV void fetch(int64_t b) {
        vl = *(const uint4 *)(ql + b * 128);
        vh = *(const uint4 *)(qh + b * 64);
        vs = *(const uint2 *)(sc + b * 16);
        vd = *(const uint16_t *)(d + b * 2);
    }
    // 4 values of 6 bits × sc, + 128, as planes of bytes: the products by
    // even and odd byte (16 bits each)
    DEV static void planes(uint32_t u, int s, uint32_t &hi, uint32_t &lo) {
        typedef short s16x2 __attribute__((ext_vector_type(2)));
        const short c = (short)(128 - 32 * s), s16 = (short)s;
        const s16x2 vsc = {s16, s16}, vc = {c, c};
        const uint32_t ue = u & 0x00FF00FFu, uo = (u >> 8) & 0x00FF00FFu;
        s16x2 e, o;
        __builtin_memcpy(&e, &ue, 4);
        __builtin_memcpy(&o, &uo, 4);
        e = e * vsc + vc;
        o = o * vsc + vc;
        uint32_t we, wo;
        __builtin_memcpy(&we, &e, 4);
        __builtin_memcpy(&wo, &o, 4);
        // v_perm selects bytes 0..3 from its second operand, 4..7 from its first
        hi = __builtin_amdgcn_perm(wo, we, 0x07030501u);
        lo = __builtin_amdgcn_perm(wo, we, 0x06020400u) ^ 0x80808080u;
    }
    DEV void store(uint8_t *buf, int t) const {
        const int h = (t >> 2) & 1, l16 = (t >> 1) & 1, kk = t & 1, r = t >> 3, sh = 16 * kk + 8 * l16;
        const int s0 = (int)(int8_t)(vs.x >> sh), s1 = (int)(int8_t)(vs.y >> sh);
        const uint32_t wl[4] = {vl.x, vl.y, vl.z, vl.w}, wh[4] = {vh.x, vh.y, vh.z, vh.w};
        u32x4 h0, l0, h1, l1;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t top = wh[i] >> (2 * kk);
            const uint32_t u0 = (wl[i] & 0x0F0F0F0Fu) | ((top << 4) & 0x30303030u);
            const uint32_t u1 = ((wl[i] >> 4) & 0x0F0F0F0Fu) | (top & 0x30303030u);
            uint32_t x, y;
            planes(u0, s0, x, y);
            h0[i] = x; l0[i] = y;
            planes(u1, s1, x, y);
            h1[i] = x; l1[i] = y;
        }
        uint8_t *dst = buf + r * MT_TS + 128 * h + 32 * kk + 16 * l16;
        *(u32x4 *)dst = h0;
        *(u32x4 *)(dst + 64) = h1;
        *(u32x4 *)(dst + MT_ROWS * MT_TS) = l0;
        *(u32x4 *)(dst + MT_ROWS * MT_TS + 64) = l1;
        if ((t & 7) == 0) *(float *)(buf + MT_Q6_D + r * 4) = h2f(vd);
    }
};

DEV void mt_q6_bstore(const MtB &B, uint8_t *buf, int t) {
    B.store(buf + MT_Q6_B, t);
    if (t < 256 && !(t & 1)) *(float *)(buf + MT_Q6_XS + (t >> 1) * 4) = B.xs;
}

DEV void mt_q6_block(const uint8_t *buf, int wr, int wc, int m, int hf, f32x16 &acc) {
    const uint8_t *wp = buf + (32 * wr + m) * MT_TS + 16 * hf;
    const uint8_t *xp = buf + MT_Q6_B + (32 * wc + m) * MT_TS + 16 * hf;
    i32x16 H = mt_magic(), L = mt_magic();
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const i32x4 x = *(const i32x4 *)(xp + 32 * j);
        H = mt_dot(x, *(const i32x4 *)(wp + 32 * j), H);
        L = mt_dot(x, *(const i32x4 *)(wp + MT_ROWS * MT_TS + 32 * j), L);
    }
    const float d = *(const float *)(buf + MT_Q6_D + (32 * wr + m) * 4);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const f32x4 xs = *(const f32x4 *)(buf + MT_Q6_XS + (32 * wc + 8 * q + 4 * hf) * 4);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float isum = __fmaf_rn(256.0f, mt_sum(H[4 * q + i]), mt_sum(L[4 * q + i]));
            acc[4 * q + i] = __fadd_rn(acc[4 * q + i], __fmul_rn(__fmul_rn(d, xs[i]), isum));
        }
    }
}

extern "C" __global__ void __launch_bounds__(512) cj_gemm_t_q6k(cj_gemv_args a) {
    __shared__ __align__(16) uint8_t mt_lds[2 * MT_Q6_BUF];
    const int t = threadIdx.x, wave = t >> 6, m = t & 31, hf = (t >> 5) & 1, wr = wave >> 2, wc = wave & 3;
    int64_t r0, c0;
    if (!mt_tile(a, r0, c0)) return;
    const int64_t nb = a.cols / 256;
    MtQ6A A;
    MtB B;
    A.init(a, r0, t);
    B.init(a, c0, t);
    A.fetch(0);
    B.fetch(0);
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.0f;
    A.store(mt_lds, t);
    mt_q6_bstore(B, mt_lds, t);
    A.fetch(min((int64_t)1, nb - 1));
    B.fetch(min((int64_t)1, nb - 1));
    lds_barrier();
    uint8_t *cur = mt_lds, *nxt = mt_lds + MT_Q6_BUF;
    for (int64_t b = 0; b < nb; b++) {
        mt_q6_block(cur, wr, wc, m, hf, acc);
        A.store(nxt, t);
        mt_q6_bstore(B, nxt, t);
        const int64_t bn = min(b + 2, nb - 1);
        A.fetch(bn);
        B.fetch(bn);
        lds_barrier();
        uint8_t *s = cur;
        cur = nxt;
        nxt = s;
    }
    mt_write(a, r0 + 32 * wr + m, c0 + 32 * wc + 4 * hf, acc);
}

// ------------------------------------------------------------------- Q8_0

// The same copies into LDS: a group of 8 blocks is 256 code bytes a row and
// a column, word w of either at w ^ (row or column % 16). Per output and
// block the reference's rounded steps are fs = Σ_j (d_j·xs_j)·dot_j over the
// group's blocks, then acc += fs; the d·xs of two blocks are one outer
// product (v_mfma_f32_32x32x1_2b_f32, one rounding a product, checked on the
// part against the f32 multiply with denormals). A short last group repeats
// the row's last block under scales of zero, whose terms (±0) change no sum.
typedef float f32x32 __attribute__((ext_vector_type(32)));

#define M8_A 0                                        // [64 rows][256]
#define M8_B (MT_ROWS * 256)                          // [128 columns][256]
#define M8_BUF (M8_B + MT_COLS * 256)
#define M8_T (2 * M8_BUF)                             // two groups' scales:
#define M8_D 0                                        //   f32 [8][64 rows]
#define M8_XS (8 * MT_ROWS * 4)                       //   f32 [8][128 columns]
#define M8_TAB (M8_XS + 8 * MT_COLS * 4)
#define M8_LDS (M8_T + 2 * M8_TAB)

// fl(a·b) for a of lane l % 32 as D's row and b of lane l % 32 as its column;
// lanes 0..31 give the first 16 results' operands, 32..63 the others'
DEV f32x32 mt_outer(float a, float b) {
    f32x32 z;
#pragma unroll
    for (int i = 0; i < 32; i++) z[i] = 0.0f;
    return __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, z, 0, 0, 0);
}

// Blocks 2p and 2p + 1 of a group: their integer dots and scale products.
struct M8Pair {
    i32x16 d0, d1;
    f32x32 s;
    // ao, bo: the lane's row and column in the buffer, its swizzle in bits 4..7
    DEV void dot(const uint8_t *buf, const uint8_t *T, int ao, int bo, int p, int row, int col, int hf, const i32x16 &M) {
        d0 = mt_dot(*(const i32x4 *)(buf + (bo ^ (64 * p))), *(const i32x4 *)(buf + (ao ^ (64 * p))), M);
        d1 = mt_dot(*(const i32x4 *)(buf + (bo ^ (64 * p + 32))), *(const i32x4 *)(buf + (ao ^ (64 * p + 32))), M);
        s = mt_outer(*(const float *)(T + M8_XS + ((2 * p + hf) * MT_COLS + col) * 4),
                     *(const float *)(T + M8_D + ((2 * p + hf) * MT_ROWS + row) * 4));
    }
    template <bool FIRST>
    DEV void fold(f32x16 &fs) const {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float t0 = __fmul_rn(s[i], mt_sum(d0[i]));
            fs[i] = FIRST ? t0 : __fadd_rn(fs[i], t0);
            fs[i] = __fadd_rn(fs[i], __fmul_rn(s[16 + i], mt_sum(d1[i])));
        }
    }
};

struct M8 {
    const uint8_t *asrc[2], *bsrc[4], *ssrc;
    uint8_t *lds;
    int64_t nb32;
    int t, wave, row, col, hf, ng, word;
    u32x4 e;
    f32x16 acc;

    DEV void init(const cj_gemv_args &a, uint8_t *l, int64_t r0, int64_t c0) {
        lds = l;
        t = threadIdx.x;
        wave = __builtin_amdgcn_readfirstlane(t >> 6);
        hf = (t >> 5) & 1;
        row = 32 * (wave >> 2) + (t & 31);
        col = 32 * (wave & 3) + (t & 31);
        nb32 = a.cols / 32;
        ng = (int)((a.cols + 255) / 256);
        const int lane = t & 63;
        // rows 8·wave + 4·i + lane / 16, columns 16·wave + 4·i + lane / 16
#pragma unroll
        for (int i = 0; i < 2; i++) asrc[i] = a.w + min(r0 + 8 * wave + 4 * i + (lane >> 4), a.rows - 1) * a.row_bytes;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = 16 * wave + 4 * i + (lane >> 4);
            bsrc[i] = a.xp + min(c0 + c, (int64_t)a.batch - 1) * a.xp_stride + 16 * ((lane & 15) ^ (c & 15));
        }
        // threads 0..255: four of a column's scales; 256..319: a row's eight
        if (t < 256) ssrc = a.xp + min(c0 + (t >> 1), (int64_t)a.batch - 1) * a.xp_stride + 288 + 16 * (t & 1);
        else ssrc = a.w + min(r0 + (t & 63), a.rows - 1) * a.row_bytes + nb32 * 32;
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] = 0.0f;
    }
    DEV void copy_a(int g, int buf, int i) {
        const int lane = t & 63, w = (lane & 15) ^ ((8 * wave + 4 * i + (lane >> 4)) & 15);
        const int64_t blk = min((int64_t)8 * g + (w >> 1), nb32 - 1);
        mt_dma(asrc[i] + blk * 32 + 16 * (w & 1), lds + buf * M8_BUF + M8_A + wave * 2048 + i * 1024);
    }
    DEV void copy_b(int g, int buf, int i) { mt_dma(bsrc[i] + (int64_t)g * 320, lds + buf * M8_BUF + M8_B + wave * 4096 + i * 1024); }
    DEV void fetch(int g) {
        if (t < 256) e = *(const u32x4 *)(ssrc + (int64_t)g * 320);
        else if (wave == 4) e = *(const u32x4 *)(ssrc + (int64_t)g * 16);
    }
    DEV void table(int g, int buf) {
        uint8_t *T = lds + M8_T + buf * M8_TAB;
        const int nj = (int)min(nb32 - 8 * (int64_t)g, (int64_t)8);
        if (t < 256) {
            const int c = t >> 1, j0 = 4 * (t & 1);
#pragma unroll
            for (int j = 0; j < 4; j++)
                *(float *)(T + M8_XS + ((j0 + j) * MT_COLS + c) * 4) = j0 + j < nj ? __uint_as_float(e[j]) : 0.0f;
        } else if (wave == 4) {
#pragma unroll
            for (int j = 0; j < 8; j++)
                *(float *)(T + M8_D + (j * MT_ROWS + (t & 63)) * 4) = j < nj ? h2f(e[j >> 1] >> (16 * (j & 1))) : 0.0f;
        }
    }
    // One pair's products are formed while the pair before is folded. The
    // empty asm ties a pair's operand addresses to the fold two before it:
    // left free, the compiler issues all the products first and spills their
    // results.
    template <class Mid>
    DEV void group(int buf, Mid &&mid) {
        const uint8_t *b = lds + buf * M8_BUF, *T = lds + M8_T + buf * M8_TAB;
        const i32x16 M = mt_magic();
        int ao = M8_A + row * 256 + 16 * ((row & 15) ^ hf), bo = M8_B + col * 256 + 16 * ((col & 15) ^ hf);
        f32x16 fs;
        M8Pair P, Q;
        P.dot(b, T, ao, bo, 0, row, col, hf, M);
        Q.dot(b, T, ao, bo, 1, row, col, hf, M);
        mid(0);
        P.fold<true>(fs);
        asm volatile("" : "+v"(ao), "+v"(bo), "+v"(fs));
        P.dot(b, T, ao, bo, 2, row, col, hf, M);
        mid(1);
        Q.fold<false>(fs);
        asm volatile("" : "+v"(ao), "+v"(bo), "+v"(fs));
        Q.dot(b, T, ao, bo, 3, row, col, hf, M);
        mid(2);
        P.fold<false>(fs);
        Q.fold<false>(fs);
#pragma unroll
        for (int i = 0; i < 16; i++) acc[i] = __fadd_rn(acc[i], fs[i]);
    }
    DEV void step(int g, int buf) {
        const int n = min(g + 1, ng - 1);
        group(buf, [&](int p) {   // (the copies spread over the step's start)
            if (p < 2) {
                copy_a(n, buf ^ 1, p);
                copy_b(n, buf ^ 1, 2 * p);
                copy_b(n, buf ^ 1, 2 * p + 1);
            }
        });
        table(n, buf ^ 1);
        mt_sync();
        fetch(min(g + 2, ng - 1));
    }
};

extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) cj_gemm_t_q80(cj_gemv_args a) {
    __shared__ __align__(16) uint8_t mt_lds[M8_LDS];
    int64_t r0, c0;
    if (!mt_tile(a, r0, c0)) return;
    M8 W;
    W.init(a, mt_lds, r0, c0);
    W.fetch(0);
#pragma unroll
    for (int i = 0; i < 2; i++) W.copy_a(0, 0, i);
#pragma unroll
    for (int i = 0; i < 4; i++) W.copy_b(0, 0, i);
    W.table(0, 0);
    mt_sync();
    W.fetch(min(1, W.ng - 1));
    for (int g = 0; g < W.ng; g += 2) {
        W.step(g, 0);
        if (g + 1 < W.ng) W.step(g + 1, 1);
    }
    mt_write(a, r0 + W.row, c0 + 32 * (W.wave & 3) + 4 * W.hf, W.acc);
}

// ------------------------------------------------- MXFP4 experts of many rows

// A workgroup (row tile, expert) over the selections of the expert, as
// moe_grp_body, its products on the int8 matrix cores. A row value is the sum
// of 32 partials by the half-wave's butterfly (16, 8, 4, 2, 1), partial L
// holding the blocks L, L + 32, L + 64 in order. Blocks ≡ j mod 8 are wave
// j's: the partials j, j + 8, j + 16, j + 24, which the butterfly's first two
// levels join; the waves' values meet in LDS for the other three. The eight
// waves read the same 128-byte lines of the weight rows (16 bytes a block) and
// of the packs together. A wave keeps its weights decoded in registers over
// the members, which go 32 a chunk; the next chunk's codes are requested
// before the current one's epilogue.
//
// VALU issue takes 55% of the SIMD cycles (counters, 300 rows, gate|up; matrix
// cores 4%): four steps an output and block (the sum's conversion, the two
// scales, the add), where the dot4 kernel spends twelve; a third of the wave
// cycles wait at two waves a SIMD.
// Measured (MI355X, 32 experts of 2880 × 2880, 4 a row): 512 rows gate|up
// 1058 → 449 us, down 604 → 261; 128 rows 281 → 263, 163 → 140. One and two
// sweeps: 8 experts of 2048 × 1024, 2 a row, 64 rows 38 → 15 and 18 → 8. At
// few rows the weights' decode and scale table bound it (2880 × 2880: 250 us
// and 124 for all the experts from 24 to 64 rows).
template <int EPI, int KB>
DEV void moe_tile_body(const cj_moe_grp_args &a) {
    constexpr int RT = EPI == CJ_EPI_GLU ? 2 : 1, ROWS = 32 * RT, NM = 4 * KB, WS = ROWS + 4;
    __shared__ __align__(16) float ws[32 * KB * WS];
    __shared__ __align__(16) float part[8 * RT * 1024];   // [wave][tile][16 rows' quads][64 lanes][4]
    __shared__ float act[32 * 33];
    __shared__ int mi[3][32];   // a wave may still read the chunk before while another requests the next
    const int e = blockIdx.y;
    const int c = a.cnt[e];
    if (c == 0) return;
    const int t = threadIdx.x, lane = t & 63, m32 = lane & 31, hf = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nb = (int)(a.cols / 32);
    const uint8_t *W = a.w + (int64_t)e * a.expert_bytes;
    const int64_t row0 = (int64_t)blockIdx.x * ROWS;
    const int32_t *mem = a.mem + (int64_t)e * a.cap;

    i32x4 x[NM];
    float xs[NM];
    auto fetch = [&](int j0, int buf) {
        const int me = mem[min(j0 + m32, c - 1)];
        if (t < 32) mi[buf][t] = me;
        const uint8_t *row = a.xp + (int64_t)(me / a.x_per) * a.xp_stride + 32 * wave;
#pragma unroll
        for (int k = 0; k < NM; k++) {
            const int q = min(8 * k + wave, nb - 1) >> 3;
            x[k] = *(const i32x4 *)(row + q * 320 + 16 * hf);
            xs[k] = *(const float *)(row + q * 320 + 288 - 28 * wave);
        }
    };
    fetch(0, 0);
    i32x4 w[RT][NM];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const uint8_t *wr = W + min(row0 + 32 * r + m32, a.rows - 1) * a.row_bytes;
#pragma unroll
        for (int k = 0; k < NM; k++) w[r][k] = *(const i32x4 *)(wr + 16 * min(8 * k + wave, nb - 1));
    }
    for (int i = t; i < ROWS * 32 * KB; i += 512) {
        const int r = i / (32 * KB), b = i % (32 * KB);
        ws[b * WS + r] = b < nb ? mxfp4_scale(W[min(row0 + r, a.rows - 1) * a.row_bytes + 16 * nb + b]) : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int k = 0; k < NM; k++)
#pragma unroll
            for (int i = 0; i < 4; i++) w[r][k][i] = (int)e2m1_x4((uint32_t)w[r][k][i] >> (4 * hf));
    __syncthreads();

    int buf = 0;
    for (int j0 = 0; j0 < c; j0 += 32, buf = buf == 2 ? 0 : buf + 1) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            // the chains of partials 0, 2, 1, 3 (in units of 8), their blocks in order
            f32x16 s, u, v;
            i32x16 Z;   // (the conversions cost less than 16 registers for mt_magic, which would spill)
#pragma unroll
            for (int i = 0; i < 16; i++) { s[i] = u[i] = v[i] = 0.0f; Z[i] = 0; }
#pragma unroll
            for (int f = 0; f < NM; f++) {
                constexpr int ORDER[4] = {0, 2, 1, 3};
                const int n = 4 * (f % KB) + ORDER[f / KB], b = 8 * n + wave;
                f32x16 &p = f / KB == 0 ? s : f / KB == 3 ? v : u;
                if (f == 2 * KB) {
#pragma unroll
                    for (int i = 0; i < 16; i++) { s[i] = __fadd_rn(s[i], u[i]); u[i] = 0.0f; }
                }
                if (b < nb) {
                    const i32x16 d = mt_dot(w[r][n], x[n], Z);
                    const float *wp = ws + b * WS + 32 * r + 4 * hf;
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const f32x4 wv = *(const f32x4 *)(wp + 8 * q);
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const float term = __fmul_rn(__fmul_rn((float)d[4 * q + k], wv[k]), xs[n]);
                            p[4 * q + k] = __fadd_rn(p[4 * q + k], term);
                        }
                    }
                }
                // the next product waits for this fold (as in the Q4_K kernel)
                if (f + 1 < NM) asm volatile("" : "+v"(x[4 * ((f + 1) % KB) + ORDER[(f + 1) / KB]]), "+v"(p));
            }
            float *pp = part + (wave * RT + r) * 1024 + 4 * lane;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                f32x4 o;
#pragma unroll
                for (int k = 0; k < 4; k++) o[k] = __fadd_rn(s[4 * q + k], __fadd_rn(u[4 * q + k], v[4 * q + k]));
                *(f32x4 *)(pp + 256 * q) = o;
            }
        }
        if (j0 + 32 < c) fetch(j0 + 32, buf == 2 ? 0 : buf + 1);
        lds_barrier();
        const int nc = min(32, c - j0);
        if (t < 256 * RT) {
            // thread (tile t / 256, quad, lane): four rows of one member
            f32x4 p[8];
#pragma unroll
            for (int k = 0; k < 8; k++) p[k] = *(const f32x4 *)(part + (k * RT + (t >> 8)) * 1024 + 4 * (t & 255));
            f32x4 o;
#pragma unroll
            for (int k = 0; k < 4; k++)
                o[k] = __fadd_rn(__fadd_rn(__fadd_rn(p[0][k], p[4][k]), __fadd_rn(p[2][k], p[6][k])),
                                 __fadd_rn(__fadd_rn(p[1][k], p[5][k]), __fadd_rn(p[3][k], p[7][k])));
            const int rl = 32 * (t >> 8) + 8 * ((t >> 6) & 3) + 4 * hf;
            if (EPI == CJ_EPI_GLU) {
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const int64_t ai = (row0 + rl) / 2 + k;
                    act[m32 * 33 + rl / 2 + k] =
                        m32 < nc && ai < a.act_n ? glu_value(a.glu_form, ai, a.act_n, o[2 * k], o[2 * k + 1]) : 0.0f;
                }
            } else if (m32 < nc && row0 + rl < a.rows) {   // (rows are a multiple of four)
                *(f32x4 *)(a.y + (int64_t)mi[buf][m32] * a.y_stride + row0 + rl) = o;
            }
        }
        lds_barrier();
        if (EPI == CJ_EPI_GLU) {
            // the 32 values of a member are one 32-block of its activation
            const int64_t ab = row0 / ROWS;
            const int o = t & 31;
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const int jj = 16 * k + (t >> 5);
                const float v = act[jj * 33 + o];
                const float bm = xmax32(fabsf(v));
                const float inv = bm > 0.0f ? __fdiv_rn(127.0f, bm) : 0.0f;
                const int q = round_away(__fmul_rn(v, inv));
                const int sq = xsum32_i(q);
                if (jj < nc) {
                    uint8_t *ob = a.outp + (int64_t)mi[buf][jj] * a.outp_stride + (ab >> 3) * 320;
                    ob[(ab & 7) * 32 + o] = (uint8_t)(int8_t)q;
                    if (o == 0) {
                        *(int32_t *)(ob + 256 + 4 * (ab & 7)) = sq;
                        *(float *)(ob + 288 + 4 * (ab & 7)) = __fdiv_rn(bm, 127.0f);
                    }
                }
            }
        }
    }
}
#define MOE_TILE_KERNEL(E, EPI, KB)                                                                                          \
    extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))                                \
        cj_moe_t_##E##_k##KB(cj_moe_grp_args a) {                                                                            \
        moe_tile_body<EPI, KB>(a);                                                                                           \
    }
MOE_TILE_KERNEL(g, CJ_EPI_GLU, 1)
MOE_TILE_KERNEL(g, CJ_EPI_GLU, 2)
MOE_TILE_KERNEL(g, CJ_EPI_GLU, 3)
MOE_TILE_KERNEL(s, CJ_EPI_STORE, 1)
MOE_TILE_KERNEL(s, CJ_EPI_STORE, 2)
MOE_TILE_KERNEL(s, CJ_EPI_STORE, 3)
