// FP32 direct sums on the BF16 matrix cores (MODE_FLOAT; direct_gemm.h has the
// method), included by pc_direct.hip.
//
// Precision: every factor is an FP32 value held as three BF16 parts (hi, mid,
// lo), which are its 24 bits without loss; a product takes the six part
// products down to 2^-16 of the term (the dropped ones are below its FP32
// rounding) and accumulates in FP32; every 240 points (fewer for small work,
// direct_chunk) the FP32 sums are folded into FP64.  Against chains of FP32 FMAs
// the sums are a little more accurate (128 random unit terms: 2.4e-7 of the sum
// against 2.8e-7; the accumulation's slight bias, -1.6e-8 of a sum, is cancelled
// by summing the negated terms of every second group).  With phases held as
// 32-bit fractions of a cycle (Fresnel) or reduced in FP64 (RS), the field's
// error against 64 bits is 3.5e-7 (Fresnel, 100k points, 3840x2160; 6.4e-7 with
// scalar FP32 FMAs) and 3.9e-7 (RS, 20k points; 7.1e-7); with 200 points, folded
// every 60, 1.2e-7 to 2.4e-7 at depths to 1.2 m (2.9e-7 to 3.1e-6), or up to 7.4e-7
// (2.1e-6) where the per-pixel kernel takes a part of the RS pairs.
//
// What bounds it: the matrix cores (48 flops per point and pixel for Fresnel, 72,
// 96 and 144 for RS of ranks 2, 3 and 4) and the generation of 256 factors per
// point and 128 x 128 tile on the VALU.  VALU instructions can issue while a BF16
// MFMA runs (not while an FP32 one does, whose 155 TFLOP/s this form beats), so one
// workgroup of 8 waves per CU, two per SIMD, and in each wave's stream the next
// batch's generation alternates, slot by slot, with this batch's products
// (double-buffered factors, one barrier per batch).  By the counters below the two
// hardly overlap all the same: what the alternation gains is the waits.
// Fresnel, 100k points at 3840x2160: 94-99 -> 32-34 ms (24.3 without the
// generation; FP32 MFMA 60, 4 waves without the alternation 40); RS, 20k points
// (rank 2): 30-31 -> 13.7-14.2 ms (7.7 without it; FP32 MFMA 27.5); 22k points at
// 1920x1080, 8 um, z 0.25 m (ranks 2 to 4, boxes inside the hologram): 12.7 -> 6.5.
// Counters: the matrix cores are busy 57 % (RS 42 %), the VALU 52 % (54 %) of the
// time; a third of a wave's time goes into waits for LDS and the barrier.
#pragma once

namespace dgemm {

constexpr int SUP = 480;                // points classified at a time: wave w holds points PW w .. PW w + PW - 1
constexpr int NTF = Kind<float>::NTH;
constexpr int GHF = Kind<float>::GH;
constexpr int PW = SUP / (NTF / 64);
constexpr int CELL = DIRECT_CELL, CELLS = SUP / CELL;   // a group (the points of a fold) is 1, 2, 4 or 8 cells
constexpr int LINES = 128;              // rows or columns of a tile
// A batch has factors for two or three K steps (16-deep MFMAs of 8 complex
// entries each); lists are padded to whole batches, per group and rank.
//  * Fresnel (rank 1): 16 points, two steps of three parts, [part][line][16 + 4]
//    (80-byte lines do not conflict).
//  * RS: step A, the large ranks in three parts, [part][line][8]; steps B, the
//    ranks that weigh less than 2^-7, in two parts, [part][line][16], the halves
//    of a line exchanged on every second 4 lines (no conflicts).  Ranks 2 and 3: 8
//    points, rank 0 in A, ranks 1 (and 2) in B.  Rank 4: 4 points, ranks 0 and 1 in
//    A, ranks 2 and 3 in B.
constexpr int ROWW = 16 + 4;
constexpr int BOFF = 3 * LINES * 8;     // of steps B
template <int R>
constexpr int batch_points() { return R == 1 ? 16 : R == 4 ? 4 : 8; }
template <int DIFF>
constexpr int side_words() { return DIFF == OHX_DIFF_FRESNEL ? 3 * LINES * ROWW : BOFF + 2 * LINES * 16; }
template <int DIFF>
constexpr int list_points() { return CELLS * (CELL + (DIFF == OHX_DIFF_FRESNEL ? 2 : 7 + 7 + 3)); }

template <int DIFF>
struct Smem32 {
    unsigned f[2][2][side_words<DIFF>()];   // [buffer][rows V, columns U]: (re, im) 16-bit pairs
    double c[DIFF == OHX_DIFF_RS ? 7 : 5][list_points<DIFF>()];
    unsigned box[list_points<DIFF>()];  // rows [b0, b1), columns [b2, b3) of the tile, byte k = bk
    int cnt[CELLS][3];                  // [cell][rank class]
    int bat[CELLS][3];                  // [group][rank class]: batches
    int left[2];                        // pairs, box edge lines of pairs left to the per-pixel kernel
};
using SmemF = Smem32<OHX_DIFF_FRESNEL>;
using SmemR = Smem32<OHX_DIFF_RS>;

__device__ inline bf16x2 pack16(float re, float im) { return bf16x2{(__bf16)re, (__bf16)im}; }
// NP parts of one factor, `plane` dwords apart; the remainders are exact
template <int NP, class Smem>
__device__ inline void put(Smem& sm, unsigned at, int plane, float re, float im)
{
    // (-1, 0) and (0, -1) from registers: as an inline constant the dot
    // instruction takes -1.0 for the other half
    unsigned m_re = 0x0000bf80u, m_im = 0xbf800000u;
    asm("" : "+s"(m_re), "+s"(m_im));
    const bf16x2 sub_re = __builtin_bit_cast(bf16x2, m_re), sub_im = __builtin_bit_cast(bf16x2, m_im);
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        const bf16x2 w = pack16(re, im);
        (&sm.f[0][0][0])[at + q * plane] = __builtin_bit_cast(unsigned, w);
        if (q == NP - 1) break;
        re = __builtin_amdgcn_fdot2_f32_bf16(w, sub_re, re, false);   // re - w.re
        im = __builtin_amdgcn_fdot2_f32_bf16(w, sub_im, im, false);
    }
}
// t mod 1 in units of 2^-32 cycles (|t| < 2^19), rounded: the low word of the
// sum with a number whose last place is that unit
__device__ inline unsigned cycles32(double t) { return (unsigned)__double2loint(t + 1572864.0); }
// the same as revolutions within half a cycle
__device__ inline float revolutions(unsigned c) { return (float)(int)c * 2.3283064365386963e-10f; }

// Fresnel factors of a batch: thread = one of its 16 points and every 32nd row
// and column, generated in 11 pieces: per side a setup, then factor by factor
// the value of one beside the stores of the last (two independent chains).
// Phase, first and second difference as 32-bit fractions of a cycle, whose
// wrap-around is the reduction mod 1: two integer adds per factor.  Each is off
// by at most 2^-33 cycles, the last phase by less than 1e-9.
template <int R>
struct Gen;
template <>
struct Gen<1> {
    static constexpr int PIECES = 11;
    unsigned at;           // this thread's first row entry in the target buffer (columns: side_words further)
    int j, grp;            // listed point, thread group
    float sg;
    int x0, y0;
    unsigned ph, d1, d2, lo, num;   // running phase and differences; box interval [lo, lo + num)
    float amp, c, s;
};
template <bool ROWS>
__device__ inline void fresnel_setup(Gen<1>& t, SmemF& sm, const Geometry& g)
{
    constexpr int NG = NTF / 16;
    const double q = sm.c[F_Q][t.j];
    const double st = ROWS ? -(NG * g.pp_y) : NG * g.pp_x;
    const double d = ROWS ? pix_y(g, t.y0 + t.grp) - sm.c[F_PY][t.j] : pix_x(g, t.x0 + t.grp) - sm.c[F_PX][t.j];
    t.ph = cycles32(fresnel_cycles(q, d) + (ROWS ? sm.c[F_CYC][t.j] : 0.0));
    const double d1 = (q * st) * fma(2.0, d, st), d2 = q * (2.0 * st * st);
    t.d1 = cycles32(d1 - rint(d1));
    t.d2 = cycles32(d2 - rint(d2));
    t.amp = ROWS ? t.sg * (float)sm.c[F_AMP][t.j] : 1.f;
    const unsigned box = sm.box[t.j];
    t.lo = (ROWS ? box : box >> 16) & 255u;
    t.num = ((ROWS ? box >> 8 : box >> 24) & 255u) - t.lo;
}
template <int I>
__device__ inline void fresnel_value(Gen<1>& t)
{
    const float f = revolutions(t.ph);
    const float a = (unsigned)(t.grp + NTF / 16 * I) - t.lo < t.num ? t.amp : 0.f;
    t.c = a * cos_rev(f);
    t.s = a * sin_rev(f);
    t.ph += t.d1;
    t.d1 += t.d2;
}
template <bool ROWS, int I>
__device__ inline void fresnel_store(const Gen<1>& t, SmemF& sm, float c, float s)
{
    put<3>(sm, t.at + (ROWS ? 0 : side_words<OHX_DIFF_FRESNEL>()) + NTF / 16 * I * ROWW, LINES * ROWW, c, s);
}
template <int K>
__device__ inline void gen_piece(Gen<1>& t, SmemF& sm, const Geometry& g)
{
    const float c = t.c, s = t.s;
    if constexpr (K == 0) fresnel_setup<true>(t, sm, g);
    if constexpr (K == 5) fresnel_setup<false>(t, sm, g);
    if constexpr (K >= 1 && K <= 4) fresnel_value<K - 1>(t);
    if constexpr (K >= 6 && K <= 9) fresnel_value<K - 6>(t);
    if constexpr (K >= 2 && K <= 5) fresnel_store<true, K - 2>(t, sm, c, s);
    if constexpr (K >= 7 && K <= 10) fresnel_store<false, K - 7>(t, sm, c, s);
}

// RS factors of a batch: thread = one of its points and every 64th (rank 4: 128th)
// row and column.  The phase to e^2 in FP64, the terms from e^3 on (below a
// tenth of a cycle) in FP32.
// Rank 2 takes e^{j theta} = (1 - b^2 Em^2 / 6)(1 - bm^2 E^2 / 6) + j theta (bm, Em
// the largest |b| and |E| on the tile), which is within theta_m^2 / 6 where 1 + j
// theta is off by theta_m^2 / 2: R_MINIMAX holds the coefficients of e^2 (low
// float, for columns) and E^2 (high, for rows), zero for the other ranks.
struct RsFactor {
    float e, bf, ur, ui;
};
__device__ inline double rs_minimax(const Geometry& g, const double* cc)
{
    const double um = (GW / 2) * g.pp_x, vm = (GHF / 2) * g.pp_y, h = 0.25 * TWO_PI * cc[R_RHO];
    const double em = h * um * (fabs(cc[R_G2X]) + um) * cc[R_IR], Em = h * vm * (fabs(cc[R_G2Y]) + vm) * cc[R_IR];
    return __hiloint2double(__float_as_int((float)(em * em * (1.0 / 6.0))), __float_as_int((float)(Em * Em * (1.0 / 6.0))));
}
struct RsPoint {
    double g2, ir, rho, mm, cyc;
    unsigned box;
    float amp;
};
template <bool ROWS>
__device__ inline void rs_load(RsPoint& q, const SmemR& sm, int j, float sg)
{
    if (ROWS) {
        q.box = sm.box[j];
        q.rho = sm.c[R_RHO][j];
        q.ir = sm.c[R_IR][j];
        q.mm = sm.c[R_MINIMAX][j];
        q.cyc = sm.c[R_CYC][j];
        q.amp = sg * (float)sm.c[R_AMP][j];
    }
    q.g2 = sm.c[ROWS ? R_G2Y : R_G2X][j];
}
__device__ inline RsFactor rs_factor(const RsPoint& q, const Geometry& g, bool rows, int k0)
{
    const unsigned lo = (rows ? q.box : q.box >> 16) & 255u, num = ((rows ? q.box >> 8 : q.box >> 24) & 255u) - lo;
    const double d = (double)(k0 - 64) * (rows ? -g.pp_y : g.pp_x);   // from the tile's centre
    const double e = d * (q.g2 + d) * q.ir;
    const float ef = (float)e, rf = (float)q.rho;
    const float f = fmaf(rf * (ef * ef * ef), fmaf(ef, -5.f / 128.f, 1.f / 16.f),
                         revolutions(cycles32(fma(q.rho, e * fma(e, -0.125, 0.5), rows ? q.cyc : 0.0))));
    const float km = __int_as_float(rows ? __double2hiint(q.mm) : __double2loint(q.mm));
    float a = pure_amp<float>(ef) * fmaf(-km * ef, ef, 1.f);
    if (rows) a *= q.amp;
    a = (unsigned)k0 - lo < num ? a : 0.f;
    return RsFactor{ef, (float)(-0.25 * TWO_PI) * rf, a * cos_rev(f), a * sin_rev(f)};
}
// in 8 pieces, per factor its value, then its stores: two rows and two columns,
// rank 4 (two pieces of stores) a row and a column
template <int R>
struct GenRs {
    static constexpr int PIECES = 8;
    unsigned at, bt;       // this thread's first row in the target buffer: steps A and B (second: ^ 8)
    int j, grp;
    float sg;
    int x0, y0;
    RsFactor r;
    RsPoint q;
};
template <>
struct Gen<2> : GenRs<2> {};
template <>
struct Gen<3> : GenRs<3> {};
template <>
struct Gen<4> : GenRs<4> {};
template <int K, int R>
__device__ inline void gen_piece(GenRs<R>& t, SmemR& sm, const Geometry& g)
{
    constexpr int NG = NTF / batch_points<R>(), i = R == 4 ? 0 : (K & 3) / 2;
    constexpr bool rows = K < 4, value = R == 4 ? K % 4 == 0 : K % 2 == 0;
    if constexpr (K == 0) rs_load<true>(t.q, sm, t.j, t.sg);
    if constexpr (value) t.r = rs_factor(t.q, g, rows, t.grp + NG * i);
    if constexpr (K == 3) rs_load<false>(t.q, sm, t.j, t.sg);
    if constexpr (!value && !(R == 4 && K % 4 == 3)) {
        constexpr int side = rows ? 0 : side_words<OHX_DIFF_RS>();
        constexpr int oa = side + NG * i * 8, ob = side + NG * i * 16;
        rs_ranks<float>(rows, R, t.r.e, t.r.bf, t.r.ur, t.r.ui, [&](int k, float re, float im) {
            if (R != 4 && k == 0) put<3>(sm, t.at + oa, LINES * 8, re, im);
            if (R != 4 && k == 1) put<2>(sm, t.bt + ob, LINES * 16, re, im);
            if (R != 4 && k == 2) put<2>(sm, (t.bt ^ 8u) + ob, LINES * 16, re, im);
            if (R == 4 && K % 4 == 1 && k < 2) put<3>(sm, t.at + oa + 4 * k, LINES * 8, re, im);
            if (R == 4 && K % 4 == 2 && k >= 2) put<2>(sm, t.bt + ob + 4 * (k - 2), LINES * 16, re, im);
        });
    }
}

// whole batch, not interleaved
template <int R, int K = 0, class Smem>
__device__ inline void gen_all(Gen<R>& t, Smem& sm, const Geometry& g)
{
    if constexpr (K < Gen<R>::PIECES) {
        gen_piece<K>(t, sm, g);
        gen_all<R, K + 1>(t, sm, g);
    }
}

struct Acc32 {
    f32x16 a[2][2];        // [32-column block][re, im]; rows 8 (i >> 2) + 4 (lane >> 5) + (i & 3)
    double d[2][2][16];
};

// The products of a batch.  A K step takes the six products of parts down to
// 2^-16 of the term (six), or the three down to 2^-8.  K entries alternate the
// real and imaginary part of U; V enters as (Re V, -Im V) for the Re block and
// (Im V, Re V) for the Im block (one row block against two column blocks).
struct Pair {
    u32x4 a, b;
};
struct Ops {
    unsigned av, au;           // this lane's row / first column in the buffer (words of sm.f), Fresnel, RS step A
    unsigned bv, bu;           // RS: first step B (second: ^ 8)
    Pair z, y, x, f;           // U parts 0, 1, 2 (two column blocks); the forms of one V part
    u32x4 v;
};
template <class Smem>
__device__ inline u32x4 ld16(const Smem& sm, unsigned at)
{
    return *reinterpret_cast<const u32x4*>(&(&sm.f[0][0][0])[at]);
}
// part q of step ks: Fresnel 0, 1; RS 0: A, 1, 2: B
template <int R, class Smem>
__device__ inline u32x4 ld_row(const Smem& sm, const Ops& o, int ks, int q)
{
    if (R == 1) return ld16(sm, o.av + ks * 8 + q * (LINES * ROWW));
    if (ks == 0) return ld16(sm, o.av + q * (LINES * 8));
    return ld16(sm, (ks == 1 ? o.bv : o.bv ^ 8u) + q * (LINES * 16));
}
template <int R, class Smem>
__device__ inline Pair ld_col(const Smem& sm, const Ops& o, int ks, int q)
{
    const unsigned p = R == 1 ? o.au + ks * 8 + q * (LINES * ROWW)
                       : ks == 0 ? o.au + q * (LINES * 8)
                                 : (ks == 1 ? o.bu : o.bu ^ 8u) + q * (LINES * 16);
    return Pair{ld16(sm, p), ld16(sm, p + 32 * (R == 1 ? ROWW : ks == 0 ? 8 : 16))};
}
__device__ inline Pair forms(u32x4 v)
{
    Pair r;
    r.a = v ^ 0x80000000u;
#pragma unroll
    for (int i = 0; i < 4; ++i) r.b[i] = __builtin_amdgcn_alignbit(v[i], v[i], 16);
    return r;
}
__device__ inline f32x16 mf(u32x4 a, u32x4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                   0);
}
__device__ inline void prod(Acc32& acc, const Pair& v, const Pair& u)
{
    acc.a[0][0] = mf(v.a, u.a, acc.a[0][0]);
    acc.a[1][0] = mf(v.a, u.b, acc.a[1][0]);
    acc.a[0][1] = mf(v.b, u.a, acc.a[0][1]);
    acc.a[1][1] = mf(v.b, u.b, acc.a[1][1]);
}

// The interleaved form: slot S holds product S of the batch (Fresnel: six of
// either K step; RS: six of step A, three of each step B), the operand reads due a
// slot before their use, and a piece of the next batch's generation, fenced so
// that the pieces stay where the matrix core is busy.  Before the last slot
// comes the batch's barrier (its operands are in registers by then) and the
// next batch's first operands are read.
template <int R, int S, class Smem>
__device__ inline void slot(Ops& o, int flip, Acc32& acc, Gen<R>& gen, Smem& sm,
                            const Geometry& g)
{
    constexpr int NS = R == 1 ? 12 : R == 3 ? 12 : 9, ks = R == 1 ? S / 6 : S < 6 ? 0 : 1 + (S - 6) / 3;
    // position within a six-product step, or 6 + that within a three-product one
    constexpr int t = (R > 1 && ks > 0) ? 6 + (S - 6) % 3 : S % 6;
    constexpr bool last = S == NS - 1;
    if constexpr (last) {
        __syncthreads();
        o.av += flip;
        o.au += flip;
        if (R > 1) {
            o.bv += flip;
            o.bu += flip;
        }
    }
    if constexpr (t == 0) {
        o.f = forms(o.v);
        o.v = ld_row<R>(sm, o, ks, 1);
        prod(acc, o.f, o.z);            // v2 u0
    } else if constexpr (t == 1) {
        o.f = forms(o.v);
        o.y = ld_col<R>(sm, o, ks, 1);
        o.v = ld_row<R>(sm, o, ks, 0);
        prod(acc, o.f, o.z);            // v1 u0
    } else if constexpr (t == 2) {
        prod(acc, o.f, o.y);            // v1 u1
    } else if constexpr (t == 3) {
        o.f = forms(o.v);
        prod(acc, o.f, o.z);            // v0 u0
    } else if constexpr (t == 4) {
        o.x = ld_col<R>(sm, o, ks, 2);
        prod(acc, o.f, o.y);            // v0 u1
    } else if constexpr (t == 5) {
        // first operands of the next step (of the next batch after the barrier)
        constexpr int nk = last ? 0 : 1;
        o.z = ld_col<R>(sm, o, nk, 0);
        o.v = ld_row<R>(sm, o, nk, (nk == 0 || R == 1) ? 2 : 1);
        prod(acc, o.f, o.x);            // v0 u2
    } else if constexpr (t == 6) {
        o.f = forms(o.v);
        o.y = ld_col<R>(sm, o, ks, 1);
        o.v = ld_row<R>(sm, o, ks, 0);
        prod(acc, o.f, o.z);            // v1 u0
    } else if constexpr (t == 7) {
        o.f = forms(o.v);
        prod(acc, o.f, o.z);            // v0 u0
    } else {
        constexpr int nk = last ? 0 : ks + 1;
        o.z = ld_col<R>(sm, o, nk, 0);
        o.v = ld_row<R>(sm, o, nk, nk == 0 ? 2 : 1);
        prod(acc, o.f, o.y);            // v0 u1
    }
    if constexpr (S < Gen<R>::PIECES) gen_piece<S>(gen, sm, g);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!last) slot<R, S + 1>(o, flip, acc, gen, sm, g);
}

// The group's `count` batches of rank R, listed from point j0 on.
template <int R, class Smem>
__device__ inline void batches(Smem& sm, const Geometry& g, Acc32& acc, int j0, int count, float sg, int x0, int y0,
                               int wave, int tid)
{
    constexpr int UN = batch_points<R>(), AW = R == 1 ? ROWW : 8;   // dwords of a line of step A
    constexpr int BUF = (int)(sizeof(sm.f[0]) / sizeof(unsigned));
    if (count == 0) return;
    const int lane = tid & 63, p0 = tid & (UN - 1), grp = tid / UN;
    constexpr int side = side_words<R == 1 ? OHX_DIFF_FRESNEL : OHX_DIFF_RS>();
    const int row = (wave >> 1) * 32 + (lane & 31), col = (wave & 1) * 64 + (lane & 31), h4 = (lane >> 5) * 4;
    auto half = [](int line) { return (line >> 2 & 1) * 8; };
    Gen<R> gen;
    Ops o;
    gen.at = grp * AW + p0;
    o.av = row * AW + h4;
    o.au = side + col * AW + h4;
    if constexpr (R > 1) {   // sm.f and BOFF are whole lines: ^ 8 is the other half
        gen.bt = BOFF + grp * 16 + half(grp) + p0;
        o.bv = BOFF + row * 16 + half(row) + h4;
        o.bu = side + BOFF + col * 16 + half(col) + h4;
    }
    gen.grp = grp;
    gen.sg = sg;
    gen.x0 = x0;
    gen.y0 = y0;
    gen.j = j0 + p0;
    gen_all(gen, sm, g);
    __syncthreads();
    o.z = ld_col<R>(sm, o, 0, 0);
    o.v = ld_row<R>(sm, o, 0, 2);
    int flip = BUF;
#pragma unroll 1
    for (int b = 1; b <= count; ++b) {
        // past the last batch the generation repeats it into the unused buffer
        gen.j = j0 + min(b, count - 1) * UN + p0;
        gen.at += flip;
        if constexpr (R > 1) gen.bt += flip;
        slot<R, 0>(o, flip, acc, gen, sm, g);
        flip = -flip;
    }
    __syncthreads();
}

// Adds points [p_begin, p_end) of s to the 128 x 128 tile `tile` of field (or
// stores the sums to the split's partial plane); returns (in every
// thread) what it left to the per-pixel kernel: LEFT_PAIRS, LEFT_LINES.  The
// FP32 sums of `group` points (direct_chunk) are folded into FP64 at a
// time; groups are counted from point 0 (p_begin is a multiple of the group), so
// that slices and splits sum alike.
template <int DIFF>
__device__ __attribute__((always_inline)) inline unsigned tile_sum(Smem32<DIFF>& sm, const Geometry& g, const PointSoA& s,
                                                               int64_t p_begin, int64_t p_end,
                                                               double2* __restrict__ field, int tile, int tiles_x,
                                                               double2* __restrict__ part, int group)
{
    constexpr int R0 = DIFF == OHX_DIFF_RS ? 2 : 1;   // rank class q has rank R0 + q
    constexpr int NLF = list_points<DIFF>();
    constexpr int NC = DIFF == OHX_DIFF_RS ? 7 : 5, NR = DIFF == OHX_DIFF_RS ? 3 : 1;
    const int cg = group / CELL;   // cells per group
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x0 = (tile % tiles_x) * GW, y0 = (tile / tiles_x) * GHF;
    const int cx1 = min(x0 + GW, g.pn_x), ry1 = min(y0 + GHF, g.pn_y);

    if (tid < 2) sm.left[tid] = 0;
    // list slots not used yet hold finite numbers
    for (int i = tid; i < NC * NLF; i += NTF) (&sm.c[0][0])[i] = 0.0;
    Acc32 acc;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            acc.a[cb][q] = f32x16{};
#pragma unroll
            for (int i = 0; i < 16; ++i) acc.d[cb][q][i] = 0.0;
        }
    __syncthreads();
    bool any = false;   // uniform: some point is listed

    for (int64_t base = p_begin; base < p_end; base += SUP) {
        // ---- classify, list the taken points by group and rank ------------------
        int rank = 0;
        double cc[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) cc[i] = 0.0;
        unsigned bb = 0u;
        const int64_t p = base + wave * PW + lane;
        bool skip = lane >= PW || p >= p_end;
        // RS: the tiles that the masked matrix-core instance took
        if (DIFF == OHX_DIFF_RS && !skip && g.rs_skip_mask)
            skip = rs_mask_bit(g.rs_skip_mask + p * g.rs_mask_words, rs_tile_index(g, x0, y0));
        if (!skip) {
            const int4 b = s.box[p];
            if (b.x < cx1 && b.y > x0 && b.z < ry1 && b.w > y0) {
                const double px = s.px[p], py = s.py[p], z = s.pz[p];
                const double q = DIFF == OHX_DIFF_FRESNEL ? s.q[p] : 0.0;
                int4 ib;
                rank = taken_rank<DIFF, float>(g, px, py, z, q, s.cyc0[p], s.kamp[p], b, x0, y0, ib);
                if (rank == 0) sm.left[0] = 1;
                else if (DIFF == OHX_DIFF_RS && edge_lines(b, ib, x0, cx1, y0, ry1)) sm.left[1] = 1;
                bb = box_bits(make_int4(ib.x, ib.y >= g.pn_x ? INT_MAX : ib.y, ib.z, ib.w >= g.pn_y ? INT_MAX : ib.w), x0, y0);
                point_constants<DIFF>(g, s, p, px, py, z, q, pix_x(g, x0 + GW / 2), pix_y(g, y0 + GHF / 2), cc);
                if constexpr (DIFF == OHX_DIFF_RS)
                    if (rank == 2) cc[R_MINIMAX] = rs_minimax(g, cc);
            }
        }
        int mine = 0;   // place among its cell's points of the same rank
        const int half = lane >= CELL ? 1 : 0, cell = 2 * wave + half;
        const unsigned long long low = (1ull << CELL) - 1;
#pragma unroll
        for (int q = 0; q < NR; ++q) {
            const int r = R0 + q;
            const unsigned long long m = __ballot(rank == r), mc = half ? m & ~low : m & low;
            if (rank == r)
                mine = __builtin_amdgcn_mbcnt_hi((unsigned)(mc >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mc, 0u));
            if (lane == 0) sm.cnt[2 * wave][q] = __popcll(m & low);
            if (lane == 1) sm.cnt[2 * wave + 1][q] = __popcll(m & ~low);
        }
        // points without amplitude in the rest of a last batch
        for (int i = tid; i < NLF; i += NTF) sm.box[i] = 0u;
        __syncthreads();
        // the list: by group, then rank, each padded to whole batches
        int beg = 0, num[3] = {0, 0, 0}, before[3] = {0, 0, 0}, j = 0, cv[3];
#pragma unroll
        for (int q = 0; q < NR; ++q) cv[q] = sm.cnt[lane & (CELLS - 1)][q];
#pragma unroll 1
        for (int w = 0; w < CELLS; ++w) {
#pragma unroll
            for (int q = 0; q < NR; ++q) {
                const int c = __builtin_amdgcn_readlane(cv[q], w);
                num[q] += c;
                if (w < cell) before[q] += c;
            }
            if ((w + 1) % cg != 0) continue;
#pragma unroll
            for (int q = 0; q < NR; ++q) {
                const int r = R0 + q, UN = r == 1 ? 16 : r == 4 ? 4 : 8, nb = (num[q] + UN - 1) / UN;
                if (rank == r && cell <= w && cell > w - cg) j = beg + mine + before[q];
                if (tid == 0) sm.bat[w / cg][q] = nb;
                beg += nb * UN;
                num[q] = before[q] = 0;
            }
        }
        if (rank != 0) {
#pragma unroll
            for (int i = 0; i < NC; ++i) sm.c[i][j] = cc[i];
            sm.box[j] = bb;
        }
        __syncthreads();

        // ---- batches, group by group -------------------------------------------
        int j0 = 0;
#pragma unroll 1
        for (int gr = 0; gr < CELLS / cg; ++gr) {
            int nb[3] = {0, 0, 0};
#pragma unroll
            for (int q = 0; q < NR; ++q) nb[q] = __builtin_amdgcn_readfirstlane(sm.bat[gr][q]);
            if (nb[0] + nb[1] + nb[2] == 0) continue;
            any = true;
            const float sg = (((int)(base / group) + gr) & 1) ? -1.f : 1.f;
            batches<R0>(sm, g, acc, j0, nb[0], sg, x0, y0, wave, tid);
            j0 += nb[0] * batch_points<R0>();
            if constexpr (NR == 3) {
                batches<3>(sm, g, acc, j0, nb[1], sg, x0, y0, wave, tid);
                j0 += nb[1] * batch_points<3>();
                batches<4>(sm, g, acc, j0, nb[2], sg, x0, y0, wave, tid);
                j0 += nb[2] * batch_points<4>();
            }
            // end of the group: FP32 sums into FP64
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc.d[cb][q][i] += (double)(sg * acc.a[cb][q][i]);
                    acc.a[cb][q] = f32x16{};
                }
        }
    }
    if (any || part) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                add_pixel(g, field, part, x0 + (wave & 1) * 64 + cb * 32 + (lane & 31),
                          y0 + (wave >> 1) * 32 + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3), acc.d[cb][0][i],
                          acc.d[cb][1][i]);
    }
    if constexpr (DIFF == OHX_DIFF_FRESNEL) {
        if (sm.left[0]) add_left<float>((int*)&sm.f, g, s, p_begin, p_end, field, part, x0, y0);
    }
    return (unsigned)(sm.left[0] | sm.left[1] << 1);
}

}  // namespace dgemm
