// FP64 direct sums on the FP64 matrix cores (MODE_DOUBLE; direct_gemm.h has
// the method), included by pc_direct.hip.
//
// What bounds it: v_mfma_f64_16x16x4, 74-79 TFLOP/s, 8 flops per point, rank
// and pixel.  The generation of the 192 factors per point and 128 x 64 tile
// comes on top: FP64 MFMA and any VALU instruction do not issue side by side
// (measured: a wave of MFMAs and one of FMAs on a SIMD take the sum of their
// times).
// Fresnel, 20k points at 3840x2160: 48.6 -> 23.3 ms (19.4 of them products); RS,
// 10k points at 1920x1080: 19.1 -> 11.1 ms.  The scalar form read one row factor
// from LDS per 4 FMAs and wave (Fresnel) and spent 23 FP64 instructions per pair
// (RS).  Two workgroups of 4 waves on 128 x 64 pixels per CU, 128 registers of sums a
// lane: while one generates, the other multiplies.  (One of 8 waves on 128 x 128
// would hold the same sums and generate a third less, without a second workgroup to
// fill its barriers; not measured.)
#pragma once

namespace dgemm {

// points per chunk: one per thread, listed in one go (120: clouds near the hologram,
// where most points miss a tile, 20k at 1 to 4 mm on 1920x1080: Fresnel 361 us, now 247;
// far ones 1 % slower)
constexpr int CH64 = 240;
constexpr int SLOTS = 8;                // K slots (two points of one rank) per batch
constexpr int ROWD = SLOTS * 4 + 2;     // padded row of factors: 272 bytes, at which the operand reads do not conflict
constexpr int NLIST = 256;              // listed points of a chunk, each rank's list padded to whole units

struct Smem64 {
    double v[64][ROWD], u[GW][ROWD];    // slot s, point i of it: re at s * 4 + i, im at s * 4 + 2 + i
    double2 tab[NTAB];                  // (cos, sin)(2 pi i / NTAB)
    double off[2][GW];                  // RS: each column's, row's distance from the tile's centre
    double c[6][NLIST];
    unsigned box[NLIST];                // rows [b0, b1), columns [b2, b3) of the tile, byte k = bk
    int cnt[2][NT / 64][Kind<double>::RMAX + 1];   // [chunk parity][wave][rank]
    int left[2];                        // pairs, box edge lines of pairs left to the per-pixel kernel
};

// (cos, sin)(2 pi (a b + c) / NTAB), the product unrounded, c in [0, NTAB] (none: 0).
// The nearest whole number of steps is what the sum with 1.5 2^52 keeps, in its low
// word the table's index (reduced by a floor first, with the index converted: Fresnel
// 23.5 ms at 20k points, 3840x2160, now 23.3).
template <bool C>
__device__ inline void cis(double a, double b, double c, const double2* tab, double& cs, double& sn)
{
    constexpr double whole = 6755399441055744.0;
    const double s = fma(a, b, whole);
    int i = __double2loint(s);
    double r = fma(a, b, whole - s);
    if (C) {
        r += c;
        const double s1 = r + whole;
        i += __double2loint(s1);
        r -= s1 - whole;
    }
    sincos_step(i, r * (TWO_PI / NTAB), tab, sn, cs);
}

// Fresnel factors of one batch (listed points j0 .. j0 + n - 1): thread = one
// point and every 16th column and row, each factor from its own phase.  (Factors
// advanced by rotations, 20k points at 3840x2160, 22.9 ms against 23.3: but their
// angles are rounded at the size of a step's phase, tens of cycles for a point
// near the hologram, which left the field off by 1.5e-13 to 3.5e-13 at all
// depths from 1 mm; by 6e-16 (1 mm) to 1.6e-13 (0.3 m) with phases of their own.)
__device__ inline void gen_fresnel(Smem64& sm, const Geometry& g, int j0, int n, int tid, int x0, int y0)
{
    constexpr int PB = 2 * SLOTS, NG = NT / PB;
    const int p = tid & (PB - 1), grp = tid / PB;
    if (p >= n) return;
    const int j = j0 + p, at = (p >> 1) * 4 + (p & 1);
    const unsigned box = sm.box[j];
    const double q = sm.c[F_Q][j] * NTAB;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        const bool rows = side == 1;
        const unsigned lo = (rows ? box : box >> 16) & 255u, hi = (rows ? box >> 8 : box >> 24) & 255u;
        const double at0 = sm.c[rows ? F_PY : F_PX][j], cyc = sm.c[F_CYC][j] * NTAB, amp = rows ? sm.c[F_AMP][j] : 1.0;
        double* dst = (rows ? sm.v[grp] : sm.u[grp]) + at;
#pragma unroll
        for (int i = 0; i < (rows ? 64 : GW) / NG; ++i) {
            const unsigned k = grp + NG * i;
            const double d = (rows ? pix_y(g, y0 + k) : pix_x(g, x0 + k)) - at0;
            double c, s;
            if (rows) cis<true>(q * d, d, cyc, sm.tab, c, s);
            else cis<false>(q * d, d, 0.0, sm.tab, c, s);
            const double a = k >= lo && k < hi ? amp : 0.0;
            dst[NG * i * ROWD] = a * c;
            dst[NG * i * ROWD + 2] = a * s;
        }
    }
}

// RS factors of one batch (listed points j0 .. j0 + m - 1 of rank R, unit u into
// slots u R .. u R + R - 1): thread = one of n >= m points (n a power of two)
// and every (NT / n)-th column and row.
__device__ inline void gen_rs(Smem64& sm, int j0, int m, int n, int R, int tid)
{
    const int p = tid & (n - 1), grp = tid / n, NG = NT / n;
    if (p >= m) return;
    const int j = j0 + p, at = (p >> 1) * R * 4 + (p & 1);
    const unsigned box = sm.box[j];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        const bool rows = side == 1;
        const unsigned lo = (rows ? box : box >> 16) & 255u, hi = (rows ? box >> 8 : box >> 24) & 255u;
        const double g2 = sm.c[rows ? R_G2Y : R_G2X][j];
        const double cyc = sm.c[R_CYC][j] * NTAB, amp = rows ? sm.c[R_AMP][j] : 1.0;
        const double ir = sm.c[R_IR][j], rho = sm.c[R_RHO][j], steps = rho * NTAB;
#pragma unroll 1
        for (int k0 = grp; k0 < (rows ? 64 : GW); k0 += NG) {
            const double d = sm.off[side][k0];
            const double e = d * (g2 + d) * ir;
            // sqrt(1 + e) - 1
            const double t =
                e * fma(e, fma(e, fma(e, fma(e, fma(e, -21.0 / 1024.0, 7.0 / 256.0), -5.0 / 128.0), 1.0 / 16.0), -0.125),
                        0.5);
            double c, s;
            if (rows) cis<true>(steps, t, cyc, sm.tab, c, s);
            else cis<false>(steps, t, 0.0, sm.tab, c, s);
            double a = amp * pure_amp<double>(e);
            a = ((unsigned)k0 >= lo && (unsigned)k0 < hi) ? a : 0.0;
            double* dst = (rows ? sm.v[k0] : sm.u[k0]) + at;
            rs_ranks<double>(rows, R, e, -0.25 * TWO_PI * rho, a * c, a * s, [&](int k, double re, double im) {
                dst[k * 4] = re;
                dst[k * 4 + 2] = im;
            });
        }
    }
}

struct Acc64 {
    f64x4 a[2][4][2];      // [16-row block][16-column block][re, im]; rows 4 i + (lane >> 4)
};

// The products of one batch.  A lane's K index: slot half, t = real or imaginary
// part of V; the Re block's column operand is (Re U, -Im U), the Im block's (Im
// U, Re U).
__device__ inline void multiply(const Smem64& sm, Acc64& acc, int nslots, int rw, int cw, int lane)
{
    const int half = lane >> 5, t = (lane >> 4) & 1, l = lane & 15;
    const unsigned sgn = t ? 0x80000000u : 0u;
    for (int s2 = 0; s2 < nslots; s2 += 2) {
        // an odd batch's last half step: the second lane half multiplies the
        // last slot's (finite) columns by zero rows
        const bool dead = s2 + half >= nslots;
        const int s = dead ? nslots - 1 : s2 + half;
        double2 a[2];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            a[rb] = *reinterpret_cast<const double2*>(&sm.v[rw * 32 + rb * 16 + l][s * 4 + t * 2]);
            if (dead) a[rb] = make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const double* r = &sm.u[cw * 64 + cb * 16 + l][s * 4];
            const double2 own = *reinterpret_cast<const double2*>(r + t * 2);
            const double2 oth = *reinterpret_cast<const double2*>(r + (t ^ 1) * 2);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const double o = i ? own.y : own.x, h = i ? oth.y : oth.x;
                const double re = __hiloint2double((int)((unsigned)__double2hiint(o) ^ sgn), __double2loint(o));
#pragma unroll
                for (int rb = 0; rb < 2; ++rb) {
                    const double av = i ? a[rb].y : a[rb].x;
                    acc.a[rb][cb][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, re, acc.a[rb][cb][0], 0, 0, 0);
                    acc.a[rb][cb][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, h, acc.a[rb][cb][1], 0, 0, 0);
                }
            }
        }
    }
}

// Adds points [p_begin, p_end) of s to the 128 x 64 tile `tile` of field (or
// stores the sums to the split's partial plane); returns (in every
// thread) what it left to the per-pixel kernel: LEFT_PAIRS, LEFT_LINES.
template <int DIFF>
__device__ __attribute__((always_inline)) inline unsigned tile_sum(Smem64& sm, const Geometry& g, const PointSoA& s,
                                                               int64_t p_begin, int64_t p_end,
                                                               double2* __restrict__ field, int tile, int tiles_x,
                                                               double2* __restrict__ part, int = 0)
{
    constexpr int UN = Kind<double>::UNIT, GH = Kind<double>::GH;
    constexpr int RMIN = DIFF == OHX_DIFF_RS ? 2 : 1, RMAX = DIFF == OHX_DIFF_RS ? Kind<double>::RMAX : 1;
    constexpr int NC = DIFF == OHX_DIFF_RS ? 6 : 5;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int x0 = (tile % tiles_x) * GW, y0 = (tile / tiles_x) * GH;
    const int cx1 = min(x0 + GW, g.pn_x), ry1 = min(y0 + GH, g.pn_y);

    for (int i = tid; i < NTAB; i += NT) {
        double sn, cs;
        sincospi(2.0 * i / NTAB, &sn, &cs);
        sm.tab[i] = make_double2(cs, sn);
    }
    if (DIFF == OHX_DIFF_RS) {
        if (tid < GW) sm.off[0][tid] = pix_x(g, x0 + tid) - pix_x(g, x0 + GW / 2);
        if (tid < GH) sm.off[1][tid] = pix_y(g, y0 + tid) - pix_y(g, y0 + GH / 2);
    }
    if (tid < 2) sm.left[tid] = 0;
    Acc64 acc;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) acc.a[rb][cb][0] = acc.a[rb][cb][1] = f64x4{};
    int par = 0;
    __syncthreads();

    bool any = false;   // uniform: some point is listed
    for (int64_t base = p_begin; base < p_end; base += CH64) {
        // ---- classify one point per thread, list the taken ones by rank ------
        int rank = 0;
        double cc[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) cc[i] = 0.0;
        unsigned bb = 0u;
        const int64_t p = base + tid;
        bool skip = tid >= CH64 || p >= p_end;
        // RS: the tiles that the masked matrix-core instance took
        if (DIFF == OHX_DIFF_RS && !skip && g.rs_skip_mask)
            skip = rs_mask_bit(g.rs_skip_mask + p * g.rs_mask_words, rs_tile_index(g, x0, y0));
        if (!skip) {
            const int4 b = s.box[p];
            if (b.x < cx1 && b.y > x0 && b.z < ry1 && b.w > y0) {
                const double px = s.px[p], py = s.py[p], z = s.pz[p];
                const double q = DIFF == OHX_DIFF_FRESNEL ? s.q[p] : 0.0;
                int4 ib;
                rank = taken_rank<DIFF, double>(g, px, py, z, q, s.cyc0[p], s.kamp[p], b, x0, y0, ib);
                if (rank == 0) sm.left[0] = 1;
                else if (DIFF == OHX_DIFF_RS && edge_lines(b, ib, x0, cx1, y0, ry1)) sm.left[1] = 1;
                bb = box_bits(ib, x0, y0);
                point_constants<DIFF>(g, s, p, px, py, z, q, pix_x(g, x0 + GW / 2), pix_y(g, y0 + GH / 2), cc);
            }
        }
        // counts per rank and wave (by chunk parity: a slower wave may still read the
        // last chunk's)
        auto& cnt = sm.cnt[par];
        par ^= 1;
        int mine = 0;   // place among its wave's points of the same rank
#pragma unroll
        for (int r = RMIN; r <= RMAX; ++r) {
            const unsigned long long m = __ballot(rank == r);
            if (rank == r)
                mine = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            if (lane == 0) cnt[wave][r] = __popcll(m);
        }
        __syncthreads();
        int beg = 0;
#pragma unroll
        for (int r = RMIN; r <= RMAX; ++r) {
            int num = 0, before = 0;
#pragma unroll
            for (int w = 0; w < NT / 64; ++w) {
                before += w < wave ? cnt[w][r] : 0;
                num += cnt[w][r];
            }
            const int end = beg + (num + UN - 1) / UN * UN;
            if (rank == r) {
                const int j = beg + mine + before;
#pragma unroll
                for (int i = 0; i < NC; ++i) sm.c[i][j] = cc[i];
                sm.box[j] = bb;
            }
            // the rest of the last unit: points without amplitude
            const int pad = beg + num + tid;
            if (pad < end) {
#pragma unroll
                for (int i = 0; i < NC; ++i) sm.c[i][pad] = 0.0;
                sm.box[pad] = 0u;
            }
            beg = end;
        }
        __syncthreads();

        // ---- batches of up to SLOTS slots of one rank --------------------------
        beg = 0;
#pragma unroll 1
        for (int r = RMIN; r <= RMAX; ++r) {
            const int units =
                (__builtin_amdgcn_readfirstlane(cnt[0][r] + cnt[1][r] + cnt[2][r] + cnt[3][r]) + UN - 1) / UN;
            any |= units > 0;
            const int per = SLOTS / r;
#pragma unroll 1
            for (int u0 = 0; u0 < units; u0 += per) {
                const int nu = min(per, units - u0);
                if constexpr (DIFF == OHX_DIFF_FRESNEL) gen_fresnel(sm, g, beg + u0 * UN, nu * UN, tid, x0, y0);
                else gen_rs(sm, beg + u0 * UN, nu * UN, per * UN, r, tid);
                __syncthreads();
                multiply(sm, acc, nu * r, wave >> 1, wave & 1, lane);
                __syncthreads();
            }
            beg += units * UN;
        }
    }
    const int xw = x0 + (wave & 1) * 64, yw = y0 + (wave >> 1) * 32;
    if (any || part) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int cb = 0; cb < 4; ++cb)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    add_pixel(g, field, part, xw + cb * 16 + (lane & 15), yw + rb * 16 + 4 * i + (lane >> 4),
                              acc.a[rb][cb][0][i], acc.a[rb][cb][1][i]);
    }
    if constexpr (DIFF == OHX_DIFF_FRESNEL) {
        if (sm.left[0]) add_left<double>((int*)&sm.v, g, s, p_begin, p_end, field, part, x0, y0);
    }
    return (unsigned)(sm.left[0] | sm.left[1] << 1);
}

}  // namespace dgemm
