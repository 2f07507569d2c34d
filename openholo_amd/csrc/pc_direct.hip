// Direct point-cloud diffraction sums for gfx950.
//
// Replaces the eight per-pixel kernels of ophgen/src/ophPCKernel.cu:66-872
// (RS / Fresnel x double / single x plain / round-to-zero), whose maths is
// ophGen::RS_Diffraction / Fresnel_Diffraction (ophgen/src/ophGen.cpp:361-514).
//
// Field model (per point p, pixel (x, y), cycles = radians / 2pi):
//   RS:      H += a z / (lambda r^2) * (sin 2pi c - j cos 2pi c),  c = r / lambda
//   Fresnel: H += a / (lambda z)     * (sin 2pi c - j cos 2pi c),  c = z/lambda + rho^2/(2 lambda z)
// over the reference's anti-aliasing mask (integer box of ophGen.cpp:384-407 /
// 467-490, plus the RS per-pixel range test of ophGen.cpp:415-429).
//
// Kernels:
//  * k_pc_prep turns the 56-byte Vertex records into FP64 structure-of-arrays
//    constants, including the exact integer mask box (same FP64 operations,
//    in the same order, as the reference, contraction off) and the per-point
//    phase constant z/lambda reduced mod 1 cycle with an exact remainder.
//  * k_pc_gemm (direct_gemm.h; direct_f64.h, direct_f32.h) takes nearly every
//    (point, tile) pair as matrix products on the FP64 or, split in three
//    parts, the BF16 matrix cores.
//  * k_pc_lines adds the one-pixel edge lines of the RS boxes, where the range
//    test is open.
//  * k_pc_rest evaluates the RS pairs that the products do not take (points near
//    the hologram), pixel by pixel on 64 x 32 tiles (FP64, few of them: 64 x 8, the
//    points shared by 16 waves), one lane per column and 8 rows per lane: FP64 mode
//    every term; FP32 mode (rest_tile) by point class --
//    FAST (whole tile inside the mask, with margin), MASKED (per-pixel mask) or
//    EXACT (FP32 series not accurate enough: FP64 terms) -- with FP32 constants
//    recentred on the tile centre, so that no phase exceeds ~65 cycles:
//    N = r^2 - r_c^2 = (2 dx_c u + u^2) + (2 dy_c v + v^2) = n_x + N_y and the
//    series r - r_c = N/(2 r_c) - N^2/(8 r_c^3), amplitude z/r^2 =
//    (z/r_c^2)(1 - N/r_c^2).  The phase splits into a column part, a row part
//    and the cross term -2 c_2 n_x N_y cycles (c_2 = 1/(8 r_c^3 lambda)), at
//    most MAX_EPS rad, taken as a first-order factor 1 + j eps folded into the
//    column factor per row: 6 FMAs per pair, no v_sin or v_cos.  Pairs with
//    a larger cross term (FASTNS) evaluate the phase per pixel.
//  * The field (interleaved FP64 complex, the reference's Complex<Real>
//    layout) is read-modify-written once per pixel and kernel.
#include <climits>

#include "line_entry.h"
#include "ohx_internal.h"

namespace ohx {

constexpr int TW = 64;            // tile width = lanes of a wave
constexpr int WAVES = 4;
constexpr int RPT = 8;            // rows per lane
constexpr int TH = WAVES * RPT;   // tile height
constexpr int NT = TW * WAVES;    // threads per workgroup
constexpr int PCH = DIRECT_CHUNK / 2; // points per LDS chunk of rest_tile, folded into FP64 per chunk

// rest_tile: FAST: whole tile inside the mask, separable form; MASKED: per-pixel
// mask; EXACT: FP64 terms; FASTNS: whole tile inside the mask, but the
// cross term of the separable form is too large, so the phase is evaluated
// per pixel.
enum { CLS_OUT = 0, CLS_FAST = 1, CLS_MASKED = 2, CLS_EXACT = 3, CLS_FASTNS = 4 };

// Largest cross-term phase (rad) of the separable RS form: e^{j eps} is taken
// as 1 + j eps, which is within eps^2/2 <= 4.5e-8.
constexpr double MAX_EPS = 3e-4;

constexpr double INV_2PI = 0.15915494309189533576888376337251436;
constexpr double TWO_PI = 6.283185307179586476925286766559;
// Largest phase excursion (cycles) over a tile that the FP32 path accepts:
// FP32 rounding then stays below ~4e-6 cycles per term; larger spans (points
// a few mm from the hologram) take the FP64 path.
constexpr double MAX_CYC = 64.0;

// ---------------------------------------------------------------------------
// reference pixel coordinates, ophGen.cpp:413 and :422 (int expression times
// pitch, then added; no contraction)
__device__ inline double pix_x(const Geometry& g, int col)
{
#pragma clang fp contract(off)
    return g.x0 + (double)(col - 1 + g.off_x) * g.pp_x;
}
__device__ inline double pix_y(const Geometry& g, int row)
{
#pragma clang fp contract(off)
    return g.y0 + (double)(g.pn_y - row + g.off_y) * g.pp_y;
}

// RS per-pixel range test, ophGen.cpp:415-429, bit-identical operation order
__device__ inline bool rs_range_ok(double px, double py, double zz, double hxc, double hyc,
                                   double xxx, double yyy)
{
#pragma clang fp contract(off)
    const double sy = sqrt((yyy - py) * (yyy - py) + zz);
    const double sx = sqrt((xxx - px) * (xxx - px) + zz);
    const double rx0 = px + fabs(hxc * sy), rx1 = px - fabs(hxc * sy);
    const double ry0 = py + fabs(hyc * sx), ry1 = py - fabs(hyc * sx);
    return ((xxx < rx0) && (xxx > rx1)) && ((yyy < ry0) && (yyy > ry1));
}

// ---------------------------------------------------------------------------
// per-point constants: Vertex (56 B) -> SoA
// boxsum (optional): adds the number of pixels inside the boxes of this
// launch's points (one atomic per workgroup), for throughput accounting.
__global__ __launch_bounds__(256) void k_pc_prep(const double* __restrict__ vtx, Geometry g, PointSoA s,
                                                 unsigned long long* __restrict__ boxsum)
{
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long area = 0;
    if (i < s.n) {
        const double* v = vtx + 7 * i;
        // genCghPointCloudCPU: scale, then distance (ophPointCloud.cpp:304-306, ophGen.cpp:379)
        const double px = v[0] * g.scale[0];
        const double py = v[1] * g.scale[1];
        const double z = v[2] * g.scale[2] + g.distance;
        const double a = v[3 + g.channel];
        double hx, hy;
        if (g.diff == OHX_DIFF_RS) {
            hx = fabs(g.hx_coef * z);
            hy = fabs(g.hy_coef * z);
        } else {
            const double operand = g.lambda * z;
            hx = fabs(operand / (2 * g.pp_x));
            hy = fabs(operand / (2 * g.pp_y));
        }
        // box bounds, ophGen.cpp:394-407 (x = -ss/2 = g.x0)
        double X0 = floor(((px + hx) - g.x0) / g.pp_x) + 1;       // exclusive upper column
        double X1 = floor(((px - hx) - g.x0) / g.pp_x) + 1;       // inclusive lower column
        double Y0 = g.pn_y - floor(((py - hy) - g.y0) / g.pp_y);  // exclusive upper row
        double Y1 = g.pn_y - floor(((py + hy) - g.y0) / g.pp_y);  // inclusive lower row
        if (X0 > g.pn_x) X0 = g.pn_x;
        if (X1 < 0) X1 = 0;
        if (Y0 > g.pn_y) Y0 = g.pn_y;
        if (Y1 < 0) Y1 = 0;
        int4 b = make_int4(0, 0, 0, 0);
        if (X1 < X0 && Y1 < Y0) b = make_int4((int)X1, (int)X0, (int)Y1, (int)Y0);

        // z / lambda mod 1 with the exact remainder of the division
        const double qz = z / g.lambda;
        const double rem = fma(-qz, g.lambda, z);
        double c = (qz - floor(qz)) + rem * g.inv_lambda;
        if (g.use_phase) c += v[6] * INV_2PI;
        c -= floor(c);

        s.px[i] = px;
        s.py[i] = py;
        s.pz[i] = z;
        s.cyc0[i] = c;
        if (g.diff == OHX_DIFF_RS) {
            s.kamp[i] = a * z / g.lambda;
            s.q[i] = 0.0;
        } else {
            s.kamp[i] = a / (g.lambda * z);
            s.q[i] = 0.5 / (g.lambda * z);
        }
        s.box[i] = b;
        area = (unsigned long long)(b.y - b.x) * (unsigned long long)(b.w - b.z);
    }
    if (boxsum) {   // uniform over the launch
        for (int off = 32; off > 0; off >>= 1) area += __shfl_xor(area, off);
        __shared__ unsigned long long part[4];
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = area;
        __syncthreads();
        if (threadIdx.x == 0) atomicAdd(boxsum, part[0] + part[1] + part[2] + part[3]);
    }
}

// Before a cloud: its box count and the direct kernels' flags of the tiles that
// leave something to the per-pixel kernels: TILE_FLAGS words, tile t at word t
// mod TILE_FLAGS (a shared word only makes a tile look for what it lacks).
__global__ __launch_bounds__(TILE_FLAGS) void k_zero_scratch(unsigned long long* boxsum, unsigned* flags)
{
    if (threadIdx.x == 0) *boxsum = 0ull;
    flags[threadIdx.x] = 0u;
}

// ---------------------------------------------------------------------------
// sin_rev / cos_rev (ohx_internal.h): the FP32 phases (below MAX_CYC + 1
// cycles by the classification) go in unreduced.

// FP64 term (1/j) amp exp(j 2pi c) of one (point, pixel) pair, added to (re, im)
template <int DIFF>
__device__ inline void exact_term(double dx, double dy, double z, double cyc0, double kamp,
                                  double q, double inv_lambda, double& re, double& im)
{
    const double rho2 = dx * dx + dy * dy;
    double cyc, amp;
    if (DIFF == OHX_DIFF_RS) {
        const double r2 = rho2 + z * z;
        const double r = sqrt(r2);
        cyc = cyc0 + (rho2 / (r + z)) * inv_lambda;   // r/lambda = z/lambda + (r-z)/lambda
        amp = kamp / r2;                               // a z / (lambda r^2)
    } else {
        cyc = cyc0 + rho2 * q;                         // z/lambda + rho^2/(2 lambda z)
        amp = kamp;                                    // a / (lambda z)
    }
    cyc -= floor(cyc);
    double sn, cs;
    sincospi(2.0 * cyc, &sn, &cs);
    re += amp * sn;
    im -= amp * cs;
}

// ---------------------------------------------------------------------------
// The sums on the matrix cores (MODE_DOUBLE: every term in FP64; MODE_FLOAT:
// FP32 factors and FP32 sums over a chunk, folded into FP64).
constexpr int NTAB = 256;  // angles of the FP64 sin/cos table

// sin and cos of 2 pi i / NTAB + x, |x| <= pi / NTAB, in FP64: the table's angle
// plus Taylor series of x (dropped terms below 2e-20), combined by angle addition; 13
// FP64 instructions and one LDS read against ~40 for sincospi.
__device__ inline void sincos_step(int i, double x, const double2* __restrict__ tab, double& s, double& c)
{
    const double2 a = tab[i & (NTAB - 1)];   // (cos, sin)(2 pi i / NTAB)
    const double x2 = x * x;
    const double cb = fma(x2, fma(x2, fma(x2, -1.0 / 720.0, 1.0 / 24.0), -0.5), 1.0);
    const double sb = x * fma(x2, fma(x2, fma(x2, -1.0 / 5040.0, 1.0 / 120.0), -1.0 / 6.0), 1.0);
    s = fma(a.y, cb, a.x * sb);
    c = fma(a.x, cb, -(a.y * sb));
}


#include "direct_gemm.h"
#include "direct_f64.h"
#include "direct_f32.h"

// ---------------------------------------------------------------------------
// LDS of one workgroup (one tile): point constants of the current chunk
struct DirectSmem {
    float4 c0[PCH];
    float4 c1[PCH];
    float2 R[WAVES][PCH][RPT];   // row factor B(row) of the separable form
    float Ny[WAVES][PCH][RPT];   // N_y(row)
    float mu[PCH];               // -1 / r_c^2
    int4 box[PCH];
    int cls[PCH];
    int cnt[2][WAVES];
};

// End of a tile: add the lane's RPT pixels into the field.
__device__ inline void store_tile(const Geometry& g, double2* __restrict__ field, int col, int rowb,
                                  const double* accr, const double* acci)
{
    if (col >= g.pn_x) return;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
        const int row = rowb + k;
        if (row < g.pn_y) {
            double2* f = field + (int64_t)row * g.pn_x + col;
            const double2 v = *f;
            *f = make_double2(v.x + accr[k], v.y + acci[k]);
        }
    }
}

// FP64 point data of a slow-list slot (px, py, z, cyc0, kamp) sits in that
// slot's row-table entries of wave 0, which these slots leave unused.
__device__ inline double* slot_fp64(float2* row_entry) { return reinterpret_cast<double*>(row_entry); }

// The matrix product left the pair of a point (box b) and the tile that holds
// pixel (x0, y0)
template <typename T>
__device__ inline bool left_pair(const Geometry& g, double px, double py, double z, double cyc0, double kamp, int4 b,
                                 int x0, int y0)
{
    int4 ib;
    return dgemm::taken_rank<OHX_DIFF_RS, T>(g, px, py, z, 0.0, cyc0, kamp, b, x0 / dgemm::GW * dgemm::GW,
                                      y0 / dgemm::Kind<T>::GH * dgemm::Kind<T>::GH, ib) == 0;
}

// RS in FP32, the pairs that the matrix product leaves (or all): accumulates points
// [p_begin, p_end) of s into one 64 x 32 tile of field.  Always inlined: a real
// call would pin the multi-job kernel at the callee's worst-case register count.
__device__ __attribute__((always_inline)) inline void rest_tile(DirectSmem& sm, const Geometry& g, const PointSoA& s,
                                                                int64_t p_begin, int64_t p_end,
                                                                double2* __restrict__ field, int x0, int y0, bool all)
{
    float4* s_c0 = sm.c0;
    float4* s_c1 = sm.c1;
    auto& s_R = sm.R;
    int4* s_box = sm.box;
    int* s_cls = sm.cls;
    auto& s_cnt = sm.cnt;

    const int tid = threadIdx.x & (NT - 1), lane = tid & 63, wave = tid >> 6;
    const int cx1 = min(x0 + TW, g.pn_x), ry1 = min(y0 + TH, g.pn_y);
    const int col = x0 + lane;
    const int rowb = y0 + wave * RPT;

    // tile centre and this lane's offset from it
    const double xc = pix_x(g, x0 + TW / 2), yc = pix_y(g, y0 + TH / 2);
    const float u = (float)((double)(lane - TW / 2) * g.pp_x);
    const float uu = u * u;
    const double xxx = pix_x(g, col);
    const float umax = (float)(TW / 2) * (float)g.pp_x, vmax = (float)(TH / 2) * (float)g.pp_y;
    // v = y_row - y_c of this wave's rows
    float vr[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) vr[k] = (float)(-(double)(wave * RPT + k - TH / 2) * g.pp_y);

    double accr[RPT], acci[RPT];
#pragma unroll
    for (int k = 0; k < RPT; ++k) accr[k] = acci[k] = 0.0;
    bool touched = false;   // uniform: some pair on this tile

    for (int64_t base = p_begin; base < p_end; base += PCH) {
        // ---- classify and prepare one point per thread --------------------
        int cls = CLS_OUT;
        float4 c0 = make_float4(0, 0, 0, 0), c1 = make_float4(0, 0, 0, 0);
        float mu = 0.f;
        int4 b = make_int4(0, 0, 0, 0);
        double px = 0, py = 0, z = 0, cyc0 = 0, kamp = 0;
        const int64_t p = base + tid;
        // RS: the tiles that the masked matrix-core instance took for this
        // point (its bit in Geometry::rs_skip_mask) are skipped
        bool skip = false;
        if (g.rs_skip_mask && tid < PCH && p < p_end)
            skip = rs_mask_bit(g.rs_skip_mask + p * g.rs_mask_words, rs_tile_index(g, x0, y0));
        if (tid < PCH && p < p_end && !skip) {
            b = s.box[p];
            if (b.x < cx1 && b.y > x0 && b.z < ry1 && b.w > y0 &&
                (all || left_pair<float>(g, s.px[p], s.py[p], s.pz[p], s.cyc0[p], s.kamp[p], b, x0, y0))) {
                const bool full = b.x <= x0 && b.y >= cx1 && b.z <= y0 && b.w >= ry1;
                px = s.px[p];
                py = s.py[p];
                z = s.pz[p];
                cyc0 = s.cyc0[p];
                kamp = s.kamp[p];
                const double dxc = xc - px, dyc = yc - py;
                const double zz = z * z;
                const double rho2 = dxc * dxc + dyc * dyc;
                const double rc2 = rho2 + zz;
                const double rc = sqrt(rc2);
                // bound on |N| = |r^2 - r_c^2| over the tile
                const double nmax = 2.0 * umax * fabs(dxc) + (double)umax * umax +
                                    2.0 * vmax * fabs(dyc) + (double)vmax * vmax;
                const double e = nmax / rc2;
                // third-order phase term e^3 r_c/(16 lambda) and second-order
                // amplitude term e^2 must be negligible; a phase that is not
                // finite is not masked by a zero amplitude
                const bool series_ok = fabs(cyc0) <= 1.0 && e * e * e * rc * g.inv_lambda < 16 * 2e-7 && e * e < 1e-7 &&
                                       nmax * 0.5 * g.inv_lambda / rc <= MAX_CYC;
                if (!series_ok) {
                    cls = CLS_EXACT;
                } else {
                    bool range_ok = false;
                    if (full) {
                        // reference range test holds on the whole tile with margin
                        const double xl = pix_x(g, x0), xh = pix_x(g, cx1 - 1);
                        const double yh = pix_y(g, y0), yl = pix_y(g, ry1 - 1);
                        const double dxmax = fmax(fabs(xl - px), fabs(xh - px));
                        const double dymax = fmax(fabs(yl - py), fabs(yh - py));
                        const double dxmin = (px >= xl && px <= xh) ? 0.0 : fmin(fabs(xl - px), fabs(xh - px));
                        const double dymin = (py >= yl && py <= yh) ? 0.0 : fmin(fabs(yl - py), fabs(yh - py));
                        const double tol = 1e-12;
                        range_ok = g.hx_coef * sqrt(dymin * dymin + zz) - dxmax > tol &&
                                   g.hy_coef * sqrt(dxmin * dxmin + zz) - dymax > tol;
                    }
                    double ph = cyc0 + (rho2 / (rc + z)) * g.inv_lambda;
                    ph -= floor(ph);
                    const double hp = 0.5 * g.inv_lambda / rc;          // 1/(2 r_c lambda)
                    const double c2 = hp / (4.0 * rc2);                  // 1/(8 r_c^3 lambda)
                    const double az = kamp / rc2;                        // a z/(lambda r_c^2)
                    const double m = az / rc2;
                    // cross term -2 c2 N_x N_y of the phase (rad) over the tile
                    const double nxm = 2.0 * umax * fabs(dxc) + (double)umax * umax;
                    const double nym = 2.0 * vmax * fabs(dyc) + (double)vmax * vmax;
                    const bool sep = 2.0 * TWO_PI * c2 * nxm * nym <= MAX_EPS;
                    cls = range_ok ? (sep ? CLS_FAST : CLS_FASTNS) : CLS_MASKED;
                    c0 = make_float4((float)ph, (float)(2.0 * dxc), (float)(-c2), (float)hp);
                    c1 = make_float4((float)(-m), (float)az, (float)(-2.0 * TWO_PI * c2), (float)(2.0 * dyc));
                    mu = (float)(-1.0 / rc2);
                }
            }
        }
        // ---- deterministic compaction (point order) ------------------------
        const unsigned long long bf = __ballot(cls == CLS_FAST);
        const unsigned long long bs = __ballot(cls >= CLS_MASKED);
        if (lane == 0) {
            s_cnt[0][wave] = __popcll(bf);
            s_cnt[1][wave] = __popcll(bs);
        }
        __syncthreads();
        int nF = 0, nS = 0, offF = 0, offS = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            if (w < wave) {
                offF += s_cnt[0][w];
                offS += s_cnt[1][w];
            }
            nF += s_cnt[0][w];
            nS += s_cnt[1][w];
        }
        // the list lengths are workgroup-uniform: scalar loop control below
        nF = __builtin_amdgcn_readfirstlane(nF);
        nS = __builtin_amdgcn_readfirstlane(nS);
        touched |= nF + nS > 0;
        if (cls != CLS_OUT) {
            const unsigned long long m = (cls == CLS_FAST) ? bf : bs;
            const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            const int slot = (cls == CLS_FAST) ? offF + rank : PCH - 1 - (offS + rank);
            s_box[slot] = b;
            if (cls != CLS_EXACT) {
                s_c0[slot] = c0;
                s_c1[slot] = c1;
                sm.mu[slot] = mu;
            }
            if (cls >= CLS_MASKED) {
                s_cls[slot] = cls;
                double* fd = slot_fp64(&s_R[0][slot][0]);
                fd[0] = px;
                fd[1] = py;
                fd[2] = z;
                fd[3] = cyc0;
                fd[4] = kamp;
            }
        }
        __syncthreads();

        // ---- row table: each wave fills its own 8 rows for every listed point
        // N_y = v (2 dy_c + v) for every non-EXACT point, and
        // for the separable list B = (1 + mu N_y) (cos, sin)(2 pi N_y (h + c_z N_y)).
        for (int jj = lane; jj < nF + nS; jj += TW) {
            const int slot = jj < nF ? jj : PCH - 1 - (jj - nF);
            if (jj >= nF && s_cls[slot] == CLS_EXACT) continue;
            const float4 c = s_c0[slot], d = s_c1[slot];
            float2 o[RPT];
            float ny[RPT];
#pragma unroll
            for (int k = 0; k < RPT; ++k) ny[k] = vr[k] * (d.w + vr[k]);
            float4* dn = (float4*)&sm.Ny[wave][slot][0];
            dn[0] = make_float4(ny[0], ny[1], ny[2], ny[3]);
            dn[1] = make_float4(ny[4], ny[5], ny[6], ny[7]);
            if (jj >= nF) continue;
            const float m1 = sm.mu[slot];
#pragma unroll
            for (int k = 0; k < RPT; ++k) {
                const float t = ny[k] * fmaf(c.z, ny[k], c.w);
                const float a = fmaf(m1, ny[k], 1.f);
                o[k] = make_float2(a * cos_rev(t), a * sin_rev(t));
            }
            float4* dst = (float4*)&s_R[wave][slot][0];
#pragma unroll
            for (int i = 0; i < RPT / 2; ++i) dst[i] = make_float4(o[2 * i].x, o[2 * i].y, o[2 * i + 1].x, o[2 * i + 1].y);
        }
        __syncthreads();

        // ---- fast list: whole tile inside the mask, separable form ----------
        // the phase
        // c0 + c_w N + c_z N^2 and amplitude az (1 + mu N), N = n_x + N_y, give
        // A(col) = az (1 + mu n_x) e^{j 2pi (c0 + c_w n_x + c_z n_x^2)} and the
        // tabulated B(row); the cross term 2 c_z n_x N_y enters as
        // B (1 + j eps), eps = k_x N_y (|eps| <= MAX_EPS), and the amplitude's
        // mu^2 n_x N_y is below 1e-7: 6 FMAs per pair, no v_sin/v_cos.
        float pr[RPT], pim[RPT];
#pragma unroll
        for (int k = 0; k < RPT; ++k) pr[k] = pim[k] = 0.f;
        for (int j = 0; j < nF; ++j) {
            // the point's own constants are read first and all reads are
            // issued before any arithmetic, so that the column factor (FP32
            // chain, v_sin, v_cos) waits only for its own constants while the
            // row factors are on their way (3 % faster)
            const float4 c = s_c0[j];
            const float4 d = s_c1[j];
            __builtin_amdgcn_sched_barrier(0);
            const float4* Rp = (const float4*)&s_R[wave][j][0];
            const float4 r0 = Rp[0], r1 = Rp[1], r2 = Rp[2], r3 = Rp[3];
            const float4 n0 = *(const float4*)&sm.Ny[wave][j][0];
            const float4 n1 = *(const float4*)&sm.Ny[wave][j][4];
            __builtin_amdgcn_sched_barrier(0);
            const float Rx[RPT] = {r0.x, r0.z, r1.x, r1.z, r2.x, r2.z, r3.x, r3.z};
            const float Ry[RPT] = {r0.y, r0.w, r1.y, r1.w, r2.y, r2.w, r3.y, r3.w};
            const float Nv[RPT] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
            const float nx = fmaf(c.y, u, uu);
            const float fa = fmaf(fmaf(c.z, nx, c.w), nx, c.x);
            const float am = fmaf(d.x, nx, d.y);
            const float kx = d.z * nx;
            const float sa = am * sin_rev(fa), ca = am * cos_rev(fa);
            // (sa, ca) against B (1 + j eps), eps = k_x N_y, regrouped per row:
            // P = sa + ca eps, Q = ca - sa eps, then pr += P Bx + Q By and
            // pim += Q Bx - P By (6 FMAs per pair)
            const float cak = ca * kx, sak = sa * kx;
#pragma unroll
            for (int k = 0; k < RPT; ++k) {
                const float P = fmaf(cak, Nv[k], sa), Q = fmaf(-sak, Nv[k], ca);
                pr[k] = fmaf(P, Rx[k], fmaf(Q, Ry[k], pr[k]));
                pim[k] = fmaf(Q, Rx[k], fmaf(-P, Ry[k], pim[k]));
            }
        }
        // ---- slow list: per-pixel mask and/or FP64 terms --------------------
        for (int j = 0; j < nS; ++j) {
            const int slot = PCH - 1 - j;
            const int cl = s_cls[slot];
            const int4 bb = s_box[slot];
            const double* fd = slot_fp64(&s_R[0][slot][0]);
            const bool colin = col >= bb.x && col < bb.y;
            if (cl == CLS_FASTNS) {
                // whole tile in the mask, phase per pixel
                const float4 c = s_c0[slot];
                const float4 d = s_c1[slot];
                const float* Ns = &sm.Ny[wave][slot][0];
                const float nx = fmaf(c.y, u, uu);
#pragma unroll
                for (int k = 0; k < RPT; ++k) {
                    const float N = nx + Ns[k];
                    const float f = fmaf(fmaf(c.z, N, c.w), N, c.x);
                    const float amp = fmaf(d.x, N, d.y);
                    pr[k] = fmaf(amp, sin_rev(f), pr[k]);
                    pim[k] = fmaf(amp, cos_rev(f), pim[k]);
                }
            } else if (cl == CLS_MASKED) {
                const float4 c = s_c0[slot];
                const float* Ns = &sm.Ny[wave][slot][0];
                const float4 d = s_c1[slot];
                const double qpx = fd[0], qpy = fd[1], qz = fd[2];
                const double zz = qz * qz;
#pragma unroll
                for (int k = 0; k < RPT; ++k) {
                    const int row = rowb + k;
                    bool in = colin && row >= bb.z && row < bb.w;
                    in = in && rs_range_ok(qpx, qpy, zz, g.hx_coef, g.hy_coef, xxx, pix_y(g, row));
                    const float N = fmaf(c.y, u, uu) + Ns[k];
                    const float f = fmaf(fmaf(c.z, N, c.w), N, c.x);
                    float amp = fmaf(d.x, N, d.y);
                    amp = in ? amp : 0.f;
                    pr[k] = fmaf(amp, sin_rev(f), pr[k]);
                    pim[k] = fmaf(amp, cos_rev(f), pim[k]);
                    __builtin_amdgcn_sched_barrier(0);  // keep one row live at a time
                }
            } else {
                // FP64 terms, one row at a time (a rolled loop keeps the kernel's
                // register count at the fast path's; the row's term is added to
                // its accumulator by selection)
                const double qpx = fd[0], qpy = fd[1], qz = fd[2];
                const double qc = fd[3], qk = fd[4];
                const double zz = qz * qz;
#pragma unroll 1
                for (int k = 0; k < RPT; ++k) {
                    const int row = rowb + k;
                    const double yyy = pix_y(g, row);
                    bool in = colin && row >= bb.z && row < bb.w;
                    in = in && rs_range_ok(qpx, qpy, zz, g.hx_coef, g.hy_coef, xxx, yyy);
                    double re = 0.0, im = 0.0;
                    if (in) exact_term<OHX_DIFF_RS>(xxx - qpx, yyy - qpy, qz, qc, qk, 0.0, g.inv_lambda, re, im);
#pragma unroll
                    for (int kk = 0; kk < RPT; ++kk) {
                        accr[kk] += (kk == k) ? re : 0.0;
                        acci[kk] += (kk == k) ? im : 0.0;
                    }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
            accr[k] += (double)pr[k];
            acci[k] -= (double)pim[k];
        }
        __syncthreads();
    }

    if (touched) store_tile(g, field, col, rowb, accr, acci);
}

struct SplitArgs {
    int tiles;           // tiles per split
    int64_t split_pts;   // points per split
    double2* part;       // (splits - 1) partial planes of pn_x * pn_y pixels
    int chunk;           // points that split_pts is a multiple of (FP32: points per fold)
};

__device__ inline void split_item(const Geometry& g, const PointSoA& s, const SplitArgs& sa, int& tile,
                                  int64_t& p0, int64_t& p1, double2*& part)
{
    const int split = blockIdx.x / sa.tiles;
    tile = blockIdx.x - split * sa.tiles;
    p0 = (int64_t)split * sa.split_pts;
    p1 = min(s.n, p0 + sa.split_pts);
    part = split == 0 ? nullptr : sa.part + (int64_t)(split - 1) * ((int64_t)g.pn_x * g.pn_y);
}

// ---------------------------------------------------------------------------
// The pairs that the matrix products leave (direct_gemm.h), pixel by pixel:
// every term in FP64 under the reference's mask, 64 columns x 8 rows a wave, a lane
// per column.  RG waves take the rows of a tile; near the hologram all points may
// be left, and where tiles are few, SHARES waves share the listed points of a row
// group, and their sums are added in a fixed order.  SHARES = 16 where the hologram
// has fewer tiles of 64 x 32 than two a CU (10k points at 320x180, z 5 to 20 mm: 3.4
// ms against 17.9 with one share; 3k at 640x360: 0.45 against 1.8), else 1 and RG =
// 4 (20k at 1920x1080, 1 to 4 mm: 0.76 ms against 1.16 with 16: more tiles to list,
// and sums to add).
constexpr int XROWS = RPT;
template <int SHARES, int RG>
union ExactSmem {
    struct {
        double d[5][64 * SHARES * RG];   // px, py, z, cyc0, kamp of the listed points of a chunk
        int4 box[64 * SHARES * RG];
        int cnt[SHARES * RG];
    };
    double2 sum[SHARES > 1 ? SHARES / 2 * RG : 1][XROWS][64];
};
inline __host__ __device__ bool few_tiles(const Geometry& g)
{
    return (int64_t)((g.pn_x + TW - 1) / TW) * ((g.pn_y + TH - 1) / TH) < 512;
}

template <int SHARES, int RG>
__device__ __attribute__((always_inline)) inline void exact_tile(ExactSmem<SHARES, RG>& sm, const Geometry& g,
                                                                 const PointSoA& s, int64_t p_begin, int64_t p_end,
                                                                 double2* __restrict__ field, int x0, int y0)
{
    constexpr int W = SHARES * RG, N = 64 * W;   // waves; threads, points per chunk
    const int tid = threadIdx.x & (N - 1), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int share = wave % SHARES, rg = wave / SHARES;
    const int cx1 = min(x0 + 64, g.pn_x), ry1 = min(y0 + RG * XROWS, g.pn_y);
    const int col = x0 + lane, row0 = y0 + rg * XROWS;
    const double xxx = pix_x(g, col);
    double accr[XROWS], acci[XROWS];
#pragma unroll
    for (int k = 0; k < XROWS; ++k) accr[k] = acci[k] = 0.0;
    bool any = false;   // uniform: some pair on this tile

    for (int64_t base = p_begin; base < p_end; base += N) {
        bool ex = false;
        const int64_t p = base + tid;
        int4 b = make_int4(0, 0, 0, 0);
        if (p < p_end) {
            b = s.box[p];
            if (b.x < cx1 && b.y > x0 && b.z < ry1 && b.w > y0)
                ex = left_pair<double>(g, s.px[p], s.py[p], s.pz[p], s.cyc0[p], s.kamp[p], b, x0, y0);
        }
        // listed in point order
        const unsigned long long m = __ballot(ex);
        if (lane == 0) sm.cnt[wave] = __popcll(m);
        __syncthreads();
        int n = 0, at = 0;
        for (int w = 0; w < W; ++w) {
            if (w == wave) at = n;
            n += sm.cnt[w];
        }
        n = __builtin_amdgcn_readfirstlane(n);
        if (ex) {
            const int j =
                at + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            sm.d[0][j] = s.px[p];
            sm.d[1][j] = s.py[p];
            sm.d[2][j] = s.pz[p];
            sm.d[3][j] = s.cyc0[p];
            sm.d[4][j] = s.kamp[p];
            sm.box[j] = b;
        }
        __syncthreads();
        any |= n > 0;
        for (int j = share; j < n; j += SHARES) {
            const int4 bb = sm.box[j];
            const double qpx = sm.d[0][j], qpy = sm.d[1][j], qz = sm.d[2][j];
            const double qc = sm.d[3][j], qk = sm.d[4][j];
            const double zz = qz * qz;
            const bool colin = col >= bb.x && col < bb.y;
#pragma unroll
            for (int k = 0; k < XROWS; ++k) {
                const int row = row0 + k;
                const double yyy = pix_y(g, row);
                bool in = colin && row >= bb.z && row < bb.w;
                in = in && rs_range_ok(qpx, qpy, zz, g.hx_coef, g.hy_coef, xxx, yyy);
                if (in) exact_term<OHX_DIFF_RS>(xxx - qpx, yyy - qpy, qz, qc, qk, 0.0, g.inv_lambda, accr[k], acci[k]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }
    if (!any) return;
    // the upper half of the shares to the lower one, until one is left
#pragma unroll
    for (int half = SHARES / 2; half > 0; half /= 2) {
        if (share >= half && share < 2 * half) {
#pragma unroll
            for (int k = 0; k < XROWS; ++k) sm.sum[rg * (SHARES / 2) + share - half][k][lane] = make_double2(accr[k], acci[k]);
        }
        __syncthreads();
        if (share < half) {
#pragma unroll
            for (int k = 0; k < XROWS; ++k) {
                const double2 v = sm.sum[rg * (SHARES / 2) + share][k][lane];
                accr[k] += v.x;
                acci[k] += v.y;
            }
        }
        __syncthreads();
    }
    if (share == 0) store_tile(g, field, col, row0, accr, acci);
}

// Workgroup = (tile, point split): blockIdx = split * tiles + tile; split 0
// adds into the field, the others store into their partial planes.
template <int DIFF, typename T>
struct GemmSmem {
    using type = dgemm::Smem64;
};
template <int DIFF>
struct GemmSmem<DIFF, float> {
    using type = dgemm::Smem32<DIFF>;
};

// Two waves per SIMD: two 4-wave workgroups (FP64) or one 8-wave one (FP32) per CU.
template <int DIFF, typename T>
__global__ __launch_bounds__(dgemm::Kind<T>::NTH, 512 / dgemm::Kind<T>::NTH) void k_pc_gemm(Geometry g, PointSoA s, double2* __restrict__ field, int tiles_x,
                                                   unsigned* __restrict__ flags, SplitArgs sa)
{
    __shared__ __align__(16) typename GemmSmem<DIFF, T>::type sm;
    int tile;
    int64_t p0, p1;
    double2* part;
    split_item(g, s, sa, tile, p0, p1, part);
    const unsigned left = dgemm::tile_sum<DIFF>(sm, g, s, p0, p1, field, tile, tiles_x, part, sa.chunk);
    if (DIFF == OHX_DIFF_RS && left && threadIdx.x == 0) atomicOr(&flags[tile & (TILE_FLAGS - 1)], left);
}

// RS: the pairs k_pc_gemm left, one workgroup per 64 x 32 (FEW: 64 x 8) tile; returns at
// once where there are none.  In FP32 mode in FP32 where the series holds on the smaller
// tile, otherwise in FP64.
template <typename T, bool FEW>
struct Rest {
    static constexpr int SHARES = FEW ? 16 : 1, RG = FEW ? 1 : WAVES;
    static constexpr int THREADS = 64 * SHARES * RG, ROWS = XROWS * RG;
    using Smem = ExactSmem<SHARES, RG>;
};
template <>
struct Rest<float, false> {
    static constexpr int THREADS = NT, ROWS = TH;
    using Smem = DirectSmem;
};

template <typename T, bool FEW>
__global__ __launch_bounds__((Rest<T, FEW>::THREADS)) void k_pc_rest(Geometry g, PointSoA s, double2* __restrict__ field,
                                                                   int tiles_x, int gemm_tiles_x,
                                                                   const unsigned* __restrict__ flags, bool all)
{
    const int x0 = (blockIdx.x % tiles_x) * TW, y0 = (blockIdx.x / tiles_x) * Rest<T, FEW>::ROWS;
    const int t = (y0 / dgemm::Kind<T>::GH) * gemm_tiles_x + x0 / dgemm::GW;
    if (!all && !(flags[t & (TILE_FLAGS - 1)] & dgemm::LEFT_PAIRS)) return;
    __shared__ typename Rest<T, FEW>::Smem sm;
    if constexpr (dgemm::Kind<T>::f64) exact_tile(sm, g, s, 0, s.n, field, x0, y0);
    else rest_tile(sm, g, s, 0, s.n, field, x0, y0, all);
}

// RS: the box edge lines of the pairs that the matrix product took (inner_box),
// one 64 x 8 strip of pixels per wave, every term in FP64 under the reference's
// mask, summed in the wave's LDS strip in a fixed order.  What it costs is the
// terms, so a line's terms are spread over the lanes: the columns of a row line, the 8 rows
// of the column lines of 8 points.  (Such pairs were evaluated whole, pixel by
// pixel, before: RS in FP64, 4k points, z 0.25 m, 1920 x 1080 at 8 um, where
// the boxes end inside the hologram: 18.4 ms, now 5.7; FP32, 22k points: 12.7 ms,
// now 6.5, of which this kernel 0.6.)
constexpr int LINE_ROWS = 8;
struct LineSmem {
    double2 acc[LINE_ROWS][64];
    int64_t queue[128];   // column lines that wait (line_entry; points from p_begin)
};

template <typename T>
__device__ __attribute__((always_inline)) inline void line_strip(LineSmem& sm, const Geometry& g, const PointSoA& s,
                                                                 int64_t p_begin, int64_t p_end,
                                                                 double2* __restrict__ field, int x0, int y0,
                                                                 unsigned left)
{
    const int lane = threadIdx.x & 63;
    const int x1 = min(x0 + 64, g.pn_x), y1 = min(y0 + LINE_ROWS, g.pn_y), col = x0 + lane;
#pragma unroll
    for (int r = 0; r < LINE_ROWS; ++r) sm.acc[r][lane] = make_double2(0.0, 0.0);
    // LDS handed from lane to lane of one wave
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    wave_sync();
    auto term = [&](int64_t p, double xxx, double yyy, double& re, double& im) {
        const double px = s.px[p], py = s.py[p], z = s.pz[p];
        re = im = 0.0;
        if (rs_range_ok(px, py, z * z, g.hx_coef, g.hy_coef, xxx, yyy))
            exact_term<OHX_DIFF_RS>(xxx - px, yyy - py, z, s.cyc0[p], s.kamp[p], 0.0, g.inv_lambda, re, im);
    };
    // the first n (up to 8) queued column lines: lane = (line, row)
    auto columns = [&](int n) {
        const int i = lane >> 3, row = y0 + (lane & 7);
        double re = 0.0, im = 0.0;
        int c = 0;
        if (i < n) {
            const int64_t e = sm.queue[i], p = p_begin + line_point(e);
            const int4 b = s.box[p];
            c = line_side(e) ? b.y - 1 : b.x;
            if (row >= b.z && row < b.w) term(p, pix_x(g, c), pix_y(g, row), re, im);
        }
        for (int k = 0; k < n; ++k) {   // line by line: the order of the sums is the queue's
            if (i == k) {
                double2& a = sm.acc[lane & 7][c - x0];
                a = make_double2(a.x + re, a.y + im);
            }
            wave_sync();
        }
    };
    int waiting = 0;
    bool any = false;
    for (int64_t base = p_begin; base < p_end; base += 64) {
        const int64_t p = base + lane;
        unsigned m = 0, cut = 0;
        if (p < p_end) {
            const int4 b = s.box[p];
            const bool meets = b.x < x1 && b.y > x0 && b.z < y1 && b.w > y0;
            if (meets && (b.x >= x0 || b.y <= x1 || b.z >= y0 || b.w <= y1) &&
                !(g.rs_skip_mask && rs_mask_bit(g.rs_skip_mask + p * g.rs_mask_words, rs_tile_index(g, x0, y0)))) {
                const double px = s.px[p], py = s.py[p], z = s.pz[p];
                int4 ib;
                if (dgemm::inner_box(g, px, py, z, b, ib) &&
                    !((left & dgemm::LEFT_PAIRS) && left_pair<T>(g, px, py, z, s.cyc0[p], s.kamp[p], b, x0, y0))) {
                    m = dgemm::edge_lines(b, ib, x0, x1, y0, y1);
                    cut = (unsigned)(ib.x - b.x) | (unsigned)(b.y - ib.y) << 1;
                }
            }
        }
        // row lines, without the column lines' pixels
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            unsigned long long todo = __ballot((m >> (2 + side)) & 1u);
            any |= todo != 0;
            while (todo) {
                const int j = __builtin_ctzll(todo);
                todo &= todo - 1;
                const unsigned ct = (unsigned)__shfl((int)cut, j);
                const int4 b = s.box[base + j];
                const int row = side ? b.w - 1 : b.z;
                double re = 0.0, im = 0.0;
                if (col >= b.x + (int)(ct & 1u) && col < b.y - (int)(ct >> 1))
                    term(base + j, pix_x(g, col), pix_y(g, row), re, im);
                double2& a = sm.acc[row - y0][lane];
                a = make_double2(a.x + re, a.y + im);
                wave_sync();
            }
        }
        // column lines wait until there are 8
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const unsigned long long has = __ballot((m >> side) & 1u);
            if ((m >> side) & 1u)
                sm.queue[waiting + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(has >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((unsigned)has, 0u))] =
                    line_entry(p - p_begin, side);
            waiting += __popcll(has);
            any |= has != 0;
            wave_sync();
            while (waiting >= 8) {
                columns(8);
                waiting -= 8;
                // up to 63 are left: move them to the front
                const int64_t e = lane < waiting ? sm.queue[lane + 8] : 0;
                wave_sync();
                if (lane < waiting) sm.queue[lane] = e;
                wave_sync();
            }
        }
    }
    if (waiting) columns(waiting);
    if (!any || col >= g.pn_x) return;
#pragma unroll
    for (int r = 0; r < LINE_ROWS; ++r) {
        const int row = y0 + r;
        if (row < g.pn_y) {
            double2* f = field + (int64_t)row * g.pn_x + col;
            const double2 v = *f, a = sm.acc[r][lane];
            *f = make_double2(v.x + a.x, v.y + a.y);
        }
    }
}

template <typename T>
__global__ __launch_bounds__(NT) void k_pc_lines(Geometry g, PointSoA s, double2* __restrict__ field, int tiles_x,
                                                 int gemm_tiles_x, const unsigned* __restrict__ flags)
{
    const int x0 = (blockIdx.x % tiles_x) * TW, y0 = (blockIdx.x / tiles_x) * TH;
    const int t = (y0 / dgemm::Kind<T>::GH) * gemm_tiles_x + x0 / dgemm::GW;
    const unsigned left = flags[t & (TILE_FLAGS - 1)];
    if (!(left & dgemm::LEFT_LINES)) return;
    __shared__ LineSmem sm[WAVES];
    const int wave = threadIdx.x >> 6;
    line_strip<T>(sm[wave], g, s, 0, s.n, field, x0, y0 + wave * LINE_ROWS, left);
}

// field += partial planes 1..splits-1, in split order (deterministic)
__global__ __launch_bounds__(256) void k_split_reduce(double2* __restrict__ field, const double2* __restrict__ part,
                                                      int64_t npx, int nparts)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < npx; i += stride) {
        double2 f = field[i];
        for (int k = 0; k < nparts; ++k) {
            const double2 q = part[(int64_t)k * npx + i];
            f.x += q.x;
            f.y += q.y;
        }
        field[i] = f;
    }
}

// Persistent multi-job form used by the serving engine, one kernel per formula
// and precision (one for all of them would take the registers of the largest):
// workgroups stride over the (job, tile) items of the table's jobs of that kind
// (item_base counts those); each item adds the job's current point slice [p0,
// p1) into that job's resident field.
template <int DIFF, typename T>
__global__ __launch_bounds__(dgemm::Kind<T>::NTH, 512 / dgemm::Kind<T>::NTH) void k_pc_gemm_jobs(
    DirectJob* __restrict__ jobs, const int* __restrict__ njobs_ptr)
{
    __shared__ __align__(16) typename GemmSmem<DIFF, T>::type sm;
    auto mine = [&](int k) { return jobs[k].g.diff == DIFF && jobs[k].fp64 == (dgemm::Kind<T>::f64 ? 1 : 0); };
    const int njobs = *njobs_ptr;
    int total = 0;
    for (int k = 0; k < njobs; ++k)
        if (mine(k)) total = jobs[k].item_base + jobs[k].tiles;
    for (int item = blockIdx.x; item < total; item += gridDim.x) {
        int j = 0;
        for (int k = 0; k < njobs; ++k)
            if (mine(k) && jobs[k].item_base <= item) j = k;
        DirectJob& jb = jobs[j];
        const unsigned left = dgemm::tile_sum<DIFF>(sm, jb.g, jb.s, jb.p0, jb.p1, jb.field, item - jb.item_base,
                                                    jb.tiles_x, nullptr, jb.chunk);
        if (left && threadIdx.x == 0) atomicOr(&jb.left, (int)left);
        __syncthreads();   // LDS reuse across items
    }
}

// The pairs those left, 64 x 32 (FP64, few tiles: 64 x 8) tiles of the jobs that have any
__global__ __launch_bounds__(NT) void k_pc_rest_jobs(const DirectJob* __restrict__ jobs,
                                                     const int* __restrict__ njobs_ptr)
{
    __shared__ union {
        DirectSmem rs;
        ExactSmem<1, WAVES> exact;
        ExactSmem<WAVES, 1> shared;
    } sm;
    const int njobs = *njobs_ptr;
    int item = blockIdx.x;
    for (int k = 0; k < njobs; ++k) {
        const DirectJob& jb = jobs[k];
        if (!jb.per_pixel && !(jb.left & dgemm::LEFT_PAIRS)) continue;
        const bool few = jb.fp64 && few_tiles(jb.g);
        const int rows = few ? XROWS : TH, xt = (jb.g.pn_x + TW - 1) / TW;
        const int tiles = xt * ((jb.g.pn_y + rows - 1) / rows);
        for (; item < tiles; item += gridDim.x) {
            const int x0 = (item % xt) * TW, y0 = (item / xt) * rows;
            if (few) exact_tile(sm.shared, jb.g, jb.s, jb.p0, jb.p1, jb.field, x0, y0);
            else if (jb.fp64) exact_tile(sm.exact, jb.g, jb.s, jb.p0, jb.p1, jb.field, x0, y0);
            else rest_tile(sm.rs, jb.g, jb.s, jb.p0, jb.p1, jb.field, x0, y0, jb.per_pixel != 0);
            __syncthreads();   // LDS reuse across items
        }
        item -= tiles;
    }
}

__global__ __launch_bounds__(NT) void k_pc_lines_jobs(const DirectJob* __restrict__ jobs,
                                                      const int* __restrict__ njobs_ptr)
{
    __shared__ LineSmem sm[WAVES];
    const int njobs = *njobs_ptr, wave = threadIdx.x >> 6;
    int item = blockIdx.x;
    for (int k = 0; k < njobs; ++k) {
        const DirectJob& jb = jobs[k];
        const unsigned left = (unsigned)jb.left;
        if (!(left & dgemm::LEFT_LINES)) continue;
        const int xt = (jb.g.pn_x + TW - 1) / TW, tiles = xt * ((jb.g.pn_y + TH - 1) / TH);
        for (; item < tiles; item += gridDim.x) {
            const int x0 = (item % xt) * TW, y0 = (item / xt) * TH + wave * LINE_ROWS;
            if (jb.fp64) line_strip<double>(sm[wave], jb.g, jb.s, jb.p0, jb.p1, jb.field, x0, y0, left);
            else line_strip<float>(sm[wave], jb.g, jb.s, jb.p0, jb.p1, jb.field, x0, y0, left);
        }
        item -= tiles;
    }
}

// ---------------------------------------------------------------------------
// FP64 accuracy probe: one thread per listed pixel, Neumaier summation
__device__ inline void neumaier(double& s, double& c, double x)
{
    const double t = s + x;
    if (fabs(s) >= fabs(x)) c += (s - t) + x;
    else c += (x - t) + s;
    s = t;
}

template <int DIFF>
__global__ __launch_bounds__(256) void k_pc_probe(Geometry g, PointSoA s, const int64_t* __restrict__ pix,
                                                  int64_t npix, double2* __restrict__ out)
{
    __shared__ double sd[6][256];
    __shared__ int4 sb[256];
    const int tid = threadIdx.x;
    const int64_t qi = (int64_t)blockIdx.x * 256 + tid;
    const int64_t npx = (int64_t)g.pn_x * g.pn_y;
    int64_t id = (qi < npix) ? pix[qi] : -1;
    const bool valid = id >= 0 && id < npx;
    const int col = valid ? (int)(id % g.pn_x) : 0;
    const int row = valid ? (int)(id / g.pn_x) : 0;
    const double xxx = pix_x(g, col), yyy = pix_y(g, row);
    double sr = 0, cr = 0, si = 0, ci = 0;
    for (int64_t base = 0; base < s.n; base += 256) {
        const int64_t p = base + tid;
        if (p < s.n) {
            sd[0][tid] = s.px[p];
            sd[1][tid] = s.py[p];
            sd[2][tid] = s.pz[p];
            sd[3][tid] = s.cyc0[p];
            sd[4][tid] = s.kamp[p];
            sd[5][tid] = s.q[p];
            sb[tid] = s.box[p];
        }
        __syncthreads();
        const int cnt = (int)min((int64_t)256, s.n - base);
        for (int j = 0; j < cnt; ++j) {
            const int4 b = sb[j];
            bool in = valid && col >= b.x && col < b.y && row >= b.z && row < b.w;
            if (DIFF == OHX_DIFF_RS && in)
                in = rs_range_ok(sd[0][j], sd[1][j], sd[2][j] * sd[2][j], g.hx_coef, g.hy_coef, xxx, yyy);
            if (in) {
                double re = 0, im = 0;
                exact_term<DIFF>(xxx - sd[0][j], yyy - sd[1][j], sd[2][j], sd[3][j], sd[4][j], sd[5][j],
                                 g.inv_lambda, re, im);
                neumaier(sr, cr, re);
                neumaier(si, ci, im);
            }
        }
        __syncthreads();
    }
    if (qi < npix) {
        const double nan = __builtin_nan("");
        out[qi] = valid ? make_double2(sr + cr, si + ci) : make_double2(nan, nan);
    }
}

// ---------------------------------------------------------------------------
int launch_prep_on(hipStream_t stream, const void* d_vertices, const Geometry& g, const PointSoA& soa,
                   unsigned long long* boxsum, unsigned* flags)
{
    const unsigned grid = (unsigned)((soa.n + 255) / 256);
    if (flags) hipLaunchKernelGGL(k_zero_scratch, dim3(1), dim3(TILE_FLAGS), 0, stream, boxsum, flags);
    hipLaunchKernelGGL(k_pc_prep, dim3(grid), dim3(256), 0, stream, (const double*)d_vertices, g, soa, boxsum);
    return hipGetLastError() == hipSuccess ? OHX_OK : OHX_ERR_DEVICE;
}

int launch_prep(ohx_ctx* ctx, const void* d_vertices, const Geometry& g, const PointSoA& soa,
                unsigned long long* boxsum, unsigned* flags)
{
    if (launch_prep_on(ctx->stream, d_vertices, g, soa, boxsum, flags) != OHX_OK)
        return check_hip(ctx, hipErrorLaunchFailure, "k_pc_prep");
    return OHX_OK;
}

// Workgroups the device holds at once for kernel k (occupancy x CUs).
static int resident_slots(ohx_ctx* ctx, const void* k, int threads)
{
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, threads, 0) != hipSuccess || per_cu < 1) per_cu = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess || cus < 1)
        cus = 1;
    return per_cu * cus;
}

// Point splits of the matrix-product kernels by their modelled time, in units of 0.1
// us: a point on a tile (FP32: with its share of a group's start and fold, 4 us for
// Fresnel, 10 for RS), a tile's start and end, and each further partial plane
// (written and read, 32 B a pixel at ~4 TB/s) with one more launch.  Split boundaries
// are multiples of `chunk` points, planes stay under 2 GiB.
constexpr int MAX_SPLITS = 64;
struct GemmCost {
    double point, tile;
};
static GemmCost gemm_cost(bool rs, bool fp64, int chunk)
{
    if (fp64) return {rs ? 16.0 : 5.0, 60.0};
    return rs ? GemmCost{4.4 + 100.0 / chunk, 200.0} : GemmCost{1.6 + 38.0 / chunk, 150.0};
}

// Time of `first` workgroups of c and then `tiles` of cl, each on the slot that is
// free first.
static double makespan(double first, double c, double tiles, double cl, double slots)
{
    const double full = std::floor(first / slots), rem = first - full * slots, open = slots - rem;
    double t = std::ceil(tiles / open) * cl;   // on the slots that the last round of c leaves open
    if (rem > 0.0) t = std::max(c, std::min(t, std::ceil((tiles + rem * c / cl) / slots) * cl));
    return full * c + t;
}

// masked: the launch skips most pairs (rs_skip_mask) and some tiles hold all of the
// rest, so its time is that of the longest workgroup after a quarter of the whole work.
static int gemm_point_splits(int64_t tiles, int64_t n, int slots, int64_t npx, int chunk, GemmCost k, bool masked,
                             double* time)
{
    int best = 1;
    for (int S = 1; S <= MAX_SPLITS; ++S) {
        if (S > 1 && (n < (int64_t)S * chunk || (double)(S - 1) * npx * 16.0 > 2.0 * (1ull << 30) ||
                      tiles * (S - 1) > 8 * (int64_t)slots))
            break;
        const int64_t per = S == 1 ? n : ((n + S - 1) / S + chunk - 1) / chunk * chunk, parts = (n + per - 1) / per;
        const double c = per * k.point + k.tile, cl = (n - (parts - 1) * per) * k.point + k.tile;
        const double run = masked ? c + (double)tiles * (n * k.point * 0.25 + parts * k.tile) / slots
                                  : makespan((double)(tiles * (parts - 1)), c, (double)tiles, cl, slots);
        const double t = run + (parts > 1 ? 40.0 + (parts - 1) * (npx * 8e-5) : 0.0);
        // the first further plane by a tenth, for the model takes every box as whole
        if (S == 1 || t < *time * (best == 1 ? 0.9 : 0.97)) {
            best = S;
            *time = t;
        }
    }
    return best;
}

// 240, or shorter ones, at whose boundaries tiles are split, where 240 would leave
// CUs without work (256 workgroups of 240 points), and shorter again where the model
// finds a tenth in it on the usual 256 CUs (500 RS points at 1920x1080: 0.31 -> 0.27
// ms; the serving engine and the no-allocation form sum alike but do not split, and
// lose 8 %).  Longer ones are faster for a few hundred points on 1920x1080, by 14 us
// of 80 for 200 points, Fresnel; but an FP32 sum of 200 points is off by 3.1e-7, of
// 60 by 1.9e-7.
int direct_chunk(const Geometry& g, int64_t n)
{
    const bool rs = g.diff == OHX_DIFF_RS;
    const int least = (rs ? 1 : 2) * DIRECT_CELL;
    int tx, best = DIRECT_CHUNK;
    const int64_t tiles = direct_tiles(g, false, &tx), npx = (int64_t)g.pn_x * g.pn_y;
    while (best > least && tiles * n < 256 * best) best /= 2;
    double best_t = 0.0;
    for (int first = best, chunk = first; chunk >= least; chunk /= 2) {
        double t;
        gemm_point_splits(tiles, n, 256, npx, chunk, gemm_cost(rs, false, chunk), false, &t);
        if (chunk == first || t < best_t * 0.9) {
            best = chunk;
            best_t = t;
        }
    }
    return best;
}

// The matrix product, and for RS the per-pixel kernels for what it leaves.
template <int DIFF, typename T>
static void launch_gemm(hipStream_t st, const Geometry& g, const PointSoA& soa, double2* f, const SplitArgs& sa,
                        int splits, int tiles_x, unsigned* flags)
{
    hipLaunchKernelGGL((k_pc_gemm<DIFF, T>), dim3((unsigned)(sa.tiles * splits)), dim3(dgemm::Kind<T>::NTH), 0, st, g,
                       soa, f, tiles_x, flags, sa);
    if constexpr (DIFF == OHX_DIFF_RS) {
        const int xt = (g.pn_x + TW - 1) / TW;
        const dim3 grid((unsigned)(xt * ((g.pn_y + TH - 1) / TH)));
        const unsigned* fl = flags;
        hipLaunchKernelGGL(k_pc_lines<T>, grid, dim3(NT), 0, st, g, soa, f, xt, tiles_x, fl);
        if constexpr (dgemm::Kind<T>::f64) {
            if (few_tiles(g)) {
                using R = Rest<T, true>;
                hipLaunchKernelGGL((k_pc_rest<T, true>), dim3((unsigned)(xt * ((g.pn_y + R::ROWS - 1) / R::ROWS))),
                                   dim3(R::THREADS), 0, st, g, soa, f, xt, tiles_x, fl, false);
                return;
            }
        }
        hipLaunchKernelGGL((k_pc_rest<T, false>), grid, dim3(NT), 0, st, g, soa, f, xt, tiles_x, fl, false);
    }
}

int launch_direct(ohx_ctx* ctx, const Geometry& g, const PointSoA& soa, double* d_field, bool fp64)
{
    return launch_direct_with(ctx, g, soa, d_field, fp64, (unsigned*)(ctx->minmax + CTX_FLAGS), true,
                              direct_chunk(g, soa.n), !fp64 && direct_per_pixel(g, soa.n));
}

int launch_direct_with(ohx_ctx* ctx, const Geometry& g, const PointSoA& soa, double* d_field, bool fp64,
                       unsigned* flags, bool allow_splits, int chunk, bool per_pixel)
{
    const bool rs = g.diff == OHX_DIFF_RS;
    const int tiles_x = (g.pn_x + dgemm::GW - 1) / dgemm::GW;
    const int gh = fp64 ? dgemm::Kind<double>::GH : dgemm::Kind<float>::GH;
    const int64_t tiles = (int64_t)tiles_x * ((g.pn_y + gh - 1) / gh);
    const int64_t npx = (int64_t)g.pn_x * g.pn_y;
    if (tiles * MAX_SPLITS > 0x7fffffff) return set_error(ctx, OHX_ERR_INVALID_ARG, "hologram too large");
    double2* f = (double2*)d_field;
    const int xt = (g.pn_x + TW - 1) / TW;
    const int64_t small_tiles = (int64_t)xt * ((g.pn_y + TH - 1) / TH);
    // counted in (tile, split) items of 64 x 32 (FP32) or 128 x 16 (FP64) pixels
    ctx->last.workgroups = fp64 ? (int64_t)tiles_x * ((g.pn_y + 15) / 16) : small_tiles;
    ctx->last.kernel_kind = fp64 ? 1 : 0;
    if (per_pixel) {
        hipLaunchKernelGGL((k_pc_rest<float, false>), dim3((unsigned)small_tiles), dim3(NT), 0, ctx->stream, g, soa, f, xt, tiles_x,
                           (const unsigned*)flags, true);
        return check_hip(ctx, hipGetLastError(), "k_pc_rest");
    }
    const void* kern = fp64 ? (rs ? (const void*)k_pc_gemm<OHX_DIFF_RS, double>
                                  : (const void*)k_pc_gemm<OHX_DIFF_FRESNEL, double>)
                            : (rs ? (const void*)k_pc_gemm<OHX_DIFF_RS, float>
                                  : (const void*)k_pc_gemm<OHX_DIFF_FRESNEL, float>);
    if (fp64) chunk = 32;
    int splits = 1;
    if (allow_splits) {
        double t;
        splits = gemm_point_splits(tiles, soa.n,
                                   resident_slots(ctx, kern, fp64 ? dgemm::Kind<double>::NTH : dgemm::Kind<float>::NTH),
                                   npx, chunk, gemm_cost(rs, fp64, chunk), g.rs_skip_mask != nullptr, &t);
    }
    SplitArgs sa{(int)tiles, soa.n, nullptr, chunk};
    if (splits > 1) {
        // split boundaries on chunk boundaries: an FP32 split sums exactly as the
        // serving engine's point slices do (FP64 ones to rounding)
        const int64_t per = (soa.n + splits - 1) / splits;
        sa.split_pts = (per + chunk - 1) / chunk * chunk;
        splits = (int)((soa.n + sa.split_pts - 1) / sa.split_pts);
    }
    if (splits > 1) {
        int st = ensure_gemm_scratch(ctx, (size_t)(splits - 1) * npx * sizeof(double2));
        if (st) return st;
        sa.part = (double2*)ctx->gemm_scratch;
    }
    hipStream_t st = ctx->stream;
    if (fp64 && rs) launch_gemm<OHX_DIFF_RS, double>(st, g, soa, f, sa, splits, tiles_x, flags);
    else if (fp64) launch_gemm<OHX_DIFF_FRESNEL, double>(st, g, soa, f, sa, splits, tiles_x, flags);
    else if (rs) launch_gemm<OHX_DIFF_RS, float>(st, g, soa, f, sa, splits, tiles_x, flags);
    else launch_gemm<OHX_DIFF_FRESNEL, float>(st, g, soa, f, sa, splits, tiles_x, flags);
    if (splits > 1) {
        const int64_t rb = std::min<int64_t>((npx + 255) / 256, 4096);
        hipLaunchKernelGGL(k_split_reduce, dim3((unsigned)rb), dim3(256), 0, st, f, (const double2*)sa.part, npx,
                           splits - 1);
    }
    ctx->last.workgroups *= splits;
    return check_hip(ctx, hipGetLastError(), "k_pc_direct");
}

int direct_tiles(const Geometry& g, bool fp64, int* tiles_x)
{
    const int gh = fp64 ? dgemm::Kind<double>::GH : dgemm::Kind<float>::GH;
    *tiles_x = (g.pn_x + dgemm::GW - 1) / dgemm::GW;
    return *tiles_x * ((g.pn_y + gh - 1) / gh);
}

int launch_direct_jobs(hipStream_t stream, DirectJob* d_jobs, const int* d_njobs, unsigned kinds)
{
    // one workgroup (FP32) or two (FP64) per CU; a kernel without work returns, but
    // costs its 4 us in the stream
    constexpr int T32 = dgemm::Kind<float>::NTH, T64 = dgemm::Kind<double>::NTH;
    constexpr unsigned rs = jobs_gemm(OHX_DIFF_RS, 0) | jobs_gemm(OHX_DIFF_RS, 1);
    if (kinds & jobs_gemm(OHX_DIFF_RS, 0))
        hipLaunchKernelGGL((k_pc_gemm_jobs<OHX_DIFF_RS, float>), dim3(256), dim3(T32), 0, stream, d_jobs, d_njobs);
    if (kinds & jobs_gemm(OHX_DIFF_FRESNEL, 0))
        hipLaunchKernelGGL((k_pc_gemm_jobs<OHX_DIFF_FRESNEL, float>), dim3(256), dim3(T32), 0, stream, d_jobs, d_njobs);
    if (kinds & jobs_gemm(OHX_DIFF_RS, 1))
        hipLaunchKernelGGL((k_pc_gemm_jobs<OHX_DIFF_RS, double>), dim3(512), dim3(T64), 0, stream, d_jobs, d_njobs);
    if (kinds & jobs_gemm(OHX_DIFF_FRESNEL, 1))
        hipLaunchKernelGGL((k_pc_gemm_jobs<OHX_DIFF_FRESNEL, double>), dim3(512), dim3(T64), 0, stream, d_jobs, d_njobs);
    if (kinds & rs) hipLaunchKernelGGL(k_pc_lines_jobs, dim3(1024), dim3(NT), 0, stream, d_jobs, d_njobs);
    if (kinds & JOBS_REST) hipLaunchKernelGGL(k_pc_rest_jobs, dim3(512), dim3(NT), 0, stream, d_jobs, d_njobs);
    return hipGetLastError() == hipSuccess ? OHX_OK : OHX_ERR_DEVICE;
}

int launch_probe(ohx_ctx* ctx, const Geometry& g, const PointSoA& soa, const int64_t* d_pix,
                 int64_t n_pix, double* d_out)
{
    const unsigned grid = (unsigned)((n_pix + 255) / 256);
    if (g.diff == OHX_DIFF_RS)
        hipLaunchKernelGGL((k_pc_probe<OHX_DIFF_RS>), dim3(grid), dim3(256), 0, ctx->stream, g, soa, d_pix, n_pix,
                           (double2*)d_out);
    else
        hipLaunchKernelGGL((k_pc_probe<OHX_DIFF_FRESNEL>), dim3(grid), dim3(256), 0, ctx->stream, g, soa, d_pix,
                           n_pix, (double2*)d_out);
    return check_hip(ctx, hipGetLastError(), "k_pc_probe");
}

}  // namespace ohx
