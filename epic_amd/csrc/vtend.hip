// vorticity_tendency (inversion.f90:321-366, 345-360) on gfx950:
//
//   vtend_c = d/dx [(xi + f_x) u_c] + d/dy [(eta + f_y) u_c] + d/dz [(zeta + f_z) u_c]
//
// with -b in the x flux of the y component and +b in the y flux of the x
// component (inversion.f90:327-335).  The spectral derivative along x only
// couples the points of one row and that along y the points of one column
// line, so no two-dimensional transform is needed: k_flux_dx takes one-
// dimensional transforms of the rows, k_flux_dy of the y lines, adds the x
// part and the second-order z difference and stores the tendency of every
// plane, the halo planes included.  Two real lines travel as the real and
// imaginary part of one complex line: multiplying the spectrum by i k keeps
// them apart.
//
// Everything is FP64 from the FP32 node fields to the one rounding of the
// stored tendency (the spectral derivative amplifies white rounding noise at
// the highest wavenumbers).  The halo planes are the linear extrapolations
// 2 v(0) - v(1) and 2 v(nz) - v(nz-1) formed from the extrapolated fluxes, so
// before that rounding; where dzeta/dt is held at zero on a wall
// (inversion.f90:345-350) the wall is 0 and its halo plane -v(1).
//
// What bounds it: HBM and L2 traffic.  Per node and component k_flux_dx reads
// 8 to 12 B and writes 8 B (the FP64 x part), k_flux_dy reads those, 8 to 12 B
// of its own flux and up to 16 B of the z neighbours, and writes 4 B; the
// two-dimensional FP64 transforms that this replaces moved 21 passes over
// FP64 spectra (sum of their five launches at 128^3: 262 us).
#include "common.h"
#include "fft.h"
#include "launch.h"

#include <algorithm>

namespace epic {

// elements a thread requests before the first LDS store, with clamped
// addresses and no branches between the loads
constexpr int VT_BATCH = 4;
// x columns of a k_flux_dy block: 64-byte segments of a row, 8 complex lines
constexpr int VT_COLS = 16, VT_PAIRS = VT_COLS / 2;

__device__ inline double flux(const VtendArgs &a, const EPIC_GLOBAL float *om, const EPIC_GLOBAL float *vel,
                              const EPIC_GLOBAL float *b, double f, double sgn, int64_t o)
{
    double v = ((double)om[o] + f) * (double)vel[o];
    if (sgn != 0.0) v += sgn * (double)b[o];
    return v;
}

// the spectrum of a line (natural order, n points) times i k / n with k = 2 pi
// kk / extent, zero at the Nyquist wavenumber (diffx / diffy,
// sta3dfft.f90:301-374), in place
__device__ inline void times_ik(double2 *Z, int L, int ls, const FftPlan &pl, double extent)
{
    const int n = pl.n;
    const double s = 2.0 * 3.14159265358979323846 / (extent * (double)n);
    for (int t = threadIdx.x; t < L * n; t += blockDim.x) {
        const int l = fdiv(t, pl.n1), q = t - l * n;
        const int kk = (2 * q < n) ? q : q - n;
        const double w = (2 * q == n) ? 0.0 : s * (double)kk;
        const double2 v = Z[l * ls + q];
        Z[l * ls + q] = double2{-w * v.y, w * v.x};
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// physical-space completion
// ---------------------------------------------------------------------------
// vor2vel: z halo of velocity (inversion.f90:241-248) and the derived
// gradient components (:278-313); one thread per (column, plane k =
// -1..nz+1).  A halo-plane thread forms its own halo values (linear
// extrapolation, or antisymmetry for w and its horizontal derivatives) from
// the interior planes before the derived components.  In a step these are
// further blocks of k_flux_dx, which reads neither the halo planes nor the
// gradient (a launch of 4 to 5 us less on small grids).
__device__ inline void vor2vel_fixup(const Grid &g, float *fld, int64_t tq)
{
    const int nz = g.nz;
    const int64_t ncol = (int64_t)g.nx * g.ny;
    if (tq >= ncol * (nz + 3)) return;
    const int k = (int)(tq / ncol) - 1;
    const int64_t col = tq - (int64_t)(k + 1) * ncol;
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    auto F = [&](int slot, int kk) -> EPIC_GLOBAL float & { return gl(fld)[slot * FS + (int64_t)(kk + 1) * PS + col]; };
    float dwdx, dudy, dwdy;
    if (k == -1 || k == nz + 1) {
        const int kb = (k < 0) ? 0 : nz, kn = (k < 0) ? 1 : nz - 1;
        auto lin = [&](int slot) { return F(slot, k) = 2.0f * F(slot, kb) - F(slot, kn); };
        auto anti = [&](int slot) { return F(slot, k) = -F(slot, kn); };
        lin(F_VELOG + 0);
        lin(F_VELOG + 1);
        anti(F_VELOG + 2);
        lin(F_VELGRADG + DUDX);
        dudy = lin(F_VELGRADG + DUDY);
        dwdx = anti(F_VELGRADG + DWDX);
        lin(F_VELGRADG + DVDY);
        dwdy = anti(F_VELGRADG + DWDY);
    } else {
        dwdx = F(F_VELGRADG + DWDX, k);
        dudy = F(F_VELGRADG + DUDY, k);
        dwdy = F(F_VELGRADG + DWDY, k);
    }
    F(F_VELGRADG + DUDZ, k) = dwdx + F(F_VORTG + 1, k);
    F(F_VELGRADG + DVDX, k) = dudy + F(F_VORTG + 2, k);
    F(F_VELGRADG + DVDZ, k) = dwdy - F(F_VORTG + 0, k);
}

__global__ __launch_bounds__(256) void k_vor2vel_fixup(const FixArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    vor2vel_fixup(tab[ib.item].g, tab[ib.item].fld, ib.blk * (int64_t)256 + threadIdx.x);
}

static int fixup_blocks(const Grid &g) { return (int)(((int64_t)g.nx * g.ny * (g.nz + 3) + 255) / 256); }

void add_vor2vel_fixup(Plan &P, int phase, const std::vector<FixArgs> &items)
{
    std::vector<int> nb;
    for (const FixArgs &a : items) nb.push_back(fixup_blocks(a.g));
    P.add((const void *)k_vor2vel_fixup, 256, 0, phase, items, nb);
}

// x derivative of the x flux of one component on planes 0..nz, rows (plane,
// j) taken in pairs; a.lines pairs per block
__global__ __launch_bounds__(256) void k_flux_dx(const VtendArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const VtendArgs &a = tab[ib.item];
    const Grid &g = a.g;
    if (ib.blk >= a.dx_blocks) {   // uniform over the block
        vor2vel_fixup(g, a.fld, (ib.blk - a.dx_blocks) * (int64_t)256 + threadIdx.x);
        return;
    }
    const int n = g.nx, L = a.lines, ls = n + 1;
    const int64_t rows = (int64_t)(g.nz + 1) * g.ny, r0 = (int64_t)ib.blk * 2 * L;
    extern __shared__ double2 lds[];
    double2 *bufa = lds, *bufb = lds + L * ls, *tw = bufb + L * ls;
    for (int t = threadIdx.x; t < n; t += blockDim.x) tw[t] = gl(a.twx)[t];
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    // rows of consecutive planes are contiguous from plane 0 on
    const EPIC_GLOBAL float *om = gl(a.fld) + (F_VORTG + 0) * FS + PS, *vel = gl(a.fld) + (F_VELOG + a.comp) * FS + PS,
                            *b = gl(a.fld) + F_TBUOYG * FS + PS;
    const double sgn = (a.comp == 1) ? -1.0 : 0.0, f = g.f_cor[0];
    const int total = L * n;
    for (int t0 = threadIdx.x; t0 < total; t0 += VT_BATCH * blockDim.x) {
        double2 z[VT_BATCH];
#pragma unroll
        for (int u = 0; u < VT_BATCH; ++u) {
            const int t = min(t0 + u * (int)blockDim.x, total - 1);
            const int l = fdiv(t, a.px.n1), q = t - l * n;
            const int64_t ra = min(r0 + 2 * l, rows - 1), rb = min(r0 + 2 * l + 1, rows - 1);
            z[u] = double2{flux(a, om, vel, b, f, sgn, ra * n + q), flux(a, om, vel, b, f, sgn, rb * n + q)};
        }
#pragma unroll
        for (int u = 0; u < VT_BATCH; ++u) {
            const int t = t0 + u * blockDim.x;
            const int l = fdiv(min(t, total - 1), a.px.n1);
            if (t < total) bufa[t + l] = z[u];   // l ls + q
        }
    }
    __syncthreads();
    double2 *Z = lds_fft(bufa, bufb, L, a.px, tw, 1, false, ls);
    times_ik(Z, L, ls, a.px, g.extent[0]);
    Z = lds_fft(Z, Z == bufa ? bufb : bufa, L, a.px, tw, 1, true, ls);
    EPIC_GLOBAL double *out = gl(a.dx) + (int64_t)a.comp * rows * n;
    for (int t = threadIdx.x; t < 2 * total; t += blockDim.x) {
        const int r = fdiv(t, a.px.n1), q = t - r * n;   // row r of the block
        const double2 v = Z[(r >> 1) * ls + q];
        if (r0 + r < rows) out[(r0 + r) * n + q] = (r & 1) ? v.y : v.x;
    }
}

// y derivative of the y flux, plus the x part and the z difference, of one
// component on planes -1..nz+1: a block takes VT_COLS columns of a.planes
// consecutive planes
__global__ __launch_bounds__(256) void k_flux_dy(const VtendArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const VtendArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int n = g.ny, nz = g.nz, ls = n + 1;
    const int nbx = (g.nx + VT_COLS - 1) / VT_COLS;
    const int i0 = (ib.blk % nbx) * VT_COLS, kb = (ib.blk / nbx) * a.planes - 1;
    const int L = VT_PAIRS * a.planes;
    extern __shared__ double2 lds[];
    double2 *bufa = lds, *bufb = lds + L * ls, *tw = bufb + L * ls;
    for (int t = threadIdx.x; t < n; t += blockDim.x) tw[t] = gl(a.twy)[t];
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    const EPIC_GLOBAL float *om = gl(a.fld) + (F_VORTG + 1) * FS + PS, *vel = gl(a.fld) + (F_VELOG + a.comp) * FS + PS,
                            *b = gl(a.fld) + F_TBUOYG * FS + PS;
    const EPIC_GLOBAL float *omz = gl(a.fld) + (F_VORTG + 2) * FS + PS;
    const double sgn = (a.comp == 0) ? 1.0 : 0.0, f = g.f_cor[1], fz = g.f_cor[2];
    // plane k as plane p0 with weight c0 plus plane p1 with weight c1
    auto weights = [&](int k, int &p0, int &p1, double &c0, double &c1) {
        p0 = p1 = max(0, min(k, nz));
        c0 = 1.0;
        c1 = 0.0;
        if (k == -1) {
            p1 = 1;
            c0 = (a.comp == 2 && g.zeta_zero[0]) ? 0.0 : 2.0;
            c1 = -1.0;
        } else if (k == nz + 1) {
            p1 = nz - 1;
            c0 = (a.comp == 2 && g.zeta_zero[1]) ? 0.0 : 2.0;
            c1 = -1.0;
        }
    };
    const int total = L * n;   // t = (plane, y, pair), pairs fastest
    for (int t0 = threadIdx.x; t0 < total; t0 += VT_BATCH * blockDim.x) {
        double2 z[VT_BATCH];
#pragma unroll
        for (int u = 0; u < VT_BATCH; ++u) {
            const int t = min(t0 + u * (int)blockDim.x, total - 1);
            const int c = t % VT_PAIRS, pj = t / VT_PAIRS, pl = fdiv(pj, a.py.n1), j = pj - pl * n;
            const int i = min(i0 + 2 * c, g.nx - 2);   // nx is even
            int p0, p1;
            double c0, c1;
            weights(kb + pl, p0, p1, c0, c1);
            const int64_t o0 = (int64_t)p0 * PS + (int64_t)j * g.nx + i;
            z[u] = double2{flux(a, om, vel, b, f, sgn, o0), flux(a, om, vel, b, f, sgn, o0 + 1)};
            if (c1 != 0.0) {
                const int64_t o1 = (int64_t)p1 * PS + (int64_t)j * g.nx + i;
                z[u].x = c0 * z[u].x + c1 * flux(a, om, vel, b, f, sgn, o1);
                z[u].y = c0 * z[u].y + c1 * flux(a, om, vel, b, f, sgn, o1 + 1);
            }
        }
#pragma unroll
        for (int u = 0; u < VT_BATCH; ++u) {
            const int t = t0 + u * blockDim.x;
            const int c = t % VT_PAIRS, pj = t / VT_PAIRS, pl = fdiv(min(pj, a.planes * n - 1), a.py.n1), j = pj - pl * n;
            if (t < total) bufa[(pl * VT_PAIRS + c) * ls + j] = z[u];
        }
    }
    __syncthreads();
    double2 *Z = lds_fft(bufa, bufb, L, a.py, tw, 1, false, ls);
    times_ik(Z, L, ls, a.py, g.extent[1]);
    Z = lds_fft(Z, Z == bufa ? bufb : bufa, L, a.py, tw, 1, true, ls);

    const EPIC_GLOBAL double *dx = gl(a.dx) + (int64_t)a.comp * (nz + 1) * PS;
    EPIC_GLOBAL float *out = gl(a.fld) + (F_VTEND + a.comp) * FS + PS;
    const double dzi = g.dxi[2];
    for (int t = threadIdx.x; t < total; t += blockDim.x) {
        const int c = t % VT_PAIRS, pj = t / VT_PAIRS, pl = fdiv(pj, a.py.n1), j = pj - pl * n;
        const int i = i0 + 2 * c, k = kb + pl;
        if (i >= g.nx || k > nz + 1) continue;
        int p0, p1;
        double c0, c1;
        weights(k, p0, p1, c0, c1);
        const int64_t col = (int64_t)j * g.nx + i;
        // x part + d/dz of (zeta + f_z) u_c, second order (central_diffz,
        // inversion_utils.f90:488-514), of plane p at columns i and i + 1
        auto rest = [&](int p) {
            auto f3 = [&](int kk) {
                const int64_t o = (int64_t)kk * PS + col;
                return double2{((double)omz[o] + fz) * (double)vel[o], ((double)omz[o + 1] + fz) * (double)vel[o + 1]};
            };
            const int lo = max(p - 1, 0), hi = min(p + 1, nz);
            const double s = (hi - lo == 2) ? 0.5 * dzi : dzi;
            const double2 h = f3(hi), l = f3(lo);
            const int64_t o = (int64_t)p * PS + col;
            return double2{dx[o] + (h.x - l.x) * s, dx[o + 1] + (h.y - l.y) * s};
        };
        const double2 r0 = rest(p0);
        double2 v = Z[(pl * VT_PAIRS + c) * ls + j];
        if (c1 == 0.0) {
            v = double2{v.x + r0.x, v.y + r0.y};
        } else {
            const double2 r1 = rest(p1);
            v = double2{v.x + (c0 * r0.x + c1 * r1.x), v.y + (c0 * r0.y + c1 * r1.y)};
        }
        if (a.comp == 2 && ((k == 0 && g.zeta_zero[0]) || (k == nz && g.zeta_zero[1]))) v = double2{0.0, 0.0};
        const int64_t o = (int64_t)k * PS + col;
        out[o] = (float)v.x;
        out[o + 1] = (float)v.y;
    }
}

// Points of complex lines a block: 1024, four to a thread, one radix-4
// butterfly a stage, and four blocks to a CU's LDS; 256 on grids whose 1024
// points a block would leave CUs without one (below 2^18 nodes a component:
// the block's own chain of stages is what such a launch takes).  Short lines
// are taken several to a block, long ones at least one row pair / one plane.
static int block_points(const Grid &g) { return (int64_t)g.nx * g.ny * (g.nz + 1) >= (1 << 18) ? 1024 : 256; }
static int dx_lines(const Grid &g) { return std::max(1, block_points(g) / g.nx); }
static int dy_planes(const Grid &g) { return std::max(1, block_points(g) / (VT_PAIRS * g.ny)); }

void add_vtend(Plan &P, int phase, const std::vector<VtendArgs> &members, bool fix)
{
    std::vector<VtendArgs> items;
    std::vector<int> bx, by;
    size_t lx = 0, ly = 0;
    for (VtendArgs a : members) {
        const Grid &g = a.g;
        a.lines = dx_lines(g);
        a.planes = dy_planes(g);
        const int64_t rows = (int64_t)(g.nz + 1) * g.ny;
        lx = std::max(lx, sizeof(double2) * (2 * (size_t)a.lines * (g.nx + 1) + g.nx));
        ly = std::max(ly, sizeof(double2) * (2 * (size_t)VT_PAIRS * a.planes * (g.ny + 1) + g.ny));
        for (int c = 0; c < 3; ++c) {
            a.comp = c;
            a.dx_blocks = (int)((rows + 2 * a.lines - 1) / (2 * a.lines));
            items.push_back(a);
            bx.push_back(a.dx_blocks + (fix && c == 0 ? fixup_blocks(g) : 0));
            by.push_back((g.nx + VT_COLS - 1) / VT_COLS * ((g.nz + 3 + a.planes - 1) / a.planes));
        }
    }
    P.add((const void *)k_flux_dx, 256, lx, phase, items, bx);
    P.add((const void *)k_flux_dy, 256, ly, phase, items, by);
}

}  // namespace epic
