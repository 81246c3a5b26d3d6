// Spectral vorticity inversion on gfx950 (inversion.f90:25-366,
// inversion_utils.f90:79-514).
//
// After the horizontal FFTs every horizontal operator of vor2vel is diagonal
// in (kx, ky), so the whole vertical part of the inversion is independent per
// spectral column.  k_vor2vel_columns gives each column to one wavefront and
// runs it in FP64, the column in registers (nz <= 191) or in LDS:
// decomposition into boundary values + sine series,
// Hou-Li filter, solenoidal projection, vertical Green's function, the
// hyperbolic boundary corrections theta/phi, the zero-mode mean flow and the
// velocity and velocity-gradient spectra.  The z transforms (DST-I / DCT-I
// with the sqrt(2/nz) normalisation of stafft.f90:410-555) are evaluated as
// one complex FFT of length 2 nz of the odd / even extension of the column.
// Tables (filter, Green, theta, phi, gamma) are evaluated on the fly in FP64
// from the same formulas as init_inversion; nothing is stored per column.
#include "common.h"
#include "fft.h"
#include "launch.h"

#include <algorithm>

namespace epic {

#define EPIC_PI 3.14159265358979323846

// columns of up to 64 COL_REG_SLOTS values (nz <= 191) keep their arrays in
// registers, and of nz <= 64 COL_PHASE_SLOTS take their transforms in phases
// of several lines
constexpr int COL_REG_SLOTS = 3, COL_PHASE_SLOTS = 2;

struct ColCtx {
    int nz;
    double2 *fa, *fb;
    const FftPlan *plan;
    const double2 *tw;   // e^{-2 pi i t / (2 nz)}, t < nz (the member's table; cached reads)
};

// One column of nz + 1 values per wave.  With NS > 0 the value at z = lane +
// 64 i sits in register slot i of the lane (NS slots, nz + 1 <= 64 NS): the
// column arrays then take no LDS, only the FFT lines do, and more columns
// share a CU.  NS == 0 keeps every column array in LDS (any nz).
template <int NS, typename T> struct ZCol {
    T r[NS > 0 ? NS : 1];
    T *l = nullptr;
    __device__ T &operator()(int i, int z)
    {
        if constexpr (NS > 0) return r[i];
        else return l[z];
    }
};

__device__ inline double read_lane(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
// the column's value at z (z uniform over the wave; with LDS storage, after
// a barrier that follows its last store)
template <int NS> __device__ __forceinline__ double2 zval(ZCol<NS, double2> &c, int z)
{
    if constexpr (NS > 0) {
        // every slot read from lane z mod 64, then the slot z / 64 chosen
        // among the scalar results (a select among the register slots
        // themselves would become an indexed access, which keeps the slots
        // in scratch memory)
        const int k = z >> 6, l = z & 63;
        double2 s = double2{0.0, 0.0};
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const double2 v = double2{read_lane(c.r[i].x, l), read_lane(c.r[i].y, l)};
            if (k == i) s = v;
        }
        return s;
    } else {
        return c.l[z];
    }
}

// slots of this lane: z = lane + 64 i for i < nsl (z < nz + 1 checked by the caller)
#define ZSLOTS(i, z) \
    _Pragma("unroll") for (int i = 0; i < nsl; ++i) if (const int z = (int)threadIdx.x + 64 * i; true)

// DST-I of col[1..nz-1] in place (col[0], col[nz] untouched)
template <int NS> __device__ __forceinline__ void zdst(const ColCtx &c, ZCol<NS, double2> &col, int nsl)
{
    const int nz = c.nz, n2 = 2 * nz;
    ZSLOTS(i, z)
    {
        if (z > 0 && z < nz) {
            const double2 v = col(i, z);
            c.fa[z] = v;
            c.fa[n2 - z] = double2{-v.x, -v.y};   // the odd extension
        } else if (z == 0 || z == nz) {
            c.fa[z] = double2{0.0, 0.0};
        }
    }
    __syncthreads();
    double2 *R = lds_fft_tw(c.fa, c.fb, 1, *c.plan, TwHalf<double2>{c.tw, nz}, false, n2);
    const double s = 0.5 * sqrt(2.0 / (double)nz);
    ZSLOTS(i, z)
    {
        if (z > 0 && z < nz) col(i, z) = double2{-s * R[z].y, s * R[z].x};   // s i R
    }
    __syncthreads();
}

// DCT-I of col[0..nz] in place
template <int NS> __device__ __forceinline__ void zdct(const ColCtx &c, ZCol<NS, double2> &col, int nsl)
{
    const int nz = c.nz, n2 = 2 * nz;
    ZSLOTS(i, z)
    {
        if (z <= nz) {
            const double2 v = col(i, z);
            c.fa[z] = v;
            if (z > 0 && z < nz) c.fa[n2 - z] = v;   // the even extension
        }
    }
    __syncthreads();
    double2 *R = lds_fft_tw(c.fa, c.fb, 1, *c.plan, TwHalf<double2>{c.tw, nz}, false, n2);
    const double s = 0.5 * sqrt(2.0 / (double)nz);
    ZSLOTS(i, z)
    {
        if (z <= nz) col(i, z) = double2{s * R[z].x, s * R[z].y};
    }
    __syncthreads();
}

// field_decompose_semi_spectral (inversion_utils.f90:372-401)
template <int NS>
__device__ __forceinline__ void decompose(const ColCtx &c, ZCol<NS, double2> &col, ZCol<NS, double> &phim, ZCol<NS, double> &phip,
                          int nsl)
{
    const int nz = c.nz;
    const double2 b0 = zval(col, 0), bn = zval(col, nz);
    __syncthreads();
    ZSLOTS(i, z)
    {
        if (z > 0 && z < nz) {
            const double2 v = col(i, z);
            const double pm = phim(i, z), pp = phip(i, z);
            col(i, z) = double2{v.x - (b0.x * pm + bn.x * pp), v.y - (b0.y * pm + bn.y * pp)};
        }
    }
    __syncthreads();
    zdst(c, col, nsl);
}

// field_combine_semi_spectral (inversion_utils.f90:426-456)
template <int NS>
__device__ __forceinline__ void combine(const ColCtx &c, ZCol<NS, double2> &col, ZCol<NS, double> &phim, ZCol<NS, double> &phip,
                        int nsl)
{
    const int nz = c.nz;
    zdst(c, col, nsl);
    const double2 b0 = zval(col, 0), bn = zval(col, nz);
    ZSLOTS(i, z)
    {
        if (z > 0 && z < nz) {
            const double2 v = col(i, z);
            const double pm = phim(i, z), pp = phip(i, z);
            col(i, z) = double2{v.x + b0.x * pm + bn.x * pp, v.y + b0.y * pm + bn.y * pp};
        }
    }
    __syncthreads();
}

__device__ inline double2 muli(double2 a, double s) { return double2{-s * a.y, s * a.x}; }   // i s a

// x^36 of the Hou-Li filter
__device__ inline double pow36(double x)
{
    const double x2 = x * x, x4 = x2 * x2, x8 = x4 * x4, x16 = x8 * x8;
    return x16 * x16 * x4;
}

// ---------------------------------------------------------------------------
// in-place transforms of L lines of n points by one wave (register form)
// ---------------------------------------------------------------------------
// One Stockham stage: the butterflies of all the lines are spread over the
// lanes (M of them a lane at most) and all read before any is written, so a
// line needs one buffer and the lines of a phase overlap their latencies.
template <int R, int M>
__device__ __forceinline__ void wave_fft_stage(double2 *buf, int ls, int L, const FastDiv &nbd, const FastDiv &nsd, int tstep,
                                               const TwHalf<double2> &tw)
{
    const int nb = nbd.d, Ns = nsd.d, total = L * nb;
    double2 v[M][R];
    int dst[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int t = (int)threadIdx.x + 64 * m;
        if (t >= total) continue;
        const int l = fdiv(t, nbd), jj = t - l * nb, o = l * ls;
#pragma unroll
        for (int r = 0; r < R; ++r) v[m][r] = buf[o + jj + r * nb];
        const int q = fdiv(jj, nsd), kk = jj - q * Ns;
        dst[m] = o + q * Ns * R + kk;
        if (Ns > 1) {   // (the first stage's twiddles are 1)
#pragma unroll
            for (int r = 1; r < R; ++r) v[m][r] = cmul(v[m][r], tw(r * kk * tstep));
        }
        butterfly<R>(v[m], false);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; ++m) {
        if ((int)threadIdx.x + 64 * m >= total) continue;
#pragma unroll
        for (int r = 0; r < R; ++r) buf[dst[m] + r * Ns] = v[m][r];
    }
    __syncthreads();
}

// butterflies of radix R a lane has at most in three lines of n <= 128 NS points
constexpr int wave_butterflies(int NS, int R) { return (3 * 128 * NS / R + 63) / 64; }

template <int NS>
__device__ __forceinline__ void wave_fft(double2 *buf, int ls, int L, const FftPlan &pl, const TwHalf<double2> &tw)
{
    const int nst = pl.nst;
    FftStage next = pl.st[0];
#pragma unroll 1
    for (int st = 0; st < nst; ++st) {
        const FftStage g = next;
        next = pl.st[min(st + 1, nst - 1)];   // requested a stage ahead
        if (g.radix == 4) wave_fft_stage<4, wave_butterflies(NS, 4)>(buf, ls, L, g.nb, g.ns, g.tstep, tw);
        else if (g.radix == 2) wave_fft_stage<2, wave_butterflies(NS, 2)>(buf, ls, L, g.nb, g.ns, g.tstep, tw);
        else if (g.radix == 3) wave_fft_stage<3, wave_butterflies(NS, 3)>(buf, ls, L, g.nb, g.ns, g.tstep, tw);
        else wave_fft_stage<5, wave_butterflies(NS, 5)>(buf, ls, L, g.nb, g.ns, g.tstep, tw);
    }
}

// A column of the phase form: the inner values z = 1 + lane + 64 i in register
// slots i < NS, the two boundary values z = 0 and nz in lanes 0 and 1 of slot
// NS.  nz = 64 and 128 then take 1 and 2 slots of inner values, not 2 and 3 of
// nz + 1.
template <int NS> struct PCol {
    double2 r[NS + 1];
    __device__ double2 low() const { return double2{read_lane(r[NS].x, 0), read_lane(r[NS].y, 0)}; }
    __device__ double2 top() const { return double2{read_lane(r[NS].x, 1), read_lane(r[NS].y, 1)}; }
};
// inner slots, and inner and boundary slots (BND: a compile-time constant)
#define ZIN(i, z) \
    _Pragma("unroll") for (int i = 0; i < NS; ++i) if (const int z = 1 + (int)threadIdx.x + 64 * i; z < nz)
#define ZBND(z) if (const int z = threadIdx.x == 0 ? 0 : nz; threadIdx.x < 2)
#define ZALL(i, z) \
    _Pragma("unroll") for (int i = 0; i <= NS; ++i) \
        if (const int z = i < NS ? 1 + (int)threadIdx.x + 64 * i : threadIdx.x == 0 ? 0 : nz; i < NS ? z < nz : threadIdx.x < 2)

template <int NS>
__global__ __launch_bounds__(64, NS == 1 ? 3 : 2) void k_vor2vel_columns(const ColArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const ColArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int nz = g.nz;
    const int col = ib.blk;
    const int kx = col % g.nxh, ky = col / g.nxh;
    const bool zero_mode = (kx == 0 && ky == 0);

    extern __shared__ double2 sm[];
    const int n2 = 2 * nz;
    double2 *const line[3] = {sm, sm + n2, sm + 2 * n2};   // the FFT lines
    double2 *const twl = sm + 3 * n2;                      // e^{-2 pi i t / (2 nz)}, t < nz
    const TwHalf<double2> tw{twl, nz};
    PCol<NS> SX, SY, C, E, DS, AS;
    double phim[NS], phip[NS];

    // wavenumbers (sta3dfft.f90:88-107, sta2dfft.f90:59-64): r = (pi/L) 2k
    const int kys = (2 * ky <= g.ny) ? ky : ky - g.ny;
    const double scx = EPIC_PI / g.extent[0], scy = EPIC_PI / g.extent[1], scz = EPIC_PI / g.extent[2];
    const double rkx = scx * (double)(2 * kx), rky = scy * (double)(2 * (kys < 0 ? -kys : kys));
    const double ikx = (2 * kx == g.nx) ? 0.0 : rkx;                       // diffx factor
    const double iky = (2 * ky == g.ny) ? 0.0 : (kys < 0 ? -rky : rky);   // diffy factor
    const double k2l2 = rkx * rkx + rky * rky;
    const double k2l2i = zero_mode ? 0.0 : 1.0 / k2l2;
    // Hou & Li filter (inversion_utils.f90:130-150)
    const double kxmaxi = 1.0 / (scx * (double)g.nx), kymaxi = 1.0 / (scy * (double)g.ny);
    const double kzmaxi = 1.0 / (scz * (double)nz);
    const double fh = exp(-36.0 * pow36(kxmaxi * rkx) + -36.0 * pow36(kymaxi * rky));
    // hyperbolic functions (inversion_utils.f90:305-351)
    const double Lz = g.extent[2];
    const double kl = sqrt(k2l2);
    const double ef = exp(-kl * Lz);
    const double dv = 1.0 / (1.0 - ef * ef);
    const double Q = dv * (1.0 + ef * ef), Rr = dv * 2.0 * ef, k2ifac = 0.5 * k2l2i;

    auto zcoord = [&](int iz, double &zm, double &zp) {
        const double z = g.lower[2] + g.dx[2] * (double)iz;
        zm = g.upper[2] - z;
        zp = z - g.lower[2];
    };

    // ---- load the three vorticity spectra and the phi tables ----
    const int64_t base = ((int64_t)ky * g.nxh + kx) * g.nzp;
    for (int t = threadIdx.x; t < nz; t += 64) twl[t] = gl(a.ztw)[t];
    ZALL(i, z)
    {
        const float2 x = gl(a.in[0])[base + z], y = gl(a.in[1])[base + z], w = gl(a.in[2])[base + z];
        SX.r[i] = double2{x.x, x.y};
        SY.r[i] = double2{y.x, y.y};
        C.r[i] = double2{w.x, w.y};
    }
    ZIN(i, z)
    {
        double zm, zp;
        zcoord(z, zm, zp);
        if (zero_mode) {
            phim[i] = zm / Lz;
            phip[i] = zp / Lz;
        } else {
            const double ep = exp(-(kl * zp)), em = exp(-(kl * zm));
            phim[i] = dv * (ep - ef * em);
            phip[i] = dv * (em - ef * ep);
        }
    }
    const double s = 0.5 * sqrt(2.0 / (double)nz);   // DST-I / DCT-I normalisation of the extended lines
    double2 ds0 = double2{0.0, 0.0}, dsn = ds0;
    double2 mb[4] = {};   // the mean flow's boundary values

    // the odd extension of col[1..nz-1] for a DST-I, col's boundary values
    // taken off in decomposed form first when dec
    auto put_odd = [&](double2 *f, const PCol<NS> &col, bool dec) {
        const double2 b0 = col.low(), bn = col.top();
        ZIN(i, z)
        {
            double2 v = col.r[i];
            if (dec) {
                const double pm = phim[i], pp = phip[i];
                v = double2{v.x - (b0.x * pm + bn.x * pp), v.y - (b0.y * pm + bn.y * pp)};
            }
            f[z] = v;
            f[n2 - z] = double2{-v.x, -v.y};
        }
        ZBND(z) f[z] = double2{0.0, 0.0};
    };
    // the even extension of col[0..nz] for a DCT-I
    auto put_even = [&](double2 *f, const PCol<NS> &col) {
        ZIN(i, z)
        {
            f[z] = col.r[i];
            f[n2 - z] = col.r[i];
        }
        ZBND(z) f[z] = col.r[NS];
    };
    // DST-I result to col[1..nz-1], the boundary values' part added when comb
    auto get_odd = [&](const double2 *f, PCol<NS> &col, bool comb) {
        const double2 b0 = col.low(), bn = col.top();
        ZIN(i, z)
        {
            double2 v = double2{-s * f[z].y, s * f[z].x};   // s i R
            if (comb) {
                const double pm = phim[i], pp = phip[i];
                v = double2{v.x + b0.x * pm + bn.x * pp, v.y + b0.y * pm + bn.y * pp};
            }
            col.r[i] = v;
        }
    };
    auto get_even = [&](const double2 *f, PCol<NS> &col) {
        ZALL(i, z) col.r[i] = double2{s * f[z].x, s * f[z].y};
    };

    // The vertical transforms come in six phases of up to three lines; a loop
    // over the phases keeps one copy of the transform's code.  A column is a
    // chain of latencies (transform stages, exponentials, and instruction
    // fetches of nine inlined transforms): against one transform after the
    // other a launch takes 30 -> 16 us at 16^3, 36 -> 21 at 32^3, 56 -> 33 at
    // 64^3 (48 with slots of nz + 1 values, which spilled), 163 -> 159 at 128^3.
    // Three waves per SIMD of one slot: of two, the 2112 waves of a 64 x 64
    // grid leave a tail (42 us at 64^3); of two slots two (the 168 registers
    // of three spill 83).
    enum { DECOMPOSE, COMBINE_ZETA, DECOMPOSE_DZ, COMBINE, VELOCITY, MEAN_FLOW };
#pragma unroll 1
    for (int ph = DECOMPOSE; ph <= (zero_mode ? MEAN_FLOW : VELOCITY); ++ph) {
        if (ph == DECOMPOSE) {   // inversion.f90:40-43
            put_odd(line[0], SX, true);
            put_odd(line[1], SY, true);
            put_odd(line[2], C, true);
        } else if (ph == COMBINE_ZETA) {   // inversion.f90:50-87: zeta, semi-spectral
            put_odd(line[0], C, false);
        } else if (ph == DECOMPOSE_DZ) {
            put_odd(line[0], E, true);
        } else if (ph == COMBINE) {
            put_odd(line[0], DS, false);
            put_odd(line[1], AS, false);
        } else if (ph == VELOCITY) {
            put_even(line[0], AS);
            put_odd(line[1], DS, false);
        } else {
            put_even(line[0], AS);
            put_even(line[1], SX);
        }
        __syncthreads();
        wave_fft<NS>(sm, n2, ph == DECOMPOSE ? 3 : ph >= COMBINE ? 2 : 1, a.zplan, tw);

        if (ph == DECOMPOSE) {   // and the filter
            get_odd(line[0], SX, false);
            get_odd(line[1], SY, false);
            get_odd(line[2], C, false);
            ZALL(i, z)
            {
                double f = fh;
                if (i < NS) f = fh * exp(-36.0 * pow36(kzmaxi * (scz * (double)z)));
                if (zero_mode) f = 1.0;
                SX.r[i] = double2{f * SX.r[i].x, f * SX.r[i].y};
                SY.r[i] = double2{f * SY.r[i].x, f * SY.r[i].y};
                C.r[i] = double2{f * C.r[i].x, f * C.r[i].y};
            }
        } else if (ph == COMBINE_ZETA) {   // and its z derivative, the neighbours through a line
            get_odd(line[0], C, true);
            double2 *fa = line[1];
            ZALL(i, z) fa[z] = C.r[i];
            __syncthreads();
            const double dzi = g.dxi[2], hdzi = 0.5 * g.dxi[2];
            ZALL(i, z)
            {
                const double w = i < NS ? hdzi : dzi;   // one-sided at the boundaries
                const double2 hi = fa[min(z + 1, nz)], lo = fa[max(z - 1, 0)];
                E.r[i] = double2{w * (hi.x - lo.x), w * (hi.y - lo.y)};
            }
        } else if (ph == DECOMPOSE_DZ) {   // and the solenoidal projection
            get_odd(line[0], E, false);
            ZALL(i, z)
            {
                if (!zero_mode) {
                    // D = B_x - A_y;  A = k2l2i (E_x + D_y), B = k2l2i (E_y - D_x)
                    const double2 sx = SX.r[i], sy = SY.r[i], e = E.r[i];
                    const double2 d = double2{muli(sy, ikx).x - muli(sx, iky).x, muli(sy, ikx).y - muli(sx, iky).y};
                    const double2 ex = muli(e, ikx), ey = muli(e, iky), dx_ = muli(d, ikx), dy_ = muli(d, iky);
                    SX.r[i] = double2{k2l2i * (ex.x + dy_.x), k2l2i * (ex.y + dy_.y)};
                    SY.r[i] = double2{k2l2i * (ey.x - dx_.x), k2l2i * (ey.y - dx_.y)};
                }
                DS.r[i] = SX.r[i];
                AS.r[i] = SY.r[i];
            }
        } else if (ph == COMBINE) {   // the filtered solenoidal vorticity (inversion.f90:91-93)
            get_odd(line[0], DS, true);
            get_odd(line[1], AS, true);
            ZALL(i, z)
            {
                const double2 ds = DS.r[i], as = AS.r[i], cz = C.r[i];
                gl(a.out[0])[base + z] = float2{(float)ds.x, (float)ds.y};
                gl(a.out[1])[base + z] = float2{(float)as.x, (float)as.y};
                gl(a.out[2])[base + z] = float2{(float)cz.x, (float)cz.y};
                // the source of the vertical velocity (inversion.f90:97-150)
                const double2 dy_ = muli(SX.r[i], iky), dx_ = muli(SY.r[i], ikx);
                DS.r[i] = double2{dy_.x - dx_.x, dy_.y - dx_.y};
            }
            ds0 = DS.low();
            dsn = DS.top();
            ZALL(i, z)
            {
                // es = ds(0) dtheta_-(z) + ds(nz) dtheta_+(z)
                double dtm = 0.0, dtp = 0.0;
                if (!zero_mode) {
                    double zm, zp;
                    zcoord(z, zm, zp);
                    const double Lm = kl * zm, Lp = kl * zp;
                    const double ep = exp(-Lp), em = exp(-Lm);
                    const double dpm = -kl * dv * (ep + ef * em), dpp = kl * dv * (em + ef * ep);
                    dtm = -k2ifac * ((Q * Lp - 1.0) * dpm - Rr * Lm * dpp);
                    dtp = -k2ifac * ((Q * Lm - 1.0) * dpp - Rr * Lp * dpm);
                }
                E.r[i] = double2{ds0.x * dtm + dsn.x * dtp, ds0.y * dtm + dsn.y * dtp};
                if (i < NS) {
                    const double rz = scz * (double)z;
                    const double green = -1.0 / (k2l2 + rz * rz);
                    const double2 ds = DS.r[i];
                    const double2 gd = double2{green * ds.x, green * ds.y};
                    DS.r[i] = gd;
                    AS.r[i] = double2{rz * gd.x, rz * gd.y};
                } else {
                    AS.r[i] = double2{0.0, 0.0};
                }
            }
        } else if (ph == VELOCITY) {   // w and dw/dz
            get_even(line[0], AS);
            get_odd(line[1], DS, false);
            DS.r[NS] = double2{0.0, 0.0};
            ZIN(i, z)
            {
                double tm = 0.0, tp = 0.0;   // bs = ds(0) theta_-(z) + ds(nz) theta_+(z)
                if (!zero_mode) {
                    double zm, zp;
                    zcoord(z, zm, zp);
                    const double Lm = kl * zm, Lp = kl * zp;
                    const double pm = phim[i], pp = phip[i];
                    tm = k2ifac * (Rr * Lm * pp - Q * Lp * pm);
                    tp = k2ifac * (Rr * Lp * pm - Q * Lm * pp);
                }
                const double2 ds = DS.r[i];
                DS.r[i] = double2{ds.x + (ds0.x * tm + dsn.x * tp), ds.y + (ds0.y * tm + dsn.y * tp)};
            }
#pragma unroll
            for (int i = 0; i <= NS; ++i) E.r[i] = double2{E.r[i].x + AS.r[i].x, E.r[i].y + AS.r[i].y};   // dw/dz
            if (zero_mode) {   // horizontally averaged flow (inversion.f90:161-176)
                mb[0] = SY.low();
                mb[1] = SY.top();
                mb[2] = SX.low();
                mb[3] = SX.top();
                AS.r[NS] = SX.r[NS] = double2{0.0, 0.0};
                ZIN(i, z)
                {
                    const double rzi = 1.0 / (scz * (double)z);
                    const double2 sy = SY.r[i], sx = SX.r[i];
                    AS.r[i] = double2{-rzi * sy.x, -rzi * sy.y};   // ubar
                    SX.r[i] = double2{rzi * sx.x, rzi * sx.y};     // vbar
                }
            }
        } else {
            get_even(line[0], AS);
            get_even(line[1], SX);
            const double2 y0 = mb[0], yn = mb[1], x0 = mb[2], xn = mb[3];
            ZALL(i, z)
            {
                double zm, zp;
                zcoord(z, zm, zp);
                const double pt = zp / Lz;
                double zm2, zp2;
                zcoord(nz - z, zm2, zp2);
                const double pb = zp2 / Lz;
                const double gt = 0.5 * Lz * (pt * pt - 1.0 / 3.0);
                const double gb = 0.5 * Lz * (pb * pb - 1.0 / 3.0);
                const double2 as = AS.r[i], sx = SX.r[i];
                AS.r[i] = double2{as.x + yn.x * gt - y0.x * gb, as.y + yn.y * gt - y0.y * gb};
                SX.r[i] = double2{sx.x - xn.x * gt + x0.x * gb, sx.y - xn.y * gt + x0.y * gb};
            }
        }
        __syncthreads();   // the lines are read before the next phase writes them
    }

    // ---- u, v, w and the velocity-gradient spectra (inversion.f90:180-233, 259-317) ----
    ZALL(i, z)
    {
        double2 u, v;
        if (zero_mode) {
            u = AS.r[i];
            v = SX.r[i];
        } else {
            const double2 e = E.r[i], cz = C.r[i];
            const double2 ex = muli(e, ikx), ey = muli(e, iky), cx = muli(cz, ikx), cy = muli(cz, iky);
            u = double2{k2l2i * (ex.x + cy.x), k2l2i * (ex.y + cy.y)};
            v = double2{k2l2i * (ey.x - cx.x), k2l2i * (ey.y - cx.y)};
        }
        const double2 w = DS.r[i];
        auto st = [&](int o, double2 val) { gl(a.out[o])[base + z] = float2{(float)val.x, (float)val.y}; };
        st(3, u);
        st(4, v);
        st(5, w);
        st(6, muli(u, ikx));    // du/dx
        st(7, muli(u, iky));    // du/dy
        st(8, muli(v, iky));    // dv/dy
        st(9, muli(w, ikx));    // dw/dx
        st(10, muli(w, iky));   // dw/dy
    }
}
#undef ZIN
#undef ZBND
#undef ZALL

// (the slot loops of the LDS form, NS == 0, have a run-time trip count: no
// full unrolling there)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wpass-failed"
// One transform after the other, each inlined: for columns of three slots, whose
// arrays all live across the phase loop above would leave one wave per SIMD
// (with three slots a launch took 236 us at 128^3, 157 here), and for the LDS
// form.
template <int NS>
__global__ __launch_bounds__(64) void k_vor2vel_columns_seq(const ColArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const ColArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int nz = g.nz, nz1 = nz + 1;
    const int nsl = NS > 0 ? NS : (nz1 + 63) / 64;
    const int col = ib.blk;
    const int kx = col % g.nxh, ky = col / g.nxh;
    const bool zero_mode = (kx == 0 && ky == 0);

    extern __shared__ double2 sm[];
    ZCol<NS, double2> SX, SY, C, E, DS, AS;
    ZCol<NS, double> phim, phip;
    double2 *fa, *fb;
    if constexpr (NS > 0) {
        fa = sm;
        fb = fa + 2 * nz;
    } else {
        SX.l = sm;
        SY.l = SX.l + nz1;
        C.l = SY.l + nz1;
        E.l = C.l + nz1;
        DS.l = E.l + nz1;
        AS.l = DS.l + nz1;
        fa = AS.l + nz1;
        fb = fa + 2 * nz;
        phim.l = (double *)(fb + 2 * nz);
        phip.l = phim.l + nz1;
    }
    ColCtx cc{nz, fa, fb, &a.zplan, a.ztw};   // twiddles from global memory (cached)

    // wavenumbers (sta3dfft.f90:88-107, sta2dfft.f90:59-64): r = (pi/L) 2k
    const int kys = (2 * ky <= g.ny) ? ky : ky - g.ny;
    const double scx = EPIC_PI / g.extent[0], scy = EPIC_PI / g.extent[1], scz = EPIC_PI / g.extent[2];
    const double rkx = scx * (double)(2 * kx), rky = scy * (double)(2 * (kys < 0 ? -kys : kys));
    const double ikx = (2 * kx == g.nx) ? 0.0 : rkx;                       // diffx factor
    const double iky = (2 * ky == g.ny) ? 0.0 : (kys < 0 ? -rky : rky);   // diffy factor
    const double k2l2 = rkx * rkx + rky * rky;
    const double k2l2i = zero_mode ? 0.0 : 1.0 / k2l2;
    // Hou & Li filter (inversion_utils.f90:130-150)
    const double kxmaxi = 1.0 / (scx * (double)g.nx), kymaxi = 1.0 / (scy * (double)g.ny);
    const double kzmaxi = 1.0 / (scz * (double)nz);
    const double fh = exp(-36.0 * pow36(kxmaxi * rkx) + -36.0 * pow36(kymaxi * rky));
    // hyperbolic functions (inversion_utils.f90:305-351)
    const double Lz = g.extent[2];
    const double kl = sqrt(k2l2);
    const double ef = exp(-kl * Lz);
    const double dv = 1.0 / (1.0 - ef * ef);
    const double Q = dv * (1.0 + ef * ef), Rr = dv * 2.0 * ef, k2ifac = 0.5 * k2l2i;

    auto zcoord = [&](int iz, double &zm, double &zp) {
        const double z = g.lower[2] + g.dx[2] * (double)iz;
        zm = g.upper[2] - z;
        zp = z - g.lower[2];
    };

    // ---- load the three vorticity spectra and the phi tables ----
    const int64_t base = ((int64_t)ky * g.nxh + kx) * g.nzp;
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            const float2 x = gl(a.in[0])[base + z], y = gl(a.in[1])[base + z], w = gl(a.in[2])[base + z];
            SX(i, z) = double2{x.x, x.y};
            SY(i, z) = double2{y.x, y.y};
            C(i, z) = double2{w.x, w.y};
            double zm, zp;
            zcoord(z, zm, zp);
            if (zero_mode) {
                phim(i, z) = zm / Lz;
                phip(i, z) = zp / Lz;
            } else {
                const double ep = exp(-(kl * zp)), em = exp(-(kl * zm));
                phim(i, z) = dv * (ep - ef * em);
                phip(i, z) = dv * (em - ef * ep);
            }
        }
    }
    __syncthreads();

    // ---- decompose + filter (inversion.f90:40-43) ----
    decompose(cc, SX, phim, phip, nsl);
    decompose(cc, SY, phim, phip, nsl);
    decompose(cc, C, phim, phip, nsl);
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            double f = fh;
            if (z > 0 && z < nz) f = fh * exp(-36.0 * pow36(kzmaxi * (scz * (double)z)));
            if (zero_mode) f = 1.0;
            const double2 sx = SX(i, z), sy = SY(i, z), cz = C(i, z);
            SX(i, z) = double2{f * sx.x, f * sx.y};
            SY(i, z) = double2{f * sy.x, f * sy.y};
            C(i, z) = double2{f * cz.x, f * cz.y};
        }
    }
    __syncthreads();

    // ---- solenoidal projection (inversion.f90:50-87) ----
    combine(cc, C, phim, phip, nsl);   // zeta, semi-spectral
    {
        // neighbours through the FFT buffer
        ZSLOTS(i, z)
        {
            if (z < nz1) fa[z] = C(i, z);
        }
        __syncthreads();
        const double dzi = g.dxi[2], hdzi = 0.5 * g.dxi[2];
        ZSLOTS(i, z)
        {
            if (z < nz1) {
                double2 d;
                if (z == 0) d = double2{dzi * (fa[1].x - fa[0].x), dzi * (fa[1].y - fa[0].y)};
                else if (z == nz) d = double2{dzi * (fa[nz].x - fa[nz - 1].x), dzi * (fa[nz].y - fa[nz - 1].y)};
                else d = double2{(fa[z + 1].x - fa[z - 1].x) * hdzi, (fa[z + 1].y - fa[z - 1].y) * hdzi};
                E(i, z) = d;
            }
        }
        __syncthreads();
    }
    decompose(cc, E, phim, phip, nsl);
    if (!zero_mode) {
        ZSLOTS(i, z)
        {
            if (z < nz1) {
                // D = B_x - A_y;  A = k2l2i (E_x + D_y), B = k2l2i (E_y - D_x)
                const double2 sx = SX(i, z), sy = SY(i, z), e = E(i, z);
                const double2 d = double2{muli(sy, ikx).x - muli(sx, iky).x, muli(sy, ikx).y - muli(sx, iky).y};
                const double2 ex = muli(e, ikx), ey = muli(e, iky), dx_ = muli(d, ikx), dy_ = muli(d, iky);
                SX(i, z) = double2{k2l2i * (ex.x + dy_.x), k2l2i * (ex.y + dy_.y)};
                SY(i, z) = double2{k2l2i * (ey.x - dx_.x), k2l2i * (ey.y - dx_.y)};
            }
        }
    }
    __syncthreads();

    // ---- filtered solenoidal vorticity (inversion.f90:91-93) ----
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            DS(i, z) = SX(i, z);
            AS(i, z) = SY(i, z);
        }
    }
    __syncthreads();
    combine(cc, DS, phim, phip, nsl);
    combine(cc, AS, phim, phip, nsl);
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            const double2 ds = DS(i, z), as = AS(i, z), cz = C(i, z);
            gl(a.out[0])[base + z] = float2{(float)ds.x, (float)ds.y};
            gl(a.out[1])[base + z] = float2{(float)as.x, (float)as.y};
            gl(a.out[2])[base + z] = float2{(float)cz.x, (float)cz.y};
        }
    }
    __syncthreads();

    // ---- vertical velocity (inversion.f90:97-150) ----
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            const double2 dy_ = muli(SX(i, z), iky), dx_ = muli(SY(i, z), ikx);
            DS(i, z) = double2{dy_.x - dx_.x, dy_.y - dx_.y};
        }
    }
    __syncthreads();
    const double2 ds0 = zval(DS, 0), dsn = zval(DS, nz);
    __syncthreads();
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            // es = ds(0) dtheta_-(z) + ds(nz) dtheta_+(z)
            double dtm = 0.0, dtp = 0.0;
            if (!zero_mode) {
                double zm, zp;
                zcoord(z, zm, zp);
                const double Lm = kl * zm, Lp = kl * zp;
                const double ep = exp(-Lp), em = exp(-Lm);
                const double dpm = -kl * dv * (ep + ef * em), dpp = kl * dv * (em + ef * ep);
                dtm = -k2ifac * ((Q * Lp - 1.0) * dpm - Rr * Lm * dpp);
                dtp = -k2ifac * ((Q * Lm - 1.0) * dpp - Rr * Lp * dpm);
            }
            E(i, z) = double2{ds0.x * dtm + dsn.x * dtp, ds0.y * dtm + dsn.y * dtp};
            if (z > 0 && z < nz) {
                const double rz = scz * (double)z;
                const double green = -1.0 / (k2l2 + rz * rz);
                const double2 ds = DS(i, z);
                const double2 gd = double2{green * ds.x, green * ds.y};
                DS(i, z) = gd;
                AS(i, z) = double2{rz * gd.x, rz * gd.y};
            } else {
                AS(i, z) = double2{0.0, 0.0};
            }
        }
    }
    __syncthreads();
    zdct(cc, AS, nsl);
    zdst(cc, DS, nsl);
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            if (z == 0 || z == nz) {
                DS(i, z) = double2{0.0, 0.0};
            } else {
                double tm = 0.0, tp = 0.0;   // bs = ds(0) theta_-(z) + ds(nz) theta_+(z)
                if (!zero_mode) {
                    double zm, zp;
                    zcoord(z, zm, zp);
                    const double Lm = kl * zm, Lp = kl * zp;
                    const double ep = exp(-Lp), em = exp(-Lm);
                    const double pm = dv * (ep - ef * em), pp = dv * (em - ef * ep);
                    tm = k2ifac * (Rr * Lm * pp - Q * Lp * pm);
                    tp = k2ifac * (Rr * Lp * pm - Q * Lm * pp);
                }
                const double2 ds = DS(i, z);
                DS(i, z) = double2{ds.x + (ds0.x * tm + dsn.x * tp), ds.y + (ds0.y * tm + dsn.y * tp)};
            }
            const double2 e = E(i, z), as = AS(i, z);
            E(i, z) = double2{e.x + as.x, e.y + as.y};   // dw/dz
        }
    }
    __syncthreads();

    // ---- horizontally averaged flow (inversion.f90:161-176) ----
    if (zero_mode) {
        const double2 y0 = zval(SY, 0), yn = zval(SY, nz), x0 = zval(SX, 0), xn = zval(SX, nz);
        __syncthreads();
        ZSLOTS(i, z)
        {
            if (z < nz1) {
                if (z == 0 || z == nz) {
                    AS(i, z) = double2{0.0, 0.0};
                    SX(i, z) = double2{0.0, 0.0};
                } else {
                    const double rzi = 1.0 / (scz * (double)z);
                    const double2 sy = SY(i, z), sx = SX(i, z);
                    AS(i, z) = double2{-rzi * sy.x, -rzi * sy.y};   // ubar
                    SX(i, z) = double2{rzi * sx.x, rzi * sx.y};     // vbar
                }
            }
        }
        __syncthreads();
        zdct(cc, AS, nsl);
        zdct(cc, SX, nsl);
        ZSLOTS(i, z)
        {
            if (z < nz1) {
                double zm, zp;
                zcoord(z, zm, zp);
                const double pt = zp / Lz;
                double zm2, zp2;
                zcoord(nz - z, zm2, zp2);
                const double pb = zp2 / Lz;
                const double gt = 0.5 * Lz * (pt * pt - 1.0 / 3.0);
                const double gb = 0.5 * Lz * (pb * pb - 1.0 / 3.0);
                const double2 as = AS(i, z), sx = SX(i, z);
                AS(i, z) = double2{as.x + yn.x * gt - y0.x * gb, as.y + yn.y * gt - y0.y * gb};
                SX(i, z) = double2{sx.x - xn.x * gt + x0.x * gb, sx.y - xn.y * gt + x0.y * gb};
            }
        }
        __syncthreads();
    }

    // ---- u, v, w and the velocity-gradient spectra (inversion.f90:180-233, 259-317) ----
    ZSLOTS(i, z)
    {
        if (z < nz1) {
            double2 u, v;
            if (zero_mode) {
                u = AS(i, z);
                v = SX(i, z);
            } else {
                const double2 e = E(i, z), cz = C(i, z);
                const double2 ex = muli(e, ikx), ey = muli(e, iky), cx = muli(cz, ikx), cy = muli(cz, iky);
                u = double2{k2l2i * (ex.x + cy.x), k2l2i * (ex.y + cy.y)};
                v = double2{k2l2i * (ey.x - cx.x), k2l2i * (ey.y - cx.y)};
            }
            const double2 w = DS(i, z);
            auto st = [&](int o, double2 val) { gl(a.out[o])[base + z] = float2{(float)val.x, (float)val.y}; };
            st(3, u);
            st(4, v);
            st(5, w);
            st(6, muli(u, ikx));    // du/dx
            st(7, muli(u, iky));    // du/dy
            st(8, muli(v, iky));    // dv/dy
            st(9, muli(w, ikx));    // dw/dx
            st(10, muli(w, iky));   // dw/dy
        }
    }
}
#pragma clang diagnostic pop
#undef ZSLOTS

// the column form for nz: 1 and 2 the phase form with that many slots of inner
// values, 3 the register slots of nz + 1 values, 0 the LDS form
static int col_slots(const Grid &g)
{
    if (g.nz <= 64 * COL_PHASE_SLOTS) return (g.nz + 63) / 64;
    return g.nz + 1 <= 64 * COL_REG_SLOTS ? COL_REG_SLOTS : 0;
}

size_t col_lds_bytes(const Grid &g)
{
    const int nz1 = g.nz + 1;
    const int ns = col_slots(g);
    if (ns > 0 && ns <= COL_PHASE_SLOTS) return (size_t)7 * g.nz * sizeof(double2);   // three lines of 2 nz points, nz twiddles
    const size_t fft = (size_t)4 * g.nz * sizeof(double2);   // the two FFT buffers of 2 nz points
    if (ns > 0) return fft;
    return (size_t)6 * nz1 * sizeof(double2) + fft + 2 * (size_t)nz1 * sizeof(double);
}

// one launch per column form present (members of one batch may differ in nz)
void add_vor2vel_columns(Plan &P, int phase, const std::vector<ColArgs> &items)
{
    static const void *const kern[COL_REG_SLOTS + 1] = {(const void *)k_vor2vel_columns_seq<0>,
                                                        (const void *)k_vor2vel_columns<1>,
                                                        (const void *)k_vor2vel_columns<2>,
                                                        (const void *)k_vor2vel_columns_seq<3>};
    for (int ns = 0; ns <= COL_REG_SLOTS; ++ns) {
        std::vector<ColArgs> sel;
        std::vector<int> nb;
        size_t lds = 0;
        for (const ColArgs &a : items) {
            if (col_slots(a.g) != ns) continue;
            sel.push_back(a);
            nb.push_back(a.g.ny * a.g.nxh);
            lds = std::max(lds, col_lds_bytes(a.g));
        }
        if (!sel.empty()) P.add(kern[ns], 64, lds, phase, sel, nb);
    }
}

}  // namespace epic
