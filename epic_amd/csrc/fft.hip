// Horizontal 2D real FFTs of the node planes z = 0..nz (FP32), the transform
// pair of fftxyp2s / fftxys2p (sta3dfft.f90:134-257) in complex half-spectrum
// form: S(kx, ky) = sum_{i,j} f(i, j) e^{-2 pi i (kx i/nx + ky j/ny)},
// kx in [0, nx/2].  The inverse carries the 1/(nx ny) normalisation.
//
// Two passes per direction (one launch for both where a plane fits LDS, the last
// section); the intermediate T[j][kx][z] and the spectra
// S[ky][kx][z] keep ZB consecutive z planes contiguous, so every pass moves
// 128-byte segments and the vertical (z) column kernels read whole columns.
//
// The parcel correction's source volg / vcell - 1 is formed in the forward x
// pass's loader.
//
// Lines lie one point apart from a multiple of 32 banks in LDS where they are
// read or written across (16 z of one point): at power-of-two lengths those
// accesses met one bank 16 ways.
#include "common.h"
#include "fft.h"
#include "launch.h"

#include <algorithm>

namespace epic {

// ---------------------------------------------------------------------------
// forward x pass: real rows -> half spectra
// ---------------------------------------------------------------------------
// The global -> LDS staging loops below request LOAD_BATCH elements per
// thread before the first LDS store, with clamped (always valid) addresses
// and no branches between the loads, so a thread waits one memory round
// trip per batch rather than one per element.
constexpr int LOAD_BATCH = 8;

// forward x input value at node offset o (mode fixed per launch item)
enum XfKind { XF_FIELD, XF_PHI };
template <int KIND> __device__ inline float phys_value(const FftXArgs &a, int64_t o, int64_t FS)
{
    // parcel-correction source: volg / vcell - 1
    if constexpr (KIND == XF_PHI) return gl(a.fld)[F_VOLG * FS + o] * (float)(1.0 / a.g.vcell) - 1.0f;
    return gl(a.fld)[a.slot * FS + o];
}

// ZB rows of nx reals (planes zp0.., row j) packed as m = nx/2 complex
// values per row into buf[r (m + 1) + q]; planes above nz are zero
template <int KIND> __device__ inline void stage_rows(const FftXArgs &a, float2 *buf, int j, int zp0, int m)
{
    const Grid &g = a.g;
    const int nz = g.nz;
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    const int total = ZB * m;
    for (int t0 = threadIdx.x; t0 < total; t0 += LOAD_BATCH * blockDim.x) {
        float2 z[LOAD_BATCH];
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = min(t0 + u * (int)blockDim.x, total - 1);
            const int r = fdiv(t, a.plan.n1), q = t - r * m;   // the x plan's length is m
            const int64_t o = (int64_t)(min(zp0 + r, nz) + 1) * PS + (int64_t)j * g.nx + 2 * q;
            z[u] = float2{phys_value<KIND>(a, o, FS), phys_value<KIND>(a, o + 1, FS)};
        }
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = t0 + u * blockDim.x, r = fdiv(min(t, total - 1), a.plan.n1);
            if (t < total) buf[t + r] = (zp0 + r <= nz) ? z[u] : float2{0, 0};
        }
    }
}

// ZB z-contiguous spectra columns: buf[r * ls + c] = in[(c * stride + col) * nzp + zp0 + r]
// for c < len
__device__ inline void stage_columns(const float2 *in, float2 *buf, int len, int ls, int64_t stride, int col, const Grid &g, int zp0)
{
    const int total = ZB * len;
    for (int t0 = threadIdx.x; t0 < total; t0 += LOAD_BATCH * blockDim.x) {
        float2 v[LOAD_BATCH];
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = min(t0 + u * (int)blockDim.x, total - 1);
            const int c = t / ZB, r = t - c * ZB;
            v[u] = gl(in)[((int64_t)c * stride + col) * g.nzp + zp0 + r];
        }
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = t0 + u * blockDim.x, c = t / ZB, r = t - c * ZB;
            if (t < total) buf[r * ls + c] = v[u];
        }
    }
}

// X_k of a real line from its packed transform at k and m - k; w = e^{-2 pi i k / nx}
__device__ inline float2 untangled(float2 zk, float2 zc, float2 w)
{
    const float2 s = cadd(zk, zc), d = csub(zk, zc);
    const float2 wd = cmul(w, d);
    return float2{0.5f * (s.x + wd.y), 0.5f * (s.y - wd.x)};   // (s - i w d) / 2
}
// and the packed transform (twice it) from X_k and X_{m-k}
__device__ inline float2 tangled(float2 xk, float2 xc, float2 tw)
{
    const float2 w = cconj(tw);   // e^{+2 pi i k / nx}
    const float2 s = cadd(xk, xc), d = csub(xk, xc);
    const float2 wd = cmul(w, d);
    return float2{s.x - wd.y, s.y + wd.x};   // s + i w d
}

__global__ __launch_bounds__(256) void k_fft_xf(const FftXArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const FftXArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int j = ib.blk % g.ny;
    const int zp0 = (ib.blk / g.ny) * ZB;
    const int m = g.nx / 2;
    extern __shared__ float2 lds[];
    float2 *bufa = lds, *bufb = lds + ZB * (m + 1);
    float2 *tw = bufb + ZB * (m + 1);   // twiddles staged in LDS
    for (int t = threadIdx.x; t < g.nx; t += blockDim.x) tw[t] = gl(a.tw)[t];
    if (a.mode == 3) stage_rows<XF_PHI>(a, bufa, j, zp0, m);
    else stage_rows<XF_FIELD>(a, bufa, j, zp0, m);
    __syncthreads();
    float2 *Z = lds_fft(bufa, bufb, ZB, a.plan, tw, 2, false, m + 1);
    float2 *other = (Z == bufa) ? bufb : bufa;
    // untangle the packed real transform: X_k, k = 0..m
    for (int t = threadIdx.x; t < ZB * (m + 1); t += blockDim.x) {
        const int kx = t / ZB, r = t - kx * ZB;
        const float2 zk = Z[r * (m + 1) + (kx == m ? 0 : kx)];              // kx mod m, kx in [0, m]
        const float2 zc = cconj(Z[r * (m + 1) + (kx == 0 ? 0 : m - kx)]);   // (m - kx) mod m
        other[r * (m + 1) + kx] = untangled(zk, zc, tw[kx]);
    }
    __syncthreads();
    const int nxh = m + 1;
    for (int t = threadIdx.x; t < ZB * nxh; t += blockDim.x) {
        const int kx = t / ZB, r = t - kx * ZB;
        gl(a.out)[((int64_t)j * nxh + kx) * g.nzp + zp0 + r] = other[r * (m + 1) + kx];
    }
}

// ---------------------------------------------------------------------------
// y pass (c2c), forward or inverse
// ---------------------------------------------------------------------------
// in place is allowed (out == in): a block reads and writes only its own
// (kx, z block) slab
__global__ __launch_bounds__(256) void k_fft_y(const FftYArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const FftYArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int kx = ib.blk % g.nxh;
    const int zp0 = (ib.blk / g.nxh) * ZB;
    const int ny = g.ny, nxh = g.nxh;
    extern __shared__ float2 lds[];
    float2 *bufa = lds, *bufb = lds + ZB * (ny + 1);
    float2 *tw = bufb + ZB * (ny + 1);   // twiddles staged in LDS
    for (int t = threadIdx.x; t < ny; t += blockDim.x) tw[t] = gl(a.tw)[t];
    stage_columns(a.in, bufa, ny, ny + 1, nxh, kx, g, zp0);
    __syncthreads();
    float2 *Rb = lds_fft(bufa, bufb, ZB, a.plan, tw, 1, a.mode != 0, ny + 1);
    for (int t = threadIdx.x; t < ZB * ny; t += blockDim.x) {
        const int jy = t / ZB, r = t - jy * ZB;
        gl(a.out)[((int64_t)jy * nxh + kx) * g.nzp + zp0 + r] = Rb[r * (ny + 1) + jy];
    }
}

// ---------------------------------------------------------------------------
// inverse x pass: half spectra -> real rows
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_fft_xi(const FftXArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const FftXArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int j = ib.blk % g.ny;
    const int zp0 = (ib.blk / g.ny) * ZB;
    const int m = g.nx / 2, nxh = m + 1;
    extern __shared__ float2 lds[];
    float2 *bufa = lds, *bufb = lds + ZB * (m + 1);
    float2 *tw = bufb + ZB * (m + 1);   // twiddles staged in LDS
    for (int t = threadIdx.x; t < g.nx; t += blockDim.x) tw[t] = gl(a.tw)[t];
    stage_columns(a.in, bufb, nxh, nxh, 1, j * nxh, g, zp0);
    __syncthreads();
    for (int t = threadIdx.x; t < ZB * m; t += blockDim.x) {
        const int r = fdiv(t, a.plan.n1), k = t - r * m;
        const float2 xk = bufb[r * nxh + k];
        const float2 xc = cconj(bufb[r * nxh + (m - k)]);
        bufa[r * m + k] = tangled(xk, xc, tw[k]);
    }
    __syncthreads();
    float2 *Z = lds_fft(bufa, bufb, ZB, a.plan, tw, 2, true, m);
    const float scale = 1.0f / ((float)g.nx * (float)g.ny);
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    for (int t = threadIdx.x; t < ZB * g.nx; t += blockDim.x) {
        const int r = fdiv(t, a.plan.n2), i = t - r * g.nx;   // 2 m = nx
        if (zp0 + r > g.nz) continue;
        const float2 z = Z[r * m + (i >> 1)];
        gl(a.fld_out)[a.slot * FS + (int64_t)(zp0 + r + 1) * PS + (int64_t)j * g.nx + i] = ((i & 1) ? z.y : z.x) * scale;
    }
}

// ---------------------------------------------------------------------------
// both passes of a direction in one launch, for planes that fit LDS
// ---------------------------------------------------------------------------
// A block takes PZ whole planes of one component (z pairs of the spectra are 16
// bytes; more planes a block leave CUs without one).  The x lines (plane, j) and
// the y lines (plane, kx) share two buffers; the untangling of the packed real
// transform moves a row into the y lines.  The operations on a line are those
// of the separate passes, so the results are the same bits.
constexpr int PZ = 2;
struct PlaneShape {
    int m, nxh, lx, ly, size;   // packed length, half spectrum, line pitches, points of a buffer per plane
};
__host__ __device__ inline PlaneShape plane_shape(const Grid &g)
{
    const int m = g.nx / 2, lx = m + 1, ly = g.ny | 1;
    const int x = g.ny * lx, y = (m + 1) * ly;
    return PlaneShape{m, m + 1, lx, ly, x > y ? x : y};
}

__global__ __launch_bounds__(1024) void k_fft_planes_f(const FftPlaneArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const FftPlaneArgs &a = tab[ib.item];
    const Grid &g = a.x.g;
    const PlaneShape s = plane_shape(g);
    const int zp0 = ib.blk * PZ, L = min(PZ, g.nz + 1 - zp0), ny = g.ny, m = s.m;
    extern __shared__ float2 lds[];
    float2 *bufa = lds, *bufb = lds + PZ * s.size, *twx = bufb + PZ * s.size, *twy = twx + g.nx;
    for (int t = threadIdx.x; t < g.nx; t += blockDim.x) twx[t] = gl(a.x.tw)[t];
    for (int t = threadIdx.x; t < ny; t += blockDim.x) twy[t] = gl(a.y.tw)[t];
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    const int rows = L * ny, total = rows * m;   // the rows of consecutive planes are consecutive
    for (int t0 = threadIdx.x; t0 < total; t0 += LOAD_BATCH * blockDim.x) {
        float2 z[LOAD_BATCH];
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = min(t0 + u * (int)blockDim.x, total - 1);
            const int64_t o = (int64_t)(zp0 + 1) * PS + 2 * t;
            if (a.x.mode == 3) z[u] = float2{phys_value<XF_PHI>(a.x, o, FS), phys_value<XF_PHI>(a.x, o + 1, FS)};
            else z[u] = float2{phys_value<XF_FIELD>(a.x, o, FS), phys_value<XF_FIELD>(a.x, o + 1, FS)};
        }
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = t0 + u * blockDim.x;
            if (t < total) bufa[t + fdiv(t, a.x.plan.n1)] = z[u];   // row lx + q
        }
    }
    __syncthreads();
    float2 *Z = lds_fft(bufa, bufb, rows, a.x.plan, twx, 2, false, s.lx);
    float2 *Y = (Z == bufa) ? bufb : bufa;
    for (int t = threadIdx.x; t < rows * s.nxh; t += blockDim.x) {
        const int row = fdiv(t, a.nxh), kx = t - row * s.nxh, r = fdiv(row, a.y.plan.n1), j = row - r * ny;
        const float2 zk = Z[row * s.lx + (kx == m ? 0 : kx)];
        const float2 zc = cconj(Z[row * s.lx + (kx == 0 ? 0 : m - kx)]);
        Y[(r * s.nxh + kx) * s.ly + j] = untangled(zk, zc, twx[kx]);
    }
    __syncthreads();
    float2 *R = lds_fft(Y, Z, L * s.nxh, a.y.plan, twy, 1, false, s.ly);
    // (z fastest: whole lines of the spectra are written by neighbouring lanes)
    for (int t = threadIdx.x; t < PZ * s.nxh * ny; t += blockDim.x) {
        const int c = t / PZ, r = t - c * PZ, j = fdiv(c, a.nxh), kx = c - j * s.nxh;
        if (r < L) gl(a.y.out)[(int64_t)c * g.nzp + zp0 + r] = R[(r * s.nxh + kx) * s.ly + j];
    }
}

__global__ __launch_bounds__(1024) void k_fft_planes_i(const FftPlaneArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const FftPlaneArgs &a = tab[ib.item];
    const Grid &g = a.x.g;
    const PlaneShape s = plane_shape(g);
    const int zp0 = ib.blk * PZ, L = min(PZ, g.nz + 1 - zp0), ny = g.ny, m = s.m;
    extern __shared__ float2 lds[];
    float2 *bufa = lds, *bufb = lds + PZ * s.size, *twx = bufb + PZ * s.size, *twy = twx + g.nx;
    for (int t = threadIdx.x; t < g.nx; t += blockDim.x) twx[t] = gl(a.x.tw)[t];
    for (int t = threadIdx.x; t < ny; t += blockDim.x) twy[t] = gl(a.y.tw)[t];
    const int total = PZ * s.nxh * ny;
    for (int t0 = threadIdx.x; t0 < total; t0 += LOAD_BATCH * blockDim.x) {
        float2 v[LOAD_BATCH];
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = min(t0 + u * (int)blockDim.x, total - 1), c = t / PZ, r = t - c * PZ;
            v[u] = gl(a.y.in)[(int64_t)c * g.nzp + zp0 + min(r, L - 1)];
        }
#pragma unroll
        for (int u = 0; u < LOAD_BATCH; ++u) {
            const int t = t0 + u * blockDim.x, c = t / PZ, r = t - c * PZ, j = fdiv(c, a.nxh), kx = c - j * s.nxh;
            if (t < total && r < L) bufa[(r * s.nxh + kx) * s.ly + j] = v[u];
        }
    }
    __syncthreads();
    float2 *Y = lds_fft(bufa, bufb, L * s.nxh, a.y.plan, twy, 1, true, s.ly);
    float2 *X = (Y == bufa) ? bufb : bufa;
    const int rows = L * ny;
    for (int t = threadIdx.x; t < rows * m; t += blockDim.x) {
        const int row = fdiv(t, a.x.plan.n1), k = t - row * m, r = fdiv(row, a.y.plan.n1), j = row - r * ny;
        const float2 *line = Y + r * s.nxh * s.ly + j;
        X[row * m + k] = tangled(line[k * s.ly], cconj(line[(m - k) * s.ly]), twx[k]);
    }
    __syncthreads();
    float2 *Z = lds_fft(X, Y, rows, a.x.plan, twx, 2, true, m);
    const float scale = 1.0f / ((float)g.nx * (float)g.ny);
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    EPIC_GLOBAL float *out = gl(a.x.fld_out) + a.x.slot * FS + (int64_t)(zp0 + 1) * PS;
    for (int t = threadIdx.x; t < rows * g.nx; t += blockDim.x) {
        const float2 z = Z[t >> 1];
        out[t] = ((t & 1) ? z.y : z.x) * scale;
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static size_t x_lds(const Grid &g) { return (2 * ZB * (size_t)(g.nx / 2 + 1) + g.nx) * sizeof(float2); }
static size_t y_lds(const Grid &g) { return (2 * ZB * (size_t)(g.ny + 1) + g.ny) * sizeof(float2); }

// The grids accepted are those whose ZB lines of nx/2 + 1 and of ny points fit
// a work-group's LDS twice at FP64: more than any of the transforms takes
size_t transform_lds_bytes(const Grid &g)
{
    const size_t x = 2 * ZB * (size_t)(g.nx / 2 + 1) + g.nx, y = 2 * ZB * (size_t)g.ny + g.ny;
    return std::max(std::max(x, y) * sizeof(double2), col_lds_bytes(g));
}

static size_t planes_lds(const Grid &g)
{
    return (2 * (size_t)PZ * plane_shape(g).size + g.nx + g.ny) * sizeof(float2);
}
// One launch where two blocks share a CU's LDS (up to 64 x 64): vor2vel takes
// 49 -> 44 us at 16^3, 55.5 -> 49.6 at 32^3, 65 -> 64 at 48x48x32 and 95.3 -> 93.2 at
// 64^3.  Larger planes leave too few blocks (single planes: 129 -> 138 us at
// 128x64x64); with four planes a block 45.0, 52.4, 64.1 and 94.1 us.
static bool planes_fit(const Grid &g) { return planes_lds(g) <= (80 << 10); }
static void add_planes(Plan &P, int phase, const void *kernel, const std::vector<FftPlaneArgs> &items)
{
    if (items.empty()) return;
    std::vector<int> nb;
    size_t lds = 0;
    int pts = 0;
    for (const FftPlaneArgs &a : items) {
        const Grid &g = a.x.g;
        nb.push_back((g.nz + PZ) / PZ);
        lds = std::max(lds, planes_lds(g));
        pts = std::max(pts, PZ * g.ny * plane_shape(g).nxh);
    }
    P.add(kernel, pts > 2048 ? 1024 : pts > 1024 ? 512 : 256, lds, phase, items, nb);
}
static void add_fft_xf(Plan &P, int phase, const std::vector<FftXArgs> &items)
{
    std::vector<int> nb;
    size_t lds = 0;
    for (const FftXArgs &a : items) {
        nb.push_back(a.g.ny * (a.g.nzp / ZB));
        lds = std::max(lds, x_lds(a.g));
    }
    P.add((const void *)k_fft_xf, 256, lds, phase, items, nb);
}

static void add_fft_y(Plan &P, int phase, const std::vector<FftYArgs> &items)
{
    std::vector<int> nb;
    size_t lds = 0;
    for (const FftYArgs &a : items) {
        nb.push_back(a.g.nxh * (a.g.nzp / ZB));
        lds = std::max(lds, y_lds(a.g));
    }
    P.add((const void *)k_fft_y, 256, lds, phase, items, nb);
}

static void add_fft_xi(Plan &P, int phase, const std::vector<FftXArgs> &items)
{
    std::vector<int> nb;
    size_t lds = 0;
    for (const FftXArgs &a : items) {
        nb.push_back(a.g.ny * (a.g.nzp / ZB));
        lds = std::max(lds, x_lds(a.g));
    }
    P.add((const void *)k_fft_xi, 256, lds, phase, items, nb);
}

// forward: the x pass of every item and the y pass in place; inverse: the y
// pass in place and the x pass
void add_fft_forward(Plan &P, int phase, const std::vector<FftXArgs> &x, const std::vector<FftYArgs> &y)
{
    std::vector<FftPlaneArgs> pl;
    std::vector<FftXArgs> xs;
    std::vector<FftYArgs> ys;
    for (size_t i = 0; i < x.size(); ++i) {
        if (planes_fit(x[i].g)) {
            pl.push_back(FftPlaneArgs{x[i], y[i], make_fastdiv(x[i].g.nxh)});
        } else {
            xs.push_back(x[i]);
            ys.push_back(y[i]);
        }
    }
    add_planes(P, phase, (const void *)k_fft_planes_f, pl);
    if (xs.empty()) return;
    add_fft_xf(P, phase, xs);
    add_fft_y(P, phase, ys);
}
void add_fft_inverse(Plan &P, int phase, const std::vector<FftYArgs> &y, const std::vector<FftXArgs> &x)
{
    std::vector<FftPlaneArgs> pl;
    std::vector<FftXArgs> xs;
    std::vector<FftYArgs> ys;
    for (size_t i = 0; i < x.size(); ++i) {
        if (planes_fit(x[i].g)) {
            pl.push_back(FftPlaneArgs{x[i], y[i], make_fastdiv(x[i].g.nxh)});
        } else {
            xs.push_back(x[i]);
            ys.push_back(y[i]);
        }
    }
    add_planes(P, phase, (const void *)k_fft_planes_i, pl);
    if (xs.empty()) return;
    add_fft_y(P, phase, ys);
    add_fft_xi(P, phase, xs);
}

}  // namespace epic
