// Horizontal 2D real FFTs of the node planes z = 0..nz (FP32), the transform
// pair of fftxyp2s / fftxys2p (sta3dfft.f90:134-257) in complex half-spectrum
// form: S(kx, ky) = sum_{i,j} f(i, j) e^{-2 pi i (kx i/nx + ky j/ny)},
// kx in [0, nx/2].  The inverse carries the 1/(nx ny) normalisation.
//
// Two passes per direction; the intermediate T[j][kx][z] and the spectra
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
        const float2 w = tw[kx];   // e^{-2 pi i kx / nx}
        const float2 s = cadd(zk, zc), d = csub(zk, zc);
        const float2 wd = cmul(w, d);
        // X = (s - i w d) / 2
        other[r * (m + 1) + kx] = float2{0.5f * (s.x + wd.y), 0.5f * (s.y - wd.x)};
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
        const float2 w = cconj(tw[k]);   // e^{+2 pi i k / nx}
        const float2 s = cadd(xk, xc), d = csub(xk, xc);
        const float2 wd = cmul(w, d);
        bufa[r * m + k] = float2{s.x - wd.y, s.y + wd.x};   // s + i w d
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

void add_fft_xf(Plan &P, int phase, const std::vector<FftXArgs> &items)
{
    std::vector<int> nb;
    size_t lds = 0;
    for (const FftXArgs &a : items) {
        nb.push_back(a.g.ny * (a.g.nzp / ZB));
        lds = std::max(lds, x_lds(a.g));
    }
    P.add((const void *)k_fft_xf, 256, lds, phase, items, nb);
}

void add_fft_y(Plan &P, int phase, const std::vector<FftYArgs> &items)
{
    std::vector<int> nb;
    size_t lds = 0;
    for (const FftYArgs &a : items) {
        nb.push_back(a.g.nxh * (a.g.nzp / ZB));
        lds = std::max(lds, y_lds(a.g));
    }
    P.add((const void *)k_fft_y, 256, lds, phase, items, nb);
}

void add_fft_xi(Plan &P, int phase, const std::vector<FftXArgs> &items)
{
    std::vector<int> nb;
    size_t lds = 0;
    for (const FftXArgs &a : items) {
        nb.push_back(a.g.ny * (a.g.nzp / ZB));
        lds = std::max(lds, x_lds(a.g));
    }
    P.add((const void *)k_fft_xi, 256, lds, phase, items, nb);
}

}  // namespace epic
