// grid2par (parcel_interpl.f90:405-470), and grid2par fused with dB/dt and
// the low-storage RK push (parcel_ellipsoid.f90:466-507, ls_rk.f90:142-217,
// parcel_bc.f90:17-40) for ls_rk_step.
//
// Per parcel: four support points from the half axes; each point gathers
// velocity (3), velocity gradient (8) and vorticity tendency (3) from the
// eight corner nodes with trilinear weights (FP64 cell fractions); the
// quarter-weighted sums update delta_pos / delta_vor.  In the fused form the
// gradient gives dB/dt (B33 from det B in FP64), the stage pushes position
// (FP64), vorticity and B by cb dt delta, applies the periodic wrap (int()
// truncation), scales the deltas by ca for the next stage and computes the
// next stage's cell key and cell histogram; on every stage but the last it
// also stores the half axes of the B it wrote (FP64 eigen-solve) and the
// next par2grid's fixed-point maxima.
#include "common.h"
#include "ellipsoid.h"
#include "launch.h"

#include <algorithm>
#include <type_traits>

namespace epic {

// two neighbouring nodes of a row in one load
struct __attribute__((packed, aligned(4))) Pair {
    float lo, hi;
};

// Stand-alone grid2par(add) (parcel_interpl.f90:405-470): support points
// from the current B (stored as the cache of the next par2grid, :442),
// quarter-weighted trilinear gathers of velocity, velocity gradient and
// vorticity tendency; delta_pos / delta_vor are set or accumulated, strain is
// set.  One parcel per thread.
// What bounds it: the number of its loads (4 points x 8 corners x 14 fields, from
// L2).  The corners of a row are neighbours, so a wave whose points do not reach
// over the end of a row takes them in pairs, half the loads: 570 -> 315 us at
// 96x64x32 (1.6 M parcels), 40 -> 30 a call at 20x36x10.
__global__ __launch_bounds__(256) void k_grid2par(const G2PArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const G2PArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int64_t PS = plane_stride(g), FS = field_stride(g);
    int e = 0;
    const int64_t q = ib.blk * (int64_t)blockDim.x + threadIdx.x;
    if (q < a.p.n) {
        const double pos[3] = {gl(a.p.x)[q], gl(a.p.y)[q], gl(a.p.z)[q]};
        double B[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) B[c] = (double)gl(a.p.B[c])[q];
        const double vol = (double)gl(a.p.vol)[q];
        double ve[3], vt[3];
        if (!support_axes(B, vol, ve, vt)) {
            e |= ERR_B33;
            ve[0] = ve[1] = ve[2] = vt[0] = vt[1] = vt[2] = 0.0;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            gl(a.p.veta[d])[q] = (float)ve[d];
            gl(a.p.vtau[d])[q] = (float)vt[d];
        }
        float dp[3], dv[3], st[8];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            dp[c] = a.add ? gl(a.p.dpos[c])[q] : 0.0f;
            dv[c] = a.add ? gl(a.p.dvor[c])[q] : 0.0f;
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) st[c] = 0.0f;
        for (int jp = 0; jp < 4; ++jp) {
            const double cs = support_cos(jp), sn = support_sin(jp);
            int ii[3];
            float w[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double pt = pos[d] + ve[d] * cs + vt[d] * sn;
                const double xyz = (pt - g.lower[d]) * g.dxi[d];
                const double fl = floor(xyz);
                ii[d] = (int)fl;
                w[d] = (float)(xyz - fl);
            }
            if (ii[2] < -1 || ii[2] > g.nz) {
                e |= ERR_OUT_OF_GRID;
                continue;
            }
            const int x0 = wrap(ii[0], g.nx), x1 = wrap(ii[0] + 1, g.nx);
            const int y0 = wrap(ii[1], g.ny), y1 = wrap(ii[1] + 1, g.ny);
            const int64_t zp0 = (int64_t)(ii[2] + 1) * PS, zp1 = zp0 + PS;
            // corners in Fortran element order of ww(0:1,0:1,0:1): k fastest;
            // the pairs along x of the first four
            const int64_t row[4] = {zp0 + (int64_t)y0 * g.nx, zp1 + (int64_t)y0 * g.nx, zp0 + (int64_t)y1 * g.nx,
                                    zp1 + (int64_t)y1 * g.nx};
            const float pxc = 1.0f - w[0], pyc = 1.0f - w[1], pzc = 1.0f - w[2];
            const float w00 = pyc * pxc, w10 = pyc * w[0], w01 = w[1] * pxc, w11 = w[1] * w[0];
            const float wt[8] = {pzc * w00, w[2] * w00, pzc * w01, w[2] * w01,
                                 pzc * w10, w[2] * w10, pzc * w11, w[2] * w11};
            auto gather = [&](auto pairs) {
                auto at_point = [&](int slot) {
                    const EPIC_GLOBAL float *f = gl(a.fld) + slot * FS;
                    float lo[4], hi[4], s = 0.0f;
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        if constexpr (decltype(pairs)::value) {
                            const Pair v = *(const EPIC_GLOBAL Pair *)(f + row[m] + x0);
                            lo[m] = v.lo;
                            hi[m] = v.hi;
                        } else {
                            lo[m] = f[row[m] + x0];
                            hi[m] = f[row[m] + x1];
                        }
                    }
#pragma unroll
                    for (int m = 0; m < 4; ++m) s += wt[m] * lo[m];
#pragma unroll
                    for (int m = 0; m < 4; ++m) s += wt[4 + m] * hi[m];
                    return 0.25f * s;
                };
#pragma unroll
                for (int c = 0; c < 3; ++c) dp[c] += at_point(F_VELOG + c);
#pragma unroll
                for (int c = 0; c < 8; ++c) st[c] += at_point(F_VELGRADG + c);
#pragma unroll
                for (int c = 0; c < 3; ++c) dv[c] += at_point(F_VTEND + c);
            };
            if (__any(x1 != x0 + 1)) gather(std::false_type{});
            else gather(std::true_type{});
        }

#pragma unroll
        for (int c = 0; c < 3; ++c) {
            gl(a.p.dpos[c])[q] = dp[c];
            gl(a.p.dvor[c])[q] = dv[c];
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) gl(a.p.strain[c])[q] = st[c];
    }
    if (e) atomicOr(a.err, e);
}

// ---------------------------------------------------------------------------
// Tiled form used by ls_rk_step: one work-group per (8x8 column tile, z chunk
// of tz cell layers).  The 14 gathered fields of the chunk's node box (node
// planes k0-1 .. k0+tz+1, x and y from -1 to 9 around the tile) are staged in
// LDS once as four planes of field groups (fields 0-3, 4-7, 8-11 as float4,
// 12-13 as float2), so every corner is three 16-byte and one 8-byte LDS read
// and neighbouring nodes sit in neighbouring banks; then every thread takes
// parcels of the chunk's slot range of the cell sort, with no barrier between
// parcels.  Support points come from the
// half axes cached for this stage.  The permutation entry of a thread's next
// parcel is loaded one round ahead, and parcel arrays are addressed as a
// table pointer plus a 32-bit byte offset.
//
// What bounds it: HBM traffic (367 B a parcel at 4.9 TB/s, a large copy's rate
// here, in a run that moves parcels by a cell in two steps), as long as no
// round waits for memory before its gather: the deltas are taken into the sums
// after the gather, LDS strides are constant, offsets are folded into the
// accesses, the fields that a step does not change are out of the maxima, and
// no register is spilled.  A launch at 128^3: 1.46 ms, 1.20 with these, 1.15
// with chunks of four layers (g2p_default_tz).
// ---------------------------------------------------------------------------
size_t g2p_lds_bytes(int tz) { return (3 * sizeof(float4) + sizeof(float2)) * (tz + 3) * P2G_BOX * P2G_BOX; }

template <int NT, int TZ>
__global__ __launch_bounds__(NT, 4) void k_g2p_tiles(const G2PTileArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const G2PTileArgs &a = tab[ib.item];
    const Grid &g = a.g;
    constexpr int tz = TZ;   // = a.tz
    const int tx = ib.blk % a.ntx;
    const int ty = (ib.blk / a.ntx) % a.nty;
    const int cz = ib.blk / (a.ntx * a.nty);
    const int i0 = tx * P2G_TX, j0 = ty * P2G_TY;
    const int k0 = -1 + cz * tz;
    const int nl = min(tz, g.nz + 1 - k0);   // layers k0 .. k0 + nl - 1
    const int tid = threadIdx.x;
    const int64_t PS = plane_stride(g), FS = field_stride(g);
    constexpr int NN = P2G_BOX * P2G_BOX;
    constexpr int nbox = tz + 3;

    extern __shared__ float4 box[];                 // [group][plane][y][x]: 3 float4 groups, then a float2 group
    constexpr int NB = nbox * NN;                   // nodes in the box
    float2 *box2 = (float2 *)(box + 3 * NB);
    __shared__ unsigned int s_pmax[3];              // the next par2grid's vorticity maxima (float bits)
    int e = 0;
    if (tid < 3) s_pmax[tid] = 0u;   // ordered by the barrier after the box is staged

    // ---- stage the node box (plane P = k0 - 1 + lp) ----
    // thread = (node of the 11 x 11 box column, half of the 14 fields, every
    // NT / 256-th plane): the wrapped column offset is found once, then the
    // thread walks its planes with its 7 loads in flight at a time
    static_assert(NN <= 128 && NT % 256 == 0, "two threads per box node column");
    {
        const int node = tid & 127, half = (tid >> 7) & 1;
        if (node < NN) {
            const int ly = node / P2G_BOX, lx = node - ly * P2G_BOX;
            int gi = i0 - 1 + lx, gj = j0 - 1 + ly;   // in [-1, n + 9]
            gi = (gi < 0) ? gi + g.nx : (gi >= g.nx ? gi - g.nx : gi);
            gj = (gj < 0) ? gj + g.ny : (gj >= g.ny ? gj - g.ny : gj);
            const EPIC_GLOBAL float *col = gl(a.fld) + (int64_t)(F_VELOG + half) * FS + (int64_t)gj * g.nx + gi;
            for (int lp = tid >> 8; lp < nbox; lp += NT / 256) {
                const int P = k0 - 1 + lp;
                const bool in = (P >= -1 && P <= g.nz + 1);
                const int64_t po = (int64_t)(P + 1) * PS;
                float v[7];
#pragma unroll
                for (int t = 0; t < 7; ++t) v[t] = in ? col[(int64_t)(2 * t) * FS + po] : 0.0f;
                const int nd = lp * NN + node;
#pragma unroll
                for (int t = 0; t < 7; ++t) {
                    const int f = 2 * t + half;
                    if (f < 12) ((float *)box)[((f >> 2) * NB + nd) * 4 + (f & 3)] = v[t];
                    else ((float *)box2)[nd * 2 + (f - 12)] = v[t];
                }
            }
        }
    }
    __syncthreads();
    // the chunk's parcels: one contiguous slot range of the sort
    const int first = gl(a.cell_start)[layer_index(g, tx, ty, k0)];
    const int total = gl(a.cell_start)[layer_index(g, tx, ty, k0 + nl)] - first;

    // The next round's entry is loaded one round ahead, and the position and
    // half axes of the parcel it names are requested in the middle of the
    // current round (after the gather), so the support points of a round
    // start without waiting for memory.
    int pi_nx = 0;
    double pn[3] = {0.0, 0.0, 0.0};
    float an[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    const bool acc_prev = a.stage > 1;
    auto prefetch = [&](int pj) {
        const unsigned oj = block_offset((unsigned)pj * 4u);
        pn[0] = gl(a.p.x)[pj];
        pn[1] = gl(a.p.y)[pj];
        pn[2] = gl(a.p.z)[pj];
#pragma unroll
        for (int c = 0; c < 6; ++c) an[c] = at(a.axes[c], oj);
    };
    if (tid < total) {
        pi_nx = gl(a.perm)[first + tid];
        prefetch(pi_nx);
    }
    for (int base = 0; base < total; base += NT) {   // uniform rounds: the ballot needs every lane
        const int q = base + tid;
        const int pi = pi_nx;
        const unsigned o4 = (unsigned)pi * 4u;   // byte offset (pi < 2^30): scalar base + 32-bit offset addressing
        const bool more = q + NT < total;
        if (more) pi_nx = gl(a.perm)[first + q + NT];
        double pos[3] = {pn[0], pn[1], pn[2]};
        int key = -1;
        bool small = false;
        auto process = [&]() {
            if (q >= total) return;
            // requested here and used after the gather
            float Bf[5];
#pragma unroll
            for (int c = 0; c < 5; ++c) Bf[c] = at(a.p.B[c], o4);
            const float volf = at(a.p.vol, o4);
            float dp[3] = {}, dv[3] = {};
            if (acc_prev) {
                const unsigned o = block_offset(o4);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    dp[c] = at(a.p.dpos[c], o);
                    dv[c] = at(a.p.dvor[c], o);
                }
            }
            int cc[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) cc[d] = (int)floor((pos[d] - g.lower[d]) * g.dxi[d]);
            const int cx = wrap(cc[0], g.nx) - i0, cy = wrap(cc[1], g.ny) - j0;
            const int k = cc[2];
            if (cx < 0 || cx >= P2G_TX || cy < 0 || cy >= P2G_TY || k < k0 || k >= k0 + nl) {
                e |= ERR_CELL_MISMATCH;
                if (more) prefetch(pi_nx);
                return;
            }
            const int own = __mul24(k - k0 + 1, NN) + __mul24(cy + 1, P2G_BOX) + cx + 1;   // own cell's lower corner in the box
            // coordinate of support point jp along axis d, in cells
            auto coord = [&](int jp, int d) {
                const double pt = pos[d] + (double)an[d] * support_cos(jp) + (double)an[3 + d] * support_sin(jp);
                return (pt - g.lower[d]) * g.dxi[d];
            };
            // A point's gathered velocity and tendency wait in sd until the
            // deltas that they are added to have arrived.
            float st[8], sd[4][6];
#pragma unroll
            for (int c = 0; c < 8; ++c) st[c] = 0.0f;
#pragma unroll
            for (int jp = 0; jp < 4; ++jp) {
                int off[3];
                float w[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const double xyz = coord(jp, d), fl = floor(xyz);
                    off[d] = (int)fl - cc[d];
                    w[d] = (float)(xyz - fl);
                }
                // box corner; -2: beyond the neighbour cells; -1: beyond the
                // halo layers (the reference fails too)
                int n0 = own + __mul24(off[2], NN) + __mul24(off[1], P2G_BOX) + off[0];
                if ((unsigned)(off[0] + 1) > 2u || (unsigned)(off[1] + 1) > 2u || (unsigned)(off[2] + 1) > 2u) n0 = -2;
                if (k + off[2] < -1 || k + off[2] > g.nz) {
                    e |= ERR_OUT_OF_GRID;
                    n0 = -1;
                }
#pragma unroll
                for (int c = 0; c < 6; ++c) sd[jp][c] = 0.0f;
                if (n0 == -1) continue;
                const float pxc = 1.0f - w[0], pyc = 1.0f - w[1], pzc = 1.0f - w[2];
                const float w00 = pyc * pxc, w10 = pyc * w[0], w01 = w[1] * pxc, w11 = w[1] * w[0];
                // corners in Fortran element order of ww(0:1,0:1,0:1): k fastest
                const float wt[8] = {pzc * w00, w[2] * w00, pzc * w01, w[2] * w01,
                                     pzc * w10, w[2] * w10, pzc * w11, w[2] * w11};
                float s[14];
#pragma unroll
                for (int f = 0; f < 14; ++f) s[f] = 0.0f;
                if (n0 >= 0) {
#pragma unroll
                    for (int m = 0; m < 8; ++m) {
                        const int dz = m & 1, dy = (m >> 1) & 1, dx = (m >> 2) & 1;
                        const int nd = n0 + dz * NN + dy * P2G_BOX + dx;
                        const float4 q0 = box[nd], q1 = box[NB + nd], q2 = box[2 * NB + nd];
                        const float2 q3 = box2[nd];
                        const float vv[14] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w,
                                              q2.x, q2.y, q2.z, q2.w, q3.x, q3.y};
#pragma unroll
                        for (int f = 0; f < 14; ++f) s[f] += wt[m] * vv[f];
                    }
                } else {
                    // strongly stretched parcels, rare: the corners from the
                    // global fields, in the same order, so the sums are the
                    // same bits (the cell again from its coordinates: offsets
                    // kept to here would spill registers of the gather)
                    const int ci = (int)floor(coord(jp, 0)), cj = (int)floor(coord(jp, 1)), ck = (int)floor(coord(jp, 2));
#pragma unroll 1
                    for (int m = 0; m < 8; ++m) {
                        const int dz = m & 1, dy = (m >> 1) & 1, dx = (m >> 2) & 1;
                        const int ii = wrap(ci + dx, g.nx), jj = wrap(cj + dy, g.ny);
                        const int64_t o = (int64_t)(ck + dz + 1) * PS + (int64_t)jj * g.nx + ii;
                        const EPIC_GLOBAL float *f0 = gl(a.fld) + (int64_t)F_VELOG * FS + o;
#pragma unroll
                        for (int f = 0; f < 14; ++f) s[f] += wt[m] * f0[(int64_t)f * FS];
                    }
                }
#pragma unroll
                for (int c = 0; c < 8; ++c) st[c] += 0.25f * s[3 + c];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    sd[jp][c] = s[c];
                    sd[jp][3 + c] = s[11 + c];
                }
            }
#pragma unroll
            for (int jp = 0; jp < 4; ++jp)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    dp[c] += 0.25f * sd[jp][c];
                    dv[c] += 0.25f * sd[jp][3 + c];
                }
            if (more) prefetch(pi_nx);   // the next round's position and axes, in flight during the rest
            float vor[3], dBo[5] = {};
            {
                const unsigned o = block_offset(o4);
#pragma unroll
                for (int c = 0; c < 3; ++c) vor[c] = at(a.p.vor[c], o);
            }
            if (acc_prev) {
                const unsigned o = block_offset(o4);
#pragma unroll
                for (int c = 0; c < 5; ++c) dBo[c] = at(a.p.dB[c], o);
            }
            // dB/dt (FP64, B33 from the volume constraint)
            const double vol = (double)volf;
            double B[5], S[8], dB[5];
#pragma unroll
            for (int c = 0; c < 5; ++c) B[c] = (double)Bf[c];
#pragma unroll
            for (int c = 0; c < 8; ++c) S[c] = (double)st[c];
            if (!dBdt(B, S, vol, dB)) {
                e |= ERR_B33;
                dB[0] = dB[1] = dB[2] = dB[3] = dB[4] = 0.0;
            }
            float db[5];
#pragma unroll
            for (int c = 0; c < 5; ++c) db[c] = dBo[c] + (float)dB[c];
            // push (ls_rk.f90:183-191), periodic wrap (parcel_bc.f90:17-21)
            const double cbdt = a.cb * (*a.dt);
#pragma unroll
            for (int c = 0; c < 3; ++c) pos[c] = pos[c] + cbdt * (double)dp[c];
#pragma unroll
            for (int c = 0; c < 3; ++c) vor[c] = (float)((double)vor[c] + cbdt * (double)dv[c]);
#pragma unroll
            for (int c = 0; c < 5; ++c) B[c] = B[c] + cbdt * (double)db[c];
            pos[0] = pos[0] - g.extent[0] * trunc((pos[0] - g.center[0]) * g.hli[0]);
            pos[1] = pos[1] - g.extent[1] * trunc((pos[1] - g.center[1]) * g.hli[1]);
            if (a.reflect) {   // parcel_bc.f90:26-40
                if (pos[2] > g.upper[2]) {
                    pos[2] = 2.0 * g.upper[2] - pos[2];
                    B[2] = -B[2];
                    B[4] = -B[4];
                } else if (pos[2] < g.lower[2]) {
                    pos[2] = 2.0 * g.lower[2] - pos[2];
                    B[2] = -B[2];
                    B[4] = -B[4];
                }
            }
            gl(a.p.x)[pi] = pos[0];
            gl(a.p.y)[pi] = pos[1];
            gl(a.p.z)[pi] = pos[2];
            {
                const unsigned o = block_offset(o4);
#pragma unroll
                for (int c = 0; c < 3; ++c) at(a.p.vor[c], o) = vor[c];
#pragma unroll
                for (int c = 0; c < 5; ++c) at(a.p.B[c], o) = (float)B[c];
            }
            if (a.stage < a.nstages) {
                const float ca = (float)a.ca;
                const unsigned o = block_offset(o4);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    at(a.p.dpos[c], o) = ca * dp[c];
                    at(a.p.dvor[c], o) = ca * dv[c];
                }
#pragma unroll
                for (int c = 0; c < 5; ++c) at(a.p.dB[c], o) = ca * db[c];
            }
            // cell of the new position for the next stage's sort
            const int ni = (int)floor((pos[0] - g.lower[0]) * g.dxi[0]);
            const int nj = (int)floor((pos[1] - g.lower[1]) * g.dxi[1]);
            const int nk = (int)floor((pos[2] - g.lower[2]) * g.dxi[2]);
            if (nk < -1 || nk > g.nz) e |= ERR_PARCEL_COUNT;
            else key = cell_index(g, wrap(ni, g.nx), wrap(nj, g.ny), nk);
            at(a.keys, block_offset(o4)) = key;
            small = (vol <= g.vmin);
            if (a.axes_next[0]) {   // the next stage's support axes, from B as stored
                double Bs[5], ve2[3], vt2[3];
#pragma unroll
                for (int c = 0; c < 5; ++c) Bs[c] = (double)(float)B[c];
                if (!support_axes(Bs, vol, ve2, vt2)) {
                    e |= ERR_B33;
                    ve2[0] = ve2[1] = ve2[2] = vt2[0] = vt2[1] = vt2[2] = 0.0;
                }
                const unsigned o = block_offset(o4);
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    at(a.axes_next[d], o) = (float)ve2[d];
                    at(a.axes_next[3 + d], o) = (float)vt2[d];
                }
            }
            if (a.tmax_next) {
                // the next par2grid's largest vorticity contributions, from
                // what was stored (the other fields' values do not change in a
                // step), into the work-group's maxima (bits of non-negative
                // floats); a lane below the running maximum skips the atomic
                const float v0 = (float)(0.25 * vol);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const float m = fabsf(v0 * vor[c]);
                    if (m > __uint_as_float(s_pmax[c])) atomicMax(&s_pmax[c], __float_as_uint(m));
                }
            }
        };
        process();
        // next stage's cell histogram, one atomic per run of equal keys
        wave_run_add(key, gl(a.count));
        if (__any(small)) wave_run_add(small ? key : -1, gl(a.scount));
    }
    if (a.tmax_next) {
        __syncthreads();
        if (tid < 3) {   // only what is above the maximum there (atomics on one address take turns)
            unsigned int *out = (unsigned int *)a.tmax_next + 1 + tid;
            if (s_pmax[tid] > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, s_pmax[tid]);
        }
    }
    if (e) atomicOr(a.err, e);
}

// (128 threads a layer at least: add_rk_stage_tiles)
template <int TZ> static const void *tiles_kernel(int nt)
{
    if constexpr (TZ <= 2)
        if (nt == 256) return (const void *)k_g2p_tiles<256, TZ>;
    if constexpr (TZ <= 4)
        if (nt == 512) return (const void *)k_g2p_tiles<512, TZ>;
    return (const void *)k_g2p_tiles<1024, TZ>;
}

void add_rk_stage_tiles(Plan &P, int phase, const std::vector<G2PTileArgs> &all)
{
    for (int tz : {2, 4, 8}) {   // one grouped launch per z chunk, the kernel specialised on it
        std::vector<G2PTileArgs> items;
        std::vector<int> nb;
        int64_t total = 0;
        for (const G2PTileArgs &a : all) {
            if (a.tz != tz) continue;
            items.push_back(a);
            nb.push_back(a.ntx * a.nty * a.nchz);
            total += nb.back();
        }
        if (items.empty()) continue;
        const int nt = std::max(tile_threads(total), 128 * tz);   // (256 at 4 layers: 187 us at 64^3)
        P.add(tz == 2 ? tiles_kernel<2>(nt) : tz == 4 ? tiles_kernel<4>(nt) : tiles_kernel<8>(nt), nt, g2p_lds_bytes(tz), phase, items, nb);
    }
}

void add_grid2par(Plan &P, int phase, const std::vector<G2PArgs> &items)
{
    std::vector<int> nb;
    for (const G2PArgs &a : items) nb.push_back((int)((a.p.n + 255) / 256));
    P.add((const void *)k_grid2par, 256, 0, phase, items, nb);
}

}  // namespace epic
