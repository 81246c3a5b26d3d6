// par2grid on gfx950: deterministic, atomic-free float accumulation.
//
// Pipeline (one member):
//   1. k_cell_keys     FP64 cell of every parcel centre (get_index,
//                      fields.f90:165-172), integer histogram of parcels and
//                      small parcels per cell (nparg / nsparg)
//   2. scan            exclusive prefix sum of the histogram -> cell_start
//   3. k_place         slot = cell_start + integer ticket (order not fixed yet)
//   4. k_cell_order    order every cell's slots by caller parcel index
//                      (epic_cell_sort only: the reference's cell order)
//   5. k_p2g_tiles     one work-group per (8x8 column tile, z chunk of tz
//                      layers), one thread per parcel: support points in FP64,
//                      each of the 4 x 8 x 7 contributions of a parcel scaled
//                      by a per-member power of two, rounded and added to a
//                      64-bit integer LDS accumulator of its node; the box is
//                      scaled back exactly and written to a per-tile FP64
//                      staging box
//   6. k_p2g_finalize  per node, sums the staging boxes that cover it in a
//                      fixed tile order (the periodic halo accumulation of
//                      field_mpi.f90), applies the free-slip folds,
//                      normalises by volume, the zeta wall condition and the
//                      z extrapolation (parcel_interpl.f90:235-319) in FP64;
//                      each field is rounded to FP32 once, on its store
// Integer node sums are exact and the staging boxes are added in a fixed
// tile order, so the result depends on the parcel set alone, never on
// scheduling or parcel order: results are bitwise reproducible.
#include "common.h"
#include "ellipsoid.h"
#include "launch.h"

#include <algorithm>
#include <type_traits>

namespace epic {

// ---------------------------------------------------------------------------
// 1. cell keys + histogram
// ---------------------------------------------------------------------------
__device__ inline int cell_key(const Grid &g, double x, double y, double z, int &err)
{
    const int i = (int)floor((x - g.lower[0]) * g.dxi[0]);
    const int j = (int)floor((y - g.lower[1]) * g.dxi[1]);
    const int k = (int)floor((z - g.lower[2]) * g.dxi[2]);
    if (k < -1 || k > g.nz) {
        err |= ERR_PARCEL_COUNT;
        return -1;
    }
    return cell_index(g, wrap(i, g.nx), wrap(j, g.ny), k);
}

__global__ __launch_bounds__(256) void k_cell_keys(const KeysArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const KeysArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int64_t n = parcel_count(a.p);
    if ((int64_t)ib.blk * PER_BLOCK >= n) return;   // uniform over the block
    int e = 0;
    // every lane runs every round (the histogram adds are wave-aggregated
    // over runs of equal keys: consecutive parcels mostly share a cell)
#pragma unroll
    for (int r = 0; r < PER_BLOCK / 256; ++r) {
        const int64_t q = (int64_t)ib.blk * PER_BLOCK + r * 256 + threadIdx.x;
        int key = -1;
        bool small = false;
        if (q < n) {
            key = cell_key(g, gl(a.p.x)[q], gl(a.p.y)[q], gl(a.p.z)[q], e);
            gl(a.keys)[q] = key;
            small = key >= 0 && gl(a.p.vol)[q] <= g.vmin;
        }
        wave_run_add(key, gl(a.count));
        wave_run_add(small ? key : -1, gl(a.scount));
    }
    if (e) atomicOr(a.err, e);
}

// ---------------------------------------------------------------------------
// 2. exclusive scan: block sums, then every block's own prefix.  A block of
// the second pass adds up the sums before it itself, so there is no launch
// for the sums' scan (up to SCAN_FUSED_BLOCKS of them: 32 KB each re-reads);
// of at most SCAN_SOLO_BLOCKS a block adds up the entries before it, and the
// scan is one launch (three blocks at 16^3: 8.8 us in two, 5.4 in one; eight
// at 24^3: 9.3 and 7.5)
// ---------------------------------------------------------------------------
constexpr int SCAN_T = 256;
constexpr int SCAN_PER = 8;
constexpr int SCAN_BLOCK = SCAN_T * SCAN_PER;

__device__ inline int block_excl_scan(int v, int *lds, int &total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int a = __shfl_up(incl, off, 64);
        if (lane >= off) incl += a;
    }
    if (lane == 63) lds[w] = incl;
    __syncthreads();
    int base = 0;
    total = 0;
#pragma unroll
    for (int u = 0; u < SCAN_T / 64; ++u) {
        if (u < w) base += lds[u];
        total += lds[u];
    }
    __syncthreads();
    return base + incl - v;
}

// the previous par2grid's far-point sums back to zero, when there were any
// (k_place then resets the flag)
__device__ inline void clear_far(const ScanArgs &a, int blk)
{
    if (!a.far_flag || *a.far_flag == 0) return;
    const int64_t step = (a.n + SCAN_BLOCK - 1) / SCAN_BLOCK * SCAN_T;
    for (int64_t q = (int64_t)blk * SCAN_T + threadIdx.x; q < a.far_n; q += step) gl(a.far_acc)[q] = 0ull;
}

__global__ __launch_bounds__(SCAN_T) void k_scan_reduce(const ScanArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    __shared__ int lds[SCAN_T / 64];
    const ItemBlock ib = item_block(bmap);
    const ScanArgs &a = tab[ib.item];
    const int64_t base = ib.blk * (int64_t)SCAN_BLOCK + threadIdx.x * SCAN_PER;
    int s = 0;
#pragma unroll
    for (int u = 0; u < SCAN_PER; ++u)
        if (base + u < a.n) s += gl(a.in)[base + u];
    int total;
    block_excl_scan(s, lds, total);
    if (threadIdx.x == 0) gl(a.bsum)[ib.blk] = total;
    clear_far(a, ib.blk);
}

// one block per item: exclusive scan of the item's block sums in place
__global__ __launch_bounds__(SCAN_T) void k_scan_blocks(const ScanArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    __shared__ int lds[SCAN_T / 64];
    const ItemBlock ib = item_block(bmap);
    const ScanArgs &a = tab[ib.item];
    const int nb = (int)((a.n + SCAN_BLOCK - 1) / SCAN_BLOCK);
    int carry = 0;
    for (int base = 0; base < nb; base += SCAN_T * SCAN_PER) {
        const int i0 = base + threadIdx.x * SCAN_PER;
        int v[SCAN_PER], s = 0;
#pragma unroll
        for (int u = 0; u < SCAN_PER; ++u) {
            v[u] = (i0 + u < nb) ? gl(a.bsum)[i0 + u] : 0;
            s += v[u];
        }
        int total;
        int ex = block_excl_scan(s, lds, total);
        int run = carry + ex;
#pragma unroll
        for (int u = 0; u < SCAN_PER; ++u) {
            if (i0 + u < nb) gl(a.bsum)[i0 + u] = run;
            run += v[u];
        }
        carry += total;
        __syncthreads();
    }
}

// out[c] = exclusive prefix, out[n] = total; clears gl(a.clear)[c] (the
// placement cursors) on the way
enum ScanForm {
    SCAN_PREFIXES,   // bsum holds the prefixes of the blocks' sums
    SCAN_SUMS,       // the sums
    SCAN_ALONE       // nothing yet
};
template <ScanForm FORM>
__global__ __launch_bounds__(SCAN_T) void k_scan_apply(const ScanArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    __shared__ int lds[SCAN_T / 64];
    const ItemBlock ib = item_block(bmap);
    const ScanArgs &a = tab[ib.item];
    const int64_t n = a.n;
    const int64_t base = ib.blk * (int64_t)SCAN_BLOCK + threadIdx.x * SCAN_PER;
    int v[SCAN_PER], s = 0;
#pragma unroll
    for (int u = 0; u < SCAN_PER; ++u) {
        v[u] = (base + u < n) ? gl(a.in)[base + u] : 0;
        s += v[u];
    }
    int total;
    int run = block_excl_scan(s, lds, total);
    if constexpr (FORM != SCAN_PREFIXES) {
        int before = 0;
        if constexpr (FORM == SCAN_SUMS) {
            for (int b = threadIdx.x; b < ib.blk; b += SCAN_T) before += gl(a.bsum)[b];
        } else {
            for (int b = 0; b < ib.blk; ++b) {
#pragma unroll
                for (int u = 0; u < SCAN_PER; ++u) before += gl(a.in)[b * SCAN_BLOCK + u * SCAN_T + threadIdx.x];
            }
            clear_far(a, ib.blk);
        }
        int all;
        (void)block_excl_scan(before, lds, all);
        run += all;
    } else {
        run += gl(a.bsum)[ib.blk];
    }
#pragma unroll
    for (int u = 0; u < SCAN_PER; ++u) {
        if (base + u < n) {
            gl(a.out)[base + u] = run;
            if (a.clear) gl(a.clear)[base + u] = 0;
        }
        run += v[u];
    }
    // the thread owning element n-1 also writes the grand total out[n]
    if (base <= n - 1 && n - 1 < base + SCAN_PER) gl(a.out)[n] = run;
}

void add_exclusive_scan(Plan &P, int phase, const std::vector<ScanArgs> &items)
{
    std::vector<int> nb, one;
    for (const ScanArgs &a : items) {
        nb.push_back((int)((a.n + SCAN_BLOCK - 1) / SCAN_BLOCK));
        one.push_back(1);
    }
    const int most = *std::max_element(nb.begin(), nb.end());
    bool apart = true;   // blocks read what others may have scanned already
    for (const ScanArgs &a : items) apart = apart && a.in != a.out && a.in != a.clear;
    if (apart && most <= SCAN_SOLO_BLOCKS) {
        P.add((const void *)k_scan_apply<SCAN_ALONE>, SCAN_T, 0, phase, items, nb);
        return;
    }
    P.add((const void *)k_scan_reduce, SCAN_T, 0, phase, items, nb);
    if (most <= SCAN_FUSED_BLOCKS) {
        P.add((const void *)k_scan_apply<SCAN_SUMS>, SCAN_T, 0, phase, items, nb);
        return;
    }
    P.add((const void *)k_scan_blocks, SCAN_T, 0, phase, items, one);
    P.add((const void *)k_scan_apply<SCAN_PREFIXES>, SCAN_T, 0, phase, items, nb);
}

int64_t scan_scratch_ints(int64_t n) { return (n + SCAN_BLOCK - 1) / SCAN_BLOCK + 1; }

// ---------------------------------------------------------------------------
// 3./4. placement and per-cell ordering
// ---------------------------------------------------------------------------
// Lanes of a wave that hold the same key in a row (the parcels are nearly in cell
// order) share one atomicAdd on the key's cursor; a lane's ticket is the cursor's
// old value and its rank in the run.
__global__ __launch_bounds__(256) void k_place(const PlaceArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const PlaceArgs &a = tab[ib.item];
    // the rounds' keys, cell starts and tickets are each requested together,
    // so a wave waits three memory round trips, not three per round
    constexpr int NR = PER_BLOCK / 256;   // every lane of a wave runs the same rounds
    const int lane = threadIdx.x & 63;
    const int64_t n = a.n_dev ? *a.n_dev : a.n;
    if (a.far_flag && ib.blk == 0 && threadIdx.x == 0) *a.far_flag = 0;   // its sums were cleared by the scan
    int key[NR], start[NR], head_lane[NR], got[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int64_t q = (int64_t)ib.blk * PER_BLOCK + r * 256 + threadIdx.x;
        key[r] = (q < n) ? gl(a.keys)[q] : -1;
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) start[r] = (key[r] >= 0) ? gl(a.cell_start)[key[r]] : 0;
#pragma unroll
    for (int r = 0; r < NR; ++r) {   // the atomics are left in flight
        const int prev = __shfl_up(key[r], 1, 64);
        const bool head = (lane == 0) || (prev != key[r]);
        const unsigned long long heads = __ballot(head);
        const unsigned long long below = heads & ((lane == 63) ? ~0ull : ((2ull << lane) - 1));
        head_lane[r] = 63 - __clzll(below);
        const unsigned long long above = heads & ~((2ull << lane) - 1 | (lane == 63 ? ~0ull : 0ull));
        const int next = above ? __ffsll((long long)above) - 1 : 64;
        got[r] = (head && key[r] >= 0) ? atomicAdd(&gl(a.cursor)[key[r]], next - lane) : 0;
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int base = __shfl(got[r], head_lane[r], 64) + (lane - head_lane[r]);
        if (key[r] >= 0) gl(a.perm)[start[r] + base] = (int)((int64_t)ib.blk * PER_BLOCK + r * 256 + threadIdx.x);
    }
}

__global__ void k_cell_order(int64_t nc, const int *__restrict__ cell_start, const int *__restrict__ perm_tmp,
                             const int *__restrict__ orig, int *__restrict__ perm)
{
    for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < nc; c += (int64_t)gridDim.x * blockDim.x) {
        const int s0 = cell_start[c], s1 = cell_start[c + 1];
        const int m = s1 - s0;
        if (m == 0) continue;
        if (m <= 32) {
            int pv[32], ov[32];
            for (int a = 0; a < m; ++a) {
                pv[a] = perm_tmp[s0 + a];
                ov[a] = orig[pv[a]];
            }
            for (int a = 1; a < m; ++a) {   // insertion sort by caller index
                const int kp = pv[a], ko = ov[a];
                int b = a - 1;
                while (b >= 0 && ov[b] > ko) {
                    pv[b + 1] = pv[b];
                    ov[b + 1] = ov[b];
                    --b;
                }
                pv[b + 1] = kp;
                ov[b + 1] = ko;
            }
            for (int a = 0; a < m; ++a) perm[s0 + a] = pv[a];
        } else {
            // crowded cell: selection by rank (stable: caller indices are unique)
            for (int a = 0; a < m; ++a) {
                const int pa = perm_tmp[s0 + a];
                const int oa = orig[pa];
                int rank = 0;
                for (int b = 0; b < m; ++b) rank += (orig[perm_tmp[s0 + b]] < oa);
                perm[s0 + rank] = pa;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// 5. tile scatter into fixed-point LDS accumulators
// ---------------------------------------------------------------------------
// One work-group per (8 x 8 column tile, tz cell layers); its parcels are one
// contiguous slot range, and a wave takes 64 consecutive ones at a time, so
// every lane has a parcel and a round's loads are whole lines.
// Every contribution w * (vol/4) * value is scaled by a power of two chosen
// per member and field from k_p2g_max's maxima (so that no single point's
// contribution exceeds 2^27),
// rounded to an integer and added to a 64-bit LDS accumulator of its node;
// the points of one parcel that fall in the same cell are combined first.
// Most points stay in their parcel's own cell, and neighbouring lanes mostly
// share a cell: four lanes of one cell exchange their (rounded) own-cell
// contributions, first the upper and lower planes within a lane pair, then
// the rows between the pairs, and each adds the four parcels' sums to two of
// the cell's eight corners, a quarter of the atomics.  Quads across a cell
// boundary exchange within matching pairs only.  Integer
// sums do not depend on the order of the additions, so the node sums are
// bitwise reproducible however the waves are scheduled, with no ordering
// pass and no barriers between parcels; the only rounding is that of each
// contribution (2^-28 of the member's largest) and of the final conversion.
// Node box of a tile: x, y in [-1, 9] around the tile, node planes
// [k0 - 1, k0 + tz + 1]; rows padded to lpitch 64-bit words (12 spreads the
// 8 x 8 lanes of a wave evenly over the 32 LDS banks).

__host__ __device__ constexpr int box_planes(int tz) { return tz + 3; }
// LDS row pitch in 64-bit words; at tz = 8 the unpadded 11 keeps two
// work-groups per CU within the LDS
__host__ __device__ constexpr int p2g_lpitch(int tz) { return tz >= 8 ? P2G_BOX : 12; }

// power-of-two scale s with max_abs * s < 2^27 (0 when max_abs is 0): the
// summed weights of up to four points of one parcel stay below 4, so every
// rounded contribution is below 2^29 and a node's sum over its parcels stays
// far below 2^47
__device__ inline float fixed_scale(float max_abs, int &e)
{
    if (!(max_abs > 0.0f)) {
        e = 0;
        return 0.0f;
    }
    frexpf(max_abs, &e);   // max_abs < 2^e
    return ldexpf(1.0f, 27 - e);
}

// values of other lanes of a quad by DPP quad permutations (all four lanes
// active): the other lane of the pair [1, 0, 3, 2], the same lane of the
// other pair [2, 3, 0, 1]
constexpr int QP_PAIR = 0xB1, QP_CROSS = 0x4E, QP_FIRST = 0x00, QP_LAST = 0xFF;
template <int QP> __device__ inline int quad_perm(int v) { return __builtin_amdgcn_mov_dpp(v, QP, 0xF, 0xF, false); }
// One fixed-point contribution as a 64-bit accumulator term, in one FP64
// FMA: w * c is exact in FP64 (two FP32 factors), and adding 1.5 * 2^52
// rounds it to the nearest integer q (ties to even) with q held in the low
// bits of the result, whose pattern is F_MAGIC + q for |q| < 2^51.  F_MAGIC
// is zero below bit 48, so a sum of such terms equals the sum of the q
// modulo 2^48 in its low 48 bits, whatever the number of terms: the node
// sums (|sum| < 2^47) are the low 48 bits sign-extended (fixed_sum).
constexpr double F_MAGIC_D = 6755399441055744.0;   // 1.5 * 2^52
__device__ inline unsigned long long fixed_term(double w, double c)
{
    return (unsigned long long)__double_as_longlong(fma(w, c, F_MAGIC_D));
}
// The same term as a plain 32-bit integer (|q| < 2^29: the sum of a quad's four
// fits too), for sums between lanes: half the lane moves, each part of its
// addition.  fixed_wide makes an accumulator term of such a sum.
__device__ inline int fixed_term32(double w, double c) { return (int)(unsigned)fixed_term(w, c); }
__device__ inline unsigned long long fixed_wide(int q) { return (unsigned long long)(long long)q; }
__device__ inline long long fixed_sum(unsigned long long acc) { return (long long)(acc << 16) >> 16; }

// the gridded quantities of parcel pi, read from its arrays (o4 = 4 pi)
__device__ inline void p2g_values(const Grid &g, const ParcelsDev &p, unsigned o4, double z, float v[P2G_NF])
{
    const float vor[3] = {at(p.vor[0], o4), at(p.vor[1], o4), at(p.vor[2], o4)};
    p2g_values_of(g, at(p.vol, o4), vor, at(p.buoy, o4), at(p.hum, o4), z, v);
}

// The largest |contribution| of every field over a member's parcels, and
// the largest |total buoyancy - buoyancy| one: one coalesced pass in
// storage order by at most P2G_MAX_BLOCKS work-groups, whose block maxima
// go to out[] by integer atomicMax on the bits of the non-negative floats.
// out[] is zero when this runs: it starts zeroed, and the finalize kernel
// of the same par2grid clears it once the tile kernel has taken its scales
// from it (a value left by an interrupted sequence would only be larger, a
// coarser but still valid scale).  Inside an RK step only the first stage
// runs this pass: volume, buoyancy and humidity do not change in a step, so
// their maxima stay for the later stages, the vorticity maxima come from the
// previous push, and the moist contributions, which follow the height, are
// bounded by the humidity: the condensate is at most the humidity (q0 >= 0;
// otherwise every stage runs this pass), so |tbuoy| <= |buoy| + glat hum and
// |tbuoy - buoy| <= glat hum (P2G_MAX_BOUND onwards; exact where there is no
// humidity).  A contribution at its maximum fills the 32 bits of a quad's sum,
// so the first bound is raised by 2^-20: its roundings and those of the
// contribution are at most seven, of 2^-24 each.  A scale from a bound is at
// most one power of two coarser.
__device__ inline void take_maxima(const Grid &g, const ParcelsDev &p, int64_t q, float mx[P2G_MAXIMA])
{
    float v[P2G_NF];
    p2g_values(g, p, (unsigned)q * 4u, gl(p.z)[q], v);
#pragma unroll
    for (int f = 0; f < P2G_NF; ++f) mx[f] = fmaxf(mx[f], fabsf(v[f]));
    mx[P2G_NF] = fmaxf(mx[P2G_NF], fabsf(v[4] - v[5]));
    const float hum = at(p.hum, (unsigned)q * 4u), hb = fabsf(v[0] * (float)g.glat * hum), b = fabsf(v[5]) + hb;
    mx[P2G_MAX_BOUND] = fmaxf(mx[P2G_MAX_BOUND], hum != 0.0f ? b * (1.0f + 0x1p-20f) : b);
    mx[P2G_MAX_BOUND + 1] = fmaxf(mx[P2G_MAX_BOUND + 1], hb);
}
// the block's maxima to out[] (256 threads).  A block whose maximum is not
// above the one already there leaves it: atomics on one address take turns
// across the chip
__device__ inline void put_maxima(float mx[P2G_MAXIMA], float *out)
{
    __shared__ float wm[4][P2G_MAXIMA];
#pragma unroll
    for (int f = 0; f < P2G_MAXIMA; ++f) {
        for (int o = 32; o > 0; o >>= 1) mx[f] = fmaxf(mx[f], __shfl_xor(mx[f], o, 64));
        if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6][f] = mx[f];
    }
    __syncthreads();
    if (threadIdx.x < P2G_MAXIMA) {
        const int f = threadIdx.x;
        const float m = fmaxf(fmaxf(wm[0][f], wm[1][f]), fmaxf(wm[2][f], wm[3][f]));
        if (m > __hip_atomic_load(out + f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax((unsigned int *)out + f, __float_as_uint(m));
    }
}
__global__ __launch_bounds__(256) void k_p2g_max(const P2GMaxArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const P2GMaxArgs &a = tab[ib.item];
    float mx[P2G_MAXIMA];
#pragma unroll
    for (int f = 0; f < P2G_MAXIMA; ++f) mx[f] = 0.0f;
    const int64_t n = parcel_count(a.p);
    for (int64_t q = (int64_t)ib.blk * 256 + threadIdx.x; q < n; q += (int64_t)a.nblk * 256) take_maxima(a.g, a.p, q, mx);
    put_maxima(mx, a.out);
}

// TZ (= a.tz) is a template parameter, so the LDS strides are constants and
// the 8 x 7 atomics of a cell are its base word plus immediate offsets.
//
// What bounds it: VALU issue (the SIMDs about 80 % busy at 128^3), then the LDS
// atomics; reads are 87 B a parcel.  One lane per consecutive slot, a quad's
// sums exchanged before its atomics, against two lanes per cell walking the
// cell's parcels (whose rounds each touched every line of four rows of cells,
// 455 B read a parcel): 0.91 -> 0.69 ms a launch at 128^3 without humidity,
// four work-groups per CU (three: 0.79).
template <int TZ>
__global__ __launch_bounds__(1024, 4) void k_p2g_tiles(const P2GArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const P2GArgs &a = tab[ib.item];
    const Grid &g = a.g;
    // stage 1 of a step after the first takes the cached axes (l_reuse)
    const float *const *axes = (a.use_alt && *a.use_alt) ? a.axes_alt : a.axes;
    constexpr int tz = TZ, lp = p2g_lpitch(TZ);
    const int tx = ib.blk % a.ntx;
    const int ty = (ib.blk / a.ntx) % a.nty;
    const int cz = ib.blk / (a.ntx * a.nty);
    const int k0 = -1 + cz * tz;
    const int tid = threadIdx.x;
    constexpr int nbox = box_planes(tz);
    constexpr int lplane = P2G_BOX * lp;          // words per LDS node plane
    constexpr int lfield = nbox * lplane;         // words per field
    extern __shared__ unsigned long long acc[];   // [field][plane][y][x]
    __shared__ int s_err, s_far;
    __shared__ unsigned short s_items[16][64];   // per wave: the pass's items (source lane, first point)

    for (int u = tid; u < P2G_NF * lfield; u += blockDim.x) acc[u] = 0ull;
    if (tid == 0) s_err = s_far = 0;

    // the chunk's parcels: one contiguous slot range of the sort
    const int i0 = tx * P2G_TX, j0 = ty * P2G_TY, nl = min(tz, g.nz + 1 - k0);
    const int first = gl(a.cell_start)[layer_index(g, tx, ty, k0)];
    const int nparc = gl(a.cell_start)[layer_index(g, tx, ty, k0 + nl)] - first;
    // fixed-point scales from the member's largest contributions; with no
    // condensation anywhere the total buoyancy equals the buoyancy (field 5
    // is a copy of field 4) and with no humidity field 6 is zero: their
    // atomics are then skipped and the results are the same bits
    float mx[P2G_NF + 1];
#pragma unroll
    for (int f = 0; f <= P2G_NF; ++f) mx[f] = gl(a.tmax)[f];
    if (a.bounds) {   // the later stages of a step
        mx[4] = gl(a.tmax)[P2G_MAX_BOUND];
        mx[P2G_NF] = gl(a.tmax)[P2G_MAX_BOUND + 1];
    }
    float sc[P2G_NF];
#pragma unroll
    for (int f = 0; f < P2G_NF; ++f) {
        int e;
        sc[f] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(fixed_scale(mx[f], e))));   // uniform: a scalar register
    }
    const bool own5 = mx[P2G_NF] > 0.0f;   // tbuoy differs from buoy somewhere
    const bool own6 = mx[6] > 0.0f;        // humidity somewhere
    __syncthreads();   // the accumulators are cleared

    // ---- support points, trilinear weights, integer accumulation ----
    const int lane = tid & 63;
    const bool zup = lane & 1, yup = lane & 2;   // this lane's corners of an own cell: its plane and row
    const float zsg = zup ? 1.0f : -1.0f, znr = zup ? 0.0f : 1.0f, zfr = 1.0f - znr;
    const float ysg = yup ? 1.0f : -1.0f, ynr = yup ? 0.0f : 1.0f, yfr = 1.0f - ynr;
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned short *items = s_items[tid >> 6];
    int err = 0;
    // two copies of the loop: without humidity anywhere the condensation's
    // exponential (whose constants would take 20 registers of the loop) and
    // two of the fields drop out at compile time
    auto scatter = [&](auto humid) {
        constexpr bool HUMID = decltype(humid)::value;
        // the lanes beyond the last parcel take it again, with zero values
        int pi_nx = (nparc > 0) ? gl(a.perm)[first + min(tid, nparc - 1)] : 0;
        for (int q0 = tid - lane; q0 < nparc; q0 += blockDim.x) {   // uniform over the wave
            const int pi = pi_nx;
            if (q0 + (int)blockDim.x < nparc) pi_nx = gl(a.perm)[first + min(q0 + (int)blockDim.x + lane, nparc - 1)];
            bool have = q0 + lane < nparc;
            const unsigned o4 = (unsigned)pi * 4u;   // byte offset (pi < 2^30): scalar base + 32-bit offset addressing
            const double pos[3] = {gl(a.p.x)[pi], gl(a.p.y)[pi], gl(a.p.z)[pi]};
            const double ve[3] = {at(axes[0], o4), at(axes[1], o4), at(axes[2], o4)};
            const double vt[3] = {at(axes[3], o4), at(axes[4], o4), at(axes[5], o4)};
            float v[P2G_NF];
            if constexpr (HUMID) {
                p2g_values(g, a.p, o4, pos[2], v);
            } else {   // p2g_values without humidity
                const float v0 = (float)(0.25 * (double)at(a.p.vol, o4));
                v[0] = v0;
#pragma unroll
                for (int c = 0; c < 3; ++c) v[1 + c] = v0 * at(a.p.vor[c], o4);
                v[4] = v[5] = v0 * at(a.p.buoy, o4);
                v[6] = 0.0f;
            }
            int cc[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) cc[d] = (int)floor((pos[d] - g.lower[d]) * g.dxi[d]);
            int cx = wrap(cc[0], g.nx) - i0, cy = wrap(cc[1], g.ny) - j0, lz = cc[2] - k0;
            if ((unsigned)cx >= (unsigned)P2G_TX || (unsigned)cy >= (unsigned)P2G_TY || (unsigned)lz >= (unsigned)tz) {
                // not in the cell it was sorted into: left out.  In lane 1 or 2 of a
                // quad it also puts its share of the others' sums at the wrong node:
                // no sum of the call counts once this is reported (a wave that took
                // such quads apart ran 0.7 % longer)
                err |= ERR_CELL_MISMATCH;
                have = false;
                cx = cy = lz = 0;
            }
            const int cown = __mul24(lz + 1, lplane) + __mul24(cy + 1, lp) + cx + 1;   // own cell's lower corner
            float cs[P2G_NF];
#pragma unroll
            for (int f = 0; f < P2G_NF; ++f) cs[f] = have ? v[f] * sc[f] : 0.0f;   // exact: sc is a power of two
            // the four support points: target cell (box corner index, -1 when
            // outside the neighbour cells) and cell fractions
            // tgt: >= 0 box corner; -1 none; < -1 a point beyond the neighbour
            // cells, -2 - its cell offsets (7 bits each, biased by 64)
            int tgt[4];
            float fr[4][3];
            unsigned farm = 0;   // bit jp: point jp lies beyond the neighbour cells
#pragma unroll
            for (int jp = 0; jp < 4; ++jp) {
                int off[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const double pt = pos[d] + ve[d] * support_cos(jp) + vt[d] * support_sin(jp);
                    const double xyz = (pt - g.lower[d]) * g.dxi[d];
                    const double fl = floor(xyz);
                    off[d] = (int)fl - cc[d];
                    fr[jp][d] = (float)(xyz - fl);
                }
                tgt[jp] = -1;
                if (cc[2] + off[2] < -1 || cc[2] + off[2] > g.nz) {   // beyond the halo layers (the reference fails too)
                    if (have) err |= ERR_OUT_OF_GRID;
                } else if (off[0] < -1 || off[0] > 1 || off[1] < -1 || off[1] > 1 || off[2] < -1 || off[2] > 1) {
                    if (have && off[0] >= -64 && off[0] < 64 && off[1] >= -64 && off[1] < 64 && off[2] >= -64 && off[2] < 64) {
                        farm |= 1u << jp;   // beyond the neighbour cells: global accumulator, below
                        tgt[jp] = -2 - (((off[2] + 64) << 14) | ((off[1] + 64) << 7) | (off[0] + 64));
                    } else if (have) {
                        err |= ERR_OUT_OF_GRID;   // more than 64 cells away
                    }
                } else {   // lower corner of the point's cell in the box
                    tgt[jp] = cown + __mul24(off[2], lplane) + __mul24(off[1], lp) + off[0];
                }
            }
            // support points beyond the neighbour cells (strongly stretched
            // parcels, rare): each point's 8 x 7 fixed-point terms go to the
            // member's global accumulator by 64-bit atomics (exact integer sums,
            // so still independent of the order), which the finalize adds
            if (farm) {
                s_far = 1;
                const int64_t FS = field_stride(g);
#pragma unroll
                for (int jp = 0; jp < 4; ++jp) {
                    if (!((farm >> jp) & 1u)) continue;
                    const int code = -2 - tgt[jp];
                    const int gi[3] = {cc[0] + (code & 127) - 64, cc[1] + ((code >> 7) & 127) - 64, cc[2] + (code >> 14) - 64};
                    const float *f3 = fr[jp];
                    const float wxy[4] = {(1.0f - f3[1]) * (1.0f - f3[0]), (1.0f - f3[1]) * f3[0], f3[1] * (1.0f - f3[0]),
                                          f3[1] * f3[0]};
#pragma unroll 1
                    for (int c = 0; c < 8; ++c) {
                        const int ii = wrap(gi[0] + (c & 1), g.nx), jj = wrap(gi[1] + ((c >> 1) & 1), g.ny);
                        const int kk = gi[2] + (c >> 2);   // in [-1, nz + 1]
                        const int64_t node = ((int64_t)(kk + 1) * g.ny + jj) * g.nx + ii;
                        const double wd = (double)(((c & 4) ? f3[2] : 1.0f - f3[2]) * wxy[c & 3]);
#pragma unroll
                        for (int f = 0; f < P2G_NF; ++f) atomicAdd(a.far_acc + f * FS + node, fixed_term(wd, (double)cs[f]));
                    }
                }
            }
            // own cell: the summed weights (in point order) of the points in it
            // by corner, [plane][row][x], this lane's plane and row first
            {
                float w[2][2][2] = {};
#pragma unroll
                for (int jp = 0; jp < 4; ++jp) {
                    const float *f3 = fr[jp];
                    // near and far weight of each axis: f or 1 - f, as one FMA
                    const float wy[2] = {fmaf(ysg, f3[1], ynr), fmaf(-ysg, f3[1], yfr)};
                    float wz[2] = {fmaf(zsg, f3[2], znr), fmaf(-zsg, f3[2], zfr)};
                    const float xl = 1.0f - f3[0], xu = f3[0];
                    if (tgt[jp] != cown) wz[0] = wz[1] = 0.0f;   // adds exact zeros
#pragma unroll
                    for (int cy_ = 0; cy_ < 2; ++cy_) {
                        const float wxy[2] = {wy[cy_] * xl, wy[cy_] * xu};
#pragma unroll
                        for (int cz_ = 0; cz_ < 2; ++cz_)
#pragma unroll
                            for (int c = 0; c < 2; ++c) w[cz_][cy_][c] = fmaf(wz[cz_], wxy[c], w[cz_][cy_][c]);
                    }
                }
                // node of [plane][row][0]
                const int dzn = zup ? lplane : 0, dzf = lplane - dzn, dyn = yup ? lp : 0, dyf = lp - dyn;
                if (quad_perm<QP_FIRST>(cown) == quad_perm<QP_LAST>(cown)) {   // (a cell's slots are consecutive)
                    const int nn = cown + dzn + dyn;
#pragma unroll
                    for (int f = 0; f < P2G_NF; ++f) {
                        if (!HUMID ? f > 4 : f == 5 && !own5) continue;   // uniform over the work-group
                        const double q = (double)cs[f];
#pragma unroll
                        for (int c = 0; c < 2; ++c) {
                            const int tn = fixed_term32((double)w[0][0][c], q) + quad_perm<QP_PAIR>(fixed_term32((double)w[1][0][c], q));
                            const int tf = fixed_term32((double)w[0][1][c], q) + quad_perm<QP_PAIR>(fixed_term32((double)w[1][1][c], q));
                            atomicAdd(&acc[f * lfield + nn + c], fixed_wide(tn + quad_perm<QP_CROSS>(tf)));
                        }
                    }
                } else {
                    const bool match = quad_perm<QP_PAIR>(cown) == cown;
                    const int mm = match ? -1 : 0;
#pragma unroll
                    for (int f = 0; f < P2G_NF; ++f) {
                        if (!HUMID ? f > 4 : f == 5 && !own5) continue;
                        const double q = (double)cs[f];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int dy = (r >> 1) ? dyf : dyn, c = r & 1;
                            const int tf = fixed_term32((double)w[1][r >> 1][c], q);
                            const int tn = fixed_term32((double)w[0][r >> 1][c], q);
                            atomicAdd(&acc[f * lfield + cown + dzn + dy + c], fixed_wide(tn + (quad_perm<QP_PAIR>(tf) & mm)));
                            if (!match) atomicAdd(&acc[f * lfield + cown + dzf + dy + c], fixed_wide(tf));
                        }
                    }
                }
            }
            // every other cell the points reach: its 8 corners take the summed
            // weights of its points (in point order), 8 x 7 atomics per cell.
            // These (lane, cell) items, about one for every second parcel, are
            // shared out over the wave: item P[k] + (rank of the lane among the
            // lanes with more than k items) is a lane's k-th; the lanes take 64
            // items per pass, find their source lane through a per-wave list and
            // read its fractions, targets and values by ds_bpermute, so the
            // atomics run with nearly every lane active (one pass per round as a
            // rule, where a loop over the four points ran up to four sparse ones).
            // Each item's weights and terms are the same arithmetic as in its
            // source lane.
            unsigned leadm = 0;   // bit jp: point jp opens a cell other than its own and earlier points'
#pragma unroll
            for (int jp = 0; jp < 4; ++jp) {
                bool lead = tgt[jp] >= 0 && tgt[jp] != cown && have;
#pragma unroll
                for (int jq = 0; jq < jp; ++jq) lead = lead && (tgt[jq] != tgt[jp]);
                leadm |= (lead ? 1u : 0u) << jp;
            }
            const int ni = __popc(leadm);
            unsigned long long lb[4];
            int pk[5];
            pk[0] = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                lb[k] = __ballot(ni > k);
                pk[k + 1] = pk[k] + __popcll(lb[k]);
            }
            const int total = pk[4];   // uniform over the wave
            if (total > 0) {
                // box corners in 16 bits each; no target (also a far point) as -1
                int tb[4];
#pragma unroll
                for (int jq = 0; jq < 4; ++jq) tb[jq] = tgt[jq] >= 0 ? tgt[jq] : -1;
                const int t01 = (tb[0] & 0xffff) | (tb[1] << 16), t23 = (tb[2] & 0xffff) | (tb[3] << 16);
                for (int r = 0; r < total; r += 64) {
                    unsigned lm = leadm;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int jp = __ffs(lm) - 1;   // the lane's k-th item: point jp
                        lm &= lm - 1u;
                        const int idx = pk[k] + __popcll(lb[k] & below) - r;
                        if (k < ni && idx >= 0 && idx < 64) items[idx] = (unsigned short)(lane | (jp << 8));
                    }
                    __builtin_amdgcn_wave_barrier();
                    const bool mine = r + lane < total;
                    const unsigned e = mine ? (unsigned)items[lane] : 0u;
                    const int sa = (int)(e & 63u) << 2, jp0 = (int)(e >> 8) & 3;
                    float g[4][3];
#pragma unroll
                    for (int jq = 0; jq < 4; ++jq)
#pragma unroll
                        for (int d = 0; d < 3; ++d) g[jq][d] = __int_as_float(__builtin_amdgcn_ds_bpermute(sa, __float_as_int(fr[jq][d])));
                    float cf[P2G_NF];
#pragma unroll
                    for (int f = 0; f < P2G_NF; ++f)
                        cf[f] = (!HUMID ? f > 4 : f == 5 && !own5) ? 0.0f
                                : __int_as_float(__builtin_amdgcn_ds_bpermute(sa, __float_as_int(cs[f])));
                    const int u01 = __builtin_amdgcn_ds_bpermute(sa, t01), u23 = __builtin_amdgcn_ds_bpermute(sa, t23);
                    __builtin_amdgcn_wave_barrier();   // the list is read before the next pass writes it
                    if (mine) {
                        const int tg[4] = {(int)(short)(u01 & 0xffff), u01 >> 16, (int)(short)(u23 & 0xffff), u23 >> 16};
                        const int t = jp0 == 0 ? tg[0] : jp0 == 1 ? tg[1] : jp0 == 2 ? tg[2] : tg[3];
                        float w[8];
#pragma unroll
                        for (int c = 0; c < 8; ++c) w[c] = 0.0f;
#pragma unroll
                        for (int jq = 0; jq < 4; ++jq) {
                            const float *f3 = g[jq];
                            // (no point before the leader has its target)
                            const bool in = tg[jq] == t;
                            const float wz[2] = {in ? 1.0f - f3[2] : 0.0f, in ? f3[2] : 0.0f};
                            const float xl = 1.0f - f3[0], yl = 1.0f - f3[1];
                            const float wxy[4] = {yl * xl, yl * f3[0], f3[1] * xl, f3[1] * f3[0]};
#pragma unroll
                            for (int c = 0; c < 8; ++c) {
                                const float wc = wz[c >> 2] * wxy[c & 3];
                                w[c] = w[c] + wc;
                            }
                        }
#pragma unroll
                        for (int c = 0; c < 8; ++c) {
                            const int node = t + (c >> 2) * lplane + ((c >> 1) & 1) * lp + (c & 1);
                            const double wd = (double)w[c];
#pragma unroll
                            for (int f = 0; f < P2G_NF; ++f) {
                                if (!HUMID ? f > 4 : f == 5 && !own5) continue;   // uniform over the work-group
                                atomicAdd(&acc[f * lfield + node], fixed_term(wd, (double)cf[f]));
                            }
                        }
                    }
                }
            }
        }
    };
    if (own6) scatter(std::true_type{});
    else scatter(std::false_type{});
    if (err) atomicOr(&s_err, err);
    __syncthreads();

    // ---- the box to staging (FP64, node-major, fields fastest) ----
    // q / scale is exact in FP64 (|q| < 2^53, the scale a power of two), so
    // the staged partial sums keep every bit of the integer sums
    double inv[P2G_NF];
#pragma unroll
    for (int f = 0; f < P2G_NF; ++f) inv[f] = (sc[f] > 0.0f) ? 1.0 / (double)sc[f] : 0.0;
    auto stage = [&](auto fields) {
        constexpr int NS = decltype(fields)::value, PLANE = P2G_BOX * P2G_BOX * NS;
        EPIC_GLOBAL double *out = gl(a.staging) + (int64_t)ib.blk * nbox * PLANE;
        for (int u = tid; u < nbox * PLANE; u += blockDim.x) {
            const int f = u % NS, nd = u / NS;
            const int pz = nd / (P2G_BOX * P2G_BOX), yx = nd - pz * (P2G_BOX * P2G_BOX);
            const int y = yx / P2G_BOX, x = yx - y * P2G_BOX;
            const int fs = (f == 5 && !own5) ? 4 : f;   // a skipped field 5 is field 4
            out[u] = (double)fixed_sum(acc[fs * lfield + pz * lplane + y * lp + x]) * inv[fs];
        }
    };
    // without humidity only the fields with sums of their own: the staging is
    // 400 MB at 128^3 otherwise, written here and read by the finalize
    const bool dry = !own5 && !own6;
    if (dry) stage(std::integral_constant<int, P2G_DRY>{});
    else stage(std::integral_constant<int, P2G_NF>{});
    if (tid == 0 && s_err) atomicOr(a.err, s_err);
    if (tid == 0 && s_far) atomicOr(a.far_flag, 1);
    if (ib.blk == 0) {   // the same in every work-group
        if (tid < P2G_NF) a.far_scale[tid] = inv[tid];
        if (tid == 0) *a.staged = dry ? P2G_DRY : P2G_NF;
    }
}

// ---------------------------------------------------------------------------
// 6. staging sum + folds + normalisation (one thread per (i, j) column)
// ---------------------------------------------------------------------------
// tile d = -1, 0, 1 beside the one of node i (of n >= P2G_BOX nodes in nt >= 2
// tiles of 8, the last one shorter when n is not a multiple of 8): its number t
// and the node's place l in its box; false when it holds nothing for the node.
// No box of such a row meets itself, and of two tiles one is beside the other
// once.  (Not here: beyond a last tile of one node, node 0 is also the last
// place of the box of the tile before it.)
__device__ inline bool box_place(int d, int i, int n, int nt, int &t, int &l)
{
    const int own = i >> 3, r = i & 7;
    t = own + d;
    l = r + 1;
    if (nt == 2) {
        if (d > 0) return false;
        if (d < 0) {
            t = 1 - own;
            l = wrap(i - (8 * t - 1), n);
        }
        return l < P2G_BOX;
    }
    if (d < 0) {
        if (r > 1) return false;
        l = r + 9;
        if (own == 0) {
            t = nt - 1;
            l = i + n - 8 * t + 1;
            return l < P2G_BOX;
        }
    } else if (d > 0) {
        l = 0;
        if (i == n - 1) t = 0;
        else if (r != 7) return false;
    }
    return true;
}

// adds the staged sums of node (i, j, k) to out[], and its far-point sums
// when there are any (far).  NS fields are staged; of P2G_DRY, field 5 is
// field 4 and field 6 zero.  A node lies in one box, or in two along each
// direction (three beside a last tile of a single node).  The kernel was bound
// by its waits, one per box; the up to four boxes of a z chunk are loaded
// together instead: 19.3 -> 11.6 us at 16^3, 24.9 -> 20.9 at 64^3, 143 -> 103 at
// 128^3 (290 MB of dry staging).  All nine combinations at once take 184
// registers: 25 and 127 us; several lanes per node do not help.
template <int NS>
__device__ inline void stage_add(const FinalizeArgs &a, int i, int j, int k, double out[P2G_NF], bool far)
{
    constexpr int PLANE = P2G_BOX * P2G_BOX * NS;
    const Grid &g = a.g;
    if (far) {
        const int64_t FS = field_stride(g), o = ((int64_t)(k + 1) * g.ny + j) * g.nx + i;
#pragma unroll
        for (int f = 0; f < P2G_NF; ++f) out[f] += (double)fixed_sum(a.far_acc[f * FS + o]) * a.far_scale[f];
    }
    auto add = [&](auto v) {
#pragma unroll
        for (int f = 0; f < NS; ++f) out[f] += v[f];
        if constexpr (NS == P2G_DRY) out[5] += v[4];
    };
    const int nbox = a.tz + 3;
    const int cza = (k + 1) / a.tz;
    // node row 0 in the box of the tile before a last one of one row, which does
    // not lie beside its own (only along y, as nx is even, and from 25 rows on:
    // the transforms do not take 17)
    const bool beyond = a.nty > 3 && g.ny == P2G_TY * (a.nty - 1) + 1 && j == 0;
    if (a.ntx >= 2 && a.nty >= 2 && g.nx >= P2G_BOX && g.ny >= P2G_BOX) {
        // offsets of the boxes' tiles and places along x and y, -1 for none:
        // its own tile's, a neighbour's, and (a last tile of one row only)
        // the other neighbour's
        int64_t ox[3], oy[3];
        auto places = [&](int64_t o[3], int p, int n, int nt, int64_t tile, int node) {
#pragma unroll
            for (int d = -1; d <= 1; ++d) {
                int t, l;
                o[d == 0 ? 0 : d < 0 ? 1 : 2] = box_place(d, p, n, nt, t, l) ? t * tile + l * node : -1;
            }
            if (o[1] < 0) {
                o[1] = o[2];
                o[2] = -1;
            }
        };
        places(ox, i, g.nx, a.ntx, nbox * PLANE, NS);
        places(oy, j, g.ny, a.nty, (int64_t)a.ntx * nbox * PLANE, P2G_BOX * NS);
#pragma unroll 1
        for (int dcz = -1; dcz <= 1; ++dcz) {
            const int cz = cza + dcz, lp = k - (cz * a.tz - 2);
            if (cz < 0 || cz >= a.nchz || lp < 0 || lp >= nbox) continue;
            const EPIC_GLOBAL double *s = gl(a.staging) + (int64_t)cz * a.nty * a.ntx * nbox * PLANE + lp * PLANE;
            double v[4][NS];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t x = ox[q & 1], y = oy[q >> 1];
#pragma unroll
                for (int f = 0; f < NS; ++f) v[q][f] = 0.0;
                if (x >= 0 && y >= 0) {
#pragma unroll
                    for (int f = 0; f < NS; ++f) v[q][f] = s[y + x + f];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) add(v[q]);
            if (ox[2] >= 0 || oy[2] >= 0) {
#pragma unroll 1
                for (int q = 0; q < 5; ++q) {
                    const int64_t x = q < 3 ? ox[2] : q == 3 ? ox[0] : ox[1], y = q == 0 ? oy[0] : q == 1 ? oy[1] : oy[2];
                    if (x >= 0 && y >= 0) add(s + y + x);
                }
            }
        }
        if (beyond) {   // (apart, so that other rows' loads wait for nothing: 281 -> 277 us of par2grid a step at 32^3)
            const int64_t y = (int64_t)(a.nty - 2) * a.ntx * nbox * PLANE + (P2G_BOX - 1) * P2G_BOX * NS;
#pragma unroll 1
            for (int q = 0; q < 9; ++q) {   // (z chunk, box along x)
                const int cz = cza + q / 3 - 1, lp = k - (cz * a.tz - 2), c = q % 3;
                const int64_t x = c == 0 ? ox[0] : c == 1 ? ox[1] : ox[2];
                if (x >= 0 && cz >= 0 && cz < a.nchz && lp >= 0 && lp < nbox)
                    add(gl(a.staging) + (int64_t)cz * a.nty * a.ntx * nbox * PLANE + lp * PLANE + y + x);
            }
        }
        return;
    }
    const int txa = i / P2G_TX, tya = j / P2G_TY;
    for (int dcz = -1; dcz <= 1; ++dcz) {
        const int cz = cza + dcz;
        if (cz < 0 || cz >= a.nchz) continue;
        const int lp = k - (cz * a.tz - 2);   // box plane index
        if (lp < 0 || lp >= nbox) continue;
        for (int dty = -1; dty <= (beyond ? 2 : 1); ++dty) {
            // distinct candidate tiles only (grids of one or two tiles wrap)
            if ((a.nty == 1 && dty != 0) || (a.nty == 2 && dty == 1)) continue;
            const int ty = dty == 2 ? a.nty - 2 : wrap(tya + dty, a.nty);
            for (int ly = wrap(j - (ty * P2G_TY - 1), g.ny); ly < P2G_BOX; ly += g.ny) {
                for (int dtx = -1; dtx <= 1; ++dtx) {
                    if ((a.ntx == 1 && dtx != 0) || (a.ntx == 2 && dtx == 1)) continue;
                    const int tx = wrap(txa + dtx, a.ntx);
                    for (int lx = wrap(i - (tx * P2G_TX - 1), g.nx); lx < P2G_BOX; lx += g.nx) {
                        const int wg = (cz * a.nty + ty) * a.ntx + tx;
                        const EPIC_GLOBAL double *s = gl(a.staging) + ((int64_t)wg * nbox + lp) * PLANE + (ly * P2G_BOX + lx) * NS;
                        double v[NS];
#pragma unroll
                        for (int f = 0; f < NS; ++f) v[f] = s[f];
                        add(v);
                    }
                }
            }
        }
    }
}

// one thread per (column, node plane k = -1..nz+1), consecutive threads on
// consecutive columns.  Planes 0, 1, nz-1, nz carry the free-slip folds, the
// halo planes -1 and nz+1 the raw sums and the z extrapolation; every thread
// recomputes the raw planes it needs, so the planes are independent.
__global__ __launch_bounds__(256) void k_p2g_finalize(const FinalizeArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const FinalizeArgs &a = tab[ib.item];
    const Grid &g = a.g;
    const int nz = g.nz;
    const int64_t ncol = (int64_t)g.nx * g.ny;
    const int64_t tq = ib.blk * (int64_t)blockDim.x + threadIdx.x;
    if (tq < P2G_MAXIMA && (a.clear_all || (tq >= 1 && tq <= 3))) gl(a.clear_tmax)[tq] = 0.0f;   // the tile kernel has read them
    if (tq >= ncol * (nz + 3)) return;
    const bool far = *a.far_flag != 0;   // reset by the next sort
    const int k = (int)(tq / ncol) - 1;
    const int64_t col = tq - (int64_t)(k + 1) * ncol;
    const int i = (int)(col % g.nx), j = (int)(col / g.nx);
    const int64_t PS = plane_stride(g), FS = field_stride(g);
    const int64_t base = (int64_t)j * g.nx + i;
    auto F = [&](int slot, int kk) -> EPIC_GLOBAL float & { return gl(a.fld)[slot * FS + (int64_t)(kk + 1) * PS + base]; };

    // the node value of plane kk (folds of parcel_interpl.f90:258-287); the
    // staged sums add exactly, the folds and the normalisation run in FP64
    // and each field is rounded to FP32 once, when it is stored
    const bool dry = *a.staged == P2G_DRY;
    auto staged = [&](int kk, double r[P2G_NF]) {
        if (dry) stage_add<P2G_DRY>(a, i, j, kk, r, far);
        else stage_add<P2G_NF>(a, i, j, kk, r, far);
    };
    auto folded = [&](int kk, double r[P2G_NF]) {
#pragma unroll
        for (int f = 0; f < P2G_NF; ++f) r[f] = 0.0;
        staged(kk, r);
        if (kk == 0 || kk == nz) {
#pragma unroll
            for (int f = 0; f < P2G_NF; ++f) r[f] *= 2.0;
        } else if (kk == 1 || kk == nz - 1) {
            staged(kk == 1 ? -1 : nz + 1, r);
        }
    };
    auto zero_zeta = [&](int kk) { return (kk == 0 && g.zeta_zero[0]) || (kk == nz && g.zeta_zero[1]); };

    if (k >= 0 && k <= nz) {
        double r[P2G_NF];
        folded(k, r);
        const double v = r[0];
        F(F_VOLG, k) = (float)v;
        F(F_VORTG + 0, k) = (float)(r[1] / v);
        F(F_VORTG + 1, k) = (float)(r[2] / v);
        F(F_VORTG + 2, k) = zero_zeta(k) ? 0.0f : (float)(r[3] / v);
        F(F_TBUOYG, k) = (float)(r[4] / v);
        F(F_DBUOYG, k) = (float)(r[5] / v);
        F(F_HUMG, k) = (float)(r[6] / v);
    } else {
        // halo planes keep the raw sums for vol/dbuoy/hum; vortg and tbuoyg
        // are extrapolated from the normalised boundary planes (:306-318)
        double r[P2G_NF];
#pragma unroll
        for (int f = 0; f < P2G_NF; ++f) r[f] = 0.0;
        staged(k, r);
        F(F_VOLG, k) = (float)r[0];
        F(F_DBUOYG, k) = (float)r[5];
        F(F_HUMG, k) = (float)r[6];
        const int kb = (k < 0) ? 0 : nz, kn = (k < 0) ? 1 : nz - 1;
        double e2[4];   // twice the boundary plane's normalised values
        folded(kb, r);
#pragma unroll
        for (int c = 0; c < 3; ++c) e2[c] = (c == 2 && zero_zeta(kb)) ? 0.0 : 2.0 * (r[1 + c] / r[0]);
        e2[3] = 2.0 * (r[4] / r[0]);
        folded(kn, r);
#pragma unroll
        for (int c = 0; c < 3; ++c) F(F_VORTG + c, k) = (float)(e2[c] - r[1 + c] / r[0]);
        F(F_TBUOYG, k) = (float)(e2[3] - r[4] / r[0]);
    }
    // parcel counts (:201-205, folds :239-243)
    auto cnt = [&](const int *c, int kk) -> int {
        return (kk >= -1 && kk <= nz) ? gl(c)[cell_index(g, i, j, kk)] : 0;
    };
    int np = cnt(a.count, k), ns = cnt(a.scount, k);
    if (k == 0) {
        np += cnt(a.count, -1);
        ns += cnt(a.scount, -1);
    }
    if (k == nz - 1) {
        np += cnt(a.count, nz);
        ns += cnt(a.scount, nz);
    }
    gl(a.nparg)[(int64_t)(k + 1) * PS + base] = np;
    gl(a.nsparg)[(int64_t)(k + 1) * PS + base] = ns;
    // clear the histogram the next push fills (never the one read here)
    if (a.clear_count && k <= nz) {
        const int c = cell_index(g, i, j, k);
        gl(a.clear_count)[c] = 0;
        gl(a.clear_scount)[c] = 0;
    }
}

// ---------------------------------------------------------------------------
// support-point half axes, once per parcel per stage (FP64 eigen-solve)
// ---------------------------------------------------------------------------
__device__ inline void store_axes(const ParcelsDev &p, float *const ax[6], int64_t q, int &e)
{
    const double B[5] = {gl(p.B[0])[q], gl(p.B[1])[q], gl(p.B[2])[q], gl(p.B[3])[q], gl(p.B[4])[q]};
    double ve[3], vt[3];
    if (!support_axes(B, (double)gl(p.vol)[q], ve, vt)) {
        e |= ERR_B33;
        ve[0] = ve[1] = ve[2] = vt[0] = vt[1] = vt[2] = 0.0;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        gl(ax[d])[q] = (float)ve[d];
        gl(ax[3 + d])[q] = (float)vt[d];
    }
}
__global__ __launch_bounds__(256) void k_axes(const AxesArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const AxesArgs &a = tab[ib.item];
    const int64_t n = parcel_count(a.p);
    int e = 0;
#pragma unroll
    for (int r = 0; r < PER_BLOCK / 256; ++r) {
        const int64_t q = (int64_t)ib.blk * PER_BLOCK + r * 256 + threadIdx.x;
        if (q >= n) break;
        store_axes(a.p, a.ax, q, e);
    }
    if (e) atomicOr(a.err, e);
}
// the axes and k_p2g_max's maxima in one pass, where a par2grid needs both
// (43 + 35 us at 64^3 in two, 62 in one; 288 + 111 and 349 at 128^3)
__global__ __launch_bounds__(256) void k_axes_max(const AxesArgs *__restrict__ tab, const int2 *__restrict__ bmap)
{
    const ItemBlock ib = item_block(bmap);
    const AxesArgs &a = tab[ib.item];
    const int64_t n = parcel_count(a.p);
    float mx[P2G_MAXIMA];
#pragma unroll
    for (int f = 0; f < P2G_MAXIMA; ++f) mx[f] = 0.0f;
    int e = 0;
    for (int64_t q = (int64_t)ib.blk * 256 + threadIdx.x; q < n; q += (int64_t)a.max.nblk * 256) {
        take_maxima(a.max.g, a.p, q, mx);
        store_axes(a.p, a.ax, q, e);
    }
    put_maxima(mx, a.max.out);
    if (e) atomicOr(a.err, e);
}

// ---------------------------------------------------------------------------
// plan builders
// ---------------------------------------------------------------------------
static std::vector<int> parcel_blocks_of(const std::vector<int64_t> &n)
{
    std::vector<int> b;
    for (int64_t v : n) b.push_back((int)((v + PER_BLOCK - 1) / PER_BLOCK));
    return b;
}

// parcels a launch's grid covers: the allocated slots when known, so that a
// plan stays the same launch sequence when the parcel count changes
static int64_t grid_parcels(const ParcelsDev &p) { return std::max(p.n, p.cap); }

void add_cell_keys(Plan &P, int phase, const std::vector<KeysArgs> &items)
{
    std::vector<int64_t> n;
    for (const KeysArgs &a : items) n.push_back(grid_parcels(a.p));
    P.add((const void *)k_cell_keys, 256, 0, phase, items, parcel_blocks_of(n));
}

void add_place(Plan &P, int phase, const std::vector<PlaceArgs> &items)
{
    std::vector<int64_t> n;
    for (const PlaceArgs &a : items) n.push_back(std::max(a.n, a.cap));
    P.add((const void *)k_place, 256, 0, phase, items, parcel_blocks_of(n));
}

void add_p2g_max(Plan &P, int phase, const std::vector<P2GMaxArgs> &items)
{
    std::vector<int> nb;
    for (const P2GMaxArgs &a : items) nb.push_back(a.nblk);
    P.add((const void *)k_p2g_max, 256, 0, phase, items, nb);
}

int p2g_max_blocks(int64_t n) { return (int)std::min<int64_t>((n + 1023) / 1024, P2G_MAX_BLOCKS); }

void add_axes(Plan &P, int phase, const std::vector<AxesArgs> &items)
{
    std::vector<int64_t> n;
    for (const AxesArgs &a : items) n.push_back(grid_parcels(a.p));
    P.add((const void *)k_axes, 256, 0, phase, items, parcel_blocks_of(n));
}
void add_axes_max(Plan &P, int phase, const std::vector<AxesArgs> &items)
{
    std::vector<int> nb;
    for (const AxesArgs &a : items) nb.push_back(a.max.nblk);
    P.add((const void *)k_axes_max, 256, 0, phase, items, nb);
}

void launch_cell_order(int64_t nc, const int *cell_start, const int *perm_tmp, const int *orig, int *perm, hipStream_t s)
{
    const int nb = (int)std::min<int64_t>((nc + 255) / 256, 8192);
    hipLaunchKernelGGL(k_cell_order, dim3(nb), dim3(256), 0, s, nc, cell_start, perm_tmp, orig, perm);
}

P2GLayout p2g_layout(const Grid &g)
{
    P2GLayout L;
    // the last tile of a row or column is partial when nx or ny is not a
    // multiple of 8: its cells beyond the grid hold no parcels
    L.ntx = (g.nx + P2G_TX - 1) / P2G_TX;
    L.nty = (g.ny + P2G_TY - 1) / P2G_TY;
    L.tz = p2g_default_tz(p2g_chunks4(g));
    L.nchz = (g.nz + 2 + L.tz - 1) / L.tz;
    L.staging_elems = (int64_t)L.ntx * L.nty * L.nchz * (L.tz + 3) * P2G_BOX * P2G_BOX * P2G_NF;
    return L;
}


size_t p2g_lds_bytes(int tz) { return sizeof(unsigned long long) * P2G_NF * box_planes(tz) * P2G_BOX * p2g_lpitch(tz); }

void add_p2g(Plan &P, int phase, const std::vector<P2GArgs> &tiles, const std::vector<FinalizeArgs> &fin)
{
    // one grouped launch per z chunk, the kernel specialised on it
    // (epic_set_tiling and the autotuner admit 2, 4 and 8 only)
    std::vector<int> tzs;
    for (const P2GArgs &a : tiles)
        if (std::find(tzs.begin(), tzs.end(), a.tz) == tzs.end()) tzs.push_back(a.tz);
    for (int tz : tzs) {
        std::vector<P2GArgs> items;
        std::vector<int> nb;
        int64_t total = 0;
        for (P2GArgs a : tiles) {
            if (a.tz != tz) continue;
            items.push_back(a);
            nb.push_back(a.ntx * a.nty * a.nchz);
            total += nb.back();
        }
        // 128 threads a layer keep four waves per SIMD within the box's LDS
        const int nt = std::max(tile_threads(total), 128 * tz);
        const void *k = tz == 2 ? (const void *)k_p2g_tiles<2> : tz == 4 ? (const void *)k_p2g_tiles<4> : (const void *)k_p2g_tiles<8>;
        P.add(k, nt, p2g_lds_bytes(tz), phase == PH_P2G ? (int)PH_P2G_TILES : phase, items, nb);
    }
    std::vector<int> nf;
    for (const FinalizeArgs &f : fin) nf.push_back((int)(((int64_t)f.g.nx * f.g.ny * (f.g.nz + 3) + 255) / 256));
    P.add((const void *)k_p2g_finalize, 256, 0, phase, fin, nf);
}

}  // namespace epic
