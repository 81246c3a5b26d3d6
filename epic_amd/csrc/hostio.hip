// Host <-> device copies of parcels and fields in the reference's layouts
// (parcel_container.f90:29-57, fields.f90:66-104).  The device puts the data
// into the order of the caller's arrays (parcels by caller index, components
// interleaved; fields z fastest with their halos) in a staging buffer, one
// copy moves it through pinned memory, and host threads only widen or narrow
// contiguous runs.  Chunks alternate between two buffers, so the copy of one
// overlaps the conversion of the other.
//
// What bounds it: the link (57 GB/s here) and the host's first touch of the
// caller's new pages.  The parcels of a 128^3 member (16.8 million, 1.14 GB)
// take 22 ms either way with arrays that have been written before and 36 to 48
// down into fresh ones; scattering and transposing on the host, single-threaded
// for fields, after one pageable copy per array took 340 ms, and 1.7 ms a
// component for the fields of a 96x64x32 grid.
#include "common.h"
#include "hostio.h"

#include <algorithm>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <tuple>

namespace epic {

namespace {

// ---------------------------------------------------------------------------
// staging buffers: a process-wide pool of at most POOL_KEEP idle sets.  When the
// last member goes the largest stays (up to STAGE_MAX a buffer: a program that
// makes one member at a time would allocate it again in each, at 64x64x32 5 ms
// of the 21 from create to destroy); when device memory is short all are given
// back (device_malloc).  A call owns the set it takes, so calls of several
// threads never share one.
// ---------------------------------------------------------------------------
constexpr size_t STAGE_MIN = size_t(1) << 20, STAGE_MAX = size_t(32) << 20, POOL_KEEP = 4;

struct Staging {
    size_t size = 0;   // bytes of each of the two buffers
    int device = 0;
    // pinned, its address on the device, device memory (null in a set made while
    // there was none: launches then work on the pinned memory)
    char *pin[2] = {}, *map[2] = {}, *dev[2] = {};
    hipEvent_t ev[2] = {};
};

std::mutex stage_mu;
std::vector<Staging *> stage_pool;

void stage_free(Staging *b)
{
    for (int i = 0; i < 2; ++i) {
        if (b->ev[i]) (void)hipEventDestroy(b->ev[i]);
        if (b->pin[i]) (void)hipHostFree(b->pin[i]);
        if (b->dev[i]) (void)hipFree(b->dev[i]);
    }
    delete b;
}

hipError_t stage_new(size_t size, int device, bool on_device, Staging **out)
{
    Staging *b = new Staging();
    b->size = size;
    b->device = device;
    hipError_t e = hipSuccess;
    for (int i = 0; i < 2 && e == hipSuccess; ++i) {
        e = hipHostMalloc((void **)&b->pin[i], size, hipHostMallocDefault);
        if (e == hipSuccess) e = hipHostGetDevicePointer((void **)&b->map[i], b->pin[i], 0);
        if (e == hipSuccess && on_device) e = device_malloc((void **)&b->dev[i], size);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&b->ev[i], hipEventDisableTiming);
    }
    if (e != hipSuccess) {
        stage_free(b);
        (void)hipGetLastError();
        return e;
    }
    *out = b;
    return hipSuccess;
}

// buffers of at least need bytes, capped at STAGE_MAX (the caller chunks), or
// smaller ones when memory is short; never less than least bytes.  A copy does
// not fail for want of device memory: without any it takes pinned buffers alone
hipError_t stage_get(size_t need, size_t least, Staging **out)
{
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    size_t size = STAGE_MIN;
    while (size < least || (size < need && size < STAGE_MAX)) size *= 2;
    {
        std::lock_guard<std::mutex> lk(stage_mu);
        for (size_t i = 0; i < stage_pool.size(); ++i)
            if (stage_pool[i]->device == device && stage_pool[i]->size >= size) {
                *out = stage_pool[i];
                stage_pool.erase(stage_pool.begin() + (long)i);
                return hipSuccess;
            }
    }
    for (const bool on_device : {true, false})
        for (size_t n = size; n >= std::max(least, STAGE_MIN); n /= 2)
            if ((e = stage_new(n, device, on_device, out)) == hipSuccess) return hipSuccess;
    return e;
}

// back to the pool, which keeps the largest
void stage_put(Staging *b)
{
    if (b->dev[1]) {
        std::lock_guard<std::mutex> lk(stage_mu);
        stage_pool.push_back(b);
        if (stage_pool.size() <= POOL_KEEP) return;
        auto it = std::min_element(stage_pool.begin(), stage_pool.end(),
                                   [](const Staging *x, const Staging *y) { return x->size < y->size; });
        b = *it;
        stage_pool.erase(it);
    }
    stage_free(b);
}

// up to so many bytes a field's launch works on the pinned memory itself, with no
// copy behind it (one component of 32x32x16: 33 us down, 25 so; 8 components of
// 32x32x16, 0.7 MB, up: 69 and 81)
constexpr int64_t DIRECT_MAX = 256 << 10;

// ---------------------------------------------------------------------------
// host threads of one call: run(job) calls job(t, nt) on the caller's thread
// and nt - 1 helpers and returns when all have finished
// ---------------------------------------------------------------------------
class Team {
public:
    explicit Team(int64_t elements)
    {
        const unsigned hw = std::thread::hardware_concurrency();
        // one thread per 2^20 elements, which one converts in 0.2 ms; to start
        // and join a helper takes 18 us, 15 of them 190
        const int nt = (int)std::min<int64_t>(std::min<unsigned>(hw ? hw : 1, 16u), elements / (1 << 20) + 1);
        try {
            for (int t = 1; t < nt; ++t) th_.emplace_back([this, t]() { work(t); });
        } catch (const std::system_error &) {   // fewer helpers than wished
        }
        std::lock_guard<std::mutex> lk(mu_);
        nt_ = (int)th_.size() + 1;
    }
    ~Team()
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        go_.notify_all();
        for (std::thread &t : th_) t.join();
    }
    void run(const std::function<void(int, int)> &job)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            job_ = &job;
            left_ = nt_ - 1;
            ++gen_;
        }
        if (nt_ > 1) go_.notify_all();
        job(0, nt_);
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [this] { return left_ == 0; });
    }

private:
    void work(int t)
    {
        unsigned seen = 0;
        for (;;) {
            const std::function<void(int, int)> *job;
            int nt;
            {
                std::unique_lock<std::mutex> lk(mu_);
                go_.wait(lk, [&] { return stop_ || gen_ != seen; });
                if (gen_ == seen) return;
                seen = gen_;
                job = job_;
                nt = nt_;
            }
            (*job)(t, nt);
            std::lock_guard<std::mutex> lk(mu_);
            if (--left_ == 0) done_.notify_one();
        }
    }
    std::vector<std::thread> th_;
    std::mutex mu_;
    std::condition_variable go_, done_;
    const std::function<void(int, int)> *job_ = nullptr;
    unsigned gen_ = 0;
    int nt_ = 1, left_ = 0;
    bool stop_ = false;
};

// runs nch chunks device -> host: fill(c, dev, pin) queues the device's part
// and the copy on s, take(c, pin) uses the pinned data
template <class Fill, class Take> hipError_t pipeline_down(Staging *b, int64_t nch, hipStream_t s, Fill fill, Take take)
{
    hipError_t e = hipSuccess;
    if (nch == 1) {
        e = fill(0, b->dev[0], b->pin[0]);
        const hipError_t e1 = hipStreamSynchronize(s);
        if (e == hipSuccess) e = e1;
        if (e == hipSuccess) take(0, b->pin[0]);
        return e;
    }
    auto start = [&](int64_t c) {
        e = fill(c, b->dev[c & 1], b->pin[c & 1]);
        if (e == hipSuccess) e = hipEventRecord(b->ev[c & 1], s);
    };
    if (nch > 0) start(0);
    for (int64_t c = 0; c < nch && e == hipSuccess; ++c) {
        if (c + 1 < nch) start(c + 1);   // its buffer was used up by chunk c - 1
        if (e == hipSuccess) e = hipEventSynchronize(b->ev[c & 1]);
        if (e == hipSuccess) take(c, b->pin[c & 1]);
    }
    const hipError_t e2 = hipStreamSynchronize(s);   // nothing queued uses the buffers any more
    return e != hipSuccess ? e : e2;
}

// host -> device: give(c, pin) writes the pinned data, drain(c, pin, dev)
// queues the copy and the device's part on s
template <class Give, class Drain> hipError_t pipeline_up(Staging *b, int64_t nch, hipStream_t s, Give give, Drain drain)
{
    hipError_t e = hipSuccess;
    for (int64_t c = 0; c < nch && e == hipSuccess; ++c) {
        if (c >= 2) e = hipEventSynchronize(b->ev[c & 1]);
        if (e != hipSuccess) break;
        give(c, b->pin[c & 1]);
        e = drain(c, b->pin[c & 1], b->dev[c & 1]);
        if (e == hipSuccess && nch > 2) e = hipEventRecord(b->ev[c & 1], s);
    }
    const hipError_t e2 = hipStreamSynchronize(s);
    return e != hipSuccess ? e : e2;
}

// ---------------------------------------------------------------------------
// parcels
// ---------------------------------------------------------------------------
// slot of every caller index
__global__ __launch_bounds__(256) void k_inverse(int64_t n, const int *__restrict__ orig, int *__restrict__ inv)
{
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int o = orig[s];
    if (o >= 0 && o < n) inv[o] = (int)s;
}

__global__ __launch_bounds__(256) void k_iota(int64_t n, int *__restrict__ p)
{
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s < n) p[s] = (int)s;
}

struct IoArrays {
    int ngroups;
    int ncomp[IO_MAX_GROUPS];
    int wide[IO_MAX_GROUPS];
    void *dev[IO_MAX_GROUPS][IO_MAX_COMP];
};

// the staging layout of m parcels: the groups one after the other, each
// [parcel][component], the FP64 groups first; byte offset of a group
__host__ __device__ inline int64_t group_offset(const IoArrays &a, int g, int64_t m)
{
    int64_t o = 0;
    for (int h = 0; h < g; ++h) o += (int64_t)a.ncomp[h] * (a.wide[h] ? 8 : 4) * m;
    return o;
}

// caller indices [lo, lo + m) to (UP: from) the staging buffer; inv null:
// slots are caller indices
template <bool UP>
__global__ __launch_bounds__(256) void k_parcel_io(IoArrays a, const int *__restrict__ inv, int64_t lo, int64_t m,
                                                   char *__restrict__ buf)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int64_t s = inv ? inv[lo + i] : lo + i;
    for (int g = 0; g < a.ngroups; ++g) {
        const int nc = a.ncomp[g];
        char *base = buf + group_offset(a, g, m);
        if (a.wide[g]) {
            double *p = (double *)base + i * nc;
            for (int d = 0; d < nc; ++d) {
                if constexpr (UP) ((double *)a.dev[g][d])[s] = p[d];
                else p[d] = ((const double *)a.dev[g][d])[s];
            }
        } else {
            float *p = (float *)base + i * nc;
            for (int d = 0; d < nc; ++d) {
                if constexpr (UP) ((float *)a.dev[g][d])[s] = p[d];
                else p[d] = ((const float *)a.dev[g][d])[s];
            }
        }
    }
}

int64_t blocks_of(int64_t n) { return (n + 255) / 256; }

// a launch with its own status: the thread's last-error slot, which may hold an
// earlier call's error, is neither read nor cleared
template <class... P, class... A> hipError_t launch(void (*kernel)(P...), int64_t blocks, hipStream_t s, A... a)
{
    std::tuple<P...> v{a...};
    return std::apply(
        [&](P &...p) {
            void *args[] = {(void *)&p...};
            return hipLaunchKernel((const void *)kernel, dim3((unsigned)blocks), dim3(256), args, 0, s);
        },
        v);
}

hipError_t parcel_io(bool up, int64_t n, const int *orig, int *inv, std::vector<IoGroup> groups, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    std::stable_sort(groups.begin(), groups.end(), [](const IoGroup &x, const IoGroup &y) { return x.wide > y.wide; });
    IoArrays a{};
    int64_t per = 0, values = 0;
    for (const IoGroup &g : groups) {
        if (!up && !g.host) continue;   // not asked for
        const int k = a.ngroups++;
        a.ncomp[k] = g.ncomp;
        a.wide[k] = g.wide ? 1 : 0;
        for (int d = 0; d < g.ncomp; ++d) a.dev[k][d] = g.dev[d];
        per += (int64_t)g.ncomp * (g.wide ? 8 : 4);
        values += g.ncomp;
    }
    if (a.ngroups == 0) return hipSuccess;
    if (!up) groups.erase(std::remove_if(groups.begin(), groups.end(), [](const IoGroup &g) { return !g.host; }), groups.end());
    Staging *b = nullptr;
    hipError_t e = stage_get((size_t)(n * per), 0, &b);
    if (e != hipSuccess) return e;
    const int64_t ch = std::min<int64_t>(n, (int64_t)b->size / per & ~int64_t(1));   // even: FP64 groups stay aligned
    const int64_t nch = (n + ch - 1) / ch;
    if (orig) e = launch(k_inverse, blocks_of(n), s, n, orig, inv);
    {
        Team team(std::min(n, ch) * values);
        auto part = [&](int64_t m, int t, int nt, int64_t &lo, int64_t &hi) {
            lo = m * t / nt;
            hi = m * (t + 1) / nt;
        };
        auto chunk = [&](int64_t c) { return std::min(ch, n - c * ch); };
        auto convert = [&](int64_t c, char *pin) {
            const int64_t m = chunk(c);
            team.run([&](int t, int nt) {
                int64_t lo, hi;
                part(m, t, nt, lo, hi);
                for (int g = 0; g < a.ngroups; ++g) {
                    const int64_t nc = a.ncomp[g];
                    char *base = pin + group_offset(a, g, m);
                    double *h = groups[g].host ? groups[g].host + c * ch * nc : nullptr;
                    if (a.wide[g]) {
                        double *p = (double *)base;
                        if (up && !h) std::fill(p + lo * nc, p + hi * nc, 0.0);
                        else if (up) std::copy(h + lo * nc, h + hi * nc, p + lo * nc);
                        else std::copy(p + lo * nc, p + hi * nc, h + lo * nc);
                    } else {
                        float *p = (float *)base;
                        if (up && !h) std::fill(p + lo * nc, p + hi * nc, 0.0f);
                        else if (up)
                            for (int64_t i = lo * nc; i < hi * nc; ++i) p[i] = (float)h[i];
                        else
                            for (int64_t i = lo * nc; i < hi * nc; ++i) h[i] = (double)p[i];
                    }
                }
            });
        };
        const int *map = orig ? inv : nullptr;
        if (e == hipSuccess && !up)
            e = pipeline_down(
                b, nch, s,
                [&](int64_t c, char *dev, char *pin) {
                    const int64_t m = chunk(c);
                    const hipError_t le = launch(k_parcel_io<false>, blocks_of(m), s, a, map, c * ch, m, dev ? dev : b->map[c & 1]);
                    return le != hipSuccess || !dev ? le : hipMemcpyAsync(pin, dev, (size_t)(m * per), hipMemcpyDeviceToHost, s);
                },
                convert);
        else if (e == hipSuccess)
            e = pipeline_up(b, nch, s, convert, [&](int64_t c, char *pin, char *dev) {
                const int64_t m = chunk(c);
                const hipError_t le = dev ? hipMemcpyAsync(dev, pin, (size_t)(m * per), hipMemcpyHostToDevice, s) : hipSuccess;
                if (le != hipSuccess) return le;
                return launch(k_parcel_io<true>, blocks_of(m), s, a, map, c * ch, m, dev ? dev : b->map[c & 1]);
            });
    }
    stage_put(b);
    return e;
}

// ---------------------------------------------------------------------------
// fields
// ---------------------------------------------------------------------------
// x columns of one staging unit: one component's columns i0 .. i0 + XB - 1 of
// the halo layout, all y and z, contiguous in the caller's array
constexpr int XB = 32;

// units [u0, u0 + nu) of 32-bit words to the staging buffer: block = (unit, y,
// 32 z), a 32 x 32 transpose through LDS (x is fastest on the device, z in
// the caller's array)
__global__ __launch_bounds__(256) void k_field_down(Grid g, const int *__restrict__ fld, int u0, int nzb, int *__restrict__ buf)
{
    __shared__ int t[32][33];
    const int hx = g.nx + 3, hy = g.ny + 3, hz = g.nz + 3, nxb = (hx + XB - 1) / XB;
    const int zb = blockIdx.x % nzb, iy = (blockIdx.x / nzb) % hy, ul = blockIdx.x / (nzb * hy);
    const int u = u0 + ul, c = u / nxb, x0 = (u % nxb) * XB, z0 = zb * 32;
    const int lx = threadIdx.x & 31, l8 = threadIdx.x >> 5;
    const int64_t FS = field_stride(g), PS = plane_stride(g);
    const int64_t row = c * FS + (int64_t)wrap(iy - 1, g.ny) * g.nx;
    const int gi = wrap(x0 + lx - 1, g.nx);   // the caller's x index 0 is node -1
    for (int r = l8; r < 32; r += 8)
        if (x0 + lx < hx && z0 + r < hz) t[r][lx] = fld[row + (int64_t)(z0 + r) * PS + gi];
    __syncthreads();
    // units of one component are consecutive in the caller's array; a unit's
    // place in the buffer follows from the columns before it
    const int64_t first = ((int64_t)(u0 / nxb) * hx + (u0 % nxb) * XB), me = (int64_t)c * hx + x0 - first;
    for (int r = l8; r < 32; r += 8)
        if (x0 + r < hx && z0 + lx < hz) buf[((me + r) * hy + iy) * hz + z0 + lx] = t[lx][r];
}

// interior columns [q0, q0 + nq) of component after component from the staging
// buffer: block = (32 columns, y, 32 z), transposed the same way
__global__ __launch_bounds__(256) void k_field_up(Grid g, const float *__restrict__ buf, int q0, int nq, int nzb, float *__restrict__ fld)
{
    __shared__ float t[32][33];
    const int hz = g.nz + 3;
    const int zb = blockIdx.x % nzb, iy = (blockIdx.x / nzb) % g.ny, c0 = blockIdx.x / (nzb * g.ny) * XB, z0 = zb * 32;
    const int lx = threadIdx.x & 31, l8 = threadIdx.x >> 5;
    for (int r = l8; r < XB; r += 8)
        if (c0 + r < nq && z0 + lx < hz) t[lx][r] = buf[((int64_t)(c0 + r) * g.ny + iy) * hz + z0 + lx];
    __syncthreads();
    const int q = q0 + c0 + lx, c = q / g.nx, x = q - c * g.nx;
    float *out = fld + c * field_stride(g) + (int64_t)iy * g.nx + x;
    for (int r = l8; r < 32; r += 8)
        if (c0 + lx < nq && z0 + r < hz) out[(int64_t)(z0 + r) * plane_stride(g)] = t[r][lx];
}

}  // namespace

void release_staging(bool all)
{
    std::vector<Staging *> idle;
    {
        std::lock_guard<std::mutex> lk(stage_mu);
        idle.swap(stage_pool);
        if (!all) {
            auto keep = idle.end();
            for (auto it = idle.begin(); it != idle.end(); ++it)
                if ((*it)->size <= STAGE_MAX && (keep == idle.end() || (*it)->size > (*keep)->size)) keep = it;
            if (keep != idle.end()) {
                stage_pool.push_back(*keep);
                idle.erase(keep);
            }
        }
    }
    for (Staging *b : idle) stage_free(b);
}

hipError_t device_malloc(void **p, size_t bytes)
{
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    release_staging(true);
    return hipMalloc(p, bytes);
}

hipError_t download_parcels(int64_t n, const int *orig, int *inv, const std::vector<IoGroup> &groups, hipStream_t s)
{
    return parcel_io(false, n, orig, inv, groups, s);
}

hipError_t upload_parcels(int64_t n, const int *orig, int *inv, const std::vector<IoGroup> &groups, hipStream_t s)
{
    return parcel_io(true, n, orig, inv, groups, s);
}

hipError_t launch_iota(int64_t n, int *p, hipStream_t s)
{
    return n > 0 ? launch(k_iota, blocks_of(n), s, n, p) : hipSuccess;
}

// Small fields.  A launch and a copy behind it cost more than the transposition
// of a few thousand values here, so small ones are copied as they lie on the
// device; not where their planes are whole pages apart, whose lines then share
// a few sets of the host's cache (32x32x16, one component: 29 us down and 50 up
// this way, 25 and 25 the other).  Pageable copies down of at most 16 KB take
// longer than larger ones (23 us and 13).  16^3, one component: 13 us down and
// 12 up; with a launch and a copy 28 and 25, with a launch that works on the
// pinned memory itself (DIRECT_MAX) 19 and 19.
constexpr size_t PAGEABLE_MIN = 16 << 10, SMALL_DOWN = 160 << 10, SMALL_UP = 320 << 10;
// bytes on the device, 0 where the planes are whole pages apart
static size_t small_field(const Grid &g, int ncomp)
{
    return plane_stride(g) % 1024 == 0 ? 0 : sizeof(float) * (size_t)ncomp * (size_t)field_stride(g);
}
// f(word on the device, value in the caller's array) of the plane -1 of every
// column, the halo columns too when x0 is -1
template <class F> static void small_columns(const Grid &g, int ncomp, int x0, F f)
{
    const int hx = g.nx + 3, hy = g.ny + 3, hz = g.nz + 3, halo = x0 < 0 ? 1 : -1;
    for (int c = 0; c < ncomp; ++c)
        for (int x = x0; x <= g.nx + halo; ++x)
            for (int y = x0; y <= g.ny + halo; ++y) {
                const int wx = (x + g.nx) % g.nx, wy = (y + g.ny) % g.ny;
                f(c * field_stride(g) + (int64_t)wy * g.nx + wx, (((int64_t)c * hx + x + 1) * hy + y + 1) * hz);
            }
}

template <class In, class Out>
hipError_t download_field(const Grid &g, const In *fld, int ncomp, Out *out, hipStream_t s)
{
    static_assert(sizeof(In) == 4, "32-bit words");
    if (const size_t bytes = small_field(g, ncomp); bytes > PAGEABLE_MIN && bytes <= SMALL_DOWN) {
        std::vector<In> h(bytes / 4);
        hipError_t e = hipMemcpyAsync(h.data(), fld, bytes, hipMemcpyDeviceToHost, s);
        const hipError_t e1 = hipStreamSynchronize(s);
        if (e == hipSuccess) e = e1;
        if (e != hipSuccess) return e;
        const In *const raw = h.data();
        small_columns(g, ncomp, -1, [=](int64_t dev, int64_t host) {
            const In *__restrict__ v = raw + dev;
            Out *__restrict__ o = out + host;
            for (int z = 0; z < g.nz + 3; ++z) o[z] = (Out)v[z * plane_stride(g)];
        });
        return hipSuccess;
    }
    const int hx = g.nx + 3, hy = g.ny + 3, hz = g.nz + 3, nxb = (hx + XB - 1) / XB, nzb = (hz + 31) / 32;
    const int64_t line = (int64_t)hy * hz;   // words of one x column
    const int nu = ncomp * nxb;
    Staging *b = nullptr;
    hipError_t e = stage_get((size_t)(4 * ncomp * hx * line), (size_t)(4 * XB * line), &b);
    if (e != hipSuccess) return e;
    const bool direct = !b->dev[0] || 4 * ncomp * hx * line <= DIRECT_MAX;
    const int uch = (int)std::min<int64_t>(nu, (int64_t)b->size / (4 * XB * line));
    const int nch = (nu + uch - 1) / uch;
    auto col = [&](int u) { return (int64_t)(u / nxb) * hx + std::min((u % nxb) * XB, hx); };   // columns before unit u
    {
        Team team(std::min<int64_t>((int64_t)uch * XB, (int64_t)ncomp * hx) * line);
        e = pipeline_down(
            b, nch, s,
            [&](int64_t c, char *dev, char *pin) {
                const int u0 = (int)c * uch, u1 = std::min(nu, u0 + uch);
                if (direct) dev = b->map[c & 1];
                const hipError_t le = launch(k_field_down, (int64_t)(u1 - u0) * hy * nzb, s, g, (const int *)fld, u0, nzb, (int *)dev);
                return le != hipSuccess || direct ? le : hipMemcpyAsync(pin, dev, (size_t)(4 * (col(u1) - col(u0)) * line), hipMemcpyDeviceToHost, s);
            },
            [&](int64_t c, char *pin) {
                const int u0 = (int)c * uch, u1 = std::min(nu, u0 + uch);
                const int64_t m = (col(u1) - col(u0)) * line;
                Out *o = out + col(u0) * line;
                const In *p = (const In *)pin;
                team.run([&](int t, int nt) {
                    for (int64_t i = m * t / nt; i < m * (t + 1) / nt; ++i) o[i] = (Out)p[i];
                });
            });
    }
    stage_put(b);
    return e;
}
template hipError_t download_field(const Grid &, const float *, int, double *, hipStream_t);
template hipError_t download_field(const Grid &, const int *, int, double *, hipStream_t);
template hipError_t download_field(const Grid &, const int *, int, int *, hipStream_t);

hipError_t upload_field(const Grid &g, float *fld, int ncomp, const double *in, hipStream_t s)
{
    if (const size_t bytes = small_field(g, ncomp); bytes > 0 && bytes <= SMALL_UP) {
        Staging *b = nullptr;
        hipError_t e = stage_get(bytes, 0, &b);
        if (e != hipSuccess) return e;
        float *h = (float *)b->pin[0];
        small_columns(g, ncomp, 0, [=](int64_t dev, int64_t host) {
            const double *__restrict__ v = in + host;
            float *__restrict__ o = h + dev;
            for (int z = 0; z < g.nz + 3; ++z) o[z * plane_stride(g)] = (float)v[z];
        });
        e = hipMemcpyAsync(fld, h, bytes, hipMemcpyHostToDevice, s);
        const hipError_t e1 = hipStreamSynchronize(s);
        stage_put(b);
        return e != hipSuccess ? e : e1;
    }
    const int hy = g.ny + 3, hz = g.nz + 3, nzb = (hz + 31) / 32, nq = ncomp * g.nx;
    const int64_t line = (int64_t)g.ny * hz, H = (int64_t)(g.nx + 3) * hy * hz;
    Staging *b = nullptr;
    hipError_t e = stage_get((size_t)(4 * nq * line), (size_t)(4 * line), &b);
    if (e != hipSuccess) return e;
    const bool direct = !b->dev[0] || 4 * nq * line <= DIRECT_MAX;
    const int qch = (int)std::min<int64_t>(nq, (int64_t)b->size / (4 * line));
    auto columns = [&](int64_t c) { return std::min(qch, nq - (int)c * qch); };
    {
        Team team((int64_t)qch * line);
        e = pipeline_up(
            b, (nq + qch - 1) / qch, s,
            [&](int64_t c, char *pin) {
                const int64_t rows = (int64_t)columns(c) * g.ny, first = c * qch * g.ny;   // (component, x, y)
                float *p = (float *)pin;
                team.run([&](int t, int nt) {
                    for (int64_t r = rows * t / nt; r < rows * (t + 1) / nt; ++r) {
                        const int64_t q = (first + r) / g.ny, y = (first + r) % g.ny, x = q % g.nx;
                        const double *src = in + q / g.nx * H + ((x + 1) * hy + (y + 1)) * hz;
                        for (int k = 0; k < hz; ++k) p[r * hz + k] = (float)src[k];
                    }
                });
            },
            [&](int64_t c, char *pin, char *dev) {
                const int n = columns(c);
                if (direct) dev = b->map[c & 1];
                const hipError_t le = direct ? hipSuccess : hipMemcpyAsync(dev, pin, (size_t)(4 * n * line), hipMemcpyHostToDevice, s);
                if (le != hipSuccess) return le;
                return launch(k_field_up, (int64_t)((n + XB - 1) / XB) * g.ny * nzb, s, g, (const float *)dev, (int)c * qch, n, nzb, fld);
            });
    }
    stage_put(b);
    return e;
}

}  // namespace epic
