// cumc_transfer.hip -- staged transfers between host arrays and device planes (transfer.hpp).
#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "transfer.hpp"

namespace {

constexpr size_t UNIT_BYTES = size_t(2) << 20;  // of device memory and of pinned host memory, per unit
constexpr int MAX_UNITS = 8;                    // per device: at most 16 MiB of either kind of memory
constexpr int MAX_DEVICES = 64;
// A transfer takes one more unit per this much: less for downloads, whose threads also take the page faults of the
// caller's fresh array.  One thread against two: download of 22^3 (2.6 MB) 143 / 119 us, upload of 24^3 (1.9 MB)
// 121 / 124; two against three: download of 30^3 (5.4 MB) 243 / 186.
constexpr size_t BYTES_PER_UNIT_IN = size_t(2) << 20, BYTES_PER_UNIT_OUT = size_t(3) << 19;
// A stream costs about 0.75 ms to make and destroy, in which one unit moves about this much.
constexpr double STREAM_BYTES = double(4 << 20);

struct Unit {
    int device = 0;
    double *dev = nullptr;
    double *pin = nullptr;
};
// Units made together are one allocation of either kind: each costs 0.3 to 0.5 ms to make and as much to
// free, whatever its size.
struct Block {
    int device = 0;
    void *dev = nullptr, *pin = nullptr;
};
struct Device {
    int units = 0, streams = 0;  // made, idle or in use
    int transfers = 0;           // since the first context, counted to three
    std::vector<hipStream_t> idle;
};

std::mutex g_mu;
std::condition_variable g_cv;
std::vector<Unit> g_free;  // idle units of every device
std::vector<Block> g_blocks;
Device g_dev[MAX_DEVICES];
int g_users = 0;

void free_block(Block &b)
{
    (void)hipFree(b.dev);
    (void)hipHostFree(b.pin);
}

// n more units of the current device among the idle ones
bool make_units(int device, int n)
{
    g_blocks.reserve(g_blocks.size() + 1);
    g_free.reserve(g_free.size() + MAX_UNITS);
    Block b;
    b.device = device;
    if (hipMalloc(&b.dev, n * UNIT_BYTES) != hipSuccess || hipHostMalloc(&b.pin, n * UNIT_BYTES, hipHostMallocDefault) != hipSuccess) {
        free_block(b);
        (void)hipGetLastError();  // (else the next launch's check on this thread reports it)
        return false;
    }
    g_blocks.push_back(b);
    for (int i = 0; i < n; i++) {
        Unit u;
        u.device = device;
        u.dev = (double *)((char *)b.dev + i * UNIT_BYTES);
        u.pin = (double *)((char *)b.pin + i * UNIT_BYTES);
        g_free.push_back(u);
    }
    g_dev[device].units += n;
    return true;
}

// The units and streams of one transfer: a unit each for as many host threads, the first on the context's
// own stream and the others on one of these.
struct Lease {
    int device = 0;
    std::vector<Unit> units;
    std::vector<hipStream_t> streams;

    // At least one unit of the current device and at most `want`, for a transfer of `bytes`.  A call waits
    // only while other transfers hold all of them; none are held while waiting, so every waiter is served
    // in the end.  No units: out of memory.
    // The first two transfers (a state up, a result down) take one more unit only while that saves them more
    // than its stream costs: a process that opens a context, moves little and closes it again must not pay for
    // eight.  From the third on a transfer takes all it can use.  64^3 opened, uploaded, stepped four times,
    // downloaded and closed: 15.5 ms with eight units made one by one at the first transfer, 6.4 ms so.
    void take(int dev, int want, double bytes)
    {
        device = dev;
        Device &d = g_dev[dev];
        units.reserve(want);
        streams.reserve(want);
        std::unique_lock<std::mutex> lock(g_mu);
        d.idle.reserve(MAX_UNITS);
        if (d.transfers < 3) d.transfers++;
        for (;;) {
            int free = 0;
            for (const Unit &u : g_free) free += u.device == dev;
            const int room = MAX_UNITS - d.units, lack = want - free < room ? want - free : room;
            // (one unit alone where there is no memory for all)
            if (lack > 0 && !make_units(dev, lack) && free == 0 && lack > 1) make_units(dev, 1);
            for (size_t i = 0; i < g_free.size() && (int)units.size() < want;) {
                if (g_free[i].device == dev) {
                    units.push_back(g_free[i]);
                    g_free.erase(g_free.begin() + (long)i);
                } else {
                    i++;
                }
            }
            if (!units.empty() || d.units == 0) break;
            g_cv.wait(lock);
        }
        while (streams.size() + 1 < units.size()) {
            hipStream_t s = nullptr;
            if (!d.idle.empty()) {
                s = d.idle.back();
                d.idle.pop_back();
            } else {
                const double k = (double)streams.size() + 1.0;
                if (d.streams >= MAX_UNITS - 1 || (d.transfers <= 2 && bytes / (k * (k + 1.0)) < STREAM_BYTES)) break;
                if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) {
                    (void)hipGetLastError();
                    break;
                }
                d.streams++;
            }
            streams.push_back(s);
        }
        while (units.size() > streams.size() + 1) {
            g_free.push_back(units.back());
            units.pop_back();
        }
    }
    ~Lease()
    {
        {
            std::lock_guard<std::mutex> lock(g_mu);
            // (room for all was reserved as they were made)
            for (Unit &u : units) g_free.push_back(u);
            for (hipStream_t s : streams) g_dev[device].idle.push_back(s);
        }
        g_cv.notify_all();
    }
};

// cells [c0, c0 + n) of the box (in the caller's cell order) between the planes and a piece
__global__ __launch_bounds__(256) void k_piece_to_aos(Lay L, const double *__restrict__ soa, int nv, long c0, int n,
                                                      double *__restrict__ aos)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const unsigned sx = L.nx + 6, sy = L.ny + 6, c = (unsigned)(c0 + t), row = c / sx;
    const long g = (long)(row / sy) * L.py + (long)(row % sy) * L.px + (c - row * sx);
    for (int v = 0; v < nv; v++) aos[(long)t * nv + v] = soa[g + v * L.ps];
}
__global__ __launch_bounds__(256) void k_piece_to_soa(Lay L, double *__restrict__ soa, int nv, long c0, int n,
                                                      const double *__restrict__ aos)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const unsigned sx = L.nx + 6, sy = L.ny + 6, c = (unsigned)(c0 + t), row = c / sx;
    const long g = (long)(row / sy) * L.py + (long)(row % sy) * L.px + (c - row * sx);
    for (int v = 0; v < nv; v++) soa[g + v * L.ps] = aos[(long)t * nv + v];
}

// the context's device made current for the calling thread, and the thread's own back afterwards
struct OnDevice {
    int own = -1;
    hipError_t e;
    explicit OnDevice(int device)
    {
        e = hipGetDevice(&own);
        if (e == hipSuccess && own != device) e = hipSetDevice(device);
    }
    ~OnDevice() { if (own >= 0) (void)hipSetDevice(own); }
};

struct Piece {
    XferArray a;
    long c0;
    int n;
};

// One thread's pieces through one unit and one stream.  A thread alone queues them until the unit is full and
// waits for them together, conversions next to each other and copies next to each other (going from one engine to
// the other and back costs about 15 us): a box that fits into a unit costs one wait.  Of several threads each waits
// for every piece, so that one does not queue what another could start.
struct Worker {
    const Lay &L;
    bool out, alone;
    const Unit &u;
    hipStream_t st;
    size_t used = 0;  // bytes of the unit that queued pieces hold
    std::vector<std::pair<const Piece *, size_t>> queued;

    static size_t bytes_of(const Piece &p) { return (size_t)p.n * p.a.nv * sizeof(double); }
    double *at(double *base, size_t off) const { return base + off / sizeof(double); }
    hipError_t convert(const Piece &p, size_t off)
    {
        const dim3 grid(nblk(p.n, 256));
        double *dev = at(u.dev, off);
        if (out)
            hipLaunchKernelGGL(k_piece_to_aos, grid, dim3(256), 0, st, L, (const double *)p.a.soa, p.a.nv, p.c0, p.n, dev);
        else
            hipLaunchKernelGGL(k_piece_to_soa, grid, dim3(256), 0, st, L, p.a.soa, p.a.nv, p.c0, p.n, (const double *)dev);
        return hipGetLastError();
    }
    // the other half of what is queued, and the wait for all of it
    hipError_t flush()
    {
        hipError_t e = hipSuccess;
        if (out && used) e = hipMemcpyAsync(u.pin, u.dev, used, hipMemcpyDeviceToHost, st);
        for (const auto &[p, off] : queued)
            if (!out && e == hipSuccess) e = convert(*p, off);
        const hipError_t w = hipStreamSynchronize(st);
        if (e == hipSuccess) e = w;
        for (const auto &[p, off] : queued)
            if (out && e == hipSuccess) std::memcpy(p->a.host + p->c0 * p->a.nv, at(u.pin, off), bytes_of(*p));
        queued.clear();
        used = 0;
        return e;
    }
    hipError_t put(const Piece &p)
    {
        const size_t bytes = bytes_of(p);
        hipError_t e = used + bytes > UNIT_BYTES ? flush() : hipSuccess;
        if (e != hipSuccess) return e;
        const size_t off = used;
        if (out) {
            e = convert(p, off);
        } else {
            std::memcpy(at(u.pin, off), p.a.host + p.c0 * p.a.nv, bytes);
            e = hipMemcpyAsync(at(u.dev, off), at(u.pin, off), bytes, hipMemcpyHostToDevice, st);
        }
        queued.emplace_back(&p, off);
        used += (bytes + 255) / 256 * 256 < UNIT_BYTES - used ? (bytes + 255) / 256 * 256 : UNIT_BYTES - used;
        return e == hipSuccess && !alone ? flush() : e;
    }
    // shares the pieces with the other workers; leaves nothing queued, after an error either (the unit goes
    // back for the next transfer to use)
    void run(const std::vector<Piece> &pieces, std::atomic<size_t> &next, std::atomic<int> &err)
    {
        hipError_t e = hipSuccess;
        for (size_t i = next++; i < pieces.size() && e == hipSuccess && err == (int)hipSuccess; i = next++) e = put(pieces[i]);
        if (e == hipSuccess) e = flush();
        else (void)hipStreamSynchronize(st);
        if (e != hipSuccess) err = (int)e;
    }
};

int transfer(cumc_ctx *ctx, const XferArray *a, int n, bool out)
{
    const Lay &L = ctx->L;
    const long ncell = (long)(L.nx + 6) * (L.ny + 6) * (L.nz + 6);
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    const OnDevice here(ctx->device);
    HIPCHK(ctx, here.e);
    const int device = ctx->device;
    if (device < 0 || device >= MAX_DEVICES) return fail(ctx, CUMC_EINVAL, "device index out of range");
    try {
        size_t bytes = 0;
        for (int i = 0; i < n; i++) bytes += (size_t)ncell * a[i].nv * sizeof(double);
        const size_t per_unit = out ? BYTES_PER_UNIT_OUT : BYTES_PER_UNIT_IN;
        const int want = bytes / per_unit + 1 > MAX_UNITS ? MAX_UNITS : (int)(bytes / per_unit + 1);
        Lease lease;
        lease.take(device, want, (double)bytes);
        if (lease.units.empty()) return fail(ctx, CUMC_ENOMEM, "transfer staging");
        // pieces of at most a unit for several threads, as many for one as for another (the fewest rounds, and the
        // smallest size that cuts all arrays into no more than that); of a third of a unit for one thread, so that
        // copying one overlaps the engine's work on the one before
        const size_t k = lease.units.size();
        size_t most = UNIT_BYTES / 3;
        auto cut = [&]() {
            size_t c = 0;
            for (int i = 0; i < n; i++) c += ((size_t)ncell * a[i].nv * sizeof(double) + most - 1) / most;
            return c;
        };
        for (size_t rounds = bytes / (k * UNIT_BYTES) + 1; k > 1; rounds++) {
            most = bytes / (k * rounds);
            while (most < UNIT_BYTES && cut() > k * rounds) most += most / 64 + 64;
            most = most < UNIT_BYTES ? most : UNIT_BYTES;
            if (cut() <= k * rounds) break;
        }
        std::vector<Piece> pieces;
        for (int i = 0; i < n; i++) {
            const long per = (long)(most / sizeof(double)) / a[i].nv;
            for (long c = 0; c < ncell; c += per) pieces.push_back({a[i], c, (int)(ncell - c < per ? ncell - c : per)});
        }
        std::atomic<size_t> next{0};
        std::atomic<int> err{(int)hipSuccess};
        std::vector<Worker> workers;
        for (size_t i = 0; i < k; i++) {
            workers.push_back(Worker{L, out, k == 1, lease.units[i], i ? lease.streams[i - 1] : ctx->stream});
            workers[i].queued.reserve(pieces.size());
        }
        std::vector<std::thread> threads;
        threads.reserve(k);
        try {
            for (size_t i = 1; i < k; i++)
                threads.emplace_back([&, i]() {
                    const hipError_t e = hipSetDevice(device);
                    if (e != hipSuccess) err = (int)e;
                    else workers[i].run(pieces, next, err);
                });
        } catch (const std::exception &) {
            // no further thread to be had: the ones that run share the pieces
        }
        workers[0].run(pieces, next, err);
        for (std::thread &t : threads) t.join();
        const hipError_t e = (hipError_t)err.load();
        if (e != hipSuccess) return fail(ctx, CUMC_EHIP, std::string("transfer: ") + hipGetErrorString(e));
    } catch (const std::exception &x) {
        return fail(ctx, CUMC_ENOMEM, std::string("transfer: ") + x.what());
    }
    return CUMC_OK;
}

}  // namespace

int transfer_in(cumc_ctx *ctx, const XferArray *a, int n) { return transfer(ctx, a, n, false); }
int transfer_out(cumc_ctx *ctx, const XferArray *a, int n) { return transfer(ctx, a, n, true); }

void staging_retain()
{
    std::lock_guard<std::mutex> lock(g_mu);
    g_users++;
}

void staging_release()
{
    std::lock_guard<std::mutex> lock(g_mu);
    if (--g_users > 0) return;
    int cur = 0;
    const bool back = hipGetDevice(&cur) == hipSuccess;
    for (Block &b : g_blocks)
        if (hipSetDevice(b.device) == hipSuccess) free_block(b);
    g_blocks.clear();
    g_free.clear();
    for (int i = 0; i < MAX_DEVICES; i++) {
        if (!g_dev[i].idle.empty() && hipSetDevice(i) == hipSuccess)
            for (hipStream_t st : g_dev[i].idle) (void)hipStreamDestroy(st);
        g_dev[i] = Device{};
    }
    if (back) (void)hipSetDevice(cur);
}
