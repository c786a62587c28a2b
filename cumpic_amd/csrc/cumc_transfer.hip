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

constexpr size_t STAGE_BYTES = size_t(2) << 20;  // one piece; a unit holds it on the device and pinned on the host
constexpr int MAX_UNITS = 8;                     // per device: at most 16 MiB of either kind of memory
constexpr size_t BYTES_PER_UNIT = size_t(2) << 20;  // a transfer takes one more unit per this much

struct Unit {
    int device = 0;
    hipStream_t stream = nullptr;
    double *dev = nullptr;
    double *pin = nullptr;
};

std::mutex g_mu;
std::condition_variable g_cv;
std::vector<Unit> g_free;   // idle units of every device
int g_made[64] = {0};       // units made per device, idle or in use
int g_users = 0;

void free_unit(Unit &u)
{
    if (u.stream) (void)hipStreamDestroy(u.stream);
    (void)hipFree(u.dev);
    (void)hipHostFree(u.pin);
}

bool make_unit(int device, Unit &u)
{
    u.device = device;
    if (hipStreamCreateWithFlags(&u.stream, hipStreamNonBlocking) == hipSuccess &&
        hipMalloc(&u.dev, STAGE_BYTES) == hipSuccess && hipHostMalloc(&u.pin, STAGE_BYTES, hipHostMallocDefault) == hipSuccess)
        return true;
    free_unit(u);
    (void)hipGetLastError();  // (else the next launch's check on this thread reports it)
    return false;
}

// Between 1 and `want` units of the current device.  A call waits only while other transfers hold all
// of them; none are held while waiting, so every waiter is served in the end.  Empty: out of memory.
std::vector<Unit> acquire(int device, int want)
{
    std::vector<Unit> got;
    got.reserve(want);
    std::unique_lock<std::mutex> lock(g_mu);
    for (;;) {
        for (size_t i = 0; i < g_free.size() && (int)got.size() < want;) {
            if (g_free[i].device == device) {
                got.push_back(g_free[i]);
                g_free.erase(g_free.begin() + (long)i);
            } else {
                i++;
            }
        }
        while ((int)got.size() < want && g_made[device] < MAX_UNITS) {
            Unit u;
            if (!make_unit(device, u)) break;
            g_made[device]++;
            got.push_back(u);
        }
        if (!got.empty() || g_made[device] == 0) return got;
        g_cv.wait(lock);
    }
}

void give_back(std::vector<Unit> &units)
{
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (Unit &u : units) {
            if (g_users > 0) {
                g_free.push_back(u);
            } else {
                g_made[u.device]--;
                free_unit(u);
            }
        }
    }
    units.clear();
    g_cv.notify_all();
}

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

hipError_t run_piece(const Lay &L, const Piece &p, bool out, const Unit &u)
{
    const size_t bytes = (size_t)p.n * p.a.nv * sizeof(double);
    double *host = p.a.host + p.c0 * p.a.nv;
    const dim3 grid(nblk(p.n, 256));
    hipError_t e;
    if (out) {
        hipLaunchKernelGGL(k_piece_to_aos, grid, dim3(256), 0, u.stream, L, (const double *)p.a.soa, p.a.nv, p.c0, p.n, u.dev);
        if ((e = hipGetLastError()) == hipSuccess) e = hipMemcpyAsync(u.pin, u.dev, bytes, hipMemcpyDeviceToHost, u.stream);
    } else {
        std::memcpy(u.pin, host, bytes);
        if ((e = hipMemcpyAsync(u.dev, u.pin, bytes, hipMemcpyHostToDevice, u.stream)) == hipSuccess) {
            hipLaunchKernelGGL(k_piece_to_soa, grid, dim3(256), 0, u.stream, L, p.a.soa, p.a.nv, p.c0, p.n, (const double *)u.dev);
            e = hipGetLastError();
        }
    }
    // (waits after an error too: the unit goes back for the next transfer to use)
    const hipError_t w = hipStreamSynchronize(u.stream);
    if (e == hipSuccess) e = w;
    if (e == hipSuccess && out) std::memcpy(host, u.pin, bytes);
    return e;
}

int transfer(cumc_ctx *ctx, const XferArray *a, int n, bool out)
{
    const Lay &L = ctx->L;
    const long ncell = (long)(L.nx + 6) * (L.ny + 6) * (L.nz + 6);
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    const OnDevice here(ctx->device);
    HIPCHK(ctx, here.e);
    const int device = ctx->device;
    if (device < 0 || device >= 64) return fail(ctx, CUMC_EINVAL, "device index out of range");
    try {
        std::vector<Piece> pieces;
        size_t bytes = 0;
        for (int i = 0; i < n; i++) {
            const long per = (long)(STAGE_BYTES / sizeof(double)) / a[i].nv;
            for (long c = 0; c < ncell; c += per) pieces.push_back({a[i], c, (int)(ncell - c < per ? ncell - c : per)});
            bytes += (size_t)ncell * a[i].nv * sizeof(double);
        }
        int want = 1 + (int)(bytes / BYTES_PER_UNIT);
        want = want > MAX_UNITS ? MAX_UNITS : want;
        std::vector<Unit> units = acquire(device, want);
        if (units.empty()) return fail(ctx, CUMC_ENOMEM, "transfer staging");
        std::atomic<size_t> next{0};
        std::atomic<int> err{(int)hipSuccess};
        auto work = [&](const Unit &u) {
            for (size_t i = next++; i < pieces.size() && err == (int)hipSuccess; i = next++) {
                const hipError_t e = run_piece(L, pieces[i], out, u);
                if (e != hipSuccess) err = (int)e;
            }
        };
        std::vector<std::thread> threads;
        try {
            threads.reserve(units.size());
            for (size_t i = 1; i < units.size(); i++)
                threads.emplace_back([&, i]() {
                    const hipError_t e = hipSetDevice(device);
                    if (e != hipSuccess) err = (int)e;
                    else work(units[i]);
                });
        } catch (const std::exception &) {
            // no further thread to be had: the ones that run share the pieces
        }
        work(units[0]);
        for (std::thread &t : threads) t.join();
        give_back(units);
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
    for (Unit &u : g_free) {
        if (hipSetDevice(u.device) == hipSuccess) free_unit(u);
        g_made[u.device]--;
    }
    g_free.clear();
    if (back) (void)hipSetDevice(cur);
}
