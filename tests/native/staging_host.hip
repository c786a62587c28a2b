// The staged transfers over a stand-in for the HIP runtime, on the CPU (tests/test_staging_host.py).
// Memory is host memory, and a stream is a queue whose work runs when somebody waits for it, and not
// before, so a missing wait shows as a wrong value or as work left behind.  As in the real runtime a
// failed call leaves its error with the thread until it is fetched.
#include "../../cumpic_amd/csrc/cumc_transfer.hip"

#include <deque>
#include <functional>
#include <map>

namespace fake {
std::recursive_mutex mu;
thread_local hipError_t last = hipSuccess;
struct Call {
    dim3 grid, block;
    hipStream_t stream;
};
thread_local std::vector<Call> calls;
long allocs_left = 1L << 40, launches_left = 1L << 40;
long streams_made = 0, allocs_made = 0, live = 0;

struct Stream {
    std::deque<std::function<void()>> work;
};
std::map<hipStream_t, Stream *> streams;

hipError_t error(hipError_t e)
{
    last = e;
    return e;
}
}  // namespace fake
using fake::error;
#define LOCK std::lock_guard<std::recursive_mutex> lock(fake::mu)

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { hipError_t e = fake::last; fake::last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
static hipError_t alloc(void **p, size_t n)
{
    LOCK;
    if (fake::allocs_left-- <= 0) return error(hipErrorOutOfMemory);
    *p = malloc(n);
    memset(*p, 0x7f, n);
    fake::allocs_made++;
    fake::live++;
    return hipSuccess;
}
static hipError_t release(void *p)
{
    LOCK;
    if (p) fake::live--;
    free(p);
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return alloc(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return alloc(p, n); }
hipError_t hipFree(void *p) { return release(p); }
hipError_t hipHostFree(void *p) { return release(p); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    LOCK;
    *s = (hipStream_t) new char;
    fake::streams[*s] = new fake::Stream;
    fake::streams_made++;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    LOCK;
    delete fake::streams[s];
    fake::streams.erase(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    LOCK;
    std::deque<std::function<void()>> &work = fake::streams.at(s)->work;
    for (; !work.empty(); work.pop_front()) work.front()();
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    LOCK;
    fake::streams.at(st)->work.push_back([=] { memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t s) { fake::calls.push_back({g, b, s}); return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shared, hipStream_t *s)
{
    *g = fake::calls.back().grid;
    *b = fake::calls.back().block;
    *s = fake::calls.back().stream;
    *shared = 0;
    fake::calls.pop_back();
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **a, size_t, hipStream_t st);
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, dim3 *, dim3 *, int *) {}
void __hipUnregisterFatBinary(void **) {}
}

// the two conversion kernels, cell by cell over the threads of the launch
template <bool OUT>
static void convert(const Lay &L, double *soa, int nv, long c0, int n, double *aos, unsigned threads)
{
    for (unsigned t = 0; t < threads && (int)t < n; t++) {
        const long c = c0 + t, sx = L.nx + 6, sy = L.ny + 6;
        const long g = c / (sx * sy) * L.py + c / sx % sy * L.px + c % sx;
        for (int v = 0; v < nv; v++) (OUT ? aos[(long)t * nv + v] : soa[g + v * L.ps]) = OUT ? soa[g + v * L.ps] : aos[(long)t * nv + v];
    }
}

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **a, size_t, hipStream_t st)
{
    LOCK;
    if (fake::launches_left-- <= 0) return error(hipErrorLaunchFailure);
    const Lay L = *(Lay *)a[0];
    double *soa = *(double **)a[1], *aos = *(double **)a[5];
    const int nv = *(int *)a[2], n = *(int *)a[4];
    const long c0 = *(long *)a[3];
    const unsigned threads = grid.x * block.x;
    const bool out = f == (const void *)k_piece_to_aos;
    fake::streams.at(st)->work.push_back([=] {
        if (out) convert<true>(L, soa, nv, c0, n, aos, threads);
        else convert<false>(L, soa, nv, c0, n, aos, threads);
    });
    return hipSuccess;
}

static hipStream_t g_stream;

extern "C" {
// A box's planes filled from host arrays and read back: 0 if every value came back, 1 a wrong value,
// 2 planes with a wrong value, 10 + code for a failed transfer.
int stg_round_trip(int nx, int ny, int nz)
{
    if (!g_stream) hipStreamCreateWithFlags(&g_stream, 0);
    cumc_ctx ctx{};
    Lay &L = ctx.L;
    L.nx = nx; L.ny = ny; L.nz = nz;
    L.px = (nx + 6 + 7) / 8 * 8;
    L.py = L.px * (ny + 6);
    L.ps = (L.py * (nz + 6) + 63) / 64 * 64;
    ctx.stream = g_stream;
    const long n = (long)(nx + 6) * (ny + 6) * (nz + 6);
    std::vector<double> planes(9 * L.ps, -1.0), in(9 * n), out(9 * n, -2.0);
    for (long i = 0; i < 9 * n; i++) in[i] = (double)(i * 7 % 1000003);
    const XferArray a[2] = {{planes.data(), in.data(), 8}, {planes.data() + 8 * L.ps, in.data() + 8 * n, 1}};
    if (int r = transfer_in(&ctx, a, 2)) return 10 + r;
    for (long c = 0; c < n; c++) {
        const long sx = nx + 6, sy = ny + 6, g = c / (sx * sy) * L.py + c / sx % sy * L.px + c % sx;
        for (int v = 0; v < 8; v++)
            if (planes[g + v * L.ps] != in[c * 8 + v]) return 2;
        if (planes[g + 8 * L.ps] != in[8 * n + c]) return 2;
    }
    const XferArray b[2] = {{planes.data(), out.data(), 8}, {planes.data() + 8 * L.ps, out.data() + 8 * n, 1}};
    if (int r = transfer_out(&ctx, b, 2)) return 10 + r;
    return in == out ? 0 : 1;
}
void stg_allow(long allocs, long launches) { fake::allocs_left = allocs; fake::launches_left = launches; }
void stg_retain() { staging_retain(); }
void stg_release() { staging_release(); }
long stg_streams_made() { return fake::streams_made; }
long stg_allocs_made() { return fake::allocs_made; }
long stg_live() { return fake::live; }
// streams with work that nobody waited for
int stg_unfinished()
{
    LOCK;
    int n = 0;
    for (auto &s : fake::streams) n += !s.second->work.empty();
    return n;
}
}
