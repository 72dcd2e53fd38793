// The host side of the field transfers (lbman3d_amd/csrc/transfer.hip) on a
// stand-in for the HIP runtime with two devices: no GPU, no HIP library. The
// stand-in keeps what the runtime documents: the current device and the last
// error belong to a thread, an event belongs to the device that was current
// when it was made, recording it on a stream of another device is an error, a
// kernel is launched on a stream of the current device, and the kernels' own
// work is done here in plain loops.
//
// transfer_check SCENARIO: prints "ok" and leaves 0, or says what is wrong.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>

#include "../../lbman3d_amd/csrc/transfer.hip"

using namespace lbm;

// ---- stand-in runtime -------------------------------------------------------------
struct ihipStream_t {
    int device;
};
struct ihipEvent_t {
    int device;
};

namespace {
thread_local int t_device = 0;
thread_local hipError_t t_last = hipSuccess;
thread_local bool t_helper = true;        // main() clears it
thread_local bool t_no_memory = false;    // operator new throws
std::atomic<bool> g_no_memory_after_event{false};
std::atomic<int> g_refuse_helpers{0};   // 1: buffers, 2: events, 3: devices
std::atomic<int> g_helpers{0}, g_launches{0};

hipError_t status(hipError_t e) {
    if (e != hipSuccess) t_last = e;
    return e;
}
struct Config {
    dim3 grid, block;
    hipStream_t stream;
};
thread_local Config t_config;

template <typename T>
bool emulate(const void* fn, dim3 grid, void** args) {
    if (fn == (const void*)pack_kernel<T>) {
        const auto& src = *(Arrays<const T>*)args[0];
        const long c0 = *(long*)args[1];
        const int n = *(int*)args[2];
        T* out = *(T**)args[3];
        for (unsigned k = 0; k < grid.y; ++k) std::memcpy(out + (size_t)k * n, src.p[k] + c0, n * sizeof(T));
        return true;
    }
    if (fn == (const void*)unpack_kernel<T>) {
        const auto& dst = *(Arrays<T>*)args[0];
        const auto& base = *(Bases*)args[1];
        const long c0 = *(long*)args[2];
        const int n = *(int*)args[3];
        const double* in = *(const double**)args[4];
        for (unsigned k = 0; k < grid.y; ++k)
            for (int i = 0; i < n; ++i) dst.p[k][c0 + i] = (T)(in[(size_t)k * n + i] - base.v[k]);
        return true;
    }
    return fn == (const void*)state_kernel<T>;
}
}  // namespace

void* operator new(size_t n) {
    if (t_no_memory) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipGetDevice(int* d) {
    *d = t_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    if (t_helper) ++g_helpers;
    if (t_helper && g_refuse_helpers == 3) return status(hipErrorInvalidDevice);
    t_device = d;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (t_helper && g_refuse_helpers == 1) return status(hipErrorOutOfMemory);
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (t_helper && g_refuse_helpers == 2) return status(hipErrorOutOfMemory);
    *e = new ihipEvent_t{t_device};
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    if (g_no_memory_after_event) t_no_memory = true;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    return e->device == s->device ? hipSuccess : status(hipErrorInvalidHandle);
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) {
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t s) {
    t_config = {grid, block, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* s) {
    *grid = t_config.grid;
    *block = t_config.block;
    *shared = 0;
    *s = t_config.stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3, void** args, size_t, hipStream_t s) {
    if (s->device != t_device) return status(hipErrorInvalidHandle);
    ++g_launches;
    return emulate<float>(fn, grid, args) || emulate<double>(fn, grid, args) ? hipSuccess : status(hipErrorInvalidValue);
}
}

namespace lbm {
thread_local std::string g_last_error;
int fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}
template <typename T>
void launch_order_director(const Fields<T>&, long, long, double*, double*, hipStream_t) {}
template void launch_order_director<double>(const Fields<double>&, long, long, double*, double*, hipStream_t);
template void launch_order_director<float>(const Fields<float>&, long, long, double*, double*, hipStream_t);
}  // namespace lbm

// ---- scenarios --------------------------------------------------------------------
namespace {
int g_failures = 0;
void expect(bool ok, const char* what) {
    if (ok) return;
    ++g_failures;
    std::printf("FAILED: %s (%s)\n", what, g_last_error.c_str());
}

// A field set of `count` arrays there and back on a handle of `device`.
void round_trip(int device, long cells, int count) {
    ihipStream_t stream{device};
    lbm_solver s;
    s.device = device;
    s.stream = &stream;
    s.V = cells;
    std::vector<double> host(cells * count), dev(cells * count, -1.0), back(cells * count, -2.0);
    for (size_t i = 0; i < host.size(); ++i) host[i] = 0.5 * (double)i;
    PutItem put[kMaxItems];
    FetchItem fetch[kMaxItems];
    for (int k = 0; k < count; ++k) {
        put[k] = {&dev[k * cells], &host[k * cells], 0.0};
        fetch[k] = {&dev[k * cells], &back[k * cells], 0.0};
    }
    staging_open();
    expect(put_fields(&s, put, count) == LBM_OK, "upload");
    expect(dev == host, "device values");
    expect(fetch_fields(&s, fetch, count) == LBM_OK, "download");
    expect(back == host, "host values");
    staging_close();
}

constexpr long kSmall = 5000, kLarge = 500000;   // 9 arrays: 0.4 MB on one thread, 36 MB on several
}  // namespace

int main(int argc, char** argv) {
    t_helper = false;
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "plain") {
        round_trip(0, kSmall, 9);
        round_trip(0, kLarge, 9);
        expect(g_helpers > 0, "helper threads took part");
    } else if (what == "earlier-error") {
        // an error that an earlier call of this thread left is not the transfer's
        for (long cells : {kSmall, kLarge}) {
            t_last = hipErrorOutOfMemory;
            round_trip(0, cells, 9);
        }
    } else if (what == "other-device") {
        // the handle's device is not the caller's current one
        round_trip(1, kSmall, 9);
        round_trip(1, kLarge, 9);
        expect(t_device == 0, "the caller's device is current again");
    } else if (what == "helper-buffer" || what == "helper-event" || what == "helper-device") {
        // helpers without a buffer, event or device leave the work to the caller
        g_refuse_helpers = what == "helper-buffer" ? 1 : (what == "helper-event" ? 2 : 3);
        round_trip(0, kLarge, 9);
        expect(g_helpers > 0, "helper threads were started");
    } else if (what == "host-memory") {
        // a transfer that ends needs no host memory
        g_no_memory_after_event = true;
        ihipStream_t stream{0};
        lbm_solver s;
        s.stream = &stream;
        s.V = kLarge;
        std::vector<double> host(9 * kLarge, 1.0), dev(9 * kLarge);
        PutItem put[9];
        for (int k = 0; k < 9; ++k) put[k] = {&dev[k * kLarge], &host[k * kLarge], 0.0};
        staging_open();
        const int r = put_fields(&s, put, 9);
        t_no_memory = false;
        g_no_memory_after_event = false;
        expect(r == LBM_OK && dev == host, "upload");
        staging_close();
    } else {
        std::printf("unknown scenario\n");
        return 2;
    }
    if (!g_failures) std::printf("ok\n");
    return g_failures ? 1 : 0;
}
