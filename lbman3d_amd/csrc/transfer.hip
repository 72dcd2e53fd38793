// transfer.hip — fields between host arrays (FP64) and device arrays.
//
// A field set moves in pieces through 1 MiB buffers of pinned host memory.
// The device side of a piece is one kernel that reads or writes the buffer
// directly: nine fields of a piece are one launch, and no device staging is
// allocated. The host side (conversion between FP64 and the device's type,
// or the copy) of a large set is split over threads that each take the next
// piece, so that conversion, the page faults of fresh arrays and the bus
// overlap. It is what bounds a call: a 256^3 FP32 state took 249 ms by
// pageable copies and one converting thread and takes 30 ms so.
//
// Built without FMA contraction: the equilibrium of an uploaded state is the
// FP64 arithmetic of the reference, bit for bit.
#include <hip/hip_runtime.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <string>
#include <exception>
#include <thread>
#include <vector>

#include "common.hpp"
#include "launch.hpp"
#include "runtime.hpp"
#include "solver_state.hpp"
#include "transfer.hpp"

namespace lbm {

namespace {

constexpr size_t kStageBytes = 1u << 20;
constexpr size_t kKeep = 16;       // buffers kept between calls (16 MiB)
constexpr int kMaxThreads = 8;

// ---- pinned buffers ------------------------------------------------------------
// Shared by every handle of the process; at most kKeep are kept, and all are
// freed with the last handle. Giving one back allocates nothing: it happens at
// the end of a helper thread, where an exception would end the process.
std::mutex g_mu;
void* g_free[kKeep];
size_t g_kept = 0;
int g_users = 0;

void* stage_acquire() {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_kept > 0) return g_free[--g_kept];
    }
    void* p = nullptr;
    return hipHostMalloc(&p, kStageBytes, hipHostMallocPortable | hipHostMallocMapped) == hipSuccess ? p : nullptr;
}
void stage_release(void* p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_users > 0 && g_kept < kKeep) {
            g_free[g_kept++] = p;
            return;
        }
    }
    (void)hipHostFree(p);
}

}  // namespace

void staging_open() {
    std::lock_guard<std::mutex> lock(g_mu);
    ++g_users;
}
void staging_close() {
    void* gone[kKeep];
    size_t count = 0;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (--g_users > 0) return;
        while (g_kept > 0) gone[count++] = g_free[--g_kept];
    }
    while (count > 0) (void)hipHostFree(gone[--count]);
}

namespace {

// Threads for a set of `bytes` host bytes. A thread costs some 30 us, and up to
// a time slice (4 ms measured) where the caller's own worker threads spin on
// every CPU, as OpenMP's do for some milliseconds after a parallel loop: sets
// below 24 MB stay on the calling thread (64 boxes of 6 MB on average: 77 ms a
// sweep against 123 ms with threads; a 59 MB state 7.0 against 11.8 ms).
int host_threads(size_t bytes) {
    if (bytes < ((size_t)24 << 20)) return 1;
    cpu_set_t set;
    CPU_ZERO(&set);
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    return std::max(1, std::min({cpus, kMaxThreads, (int)std::min<size_t>(bytes >> 23, kMaxThreads)}));
}

// work(first cell, cells, buffer, finish) for pieces of at most `most` cells;
// finish() waits for what the piece has put on the stream. `arrays` host values
// belong to a cell. The caller's thread and the helpers work on the handle's
// device: an event can be recorded on a stream of its own device only.
template <typename F>
int for_pieces(const lbm_solver* s, int arrays, long most, F&& work) {
    const OnDevice on(s);
    const hipStream_t stream = s->stream;
    const long cells = s->V;
    const long pieces = (cells + most - 1) / most;
    const long piece = std::min(most, ((cells + pieces - 1) / pieces + 63) / 64 * 64);
    const int threads = (int)std::min<long>(host_threads((size_t)cells * arrays * sizeof(double)), pieces);
    std::atomic<long> next{0};
    std::atomic<int> error{0};
    // The threads join once the stream's earlier work is done: waiting for it
    // in each of them would hold that many CPUs.
    if (threads > 1 && hipStreamSynchronize(stream) != hipSuccess)
        return fail(LBM_ERR_HIP, "field transfer: synchronize failed");
    // A helper that cannot have the device, a buffer or an event leaves the
    // pieces to the others; only the caller's own thread must have them.
    auto run = [&](bool helper) {
        if (helper && hipSetDevice(s->device) != hipSuccess) return;
        void* buffer = stage_acquire();
        hipEvent_t done = nullptr;
        if (!buffer || hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess) {
            stage_release(buffer);
            if (!helper) error = (int)hipErrorOutOfMemory;
            return;
        }
        auto finish = [&]() -> bool {
            hipError_t e = hipGetLastError();
            if (e == hipSuccess) e = hipEventRecord(done, stream);
            if (e == hipSuccess) e = hipEventSynchronize(done);
            if (e != hipSuccess) error = (int)e;
            return e == hipSuccess;
        };
        for (long i; !error && (i = next++) < pieces;) {
            (void)hipGetLastError();   // what an earlier call left is not this piece's error
            work(i * piece, std::min(piece, cells - i * piece), buffer, finish);
        }
        if (error) (void)hipStreamSynchronize(stream);   // nothing may still use the buffer
        (void)hipEventDestroy(done);
        stage_release(buffer);
    };
    std::vector<std::thread> others;
    try {
        others.reserve(threads);
        for (int t = 1; t < threads; ++t) others.emplace_back(run, true);
    } catch (const std::exception&) {
        // fewer threads than asked for: the ones there are take every piece
    }
    run(false);
    for (auto& t : others) t.join();
    if (const int e = error)
        return fail(LBM_ERR_HIP, std::string("field transfer: ") + hipGetErrorString((hipError_t)e));
    return LBM_OK;
}

long piece_cells(int arrays, size_t value) { return (long)(kStageBytes / (arrays * value) / 64 * 64); }

// ---- device side -----------------------------------------------------------------
template <typename T>
struct Arrays {
    T* p[kMaxItems];
};

template <typename T>
__global__ void __launch_bounds__(256) pack_kernel(Arrays<const T> src, long c0, int n, T* out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[(size_t)blockIdx.y * n + i] = src.p[blockIdx.y][c0 + i];
}

struct Bases {
    double v[kMaxItems];
};
template <typename T>
__global__ void __launch_bounds__(256) unpack_kernel(Arrays<T> dst, Bases base, long c0, int n, const double* in) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst.p[blockIdx.y][c0 + i] = (T)(in[(size_t)blockIdx.y * n + i] - base.v[blockIdx.y]);
}

// State of n cells from c0 on: the fields that `has` names come from the
// buffer (one block of n values each, in the order rho, ux, uy, uz, Q), the
// others are the device's own; populations Feq(rho, u) (LbmSolver::Initialize,
// src/lbm_solver.tpp:59-87) from the FP64 values where given. rest: rho0 and
// the device's velocity, nothing from the buffer.
template <typename T>
__global__ void __launch_bounds__(256)
state_kernel(Fields<T> f, double rho0, double base, unsigned has, bool rest, long c0, int n, const double* in) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const long c = c0 + i;
    int block = 0;
    auto given = [&](int field) { return (has >> field) & 1; };
    auto next = [&]() { return in[(size_t)block++ * n + i]; };
    double rho, u[3];
    if (rest || given(0)) {
        rho = rest ? rho0 : next();
        f.rho[c] = (T)(rho - base);
    } else {
        rho = base + (double)f.rho[c];
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (given(1 + a)) {
            u[a] = next();
            f.u[a][c] = (T)u[a];
        } else {
            u[a] = (double)f.u[a][c];
        }
    }
    if (given(4)) {
#pragma unroll
        for (int m = 0; m < 5; ++m) f.q[m][c] = (T)next();
    }
    double fe[kQ];
    feq_node(rho, u[0], u[1], u[2], fe);
#pragma unroll
    for (int j = 0; j < kQ; ++j) f.g[j * f.vs + c] = sizeof(T) == 4 ? (T)(fe[j] - wgt(j) * rho0) : (T)fe[j];
}

dim3 piece_grid(long n, int arrays) { return dim3((unsigned)((n + 255) / 256), (unsigned)arrays); }

template <typename T>
int fetch_typed(const lbm_solver* s, const FetchItem* items, int count) {
    Arrays<const T> src{};
    for (int k = 0; k < count; ++k) src.p[k] = (const T*)items[k].dev;
    return for_pieces(s, count, piece_cells(count, sizeof(T)), [&](long c0, long n, void* buffer, auto finish) {
        hipLaunchKernelGGL(pack_kernel<T>, piece_grid(n, count), dim3(256), 0, s->stream, src, c0, (int)n, (T*)buffer);
        if (!finish()) return;
        const T* in = (const T*)buffer;
        for (int k = 0; k < count; ++k, in += n) {
            double* out = items[k].host + c0;
            if constexpr (sizeof(T) == 8) {
                std::memcpy(out, in, n * sizeof(double));
            } else {
                const double base = items[k].base;
                for (long i = 0; i < n; ++i) out[i] = base + (double)in[i];
            }
        }
    });
}

template <typename T>
int put_typed(const lbm_solver* s, const PutItem* items, int count) {
    Arrays<T> dst{};
    Bases base{};
    for (int k = 0; k < count; ++k) {
        dst.p[k] = (T*)items[k].dev;
        base.v[k] = items[k].base;
    }
    return for_pieces(s, count, piece_cells(count, sizeof(double)), [&](long c0, long n, void* buffer, auto finish) {
        for (int k = 0; k < count; ++k)
            std::memcpy((double*)buffer + k * n, items[k].host + c0, n * sizeof(double));
        hipLaunchKernelGGL(unpack_kernel<T>, piece_grid(n, count), dim3(256), 0, s->stream, dst, base, c0, (int)n,
                           (const double*)buffer);
        (void)finish();
    });
}

template <typename T>
int put_state_typed(const lbm_solver* s, const Fields<T>& f, const double* rho, const double* const u[3],
                    const double* q) {
    const double rho0 = s->cfg.p.density;
    const double base = sizeof(T) == 4 ? rho0 : 0.0;
    const double* src[9];
    unsigned has = 0;
    int count = 0;
    if (rho) {
        has |= 1;
        src[count++] = rho;
    }
    for (int a = 0; a < 3; ++a)
        if (u[a]) {
            has |= 2u << a;
            src[count++] = u[a];
        }
    if (q) {
        has |= 16;
        for (int m = 0; m < 5; ++m) src[count++] = q + m * s->V;
    }
    return for_pieces(s, count, piece_cells(std::max(count, 1), sizeof(double)),
                      [&](long c0, long n, void* buffer, auto finish) {
        for (int k = 0; k < count; ++k) std::memcpy((double*)buffer + k * n, src[k] + c0, n * sizeof(double));
        hipLaunchKernelGGL(state_kernel<T>, piece_grid(n, 1), dim3(256), 0, s->stream, f, rho0, base, has, false, c0,
                           (int)n, (const double*)buffer);
        (void)finish();
    });
}

template <typename T>
int rest_typed(hipStream_t stream, const Fields<T>& f, double rho0, long cells) {
    constexpr long kPiece = 1 << 28;   // cells per launch
    (void)hipGetLastError();           // what an earlier call left is not this one's error
    for (long c0 = 0; c0 < cells; c0 += kPiece) {
        const long n = std::min(kPiece, cells - c0);
        hipLaunchKernelGGL(state_kernel<T>, piece_grid(n, 1), dim3(256), 0, stream, f, rho0,
                           sizeof(T) == 4 ? rho0 : 0.0, 0u, true, c0, (int)n, (const double*)nullptr);
    }
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(stream) != hipSuccess)
        return fail(LBM_ERR_HIP, "initial state failed");
    return LBM_OK;
}

}  // namespace

int fetch_fields(lbm_solver* s, const FetchItem* items, int count) {
    if (count == 0) return LBM_OK;
    return s->fp64 ? fetch_typed<double>(s, items, count) : fetch_typed<float>(s, items, count);
}
int put_fields(lbm_solver* s, const PutItem* items, int count) {
    if (count == 0) return LBM_OK;
    return s->fp64 ? put_typed<double>(s, items, count) : put_typed<float>(s, items, count);
}
int put_state(lbm_solver* s, const double* rho, const double* const u[3], const double* q) {
    return s->fp64 ? put_state_typed(s, s->d64, rho, u, q) : put_state_typed(s, s->d32, rho, u, q);
}
int put_rest(lbm_solver* s) {
    const double rho0 = s->cfg.p.density;
    return s->fp64 ? rest_typed(s->stream, s->d64, rho0, s->V) : rest_typed(s->stream, s->d32, rho0, s->V);
}

int fetch_order_director(lbm_solver* s, double* order, double* director) {
    return for_pieces(s, 4, piece_cells(4, sizeof(double)), [&](long c0, long n, void* buffer, auto finish) {
        double* o = (double*)buffer;
        if (s->fp64) launch_order_director(s->d64, c0, n, o, o + n, s->stream);
        else launch_order_director(s->d32, c0, n, o, o + n, s->stream);
        if (!finish()) return;
        std::memcpy(order + c0, o, n * sizeof(double));
        std::memcpy(director + 3 * c0, o + n, 3 * n * sizeof(double));
    });
}

}  // namespace lbm
