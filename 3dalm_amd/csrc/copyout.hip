// copyout.hip -- device fields to host arrays: components interleaved per cell, FP64.
//
// A kernel interleaves (and widens) the components straight into a pair of pinned host
// slots, while the host copies the other slot into the caller's array.  The caller's
// array is ordinary memory whose pages mostly do not exist yet: one thread faults and
// fills it at 14 GB/s, so kCopyThreads share each slot.  Twelve components of 256x128x128
// (434 MB): 13.4 ms with 8 threads, 33.9, 22.9, 16.5 and 14.9 with 1, 2, 4 and 6 (slots of 2 MiB
// instead of 8: 24 with 4), where the link would take about 8; copying each component whole
// into a temporary array and interleaving it in a host loop took 108 ms.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

#include "ctx.h"

namespace {

constexpr int kCopyThreads = 8;
constexpr long long kSlot = 1 << 20;           // doubles of a slot (8 MiB)
constexpr long long kShare = 1 << 18;          // a thread shares from this many doubles each on
constexpr long long kSmall = 1 << 18;          // fields below take the plain copies

template <typename T>
__global__ __launch_bounds__(BLOCK) void k_interleave(const T* c0, const T* c1, const T* c2, int nc, long long from,
                                                      long long n, double* out) {
    const long long stride = (long long)gridDim.x * BLOCK;
    for (long long o = (long long)blockIdx.x * BLOCK + threadIdx.x; o < n; o += stride) {
        const long long e = from + o;
        double v;
        if (nc == 1) {
            v = (double)c0[e];
        } else {
            const long long cell = e / 3;
            const int q = (int)(e - 3 * cell);
            v = (double)(q == 0 ? c0 : q == 1 ? c1 : c2)[cell];
        }
        out[o] = v;
    }
}

}  // namespace

// two pinned slots of n doubles; false where the host grants none, which is no failure of the
// copy and leaves no text in dalm_last_error
static bool ensure_slots(dalm_ctx* ctx, long long n) {
    if (ctx->out_slot >= n && ctx->may_take(DALM_PATH_COPY_SLOTS)) return true;
    if (ctx->out_pin) {
        (void)hipHostFree(ctx->out_pin);
        ctx->out_pin = nullptr;
        ctx->out_slot = 0;
    }
    hipError_t rc = ctx->may_take(DALM_PATH_COPY_SLOTS) ? hipSuccess : hipErrorOutOfMemory;
    for (hipEvent_t& e : ctx->out_ev)
        if (rc == hipSuccess && !e) rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (rc == hipSuccess)
        rc = hipHostMalloc((void**)&ctx->out_pin, 2 * (size_t)n * sizeof(double), hipHostMallocCoherent);
    if (rc != hipSuccess) {
        (void)hipGetLastError();
        ctx->out_pin = nullptr;
        return false;
    }
    ctx->out_slot = n;
    return true;
}

int copy_out(dalm_ctx* ctx, void* const c[3], int nc, bool f32, double* host) {
    const long long total = ctx->L * nc, slot = std::min({kSlot, std::max((total + 3) / 4, kSmall), total});
    if (total < kSmall || !ensure_slots(ctx, slot)) {
        // no pinned slots: making them takes longer than they save at first (0.71 against 0.34 ms
        // for six fields of 32x20x20, 2.6 against 2.9 at 64x48x48);
        // nor where the host grants none
        ++ctx->taken[DALM_PATH_COPY_PLAIN];
        std::vector<double> tmp(ctx->L);
        std::vector<float> tmpf(f32 ? ctx->L : 0);
        for (int q = 0; q < nc; ++q) {
            void* to = f32 ? (void*)tmpf.data() : (void*)tmp.data();
            HIP_TRY(hipMemcpy(to, c[q], ctx->L * (f32 ? sizeof(float) : sizeof(double)), hipMemcpyDeviceToHost));
            for (long long e = 0; e < ctx->L; ++e) host[e * nc + q] = f32 ? (double)tmpf[e] : tmp[e];
        }
        return DALM_OK;
    }
    ++ctx->taken[DALM_PATH_COPY_SLOTS];
    const long long chunks = (total + slot - 1) / slot;
    const auto length = [&](long long n) { return std::min(slot, total - n * slot); };
    const auto pack = [&](long long n) -> int {
        const long long m = length(n);
        double* out = ctx->out_pin + (n & 1) * slot;
        const dim3 grid((unsigned)std::min<long long>((m + BLOCK - 1) / BLOCK, 1024));
        if (f32)
            hipLaunchKernelGGL(k_interleave<float>, grid, dim3(BLOCK), 0, ctx->stream, (const float*)c[0],
                               (const float*)c[1], (const float*)c[2], nc, n * slot, m, out);
        else
            hipLaunchKernelGGL(k_interleave<double>, grid, dim3(BLOCK), 0, ctx->stream, (const double*)c[0],
                               (const double*)c[1], (const double*)c[2], nc, n * slot, m, out);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventRecord(ctx->out_ev[n & 1], ctx->stream));
        return DALM_OK;
    };
    std::atomic<long long> ready{0}, done{0};
    std::atomic<int> parts{1};  // threads that share a slot, this one included
    const auto copy = [&](long long n, int w) {
        const long long m = length(n), per = (m + parts - 1) / parts, a = std::min(m, w * per), b = std::min(m, a + per);
        memcpy(host + n * slot + a, ctx->out_pin + (n & 1) * slot + a, (size_t)(b - a) * sizeof(double));
    };
    std::vector<std::thread> workers;
    const int want = (int)std::min<long long>(kCopyThreads, total / kShare);
    try {
        workers.reserve(kCopyThreads);
        for (int w = 1; w < want; ++w)
            workers.emplace_back([&, w] {
                for (long long n = 0; n < chunks; ++n) {
                    while (ready.load(std::memory_order_acquire) <= n) std::this_thread::yield();
                    if (ready.load(std::memory_order_relaxed) > chunks) return;  // a failure
                    copy(n, w);
                    done.fetch_add(1, std::memory_order_release);
                }
            });
    } catch (const std::exception&) {  // no thread to be had: the ones there are
    }
    const long long helpers = (long long)workers.size();
    parts = (int)helpers + 1;
    int rc = DALM_OK;
    for (long long n = 0; n < 2 && n < chunks && !rc; ++n) rc = pack(n);
    for (long long n = 0; n < chunks && !rc; ++n) {
        const hipError_t e = hipEventSynchronize(ctx->out_ev[n & 1]);
        if (e != hipSuccess) {
            rc = dalm_fail(ctx, e, "copy to the host", __FILE__, __LINE__);
            break;
        }
        ready.store(n + 1, std::memory_order_release);
        copy(n, 0);
        while (done.load(std::memory_order_acquire) < (n + 1) * helpers) std::this_thread::yield();
        if (n + 2 < chunks) rc = pack(n + 2);
    }
    if (rc) ready.store(chunks + 1, std::memory_order_release);
    for (std::thread& t : workers) t.join();
    if (rc) (void)hipStreamSynchronize(ctx->stream);
    return rc;
}
