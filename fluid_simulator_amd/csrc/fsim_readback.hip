// fsim_readback.hip — results to host memory.
//
// Particles: the reference keeps them in one vector (hashedParticles.h), here
// they are planes in cell order.  One kernel writes them interleaved, each at
// its index in that vector, and the arrays are copied out as they are.
//
// Copies: a program takes fields, snapshots and particles into memory that it
// has just allocated.  hipMemcpy into such memory runs at 10 GB/s (67 MB in
// 6.7 ms; 4.0 where the pages exist), since it pins the pages of each call and
// one thread makes them.  Here the device writes pieces into pinned slots at up
// to 54 GB/s and several threads copy them on, each piece by one thread, so
// that the pages of the destination are made in parallel.
#include <hip/hip_runtime.h>

#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "fsim_internal.hpp"

namespace fsim {

constexpr size_t kSlotBytes = size_t(2) << 20;
constexpr int kMaxThreads = 8;               // 67 MB of new pages: 1.2 ms by 8 threads, 1.0 by 16, 5.1 by one
// Below it hipMemcpy, which copies pages that exist (small arrays come from a
// program's heap) in 0.1 ms.
constexpr size_t kDirectBytes = size_t(1) << 20;
// A piece costs 10 to 20 us beside its bytes, but the threads need several
// each: 1 MB pieces take 0.40 / 0.63 / 1.33 / 2.46 ms for 8 / 15 / 34 / 67 MB of
// existing pages, 2 MB pieces 0.48 / 0.77 / 1.08 / 1.91 (hipMemcpy 0.49 / 0.86 /
// 1.95 / 3.91; new pages 0.5 / 0.7 / 1.5 / 2.3 against 1.1 / 2.0 / 3.7 / 6.7).
static size_t piece_of(size_t bytes) {
    return bytes >= size_t(24) << 20 ? kSlotBytes : bytes >= size_t(4) << 20 ? kSlotBytes / 2 : kSlotBytes / 4;
}

struct Gather {
    const float* src[15];
    const int32_t* pid;
    float *pos, *vel, *c;   // null: not wanted
    int64_t n;
    int32_t* bad;
};
__global__ void __launch_bounds__(kBlock) k_particles_out(Gather G) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= G.n) return;
    const int32_t id = G.pid[i];
    if (id < 0 || id >= G.n) {
        atomicOr(G.bad, 1);
        return;
    }
    float v[9];
    auto put = [&](float* dst, int first, int count) {
#pragma unroll
        for (int k = 0; k < 9; k++)
            if (k < count) v[k] = G.src[first + k][i];
#pragma unroll
        for (int k = 0; k < 9; k++)
            if (k < count) dst[(int64_t)count * id + k] = v[k];
    };
    if (G.pos) put(G.pos, 0, 3);
    if (G.vel) put(G.vel, 3, 3);
    if (G.c) put(G.c, 6, 9);
}

static int usable_cpus() {
    cpu_set_t set;
    CPU_ZERO(&set);
    return sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
}

// Pinned slots.  A call borrows a set; one idle set is kept for the next call of
// any context (making one takes 1 to 2 ms) until the last context goes.
static std::mutex g_mu;
static char* g_idle = nullptr;
static int g_contexts = 0;

void readback_init(fsim_ctx* ctx) {
    std::lock_guard<std::mutex> lock(g_mu);
    ctx->rb_counted = true;
    g_contexts++;
}
void readback_free(fsim_ctx* ctx) {
    for (auto& e : ctx->rb_ev)
        if (e) (void)hipEventDestroy(e);
    if (!ctx->rb_counted) return;
    char* unused = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        if (--g_contexts == 0) std::swap(unused, g_idle);
    }
    if (unused) (void)hipHostFree(unused);
}

struct PinnedSlots {
    char* p = nullptr;
    PinnedSlots() {
        {
            std::lock_guard<std::mutex> lock(g_mu);
            std::swap(p, g_idle);
        }
        if (p) return;
        // portable: the next borrower may be a context of another GPU
        if (hipHostMalloc(reinterpret_cast<void**>(&p), kSlotBytes * kReadSlots, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
        }
    }
    ~PinnedSlots() {
        {
            std::lock_guard<std::mutex> lock(g_mu);
            if (!g_idle && g_contexts > 0) std::swap(p, g_idle);
        }
        if (p) (void)hipHostFree(p);
    }
    PinnedSlots(const PinnedSlots&) = delete;
    PinnedSlots& operator=(const PinnedSlots&) = delete;
};

static bool make_events(fsim_ctx* ctx) {
    for (auto& e : ctx->rb_ev) {
        if (e || hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess) continue;
        (void)hipGetLastError();
        e = nullptr;
        return false;
    }
    return true;
}

// One copy: the calling thread has the device fill the slots in order and says
// how many pieces have arrived; thread t copies the pieces t, t + threads, ...
struct Copy {
    char* dst;
    const char* src;
    size_t bytes, piece, skew;   // pieces end at multiples of `piece` in the destination's addresses
    int pieces, threads;
    char* pin;
    std::atomic<int> arrived{0};
    std::atomic<bool> stop{false};
    std::atomic<int> left[kReadSlots];   // last piece copied out of the slot, + 1

    size_t from(int k) const { return k == 0 ? 0 : (size_t)k * piece - skew; }
    size_t upto(int k) const { return k + 1 == pieces ? bytes : (size_t)(k + 1) * piece - skew; }
    char* slot(int k) const { return pin + (size_t)(k % kReadSlots) * kSlotBytes; }
    void copy_out(int k) {
        std::memcpy(dst + from(k), slot(k), upto(k) - from(k));
        left[k % kReadSlots].store(k + 1, std::memory_order_release);
    }
    void work(int t) {
        for (int k = t; k < pieces; k += threads) {
            while (arrived.load(std::memory_order_acquire) <= k) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            copy_out(k);
        }
    }
    bool slot_free(int k) const {
        return k < kReadSlots || left[k % kReadSlots].load(std::memory_order_acquire) == k - kReadSlots + 1;
    }
};

static int run_copy(fsim_ctx* ctx, Copy& C, bool alone) {
    int asked = 0;
    for (int k = 0; k < C.pieces; k++) {
        while (asked < C.pieces && asked < k + kReadSlots && (C.slot_free(asked) || asked == k)) {
            while (!C.slot_free(asked)) std::this_thread::yield();   // asked == k: nothing else to wait for
            FSIM_HIP(ctx, hipMemcpyAsync(C.slot(asked), C.src + C.from(asked), C.upto(asked) - C.from(asked),
                                         hipMemcpyDeviceToHost, ctx->stream));
            FSIM_HIP(ctx, hipEventRecord(ctx->rb_ev[asked % kReadSlots], ctx->stream));
            asked++;
        }
        FSIM_HIP(ctx, hipEventSynchronize(ctx->rb_ev[k % kReadSlots]));
        if (alone) C.copy_out(k);
        else C.arrived.store(k + 1, std::memory_order_release);
    }
    return FSIM_OK;
}

static int direct_copy(fsim_ctx* ctx, void* dst, const void* src, size_t bytes) {
    FSIM_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return FSIM_OK;
}

int read_back(fsim_ctx* ctx, void* dst, const void* src, size_t bytes) {
    if (bytes < kDirectBytes) return direct_copy(ctx, dst, src, bytes);
    const PinnedSlots pinned;
    if (!pinned.p || !make_events(ctx)) return direct_copy(ctx, dst, src, bytes);
    Copy C;
    C.dst = static_cast<char*>(dst);
    C.src = static_cast<const char*>(src);
    C.bytes = bytes;
    C.piece = piece_of(bytes);
    C.skew = reinterpret_cast<uintptr_t>(dst) % C.piece;
    C.pieces = (int)((bytes + C.skew + C.piece - 1) / C.piece);
    C.threads = (int)std::min<size_t>({(size_t)kMaxThreads, (size_t)std::max(1, usable_cpus() - 1), bytes / kSlotBytes + 1});
    C.pin = pinned.p;
    for (auto& v : C.left) v.store(0, std::memory_order_relaxed);
    std::thread team[kMaxThreads];
    int started = 0;
    if (C.threads > 1) {
        try {
            for (; started < C.threads; started++) team[started] = std::thread([&C, t = started] { C.work(t); });
        } catch (const std::exception&) {   // no more threads: the copy is made by this one
            C.stop.store(true);
            for (int t = 0; t < started; t++) team[t].join();
            started = 0;
        }
    }
    const int rc = run_copy(ctx, C, started == 0);
    if (rc != FSIM_OK) {
        C.stop.store(true);
        (void)hipStreamSynchronize(ctx->stream);   // nothing writes the slots any more
    }
    for (int t = 0; t < started; t++) team[t].join();
    return rc;
}

int particles_out(fsim_ctx* ctx, float* pos, float* vel, float* c) {
    const int64_t n = ctx->P.n;
    if (n == 0) return FSIM_OK;
    const bool with_c = c && ctx->c_valid;
    if (c && !with_c) std::memset(c, 0, sizeof(float) * 9 * (size_t)n);
    if (!pos && !vel && !with_c) return FSIM_OK;
    // the other particle buffer holds nothing between stages, and has 16 floats a particle
    Gather G{};
    for (int a = 0; a < 3; a++) {
        G.src[a] = ctx->P.pos[a];
        G.src[3 + a] = ctx->P.vel[a];
    }
    for (int k = 0; k < 9; k++) G.src[6 + k] = ctx->P.c[k];
    G.pid = ctx->P.pid;
    G.n = n;
    float* const base = ctx->Palt.base;
    if (pos) G.pos = base;
    if (vel) G.vel = base + 3 * n;
    if (with_c) G.c = base + 6 * n;
    G.bad = ctx->rank;   // free between stages as well
    FSIM_HIP(ctx, hipMemsetAsync(G.bad, 0, sizeof(int32_t), ctx->stream));
    hipLaunchKernelGGL(k_particles_out, dim3(nblocks(n)), dim3(kBlock), 0, ctx->stream, G);
    FSIM_HIP(ctx, hipGetLastError());
    int32_t bad = 0;
    FSIM_HIP(ctx, hipMemcpyAsync(&bad, G.bad, sizeof(bad), hipMemcpyDeviceToHost, ctx->stream));
    FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (bad) return set_err(ctx, FSIM_ERR_INVALID, "corrupt particle ids");
    if (G.pos) FSIM_TRY(read_back(ctx, pos, G.pos, sizeof(float) * 3 * (size_t)n));
    if (G.vel) FSIM_TRY(read_back(ctx, vel, G.vel, sizeof(float) * 3 * (size_t)n));
    if (G.c) FSIM_TRY(read_back(ctx, c, G.c, sizeof(float) * 9 * (size_t)n));
    return FSIM_OK;
}

}  // namespace fsim
