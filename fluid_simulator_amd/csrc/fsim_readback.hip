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
#include <chrono>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "fsim_internal.hpp"

namespace fsim {

constexpr size_t kSlotBytes = size_t(2) << 20;
constexpr int kReadSlots = 12;                // pinned slots
constexpr int kMaxThreads = 8;               // 67 MB of new pages: 1.2 ms by 8 threads, 1.0 by 16, 5.1 by one
// Below it hipMemcpy, which copies pages that exist (small arrays come from a
// program's heap) in 0.1 ms.  us by hipMemcpy, and by hipMemcpyAsync with the
// stream's synchronisation: 4 KB 15 and 23, 16 KB 19 and 27, 64 KB 36 and 36,
// 128 KB 15 and 23, 160 KB 17 and 73, 512 KB 31 and 31.  Where the two take
// turns, each is slower than by itself (128 KB 62).
constexpr size_t kDirectBytes = size_t(1) << 20;
// The threads need several pieces each, and a piece costs its launch.  ms for
// existing pages of 4 / 8 / 15 / 34 / 67 MB: 0.19 / 0.32 / 0.52 / 0.95 / 1.7
// (with hipMemcpyAsync and an event per piece 0.25 / 0.41 / 0.67 / 1.1 / 2.0,
// hipMemcpy 0.25 / 0.49 / 0.86 / 1.95 / 3.91); new pages 0.4 / 0.45 / 0.66 / 1.4
// / 2.1 (hipMemcpy 0.7 / 1.1 / 2.0 / 3.7 / 6.7).
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
// any context until the last context goes.  Making and releasing one takes 0.1
// to 1 ms: a program that holds one context at a time pays it for each (create,
// a result of 2.9 / 8.4 / 21 MB and close: 3.6 / 5.3 / 7.9 ms, of which copies
// by hipMemcpy alone would save up to 0.8, but 6.5 more in the first context of
// the process).
static std::mutex g_mu;
static char* g_idle = nullptr;
static int g_contexts = 0;

void readback_init(fsim_ctx* ctx) {
    std::lock_guard<std::mutex> lock(g_mu);
    ctx->rb_counted = true;
    g_contexts++;
}
void readback_free(fsim_ctx* ctx) {
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
        // portable: the next borrower may be a context of another GPU.  coherent: the host takes flags and data
        // while later kernels run, and any flag but this one would leave that to HIP_HOST_COHERENT (off by
        // default), with the data promised only once the stream has been synchronised
        if (hipHostMalloc(reinterpret_cast<void**>(&p), kSlotBytes * kReadSlots + sizeof(unsigned) * kReadSlots,
                          hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
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

// A piece into its pinned slot, by a kernel: the next piece's follows without an
// event between them (which cost 20 us a piece), and the last block to finish
// stores the piece's number + 1 in the slot's flag, behind the data.  The flags
// are in pinned memory as well.
constexpr int kPieceBlocks = 64;
struct Piece {
    const char* src;
    char* slot;
    unsigned bytes;
    unsigned* finished;   // blocks done (0 between launches)
    unsigned* flag;
    unsigned value;
};
__global__ void __launch_bounds__(256) k_piece(Piece P) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const unsigned words = P.bytes / 16, step = gridDim.x * 256;
    // 16 bytes at a time where the source allows it (the slots are aligned), 4 otherwise
    if ((reinterpret_cast<uintptr_t>(P.src) & 15) == 0) {
        const u32x4* const from = reinterpret_cast<const u32x4*>(P.src);
        u32x4* const to = reinterpret_cast<u32x4*>(P.slot);
        for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < words; i += step) to[i] = from[i];
        for (unsigned i = words * 16 + blockIdx.x * 256 + threadIdx.x; i < P.bytes; i += step) P.slot[i] = P.src[i];
    } else if ((reinterpret_cast<uintptr_t>(P.src) & 3) == 0) {
        for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < P.bytes / 4; i += step)
            reinterpret_cast<unsigned*>(P.slot)[i] = reinterpret_cast<const unsigned*>(P.src)[i];
        for (unsigned i = P.bytes / 4 * 4 + blockIdx.x * 256 + threadIdx.x; i < P.bytes; i += step) P.slot[i] = P.src[i];
    } else {
        for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < P.bytes; i += step) P.slot[i] = P.src[i];
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) {
        if (__hip_atomic_fetch_add(P.finished, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
            __hip_atomic_store(P.finished, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __threadfence_system();
            __hip_atomic_store(P.flag, P.value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// One copy: the calling thread has the device fill the slots in order; thread t
// copies the pieces t, t + threads, ... as their flags arrive.
struct Copy {
    char* dst;
    const char* src;
    size_t bytes, piece, skew;   // pieces end at multiples of `piece` in the destination's addresses
    int pieces, threads;
    char* pin;
    unsigned* flags;                     // of the slots, pinned
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
            while (!arrived(k)) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            copy_out(k);
        }
    }
    bool arrived(int k) const { return __atomic_load_n(&flags[k % kReadSlots], __ATOMIC_ACQUIRE) == (unsigned)k + 1; }
    bool slot_free(int k) const {
        return k < kReadSlots || left[k % kReadSlots].load(std::memory_order_acquire) == k - kReadSlots + 1;
    }
};

// The stream's work is done: a piece whose flag is not there now never arrives.
static int expect_arrived(fsim_ctx* ctx, const Copy& C, int k) {
    return C.arrived(k) ? FSIM_OK : set_err(ctx, FSIM_ERR_HIP, "a piece of the copy to host memory did not arrive");
}

// Waits for `there`, which follows once piece k has arrived.  A device that
// takes long is waited for as a whole, which also reports its failure.
template <class F>
static int wait_until(fsim_ctx* ctx, const Copy& C, int k, F&& there) {
    auto t0 = std::chrono::steady_clock::now();
    while (!there()) {
        std::this_thread::yield();
        if (std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(100)) continue;
        FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
        FSIM_TRY(expect_arrived(ctx, C, k));
        t0 = std::chrono::steady_clock::now();
    }
    return FSIM_OK;
}

static int run_copy(fsim_ctx* ctx, Copy& C, bool alone) {
    auto ask = [&](int k) -> int {
        const Piece P{C.src + C.from(k), C.slot(k), (unsigned)(C.upto(k) - C.from(k)), ctx->red_count,
                      &C.flags[k % kReadSlots], (unsigned)k + 1};
        hipLaunchKernelGGL(k_piece, dim3(kPieceBlocks), dim3(256), 0, ctx->stream, P);
        FSIM_HIP(ctx, hipGetLastError());
        return FSIM_OK;
    };
    int asked = 0;
    for (int k = 0; k < C.pieces; k++) {
        if (alone) {
            for (; asked < std::min(C.pieces, k + kReadSlots); asked++) FSIM_TRY(ask(asked));
            FSIM_TRY(wait_until(ctx, C, k, [&] { return C.arrived(k); }));
            C.copy_out(k);
        } else {
            FSIM_TRY(wait_until(ctx, C, k - kReadSlots, [&] { return C.slot_free(k); }));
            FSIM_TRY(ask(k));
        }
    }
    FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    // the threads wait for the last pieces' flags (the others' have been copied out)
    for (int k = std::max(0, C.pieces - kReadSlots); k < C.pieces; k++) FSIM_TRY(expect_arrived(ctx, C, k));
    return FSIM_OK;
}

static int direct_copy(fsim_ctx* ctx, void* dst, const void* src, size_t bytes) {
    FSIM_HIP(ctx, hipStreamSynchronize(ctx->stream));
    FSIM_HIP(ctx, hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return FSIM_OK;
}

int read_back(fsim_ctx* ctx, void* dst, const void* src, size_t bytes) {
    if (bytes < kDirectBytes) return direct_copy(ctx, dst, src, bytes);
    const PinnedSlots pinned;
    if (!pinned.p) return direct_copy(ctx, dst, src, bytes);
    Copy C;
    C.dst = static_cast<char*>(dst);
    C.src = static_cast<const char*>(src);
    C.bytes = bytes;
    C.piece = piece_of(bytes);
    C.skew = reinterpret_cast<uintptr_t>(dst) % C.piece;
    C.pieces = (int)((bytes + C.skew + C.piece - 1) / C.piece);
    C.threads = (int)std::min<size_t>({(size_t)kMaxThreads, (size_t)std::max(1, usable_cpus() - 1), bytes / kSlotBytes + 1});
    C.pin = pinned.p;
    C.flags = reinterpret_cast<unsigned*>(pinned.p + kSlotBytes * kReadSlots);
    for (int k = 0; k < kReadSlots; k++) __atomic_store_n(&C.flags[k], 0u, __ATOMIC_RELEASE);
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
