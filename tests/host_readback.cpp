// The host side of fsim_readback.hip over a stand-in runtime: copies run at once in the launching thread, so that what
// the host does (the memory it asks for, its waits, its threads) can be tested without a device.  One case per run.
#include "../fluid_simulator_amd/csrc/fsim_readback.hip"

#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

static int g_mallocs = 0, g_frees = 0, g_copies = 0, g_plain = 0, g_launches = 0, g_lost = -1;
static unsigned g_flags = 0;

extern "C" {
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags) {
    g_mallocs++;
    g_flags = flags;
    *p = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    g_frees++;
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
    g_copies++;
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind) {
    g_plain++;
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* dst, int v, size_t bytes, hipStream_t) {
    std::memset(dst, v, bytes);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
// k_piece; the one numbered g_lost is never seen to finish
hipError_t hipLaunchKernel(const void*, dim3, dim3, void** args, size_t, hipStream_t) {
    const fsim::Piece& P = *static_cast<const fsim::Piece*>(args[0]);
    if (g_launches++ == g_lost) return hipSuccess;
    std::memcpy(P.slot, P.src, P.bytes);
    __atomic_store_n(P.flag, P.value, __ATOMIC_RELEASE);
    return hipSuccess;
}
static dim3 g_grid, g_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
    g_grid = g;
    g_block = b;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shared, hipStream_t* s) {
    *g = g_grid;
    *b = g_block;
    *shared = 0;
    *s = nullptr;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}
namespace fsim {
int set_err(fsim_ctx* ctx, int code, const std::string& msg) {
    ctx->err = msg;
    return code;
}
}  // namespace fsim

// copies `bytes` out and says whether they came back whole
static int copy(fsim_ctx* ctx, size_t bytes) {
    std::vector<char> src(bytes), dst(bytes + 64);
    for (size_t i = 0; i < bytes; i++) src[i] = (char)(i * 2654435761u >> 24);
    const int rc = fsim::read_back(ctx, dst.data() + 4, src.data(), bytes);
    const bool whole = std::memcmp(dst.data() + 4, src.data(), bytes) == 0;
    std::printf("copy %zu status %d whole %d mallocs %d frees %d direct %d\n", bytes, rc, whole, g_mallocs, g_frees, g_copies);
    return rc;
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (argc > 2 && std::string(argv[2]) == "alone") {   // one CPU: the calling thread copies alone
        cpu_set_t one;
        CPU_ZERO(&one);
        CPU_SET(sched_getcpu(), &one);
        sched_setaffinity(0, sizeof(one), &one);
    }
    unsigned count = 0;
    fsim_ctx ctx;
    ctx.red_count = &count;
    fsim::readback_init(&ctx);
    if (what == "memory") {
        copy(&ctx, size_t(67) << 20);
        std::printf("flags coherent %d portable %d noncoherent %d\n", (g_flags & hipHostMallocCoherent) != 0,
                    (g_flags & hipHostMallocPortable) != 0, (g_flags & hipHostMallocNonCoherent) != 0);
    } else if (what == "lost") {
        g_lost = argc > 3 ? std::atoi(argv[3]) : 0;
        copy(&ctx, size_t(67) << 20);
        std::printf("said: %s\n", ctx.err.c_str());
        g_lost = -1;
        copy(&ctx, size_t(67) << 20);
    } else if (what == "direct") {
        for (int k = 2; k < argc; k++) {
            g_copies = g_plain = 0;
            copy(&ctx, (size_t)std::atoll(argv[k]));
            std::printf("plain %d on the stream %d\n", g_plain, g_copies);
        }
    } else {
        return 2;
    }
    fsim::readback_free(&ctx);
    std::printf("end mallocs %d frees %d\n", g_mallocs, g_frees);
    return 0;
}
