// The solver's wait for its scalars (fsim_solver.hip) without a device: a thread stands in for the kernel that writes
// them, and the processor is given up through the sched_yield below.
#include "../fluid_simulator_amd/csrc/fsim_solver.hip"

#include <cstdio>
#include <cstdlib>
#include <thread>

static std::atomic<long> g_yields{0};
extern "C" {
int sched_yield() {
    g_yields++;
    return 0;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
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

int main(int argc, char** argv) {
    const int ms = argc > 1 ? std::atoi(argv[1]) : 0;   // until the scalars arrive; below 0: never
    fsim_ctx ctx;
    fsim::SolveScalars host{};
    ctx.scal_host = &host;
    ctx.scal_seq = 7;
    if (ms == 0) host.seq = 7;
    std::thread kernel([&] {
        if (ms <= 0) return;
        std::this_thread::sleep_for(std::chrono::milliseconds(ms));
        __atomic_store_n(&host.seq, 7u, __ATOMIC_RELEASE);
    });
    const int rc = fsim::wait_scalars(&ctx);
    kernel.join();
    std::printf("status %d yields %ld\n", rc, g_yields.load());
    return 0;
}
