// for_rotated (fsim_internal.hpp) against ridx for every cell of the grid sizes given as nx ny nz ...; prints the cells compared.
#include "../fluid_simulator_amd/csrc/fsim_internal.hpp"

#include <cstdio>
#include <cstdlib>

int main(int argc, char** argv) {
    long long cells = 0;
    for (int k = 1; k + 2 < argc; k += 3) {
        const int nx = std::atoi(argv[k]), ny = std::atoi(argv[k + 1]), nz = std::atoi(argv[k + 2]), nxp = fsim::rot_planes(nx);
        int64_t next = 0;
        bool good = true;
        fsim::for_rotated(nx, ny, nz, nxp, [&](int64_t i, int64_t r) {
            const int z = (int)(i % nz), y = (int)(i / nz % ny), x = (int)(i / ((int64_t)nz * ny));
            good = good && i == next++ && r == fsim::ridx(x, y, z, nxp, ny, nz) && r < (int64_t)nxp * ny * nz;
        });
        if (!good || next != (int64_t)nx * ny * nz) {
            std::printf("wrong at %d %d %d\n", nx, ny, nz);
            return 1;
        }
        cells += next;
    }
    std::printf("%lld\n", cells);
    return 0;
}
