// Steps an ensemble of two PIC/FLIP dam breaks from captured graphs and prints,
// after each step, the largest iteration count and how many graphs have been
// instantiated: the library's calls of hipGraphInstantiate come here first.
//
// usage: graph_captures <columns> <steps>
#include <dlfcn.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../include/fs2d.h"

static int g_instantiated = 0;

extern "C" __attribute__((visibility("default"))) int hipGraphInstantiate(void** exec, void* graph, void** node,
                                                                           char* log, size_t size) {
    typedef int (*Fn)(void**, void*, void**, char*, size_t);
    static const Fn next = (Fn)dlsym(RTLD_NEXT, "hipGraphInstantiate");
    if (!next) return 1;
    g_instantiated++;
    return next(exec, graph, node, log, size);
}

int main(int argc, char** argv) {
    if (argc != 3) return 2;
    const int nx = std::atoi(argv[1]), ny = 300, steps = std::atoi(argv[2]);
    std::vector<uint8_t> cells((size_t)nx * ny, FS2D_EMPTY);
    for (int j = 0; j < ny; j++)
        for (int i = 0; i < nx; i++) {
            if (i == 0 || j == 0 || i == nx - 1 || j == ny - 1) cells[(size_t)j * nx + i] = FS2D_SOLID;
            else if (i < 60 && j < 280) cells[(size_t)j * nx + i] = FS2D_FLUID;
        }
    fs2d_config c[2];
    for (fs2d_config& x : c) {
        fs2d_config_init(&x);
        x.size_x = nx;
        x.size_y = ny;
        x.dt = 0.002;
        x.dx = 1.0 / 64;
        x.pic_flip_alpha = 0.05;
        x.initial_values = cells.data();
        x.tau = 0.97;
        x.pcg_tol = 1e-6;
        x.pcg_max_iters = 500;
    }
    fs2d_batch* b = nullptr;
    if (fs2d_batch_create(c, 2, &b) != FS2D_OK || fs2d_batch_set_graph(b, 1) != FS2D_OK) {
        std::fprintf(stderr, "%s\n", fs2d_batch_last_error(b));
        return 1;
    }
    for (int k = 0; k < steps; k++) {
        if (fs2d_batch_step(b) < 0) {
            std::fprintf(stderr, "%s\n", fs2d_batch_last_error(b));
            return 1;
        }
        fs2d_stats st;
        if (fs2d_get_stats(fs2d_batch_sim(b, 0), &st) != FS2D_OK) return 1;
        std::printf("%d %d\n", (int)st.pcg_iters, g_instantiated);
        std::fflush(stdout);
    }
    fs2d_batch_destroy(b);
    return 0;
}
