// The sweep kernels of a complex64 arena.
#include "gs_sweep.h"

namespace gs {

void* sweep_kernel_c64(int lr, int vg, int ntq, int route, int sweep, int route2) {
    return sweep_for<float2>(lr, vg, ntq, route, sweep, route2);
}

}  // namespace gs
