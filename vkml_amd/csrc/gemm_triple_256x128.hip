#include "gemm_triple.h"

namespace vkhip {

int launch_triple_256x128(const GemmArgs& g, const Im2colB& im, dim3 grid, int am, int bm) {
    return launch_triple<256, 128, 64, 64, 1, 2, 2, 2>(g, im, grid, am, bm);
}

}  // namespace vkhip
