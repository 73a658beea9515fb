#include "gemm_triple.h"

namespace vkhip {

int launch_triple_128x128(const GemmArgs& g, const Im2colB& im, dim3 grid, int am, int bm) {
    return launch_triple<128, 128, 64, 32, 1, 1, 4, 2>(g, im, grid, am, bm);
}

}  // namespace vkhip
