#include "gemm_triple.h"

namespace vkhip {

int launch_triple_64x64(const GemmArgs& g, const Im2colB& im, dim3 grid, int am, int bm) {
    return launch_triple<64, 64, 32, 32, 2, 2, 2, 2>(g, im, grid, am, bm);
}

}  // namespace vkhip
