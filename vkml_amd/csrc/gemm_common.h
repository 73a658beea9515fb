// What the GEMM sources share: launch arguments, epilogues, the tile order and
// the implicit-im2col map.
#pragma once

#include "common.h"

namespace vkhip {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// An epilogue adds bias[(i % ncols) * bias_stride] to the folded value and
// then applies relu (v <= 0 ? 0 : v) when asked -- the ADD and RELU nodes'
// arithmetic on the product's output -- or (mask != null) takes the relu
// gradient mask[i] <= 0 ? +0 : v, mask laid out as the output (RELU_BACKWARD
// with the product as its incoming gradient; a NaN mask passes v).
struct FoldEpilogue {
    const float* bias;
    int64_t bias_stride;
    uint32_t ncols, relu;
    const float* mask;
};

__device__ __forceinline__ float apply_epilogue(const FoldEpilogue& epi, uint64_t i, float v) {
    if (epi.bias) {
        v = v + epi.bias[static_cast<int64_t>(i % epi.ncols) * epi.bias_stride];
        if (epi.relu) v = v <= 0.0f ? 0.0f : v;
    }
    if (epi.mask && epi.mask[i] <= 0.0f) v = 0.0f;
    return v;
}

struct GemmArgs {
    const float* a;
    const float* b;
    float* c;
    int64_t sa0, sa1, sam, sak;  // A strides: batch0, batch1, m, k (elements)
    int64_t sb0, sb1, sbk, sbn;  // B strides: batch0, batch1, k, n
    uint32_t b1;                 // extent of batch axis 1
    uint32_t m, n, k;
    uint32_t tiles_m, tiles_n;
    uint32_t ktiles;             // ceil(K / BK)
    uint32_t chunk;              // K-tiles per split partition
    uint64_t split_stride;       // elements between partition slices of c
    uint32_t a_vec, b_vec;       // 16-byte loads along k are legal
    uint32_t flat_splits;        // > 0: split grid launched flat, grid.x = tiles * flat_splits
    uint32_t pairs;              // paired direct kernel: partition pairs per tile
    // Convolution epilogue (unsplit register-path conv kernel only): out =
    // acc + bias[row * bias_stride] when bias is set, then relu (x <= 0 ? 0 :
    // x) when relu is set -- the ADD and RELU nodes' arithmetic.
    const float* bias;
    int64_t bias_stride;
    uint32_t relu;
    // A product's epilogue (MATMUL_BIAS, MATMUL_RELU_BACKWARD) applied by the
    // kernel that writes the output (unsplit plans; split plans: the fold).
    FoldEpilogue epi;
};

// The product epilogue at output (z, row, col), when the launch has one.
__device__ __forceinline__ float product_epilogue(const GemmArgs& g, uint32_t z, uint32_t row,
                                                  uint32_t col, float v) {
    if (!g.epi.bias && !g.epi.mask) return v;
    return apply_epilogue(g.epi, (static_cast<uint64_t>(z) * g.m + row) * g.n + col, v);
}

// Output tile (tm, tn) and K partition of this workgroup.
//  - Unsplit grids (blockIdx.x = tile): the hardware deals workgroups to the
//    8 XCDs round-robin, so the tile index is remapped to give each XCD a
//    contiguous tile range, walked in groups of 8 tile-rows for L2 reuse.
//  - Split grids launched flat (flat_splits > 0, grid.x = tiles * partitions):
//    the workgroups one XCD receives (linear id % 8) take a contiguous range
//    of (partition, tile) pairs, so the tiles of one partition, which read the
//    same K slices of A and B, share that XCD's L2 instead of each fetching
//    them from memory.
//  - Otherwise blockIdx.y is the partition.
// Which workgroup computes what never changes what it computes: same bits.
__device__ __forceinline__ void tile_of(const GemmArgs& g, uint32_t& tm, uint32_t& tn,
                                        uint32_t& split) {
    const uint32_t ntiles = g.tiles_m * g.tiles_n;
    uint32_t bid = blockIdx.x;
    split = blockIdx.y;
    if (g.flat_splits) {
        const uint32_t total = ntiles * g.flat_splits;
        const uint32_t xcd = bid & 7u, slot = bid >> 3, q = total >> 3, r = total & 7u;
        const uint32_t v = xcd * q + min(xcd, r) + slot;
        split = v / ntiles;
        bid = v - split * ntiles;
    } else if ((ntiles & 7u) == 0) {
        bid = (bid & 7u) * (ntiles >> 3) + (bid >> 3);
    }
    const uint32_t group_span = 8u * g.tiles_n;
    const uint32_t first_m = (bid / group_span) * 8u;
    const uint32_t gsize = min(g.tiles_m - first_m, 8u);
    tm = first_m + (bid % group_span) % gsize;
    tn = (bid % group_span) / gsize;
}

// The B operand of a convolution read straight from the image (implicit
// im2col): element (row, pos) of image n's cols matrix [C*kh*kw, out_h*out_w]
// is x[n, c, h, w] with row = c*kh*kw + ki*kw + kj, pos = oh*out_w + ow,
// h = oh*stride_h - pad_h + ki*dil_h, w = ow*stride_w - pad_w + kj*dil_w, and
// 0 outside the image (kernels_movement.cpp:438-483, the im2col kernel's map).
struct Im2colB {
    const float* x;  // image 0
    int64_t sn;      // image (batch) stride in elements
    // Within one image every offset fits 32 bits (checked by make_im2col).
    int32_t sc, sh, sw;  // channel, row and column strides in elements
    int32_t H, W, kh, kw, kk, strh, strw, padh, padw, dilh, dilw, ow;
    FastDiv div_kk, div_kw, div_ow;  // by kh*kw, kw, out_w
    const int32_t* rows;             // row table (see below)
    uint32_t L, images;              // IMGTB: positions per image, images
    FastDiv div_L;                   // IMGTB: by L
};

// The map splits into a part that depends only on the output position (one
// per lane, fixed for the whole kernel) and a part that depends only on the
// cols row (the same for every lane of a wave in the loader below). Whether
// an element is inside the image depends on the position and on the row's
// window element r = ki*kw + kj only: each position keeps a bit mask over r
// of the elements that fall in the padding.
constexpr int kMaxWindow = 63;  // kh*kw; bit 63 marks rows past K

struct ImgPos {
    int32_t h0, w0;    // top-left image coordinate of the window
    int32_t base;      // its offset (may lie outside the image)
    uint64_t outside;  // bit r set: window element r lies in the padding
};

__host__ __device__ __forceinline__ ImgPos img_pos(const Im2colB& g, uint32_t pos, bool valid) {
    const uint32_t oh = g.div_ow.div(pos);
    const uint32_t ow = pos - oh * static_cast<uint32_t>(g.ow);
    ImgPos p;
    p.h0 = static_cast<int32_t>(oh) * g.strh - g.padh;
    p.w0 = static_cast<int32_t>(ow) * g.strw - g.padw;
    p.base = p.h0 * g.sh + p.w0 * g.sw;
    p.outside = ~0ull;
    if (valid) {
        for (int ki = 0; ki < g.kh; ++ki) {
            const bool row_in = static_cast<uint32_t>(p.h0 + ki * g.dilh) < static_cast<uint32_t>(g.H);
            for (int kj = 0; kj < g.kw; ++kj) {
                const bool in = row_in && static_cast<uint32_t>(p.w0 + kj * g.dilw) <
                                              static_cast<uint32_t>(g.W);
                if (in) p.outside &= ~(1ull << (ki * g.kw + kj));
            }
        }
    }
    return p;
}

// The row part of cols row `row` (channel c, window element ki, kj): its
// offset and its window element.
struct ImgRow {
    int32_t off, r;
};

__host__ __device__ __forceinline__ ImgRow img_row(const Im2colB& g, uint32_t row) {
    const uint32_t c = g.div_kk.div(row);
    const uint32_t r = row - c * static_cast<uint32_t>(g.kk);
    const uint32_t ki = g.div_kw.div(r);
    const uint32_t kj = r - ki * static_cast<uint32_t>(g.kw);
    ImgRow q;
    q.off = static_cast<int32_t>(c) * g.sc + static_cast<int32_t>(ki) * g.dilh * g.sh +
            static_cast<int32_t>(kj) * g.dilw * g.sw;
    q.r = static_cast<int32_t>(r);
    return q;
}

// The gather reads the row part from a table built once per geometry:
// groups of 16 rows as {4*off[16], r[16]} (byte offsets), padded past K with
// rows whose r = 63 is outside for every position, so the loader needs no K
// bound. The table is read through the constant address space: a wave's rows
// are uniform, so these are scalar loads.
constexpr int kRowGroup = 16;
typedef const int32_t __attribute__((address_space(4)))* RowTable;

}  // namespace vkhip
