// fp32 products on the bf16 matrix cores. An fp32 value x is exactly the sum
// of three bf16 terms, x = h + m + l: h the nearest bf16 to x, m the nearest to
// x - h, l = x - h - m (24 significant bits, at least 8 per term). The product
// of two such sums has nine term products; all but ll' are computed, each exact
// in fp32, and summed in fp32 by v_mfma_f32_32x32x16_bf16. |m| reaches 2^-8 of
// x and |l| 2^-17, so ll' is at most 2^-34 of the product, while ml' and lm'
// together reach 2^-24: without them a sum of one non-zero term (a diagonal
// matrix, a selection) was off by up to 1.2e-7 of it, twice fp32's rounding;
// with them by 5.97e-8. A K step of 16 takes eight MFMAs of 32 cycles against
// eight of 64 for v_mfma_f32_32x32x2_f32.
//
// The matrix core drops the bits of a product that lie too far below the
// accumulator it is added to, always downwards: added to the sum of the hh'
// products, the smaller ones left it too small by a mean of 0.06 to 0.2 of
// its (random) error, which shows where many outputs are summed again (2.3e-6
// of a bias gradient, 6e-7 on the fp32 cores). They have an accumulator of
// their own: the mean is below 0.02 of the error (a bias gradient 1.2e-7), and
// the sum of the hh' products is rounded once per 16 k.
//
// What the terms cannot hold is computed again in fp32. Inf and NaN inputs, and
// values that round up to inf as h, make every output they reach non-finite: a
// workgroup that ends with a non-finite accumulator runs its K range again on
// v_mfma_f32_32x32x2_f32 and keeps that. The terms of an input with 0 < |x| <
// 2^-110 may end at bf16's smallest value 2^-133 and so leave out up to 2^-134
// of it. All such inputs together change an output by at most K 2^-133 of the
// largest input, so a workgroup that has staged one reads its operands again for
// that and runs again only where an output is below K 2^-103 of it, 2^30 times
// as much. (4096^3 on one card: 0.87 ms; with such an input in every tile, a
// probability of 1e-34 among ordinary ones, 1.12, and 2.36 with a second pass
// for all of them; 0.93 on the fp32 matrix cores.)
//
// Error of N(0,1) products against 64 bits (relative, 2-norm), the fp32 matrix
// cores' in brackets: 1024^3 1.3e-7 (4.1e-7), 2048^3 2.7e-7 (8.1e-7), 4096^3
// 4.0e-7 (1.15e-6). Operands of one sign, uniform in 0..1: 0.9e-7 (2.2e-7),
// 2.2e-7 (6.0e-7), 3.0e-7 (8.4e-7), with a mean of -4e-9 of the sum at 4096^3
// (-4e-9) from the floors; relu(N) on both sides 3.2e-7 (4.9e-7) at 4096^3.
//
// Layout: a stage is 16 k of a tile's rows of both operands, three planes (h,
// m, l) of 32 bytes per row in LDS, double buffered; the loads run D stages
// ahead in registers, which are split into the planes beside the MFMAs of the
// stage before; one barrier per stage. Planes of a k-contiguous operand are
// rows of 16 k, an MFMA operand one 16-byte read; planes of a row-contiguous
// one lie as in memory, k rows of R values, and are read through the
// transposing 8-byte LDS reads (two per MFMA operand), so that no layout
// transposes in registers. Either way lane l supplies row l % 32 and k = 8 *
// (l / 32) + 0..7 of a 32-row block: every layout sums in the same order.
// KG > 1: the workgroup is KG groups, group i taking stages i, i + KG, ...,
// their accumulators added in LDS in order.
//
// What bounds it: power, then the splitting and the LDS reads per MFMA. A loop
// of nothing but these MFMAs reaches 1.45-1.7 PFLOP/s of bf16 on this card, 180
// to 210 TFLOP/s of fp32 products; the 256x128 tile runs 4096^3 at 170 (810 us;
// 930 on the fp32 cores). Counted there, the matrix cores are busy 69% of the
// cycles, at a clock of 1.73 GHz; at 2048^3 (128x128 tiles, one workgroup per
// CU, 120 us; 126) 50%, at 1024^3 22%: a stage of the 128x128 tile reads 72 KB
// and writes 24 KB of LDS for 1024 cycles of MFMAs, of the 64x64 tile half of
// that for a quarter of the MFMAs. The 128x128 tile's 128 registers, for two
// workgroups per CU, spill up to three values around the loop, none inside it;
// with both operands transposed fifteen, of which a stage reads one (2048^3 128
// us; 116 to 129 in the other layouts).
#pragma once

#include <algorithm>

#include "gemm_common.h"

namespace vkhip {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any float
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) char* Lds;
template <class V>
__device__ __forceinline__ __attribute__((address_space(3))) V& lds_at(Lds p) {
    return *reinterpret_cast<__attribute__((address_space(3))) V*>(p);
}

// How an operand's stage is read (rows are A's m or B's n):
//   TK   unit k stride: groups of four k, 16-byte loads at any float address.
//   TR   unit row stride: four rows of one k, 16-byte loads along the rows.
//   TG   any strides: 4-byte loads.
//   TKB  TK with the batch folded into K (conv weight gradient summed over
//        the batch: k = image * L + position, L a multiple of 32).
//   TI   B gathered from the image (IMG), TT its transpose (IMGT), TTB the
//        transpose with the batch folded into K (IMGTB).
enum TripleMode { TK = 0, TR, TG, TKB, TI, TT, TTB };
// Modes whose planes are k rows of R values (the others': rows of 16 k).
constexpr bool triple_k_rows(int mode) { return mode == TR || mode == TT || mode == TTB; }

constexpr uint32_t kTripleTiny = 0x11000000u - 1u;  // 2 * bits(2^-110) - 1

__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}
// The terms of x and y, packed as bf16 pairs; `tiny` keeps the least
// 2 * |bits| - 1 seen (a zero wraps to the largest value).
__device__ __forceinline__ void split_pair(float x, float y, uint32_t& h, uint32_t& m, uint32_t& l, uint32_t& tiny) {
    const uint32_t bx = (__builtin_bit_cast(uint32_t, x) << 1) - 1u, by = (__builtin_bit_cast(uint32_t, y) << 1) - 1u;
    tiny = min(tiny, min(bx, by));
    h = bf16_pair(x, y);
    x -= __builtin_bit_cast(float, h << 16);
    y -= __builtin_bit_cast(float, h & 0xffff0000u);
    m = bf16_pair(x, y);
    x -= __builtin_bit_cast(float, m << 16);
    y -= __builtin_bit_cast(float, m & 0xffff0000u);
    l = bf16_pair(x, y);
}

// Byte address of the 16-byte half g (k 8 g .. 8 g + 7) of row r in a plane of
// 16-k rows. The halves swap every eight rows, so that the 16 rows of an MFMA
// read's pass over the 64 banks fall on all of them.
__host__ __device__ __forceinline__ constexpr uint32_t triple_slot(uint32_t r, uint32_t g) {
    return r * 32u + ((g ^ ((r >> 3) & 1u)) << 4);
}
// Byte address of rows r .. r + 3 (r a multiple of four) of k in a plane of 16 k
// rows of R values. A transposing read's pass takes 32 rows (64 bytes) of four
// consecutive k: their 64-byte blocks are exchanged so that the four fall on
// distinct banks. Every other four k the 32-byte halves swap as well, for the
// image modes' writes (16 k of 16 rows at a time).
template <int R>
__host__ __device__ __forceinline__ constexpr uint32_t triple_slot_t(uint32_t r, uint32_t k) {
    return k * (2 * R) + ((2 * r) ^ (R == 64 ? ((k >> 1) & 1u) << 6 : (k & 3u) << 6) ^ (((k >> 2) & 1u) << 5));
}
constexpr uint32_t kTriplePitch32 = 20;  // floats per 16-k row in the fp32 pass

// One operand's stages: R rows x 16 k by T threads, NG groups of four each.
template <int MODE, int R, int T>
struct TripleOperand {
    static constexpr int NG = R * 16 / T / 4;
    static_assert(NG >= 1, "at least one group of four per thread");
    static constexpr uint32_t kBytes = 3 * R * 32, kBytes32 = R * kTriplePitch32 * 4;  // of a stage
    static constexpr bool KMAP = MODE == TK || MODE == TKB || MODE == TG;

    const char* base;  // this batch's operand
    int64_t s_k;
    uint32_t kdim;
    uint32_t voff[MODE == TK || MODE == TKB || MODE == TR ? NG : 1];
    int64_t goff[MODE == TG ? NG : 1];
    uint32_t slot;
    // TI: a lane has one position for all its groups, a wave's k are the same
    // for all its lanes. An element's byte offset is the sum of the position's
    // part (vector) and the k's part (scalar, from the row table), the first
    // counted from a point the padding's extent before the image so that it
    // is not negative; a padded element's has bit 31 set and reads as 0 (a
    // buffer of 2^31 bytes).
    uint32_t lane4;
    uint32_t out_lo, out_hi;  // bit r: window element r of the position is padding
    // TT: a lane has one position per stage and four window rows per group, so
    // that a load of 64 lanes covers 16 consecutive positions of four rows.
    static constexpr bool IMAGE_T = MODE == TT || MODE == TTB;
    int32_t off4[IMAGE_T ? 4 * NG : 1];     // a row's byte offset
    uint32_t disp[IMAGE_T ? 4 * NG : 1];    // and displacement: h, and w << 16

    // (row, k group of four) of group i, for the modes that hold such groups
    __device__ __forceinline__ static void row_kq(int t, int i, int& r, int& kq) {
        if (KMAP) {
            kq = t & 3;
            r = (t >> 2) + i * (T / 4);
        } else {
            r = t % R;
            kq = t / R + i * (T / R);
        }
    }
    // Modes with k rows: group i is one k of rows quad(i) .. + 3. TR: lanes
    // along the rows, TT: along k.
    static constexpr int KSTEP = 4 * T / R, QSTEP = T / 4;
    __device__ __forceinline__ static int quad_k(int t, int i) { return IMAGE_T ? t & 15 : t / (R / 4) + i * KSTEP; }
    __device__ __forceinline__ static int quad(int t, int i) { return IMAGE_T ? (t >> 4) * 4 + i * QSTEP : 4 * (t % (R / 4)); }

    // The operand's row that the tile's row x (counted from the operand's
    // start) holds, and whether the output has it. TR loads four rows at a
    // time: where the operand ends inside such a group, the group holds the
    // operand's last four rows.
    __device__ __forceinline__ static bool real_row(uint32_t x, uint32_t rows, uint32_t& real) {
        real = x;
        if constexpr (MODE == TR) {
            const uint32_t end = rows & ~3u;
            if (x < end) return true;
            real = rows - 4u + (x - end);
            return x < end + 4u && real >= end;
        }
        return x < rows;
    }

    __device__ __forceinline__ void init(const float* b, int64_t srow, int64_t sk, uint32_t row0, uint32_t rows,
                                         uint32_t k, const Im2colB& im, int t) {
        base = reinterpret_cast<const char*>(b);
        s_k = sk;
        kdim = k;
        if constexpr (MODE == TR) {
            const uint32_t rb = min(row0 + quad(t, 0), rows - 4u);
#pragma unroll
            for (int i = 0; i < NG; ++i) voff[i] = (static_cast<uint32_t>(quad_k(t, i) * sk) + rb) * 4u;
            slot = triple_slot_t<R>(quad(t, 0), quad_k(t, 0));
        } else if constexpr (IMAGE_T) {
            slot = triple_slot_t<R>(quad(t, 0), quad_k(t, 0));
#pragma unroll
            for (int i = 0; i < 4 * NG; ++i) {
                const uint32_t x = row0 + quad(t, i / 4) + i % 4;
                const ImgRow q = img_row(im, x < rows ? x : 0u);
                const uint32_t ki = im.div_kw.div(static_cast<uint32_t>(q.r));
                const uint32_t kj = static_cast<uint32_t>(q.r) - ki * static_cast<uint32_t>(im.kw);
                // a row past the operand gets a displacement outside every image
                disp[i] = (x < rows ? ki * im.dilh : 0x6000u) | (kj * im.dilw) << 16;
                off4[i] = q.off * 4;
            }
        } else {
            int r, kq;
            row_kq(t, 0, r, kq);
            slot = triple_slot(r, kq >> 1) + ((kq & 1) << 3);
            if constexpr (MODE == TK || MODE == TKB || MODE == TG) {
#pragma unroll
                for (int i = 0; i < NG; ++i) {
                    row_kq(t, i, r, kq);
                    const uint32_t gr = min(row0 + r, rows - 1u);  // rows past the operand: the last one again
                    if constexpr (MODE == TG)
                        goff[i] = (static_cast<int64_t>(gr) * srow + 4 * kq * sk) * 4;
                    else
                        voff[i] = static_cast<uint32_t>((static_cast<int64_t>(gr) * srow + 4 * kq) * 4);
                }
            } else {
                const uint32_t before = static_cast<uint32_t>(im.padh * im.sh + im.padw * im.sw) * 4u;
                base -= before;
                const uint32_t x = row0 + r;
                const ImgPos at = img_pos(im, x < rows ? x : 0u, x < rows);
                lane4 = static_cast<uint32_t>(at.base * 4) + before;
                out_lo = static_cast<uint32_t>(at.outside);
                out_hi = static_cast<uint32_t>(at.outside >> 32);
            }
        }
    }

    // Reads this thread's elements of stage kt (k from 16 kt). TAIL: the stage
    // that K ends in; without it the stage is wholly inside K.
    template <bool TAIL>
    __device__ __forceinline__ void fetch(f32x4 (&v)[NG], uint32_t kt, const Im2colB& im, int t) const {
        const uint32_t k0 = kt * 16u;
        if constexpr (MODE == TK) {
            const char* p = base + static_cast<int64_t>(k0) * 4;
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                if constexpr (!TAIL) {
                    v[i] = *reinterpret_cast<const f32x4u*>(p + voff[i]);
                } else {
                    const uint32_t k = k0 + 4u * (t & 3);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        v[i][j] = k + j < kdim ? *reinterpret_cast<const float*>(p + voff[i] + 4 * j) : 0.0f;
                }
            }
        } else if constexpr (MODE == TKB) {
            const uint32_t n = im.div_L.div(k0);
            const char* p = base + (static_cast<int64_t>(n) * s_k + (k0 - n * im.L)) * 4;  // s_k: image stride
#pragma unroll
            for (int i = 0; i < NG; ++i) v[i] = *reinterpret_cast<const f32x4u*>(p + voff[i]);
        } else if constexpr (MODE == TR) {
            const char* p = base + static_cast<int64_t>(k0) * s_k * 4;
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                if (!TAIL || k0 + quad_k(t, i) < kdim)
                    v[i] = *reinterpret_cast<const f32x4u*>(p + voff[i]);
                else
                    v[i] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
            }
        } else if constexpr (MODE == TG) {
            const uint32_t k = k0 + 4u * (t & 3);
            const char* p = base + static_cast<int64_t>(k0) * s_k * 4;
#pragma unroll
            for (int i = 0; i < NG; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    v[i][j] = !TAIL || k + j < kdim ? *reinterpret_cast<const float*>(p + goff[i] + j * s_k * 4) : 0.0f;
        } else if constexpr (MODE == TI) {
            const __amdgpu_buffer_rsrc_t img = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<char*>(base), 0, static_cast<int32_t>(0x80000000u), 0x00020000);
            const uint32_t kq = __builtin_amdgcn_readfirstlane(t / R);
            const RowTable tab = (RowTable)im.rows + kt * (2 * kRowGroup);
#pragma unroll
            for (int i = 0; i < NG; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t e = 4u * (kq + i * (T / R)) + j;
                    const int32_t r = tab[kRowGroup + e];
                    const uint32_t pad = ((r & 32) ? out_hi : out_lo) << (31 - (r & 31));
                    v[i][j] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(
                                   img, static_cast<int32_t>((pad & 0x80000000u) | lane4), tab[e], 0));
                }
        } else {
            uint32_t p = k0 + quad_k(t, 0), positions = kdim;
            const char* image = base;
            if constexpr (MODE == TTB) {
                const uint32_t n = im.div_L.div(k0);
                image += static_cast<int64_t>(n) * im.sn * 4;
                p -= n * im.L;
                positions = im.L;
            }
            const __amdgpu_buffer_rsrc_t img = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<char*>(image), 0, static_cast<int32_t>(0x80000000u), 0x00020000);
            const uint32_t oh = im.div_ow.div(p), ow = p - oh * static_cast<uint32_t>(im.ow);
            const int32_t h0 = static_cast<int32_t>(oh) * im.strh - im.padh;
            const int32_t w0 = static_cast<int32_t>(ow) * im.strw - im.padw;
            const int32_t at4 = (h0 * im.sh + w0 * im.sw) * 4;
            // both coordinates in 16 bits (triple_image_fits): inside when the
            // lesser of (h, w) and (H - 1, W - 1), unsigned, is (h, w); a
            // position past K lies outside every image
            typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
            const u16x2 origin = {static_cast<uint16_t>(p < positions ? h0 : 0x6000), static_cast<uint16_t>(w0)};
            const u16x2 last = {static_cast<uint16_t>(im.H - 1), static_cast<uint16_t>(im.W - 1)};
#pragma unroll
            for (int i = 0; i < 4 * NG; ++i) {
                const u16x2 hw = origin + __builtin_bit_cast(u16x2, disp[i]);
                const bool inside = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(hw, last)) ==
                                    __builtin_bit_cast(uint32_t, hw);
                const uint32_t at = inside ? static_cast<uint32_t>(at4 + off4[i]) : 0x80000000u;
                v[i / 4][i % 4] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(img, static_cast<int32_t>(at), 0, 0));
            }
        }
    }

    // Writes the elements to the stage's planes.
    __device__ __forceinline__ void put(Lds lds, const f32x4 (&v)[NG], uint32_t& tiny) const {
        constexpr uint32_t P = R * 32;
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            // group i: KSTEP k or QSTEP rows further on, T / 4 rows further on,
            // or another k group
            const Lds p = MODE == TR   ? lds + slot + i * (KSTEP * 2 * R)
                          : IMAGE_T    ? lds + (slot ^ (i * (QSTEP * 2)))
                          : KMAP       ? lds + slot + i * (T / 4 * 32)
                                       : lds + (slot ^ (i * (8 * T / R)));
            static_assert(MODE != TR || NG == 1 || KSTEP % 8 == 0, "the exchanges repeat every eight k");
            static_assert(!KMAP || (T / 4) % 16 == 0, "the exchange of halves repeats every 16 rows");
            uint32_t h0, m0, l0, h1, m1, l1;
            split_pair(v[i][0], v[i][1], h0, m0, l0, tiny);
            split_pair(v[i][2], v[i][3], h1, m1, l1, tiny);
            lds_at<u32x2>(p) = (u32x2){h0, h1};
            lds_at<u32x2>(p + P) = (u32x2){m0, m1};
            lds_at<u32x2>(p + 2 * P) = (u32x2){l0, l1};
        }
    }

    // The same as fp32 rows of 16 k (the fp32 pass).
    __device__ __forceinline__ void put32(Lds lds, const f32x4 (&v)[NG], int t) const {
        int r = quad(t, 0), kq = 0;
        if constexpr (!triple_k_rows(MODE)) row_kq(t, 0, r, kq);
        const uint32_t slot32 = r * (kTriplePitch32 * 4) + (triple_k_rows(MODE) ? quad_k(t, 0) * 4u : 16u * kq);
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            if constexpr (triple_k_rows(MODE)) {
                const uint32_t step = IMAGE_T ? QSTEP * (kTriplePitch32 * 4) : KSTEP * 4;
#pragma unroll
                for (int j = 0; j < 4; ++j) lds_at<float>(lds + slot32 + i * step + j * (kTriplePitch32 * 4)) = v[i][j];
            } else {
                const uint32_t at = slot32 + (KMAP ? i * (T / 4) * (kTriplePitch32 * 4) : i * (T / R) * 16u);
                lds_at<f32x4>(lds + at) = v[i];
            }
        }
    }
};

// A lane's reads of one operand's MFMA blocks (N of 32 rows from row w0) in a
// plane of R rows.
template <int MODE, int R, int N>
struct TripleReads {
    static constexpr bool K_ROWS = triple_k_rows(MODE);
    uint32_t at[K_ROWS ? N : 1];
    __device__ __forceinline__ void init(uint32_t stage_at, uint32_t w0, int lane) {
        if constexpr (K_ROWS) {
            // lane s of 16 reads k s / 4, rows 4 (s % 4) .. + 3; it receives
            // row s of k 0..3
            const uint32_t k = 8u * (lane >> 5) + ((lane >> 2) & 3), r = w0 + 16u * ((lane >> 4) & 1) + 4u * (lane & 3);
#pragma unroll
            for (int i = 0; i < N; ++i) at[i] = stage_at + triple_slot_t<R>(r + 32 * i, k);
        } else {
            at[0] = stage_at + triple_slot(w0 + (lane & 31), lane >> 5);
        }
    }
    __device__ __forceinline__ bf16x8 read(Lds stage, int plane, int i) const {
        if constexpr (K_ROWS) {
            typedef __attribute__((address_space(3))) s16x4* Quad;
            const uint32_t p = at[K_ROWS ? i : 0] + plane * (R * 32);
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<Quad>(stage + p));
            // four k further on: the next four k rows, 32-byte halves swapped
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                reinterpret_cast<Quad>(stage + ((at[K_ROWS ? i : 0] ^ 32u) + plane * (R * 32) + 4 * 2 * R)));
            return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        } else {
            return lds_at<bf16x8>(stage + at[0] + plane * (R * 32) + i * 1024);
        }
    }
};

// What a thread stages: groups of both operands.
template <class OA, class OB, int D>
struct TripleStager {
    OA a;
    OB b;
    int t;
    f32x4 va[D][OA::NG], vb[D][OB::NG];
    template <bool TAIL>
    __device__ __forceinline__ void fetch(int d, uint32_t kt, const Im2colB& im) {
        a.template fetch<TAIL>(va[d], kt, im, t);
        b.template fetch<TAIL>(vb[d], kt, im, t);
    }
    __device__ __forceinline__ void put(Lds stage, int d, uint32_t& tiny) const {
        a.put(stage, va[d], tiny);
        b.put(stage + OA::kBytes, vb[d], tiny);
    }
    __device__ __forceinline__ uint32_t largest(int d) const {
        uint32_t most = 0;
#pragma unroll
        for (int i = 0; i < OA::NG; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) most = max(most, __builtin_bit_cast(uint32_t, va[d][i][j]) & 0x7fffffffu);
#pragma unroll
        for (int i = 0; i < OB::NG; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) most = max(most, __builtin_bit_cast(uint32_t, vb[d][i][j]) & 0x7fffffffu);
        return most;
    }
    __device__ __forceinline__ void put32(Lds stage, int d) const {
        a.put32(stage, va[d], t);
        b.put32(stage + OA::kBytes32, vb[d], t);
    }
};

// A wave's share of the multiplication: MI x NI blocks of 32 x 32.
template <int BM, int BN, int MI, int NI, int KG, int D, int AM, int BMODE>
struct TripleTile {
    static constexpr int PA = BM * 32, PB = BN * 32;  // plane bytes
    static constexpr int STAGE = 3 * (PA + PB);

    f32x16 acc[MI][NI], cor[MI][NI];  // the hh' products; the smaller ones
    TripleReads<AM, BM, MI> ra;
    TripleReads<BMODE, BN, NI> rb;
    uint32_t kt0, full;   // this partition's first stage, and the end of its whole stages
    int kg, ns, mine;     // whole stages of the longest group, and of this one
    bool tail;            // K ends inside the partition's last stage

    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = cor[i][j][r] = 0.0f;
    }
    __device__ __forceinline__ void gather() {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] += cor[i][j][r];
    }
    // The whole stage that is this group's s-th, or the last whole one.
    __device__ __forceinline__ uint32_t stage_of(int s) const { return min(kt0 + kg + s * KG, full - 1u); }

    // One stage's products; `next` (staging of the next stage) is called where
    // it can run beside them.
    template <class F>
    __device__ __forceinline__ void multiply(Lds cur, F&& next) {
        // smallest products first: ml' lm' hl' lh' mm' hm' mh' hh'
        constexpr int TA[8] = {1, 2, 0, 2, 1, 0, 1, 0}, TB[8] = {2, 1, 2, 0, 1, 1, 0, 0};
        bf16x8 fa[3][MI], fb[3][NI];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int j = 0; j < NI; ++j) fb[p][j] = rb.read(cur, p, j);
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < MI; ++i) fa[p][i] = ra.read(cur, p, i);
        next();
#pragma unroll
        for (int q = 0; q < 8; ++q)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    f32x16& c = q < 7 ? cor[i][j] : acc[i][j];
                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[TA[q]][i], fb[TB[q]][j], c, 0, 0, 0);
                }
    }

    template <class S>
    __device__ __forceinline__ void run(S& st, Lds lds, const Im2colB& im, uint32_t& tiny) {
#pragma unroll
        for (int d = 0; d < D; ++d) st.template fetch<false>(d, stage_of(d), im);
        st.put(lds, 0, tiny);
        st.template fetch<false>(0, stage_of(D), im);
        __syncthreads();
        // D register sets are addressed by unrolling; one set needs none
        for (int s0 = 0; s0 < ns; s0 += D) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                const int s = s0 + u;
                if (s >= ns) break;
                const int buf = (D % 2 ? s : u) & 1;
                if (KG == 1 || s < mine)
                    multiply(lds + buf * STAGE, [&] {
                        st.put(lds + (buf ^ 1) * STAGE, (u + 1) % D, tiny);
                        st.template fetch<false>((u + 1) % D, stage_of(s + 1 + D), im);
                    });
                __syncthreads();
            }
        }
        if (tail) {  // group 0's
            if (kg == 0) {
                st.template fetch<true>(0, full, im);
                st.put(lds, 0, tiny);
            }
            __syncthreads();
            if (kg == 0) multiply(lds, [] {});
        }
    }

    // The bits of the largest magnitude this thread's loads have had.
    template <class S>
    __device__ __forceinline__ uint32_t largest(S& st, const Im2colB& im) {
        uint32_t most = 0;
#pragma unroll 1
        for (int s = 0; s < ns + (tail ? 1 : 0); ++s) {
            if (s == ns)
                st.template fetch<true>(0, full, im);
            else
                st.template fetch<false>(0, stage_of(s), im);
            most = max(most, st.largest(0));
        }
        return most;
    }

    // The same stages and order of groups in fp32.
    template <class S>
    __device__ __forceinline__ void run32(S& st, Lds lds, const Im2colB& im, int wm0, int wn0, int lane) {
        zero();
#pragma unroll 1
        for (int s = 0; s < ns + (tail ? 1 : 0); ++s) {
            __syncthreads();
            if (s == ns)
                st.template fetch<true>(0, full, im);
            else
                st.template fetch<false>(0, stage_of(s), im);
            st.put32(lds, 0);
            __syncthreads();
            if (KG > 1 && (s == ns ? kg != 0 : s >= mine)) continue;
            const Lds as = lds + ((wm0 + (lane & 31)) * kTriplePitch32 + (lane >> 5)) * 4;
            const Lds bs = lds + ((BM + wn0 + (lane & 31)) * kTriplePitch32 + (lane >> 5)) * 4;
#pragma unroll 1
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NI; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                            lds_at<float>(as + (32 * i * kTriplePitch32 + 2 * q) * 4),
                            lds_at<float>(bs + (32 * j * kTriplePitch32 + 2 * q) * 4), acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
};

template <int BM, int BN, int WM, int WN, int KG, int D, int OCC, int AM, int BMODE>
__global__ __launch_bounds__(BM / WM * (BN / WN) * 64 * KG, OCC) void gemm_triple_kernel(GemmArgs g, Im2colB im) {
    constexpr int T = BM / WM * (BN / WN) * 64, MI = WM / 32, NI = WN / 32;
    using Tile = TripleTile<BM, BN, MI, NI, KG, D, AM, BMODE>;
    constexpr int STAGE = Tile::STAGE, FOLD = (KG - 1) * BM * BN * 4;
    constexpr int LDS = 2 * STAGE * KG > FOLD ? 2 * STAGE * KG : FOLD;
    using OA = TripleOperand<AM, BM, T>;
    using OB = TripleOperand<BMODE, BN, T>;
    __shared__ __attribute__((aligned(16))) char lds_all[LDS];

    const int lane = threadIdx.x & 63;
    const int gwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = KG > 1 ? gwave / (T / 64) : 0;
    const int wave = gwave - kg * (T / 64);
    const Lds lds = (Lds)lds_all + kg * (2 * STAGE);
    const int wm0 = (wave / (BN / WN)) * WM, wn0 = (wave % (BN / WN)) * WN;
    const int lrow = lane & 31, kh = lane >> 5;

    uint32_t tm, tn, split;
    tile_of(g, tm, tn, split);
    const uint32_t row0 = tm * BM, col0 = tn * BN;
    const uint32_t z = blockIdx.z, i0 = z / g.b1, i1 = z % g.b1;

    Tile tile;
    tile.kg = kg;
    tile.kt0 = split * 2u * g.chunk;
    const uint32_t kt1 = min((g.k + 15u) / 16u, tile.kt0 + 2u * g.chunk);
    tile.full = min(kt1, g.k / 16u);
    tile.tail = kt1 > tile.full;
    // (a partition of a tail alone has no whole stage: its prefetches read the
    // stage before it)
    const int whole = static_cast<int>(tile.full - tile.kt0);
    tile.ns = (whole + KG - 1) / KG;
    tile.mine = (whole - kg + KG - 1) / KG;
    tile.ra.init(0, wm0, lane);
    tile.rb.init(3 * Tile::PA, wn0, lane);
    tile.zero();

    TripleStager<OA, OB, D> st;
    st.t = wave * 64 + lane;
    st.a.init(g.a + i0 * g.sa0 + i1 * g.sa1, g.sam, AM == TKB ? g.sa1 : g.sak, row0, g.m, g.k, im, st.t);
    st.b.init(BMODE >= TI ? im.x + (BMODE == TTB ? 0 : static_cast<int64_t>(z) * im.sn)
                          : g.b + i0 * g.sb0 + i1 * g.sb1,
              g.sbn, g.sbk, col0, g.n, g.k, im, st.t);
    uint32_t tiny = ~0u;
    tile.run(st, lds, im, tiny);

    tile.gather();
    auto& acc = tile.acc;
    // (rows past an operand's end hold whatever the LDS held)
    auto inside = [&](int i, int j, int r) {
        uint32_t row, col;
        return OA::real_row(row0 + wm0 + 32 * i + 8 * (r / 4) + 4 * kh + (r % 4), g.m, row) &&
               OB::real_row(col0 + wn0 + 32 * j + lrow, g.n, col);
    };
    float finite = 0.0f;  // becomes NaN with any non-finite accumulator of the output
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) finite = __builtin_fmaf(inside(i, j, r) ? acc[i][j][r] : 0.0f, 0.0f, finite);
    if (__syncthreads_or(!(finite == 0.0f) || tiny < kTripleTiny)) {
        uint32_t* most = reinterpret_cast<uint32_t*>(lds_all);
        if (threadIdx.x == 0) *most = 0u;
        __syncthreads();
        atomicMax(most, tile.largest(st, im));
        __syncthreads();
        const float bound = static_cast<float>(g.k) * 0x1p-103f * __builtin_bit_cast(float, *most);
        bool far = finite == 0.0f;  // every output far above what the tiny inputs lose
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) far = far && (!inside(i, j, r) || __builtin_fabsf(acc[i][j][r]) >= bound);
        if (__syncthreads_or(!far)) tile.run32(st, lds, im, wm0, wn0, lane);
    }
    if constexpr (KG > 1) {
        float* part = reinterpret_cast<float*>(lds_all);
        __syncthreads();
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        part[(((kg - 1) * MI + i) * NI + j) * (16 * T) + r * T + wave * 64 + lane] = acc[i][j][r];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int q = 1; q < KG; ++q)
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int j = 0; j < NI; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        acc[i][j][r] += part[(((q - 1) * MI + i) * NI + j) * (16 * T) + r * T + wave * 64 + lane];
    }

    // register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32
    float* cbase = g.c + static_cast<uint64_t>(split) * g.split_stride + static_cast<uint64_t>(z) * g.m * g.n;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            uint32_t col;
            const bool col_in = OB::real_row(col0 + wn0 + 32 * j + lrow, g.n, col);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                uint32_t row;
                if (OA::real_row(row0 + wm0 + 32 * i + 8 * (r / 4) + 4 * kh + (r % 4), g.m, row) && col_in) {
                    float* at = cbase + static_cast<uint64_t>(row) * g.n + col;
                    // outputs of large tiles and convolutions, and split-K
                    // partials, are read by later kernels only
                    if constexpr (BM >= 128 || BMODE >= TI)
                        __builtin_nontemporal_store(acc[i][j][r], at);
                    else
                        *at = acc[i][j][r];
                }
            }
        }
}

// Whether the transposed image gather's 16-bit coordinates hold the geometry.
inline bool triple_image_fits(const Im2colB& im, int64_t out_h) {
    const int64_t h = std::max<int64_t>(im.H, (out_h - 1) * im.strh) + im.padh + static_cast<int64_t>(im.dilh) * im.kh;
    const int64_t w = std::max<int64_t>(im.W, (im.ow - 1) * static_cast<int64_t>(im.strw)) + im.padw +
                      static_cast<int64_t>(im.dilw) * im.kw;
    return h < 8192 && w < 8192;
}

// One tile size's launches (gemm_triple_*.hip). The gathers of the transposed
// image hold four window rows per thread: OCC_T waves per SIMD instead of OCC.
template <int BM, int BN, int WM, int WN, int KG, int D, int OCC, int OCC_T>
int launch_triple(const GemmArgs& g, const Im2colB& im, dim3 grid, int am, int bm) {
    constexpr int threads = BM / WM * (BN / WN) * 64 * KG;
#define VKHIP_TRIPLE(A, B)                                                                                   \
    if (am == A && bm == B) {                                                                                \
        hipLaunchKernelGGL((gemm_triple_kernel<BM, BN, WM, WN, KG, D, (B >= TT ? OCC_T : OCC), A, B>), \
                           grid, dim3(threads), 0, ctx().stream, g, im);                                     \
        VKHIP_LAUNCH_CHECK();                                                                                \
        return VKHIP_OK;                                                                                     \
    }
    VKHIP_TRIPLE(TK, TR)
    VKHIP_TRIPLE(TK, TK)
    VKHIP_TRIPLE(TR, TR)
    VKHIP_TRIPLE(TR, TK)
    VKHIP_TRIPLE(TG, TG)
    VKHIP_TRIPLE(TK, TI)
    VKHIP_TRIPLE(TK, TT)
    VKHIP_TRIPLE(TKB, TTB)
#undef VKHIP_TRIPLE
    return fail(VKHIP_ERR_INVALID, "gemm_triple: no kernel for operand modes %d, %d", am, bm);
}

int launch_triple_64x64(const GemmArgs& g, const Im2colB& im, dim3 grid, int am, int bm);
int launch_triple_128x128(const GemmArgs& g, const Im2colB& im, dim3 grid, int am, int bm);
int launch_triple_256x128(const GemmArgs& g, const Im2colB& im, dim3 grid, int am, int bm);

}  // namespace vkhip
