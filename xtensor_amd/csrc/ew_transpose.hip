// ew_transpose.hip — copies between two layouts whose contiguous dimensions
// differ (a materialised transpose) on gfx950.
//
// One work unit per chunk of an output row reads such a leaf element by
// element, each from a cache line of its own; past the caches every line
// travels several times.  Here a workgroup copies a 64 x 64 tile through LDS:
// 16-byte loads along the leaf's contiguous dimension, 16-byte stores along
// the output's, each line touched by one workgroup (two at the tile's edge).
//   bound: memory.  NCHW -> NHWC of [32, 128, 56, 56], repeated on the same
//   arrays (in the 256 MB cache): float32 37.5 us a call with one unit per
//   output chunk, 15.6 here (6.6 TB/s); bfloat16 30.5 -> 9.7, float64 129 ->
//   29.7; a [3000, 4000] float32 matrix 67.3 -> 15.6.  Over arrays past the
//   cache the float32 images take 36.6 -> 20.1 (5.1 TB/s, a copy's rate).
//   Plain accesses: non-temporal ones leave float32 as it is and cost float64
//   30 -> 38 us (a tile's rows end inside lines that its neighbour completes).
//   tile: 64 elements are 128 to 512 bytes either way; 17 KB of LDS (33 for
//   8-byte types) leave 8 (4) workgroups of 4 waves a CU, each with its
//   16 to 128 bytes a lane in flight.
//   LDS: one cell of 4 (8) bytes an element, rows 65 cells apart, written along
//   one dimension and read along the other: lanes l of a row and rows r hit
//   cell 65 r + V l (writing) and 65 V l + r (reading), distinct banks both.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ew.hpp"
#include "ew_kernels.hpp"
#include "interp.hpp"

namespace xg {

namespace {

constexpr uint32_t kTile = 64;

struct TransposePlan {
    const char* in;
    char* out;
    uint32_t ni, nt;            // extents: along the output's rows, along the leaf's
    uint32_t in_i, out_t;       // element strides of the leaf along i, of the output along t
    uint32_t in_o[2], out_o[2]; // the other dimensions
    FastDiv tiles_i, tiles_t, n1;
};

// bits of one element as the element-wise program stores them
template <class T, bool BF16> __device__ __forceinline__ T passed(T x) {
    if constexpr (BF16) return (x & 0x7fff) > 0x7f80 ? T(x | 0x40) : x;  // NaN kept quiet
    return x;
}

template <class T, bool BF16>
__global__ __launch_bounds__(256) void transpose_kernel(const TransposePlan p) {
    constexpr uint32_t E = sizeof(T), V = 16 / E;
    constexpr uint32_t LPR = kTile / V;       // lanes a row
    constexpr uint32_t ROWS = 256 / LPR;      // rows a pass
    constexpr uint32_t PASSES = kTile / ROWS;
    using Cell = std::conditional_t<E == 8, uint64_t, uint32_t>;
    __shared__ Cell tile[kTile * (kTile + 1)];
    union Vec {
        u32x4_t q;
        T e[V];
    };

    uint32_t b = xcd_block(1);
    uint32_t q = fastdiv(b, p.tiles_i);
    const uint32_t i0 = (b - q * p.tiles_i.d) * kTile;
    b = q;
    q = fastdiv(b, p.tiles_t);
    const uint32_t t0 = (b - q * p.tiles_t.d) * kTile;
    b = q;
    q = fastdiv(b, p.n1);
    const uint32_t o1 = b - q * p.n1.d;
    const char* in = p.in + (uint64_t(q) * p.in_o[0] + uint64_t(o1) * p.in_o[1] + uint64_t(i0) * p.in_i + t0) * E;
    char* out = p.out + (uint64_t(q) * p.out_o[0] + uint64_t(o1) * p.out_o[1] + uint64_t(t0) * p.out_t + i0) * E;
    const uint32_t ni = min(kTile, p.ni - i0), nt = min(kTile, p.nt - t0);  // this tile's part
    const uint32_t row = threadIdx.x / LPR, col = (threadIdx.x % LPR) * V;

    Vec v[PASSES];
    if (ni == kTile && nt == kTile) {
#pragma unroll
        for (uint32_t k = 0; k < PASSES; ++k)
            v[k].q = ld16<false>(in + (uint64_t(row + k * ROWS) * p.in_i + col) * E);
    } else {
#pragma unroll
        for (uint32_t k = 0; k < PASSES; ++k) {
            const uint32_t r = row + k * ROWS;
            const char* src = in + (uint64_t(r) * p.in_i + col) * E;
            if (r < ni && col + V <= nt) {
                v[k].q = ld16<false>(src);
            } else {
#pragma unroll
                for (uint32_t j = 0; j < V; ++j)
                    v[k].e[j] = (r < ni && col + j < nt) ? reinterpret_cast<const T*>(src)[j] : T(0);
            }
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < PASSES; ++k)
#pragma unroll
        for (uint32_t j = 0; j < V; ++j) tile[(row + k * ROWS) * (kTile + 1) + col + j] = Cell(v[k].e[j]);
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < PASSES; ++k) {
        const uint32_t r = row + k * ROWS;  // a position along t
#pragma unroll
        for (uint32_t j = 0; j < V; ++j) v[k].e[j] = passed<T, BF16>(T(tile[(col + j) * (kTile + 1) + r]));
    }
#pragma unroll
    for (uint32_t k = 0; k < PASSES; ++k) {
        const uint32_t r = row + k * ROWS;
        char* dst = out + (uint64_t(r) * p.out_t + col) * E;
        if (r < nt && col + V <= ni) {
            st16<false>(dst, v[k].q);
        } else {
#pragma unroll
            for (uint32_t j = 0; j < V; ++j)
                if (r < nt && col + j < ni) reinterpret_cast<T*>(dst)[j] = v[k].e[j];
        }
    }
}

template <class T, bool BF16>
void launch_tiles(const TransposePlan& t, uint32_t blocks, hipStream_t stream) {
    hipLaunchKernelGGL((transpose_kernel<T, BF16>), dim3(blocks), dim3(256), 0, stream, t);
}

}  // namespace

bool ew_is_transpose(const EwPlan& p) {
    const LeafView& in = p.leaves[0];
    const Program& g = p.prog;
    if (!p.compact || p.units == 0 || p.rank < 2 || p.rank > 4) return false;
    if (g.nleaves != 1 || g.leaf_gather[0] || g.nops != 1 || g.ops[0].op != MO_LOAD) return false;
    // the stored bits are the loaded ones
    if (in.dtype != p.out_dtype) return false;
    if (g.result_dtype != (in.dtype == XG_BFLOAT16 ? int(XG_FLOAT32) : in.dtype)) return false;
    const int esz = dtype_size(in.dtype);
    if (esz < 2) return false;
    if (lm_base(p.out_mode) != LM_CONTIG || (p.out_mode & LM_FILL) || lm_base(in.mode) != LM_STRIDED) return false;
    if (reinterpret_cast<uintptr_t>(in.ptr) % uintptr_t(esz) || reinterpret_cast<uintptr_t>(p.out_ptr) % uintptr_t(esz))
        return false;
    const int ki = p.rank - 1;
    int kt = -1;
    for (int k = 0; k < ki; ++k) {
        if (in.stride[k] < 0) return false;
        if (in.stride[k] == 1) kt = k;
    }
    if (kt < 0 || in.stride[ki] < p.shape[kt]) return false;  // rows of the leaf apart
    // A tile takes the same 1.8 ns of the chip (8-byte types 2.8) however full it
    // is, and at 4/15 full that is what its bytes take at a copy's rate.  Measured
    // against one unit per output chunk: 16 channels of 2500 pixels (0.24 full)
    // float32 18.3 us there, 20.2 by tiles; 18 channels (0.27) 23.2 and 20.4,
    // bfloat16 23.6 and 19.9, float64 43.5 and 34.4; 20 x 20 matrices (0.10) 8.2
    // and 16.7.
    const uint64_t ni = uint64_t(p.shape[ki]), nt = uint64_t(p.shape[kt]);
    const uint64_t area = (ni + kTile - 1) / kTile * ((nt + kTile - 1) / kTile) * kTile * kTile;
    return ni * nt * 15 >= area * 4;
}

hipError_t launch_ew_transpose(const EwPlan& p, hipStream_t stream) {
    const LeafView& in = p.leaves[0];
    const int ki = p.rank - 1;
    int kt = 0;
    while (in.stride[kt] != 1) ++kt;
    TransposePlan t{};
    t.in = in.ptr;
    t.out = p.out_ptr;
    t.ni = uint32_t(p.shape[ki]);
    t.nt = uint32_t(p.shape[kt]);
    t.in_i = uint32_t(in.stride[ki]);
    t.out_t = uint32_t(p.out_stride[kt]);
    uint32_t n[2] = {1, 1};
    int o = 1;
    for (int k = ki - 1; k >= 0; --k) {
        if (k == kt) continue;
        n[o] = uint32_t(p.shape[k]);
        t.in_o[o] = uint32_t(in.stride[k]);
        t.out_o[o] = uint32_t(p.out_stride[k]);
        --o;
    }
    const uint32_t ti = (t.ni + kTile - 1) / kTile, tt = (t.nt + kTile - 1) / kTile;
    const uint64_t blocks = uint64_t(ti) * tt * n[0] * n[1];
    t.tiles_i = make_fastdiv(ti);
    t.tiles_t = make_fastdiv(tt);
    t.n1 = make_fastdiv(n[1]);
    switch (dtype_size(in.dtype)) {
        case 2:
            if (in.dtype == XG_BFLOAT16) launch_tiles<uint16_t, true>(t, uint32_t(blocks), stream);
            else launch_tiles<uint16_t, false>(t, uint32_t(blocks), stream);
            break;
        case 4: launch_tiles<uint32_t, false>(t, uint32_t(blocks), stream); break;
        default: launch_tiles<uint64_t, false>(t, uint32_t(blocks), stream); break;
    }
    return hipGetLastError();
}

}  // namespace xg
