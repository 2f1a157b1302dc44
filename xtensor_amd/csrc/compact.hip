// compact.hip — xg_argwhere: the multi-indices of the nonzero elements of an
// expression, listed on the device (stream compaction).
//
// xt::argwhere<L> (core/xoperation.hpp:893-930) walks the expression in
// traversal order L and pushes the index of every element that converts to
// true.  Here: flags = (bool)e, a byte each, evaluated in that order; every
// workgroup counts the flags of 4096 positions; one workgroup turns the counts
// into offsets; and every workgroup lists its positions in LDS and writes
// their multi-indices from its offset on, consecutive lanes consecutive rows.
// Bytes bound it: the flags are written once and read twice (3 bytes a
// position) beside the condition's operands and the rows.  As int64 flags,
// scanned in place, with a thread per position writing its own row, they took
// 32 bytes a position: on a float32 [2048, 3000] with 30 % true the flags, scan
// and list kernels 62 us, 24 us now.
// For column-major traversal the expression is read through its reversed axes,
// so that its row-major order is the column-major order of the original.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "ew.hpp"
#include "planner.hpp"
#include "xg_api_internal.hpp"

namespace xg {

namespace {

constexpr uint32_t kPerBlock = 4096;  // positions of a workgroup: 16 a thread

// Layout of the two-step form's buffer: offsets int64[blocks + 1] (the last one
// the total), counts uint32[blocks], flags uint8[n].
struct ArgBuf {
    uint64_t blocks;
    size_t counts_at, flags_at, bytes;
    explicit ArgBuf(int64_t n) {
        blocks = (uint64_t(n) + kPerBlock - 1) / kPerBlock;
        counts_at = (blocks + 1) * 8;
        flags_at = (counts_at + blocks * 4 + 255) & ~size_t(255);
        bytes = flags_at + ((size_t(n) + 255) & ~size_t(255));  // whole vectors past the last flag stay inside
    }
};

// the 16 flags (0 or 1 each) of the calling thread as a bit mask
__device__ __forceinline__ uint32_t flag_bits(const uint8_t* flags, uint64_t n) {
    const uint64_t i = uint64_t(blockIdx.x) * kPerBlock + threadIdx.x * 16u;
    if (i >= n) return 0;
    const uint4 w = *reinterpret_cast<const uint4*>(flags + i);
    auto nib = [](uint32_t x) { return ((x & 0x01010101u) * 0x01020408u) >> 24 & 0xfu; };
    uint32_t m = nib(w.x) | nib(w.y) << 4 | nib(w.z) << 8 | nib(w.w) << 12;
    if (n - i < 16) m &= (1u << (n - i)) - 1u;  // bytes past the last flag are not flags
    return m;
}

__global__ __launch_bounds__(256) void argwhere_count_kernel(const uint8_t* flags, uint64_t n, uint32_t* counts) {
    __shared__ uint32_t part[4];
    uint32_t c = __popc(flag_bits(flags, n));
    for (int m = 1; m < 64; m <<= 1) c += __shfl_xor(c, m);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// inclusive sum over the wave
template <class T> __device__ __forceinline__ T wave_sums(T x) {
    const int lane = threadIdx.x & 63;
    for (int d = 1; d < 64; d <<= 1) {
        const T y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    return x;
}

// one workgroup of 1024: counts -> exclusive offsets, the total behind them
__global__ __launch_bounds__(1024) void argwhere_offsets_kernel(const uint32_t* counts, uint64_t blocks,
                                                                int64_t* offs) {
    __shared__ int64_t wtot[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int64_t carry = 0;
    for (uint64_t b0 = 0; b0 < blocks; b0 += 4096) {  // uniform; four counts a thread
        const uint64_t b = b0 + threadIdx.x * 4u;
        int64_t c[4], t = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            c[k] = b + uint64_t(k) < blocks ? int64_t(counts[b + uint64_t(k)]) : 0;
            t += c[k];
        }
        const int64_t incl = wave_sums(t);
        if (lane == 63) wtot[wave] = incl;
        __syncthreads();
        int64_t at = carry + incl - t;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) at += wtot[w];
            carry += wtot[w];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (b + uint64_t(k) < blocks) offs[b + uint64_t(k)] = at;
            at += c[k];
        }
        __syncthreads();  // wtot is written again
    }
    if (threadIdx.x == 0) offs[blocks] = carry;
}

struct ListArgs {
    const uint8_t* flags;
    const int64_t* offs;
    uint64_t n;
    int64_t shape[XG_MAX_RANK];
    FastDiv div[XG_MAX_RANK];  // n < 2^31
    int32_t nd;
    int32_t reverse;           // components written in reverse order (column-major traversal)
    char* out;
    int64_t rows, s_row, s_col;
};

// BIG: positions of 2^31 and more
template <bool BIG>
__global__ __launch_bounds__(256) void argwhere_list_kernel(const ListArgs a) {
    __shared__ uint16_t pos[kPerBlock];
    __shared__ uint32_t wtot[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t m = flag_bits(a.flags, a.n);
    const uint32_t c = __popc(m);
    const uint32_t incl = wave_sums(c);
    if (lane == 63) wtot[wave] = incl;
    __syncthreads();
    uint32_t at = incl - c, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        if (w < wave) at += wtot[w];
        total += wtot[w];
    }
    for (uint32_t x = m; x; x &= x - 1u) pos[at++] = uint16_t(threadIdx.x * 16u + uint32_t(__ffs(x)) - 1u);
    __syncthreads();
    const uint64_t base = uint64_t(blockIdx.x) * kPerBlock;
    const int64_t k0 = a.offs[blockIdx.x];
    for (uint32_t e = threadIdx.x; e < total; e += 256u) {
        const int64_t k = k0 + int64_t(e);
        if (k >= a.rows) break;  // rows past the output are dropped
        int64_t* dst = reinterpret_cast<int64_t*>(a.out) + k * a.s_row;
        uint64_t q = base + pos[e];
        for (int d = a.nd - 1; d >= 0; --d) {  // uniform
            uint64_t p, r;
            if constexpr (BIG) p = q / uint64_t(a.shape[d]);
            else p = fastdiv(uint32_t(q), a.div[d]);
            r = q - p * uint64_t(a.shape[d]);
            q = p;
            dst[int64_t(a.reverse ? a.nd - 1 - d : d) * a.s_col] = int64_t(r);
        }
    }
}

// flags = (bool)cond in traversal order into `flags` (contiguous bytes), the
// counts of every workgroup's positions and their offsets
void mark(const xg_expr* cond, const ExprInfo& info, bool column_major, char* buf, const ArgBuf& lay, hipStream_t st) {
    const int nd = int(info.shape.size());
    const int64_t n = numel(info.shape);
    // the traversal shape, and the expression read through reversed axes
    // for column-major order (leaves padded to the full rank first, so
    // that broadcasting stays right-aligned)
    Shape trav = info.shape;
    std::vector<xg_tensor> leaves(cond->leaves, cond->leaves + cond->n_leaves);
    if (column_major) {
        std::reverse(trav.begin(), trav.end());
        std::vector<bool> gathered(size_t(cond->n_leaves), false);  // addressed by value, not position
        for (int i = 0; i < cond->n_nodes; ++i)
            if (cond->nodes[i].op == XG_OP_GATHER && cond->nodes[i].index >= 0 && cond->nodes[i].index < cond->n_leaves)
                gathered[size_t(cond->nodes[i].index)] = true;
        for (int l = 0; l < cond->n_leaves; ++l) {
            if (gathered[size_t(l)]) continue;
            xg_tensor& t = leaves[size_t(l)];
            const int pad = nd - t.ndim;
            if (pad < 0) raise(XG_BROADCAST_ERROR, "leaf of higher rank than the expression");
            xg_tensor r = t;
            r.ndim = nd;
            for (int k = 0; k < nd; ++k) {
                const int src = nd - 1 - k - pad;  // the leaf axis that lands on reversed axis k
                r.shape[k] = src >= 0 ? t.shape[src] : 1;
                r.strides[k] = src >= 0 ? t.strides[src] : 0;
            }
            t = r;
        }
    }
    // the tree, then a cast to bool as new root
    std::vector<xg_node> nodes(cond->nodes, cond->nodes + cond->n_nodes);
    xg_node to_bool{};
    to_bool.op = XG_OP_CAST;
    to_bool.nargs = 1;
    to_bool.args[0] = cond->n_nodes - 1;
    to_bool.index = XG_BOOL;
    nodes.push_back(to_bool);
    xg_expr fe = *cond;
    fe.n_nodes = int32_t(nodes.size());
    fe.nodes = nodes.data();
    fe.leaves = leaves.data();
    xg_tensor grid{};  // the flags laid out row-major in the traversal shape
    grid.dtype = XG_BOOL;
    grid.data = buf + lay.flags_at;
    grid.ndim = nd;
    for (int64_t k = nd - 1, stv = 1; k >= 0; --k) {
        grid.shape[k] = trav[size_t(k)];
        grid.strides[k] = stv;
        stv *= std::max<int64_t>(trav[size_t(k)], 1);
    }
    assign_any(&fe, &grid, st);
    const uint8_t* flags = reinterpret_cast<const uint8_t*>(buf + lay.flags_at);
    uint32_t* counts = reinterpret_cast<uint32_t*>(buf + lay.counts_at);
    hipLaunchKernelGGL(argwhere_count_kernel, dim3(uint32_t(lay.blocks)), dim3(256), 0, st, flags, uint64_t(n), counts);
    hipLaunchKernelGGL(argwhere_offsets_kernel, dim3(1), dim3(1024), 0, st, counts, lay.blocks,
                       reinterpret_cast<int64_t*>(buf));
    check_hip(hipGetLastError(), "argwhere count launch");
}

void list(const ExprInfo& info, bool column_major, const char* buf, const ArgBuf& lay, const xg_tensor* out,
          hipStream_t st) {
    const int nd = int(info.shape.size());
    ListArgs a{};
    a.flags = reinterpret_cast<const uint8_t*>(buf + lay.flags_at);
    a.offs = reinterpret_cast<const int64_t*>(buf);
    a.n = uint64_t(numel(info.shape));
    a.nd = nd;
    a.reverse = column_major ? 1 : 0;
    for (int k = 0; k < nd; ++k) {
        a.shape[k] = info.shape[size_t(column_major ? nd - 1 - k : k)];
        a.div[k] = make_fastdiv(uint32_t(std::min<int64_t>(a.shape[k], 0x7fffffff)));
    }
    a.out = static_cast<char*>(out->data) + out->offset * 8;
    a.rows = out->shape[0];
    a.s_row = out->strides[0];
    a.s_col = out->shape[1] == 1 ? 0 : out->strides[1];
    if (a.n < (uint64_t(1) << 31))
        hipLaunchKernelGGL(argwhere_list_kernel<false>, dim3(uint32_t(lay.blocks)), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(argwhere_list_kernel<true>, dim3(uint32_t(lay.blocks)), dim3(256), 0, st, a);
    check_hip(hipGetLastError(), "argwhere launch");
    note_kernel("argwhere");
}

// the condition's type and shape, and the checks of an argwhere call
ExprInfo check_cond(const xg_expr* cond) {
    if (!cond || !cond->nodes || cond->n_nodes < 1) raise(XG_INVALID_ARGUMENT, "empty expression");
    ExprInfo info = analyse(cond);
    if (info.shape.empty()) raise(XG_INVALID_ARGUMENT, "argwhere of a 0-d expression");
    if (numel(info.shape) >= (int64_t(1) << 43)) raise(XG_UNSUPPORTED, "argwhere: too many elements");
    return info;
}

void check_rows(const xg_tensor* out, const ExprInfo& info) {
    if (!out || out->dtype != XG_INT64 || out->ndim != 2) raise(XG_INVALID_ARGUMENT, "output must be int64 [count, ndim]");
    if (out->shape[1] != int64_t(info.shape.size()))
        raise(XG_BROADCAST_ERROR, "output rows must have one column per dimension");
}

}  // namespace

}  // namespace xg

using namespace xg;

extern "C" {

xg_status xg_argwhere(const xg_expr* cond, int32_t column_major, const xg_tensor* out, xg_stream_t stream) {
    return guard([&] {
        if (!cond || !cond->nodes || cond->n_nodes < 1) raise(XG_INVALID_ARGUMENT, "empty expression");
        if (!out || out->dtype != XG_INT64 || out->ndim != 2) raise(XG_INVALID_ARGUMENT, "output must be int64 [count, ndim]");
        const ExprInfo info = check_cond(cond);
        check_rows(out, info);
        const int64_t n = numel(info.shape);
        if (n == 0 || out->shape[0] == 0) return;
        hipStream_t st = reinterpret_cast<hipStream_t>(stream);
        const ArgBuf lay(n);
        char* buf = static_cast<char*>(workspace(lay.bytes, st));
        mark(cond, info, column_major != 0, buf, lay, st);
        list(info, column_major != 0, buf, lay, out, st);
    });
}

xg_status xg_argwhere_buffer(int64_t n, size_t* bytes, size_t* total_at) {
    return guard([&] {
        if (n < 0 || !bytes || !total_at) raise(XG_INVALID_ARGUMENT, "bad argument");
        const ArgBuf lay(n);
        *bytes = lay.bytes;
        *total_at = size_t(lay.blocks) * 8;
    });
}

xg_status xg_argwhere_mark(const xg_expr* cond, int32_t column_major, void* buffer, xg_stream_t stream) {
    return guard([&] {
        const ExprInfo info = check_cond(cond);
        const int64_t n = numel(info.shape);
        if (n == 0) raise(XG_INVALID_ARGUMENT, "argwhere of an empty expression");
        if (!buffer || reinterpret_cast<uintptr_t>(buffer) % 16) raise(XG_INVALID_ARGUMENT, "buffer must be 16-byte aligned");
        mark(cond, info, column_major != 0, static_cast<char*>(buffer), ArgBuf(n), reinterpret_cast<hipStream_t>(stream));
    });
}

xg_status xg_argwhere_list(const xg_expr* cond, int32_t column_major, const void* buffer, const xg_tensor* out,
                           xg_stream_t stream) {
    return guard([&] {
        const ExprInfo info = check_cond(cond);
        check_rows(out, info);
        const int64_t n = numel(info.shape);
        if (n == 0 || out->shape[0] == 0) return;
        if (!buffer || reinterpret_cast<uintptr_t>(buffer) % 16) raise(XG_INVALID_ARGUMENT, "buffer must be 16-byte aligned");
        list(info, column_major != 0, static_cast<const char*>(buffer), ArgBuf(n), out, reinterpret_cast<hipStream_t>(stream));
    });
}

}  // extern "C"
