// ew_interp.hip — the generic interpreter of elementwise plans on gfx950:
// programs without a compiled kernel.
#include <hip/hip_runtime.h>

#include "chunk.hpp"
#include "ew.hpp"
#include "interp.hpp"

namespace xg {

// ---------------------------------------------------------------- generic interpreter
// Launches too small to compile for, plans beyond rank 4 or 32-bit offsets.
// What bounds it is the work per micro-op, not memory, so a lane carries V
// elements and every per-op cost is paid once for them:
//   * the program's registers sit in VGPRs as vectors indexed by the op's
//     operand numbers, which are the same for the whole wave (an indexed move,
//     no LDS or scratch);
//   * the op is decoded by wave-uniform branches, and the light ops
//     (arithmetic, compares, selects, conversions, exp, log, sqrt, rounding)
//     run on all V elements inside their case;
//   * LIGHT programs (only those ops, at most kInterpPre leaves) have all
//     their leaves read before the first op, so the latencies overlap and no
//     lane-dependent branch is left in the op loop.  One such branch makes the
//     compiler rebuild the whole dispatch as a cascade of flag tests, which
//     costs several times the op itself; the other programs (libm, 64-bit
//     integer division, gathers, many leaves) keep theirs in functions that
//     are called.
// W64 = false: programs without a 64-bit type, whose registers are 32 bits
// wide and carry V = 4 elements; otherwise V = 2; V = 1 for few elements of a
// program that calls (ew_interp_width).  Float32 standardisation
// (five leaves, nine ops) of [1013, 771]: 21.8 us a launch with one element a
// lane, registers in LDS and an out-of-line call per op, 9.2 us now (float64 22.0 ->
// 13.2; the headline expression forced through it 1.82 -> 0.61 ms).
constexpr int kInterpPre = 8;
typedef uint32_t reg_file_t __attribute__((ext_vector_type(kMaxRegs)));
typedef uint32_t pre_file_t __attribute__((ext_vector_type(kInterpPre)));

template <int V, bool W64> struct RegFile {
    reg_file_t lo[V], hi[W64 ? V : 1];
    __device__ __forceinline__ void get(uint32_t r, Reg (&x)[V]) const {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            x[v] = lo[v][r];
            if constexpr (W64) x[v] |= Reg(hi[v][r]) << 32;
        }
    }
    __device__ __forceinline__ void set(uint32_t r, const Reg (&x)[V]) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            lo[v][r] = uint32_t(x[v]);
            if constexpr (W64) hi[v][r] = uint32_t(x[v] >> 32);
        }
    }
};

// V elements of a leaf as raw bits, packed from w[0] up (V * 16 / V bytes at
// most); a leaf broadcast along the row holds its one element
template <int V>
__device__ __forceinline__ void load_raw_chunk(const char* p, int dt, int mode, int64_t inner_stride, int nvalid,
                                               uint32_t (&w)[4]) {
    const int esz = dtype_size(dt);
    w[0] = w[1] = w[2] = w[3] = 0;
    if (V == 1 || mode == LM_BCAST) {
        const uint64_t x = load_raw(p, esz);
        w[0] = uint32_t(x);
        w[1] = uint32_t(x >> 32);
    } else if (mode == LM_CONTIG && nvalid == V) {
        const int bytes = V * esz;
        if (bytes == 16) {
            const u32x4_t x = ld16<false>(p);
            w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
        } else if (bytes == 8) {
            const u32x2_t x = ld8<false>(p);
            w[0] = x.x; w[1] = x.y;
        } else if (bytes == 4) {
            w[0] = ld4<false>(p);
        } else {
            w[0] = uint32_t(load_raw(p, 1)) | (uint32_t(load_raw(p + 1, 1)) << 8);
        }
    } else {
        const int64_t is = inner_stride * esz;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if (v >= nvalid) continue;
            const uint64_t x = load_raw(p + int64_t(v) * is, esz);
            if (esz == 8) {
                if (2 * v < 4) w[2 * v] = uint32_t(x), w[2 * v + 1] = uint32_t(x >> 32);
            } else if (esz == 4) {
                w[v] = uint32_t(x);
            } else if (esz == 2) {
                w[v >> 1] |= uint32_t(x) << (16 * (v & 1));
            } else {
                w[0] |= uint32_t(x) << (8 * v);
            }
        }
    }
}

template <int V>
__device__ __forceinline__ void unpack_chunk(const uint32_t (&w)[4], bool bcast, int dt, Reg (&x)[V]) {
    const int esz = dtype_size(dt);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        uint64_t raw;
        if (esz == 8) raw = bcast || 2 * v >= 4 ? uint64_t(w[0]) | (uint64_t(w[1]) << 32)
                                                : uint64_t(w[(2 * v) & 3]) | (uint64_t(w[(2 * v + 1) & 3]) << 32);
        else if (esz == 4) raw = bcast ? w[0] : w[v];
        else if (esz == 2) raw = bcast ? w[0] : w[v >> 1] >> (16 * (v & 1));
        else raw = bcast ? w[0] : w[0] >> (8 * v);
        x[v] = from_storage(raw, dt);
    }
}

// the light ops on V elements; false: not one of them
template <class T, int V>
__device__ __forceinline__ bool light_float(int op, const Reg (&a)[V], const Reg (&b)[V], Reg (&r)[V]) {
#define XG_LIGHT(OP)                                                                      \
    case OP: {                                                                            \
        _Pragma("unroll") for (int v = 0; v < V; ++v) r[v] = flt_binop<T>(OP, a[v], b[v]); \
        return true;                                                                      \
    }
#define XG_LIGHT1(OP)                                                              \
    case OP: {                                                                     \
        _Pragma("unroll") for (int v = 0; v < V; ++v) r[v] = flt_unop<T>(OP, a[v]); \
        return true;                                                               \
    }
    switch (op) {
        XG_LIGHT(MO_ADD)
        XG_LIGHT(MO_SUB)
        XG_LIGHT(MO_MUL)
        XG_LIGHT(MO_DIV)
        XG_LIGHT(MO_LT)
        XG_LIGHT(MO_LE)
        XG_LIGHT(MO_GT)
        XG_LIGHT(MO_GE)
        XG_LIGHT(MO_EQ)
        XG_LIGHT(MO_NE)
        XG_LIGHT1(MO_NEG)
        XG_LIGHT1(MO_ABS)
        XG_LIGHT1(MO_EXP)
        XG_LIGHT1(MO_LOG)
        XG_LIGHT1(MO_SQRT)
        XG_LIGHT1(MO_FLOOR)
        XG_LIGHT1(MO_CEIL)
        XG_LIGHT1(MO_TRUNC)
        XG_LIGHT1(MO_ROUND)
    default: return false;
    }
#undef XG_LIGHT
#undef XG_LIGHT1
}

template <class T, int V>
__device__ __forceinline__ bool light_int(int op, const Reg (&a)[V], const Reg (&b)[V], Reg (&r)[V]) {
#define XG_LIGHT(OP)                                                                      \
    case OP: {                                                                            \
        _Pragma("unroll") for (int v = 0; v < V; ++v) r[v] = int_binop<T>(OP, a[v], b[v]); \
        return true;                                                                      \
    }
    switch (op) {
        XG_LIGHT(MO_ADD)
        XG_LIGHT(MO_SUB)
        XG_LIGHT(MO_MUL)
        XG_LIGHT(MO_BAND)
        XG_LIGHT(MO_BOR)
        XG_LIGHT(MO_BXOR)
        XG_LIGHT(MO_SHL)
        XG_LIGHT(MO_SHR)
        XG_LIGHT(MO_LT)
        XG_LIGHT(MO_LE)
        XG_LIGHT(MO_GT)
        XG_LIGHT(MO_GE)
        XG_LIGHT(MO_EQ)
        XG_LIGHT(MO_NE)
    default: return false;
    }
#undef XG_LIGHT
}

// the conversions among the light ops
#define XG_LIGHT_CVT32                                                                                          \
    XG_CVT(XG_INT32, XG_FLOAT32) XG_CVT(XG_FLOAT32, XG_INT32) XG_CVT(XG_BOOL, XG_FLOAT32) XG_CVT(XG_BOOL, XG_INT32) \
    XG_CVT(XG_FLOAT32, XG_BOOL) XG_CVT(XG_INT32, XG_BOOL) XG_CVT(XG_UINT8, XG_INT32) XG_CVT(XG_UINT8, XG_FLOAT32)   \
    XG_CVT(XG_INT8, XG_INT32) XG_CVT(XG_INT16, XG_INT32)
#define XG_LIGHT_CVT64                                                                                               \
    XG_CVT(XG_FLOAT32, XG_FLOAT64) XG_CVT(XG_FLOAT64, XG_FLOAT32) XG_CVT(XG_INT32, XG_FLOAT64) XG_CVT(XG_INT32, XG_INT64) \
    XG_CVT(XG_INT64, XG_FLOAT64) XG_CVT(XG_BOOL, XG_INT64) XG_CVT(XG_BOOL, XG_FLOAT64) XG_CVT(XG_FLOAT64, XG_BOOL)

template <int V, bool W64>
__device__ __forceinline__ bool light_op(const MicroOp& m, const Reg (&a)[V], const Reg (&b)[V], const Reg (&c)[V],
                                         const uint64_t* kconst, Reg (&r)[V]) {
    switch (m.op) {
    case MO_CONST: {
        const Reg k = kconst[m.aux];
#pragma unroll
        for (int v = 0; v < V; ++v) r[v] = k;
        return true;
    }
    case MO_LNOT:
#pragma unroll
        for (int v = 0; v < V; ++v) r[v] = uint32_t(a[v]) == 0;
        return true;
    case MO_LAND:
#pragma unroll
        for (int v = 0; v < V; ++v) r[v] = (uint32_t(a[v]) != 0) & (uint32_t(b[v]) != 0);
        return true;
    case MO_LOR:
#pragma unroll
        for (int v = 0; v < V; ++v) r[v] = (uint32_t(a[v]) != 0) | (uint32_t(b[v]) != 0);
        return true;
    case MO_SEL:
#pragma unroll
        for (int v = 0; v < V; ++v) r[v] = uint32_t(a[v]) != 0 ? b[v] : c[v];
        return true;
    case MO_CVT:
#define XG_CVT(FROM, TO)                                                            \
    if (m.t == FROM && m.aux == TO) {                                               \
        _Pragma("unroll") for (int v = 0; v < V; ++v) r[v] = cvt(a[v], FROM, TO);    \
        return true;                                                                \
    }
        XG_LIGHT_CVT32
        if constexpr (W64) { XG_LIGHT_CVT64 }
#undef XG_CVT
        return false;
    default: break;
    }
    switch (m.t) {
    case XG_FLOAT32: return light_float<float>(m.op, a, b, r);
    case XG_INT32: return light_int<int32_t>(m.op, a, b, r);
    case XG_FLOAT64:
        if constexpr (W64) return light_float<double>(m.op, a, b, r);
        return false;
    case XG_INT64:
        if constexpr (W64) return light_int<int64_t>(m.op, a, b, r);
        return false;
    default: return false;
    }
}

// V raw elements of a leaf, out of line (see LIGHT above)
template <int V>
static __device__ __noinline__ u32x4_t load_chunk_call(const char* p, int dt, int mode, int64_t inner_stride, int nvalid) {
    uint32_t w[4];
    load_raw_chunk<V>(p, dt, mode, inner_stride, nvalid, w);
    return u32x4_t{w[0], w[1], w[2], w[3]};
}

static __device__ __noinline__ Reg gather_call(const LeafView* lv, bool valid, Reg off) {
    const Reg o[1] = {off};
    Reg r[1];
    gather_vals<1>(lv->ptr, lv->dtype, lv->stride[0], lv->stride[1], valid ? 1 : 0, o, r);
    return r[0];
}

template <int V, bool W64, bool COMPACT, bool LIGHT>
__global__ __launch_bounds__(256) void ew_interp_kernel(const EwPlan plan_arg) {
    const EwPlan& plan = kernel_plan<DynSpec>(plan_arg);
    const uint32_t nunits = uint32_t(plan.units);
    const uint32_t step = gridDim.x * 256u;
    const int rank = plan.rank, nleaves = plan.prog.nleaves, nops = plan.prog.nops;
    for (uint32_t u = blockIdx.x * 256u + threadIdx.x; u < nunits; u += step) {
        const uint32_t row = fastdiv(u, plan.div_chunks);
        const uint32_t j0 = (u - row * plan.nchunks) * uint32_t(V);
        const int nvalid = min(V, int(plan.inner - j0));
        uint32_t idx[kMaxRank] = {};
        uint32_t q = row;
        if constexpr (COMPACT) {
            if (rank == 4) {
                const uint32_t d = fastdiv(q, plan.div[2]);
                idx[2] = q - d * plan.shape32[2];
                q = d;
            }
            if (rank >= 3) {
                const uint32_t d = fastdiv(q, plan.div[1]);
                idx[1] = q - d * plan.shape32[1];
                q = d;
            }
            idx[0] = rank >= 2 ? q : 0u;
        } else {
#pragma unroll
            for (int k = kMaxRank - 2; k >= 0; --k) {
                if (k <= rank - 2) {
                    const uint32_t d = fastdiv(q, plan.div[k]);
                    idx[k] = q - d * uint32_t(plan.shape[k]);
                    q = d;
                }
            }
        }
        // element offset of the unit in operand l (kMaxLeaves: the output)
        auto offset = [&](int l) -> int64_t {
            if constexpr (COMPACT) {
                const int32_t(&st)[4] = plan.cst[l];
                return int32_t(j0) * st[rank - 1] + int32_t(idx[0]) * st[0] + int32_t(idx[1]) * st[1] + int32_t(idx[2]) * st[2];
            } else {
                return unit_offset<true>(l == kMaxLeaves ? plan.out_stride : plan.leaves[l].stride, idx, rank, j0);
            }
        };
        pre_file_t pw[4];
        if constexpr (LIGHT) {
#pragma unroll
            for (int l = 0; l < kInterpPre; ++l) {
                uint32_t w[4] = {0, 0, 0, 0};
                if (l < nleaves) {
                    const LeafView& lv = plan.leaves[l];
                    load_raw_chunk<V>(lv.ptr + offset(l) * dtype_size(lv.dtype), lv.dtype, lm_base(lv.mode),
                                      lv.stride[rank - 1], nvalid, w);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) pw[k][l] = w[k];
            }
        }
        RegFile<V, W64> file;
        MicroOp next = plan.prog.ops[0];
        for (int pc = 0; pc < nops; ++pc) {
            const MicroOp m = next;
            next = plan.prog.ops[min(pc + 1, kMaxOps - 1)];
            Reg r[V];
            if (m.op == MO_LOAD) {
                const LeafView& lv = plan.leaves[m.aux];
                uint32_t w[4];
                if constexpr (LIGHT) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) w[k] = pw[k][m.aux];
                } else {
                    const u32x4_t x = load_chunk_call<V>(lv.ptr + offset(m.aux) * dtype_size(lv.dtype), lv.dtype,
                                                         lm_base(lv.mode), lv.stride[rank - 1], nvalid);
                    w[0] = x.x, w[1] = x.y, w[2] = x.z, w[3] = x.w;
                }
                unpack_chunk<V>(w, lm_base(lv.mode) == LM_BCAST, lv.dtype, r);
            } else {
                Reg a[V], b[V], c[V];
                file.get(m.a, a);
                file.get(m.b, b);
                file.get(m.c, c);
                const bool done = light_op<V, W64>(m, a, b, c, plan.prog.consts, r);
                if constexpr (!LIGHT) {
                    if (!done) {
                        const bool gather = m.op == MO_GATHER;
#pragma unroll 1
                        for (int v = 0; v < V; ++v) {  // the V operands rotate through slot 0
                            const Reg x = gather ? gather_call(&plan.leaves[m.aux], v < nvalid, a[0])
                                                 : exec_scalar_dyn(m, a[0], b[0], c[0], plan.prog.consts);
#pragma unroll
                            for (int k = 0; k + 1 < V; ++k) {
                                a[k] = a[k + 1];
                                b[k] = b[k + 1];
                                c[k] = c[k + 1];
                                r[k] = r[k + 1];
                            }
                            r[V - 1] = x;
                        }
                    }
                }
            }
            file.set(m.dst, r);
        }
        Reg res[V];
        file.get(plan.prog.result_reg, res);
        const int odt = plan.out_dtype, esz = dtype_size(odt);
        char* p = plan.out_ptr + offset(kMaxLeaves) * esz;
        if (V > 1 && lm_base(plan.out_mode) == LM_CONTIG && nvalid == V) {
            if constexpr (V > 1) store_vec<V>(p, esz, odt, res);
        } else {
            const int64_t os = plan.out_stride[rank - 1] * esz;
#pragma unroll
            for (int v = 0; v < V; ++v)
                if (v < nvalid) store_raw(p + int64_t(v) * os, esz, to_storage(res[v], odt));
        }
    }
}

// ops that light_op does not take
int called_ops(const EwPlan& p) {
    auto cvt_ok = [](int from, int to) {
#define XG_CVT(FROM, TO) if (from == FROM && to == TO) return true;
        XG_LIGHT_CVT32
        XG_LIGHT_CVT64
#undef XG_CVT
        return false;
    };
    auto light = [&](const MicroOp& m) {
        switch (m.op) {
        case MO_LOAD: case MO_CONST: case MO_LNOT: case MO_LAND: case MO_LOR: case MO_SEL: return true;
        case MO_CVT: return cvt_ok(m.t, m.aux);
        case MO_ADD: case MO_SUB: case MO_MUL: case MO_LT: case MO_LE: case MO_GT: case MO_GE: case MO_EQ: case MO_NE:
            return m.t == XG_FLOAT32 || m.t == XG_FLOAT64 || m.t == XG_INT32 || m.t == XG_INT64;
        case MO_DIV: case MO_NEG: case MO_ABS: case MO_EXP: case MO_LOG: case MO_SQRT: case MO_FLOOR: case MO_CEIL:
        case MO_TRUNC: case MO_ROUND:
            return m.t == XG_FLOAT32 || m.t == XG_FLOAT64;
        case MO_BAND: case MO_BOR: case MO_BXOR: case MO_SHL: case MO_SHR: return m.t == XG_INT32 || m.t == XG_INT64;
        default: return false;
        }
    };
    int n = 0;
    for (int i = 0; i < p.prog.nops; ++i) n += light(p.prog.ops[i]) ? 0 : 1;
    return n;
}

// LIGHT: every op is one light_op takes, and the leaves fit the registers
bool interp_light(const EwPlan& p) {
    if (p.prog.nleaves > kInterpPre) return false;
    for (int l = 0; l < p.prog.nleaves; ++l)
        if (p.prog.leaf_gather[l]) return false;
    return called_ops(p) == 0;
}

using InterpFn = void (*)(const EwPlan);

template <int V, bool W64> InterpFn interp_kernel(bool compact, bool light) {
    if (light) return compact ? ew_interp_kernel<V, W64, true, true> : ew_interp_kernel<V, W64, false, true>;
    return compact ? ew_interp_kernel<V, W64, true, false> : ew_interp_kernel<V, W64, false, false>;
}

// one element a lane: the programs that call
InterpFn interp_kernel_1(bool compact, bool w64) {
    if (w64) return compact ? ew_interp_kernel<1, true, true, false> : ew_interp_kernel<1, true, false, false>;
    return compact ? ew_interp_kernel<1, false, true, false> : ew_interp_kernel<1, false, false, false>;
}

// something in the program or its operands is 64 bits wide
bool interp_64(const EwPlan& p) {
    if (dtype_size(p.out_dtype) == 8) return true;
    for (int l = 0; l < p.prog.nleaves; ++l)
        if (p.prog.leaf_gather[l] || dtype_size(p.leaves[l].dtype) == 8) return true;
    for (int i = 0; i < p.prog.nops; ++i) {
        const MicroOp& m = p.prog.ops[i];
        if (m.op == MO_GATHER || (m.op != MO_LOAD && is_64bit(m.t)) || (m.op == MO_CVT && is_64bit(m.aux))) return true;
    }
    return false;
}

// Elements per lane.  Light programs: four when nothing is 64 bits wide, else
// two.  The others call a function per op and element, one after the other in a
// lane: with few elements, whose waves do not fill the GPU, they take one a
// lane (float32 tanh(sin(a) + cos(b)) * erf(a) + atan(b) of 30,000 elements
// 20.8 us with four, 9.7 with one; of 400,000 22.8 and 18.1; of 900,000 29.0
// and 30.6; float64 of 120,000 15.0 and 11.2, of 400,000 21.6 and 22.7; nine
// float32 leaves added, of 250,000 15.6 and 13.3, of 400,000 15.8 and 20.1).
int ew_interp_width(const EwPlan& p) {
    const bool w64 = interp_64(p);
    const uint64_t n = p.nchunks ? p.units / p.nchunks * p.inner : 0;
    if (n < (uint64_t(1) << 19) && !interp_light(p) &&
        (n < (uint64_t(1) << 18) || (!w64 && called_ops(p) * 4 >= p.prog.nops)))
        return 1;
    return w64 ? 2 : 4;
}

hipError_t launch_ew_interp(const EwPlan& p, int V, dim3 grid, hipStream_t stream) {
    if (V != ew_interp_width(p)) return hipErrorInvalidValue;
    const bool light = interp_light(p);
    InterpFn f = V == 1 ? interp_kernel_1(p.compact != 0, interp_64(p)) : V == 4 ? interp_kernel<4, false>(p.compact != 0, light) : interp_kernel<2, true>(p.compact != 0, light);
    hipLaunchKernelGGL(f, grid, dim3(256), 0, stream, p);
    return hipGetLastError();
}

}  // namespace xg
