/*
 * m3_hip_binary.hip - broadcast elementwise ADD/MUL/SUB/DIV for gfx950.
 *
 * Semantics are the reference's m3_host_binary (src/m3_op_execute_basic.c:
 * 61-77) and Metal m3_binary_apply (src/m3_backend_metal_basic.m:66-104):
 * out[i] = round_out(float(left[b_l(i)]) (op) float(right[b_r(i)])) with
 * right-aligned broadcasting, one F32 operation per element, round to
 * nearest even on store.
 *
 * Launch planning (host side):
 *   1. the output index space is coalesced: size-1 axes are dropped and
 *      neighbouring axes merge when every operand steps across them as one
 *      axis (m3_plan_index_space);
 *   2. each input is classified by how its element offset depends on the
 *      flat output index f:
 *        FULL     offset = f                 (same layout as the output)
 *        TRAIL    offset = f mod P           (trailing-axis broadcast,
 *                                             e.g. x[8,1024,1536]*c[1536])
 *        ROW      offset = (f / I) mod P     (broadcast over inner axes,
 *                                             I a multiple of 4)
 *        SCALAR   offset = 0
 *        TRAIL_CUT, ROW_CUT                  (the same two with P or I at
 *                                             least 4 but no multiple of
 *                                             it: a group of 4 may wrap or
 *                                             take two elements)
 *        PERIODIC offset = (f / I) mod P     (any I, per-element loads)
 *   3. when both inputs classify, and there are enough elements (or their
 *      loads are known when a kernel is compiled, m3_operand_kind), the
 *      vector kernel runs: each lane handles groups of 4 consecutive
 *      outputs with 16-byte (F32) or 8-byte (F16/BF16) loads and stores at
 *      any alignment, two groups in flight per lane, grid-stride over the
 *      tensor; with F32 operands and a tensor whose lanes are all resident
 *      at once, its held form instead (all loads, then the stores after a
 *      timed wait); divisions by I and P use precomputed multiply-shift
 *      divisors;
 *   4. anything else runs the general kernel: per-element offsets from the
 *      coalesced stride table.
 * A run of such operations and float casts in which each takes the one
 * before as an operand is one launch of the chain kernel (m3_chain_kernel):
 * every result is stored, none is read back.
 * All operands are read as F32 bit patterns, so NaN payloads survive
 * loads; m3_binary_f32_bits applies the operation and the NaN rule.
 */
#include "m3_hip_internal.h"

#include <cstring>

namespace {

enum m3_bin_mode : uint32_t {
    M3_BIN_FULL = 0,
    M3_BIN_TRAIL = 1,
    M3_BIN_ROW = 2,
    M3_BIN_SCALAR = 3,
    M3_BIN_PERIODIC = 4,
    M3_BIN_TRAIL_CUT = 5,
    M3_BIN_ROW_CUT = 6
};

struct m3_bin_operand {
    const uint8_t *base; /* first element (byte offset applied) */
    uint32_t mode;
    uint32_t dtype;
    m3_fast_div inner;
    m3_fast_div period;
};

struct m3_bin_vec_args {
    m3_bin_operand left;
    m3_bin_operand right;
    uint8_t *out;
    uint32_t out_dtype;
    uint32_t count;  /* elements, < 2^32 */
    uint32_t groups; /* count / 4 */
    m3_hip_gate list_gate;
};

constexpr uint32_t kThreads = 256U;
/* a kernel's element type: one dtype throughout, or each operand's own */
constexpr uint32_t kAnyDtype = 0xffffffffU;
constexpr uint32_t kUnroll = 2U; /* groups in flight per lane (measured best) */

__device__ __forceinline__ uint32_t m3_load_raw(const uint8_t *p,
                                                uint32_t dtype)
{
    return dtype == M3N_F32 ? *(const uint32_t *)p
                            : (uint32_t) * (const uint16_t *)p;
}

__device__ __forceinline__ uint32_t m3_operand_index(const m3_bin_operand &o,
                                                     uint32_t f)
{
    switch (o.mode) {
    case M3_BIN_FULL:
        return f;
    case M3_BIN_TRAIL:
    case M3_BIN_TRAIL_CUT:
        return f - m3_fast_div_q(o.period, f) * o.period.divisor;
    case M3_BIN_SCALAR:
        return 0U;
    default: {
        uint32_t q = m3_fast_div_q(o.inner, f);

        return q - m3_fast_div_q(o.period, q) * o.period.divisor;
    }
    }
}

/* F32 bits of the operand's element at `index`. */
template <uint32_t DT>
__device__ __forceinline__ uint32_t m3_operand_at(const m3_bin_operand &o,
                                                  uint32_t index)
{
    uint32_t dtype = DT == kAnyDtype ? o.dtype : DT;
    uint32_t esize = dtype == M3N_F32 ? 4U : 2U;

    return m3_load_as_f32_bits(
        m3_load_raw(o.base + (uint64_t)index * esize, dtype), dtype);
}

template <uint32_t DT>
__device__ __forceinline__ uint32_t m3_operand_element(const m3_bin_operand &o,
                                                       uint32_t f)
{
    return m3_operand_at<DT>(o, m3_operand_index(o, f));
}

/* F32 bits of operand elements f..f+3 (f a multiple of 4). */
template <uint32_t DT>
__device__ __forceinline__ uint4 m3_operand_load4(const m3_bin_operand &o,
                                                  uint32_t f)
{
    uint32_t dtype = DT == kAnyDtype ? o.dtype : DT;

    if (o.mode == M3_BIN_FULL || o.mode == M3_BIN_TRAIL) {
        uint32_t index = o.mode == M3_BIN_FULL
                             ? f
                             : f - m3_fast_div_q(o.period, f) *
                                       o.period.divisor;

        /* a full operand is read once per launch: streamed; a trailing
         * broadcast operand is reread by every row: cached, and written
         * element by element (the compiler joins the accesses later): as
         * one vector load it is merged with the streamed one above, which
         * then is no longer nontemporal (x[8,1024,1536] * c[1536] 24.1
         * against 17.7 us). */
        if (dtype == M3N_F32) {
            const uint8_t *p = o.base + (uint64_t)index * 4U;

            if (o.mode == M3_BIN_FULL) {
                return m3_stream_load((const uint4 *)p);
            }
            const uint32_t *w = (const uint32_t *)p;

            return make_uint4(w[0], w[1], w[2], w[3]);
        }
        const uint8_t *p = o.base + (uint64_t)index * 2U;
        uint2 half;

        if (o.mode == M3_BIN_FULL) {
            half = m3_stream_load((const uint2 *)p);
        } else {
            const uint16_t *h = (const uint16_t *)p;

            half = make_uint2(h[0] | ((uint32_t)h[1] << 16U),
                              h[2] | ((uint32_t)h[3] << 16U));
        }
        return m3_widen4_bits(half, dtype);
    }
    if (o.mode == M3_BIN_SCALAR) {
        uint32_t v = m3_operand_element<DT>(o, f);

        return make_uint4(v, v, v, v);
    }
    if (o.mode == M3_BIN_ROW) {
        /* one element, from cache; a wave whose groups lie in one run, as
         * most do when runs are long, finds and converts it once, in scalar
         * registers */
        const uint32_t q = m3_fast_div_q(o.inner, f);
        const uint32_t run = (uint32_t)__builtin_amdgcn_readfirstlane((int)q);

        if (__all(q == run)) {
            const uint32_t v = m3_operand_at<DT>(
                o, run - m3_fast_div_q(o.period, run) * o.period.divisor);

            return make_uint4(v, v, v, v);
        }
        const uint32_t v = m3_operand_at<DT>(
            o, q - m3_fast_div_q(o.period, q) * o.period.divisor);

        return make_uint4(v, v, v, v);
    }
    if (o.mode == M3_BIN_ROW_CUT) {
        /* the same, or two elements for a group in which a run of I ends:
         * both from cache (the second is the first again in the others) */
        const uint32_t q = m3_fast_div_q(o.inner, f);
        const uint32_t here = (q + 1U) * o.inner.divisor - f;
        const uint32_t run = (uint32_t)__builtin_amdgcn_readfirstlane((int)q);

        if (__all(q == run && here >= 4U)) {
            const uint32_t v = m3_operand_at<DT>(
                o, run - m3_fast_div_q(o.period, run) * o.period.divisor);

            return make_uint4(v, v, v, v);
        }
        const uint32_t next = here < 4U ? q + 1U : q;
        const uint32_t v = m3_operand_at<DT>(
            o, q - m3_fast_div_q(o.period, q) * o.period.divisor);
        const uint32_t w = m3_operand_at<DT>(
            o, next - m3_fast_div_q(o.period, next) * o.period.divisor);

        return make_uint4(v, here > 1U ? v : w, here > 2U ? v : w,
                          here > 3U ? v : w);
    }
    if (o.mode == M3_BIN_TRAIL_CUT) {
        /* consecutive elements that may wrap to the period's start */
        const uint32_t p = o.period.divisor;
        const uint32_t i = f - m3_fast_div_q(o.period, f) * p;

        return make_uint4(
            m3_operand_at<DT>(o, i),
            m3_operand_at<DT>(o, i + 1U < p ? i + 1U : i + 1U - p),
            m3_operand_at<DT>(o, i + 2U < p ? i + 2U : i + 2U - p),
            m3_operand_at<DT>(o, i + 3U < p ? i + 3U : i + 3U - p));
    }
    return make_uint4(m3_operand_element<DT>(o, f),
                      m3_operand_element<DT>(o, f + 1U),
                      m3_operand_element<DT>(o, f + 2U),
                      m3_operand_element<DT>(o, f + 3U));
}

template <uint32_t DT>
__device__ __forceinline__ void m3_store4(uint8_t *out, uint32_t dtype,
                                          uint32_t f, uint4 v)
{
    if (DT == M3N_F32 || dtype == M3N_F32) {
        m3_stream_store((uint4 *)(out + (uint64_t)f * 4U), v);
        return;
    }
    m3_stream_store((uint2 *)(out + (uint64_t)f * 2U),
                    m3_narrow4_bits(v, dtype));
}

/* What a group loads of an F32 operand, where that is known when the kernel
 * is compiled: its own four elements, four of a trailing broadcast, or one
 * element (of a row; a scalar is a row operand whose inner axis and period
 * are 1). ANY: by the operand's mode. */
enum m3_operand_kind : uint32_t {
    M3_KIND_FULL = 0,
    M3_KIND_TRAIL = 1,
    M3_KIND_ONE = 2,
    M3_KIND_ANY = 3
};

/* F32 bits of elements f..f+3 of an F32 operand of kind KIND (not ANY). */
template <uint32_t KIND>
__device__ __forceinline__ uint4 m3_kind_load4(const m3_bin_operand &o,
                                               uint32_t f)
{
    if constexpr (KIND == M3_KIND_FULL) {
        return m3_stream_load((const uint4 *)(o.base + (uint64_t)f * 4U));
    } else if constexpr (KIND == M3_KIND_TRAIL) {
        const uint32_t index =
            f - m3_fast_div_q(o.period, f) * o.period.divisor;
        const m3_u32x4 w =
            *(const m3_u32x4_any *)(o.base + (uint64_t)index * 4U);

        return make_uint4(w[0], w[1], w[2], w[3]);
    } else {
        const uint32_t run = m3_fast_div_q(o.inner, f);
        const uint32_t v = m3_operand_at<M3N_F32>(
            o, run - m3_fast_div_q(o.period, run) * o.period.divisor);

        return make_uint4(v, v, v, v);
    }
}

/* F32 operands of known kinds have an instance per pair of kinds: with all
 * modes in one kernel, calls that need the simplest loads pay for the others'
 * instructions (20,000 elements 3.3 us against 2.6, 3,000,000 times a scalar
 * 6.1 against 4.8, 4,194,304 in rows of 8 times a column 8.1 against 5.8;
 * without the modes that cut groups 3.1, 5.6 and 6.8). Otherwise the loads
 * go by the modes (kinds ANY). */
template <int OP, uint32_t DT, uint32_t LEFT, uint32_t RIGHT>
__global__ __launch_bounds__(256) void m3_binary_vec_kernel(m3_bin_vec_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    constexpr uint32_t UNROLL = kUnroll;
    const uint32_t out_dtype = DT == kAnyDtype ? a.out_dtype : DT;
    const uint32_t step = gridDim.x * kThreads * UNROLL;

    for (uint32_t first = blockIdx.x * kThreads * UNROLL + threadIdx.x;
         first < a.groups; first += step) {
        uint4 left[UNROLL];
        uint4 right[UNROLL];

#pragma unroll
        for (uint32_t u = 0U; u < UNROLL; ++u) {
            uint32_t g = first + u * kThreads;

            if constexpr (LEFT == M3_KIND_ANY) {
                if (g < a.groups) {
                    left[u] = m3_operand_load4<DT>(a.left, g * 4U);
                    right[u] = m3_operand_load4<DT>(a.right, g * 4U);
                }
            } else {
                /* groups past the end read the last one, store nothing */
                const uint32_t f = 4U * min(g, a.groups - 1U);

                left[u] = m3_kind_load4<LEFT>(a.left, f);
                right[u] = m3_kind_load4<RIGHT>(a.right, f);
            }
        }
#pragma unroll
        for (uint32_t u = 0U; u < UNROLL; ++u) {
            uint32_t g = first + u * kThreads;

            if (g < a.groups) {
                uint4 r;

                r.x = m3_binary_f32_bits(OP, left[u].x, right[u].x);
                r.y = m3_binary_f32_bits(OP, left[u].y, right[u].y);
                r.z = m3_binary_f32_bits(OP, left[u].z, right[u].z);
                r.w = m3_binary_f32_bits(OP, left[u].w, right[u].w);
                m3_store4<DT>(a.out, out_dtype, g * 4U, r);
            }
        }
    }
    /* Tail: the last count % 4 elements. */
    if (blockIdx.x == 0U && threadIdx.x < a.count - a.groups * 4U) {
        uint32_t f = a.groups * 4U + threadIdx.x;
        uint32_t r = m3_binary_f32_bits(
            OP, m3_operand_element<DT>(a.left, f),
            m3_operand_element<DT>(a.right, f));
        uint32_t raw = m3_store_from_f32_bits(r, out_dtype);

        if (out_dtype == M3N_F32) {
            *(uint32_t *)(a.out + (uint64_t)f * 4U) = raw;
        } else {
            *(uint16_t *)(a.out + (uint64_t)f * 2U) = (uint16_t)raw;
        }
    }
}

/* Groups of four outputs per lane of the held form, and its workgroups
 * per CU (at most 128 VGPRs: four waves per SIMD, all resident at once). */
constexpr int kHeldGroups = 12;
constexpr uint32_t kHeldBlocksPerCu = 4U;
/* Its wait before the stores, as a multiple of the time the launch's
 * reads of its full operands take at 8 TB/s. Measured in bench.py on
 * MUL x[8,1024,1536] * c[1536], alternating libraries on one box: 17.6-17.9
 * us at 1.0 and 1.19 against 18.1-18.6 us with the streaming kernel (1.4:
 * 18.5-18.8; eight groups per lane, whose workgroups were not all
 * resident, 20-31 us). */
constexpr double kBinaryHoldFactor = 1.1;

/* The held form of the F32 vector kernel, for a launch whose workgroups
 * are all resident at once: each lane loads its K groups of both operands,
 * forms the results, and stores them only hold_ticks after its start
 * (s_memrealtime), so that the launch's writes do not compete with its reads
 * still in flight. The wait is bounded by the clock; results are those of
 * m3_binary_vec_kernel. An instance per pair of operand kinds, and lanes
 * past the end read the last group, so that the loads are one straight line,
 * all in flight: with the kinds tested among the loads, the time moved with
 * every change of the code around them (x[131072,64] * c[64], the same loads:
 * 12.5, 14.0 and 20.2 us; 12.8 here, and 12.8 instead of 19.2 times a
 * column of 131,072). */
template <int OP, int K, uint32_t LEFT, uint32_t RIGHT>
__global__ __launch_bounds__(256) void m3_binary_held_kernel(
    m3_bin_vec_args a, uint32_t hold_ticks)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t start = __builtin_amdgcn_s_memrealtime();
    const uint32_t first = blockIdx.x * kThreads * K + threadIdx.x;
    uint4 left[K];
    uint4 right[K];

#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t f =
            4U * min(first + (uint32_t)k * kThreads, a.groups - 1U);

        left[k] = m3_kind_load4<LEFT>(a.left, f);
        right[k] = m3_kind_load4<RIGHT>(a.right, f);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        left[k].x = m3_binary_f32_bits(OP, left[k].x, right[k].x);
        left[k].y = m3_binary_f32_bits(OP, left[k].y, right[k].y);
        left[k].z = m3_binary_f32_bits(OP, left[k].z, right[k].z);
        left[k].w = m3_binary_f32_bits(OP, left[k].w, right[k].w);
    }
    while (__builtin_amdgcn_s_memrealtime() - start < (uint64_t)hold_ticks) {
        __builtin_amdgcn_s_sleep(2);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t g = first + (uint32_t)k * kThreads;

        if (g < a.groups) {
            m3_store4<M3N_F32>(a.out, M3N_F32, g * 4U, left[k]);
        }
    }
    /* Tail: the last count % 4 elements. */
    if (blockIdx.x == 0U && threadIdx.x < a.count - a.groups * 4U) {
        uint32_t f = a.groups * 4U + threadIdx.x;

        *(uint32_t *)(a.out + (uint64_t)f * 4U) = m3_binary_f32_bits(
            OP, m3_operand_element<M3N_F32>(a.left, f),
            m3_operand_element<M3N_F32>(a.right, f));
    }
}

/* ---- chains ----------------------------------------------------------------- */

constexpr uint32_t kChainCast = 4U; /* an op after the four of m3_numeric.h */

/* One operation of a chain: value = value (op) other, or other (op) value,
 * or a cast; the result rounded to out_dtype and stored at out. */
struct m3_chain_step {
    m3_bin_operand other;
    uint8_t *out;
    uint32_t out_dtype;
    uint32_t op;
    uint32_t other_left;
};

struct m3_chain_args {
    m3_bin_operand value; /* the first operation's left operand */
    m3_chain_step steps[M3_HIP_MAX_CHAIN];
    uint32_t count;  /* elements, < 2^32 */
    uint32_t groups; /* count / 4 */
    m3_hip_gate list_gate;
};

/* Four results of one operation (the same in every lane), with the NaN
 * rule applied only in a wave that holds a NaN. */
__device__ __forceinline__ uint4 m3_chain_op4(uint32_t op, uint4 x, uint4 y)
{
    const float4 a = make_float4(m3_bits_f32(x.x), m3_bits_f32(x.y),
                                 m3_bits_f32(x.z), m3_bits_f32(x.w));
    const float4 b = make_float4(m3_bits_f32(y.x), m3_bits_f32(y.y),
                                 m3_bits_f32(y.z), m3_bits_f32(y.w));
    float4 r;

    if (op == M3N_ADD) {
        r = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
    } else if (op == M3N_MUL) {
        r = make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
    } else if (op == M3N_SUB) {
        r = make_float4(a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w);
    } else {
        r = make_float4(a.x / b.x, a.y / b.y, a.z / b.z, a.w / b.w);
    }
    uint4 v = make_uint4(m3_f32_bits(r.x), m3_f32_bits(r.y),
                         m3_f32_bits(r.z), m3_f32_bits(r.w));

    if (__any(r.x != r.x || r.y != r.y || r.z != r.z || r.w != r.w)) {
        const int commutative = op == M3N_ADD || op == M3N_MUL;

        v.x = m3_binary_nan_fix(v.x, x.x, y.x, commutative);
        v.y = m3_binary_nan_fix(v.y, x.y, y.y, commutative);
        v.z = m3_binary_nan_fix(v.z, x.z, y.z, commutative);
        v.w = m3_binary_nan_fix(v.w, x.w, y.w, commutative);
    }
    return v;
}

/* Runs of up to M3_HIP_MAX_CHAIN operations over one element space, each
 * taking the one before as an operand: a lane loads every operand of its
 * groups of four, applies the operations in order, rounding each result to
 * its output's dtype as a store and a load back would, and stores all
 * results. Bound by HBM: a separate launch per operation also reads every
 * intermediate result back. DT: every operand and output is of that dtype
 * (kAnyDtype: each its own), which drops the choice per value that bound
 * 16-bit chains by instructions. Measured against one launch per
 * operation, passes over the same buffers: F32 x[2,512,24001] * s[512,1] +
 * b[512,1] 67.5 -> 44.8 us (6.6 TB/s; over buffers that change from pass to
 * pass 66.6 -> 54.6, 5.4 TB/s), BF16 107 -> 32.7, F16 120 -> 40.4;
 * x[8,1024,1536] * c[1536] then to BF16 and back to F32 47.4 -> 28.8. Two
 * groups per lane and one tile per workgroup: one group 29.8 and 46.0, four
 * 30.6 and 46.8; 16 workgroups per CU in a loop the same within 1%. */
template <int STEPS, uint32_t DT, int UNROLL>
__global__ __launch_bounds__(256) void m3_chain_kernel(m3_chain_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint32_t step = gridDim.x * kThreads * UNROLL;

    for (uint32_t first = blockIdx.x * kThreads * UNROLL + threadIdx.x;
         first < a.groups; first += step) {
        uint4 value[UNROLL];
        uint4 other[UNROLL][STEPS];

#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            /* groups past the end read the last one and store nothing */
            const uint32_t f =
                4U * min(first + u * kThreads, a.groups - 1U);

            value[u] = m3_operand_load4<DT>(a.value, f);
#pragma unroll
            for (int k = 0; k < STEPS; ++k) {
                if (a.steps[k].op != kChainCast) {
                    other[u][k] =
                        m3_operand_load4<DT>(a.steps[k].other, f);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const uint32_t g = first + u * kThreads;

#pragma unroll
            for (int k = 0; k < STEPS; ++k) {
                const m3_chain_step &s = a.steps[k];
                const uint32_t dtype = DT == kAnyDtype ? s.out_dtype : DT;

                if (s.op != kChainCast) {
                    const bool left = s.other_left != 0U;

                    value[u] = m3_chain_op4(s.op,
                                            left ? other[u][k] : value[u],
                                            left ? value[u] : other[u][k]);
                }
                if (dtype == M3N_F32) {
                    if (g < a.groups) {
                        m3_stream_store((uint4 *)s.out + g, value[u]);
                    }
                    continue;
                }
                const uint2 raw = m3_narrow4_bits(value[u], dtype);

                if (g < a.groups) {
                    m3_stream_store((uint2 *)s.out + g, raw);
                }
                value[u] = m3_widen4_bits(raw, dtype);
            }
        }
    }
    /* Tail: the last count % 4 elements. */
    if (blockIdx.x == 0U && threadIdx.x < a.count - a.groups * 4U) {
        const uint32_t f = a.groups * 4U + threadIdx.x;
        uint32_t v = m3_operand_element<DT>(a.value, f);

#pragma unroll
        for (int k = 0; k < STEPS; ++k) {
            const m3_chain_step &s = a.steps[k];
            const uint32_t dtype = DT == kAnyDtype ? s.out_dtype : DT;

            if (s.op != kChainCast) {
                const uint32_t o = m3_operand_element<DT>(s.other, f);
                const bool left = s.other_left != 0U;

                v = m3_binary_f32_bits(s.op, left ? o : v, left ? v : o);
            }
            const uint32_t raw = m3_store_from_f32_bits(v, dtype);

            if (dtype == M3N_F32) {
                *(uint32_t *)(s.out + (uint64_t)f * 4U) = raw;
            } else {
                *(uint16_t *)(s.out + (uint64_t)f * 2U) = (uint16_t)raw;
            }
            v = m3_load_as_f32_bits(raw, dtype);
        }
    }
}

struct m3_bin_general_args {
    const uint8_t *left;
    const uint8_t *right;
    uint8_t *out;
    uint32_t left_dtype;
    uint32_t right_dtype;
    uint32_t out_dtype;
    uint32_t rank;
    uint64_t count;
    uint64_t shape[M3_HIP_MAX_RANK];
    int64_t left_strides[M3_HIP_MAX_RANK];
    int64_t right_strides[M3_HIP_MAX_RANK];
    m3_hip_gate list_gate;
};

template <int OP>
__global__ __launch_bounds__(256) void m3_binary_general_kernel(
    m3_bin_general_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint32_t out_size = a.out_dtype == M3N_F32 ? 4U : 2U;

    for (uint64_t f = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
         f < a.count; f += stride) {
        uint64_t rest = f;
        int64_t lo = 0;
        int64_t ro = 0;

        for (int axis = (int)a.rank - 1; axis >= 0; --axis) {
            uint64_t dim = a.shape[axis];
            uint64_t q = rest / dim;
            uint64_t c = rest - q * dim;

            rest = q;
            lo += (int64_t)c * a.left_strides[axis];
            ro += (int64_t)c * a.right_strides[axis];
        }
        uint32_t x = m3_load_as_f32_bits(m3_load_raw(a.left + lo,
                                                     a.left_dtype),
                                         a.left_dtype);
        uint32_t y = m3_load_as_f32_bits(m3_load_raw(a.right + ro,
                                                     a.right_dtype),
                                         a.right_dtype);
        uint32_t raw =
            m3_store_from_f32_bits(m3_binary_f32_bits(OP, x, y), a.out_dtype);

        if (out_size == 4U) {
            *(uint32_t *)(a.out + f * 4U) = raw;
        } else {
            *(uint16_t *)(a.out + f * 2U) = (uint16_t)raw;
        }
    }
}

/* Classifies operand k of `plan` (strides in bytes, element size esize). */
bool m3_classify_operand(const m3_index_plan &plan, uint32_t k,
                         const m3_hip_view *view, m3_bin_operand *operand)
{
    const int64_t esize = (int64_t)m3_dtype_bytes(view->dtype);
    const uint8_t *base = (const uint8_t *)view->base + view->byte_offset;
    uint64_t contiguous = 1U; /* output-layout element stride of an axis */
    uint64_t expected[M3_HIP_MAX_RANK];
    int live = -1;
    uint32_t live_count = 0U;
    bool full = true;

    for (int axis = (int)plan.rank - 1; axis >= 0; --axis) {
        expected[axis] = contiguous;
        contiguous *= plan.shape[axis];
    }
    for (uint32_t axis = 0U; axis < plan.rank; ++axis) {
        int64_t s = plan.strides[k][axis];

        if (s != (int64_t)expected[axis] * esize) {
            full = false;
        }
        if (s != 0) {
            live = (int)axis;
            live_count += 1U;
        }
    }
    std::memset(operand, 0, sizeof(*operand));
    operand->base = base;
    operand->dtype = view->dtype;
    if (full && contiguous < (1ULL << 32U)) {
        operand->mode = M3_BIN_FULL;
        return true;
    }
    if (live_count == 0U) {
        operand->mode = M3_BIN_SCALAR;
        return true;
    }
    if (live_count != 1U || plan.strides[k][live] != esize ||
        contiguous >= (1ULL << 32U)) {
        return false;
    }
    operand->inner = m3_fast_div_make((uint32_t)expected[live]);
    operand->period = m3_fast_div_make((uint32_t)plan.shape[live]);
    operand->mode = M3_BIN_PERIODIC;
    if (expected[live] == 1U && plan.shape[live] >= 4U) {
        operand->mode = plan.shape[live] % 4U == 0U ? M3_BIN_TRAIL
                                                    : M3_BIN_TRAIL_CUT;
    } else if (expected[live] >= 4U) {
        operand->mode = expected[live] % 4U == 0U ? M3_BIN_ROW
                                                  : M3_BIN_ROW_CUT;
    }
    return true;
}

/* The kind of an F32 operand. */
uint32_t m3_kind_of(const m3_bin_operand &o)
{
    return o.mode == M3_BIN_FULL    ? M3_KIND_FULL
           : o.mode == M3_BIN_TRAIL ? M3_KIND_TRAIL
           : o.mode == M3_BIN_ROW || o.mode == M3_BIN_SCALAR ? M3_KIND_ONE
                                                             : M3_KIND_ANY;
}

/* True for an operand that gives a group one element or one 16-byte
 * aligned vector. */
bool m3_operand_whole(const m3_bin_operand &o)
{
    const uint32_t kind = m3_kind_of(o);

    return kind == M3_KIND_ONE ||
           (kind != M3_KIND_ANY && ((uintptr_t)o.base & 15U) == 0U);
}

/* How many elements (m3_least_elements) operands that go by their modes want
 * for the vector kernel; below, one element per lane is faster, contiguous or
 * not. General against vector kernel, us: F32 in rows of 7 times a column
 * 100,000 3.2 and 3.8, 300,000 3.6 and 3.9, 400,000 4.1 and 4.0; BF16 times
 * BF16 20,000 3.0 and 4.0, 300,000 3.4 and 4.1, 524,288 3.8 and 4.2, 650,000
 * 4.4 and 4.3; F16 in rows of 3 times a column 20,000 3.4 and 5.6, 650,000
 * 5.4 and 5.8, 800,000 6.1 and 5.9. */
uint32_t m3_any_quarters(const m3_bin_vec_args &vec, bool f32)
{
    const bool cut = m3_kind_of(vec.left) == M3_KIND_ANY ||
                     m3_kind_of(vec.right) == M3_KIND_ANY;

    return f32 ? 3U : cut ? 6U : 4U;
}

/* The F32 kernels of one pair of kinds: streamed (hold_ticks null) or held. */
typedef void (*m3_binary_launcher)(dim3, hipStream_t, hipEvent_t, hipEvent_t,
                                   const m3_bin_vec_args &, const uint32_t *);

template <int OP, uint32_t LEFT, uint32_t RIGHT>
void m3_launch_kinds(dim3 grid, hipStream_t stream, hipEvent_t start,
                     hipEvent_t stop, const m3_bin_vec_args &args,
                     const uint32_t *hold_ticks)
{
    if (hold_ticks != nullptr) {
        hipExtLaunchKernelGGL(
            (m3_binary_held_kernel<OP, kHeldGroups, LEFT, RIGHT>), grid,
            dim3(kThreads), 0, stream, start, stop, 0U, args, *hold_ticks);
        return;
    }
    hipExtLaunchKernelGGL((m3_binary_vec_kernel<OP, M3N_F32, LEFT, RIGHT>),
                          grid, dim3(kThreads), 0, stream, start, stop, 0U,
                          args);
}

/* [left kind][right kind] */
template <int OP>
m3_binary_launcher m3_binary_launcher_of(uint32_t left, uint32_t right)
{
    static const m3_binary_launcher launchers[3][3] = {
        {&m3_launch_kinds<OP, M3_KIND_FULL, M3_KIND_FULL>,
         &m3_launch_kinds<OP, M3_KIND_FULL, M3_KIND_TRAIL>,
         &m3_launch_kinds<OP, M3_KIND_FULL, M3_KIND_ONE>},
        {&m3_launch_kinds<OP, M3_KIND_TRAIL, M3_KIND_FULL>,
         &m3_launch_kinds<OP, M3_KIND_TRAIL, M3_KIND_TRAIL>,
         &m3_launch_kinds<OP, M3_KIND_TRAIL, M3_KIND_ONE>},
        {&m3_launch_kinds<OP, M3_KIND_ONE, M3_KIND_FULL>,
         &m3_launch_kinds<OP, M3_KIND_ONE, M3_KIND_TRAIL>,
         &m3_launch_kinds<OP, M3_KIND_ONE, M3_KIND_ONE>}};

    return launchers[left][right];
}

template <int OP>
int m3_launch_binary_op(m3_hip_device *device, const m3_hip_view *left,
                        const m3_hip_view *right, const m3_hip_view *output,
                        char *message, size_t capacity)
{
    static const char *const names[4] = {"m3_binary_add", "m3_binary_mul",
                                         "m3_binary_sub", "m3_binary_div"};
    const m3_hip_view *operands[3] = {output, left, right};
    m3_index_plan plan;
    m3_bin_vec_args vec;
    uint8_t *out = (uint8_t *)output->base + output->byte_offset;

    m3_plan_index_space(output, operands, 3U, &plan);
    std::memset(&vec, 0, sizeof(vec));
    vec.list_gate = device->gate;
    if (output->element_count < (1ULL << 32U) &&
        m3_classify_operand(plan, 1U, left, &vec.left) &&
        m3_classify_operand(plan, 2U, right, &vec.right)) {
        bool f32 = left->dtype == M3N_F32 && right->dtype == M3N_F32 &&
                   output->dtype == M3N_F32;

        vec.out = out;
        vec.out_dtype = output->dtype;
        vec.count = (uint32_t)output->element_count;
        vec.groups = vec.count / 4U;
        uint32_t blocks = m3_grid_blocks(device,
                                         (uint64_t)vec.groups == 0U
                                             ? 1U
                                             : vec.groups,
                                         kThreads * kUnroll, 16U);

        const uint64_t held =
            ((uint64_t)vec.groups + kThreads * kHeldGroups - 1U) /
            (kThreads * kHeldGroups);
        /* held only when its workgroups fill at least half of what the
         * device holds at once (a smaller tensor in few workgroups of
         * twelve groups per lane runs slower than streamed: 2 MB MUL, 9.0
         * against 4.5 us) and fit in it */
        const uint64_t slots =
            (uint64_t)device->compute_units * kHeldBlocksPerCu;
        const bool hold = f32 && device->wall_clock_khz != 0U &&
                          2U * held >= slots && held <= slots &&
                          m3_operand_whole(vec.left) &&
                          m3_operand_whole(vec.right);
        /* the full operands' bytes (broadcast ones are read from cache) */
        const double read_bytes =
            4.0 * (double)vec.count *
            (double)((vec.left.mode == M3_BIN_FULL) +
                     (vec.right.mode == M3_BIN_FULL));
        const uint32_t hold_ticks = (uint32_t)(
            kBinaryHoldFactor * read_bytes / 8.0e6 *
            (double)device->wall_clock_khz / 1000.0);
        const uint32_t left_kind = f32 ? m3_kind_of(vec.left) : M3_KIND_ANY;
        const uint32_t right_kind = f32 ? m3_kind_of(vec.right) : M3_KIND_ANY;

        if (left_kind != M3_KIND_ANY && right_kind != M3_KIND_ANY) {
            const m3_binary_launcher launcher =
                m3_binary_launcher_of<OP>(left_kind, right_kind);

            for (m3_bin_operand *o : {&vec.left, &vec.right}) {
                if (o->mode == M3_BIN_SCALAR) {
                    o->inner = m3_fast_div_make(1U);
                    o->period = m3_fast_div_make(1U);
                }
            }
            return m3_hip_launch(
                device, names[OP],
                [&](hipEvent_t start, hipEvent_t stop) {
                    launcher(dim3(hold ? (uint32_t)held : blocks),
                             device->stream, start, stop, vec,
                             hold ? &hold_ticks : nullptr);
                },
                message, capacity);
        }
        if (vec.count >= m3_least_elements(
                             device, m3_any_quarters(vec, f32))) {
            return m3_hip_launch(
                device, names[OP],
                [&](hipEvent_t start, hipEvent_t stop) {
                    if (f32) {
                        hipExtLaunchKernelGGL(
                            (m3_binary_vec_kernel<OP, M3N_F32, M3_KIND_ANY,
                                                  M3_KIND_ANY>),
                            dim3(blocks), dim3(kThreads), 0, device->stream,
                            start, stop, 0U, vec);
                    } else {
                        hipExtLaunchKernelGGL(
                            (m3_binary_vec_kernel<OP, kAnyDtype, M3_KIND_ANY,
                                                  M3_KIND_ANY>),
                            dim3(blocks), dim3(kThreads), 0, device->stream,
                            start, stop, 0U, vec);
                    }
                },
                message, capacity);
        }
    }

    m3_bin_general_args general;

    std::memset(&general, 0, sizeof(general));
    general.list_gate = device->gate;
    general.left = (const uint8_t *)left->base + left->byte_offset;
    general.right = (const uint8_t *)right->base + right->byte_offset;
    general.out = out;
    general.left_dtype = left->dtype;
    general.right_dtype = right->dtype;
    general.out_dtype = output->dtype;
    general.rank = plan.rank;
    general.count = output->element_count;
    for (uint32_t axis = 0U; axis < plan.rank; ++axis) {
        general.shape[axis] = plan.shape[axis];
        general.left_strides[axis] = plan.strides[1][axis];
        general.right_strides[axis] = plan.strides[2][axis];
    }
    uint32_t blocks = m3_grid_blocks(device, general.count, 256U, 16U);

    return m3_hip_launch(
        device, names[OP],
        [&](hipEvent_t start, hipEvent_t stop) {
            hipExtLaunchKernelGGL((m3_binary_general_kernel<OP>), dim3(blocks),
                                  dim3(256), 0, device->stream, start, stop,
                                  0U, general);
        },
        message, capacity);
}

typedef void (*m3_chain_launcher)(dim3, hipStream_t, hipEvent_t, hipEvent_t,
                                  const m3_chain_args &);

constexpr int kChainUnroll = 2; /* groups in flight per lane */
constexpr uint32_t kChainBlocksPerCu = 1024U; /* one tile per workgroup */

template <int STEPS, uint32_t DT>
void m3_launch_chain(dim3 grid, hipStream_t stream, hipEvent_t start,
                     hipEvent_t stop, const m3_chain_args &args)
{
    hipExtLaunchKernelGGL((m3_chain_kernel<STEPS, DT, kChainUnroll>),
                          grid, dim3(kThreads), 0, stream, start, stop, 0U,
                          args);
}

bool m3_chain_is_float(const m3_hip_view *view)
{
    return m3_view_is_valid(view) && view->dtype != M3_HIP_I32;
}

/* True when the two views are of one shape. */
bool m3_chain_same_shape(const m3_hip_view *a, const m3_hip_view *b)
{
    return a->rank == b->rank && m3_view_broadcasts_to(a, b) &&
           a->element_count == b->element_count;
}

/* Fills the kernel's arguments from a chain of binary operations and casts;
 * false when the chain kernel does not take it: an operand that does not
 * classify, no elements, 2^32 of them or more, or an output that overlaps what
 * another operation reads or writes (the launch would no longer equal the
 * operations in order). */
bool m3_chain_plan(const m3_hip_chain_command *commands, uint32_t count,
                   m3_chain_args *args)
{
    const m3_hip_view *space = &commands[0].output;

    /* before any divisor is formed from an extent: none of them is zero */
    if (space->element_count == 0U ||
        space->element_count >= (1ULL << 32U)) {
        return false;
    }
    for (uint32_t k = 0U; k < count; ++k) {
        const m3_hip_chain_command &c = commands[k];
        const bool cast = c.kind == M3_HIP_CHAIN_CAST;
        /* the operand that is not the chain's value (none of a cast) */
        const bool other_left = k != 0U && !cast && c.link != 0U;
        const m3_hip_view *value = other_left ? &c.right : &c.left;
        const m3_hip_view *other = other_left ? &c.left : &c.right;
        m3_chain_step *step = &args->steps[k];

        if ((!cast && (c.kind != M3_HIP_CHAIN_BINARY || c.op > M3_HIP_DIV)) ||
            !m3_chain_is_float(&c.output) || !m3_chain_is_float(value) ||
            (!cast && !m3_chain_is_float(other)) ||
            !m3_view_is_contiguous(&c.output) ||
            !m3_chain_same_shape(&c.output, space)) {
            return false;
        }
        for (uint32_t i = 0U; i < k; ++i) {
            if (m3_views_overlap(&commands[i].output, &c.output) ||
                (!cast && m3_views_overlap(&commands[i].output, other))) {
                return false;
            }
        }
        /* what this and earlier operations load, against this output */
        for (uint32_t i = 0U; i <= k; ++i) {
            const m3_hip_chain_command &e = commands[i];
            const bool e_cast = e.kind == M3_HIP_CHAIN_CAST;
            const bool e_left = i == 0U || (!e_cast && e.link != 0U);
            const bool e_right = !e_cast && (i == 0U || e.link == 0U);

            if ((e_left && m3_views_overlap(&e.left, &c.output)) ||
                (e_right && m3_views_overlap(&e.right, &c.output))) {
                return false;
            }
        }
        const m3_hip_view *operands[3] = {&c.output, value,
                                          cast ? value : other};
        m3_index_plan plan;

        if ((k == 0U && !m3_view_broadcasts_to(value, &c.output)) ||
            (!cast && !m3_view_broadcasts_to(other, &c.output))) {
            return false;
        }
        m3_plan_index_space(&c.output, operands, 3U, &plan);
        if ((k == 0U && !m3_classify_operand(plan, 1U, value, &args->value)) ||
            (!cast && !m3_classify_operand(plan, 2U, other, &step->other))) {
            return false;
        }
        step->out = (uint8_t *)c.output.base + c.output.byte_offset;
        step->out_dtype = c.output.dtype;
        step->op = cast ? kChainCast : c.op;
        step->other_left = other_left ? 1U : 0U;
    }
    args->count = (uint32_t)space->element_count;
    args->groups = args->count / 4U;
    return true;
}

} // namespace

extern "C" int m3_hip_launch_chain(m3_hip_device *device,
                                   const m3_hip_chain_command *commands,
                                   uint32_t count, int *taken, char *message,
                                   size_t capacity)
{
    /* [operations - 2][the one dtype throughout, or 3: several] */
    static const m3_chain_launcher launchers[M3_HIP_MAX_CHAIN - 1][4] = {
        {&m3_launch_chain<2, M3N_F32>, &m3_launch_chain<2, M3N_F16>,
         &m3_launch_chain<2, M3N_BF16>, &m3_launch_chain<2, kAnyDtype>},
        {&m3_launch_chain<3, M3N_F32>, &m3_launch_chain<3, M3N_F16>,
         &m3_launch_chain<3, M3N_BF16>, &m3_launch_chain<3, kAnyDtype>}};
    m3_chain_args args;
    uint32_t dtype;

    if (device == nullptr || commands == nullptr || taken == nullptr ||
        count < 2U || count > M3_HIP_MAX_CHAIN) {
        return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                           "chain launch arguments are malformed");
    }
    *taken = 0;
    if (count == 2U && commands[0].kind == M3_HIP_CHAIN_SNAKE1D &&
        commands[1].kind == M3_HIP_CHAIN_TANH) {
        return m3_snake1d_tanh(device, commands, taken, message, capacity);
    }
    std::memset(&args, 0, sizeof(args));
    if (!m3_chain_plan(commands, count, &args)) {
        return M3_HIP_OK;
    }
    args.list_gate = device->gate;
    dtype = args.value.dtype;
    for (uint32_t k = 0U; k < count; ++k) {
        if (args.steps[k].out_dtype != dtype ||
            (args.steps[k].op != kChainCast &&
             args.steps[k].other.dtype != dtype)) {
            dtype = 3U;
            break;
        }
    }
    const dim3 grid(m3_grid_blocks(device,
                                   args.groups == 0U ? 1U : args.groups,
                                   kThreads * kChainUnroll,
                                   kChainBlocksPerCu));
    const m3_chain_launcher launcher = launchers[count - 2U][dtype];

    *taken = 1;
    return m3_hip_launch(
        device, "m3_chain",
        [&](hipEvent_t start, hipEvent_t stop) {
            launcher(grid, device->stream, start, stop, args);
        },
        message, capacity);
}

extern "C" int m3_hip_launch_binary(m3_hip_device *device, uint32_t op,
                                    const m3_hip_view *left,
                                    const m3_hip_view *right,
                                    const m3_hip_view *output, char *message,
                                    size_t capacity)
{
    if (device == nullptr || op > M3_HIP_DIV || !m3_view_is_valid(left) ||
        !m3_view_is_valid(right) || !m3_view_is_valid(output) ||
        left->dtype == M3_HIP_I32 || right->dtype == M3_HIP_I32 ||
        output->dtype == M3_HIP_I32 || !m3_view_is_contiguous(output) ||
        !m3_view_broadcasts_to(left, output) ||
        !m3_view_broadcasts_to(right, output)) {
        return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                           "binary launch arguments are malformed");
    }
    if (output->element_count == 0U) {
        return M3_HIP_OK;
    }
    switch (op) {
    case M3_HIP_ADD:
        return m3_launch_binary_op<M3N_ADD>(device, left, right, output,
                                            message, capacity);
    case M3_HIP_MUL:
        return m3_launch_binary_op<M3N_MUL>(device, left, right, output,
                                            message, capacity);
    case M3_HIP_SUB:
        return m3_launch_binary_op<M3N_SUB>(device, left, right, output,
                                            message, capacity);
    default:
        return m3_launch_binary_op<M3N_DIV>(device, left, right, output,
                                            message, capacity);
    }
}
