/*
 * m3_hip_activation.hip - TANH and GATED_SILU for gfx950, bit-exact with
 * the CPU provider of the reference.
 *
 * Reference semantics:
 *   TANH       (src/m3_op_execute_basic.c:217-229) out = tanhf(in), F32;
 *              every element is m3_tanhf_uniform, the C library's tanhf
 *              restated bit for bit (m3_libm.h).
 *   GATED_SILU (src/m3_op_execute_basic.c:104-122) out = round_gate(gate /
 *              (1 + expf(-gate))) * up; m3_activation.h states it with
 *              the host's NaN bits.
 *
 * Both are elementwise and bound by HBM traffic at large sizes: TANH moves
 * 8 bytes per F32 element, GATED_SILU 12 (F32) or 6 (16-bit operands).
 * The vector kernels take contiguous operands of one dtype at any
 * alignment, and for GATED_SILU also a gate and up whose rows are
 * contiguous and evenly spaced (both halves of one projection), of about as
 * many elements as the device has lanes or more (m3_least_elements): a lane
 * handles four consecutive elements per group, kUnroll groups in flight,
 * loads and stores streaming (every element is read and written once). The
 * last count % 4 elements are done by the first lanes of block 0. Smaller
 * tensors and every other layout (strided inputs, mixed dtypes for
 * GATED_SILU) run the general kernel over the coalesced index space with
 * per-element offsets.
 *
 * GATED_SILU's NaN rule costs a recomputation only in a wave where some
 * product is NaN: the plain arithmetic gives the host's bits for every
 * non-NaN result, and m3_gated_silu_bits gives them for all.
 *
 * All-BF16 GATED_SILU looks its activation up in a 16 KB table that each
 * device builds once (m3_gated_silu_bf16_kernel): a BF16 gate has only
 * 65,536 values, and the rounded activation depends on the gate alone.
 * That takes the kernel from 52 VALU instructions per element, clock-bound,
 * to 25, bound by HBM.
 */
#include "m3_activation.h"
#include "m3_hip_internal.h"
#include "m3_libm.h"

#include <algorithm>
#include <cstring>

namespace {

constexpr uint32_t kThreads = 256U;
constexpr uint32_t kUnroll = 4U;
/* TANH's groups per lane: with ~100 instructions per element, two groups
 * in flight already cover the load latency, and the smaller tile lets the
 * dispatcher spread the work more evenly (3% faster than four, measured
 * alternating in one process on x[2,1536,65536]). */
constexpr uint32_t kTanhUnroll = 2U;
/* Grid cap of the vector kernels: 1,024 workgroups per CU, so every
 * tensor below 2^30 elements runs as one workgroup per tile (1,024 groups
 * of four elements) and the hardware dispatcher, not the grid-stride
 * loop, spreads the tiles. Measured against 16 per CU, alternating in one
 * process: GATED_SILU [16384, 3072] 94.5 against 100.5 us in F32 and 68.5
 * against 72.3 us in BF16; TANH x[2,1536,65536] 484 against 506 us. */
constexpr uint32_t kBlocksPerCu = 1024U;
/* general against vector kernel: 20,000 elements 2.9 and 3.4 us, 100,000 3.0
 * and 3.6, 300,000 3.4 and 3.7, 600,000 4.2 and 4.0 */
constexpr uint32_t kTanhQuarters = 3U;

/* Stores four F32 results (as bits) rounded to dtype D at group g. */
template <uint32_t D>
__device__ __forceinline__ void m3_store4(uint8_t *base, uint32_t g,
                                          const uint32_t r[4])
{
    if (D == M3N_F32) {
        m3_stream_store((uint4 *)base + g, make_uint4(r[0], r[1], r[2], r[3]));
    } else {
        uint32_t lo = m3_store_from_f32_bits(r[0], D) |
                      (m3_store_from_f32_bits(r[1], D) << 16U);
        uint32_t hi = m3_store_from_f32_bits(r[2], D) |
                      (m3_store_from_f32_bits(r[3], D) << 16U);

        m3_stream_store((uint2 *)base + g, make_uint2(lo, hi));
    }
}

__device__ __forceinline__ uint32_t m3_load_element(const uint8_t *p,
                                                    uint32_t dtype)
{
    uint32_t raw = dtype == M3N_F32 ? *(const uint32_t *)p
                                    : (uint32_t) * (const uint16_t *)p;

    return m3_load_as_f32_bits(raw, dtype);
}

__device__ __forceinline__ void m3_store_element(uint8_t *p, uint32_t dtype,
                                                 uint32_t bits)
{
    uint32_t raw = m3_store_from_f32_bits(bits, dtype);

    if (dtype == M3N_F32) {
        *(uint32_t *)p = raw;
    } else {
        *(uint16_t *)p = (uint16_t)raw;
    }
}

/* ---- TANH ---------------------------------------------------------------- */

struct m3_tanh_vec_args {
    const uint8_t *input;
    uint8_t *output;
    uint32_t groups; /* count / 4 */
    uint32_t tail;   /* count % 4 */
    m3_hip_gate list_gate;
};

__global__ __launch_bounds__(256) void m3_tanh_vec_kernel(m3_tanh_vec_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint32_t step = gridDim.x * kThreads * kTanhUnroll;

    for (uint32_t first = blockIdx.x * kThreads * kTanhUnroll + threadIdx.x;
         first < a.groups; first += step) {
        float4 x[kTanhUnroll];

        /* unconditional loads (groups past the end re-read the last one)
         * so that all of them are in flight before the first use */
#pragma unroll
        for (uint32_t u = 0U; u < kTanhUnroll; ++u) {
            x[u] = m3_stream_load((const float4 *)a.input +
                                  min(first + u * kThreads, a.groups - 1U));
        }
#pragma unroll
        for (uint32_t u = 0U; u < kTanhUnroll; ++u) {
            uint32_t g = first + u * kThreads;

            if (g < a.groups) {
                m3_stream_store((float4 *)a.output + g,
                                make_float4(m3_tanhf_uniform(x[u].x),
                                            m3_tanhf_uniform(x[u].y),
                                            m3_tanhf_uniform(x[u].z),
                                            m3_tanhf_uniform(x[u].w)));
            }
        }
    }
    if (blockIdx.x == 0U && threadIdx.x < a.tail) {
        const uint64_t e = 4ULL * a.groups + threadIdx.x;
        float x = m3_bits_f32(*(const uint32_t *)(a.input + 4ULL * e));

        *(uint32_t *)(a.output + 4ULL * e) = m3_f32_bits(m3_tanhf_uniform(x));
    }
}

/* Coalesced index space: operand 0 is the contiguous output, 1 and 2 the
 * inputs (byte strides per axis). */
struct m3_activation_general_args {
    const uint8_t *inputs[2];
    uint8_t *output;
    uint32_t dtypes[3]; /* output, input 0, input 1 */
    uint32_t rank;
    uint64_t count;
    uint64_t shape[M3_HIP_MAX_RANK];
    int64_t strides[2][M3_HIP_MAX_RANK];
    m3_hip_gate list_gate;
};

__device__ __forceinline__ void m3_general_offsets(
    const m3_activation_general_args &a, uint64_t f, int64_t offsets[2])
{
    uint64_t rest = f;

    offsets[0] = 0;
    offsets[1] = 0;
    for (int axis = (int)a.rank - 1; axis >= 0; --axis) {
        uint64_t dim = a.shape[axis];
        uint64_t q = rest / dim;
        int64_t c = (int64_t)(rest - q * dim);

        offsets[0] += c * a.strides[0][axis];
        offsets[1] += c * a.strides[1][axis];
        rest = q;
    }
}

__global__ __launch_bounds__(256) void m3_tanh_general_kernel(
    m3_activation_general_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;

    for (uint64_t f = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
         f < a.count; f += step) {
        int64_t offsets[2];

        m3_general_offsets(a, f, offsets);
        float x = m3_bits_f32(*(const uint32_t *)(a.inputs[0] + offsets[0]));

        *(uint32_t *)(a.output + 4ULL * f) = m3_f32_bits(m3_tanhf_uniform(x));
    }
}

/* ---- GATED_SILU ---------------------------------------------------------- */

struct m3_silu_vec_args {
    const uint8_t *gate;
    const uint8_t *up;
    uint8_t *output;
    uint32_t groups;
    uint32_t tail;
    /* rows of `width` (at least 4) elements whose starts are this many
     * elements apart; unused when gate and up are contiguous */
    m3_fast_div width;
    uint64_t gate_pitch;
    uint64_t up_pitch;
    m3_hip_gate list_gate;
};

/* Element `e` of an operand in rows of a.width elements, `pitch` apart. */
__device__ __forceinline__ uint64_t m3_silu_row_offset(
    const m3_silu_vec_args &a, uint64_t pitch, uint32_t e)
{
    const uint32_t row = m3_fast_div_q(a.width, e);

    return row * pitch + (e - row * a.width.divisor);
}

/* Four consecutive elements of dtype D at group g, raw (zero-extended);
 * ROWS: from rows, four elements that a row's end cuts one by one. Packed
 * [3001, 2 x 3072] took 47 (BF16), 46 (F32) and 57 us (F16) in the general
 * kernel, one element per lane, and takes 18.8, 20 and 32 in this one. */
template <uint32_t D, bool ROWS>
__device__ __forceinline__ uint4 m3_silu_load4(const m3_silu_vec_args &a,
                                               const uint8_t *base,
                                               uint64_t pitch, uint32_t g)
{
    constexpr uint32_t size = D == M3N_F32 ? 4U : 2U;
    const uint32_t e = 4U * g;
    uint64_t offset = e;

    if (ROWS) {
        offset = m3_silu_row_offset(a, pitch, e);
        if (m3_fast_div_q(a.width, e) != m3_fast_div_q(a.width, e + 3U)) {
            uint32_t x[4];

#pragma unroll
            for (uint32_t i = 0U; i < 4U; ++i) {
                const uint8_t *p =
                    base + m3_silu_row_offset(a, pitch, e + i) * size;

                x[i] = size == 4U ? *(const uint32_t *)p
                                  : (uint32_t) * (const uint16_t *)p;
            }
            return make_uint4(x[0], x[1], x[2], x[3]);
        }
    }
    if (size == 4U) {
        return m3_stream_load((const uint4 *)(base + offset * 4U));
    }
    const uint2 h = m3_stream_load((const uint2 *)(base + offset * 2U));

    return make_uint4(h.x & 0xffffU, h.x >> 16U, h.y & 0xffffU, h.y >> 16U);
}

/* Four GATED_SILU elements with a gate of dtype D, as F32 bits; `table`
 * is the expf table in LDS. */
template <uint32_t D>
__device__ __forceinline__ void m3_silu4(const float g[4], const float u[4],
                                         const uint64_t *table, uint32_t r[4])
{
    float p[4];

#pragma unroll
    for (uint32_t k = 0U; k < 4U; ++k) {
        float activation = m3_silu_quotient_fast(g[k], table);

        if (D == M3N_BF16) {
            activation = m3_bits_f32(
                m3_round_through_bf16_finite(m3_f32_bits(activation)));
        } else if (D == M3N_F16) {
            activation = m3_bits_f32(
                m3_round_through_bits(m3_f32_bits(activation), D));
        }
        p[k] = activation * u[k];
    }
    /* a NaN activation makes its product NaN, so one test covers both */
    if ((__ballot(p[0] != p[0]) | __ballot(p[1] != p[1]) |
         __ballot(p[2] != p[2]) | __ballot(p[3] != p[3])) != 0U) {
#pragma unroll
        for (uint32_t k = 0U; k < 4U; ++k) {
            p[k] = m3_bits_f32(m3_gated_silu_bits(g[k], u[k], D));
        }
    }
#pragma unroll
    for (uint32_t k = 0U; k < 4U; ++k) {
        r[k] = m3_f32_bits(p[k]);
    }
}

/* GATED_SILU BF16 through a table of activations. A BF16 gate has 65,536
 * bit patterns, and the activation, rounded through BF16, depends on the
 * gate alone; the table holds it for every gate of magnitude in
 * [2^-25, 2^7) (exponent fields 102-133, 32 binades of 128 values, both
 * signs: 8,192 entries, 16 KB), which covers every gate that is not tiny,
 * huge, infinite or NaN. The entries are the bits m3_gated_silu_bits gives
 * with up = 1 (exact: the product of a finite BF16 activation and 1), built
 * on the device when it is opened. Each workgroup copies the table into
 * LDS; an element then costs one LDS read instead of the ~35 instructions
 * of expf and the division. Gates outside the table take the arithmetic
 * of m3_silu4 in the waves where a lane has one, and NaN products the
 * exact recomputation, as in m3_gated_silu_vec_kernel. */
constexpr uint32_t kSiluTableFirstField = 102U; /* exponent field of 2^-25 */
constexpr uint32_t kSiluTableSpan = 32U << 7U;  /* entries per sign */
constexpr uint32_t kSiluTableEntries = 2U * kSiluTableSpan;

/* The BF16 bits of table entry i: bit 12 is the sign, the rest counts up
 * from the first exponent field. */
__host__ __device__ inline uint32_t m3_silu_table_gate(uint32_t i)
{
    return ((i & kSiluTableSpan) << 3U) |
           ((kSiluTableFirstField << 7U) + (i & (kSiluTableSpan - 1U)));
}

__global__ __launch_bounds__(256) void m3_silu_table_build_kernel(
    uint16_t *table)
{
    const uint32_t i = blockIdx.x * 256U + threadIdx.x;

    if (i < kSiluTableEntries) {
        const float gate = m3_bits_f32(m3_silu_table_gate(i) << 16U);

        table[i] = (uint16_t)(m3_gated_silu_bits(gate, 1.0F, M3N_BF16) >>
                              16U);
    }
}

/* The activation of BF16 gate bits `raw` as F32 bits from the LDS table;
 * *miss is set (and 0 returned) for a gate outside it. */
__device__ __forceinline__ uint32_t m3_silu_table_lookup(
    uint32_t raw, const uint16_t *table, bool *miss)
{
    const uint32_t index = (raw & 0x7fffU) - (kSiluTableFirstField << 7U);
    const bool inside = index < kSiluTableSpan;

    *miss = !inside;
    return inside ? (uint32_t)table[index | ((raw >> 3U) & kSiluTableSpan)]
                        << 16U
                  : 0U;
}

template <bool ROWS>
__global__ __launch_bounds__(256) void m3_gated_silu_bf16_kernel(
    m3_silu_vec_args a, const uint4 *source)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint32_t step = gridDim.x * kThreads * kUnroll;
    __shared__ uint16_t table[kSiluTableEntries];
    __shared__ uint64_t exp_table[32];

    for (uint32_t i = threadIdx.x; i < kSiluTableEntries / 8U; i += kThreads) {
        ((uint4 *)table)[i] = source[i];
    }
    if (threadIdx.x < 32U) {
        exp_table[threadIdx.x] = m3_expf_table[threadIdx.x];
    }
    __syncthreads();
    for (uint32_t first = blockIdx.x * kThreads * kUnroll + threadIdx.x;
         first < a.groups; first += step) {
        uint4 gate[kUnroll];
        uint4 up[kUnroll];

        /* unconditional loads (groups past the end re-read the last one)
         * so that all of them are in flight before the first use */
#pragma unroll
        for (uint32_t k = 0U; k < kUnroll; ++k) {
            const uint32_t index = min(first + k * kThreads, a.groups - 1U);

            gate[k] = m3_silu_load4<M3N_BF16, ROWS>(a, a.gate, a.gate_pitch,
                                                    index);
            up[k] = m3_silu_load4<M3N_BF16, ROWS>(a, a.up, a.up_pitch, index);
        }
#pragma unroll
        for (uint32_t k = 0U; k < kUnroll; ++k) {
            const uint32_t index = first + k * kThreads;

            if (index < a.groups) {
                const uint32_t raw[4] = {gate[k].x, gate[k].y, gate[k].z,
                                         gate[k].w};
                const float u[4] = {m3_bits_f32(up[k].x << 16U),
                                    m3_bits_f32(up[k].y << 16U),
                                    m3_bits_f32(up[k].z << 16U),
                                    m3_bits_f32(up[k].w << 16U)};
                uint32_t activation[4];
                bool miss[4];
                float p[4];
                uint32_t r[4];

#pragma unroll
                for (uint32_t e = 0U; e < 4U; ++e) {
                    activation[e] = m3_silu_table_lookup(raw[e], table,
                                                         &miss[e]);
                }
                if ((__ballot(miss[0]) | __ballot(miss[1]) |
                     __ballot(miss[2]) | __ballot(miss[3])) != 0U) {
#pragma unroll
                    for (uint32_t e = 0U; e < 4U; ++e) {
                        if (miss[e]) {
                            activation[e] = m3_round_through_bf16_finite(
                                m3_f32_bits(m3_silu_quotient_fast(
                                    m3_bits_f32(raw[e] << 16U), exp_table)));
                        }
                    }
                }
#pragma unroll
                for (uint32_t e = 0U; e < 4U; ++e) {
                    p[e] = m3_bits_f32(activation[e]) * u[e];
                }
                /* a NaN activation makes its product NaN, so one test
                 * covers both */
                if ((__ballot(p[0] != p[0]) | __ballot(p[1] != p[1]) |
                     __ballot(p[2] != p[2]) | __ballot(p[3] != p[3])) != 0U) {
#pragma unroll
                    for (uint32_t e = 0U; e < 4U; ++e) {
                        p[e] = m3_bits_f32(m3_gated_silu_bits(
                            m3_bits_f32(raw[e] << 16U), u[e], M3N_BF16));
                    }
                }
#pragma unroll
                for (uint32_t e = 0U; e < 4U; ++e) {
                    r[e] = m3_f32_bits(p[e]);
                }
                m3_store4<M3N_BF16>(a.output, index, r);
            }
        }
    }
    if (blockIdx.x == 0U && threadIdx.x < a.tail) {
        const uint64_t e = 4ULL * a.groups + threadIdx.x;
        const uint64_t ge =
            ROWS ? m3_silu_row_offset(a, a.gate_pitch, (uint32_t)e) : e;
        const uint64_t ue =
            ROWS ? m3_silu_row_offset(a, a.up_pitch, (uint32_t)e) : e;
        float g = m3_bits_f32(m3_load_element(a.gate + 2U * ge, M3N_BF16));
        float u = m3_bits_f32(m3_load_element(a.up + 2U * ue, M3N_BF16));

        m3_store_element(a.output + 2U * e, M3N_BF16,
                         m3_gated_silu_bits(g, u, M3N_BF16));
    }
}

/* Gate, up and output all of dtype D. */
template <uint32_t D, bool ROWS>
__global__ __launch_bounds__(256) void m3_gated_silu_vec_kernel(
    m3_silu_vec_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint32_t step = gridDim.x * kThreads * kUnroll;
    constexpr uint32_t size = D == M3N_F32 ? 4U : 2U;
    __shared__ uint64_t table[32];

    if (threadIdx.x < 32U) {
        table[threadIdx.x] = m3_expf_table[threadIdx.x];
    }
    __syncthreads();
    for (uint32_t first = blockIdx.x * kThreads * kUnroll + threadIdx.x;
         first < a.groups; first += step) {
        float g[kUnroll][4];
        float u[kUnroll][4];

        /* unconditional loads (groups past the end re-read the last one)
         * so that all of them are in flight before the first use */
#pragma unroll
        for (uint32_t k = 0U; k < kUnroll; ++k) {
            const uint32_t index = min(first + k * kThreads, a.groups - 1U);

            const uint4 gr =
                m3_silu_load4<D, ROWS>(a, a.gate, a.gate_pitch, index);
            const uint4 ur =
                m3_silu_load4<D, ROWS>(a, a.up, a.up_pitch, index);

            g[k][0] = m3_bits_f32(m3_load_as_f32_bits(gr.x, D));
            g[k][1] = m3_bits_f32(m3_load_as_f32_bits(gr.y, D));
            g[k][2] = m3_bits_f32(m3_load_as_f32_bits(gr.z, D));
            g[k][3] = m3_bits_f32(m3_load_as_f32_bits(gr.w, D));
            u[k][0] = m3_bits_f32(m3_load_as_f32_bits(ur.x, D));
            u[k][1] = m3_bits_f32(m3_load_as_f32_bits(ur.y, D));
            u[k][2] = m3_bits_f32(m3_load_as_f32_bits(ur.z, D));
            u[k][3] = m3_bits_f32(m3_load_as_f32_bits(ur.w, D));
        }
#pragma unroll
        for (uint32_t k = 0U; k < kUnroll; ++k) {
            uint32_t index = first + k * kThreads;

            if (index < a.groups) {
                uint32_t r[4];

                m3_silu4<D>(g[k], u[k], table, r);
                m3_store4<D>(a.output, index, r);
            }
        }
    }
    if (blockIdx.x == 0U && threadIdx.x < a.tail) {
        const uint64_t e = 4ULL * a.groups + threadIdx.x;
        const uint64_t ge =
            ROWS ? m3_silu_row_offset(a, a.gate_pitch, (uint32_t)e) : e;
        const uint64_t ue =
            ROWS ? m3_silu_row_offset(a, a.up_pitch, (uint32_t)e) : e;
        float g = m3_bits_f32(m3_load_element(a.gate + size * ge, D));
        float u = m3_bits_f32(m3_load_element(a.up + size * ue, D));

        m3_store_element(a.output + size * e, D, m3_gated_silu_bits(g, u, D));
    }
}

__global__ __launch_bounds__(256) void m3_gated_silu_general_kernel(
    m3_activation_general_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t out_size = a.dtypes[0] == M3N_F32 ? 4U : 2U;

    for (uint64_t f = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
         f < a.count; f += step) {
        int64_t offsets[2];

        m3_general_offsets(a, f, offsets);
        float g = m3_bits_f32(
            m3_load_element(a.inputs[0] + offsets[0], a.dtypes[1]));
        float u = m3_bits_f32(
            m3_load_element(a.inputs[1] + offsets[1], a.dtypes[2]));

        m3_store_element(a.output + out_size * f, a.dtypes[0],
                         m3_gated_silu_bits(g, u, a.dtypes[1]));
    }
}

/* ---- launch planning ----------------------------------------------------- */

bool m3_same_shape(const m3_hip_view *a, const m3_hip_view *b)
{
    if (a->rank != b->rank) {
        return false;
    }
    for (uint32_t axis = 0U; axis < a->rank; ++axis) {
        if (a->shape[axis] != b->shape[axis]) {
            return false;
        }
    }
    return true;
}

bool m3_is_float(uint32_t dtype)
{
    return dtype == M3_HIP_F32 || dtype == M3_HIP_F16 ||
           dtype == M3_HIP_BF16;
}

/* Fills the general kernel's arguments from the coalesced index space of
 * `output` with inputs `first` and `second` (second may be null). */
void m3_general_args(const m3_hip_view *output, const m3_hip_view *first,
                     const m3_hip_view *second,
                     m3_activation_general_args *args)
{
    const m3_hip_view *operands[3] = {output, first,
                                      second != nullptr ? second : first};
    m3_index_plan plan;

    m3_plan_index_space(output, operands, 3U, &plan);
    std::memset(args, 0, sizeof(*args));
    args->inputs[0] = (const uint8_t *)first->base + first->byte_offset;
    args->inputs[1] =
        second != nullptr
            ? (const uint8_t *)second->base + second->byte_offset
            : args->inputs[0];
    args->output = (uint8_t *)output->base + output->byte_offset;
    args->dtypes[0] = output->dtype;
    args->dtypes[1] = first->dtype;
    args->dtypes[2] = second != nullptr ? second->dtype : first->dtype;
    args->rank = plan.rank;
    args->count = output->element_count;
    for (uint32_t axis = 0U; axis < plan.rank; ++axis) {
        args->shape[axis] = plan.shape[axis];
        args->strides[0][axis] = plan.strides[1][axis];
        args->strides[1][axis] = plan.strides[2][axis];
    }
}

/* True when `view`, of the output's element count, is rows of *width
 * contiguous elements, *pitch elements apart (a contiguous view: one row),
 * after merging its axes. */
bool m3_silu_rows(const m3_hip_view *view, uint64_t *width, uint64_t *pitch)
{
    const uint64_t size = m3_dtype_bytes(view->dtype);
    const m3_hip_view *operands[1] = {view};
    m3_index_plan plan;

    m3_plan_index_space(view, operands, 1U, &plan);
    if (plan.rank > 2U || plan.strides[0][plan.rank - 1U] != (int64_t)size) {
        return false;
    }
    *width = plan.shape[plan.rank - 1U];
    *pitch = plan.rank == 1U ? *width
                             : (uint64_t)plan.strides[0][0] / size;
    return plan.rank == 1U || (uint64_t)plan.strides[0][0] % size == 0U;
}

template <uint32_t D, bool ROWS>
void m3_launch_silu_vec(m3_hip_device *device, const m3_silu_vec_args &args,
                        uint32_t blocks, hipEvent_t start, hipEvent_t stop)
{
    if (D == M3N_BF16) {
        hipExtLaunchKernelGGL((m3_gated_silu_bf16_kernel<ROWS>), dim3(blocks),
                              dim3(kThreads), 0, device->stream, start, stop,
                              0U, args,
                              (const uint4 *)device->silu_bf16_table);
        return;
    }
    hipExtLaunchKernelGGL((m3_gated_silu_vec_kernel<D, ROWS>), dim3(blocks),
                          dim3(kThreads), 0, device->stream, start, stop, 0U,
                          args);
}

} // namespace

int m3_silu_table_build(m3_hip_device *device, char *message,
                        size_t capacity)
{
    int code = m3_hip_check((hipError_t)m3_hip_malloc((void **)&device->silu_bf16_table,
                                      kSiluTableEntries * sizeof(uint16_t)),
                            "hipMalloc(GATED_SILU table)", message, capacity);

    if (code != M3_HIP_OK) {
        device->silu_bf16_table = nullptr;
        return code;
    }
    hipLaunchKernelGGL(m3_silu_table_build_kernel,
                       dim3(kSiluTableEntries / 256U), dim3(256), 0,
                       device->stream, device->silu_bf16_table);
    return m3_hip_check(hipGetLastError(), "m3_silu_table_build", message,
                        capacity);
}

void m3_silu_table_release(m3_hip_device *device)
{
    if (device->silu_bf16_table != nullptr) {
        (void)hipFree(device->silu_bf16_table);
        device->silu_bf16_table = nullptr;
    }
}

extern "C" int m3_hip_launch_tanh(m3_hip_device *device,
                                  const m3_hip_view *input,
                                  const m3_hip_view *output, char *message,
                                  size_t capacity)
{
    if (device == nullptr || !m3_view_is_valid(input) ||
        !m3_view_is_valid(output) || input->dtype != M3_HIP_F32 ||
        output->dtype != M3_HIP_F32 || input->rank == 0U ||
        !m3_same_shape(input, output) || !m3_view_is_contiguous(output)) {
        return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                           "tanh launch arguments are malformed");
    }
    const uint64_t count = output->element_count;

    if (count == 0U) {
        return M3_HIP_OK;
    }
    /* below 2^32 elements the vector kernel's 32-bit group indices, plus
     * one grid stride (at most 2^28), stay below 2^32 */
    if (m3_view_is_contiguous(input) &&
        count >= m3_least_elements(device, kTanhQuarters) &&
        count < (1ULL << 32U)) {
        m3_tanh_vec_args args;

        args.list_gate = device->gate;
        args.input = (const uint8_t *)input->base + input->byte_offset;
        args.output = (uint8_t *)output->base + output->byte_offset;
        args.groups = (uint32_t)(count / 4U);
        args.tail = (uint32_t)(count % 4U);
        uint32_t blocks = m3_grid_blocks(
            device, args.groups == 0U ? 1U : args.groups,
            kThreads * kTanhUnroll, kBlocksPerCu);

        return m3_hip_launch(
            device, "m3_tanh",
            [&](hipEvent_t start, hipEvent_t stop) {
                hipExtLaunchKernelGGL(m3_tanh_vec_kernel, dim3(blocks),
                                      dim3(kThreads), 0, device->stream, start,
                                      stop, 0U, args);
            },
            message, capacity);
    }
    m3_activation_general_args args;

    m3_general_args(output, input, nullptr, &args);
    args.list_gate = device->gate;
    uint32_t blocks = m3_grid_blocks(device, count, 256U, 16U);

    return m3_hip_launch(
        device, "m3_tanh_strided",
        [&](hipEvent_t start, hipEvent_t stop) {
            hipExtLaunchKernelGGL(m3_tanh_general_kernel, dim3(blocks),
                                  dim3(256), 0, device->stream, start, stop,
                                  0U, args);
        },
        message, capacity);
}

extern "C" int m3_hip_launch_gated_silu(m3_hip_device *device,
                                        const m3_hip_view *gate,
                                        const m3_hip_view *up,
                                        const m3_hip_view *output,
                                        char *message, size_t capacity)
{
    if (device == nullptr || !m3_view_is_valid(gate) ||
        !m3_view_is_valid(up) || !m3_view_is_valid(output) ||
        !m3_is_float(gate->dtype) || !m3_is_float(up->dtype) ||
        !m3_is_float(output->dtype) || !m3_same_shape(gate, up) ||
        !m3_same_shape(gate, output) || !m3_view_is_contiguous(output)) {
        return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                           "gated SiLU launch arguments are malformed");
    }
    const uint64_t count = output->element_count;

    if (count == 0U) {
        return M3_HIP_OK;
    }
    const uint32_t dtype = output->dtype;
    uint64_t gate_width = 0U;
    uint64_t up_width = 0U;
    uint64_t gate_pitch = 0U;
    uint64_t up_pitch = 0U;
    const bool contiguous =
        m3_view_is_contiguous(gate) && m3_view_is_contiguous(up);
    /* rows: each operand contiguous or in rows, the same ones; four
     * consecutive elements then lie in at most two rows */
    const bool in_rows =
        !contiguous && m3_silu_rows(gate, &gate_width, &gate_pitch) &&
        m3_silu_rows(up, &up_width, &up_pitch) &&
        (gate_width == up_width || gate_width == count ||
         up_width == count) &&
        std::min(gate_width, up_width) >= 4U;
    /* General against vector kernel, us, contiguous: F32 64K elements 3.4
     * and 3.9, 384K 4.1 and 4.1, 512K 4.7 and 4.2; F16 64K 3.6 and 6.0, 768K
     * 6.5 and 6.5, 1M 7.7 and 6.6; BF16 64K 3.4 and 4.8, 512K 4.7 and 4.9,
     * 768K 5.8 and 5.0. Halves of rows of 2 x 3,072: F32 192K (64 rows) 3.6
     * and 4.6, 512K 5.0 and 4.8; F16 192K 4.0 and 7.2, 768K 7.2 and 8.1, 1M
     * 8.6 and 7.9; BF16 192K 3.8 and 5.9, 768K 6.3 and 6.7, 1M 7.6 and
     * 6.1. */
    static const uint32_t quarters[3][2] = {{3U, 4U}, {6U, 7U}, {4U, 7U}};

    if (gate->dtype == dtype && up->dtype == dtype &&
        (contiguous || in_rows) &&
        count >= m3_least_elements(device, quarters[dtype][in_rows]) &&
        count < (1ULL << 32U)) { /* 32-bit group indices, as for TANH */
        m3_silu_vec_args args;

        std::memset(&args, 0, sizeof(args));
        args.list_gate = device->gate;
        args.gate = (const uint8_t *)gate->base + gate->byte_offset;
        args.up = (const uint8_t *)up->base + up->byte_offset;
        args.output = (uint8_t *)output->base + output->byte_offset;
        args.groups = (uint32_t)(count / 4U);
        args.tail = (uint32_t)(count % 4U);
        if (in_rows) {
            const uint64_t width = std::min(gate_width, up_width);

            args.width = m3_fast_div_make((uint32_t)width);
            args.gate_pitch = gate_width == width ? gate_pitch : width;
            args.up_pitch = up_width == width ? up_pitch : width;
        }
        uint32_t blocks = m3_grid_blocks(
            device, args.groups == 0U ? 1U : args.groups,
            kThreads * kUnroll, kBlocksPerCu);
        void (*launch)(m3_hip_device *, const m3_silu_vec_args &, uint32_t,
                       hipEvent_t, hipEvent_t) =
            dtype == M3_HIP_F32
                ? in_rows ? &m3_launch_silu_vec<M3N_F32, true>
                          : &m3_launch_silu_vec<M3N_F32, false>
            : dtype == M3_HIP_F16
                ? in_rows ? &m3_launch_silu_vec<M3N_F16, true>
                          : &m3_launch_silu_vec<M3N_F16, false>
            : in_rows ? &m3_launch_silu_vec<M3N_BF16, true>
                      : &m3_launch_silu_vec<M3N_BF16, false>;
        const char *name = dtype == M3_HIP_F32   ? "m3_gated_silu"
                           : dtype == M3_HIP_F16 ? "m3_gated_silu_f16"
                                                 : "m3_gated_silu_bf16";

        return m3_hip_launch(
            device, name,
            [&](hipEvent_t start, hipEvent_t stop) {
                launch(device, args, blocks, start, stop);
            },
            message, capacity);
    }
    m3_activation_general_args args;

    m3_general_args(output, gate, up, &args);
    args.list_gate = device->gate;
    uint32_t blocks = m3_grid_blocks(device, count, 256U, 16U);

    return m3_hip_launch(
        device, "m3_gated_silu_strided",
        [&](hipEvent_t start, hipEvent_t stop) {
            hipExtLaunchKernelGGL(m3_gated_silu_general_kernel, dim3(blocks),
                                  dim3(256), 0, device->stream, start, stop,
                                  0U, args);
        },
        message, capacity);
}
