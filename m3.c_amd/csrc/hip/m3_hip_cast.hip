/*
 * m3_hip_cast.hip - CAST and COPY for gfx950.
 *
 * Semantics are the reference's m3_host_cast / m3_host_copy
 * (src/m3_op_execute_basic.c:11-59) and Metal m3_cast / m3_copy
 * (src/m3_backend_metal_basic.m:29-63):
 *   - same dtype: the element bytes are copied;
 *   - I32 -> float: (float)i, rounded to nearest even, then stored like
 *     any F32 value (so I32 -> F16 rounds twice, as the reference does);
 *   - float -> I32: truncation toward zero (inputs were scanned first);
 *   - float -> float: exact widening to F32, then the bit-exact RNE
 *     narrowing of m3_numeric.h. NaN payloads follow the reference rules.
 * The output is contiguous. A contiguous, aligned input runs the vector
 * kernel (four elements per lane per group, two groups in flight, output
 * written with streaming stores), or, for the cheap conversions of a
 * tensor whose lanes are all resident at once, its held form (all loads,
 * then the stores after a timed wait);
 * an input whose unit-stride axis is another than the output's innermost
 * one (a permuted view) goes through transposing tiles in LDS; other
 * strided inputs run a per-element kernel over the coalesced index space.
 */
#include "m3_hip_internal.h"

#include <algorithm>
#include <cstring>

namespace {

constexpr uint32_t kThreads = 256U;
constexpr uint32_t kUnroll = 2U; /* groups in flight per lane, copies */
/* Groups in flight per lane of a conversion: 4 when it narrows (4-byte to
 * 16-bit elements), 2 otherwise. Against 2, in bench.py alternating
 * libraries on one box: F32 -> F16 17.4-17.5 against 17.6-17.8 us and
 * F32 -> BF16 16.9-17.0 against 17.0-17.1 us; the widening casts measured
 * the same or slower with 1 or 4. */
constexpr uint32_t m3_cast_unroll(uint32_t in_size, uint32_t out_size)
{
    return in_size > out_size ? 4U : 2U;
}
/* workgroups per CU of a conversion: up to 32, so that a 16M-element
 * cast runs each lane's groups in one pass instead of a grid-stride loop
 * (measured 2% faster for F16 -> F32 than 16 per CU) */
constexpr uint32_t kCastBlocksPerCu = 32U;

template <uint32_t DT>
struct m3_vec_io;

/* Four 4-byte elements: one 16-byte access, read with a streaming load
 * (each input byte is read once). */
template <>
struct m3_vec_io<4U> {
    using type = uint4;
    __device__ static type load(const type *p) { return m3_stream_load(p); }
    __device__ static uint4 unpack(type v) { return v; }
    __device__ static type pack(uint4 v) { return v; }
};

/* Four 2-byte elements: one 8-byte access, read with a streaming load
 * (F16 -> F32 17.8-18.0 against 18.3-18.5 us with an ordinary one, BF16 ->
 * F32 17.8-18.0 against 18.3-18.5 us; bench.py alternating libraries on
 * one box). */
template <>
struct m3_vec_io<2U> {
    using type = uint2;
    __device__ static type load(const type *p) { return m3_stream_load(p); }
    __device__ static uint4 unpack(type v)
    {
        return make_uint4(v.x & 0xffffU, v.x >> 16U, v.y & 0xffffU,
                          v.y >> 16U);
    }
    __device__ static type pack(uint4 v)
    {
        return make_uint2((v.x & 0xffffU) | (v.y << 16U),
                          (v.z & 0xffffU) | (v.w << 16U));
    }
};

constexpr uint32_t m3_size_of(uint32_t dtype)
{
    return dtype == M3N_F16 || dtype == M3N_BF16 ? 2U : 4U;
}

template <uint32_t IN, uint32_t OUT>
__device__ __forceinline__ uint32_t m3_convert(uint32_t raw)
{
    return m3_store_from_f32_bits(m3_load_as_f32_bits(raw, IN), OUT);
}

template <uint32_t IN, uint32_t OUT>
__global__ __launch_bounds__(256) void m3_cast_vec_kernel(
    const uint8_t *input, uint8_t *output, uint64_t count, uint64_t groups,
    m3_hip_gate gate)
{
    if (m3_gate_closed(gate)) {
        return; /* a check earlier in the list failed */
    }
    using in_io = m3_vec_io<m3_size_of(IN)>;
    using out_io = m3_vec_io<m3_size_of(OUT)>;
    const typename in_io::type *in = (const typename in_io::type *)input;
    typename out_io::type *out = (typename out_io::type *)output;
    constexpr uint32_t unroll = m3_cast_unroll(m3_size_of(IN), m3_size_of(OUT));
    const uint64_t step = (uint64_t)gridDim.x * kThreads * unroll;

    for (uint64_t first = (uint64_t)blockIdx.x * kThreads * unroll +
                          threadIdx.x;
         first < groups; first += step) {
        uint4 v[unroll];

#pragma unroll
        for (uint32_t u = 0U; u < unroll; ++u) {
            uint64_t g = first + u * kThreads;

            if (g < groups) {
                v[u] = in_io::unpack(in_io::load(&in[g]));
            }
        }
#pragma unroll
        for (uint32_t u = 0U; u < unroll; ++u) {
            uint64_t g = first + u * kThreads;

            if (g < groups) {
                uint4 r = make_uint4(m3_convert<IN, OUT>(v[u].x),
                                     m3_convert<IN, OUT>(v[u].y),
                                     m3_convert<IN, OUT>(v[u].z),
                                     m3_convert<IN, OUT>(v[u].w));

                m3_stream_store(&out[g], out_io::pack(r));
            }
        }
    }
    if (blockIdx.x == 0U && threadIdx.x < count - groups * 4U) {
        uint64_t f = groups * 4U + threadIdx.x;
        uint32_t raw = m3_size_of(IN) == 4U
                           ? ((const uint32_t *)input)[f]
                           : (uint32_t)((const uint16_t *)input)[f];
        uint32_t r = m3_convert<IN, OUT>(raw);

        if (m3_size_of(OUT) == 4U) {
            ((uint32_t *)output)[f] = r;
        } else {
            ((uint16_t *)output)[f] = (uint16_t)r;
        }
    }
}

struct m3_strided_args {
    const uint8_t *input;
    uint8_t *output;
    uint32_t in_dtype;
    uint32_t out_dtype;
    uint32_t rank;
    uint64_t count;
    uint64_t shape[M3_HIP_MAX_RANK];
    int64_t strides[M3_HIP_MAX_RANK];
    m3_hip_gate list_gate;
};

/* Strided input, contiguous output; `convert` false copies raw elements. */
__global__ __launch_bounds__(256) void m3_cast_strided_kernel(
    m3_strided_args a, bool convert)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    const uint32_t in_size = m3_size_of(a.in_dtype);
    const uint32_t out_size = m3_size_of(a.out_dtype);

    for (uint64_t f = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
         f < a.count; f += step) {
        uint64_t rest = f;
        int64_t offset = 0;

        for (int axis = (int)a.rank - 1; axis >= 0; --axis) {
            uint64_t dim = a.shape[axis];
            uint64_t q = rest / dim;

            offset += (int64_t)(rest - q * dim) * a.strides[axis];
            rest = q;
        }
        uint32_t raw = in_size == 4U
                           ? *(const uint32_t *)(a.input + offset)
                           : (uint32_t) * (const uint16_t *)(a.input + offset);
        uint32_t r = convert ? m3_store_from_f32_bits(
                                   m3_load_as_f32_bits(raw, a.in_dtype),
                                   a.out_dtype)
                             : raw;

        if (out_size == 4U) {
            *(uint32_t *)(a.output + f * 4U) = r;
        } else {
            *(uint16_t *)(a.output + f * 2U) = (uint16_t)r;
        }
    }
}

/* Contiguous byte copy with 16-byte words; `tail` bytes finish it. */
__global__ __launch_bounds__(256) void m3_copy_bytes_kernel(
    const uint4 *input, uint4 *output, uint64_t words, const uint8_t *tail_in,
    uint8_t *tail_out, uint32_t tail, m3_hip_gate gate)
{
    if (m3_gate_closed(gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t step = (uint64_t)gridDim.x * kThreads * kUnroll;

    for (uint64_t first = (uint64_t)blockIdx.x * kThreads * kUnroll +
                          threadIdx.x;
         first < words; first += step) {
        uint4 v[kUnroll];

#pragma unroll
        for (uint32_t u = 0U; u < kUnroll; ++u) {
            uint64_t g = first + u * kThreads;

            if (g < words) {
                v[u] = m3_stream_load(&input[g]);
            }
        }
#pragma unroll
        for (uint32_t u = 0U; u < kUnroll; ++u) {
            uint64_t g = first + u * kThreads;

            if (g < words) {
                m3_stream_store(&output[g], v[u]);
            }
        }
    }
    if (blockIdx.x == 0U && threadIdx.x < tail) {
        tail_out[threadIdx.x] = tail_in[threadIdx.x];
    }
}

/* ---- transposing tiles ------------------------------------------------------ */

/* An input whose consecutive elements lie along another axis (u) than the
 * output's (n): the output's innermost axis n steps by n_stride bytes in
 * the input, and axis u, whose consecutive elements are out_u_stride
 * elements apart in the output, is the input's unit-stride one. */
struct m3_transpose_args {
    const uint8_t *input;
    uint8_t *output;
    uint32_t n;
    uint32_t u;
    int64_t n_stride;
    uint64_t out_u_stride;
    uint32_t tiles; /* tiles_n * tiles_u * the outer axes' extents */
    m3_fast_div tiles_n;
    m3_fast_div tiles_u;
    uint32_t outer_rank;
    uint64_t outer_shape[M3_HIP_MAX_RANK];
    int64_t outer_in[M3_HIP_MAX_RANK];   /* bytes */
    uint64_t outer_out[M3_HIP_MAX_RANK]; /* elements */
    m3_hip_gate list_gate;
};

/* When tiles are used: both extents at least 16 (below it a tile's lanes are
 * less than a quarter (u) or an eighth (n) full), and so much of the tiles
 * that cover the two axes inside the tensor that the tile kernel's work for
 * nothing stays below what one element per lane costs: 5 of 64 parts for a
 * copy, 6 for a conversion, 9 for one from or to F16 (in integer
 * instructions). Against the per-element kernel, many small planes of n x u,
 * F32, BF16 and F16 to F32: 16 x 16 (2 parts) 60 -> 120, 59 -> 90 and 65 ->
 * 209 us, 24 x 24 (4.5) 63 -> 61, 58 -> 46 and 65 -> 100, 24 x 32 (6) 62 ->
 * 51, 58 -> 38 and 66 -> 78, 32 x 32 (8) 61 -> 39, 59 -> 29 and 66 -> 60, 32
 * x 40 (10) 64 -> 34, 58 -> 26 and 66 -> 51; a plane that only just needs a
 * second tile, 17 x 70 (4.6), 60 -> 84, 59 -> 65 and 65 -> 115. */
constexpr uint32_t kTransposeLeast = 16U;
constexpr uint32_t kTransposeFillCopy = 5U;
constexpr uint32_t kTransposeFill = 6U;
constexpr uint32_t kTransposeFillF16 = 9U;
constexpr uint32_t kTileU = 64U;
constexpr uint32_t kTileN = 128U;
constexpr uint32_t kXcds = 8U;
constexpr uint32_t kMaxTransposeGrid = 1U << 20; /* workgroups; they loop */

/* Four consecutive elements at any alignment, zero-extended. */
template <uint32_t SIZE>
__device__ __forceinline__ uint4 m3_load4_any(const uint8_t *p)
{
    if (SIZE == 4U) {
        const m3_u32x4_any w = *(const m3_u32x4_any *)p;

        return make_uint4(w[0], w[1], w[2], w[3]);
    }
    const m3_u32x2_any h = *(const m3_u32x2_any *)p;

    return make_uint4(h[0] & 0xffffU, h[0] >> 16U, h[1] & 0xffffU,
                      h[1] >> 16U);
}

/* A tile of 64 (u) by 128 (n) elements through LDS: each lane reads four
 * elements along u at four consecutive n, transposes the 4 x 4 block in
 * registers, converts it and writes it as four vectors along n; the tile is
 * then stored along n. Both sides of memory move whole runs (256 bytes and
 * 512 for 4-byte elements), at any alignment. The vector slot of a row in
 * LDS is rotated by an exclusive or with the row's group of four, so that
 * the lanes of a write (consecutive u) and of a read (consecutive n) both
 * fall on distinct banks. IN == OUT copies raw elements.
 *
 * Bound by HBM; against one element per lane with 64-bit divisions and
 * strided reads: F32 [2,8191,512] 36.5 -> 13.9 us (4.8 TB/s; 9.9 us at
 * length 8192, whose stores are aligned), F32 [1,32000,1024] 610 -> 40.5,
 * BF16 [2,8191,512] 37.4 -> 7.8, BF16 to F32 [4,8000,1001] 283 -> 31.
 * Nontemporal stores against ordinary ones: 9.9 against 11.9 us at length
 * 8192, 31 against 36 for [4,8000,1001], 13.0 against 12.4 at 8191. Tiles
 * of 64 along n: 14.5 at 8191, 64 against 49 for F32 [1,31999,1024];
 * neighbouring tiles dealt to different XCDs: 47 against 40.5. */
template <uint32_t IN, uint32_t OUT>
__global__ __launch_bounds__(256) void m3_transpose_kernel(m3_transpose_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    constexpr uint32_t in_size = m3_size_of(IN);
    constexpr uint32_t out_size = m3_size_of(OUT);
    using out_io = m3_vec_io<out_size>;
    using slot_type = typename out_io::type;
    constexpr uint32_t kSlots = kTileN / 4U; /* vectors per tile row */
    __shared__ slot_type lds[kTileU][kSlots];
    const uint32_t ul = threadIdx.x & 15U;
    const uint32_t nl = threadIdx.x >> 4U;

    for (uint32_t block = blockIdx.x; block < a.tiles; block += gridDim.x) {
        uint32_t tile = block;

        if (gridDim.x == a.tiles) {
            /* neighbouring tiles, which share lines at their edges, on one
             * XCD (workgroups go round the XCDs) */
            const uint32_t xcd = block % kXcds;
            const uint32_t share = a.tiles / kXcds;
            const uint32_t rest = a.tiles % kXcds;

            tile = xcd * share + min(xcd, rest) + block / kXcds;
        }
        const uint32_t q = m3_fast_div_q(a.tiles_n, tile);
        const uint32_t tile_n = (tile - q * a.tiles_n.divisor) * kTileN;
        uint64_t outer = m3_fast_div_q(a.tiles_u, q);
        const uint32_t tile_u =
            (q - (uint32_t)outer * a.tiles_u.divisor) * kTileU;
        const uint8_t *in = a.input;
        uint8_t *out = a.output;

        for (int axis = (int)a.outer_rank - 1; axis >= 0; --axis) {
            const uint64_t dim = a.outer_shape[axis];
            const uint64_t rest = outer / dim;
            const uint64_t c = outer - rest * dim;

            in += (int64_t)c * a.outer_in[axis];
            out += c * a.outer_out[axis] * out_size;
            outer = rest;
        }
        /* the tile's last partial vector along u is read from the row's
         * last four elements (u >= 4), which repeat the lanes before it */
        const uint32_t u0 = min(tile_u + 4U * ul, a.u - 4U);
        const bool inside = tile_u + 4U * ul < a.u;
        uint4 v[kSlots / 16U][4];

#pragma unroll
        for (uint32_t k = 0U; k < kSlots / 16U; ++k) {
#pragma unroll
            for (uint32_t i = 0U; i < 4U; ++i) {
                const uint32_t n = tile_n + 64U * k + 4U * nl + i;

                v[k][i] = m3_load4_any<in_size>(
                    in + (int64_t)min(n, a.n - 1U) * a.n_stride +
                    (uint64_t)u0 * in_size);
            }
        }
#pragma unroll
        for (uint32_t k = 0U; k < kSlots / 16U; ++k) {
            const uint4 t[4] = {
                make_uint4(v[k][0].x, v[k][1].x, v[k][2].x, v[k][3].x),
                make_uint4(v[k][0].y, v[k][1].y, v[k][2].y, v[k][3].y),
                make_uint4(v[k][0].z, v[k][1].z, v[k][2].z, v[k][3].z),
                make_uint4(v[k][0].w, v[k][1].w, v[k][2].w, v[k][3].w)};

#pragma unroll
            for (uint32_t e = 0U; e < 4U; ++e) {
                /* rows before the tile wrap and are dropped */
                const uint32_t r = u0 + e - tile_u;
                uint4 w = t[e];

                if (IN != OUT) {
                    w = make_uint4(m3_convert<IN, OUT>(w.x),
                                   m3_convert<IN, OUT>(w.y),
                                   m3_convert<IN, OUT>(w.z),
                                   m3_convert<IN, OUT>(w.w));
                }
                if (inside && r < kTileU) {
                    lds[r][(16U * k + nl) ^ ((r >> 2U) & 15U)] =
                        out_io::pack(w);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t s = 0U; s < kTileU * kSlots / kThreads; ++s) {
            const uint32_t index = s * kThreads + threadIdx.x;
            const uint32_t r = index / kSlots;
            const uint32_t slot = index % kSlots;
            const uint32_t n = tile_n + 4U * slot;

            if (tile_u + r >= a.u || n >= a.n) {
                continue;
            }
            const slot_type w = lds[r][slot ^ ((r >> 2U) & 15U)];
            uint8_t *p =
                out + ((tile_u + r) * a.out_u_stride + n) * out_size;

            if (n + 4U <= a.n) {
                m3_stream_store((slot_type *)p, w);
                continue;
            }
            const uint4 x = out_io::unpack(w);
            const uint32_t rest[3] = {x.x, x.y, x.z};

#pragma unroll
            for (uint32_t i = 0U; i < 3U; ++i) {
                if (n + i >= a.n) {
                    continue;
                }
                if (out_size == 4U) {
                    ((uint32_t *)p)[i] = rest[i];
                } else {
                    ((uint16_t *)p)[i] = (uint16_t)rest[i];
                }
            }
        }
        __syncthreads(); /* the next tile overwrites the LDS */
    }
}

/* Groups of four elements per lane of the held form. */
constexpr int kHeldGroups = 8;
/* Workgroups per CU that are all resident at once in the held form (its
 * lanes take at most 64 VGPRs: eight waves per SIMD). */
constexpr uint32_t kHeldBlocksPerCu = 8U;

/* How long the held form of a conversion waits before its stores, as a
 * multiple of the time the launch's reads take at 8 TB/s; 0 where it is
 * not used. Measured in bench.py, alternating libraries on one box
 * (4096 x 4096): F16 -> F32 and BF16 -> F32 16.7-17.1 us at 1.4 against
 * 18.0-18.5 us with the streaming kernel (1.19: 17.1-17.5, 1.6: 17.5-17.8);
 * F32 -> BF16 16.3-16.4 against 16.7-17.0 us at 1.19 (1.4: 18.1). F32 ->
 * F16, whose conversion takes several times the instructions, measured
 * slower held at every factor (19.6-21.4 against 17.2-17.4 us): its
 * conversions, all after the loads, then delay the stores. */
constexpr double m3_cast_hold_factor(uint32_t in, uint32_t out)
{
    return (in == M3N_F16 || in == M3N_BF16) && out == M3N_F32 ? 1.4
           : in == M3N_F32 && out == M3N_BF16                  ? 1.19
                                                                : 0.0;
}

/* The held form of the vector conversion, for a launch whose workgroups
 * are all resident at once: each lane loads its kHeldGroups groups, forms
 * their results, and stores them only hold_ticks (s_memrealtime) after its
 * start, so that the launch's writes do not compete with its reads still
 * in flight (HBM serves a phase of reads, then one of writes). The wait is
 * bounded by the clock; results are those of m3_cast_vec_kernel. */
template <uint32_t IN, uint32_t OUT, int K>
__global__ __launch_bounds__(256) void m3_cast_held_kernel(
    const uint8_t *input, uint8_t *output, uint64_t count, uint64_t groups,
    uint32_t hold_ticks, m3_hip_gate gate)
{
    if (m3_gate_closed(gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t start = __builtin_amdgcn_s_memrealtime();
    using in_io = m3_vec_io<m3_size_of(IN)>;
    using out_io = m3_vec_io<m3_size_of(OUT)>;
    const typename in_io::type *in = (const typename in_io::type *)input;
    typename out_io::type *out = (typename out_io::type *)output;
    const uint64_t first = (uint64_t)blockIdx.x * kThreads * K + threadIdx.x;
    typename out_io::type result[K];

#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint64_t g = first + (uint64_t)k * kThreads;
        uint4 v = make_uint4(0U, 0U, 0U, 0U);

        if (g < groups) {
            v = in_io::unpack(in_io::load(&in[g]));
        }
        result[k] = out_io::pack(make_uint4(m3_convert<IN, OUT>(v.x),
                                            m3_convert<IN, OUT>(v.y),
                                            m3_convert<IN, OUT>(v.z),
                                            m3_convert<IN, OUT>(v.w)));
    }
    while (__builtin_amdgcn_s_memrealtime() - start < (uint64_t)hold_ticks) {
        __builtin_amdgcn_s_sleep(2);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint64_t g = first + (uint64_t)k * kThreads;

        if (g < groups) {
            m3_stream_store(&out[g], result[k]);
        }
    }
    if (blockIdx.x == 0U && threadIdx.x < count - groups * 4U) {
        uint64_t f = groups * 4U + threadIdx.x;
        uint32_t raw = m3_size_of(IN) == 4U
                           ? ((const uint32_t *)input)[f]
                           : (uint32_t)((const uint16_t *)input)[f];
        uint32_t r = m3_convert<IN, OUT>(raw);

        if (m3_size_of(OUT) == 4U) {
            ((uint32_t *)output)[f] = r;
        } else {
            ((uint16_t *)output)[f] = (uint16_t)r;
        }
    }
}

template <uint32_t IN, uint32_t OUT>
void m3_launch_cast_vec(m3_hip_device *device, const uint8_t *input,
                        uint8_t *output, uint64_t count, uint32_t blocks,
                        hipEvent_t start, hipEvent_t stop)
{
    constexpr double factor = m3_cast_hold_factor(IN, OUT);
    const uint64_t groups = count / 4U;
    const uint64_t held =
        (groups + kThreads * kHeldGroups - 1U) / (kThreads * kHeldGroups);

    const uint64_t slots =
        (uint64_t)device->compute_units * kHeldBlocksPerCu;

    /* held only when its workgroups fill at least half of what the device
     * holds at once (few workgroups of eight groups per lane would leave
     * most CUs idle) and fit in it */
    if (factor > 0.0 && device->wall_clock_khz != 0U && 2U * held >= slots &&
        held <= slots) {
        const double us = factor * (double)count * m3_size_of(IN) / 8.0e6;
        const uint32_t ticks =
            (uint32_t)(us * (double)device->wall_clock_khz / 1000.0);

        hipExtLaunchKernelGGL((m3_cast_held_kernel<IN, OUT, kHeldGroups>),
                              dim3((uint32_t)held), dim3(kThreads), 0,
                              device->stream, start, stop, 0U, input, output,
                              count, groups, ticks, device->gate);
        return;
    }
    hipExtLaunchKernelGGL((m3_cast_vec_kernel<IN, OUT>), dim3(blocks),
                          dim3(kThreads), 0, device->stream, start, stop, 0U,
                          input, output, count, count / 4U, device->gate);
}

typedef void (*m3_cast_launcher)(m3_hip_device *, const uint8_t *, uint8_t *,
                                 uint64_t, uint32_t, hipEvent_t, hipEvent_t);

m3_cast_launcher m3_cast_vec_launcher(uint32_t in, uint32_t out)
{
#define M3_CAST_CASE(I, O)                                                    \
    if (in == (I) && out == (O)) {                                           \
        return &m3_launch_cast_vec<(I), (O)>;                                \
    }
    M3_CAST_CASE(M3N_F32, M3N_F16)
    M3_CAST_CASE(M3N_F32, M3N_BF16)
    M3_CAST_CASE(M3N_F32, M3N_I32)
    M3_CAST_CASE(M3N_F16, M3N_F32)
    M3_CAST_CASE(M3N_F16, M3N_BF16)
    M3_CAST_CASE(M3N_F16, M3N_I32)
    M3_CAST_CASE(M3N_BF16, M3N_F32)
    M3_CAST_CASE(M3N_BF16, M3N_F16)
    M3_CAST_CASE(M3N_BF16, M3N_I32)
    M3_CAST_CASE(M3N_I32, M3N_F32)
    M3_CAST_CASE(M3N_I32, M3N_F16)
    M3_CAST_CASE(M3N_I32, M3N_BF16)
#undef M3_CAST_CASE
    return nullptr;
}

typedef void (*m3_transpose_launcher)(dim3, hipStream_t, hipEvent_t,
                                      hipEvent_t, m3_transpose_args);

template <uint32_t IN, uint32_t OUT>
void m3_launch_transpose(dim3 grid, hipStream_t stream, hipEvent_t start,
                         hipEvent_t stop, m3_transpose_args args)
{
    hipExtLaunchKernelGGL((m3_transpose_kernel<IN, OUT>), grid,
                          dim3(kThreads), 0, stream, start, stop, 0U, args);
}

/* The transposing kernel of a conversion; copies of one element size share
 * one. */
m3_transpose_launcher m3_transpose_of(uint32_t in, uint32_t out)
{
    static const m3_transpose_launcher launchers[4][4] = {
        {&m3_launch_transpose<M3N_F32, M3N_F32>,
         &m3_launch_transpose<M3N_F32, M3N_F16>,
         &m3_launch_transpose<M3N_F32, M3N_BF16>,
         &m3_launch_transpose<M3N_F32, M3N_I32>},
        {&m3_launch_transpose<M3N_F16, M3N_F32>,
         &m3_launch_transpose<M3N_F16, M3N_F16>,
         &m3_launch_transpose<M3N_F16, M3N_BF16>,
         &m3_launch_transpose<M3N_F16, M3N_I32>},
        {&m3_launch_transpose<M3N_BF16, M3N_F32>,
         &m3_launch_transpose<M3N_BF16, M3N_F16>,
         &m3_launch_transpose<M3N_F16, M3N_F16>,
         &m3_launch_transpose<M3N_BF16, M3N_I32>},
        {&m3_launch_transpose<M3N_I32, M3N_F32>,
         &m3_launch_transpose<M3N_I32, M3N_F16>,
         &m3_launch_transpose<M3N_I32, M3N_BF16>,
         &m3_launch_transpose<M3N_F32, M3N_F32>}};

    return launchers[in][out];
}

/* Fills `args` when the plan (operand 1 the input) is one that the
 * transposing kernel takes: the innermost axis strided in the input, some
 * other axis of unit stride there, both of at least kTransposeLeast and
 * filling `fill` of 64 parts of their tiles. */
bool m3_plan_transpose(const m3_index_plan &plan, uint32_t in_size,
                       uint32_t fill, m3_transpose_args *args)
{
    const uint32_t inner = plan.rank - 1U;
    uint64_t out_strides[M3_HIP_MAX_RANK];
    uint64_t elements = 1U;
    uint64_t outer = 1U;
    uint32_t unit = plan.rank;

    for (int axis = (int)inner; axis >= 0; --axis) {
        out_strides[axis] = elements;
        elements *= plan.shape[axis];
        if (plan.strides[1][axis] == (int64_t)in_size) {
            unit = (uint32_t)axis;
        }
    }
    if (unit >= inner || plan.shape[inner] < kTransposeLeast ||
        plan.shape[unit] < kTransposeLeast ||
        plan.shape[inner] > 0x7fffffffULL ||
        plan.shape[unit] > 0x7fffffffULL) {
        return false;
    }
    for (uint32_t axis = 0U; axis < inner; ++axis) {
        if (axis == unit) {
            continue;
        }
        args->outer_shape[args->outer_rank] = plan.shape[axis];
        args->outer_in[args->outer_rank] = plan.strides[1][axis];
        args->outer_out[args->outer_rank] = out_strides[axis];
        args->outer_rank += 1U;
        outer *= plan.shape[axis];
    }
    const uint64_t tiles_n = (plan.shape[inner] + kTileN - 1U) / kTileN;
    const uint64_t tiles_u = (plan.shape[unit] + kTileU - 1U) / kTileU;

    /* two factors below 2^32 each, checked before the third */
    if (plan.shape[inner] * plan.shape[unit] <
            tiles_n * tiles_u * (kTileN * kTileU / 64U * fill) ||
        tiles_n * tiles_u > 0x7fffffffULL ||
        outer > 0x7fffffffULL / (tiles_n * tiles_u)) {
        return false;
    }
    args->n = (uint32_t)plan.shape[inner];
    args->u = (uint32_t)plan.shape[unit];
    args->n_stride = plan.strides[1][inner];
    args->out_u_stride = out_strides[unit];
    args->tiles = (uint32_t)(tiles_n * tiles_u * outer);
    args->tiles_n = m3_fast_div_make((uint32_t)tiles_n);
    args->tiles_u = m3_fast_div_make((uint32_t)tiles_u);
    return true;
}

const char *m3_cast_kernel_name(uint32_t in, uint32_t out)
{
    static const char *const names[4][4] = {
        {"m3_copy", "m3_cast_f32_f16", "m3_cast_f32_bf16", "m3_cast_f32_i32"},
        {"m3_cast_f16_f32", "m3_copy", "m3_cast_f16_bf16", "m3_cast_f16_i32"},
        {"m3_cast_bf16_f32", "m3_cast_bf16_f16", "m3_copy",
         "m3_cast_bf16_i32"},
        {"m3_cast_i32_f32", "m3_cast_i32_f16", "m3_cast_i32_bf16",
         "m3_copy"}};

    return names[in][out];
}

int m3_launch_unary(m3_hip_device *device, const m3_hip_view *input,
                    const m3_hip_view *output, char *message,
                    size_t capacity)
{
    const uint8_t *in = (const uint8_t *)input->base + input->byte_offset;
    uint8_t *out = (uint8_t *)output->base + output->byte_offset;
    const m3_hip_view *operands[2] = {output, input};
    const char *name = m3_cast_kernel_name(input->dtype, output->dtype);
    bool same = input->dtype == output->dtype;
    m3_index_plan plan;
    uint64_t count = output->element_count;

    m3_plan_index_space(output, operands, 2U, &plan);
    bool input_contiguous =
        plan.rank == 1U &&
        plan.strides[1][0] == (int64_t)m3_dtype_bytes(input->dtype);

    if (input_contiguous && same && ((uintptr_t)in & 15U) == 0U &&
        ((uintptr_t)out & 15U) == 0U) {
        uint64_t bytes = count * m3_dtype_bytes(input->dtype);
        uint64_t words = bytes / 16U;
        uint32_t tail = (uint32_t)(bytes % 16U);
        uint32_t blocks = m3_grid_blocks(device, words == 0U ? 1U : words,
                                         kThreads * kUnroll, 16U);

        return m3_hip_launch(
            device, name,
            [&](hipEvent_t start, hipEvent_t stop) {
                hipExtLaunchKernelGGL(m3_copy_bytes_kernel, dim3(blocks),
                                      dim3(kThreads), 0, device->stream, start,
                                      stop, 0U, (const uint4 *)in,
                                      (uint4 *)out, words, in + words * 16U,
                                      out + words * 16U, tail, device->gate);
            },
            message, capacity);
    }
    if (input_contiguous && !same) {
        uint32_t in_align = 4U * (uint32_t)m3_dtype_bytes(input->dtype);
        uint32_t out_align = 4U * (uint32_t)m3_dtype_bytes(output->dtype);
        m3_cast_launcher launcher =
            m3_cast_vec_launcher(input->dtype, output->dtype);

        if (launcher != nullptr && ((uintptr_t)in % in_align) == 0U &&
            ((uintptr_t)out % out_align) == 0U) {
            uint64_t groups = count / 4U;
            uint32_t blocks = m3_grid_blocks(device,
                                             groups == 0U ? 1U : groups,
                                             kThreads * m3_cast_unroll(
                                                 in_align / 4U,
                                                 out_align / 4U),
                                             kCastBlocksPerCu);

            return m3_hip_launch(
                device, name,
                [&](hipEvent_t start, hipEvent_t stop) {
                    launcher(device, in, out, count, blocks, start, stop);
                },
                message, capacity);
        }
    }
    m3_transpose_args transpose;

    std::memset(&transpose, 0, sizeof(transpose));
    const uint32_t fill = input->dtype == output->dtype ? kTransposeFillCopy
                          : input->dtype == M3_HIP_F16 ||
                                  output->dtype == M3_HIP_F16
                              ? kTransposeFillF16
                              : kTransposeFill;

    if (m3_plan_transpose(plan, (uint32_t)m3_dtype_bytes(input->dtype), fill,
                          &transpose)) {
        const m3_transpose_launcher launcher =
            m3_transpose_of(input->dtype, output->dtype);
        const dim3 grid(std::min(transpose.tiles, kMaxTransposeGrid));

        transpose.list_gate = device->gate;
        transpose.input = in;
        transpose.output = out;
        return m3_hip_launch(
            device, name,
            [&](hipEvent_t start, hipEvent_t stop) {
                launcher(grid, device->stream, start, stop, transpose);
            },
            message, capacity);
    }
    m3_strided_args args;

    std::memset(&args, 0, sizeof(args));
    args.list_gate = device->gate;
    args.input = in;
    args.output = out;
    args.in_dtype = input->dtype;
    args.out_dtype = output->dtype;
    args.rank = plan.rank;
    args.count = count;
    for (uint32_t axis = 0U; axis < plan.rank; ++axis) {
        args.shape[axis] = plan.shape[axis];
        args.strides[axis] = plan.strides[1][axis];
    }
    uint32_t blocks = m3_grid_blocks(device, count, 256U, 16U);

    return m3_hip_launch(
        device, name,
        [&](hipEvent_t start, hipEvent_t stop) {
            hipExtLaunchKernelGGL(m3_cast_strided_kernel, dim3(blocks),
                                  dim3(256), 0, device->stream, start, stop,
                                  0U, args, !same);
        },
        message, capacity);
}

bool m3_unary_views_ok(const m3_hip_view *input, const m3_hip_view *output)
{
    if (!m3_view_is_valid(input) || !m3_view_is_valid(output) ||
        input->rank != output->rank || !m3_view_is_contiguous(output)) {
        return false;
    }
    for (uint32_t axis = 0U; axis < input->rank; ++axis) {
        if (input->shape[axis] != output->shape[axis]) {
            return false;
        }
    }
    return true;
}

} // namespace

extern "C" int m3_hip_launch_cast(m3_hip_device *device,
                                  const m3_hip_view *input,
                                  const m3_hip_view *output, char *message,
                                  size_t capacity)
{
    if (device == nullptr || !m3_unary_views_ok(input, output)) {
        return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                           "cast launch arguments are malformed");
    }
    if (output->element_count == 0U) {
        return M3_HIP_OK;
    }
    return m3_launch_unary(device, input, output, message, capacity);
}

extern "C" int m3_hip_launch_copy(m3_hip_device *device,
                                  const m3_hip_view *input,
                                  const m3_hip_view *output, char *message,
                                  size_t capacity)
{
    if (device == nullptr || !m3_unary_views_ok(input, output) ||
        input->dtype != output->dtype) {
        return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                           "copy launch arguments are malformed");
    }
    if (output->element_count == 0U) {
        return M3_HIP_OK;
    }
    return m3_launch_unary(device, input, output, message, capacity);
}
