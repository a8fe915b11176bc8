/*
 * m3_hip_snake1d.hip - Snake1d activation for gfx950, bit-exact with the
 * CPU provider of the reference.
 *
 * Reference semantics (src/m3_op_execute_basic.c:182-215): for x[B, C, L]
 * and alpha[1, C, 1], every output element is the result of seven F32
 * statements, each rounded, with contraction off:
 *   d = a + 0x1.12e0bep-30 (bits 0x3089705f); inv = 1 / d; ang = a * x;
 *   s = sinf(ang); q = s * s; t = inv * q; y = x + t.
 * sinf is m3_sinf, the C library algorithm restated bit for bit; the
 * division is the IEEE F32 quotient; this file is compiled with
 * -ffp-contract=off so no statement fuses. inv depends only on the channel
 * and is formed once per lane and loop iteration when the lane's groups lie
 * in one channel, else once per group of four outputs (twice in a wave
 * where a channel ends inside a group).
 *
 * The vector kernel handles contiguous x and output of any length L of at
 * least 4, at any alignment, of about as many elements as the device has
 * lanes or more: a lane takes four consecutive elements, four groups in
 * flight. Smaller tensors and other layouts run per element over stride
 * tables.
 */
#include "m3_hip_internal.h"
#include "m3_libm.h"

#include <cstring>

namespace {

constexpr uint32_t kThreads = 256U;
constexpr uint32_t kUnroll = 4U;
/* Grid cap: 1,024 workgroups per CU, so the vector kernel runs one
 * workgroup per tile (1,024 groups of four elements) and the hardware
 * dispatcher spreads the tiles. Measured alternating in one process on
 * x[2,1536,65536]: 274 us against 292 us with 16 workgroups per CU. The
 * vector path takes fewer than 2^32 elements, so group indices plus one
 * grid stride (at most 2^28) stay below 2^32. */
constexpr uint32_t kBlocksPerCu = 1024U;
/* general against vector kernel (m3_least_elements): x[1,512,7] 2.8 and 3.8
 * us, [1,128,255] 2.8 and 4.2, [2,64,1001] 3.1 and 3.9, [2,192,1001] 4.1 and
 * 4.1, [2,192,2001] 5.8 and 3.8 */
constexpr uint32_t kVectorQuarters = 3U;

/* y = x + inverse * sin(a*x)^2 given sine = sin(a*x). */
__device__ __forceinline__ float m3_snake_finish(float x, float sine,
                                                 float inverse)
{
    float square = sine * sine;
    float scaled = inverse * square;

    return x + scaled;
}

__device__ __forceinline__ float m3_snake(float x, float a, float inverse)
{
    return m3_snake_finish(x, m3_sinf(a * x), inverse);
}

/* Four outputs, given each one's alpha and inverse. When no lane of the wave has an angle with
 * |a*x| >= 120 or a NaN angle (the common case by far), all four take the
 * branch-free sinf path, so the large-argument reduction costs one uniform
 * test per group instead of a divergent branch per element. That path
 * drops the sign of sinf: only its square is used, and the magnitude is
 * that of sinf for every |angle| < 120. */
__device__ __forceinline__ float4 m3_snake4(float4 x, float4 a,
                                            float4 inverse)
{
    const float4 angle =
        make_float4(a.x * x.x, a.y * x.y, a.z * x.z, a.w * x.w);
    /* one compare per element into a lane mask, the masks OR-ed as
     * scalars */
    const uint64_t large = __ballot(!(fabsf(angle.x) < 120.0F)) |
                           __ballot(!(fabsf(angle.y) < 120.0F)) |
                           __ballot(!(fabsf(angle.z) < 120.0F)) |
                           __ballot(!(fabsf(angle.w) < 120.0F));
    float4 sine;

    if (large != 0U) {
        sine = make_float4(m3_sinf(angle.x), m3_sinf(angle.y),
                           m3_sinf(angle.z), m3_sinf(angle.w));
    } else {
        sine = make_float4(m3_sinf_medium_magnitude(angle.x),
                           m3_sinf_medium_magnitude(angle.y),
                           m3_sinf_medium_magnitude(angle.z),
                           m3_sinf_medium_magnitude(angle.w));
    }
    return make_float4(m3_snake_finish(x.x, sine.x, inverse.x),
                       m3_snake_finish(x.y, sine.y, inverse.y),
                       m3_snake_finish(x.z, sine.z, inverse.z),
                       m3_snake_finish(x.w, sine.w, inverse.w));
}

__device__ __forceinline__ float m3_snake_inverse(float a)
{
    float denominator = a + m3_bits_f32(0x3089705fU);

    return 1.0F / denominator;
}

struct m3_snake_vec_args {
    const float *input;
    const uint8_t *alpha; /* alpha element of channel 0 */
    int64_t alpha_stride; /* bytes between channels */
    float *output;
    float *tanh_output;   /* tanhf of the output (TANH) */
    uint32_t groups;      /* elements / 4 */
    uint32_t tail;        /* elements % 4 */
    m3_fast_div length;   /* L >= 4 */
    m3_fast_div channels;
    m3_hip_gate list_gate;
};

__device__ __forceinline__ float4 m3_splat4(float v)
{
    return make_float4(v, v, v, v);
}

/* The alpha of row b*C + c. */
__device__ __forceinline__ float m3_snake_alpha(const m3_snake_vec_args &a,
                                                uint32_t row)
{
    const uint32_t channel =
        row - m3_fast_div_q(a.channels, row) * a.channels.divisor;

    return *(const float *)(a.alpha + (int64_t)channel * a.alpha_stride);
}

template <bool TANH>
__device__ __forceinline__ void m3_snake_put4(const m3_snake_vec_args &a,
                                              uint32_t g, float4 y)
{
    m3_stream_store((float4 *)a.output + g, y);
    if (TANH) {
        m3_stream_store((float4 *)a.tanh_output + g,
                        make_float4(m3_tanhf_uniform(y.x),
                                    m3_tanhf_uniform(y.y),
                                    m3_tanhf_uniform(y.z),
                                    m3_tanhf_uniform(y.w)));
    }
}

/* Groups of four consecutive elements, kUnroll per lane. L need not be a
 * multiple of 4: a group that a row's end cuts takes the next row's alpha
 * for its last elements, in the waves that hold one. Bound by HBM
 * (x[2,1536,65536] 264 us, 6.1 TB/s; x[2,192,60001] 30.5 us, 6.0 TB/s,
 * where one element per lane with 64-bit divisions took about 75). TANH:
 * tanhf of the output is stored too, in the launch of the TANH command
 * after it, which then does not read it back: 30.5 + 34.0 us for the two
 * over x[2,192,60001], 52.3 together, by then bound by instructions (100 per
 * element, 38 us of issue) as much as by HBM. */
template <bool TANH>
__global__ __launch_bounds__(256) void m3_snake1d_vec_kernel(
    m3_snake_vec_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint32_t step = gridDim.x * kThreads * kUnroll;

    for (uint32_t first = blockIdx.x * kThreads * kUnroll + threadIdx.x;
         first < a.groups; first += step) {
        const uint32_t last = first + (kUnroll - 1U) * kThreads;
        const uint32_t row = m3_fast_div_q(a.length, 4U * first);
        float4 x[kUnroll];

        /* The row b*C + c of an element is nondecreasing in its index, so
         * when a lane's first and last element share a row, all of them
         * do: one channel, one alpha and one division for the lane. */
        if (__all(last < a.groups &&
                  m3_fast_div_q(a.length, 4U * last + 3U) == row)) {
            const float alpha = m3_snake_alpha(a, row);

#pragma unroll
            for (uint32_t u = 0U; u < kUnroll; ++u) {
                x[u] = m3_stream_load((const float4 *)a.input + first +
                                      u * kThreads);
            }
            const float inverse = m3_snake_inverse(alpha);

#pragma unroll
            for (uint32_t u = 0U; u < kUnroll; ++u) {
                m3_snake_put4<TANH>(a, first + u * kThreads,
                                    m3_snake4(x[u], m3_splat4(alpha),
                                              m3_splat4(inverse)));
            }
            continue;
        }

        uint32_t rows[kUnroll];
        float alpha[kUnroll];
        /* the wave's groups before the end, in steps of kThreads */
        const uint32_t live =
            (a.groups -
             (uint32_t)__builtin_amdgcn_readfirstlane((int)first) +
             kThreads - 1U) /
            kThreads;

#pragma unroll
        for (uint32_t u = 0U; u < kUnroll; ++u) {
            const uint32_t g = min(first + u * kThreads, a.groups - 1U);

            rows[u] = m3_fast_div_q(a.length, 4U * g);
            x[u] = m3_stream_load((const float4 *)a.input + g);
            alpha[u] = m3_snake_alpha(a, rows[u]);
        }
#pragma unroll
        for (uint32_t u = 0U; u < kUnroll; ++u) {
            if (u >= live) {
                break; /* a wave past the end forms nothing */
            }
            const uint32_t at = first + u * kThreads;
            const uint32_t g = min(at, a.groups - 1U);
            /* elements of the group before the row's end */
            const uint32_t here =
                a.length.divisor - (4U * g - rows[u] * a.length.divisor);
            const float inverse = m3_snake_inverse(alpha[u]);
            float4 alpha4 = m3_splat4(alpha[u]);
            float4 inverse4 = m3_splat4(inverse);

            if (M3_ANY_LANE(here < 4U)) {
                /* every row has at least 4 elements: at most one end; a
                 * group it does not cut takes its own row again */
                const float other =
                    m3_snake_alpha(a, rows[u] + (here < 4U ? 1U : 0U));
                const float other_inverse = m3_snake_inverse(other);

                alpha4.y = here > 1U ? alpha4.y : other;
                alpha4.z = here > 2U ? alpha4.z : other;
                alpha4.w = here > 3U ? alpha4.w : other;
                inverse4.y = here > 1U ? inverse4.y : other_inverse;
                inverse4.z = here > 2U ? inverse4.z : other_inverse;
                inverse4.w = here > 3U ? inverse4.w : other_inverse;
            }
            const float4 y = m3_snake4(x[u], alpha4, inverse4);

            if (at < a.groups) {
                m3_snake_put4<TANH>(a, g, y);
            }
        }
    }
    if (blockIdx.x == 0U && threadIdx.x < a.tail) {
        /* the last elements % 4, in the last row */
        const uint64_t e = 4ULL * a.groups + threadIdx.x;
        const float alpha =
            m3_snake_alpha(a, m3_fast_div_q(a.length, (uint32_t)e));

        const float y =
            m3_snake(a.input[e], alpha, m3_snake_inverse(alpha));

        a.output[e] = y;
        if (TANH) {
            a.tanh_output[e] = m3_tanhf_uniform(y);
        }
    }
}

struct m3_snake_general_args {
    const uint8_t *input;
    const uint8_t *alpha;
    float *output;
    uint64_t count;
    uint64_t shape[3];
    int64_t input_strides[3];
    int64_t alpha_stride;
    m3_hip_gate list_gate;
};

__global__ __launch_bounds__(256) void m3_snake1d_general_kernel(
    m3_snake_general_args a)
{
    if (m3_gate_closed(a.list_gate)) {
        return; /* a check earlier in the list failed */
    }
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;

    for (uint64_t f = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
         f < a.count; f += step) {
        uint64_t l = f % a.shape[2];
        uint64_t rest = f / a.shape[2];
        uint64_t c = rest % a.shape[1];
        uint64_t b = rest / a.shape[1];
        float x = *(const float *)(a.input + (int64_t)b * a.input_strides[0] +
                                   (int64_t)c * a.input_strides[1] +
                                   (int64_t)l * a.input_strides[2]);
        float alpha = *(const float *)(a.alpha + (int64_t)c * a.alpha_stride);

        a.output[f] = m3_snake(x, alpha, m3_snake_inverse(alpha));
    }
}

} // namespace

/* True for the layouts of the vector kernel. */
static bool m3_snake_vector(const m3_hip_view *input,
                            const m3_hip_view *output)
{
    /* 32-bit element indices: below 2^32 with the lanes past the end (they
     * read the last group) */
    return m3_view_is_contiguous(input) && input->shape[2] >= 4U &&
           output->element_count < (1ULL << 32U);
}

/* SNAKE1D, and tanhf of its output into tanh_output when not null (which
 * the caller passes only for the vector kernel's layouts). */
static int m3_snake_launch(m3_hip_device *device, const m3_hip_view *input,
                           const m3_hip_view *alpha,
                           const m3_hip_view *output, float *tanh_output,
                           char *message, size_t capacity)
{
    if (device == nullptr || !m3_view_is_valid(input) ||
        !m3_view_is_valid(alpha) || !m3_view_is_valid(output) ||
        input->rank != 3U || alpha->rank != 3U || output->rank != 3U ||
        input->dtype != M3_HIP_F32 || alpha->dtype != M3_HIP_F32 ||
        output->dtype != M3_HIP_F32 || !m3_view_is_contiguous(output) ||
        alpha->shape[0] != 1U || alpha->shape[2] != 1U ||
        alpha->shape[1] != input->shape[1]) {
        return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                           "Snake1d launch arguments are malformed");
    }
    for (uint32_t axis = 0U; axis < 3U; ++axis) {
        if (input->shape[axis] != output->shape[axis]) {
            return m3_hip_fail(message, capacity, M3_HIP_INVALID,
                               "Snake1d input and output shapes differ");
        }
    }
    if (output->element_count == 0U) {
        return M3_HIP_OK;
    }
    const uint8_t *in = (const uint8_t *)input->base + input->byte_offset;
    const uint8_t *al = (const uint8_t *)alpha->base + alpha->byte_offset;
    uint8_t *out = (uint8_t *)output->base + output->byte_offset;
    uint64_t length = input->shape[2];
    int64_t alpha_stride = input->shape[1] > 1U
                               ? (int64_t)alpha->byte_strides[1]
                               : 0;

    /* With the TANH of the command after it the vector kernel saves a
     * launch, which counts for more than its lanes' turns. */
    if (m3_snake_vector(input, output) &&
        (tanh_output != nullptr ||
         output->element_count >= m3_least_elements(device, kVectorQuarters))) {
        m3_snake_vec_args args;

        std::memset(&args, 0, sizeof(args));
        args.list_gate = device->gate;
        args.input = (const float *)in;
        args.alpha = al;
        args.alpha_stride = alpha_stride;
        args.output = (float *)out;
        args.tanh_output = tanh_output;
        args.groups = (uint32_t)(output->element_count / 4U);
        args.tail = (uint32_t)(output->element_count % 4U);
        args.length = m3_fast_div_make((uint32_t)length);
        args.channels = m3_fast_div_make((uint32_t)input->shape[1]);
        uint32_t blocks = m3_grid_blocks(device, args.groups,
                                         kThreads * kUnroll, kBlocksPerCu);

        return m3_hip_launch(
            device, tanh_output != nullptr ? "m3_snake1d_tanh" : "m3_snake1d",
            [&](hipEvent_t start, hipEvent_t stop) {
                if (tanh_output != nullptr) {
                    hipExtLaunchKernelGGL((m3_snake1d_vec_kernel<true>),
                                          dim3(blocks), dim3(kThreads), 0,
                                          device->stream, start, stop, 0U,
                                          args);
                } else {
                    hipExtLaunchKernelGGL((m3_snake1d_vec_kernel<false>),
                                          dim3(blocks), dim3(kThreads), 0,
                                          device->stream, start, stop, 0U,
                                          args);
                }
            },
            message, capacity);
    }

    m3_snake_general_args general;

    std::memset(&general, 0, sizeof(general));
    general.list_gate = device->gate;
    general.input = in;
    general.alpha = al;
    general.output = (float *)out;
    general.count = output->element_count;
    for (uint32_t axis = 0U; axis < 3U; ++axis) {
        general.shape[axis] = input->shape[axis];
        general.input_strides[axis] = (int64_t)input->byte_strides[axis];
    }
    general.alpha_stride = alpha_stride;
    uint32_t blocks = m3_grid_blocks(device, general.count, 256U, 16U);

    return m3_hip_launch(
        device, "m3_snake1d_strided",
        [&](hipEvent_t start, hipEvent_t stop) {
            hipExtLaunchKernelGGL(m3_snake1d_general_kernel, dim3(blocks),
                                  dim3(256), 0, device->stream, start, stop,
                                  0U, general);
        },
        message, capacity);
}

extern "C" int m3_hip_launch_snake1d(m3_hip_device *device,
                                     const m3_hip_view *input,
                                     const m3_hip_view *alpha,
                                     const m3_hip_view *output,
                                     char *message, size_t capacity)
{
    return m3_snake_launch(device, input, alpha, output, nullptr, message,
                           capacity);
}

int m3_snake1d_tanh(m3_hip_device *device,
                    const m3_hip_chain_command *commands, int *taken,
                    char *message, size_t capacity)
{
    const m3_hip_view *input = &commands[0].left;
    const m3_hip_view *alpha = &commands[0].right;
    const m3_hip_view *output = &commands[0].output;
    const m3_hip_view *wave = &commands[1].output;

    /* shapes as m3_snake_launch checks them; the second output apart from
     * all the others, the first from alpha (in place over the input the
     * launch of SNAKE1D alone is as good) */
    if (!m3_view_is_valid(input) || !m3_view_is_valid(alpha) ||
        !m3_view_is_valid(output) || !m3_view_is_valid(wave) ||
        input->rank != 3U || output->rank != 3U ||
        output->element_count == 0U || wave->dtype != M3_HIP_F32 ||
        wave->element_count != output->element_count ||
        !m3_view_is_contiguous(wave) || !m3_snake_vector(input, output) ||
        m3_views_overlap(input, output) || m3_views_overlap(alpha, output) ||
        m3_views_overlap(input, wave) || m3_views_overlap(alpha, wave) ||
        m3_views_overlap(output, wave)) {
        return M3_HIP_OK;
    }
    *taken = 1;
    return m3_snake_launch(
        device, input, alpha, output,
        (float *)((uint8_t *)wave->base + wave->byte_offset), message,
        capacity);
}
