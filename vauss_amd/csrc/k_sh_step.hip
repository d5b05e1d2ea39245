// k_sh_step.hip -- the trainer's SH-coefficient step: lazy Adam on f16
// coefficients whose first moment is stored block-scaled in 8 bits, with the
// coefficient gradient rebuilt from the fused update's colour gradient and
// view direction; plus that moment's codec (encode, decode, zero rows).
//
// Restates crates/splat-train/src/optim.rs:391-498 (step_sh_color,
// step_quantized) and crates/splat-train/src/quant_kernels.rs:582-777
// (step_kernel_w4, sh_basis, stochastic_half), 438-498 (pack_block, unpack,
// encode/decode) and 911-925 (zero_moment_rows_kernel).
//
// Moment layout: the flat [N*K*3] values in blocks of 128; block b has one
// f32 scale (absmax / 127) and 32 u32 words of four biased 8-bit codes,
// value 4w+j in byte j of word w.  gfx950 mapping: one wave64 owns two
// blocks, each 32-lane half one block and each lane one word (four
// consecutive values), so a block's absmax is five steps inside the half-wave
// and needs no LDS or barrier.
#include "vs_device.h"
#include "vs_sh.h"
#include "vs_internal.h"

namespace vs {

constexpr uint32_t B8_VALUES = 128;            // quant.rs:15
constexpr uint32_t B8_WORDS = B8_VALUES / 4;   // one word per lane of a half-wave
constexpr int SH_STEP_BLOCK = 256;             // 4 waves = 8 moment blocks at a time
constexpr uint32_t SH_STEP_ROWS = 128;         // splats per workgroup: K*3 whole moment blocks at every degree

// quant_kernels.rs:866-894: round to one of the two f16 values adjacent to
// `value` with probability proportional to distance; a per-value, per-step
// integer hash gives 24 uniform bits.  Values beyond the f16 range (and NaN)
// pass through for the conversion to turn into infinities.
// Above the f16 subnormals (spacing 2^-24) the distance from the lower
// neighbour is the 13 bits f16 drops, so hash / 2^24 < distance / spacing is
// the integer comparison hash < bits * 2^11.
VS_DEV float stochastic_half(float value, uint32_t index, uint32_t step) {
    const float magnitude = __builtin_fabsf(value);
    uint32_t h = index ^ (step * 0x9e3779b9u);
    h = (h ^ (h >> 16)) * 0x7feb352du;
    h = (h ^ (h >> 15)) * 0x846ca68bu;
    h = (h ^ (h >> 16)) >> 8;
    const uint32_t bits = as_u(magnitude), dropped = bits & 0x1fffu;
    const float normal = as_f(bits - dropped + (h < (dropped << 11) ? 8192u : 0u));
    const float scaled = magnitude * 16777216.0f;
    const float below = __builtin_floorf(scaled);
    const float sub = ((float)h * 0x1p-24f < scaled - below ? below + 1.0f : below) * 0x1p-24f;
    const float r = magnitude < 6.103515625e-05f ? sub : normal;
    return !(magnitude <= 65504.0f) ? value : (value < 0.0f ? -r : r);
}

// 1 / b with the division's bits for 2^-60 <= |b| <= 2^60 (div_cr's sequence
// for a = 1, compared with the division at all such b).
VS_DEV float sh_recip(float b) {
    const float r0 = __builtin_amdgcn_rcpf(b);
    const float r1 = __builtin_fmaf(__builtin_fmaf(-b, r0, 1.0f), r0, r0);
    return __builtin_fmaf(__builtin_fmaf(-b, r1, 1.0f), r1, r1);
}

// a / b from r = 1 / b correctly rounded: the first correction brings the
// quotient within an ulp, and the second then rounds it correctly (Markstein)
// where no remainder underflows.
VS_DEV float sh_quotient(float a, float b, float r) {
    const float q0 = a * r;
    const float q1 = __builtin_fmaf(__builtin_fmaf(-b, q0, a), r, q0);
    return __builtin_fmaf(__builtin_fmaf(-b, q1, a), r, q1);
}

VS_DEV bool sh_mid_range(float v) {
    const float m = __builtin_fabsf(v);
    return m >= 0x1p-60f && m <= 0x1p60f;
}

// Block absmax over the 32 lanes of this half-wave (NaN-ignoring max).
// Rotations within 16 lanes, then the neighbouring 16.
template <int N>
VS_DEV float row_rotated(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xF, 0xF, false));
}
VS_DEV float half_wave_max(float v) {
    v = mx(v, row_rotated<8>(v));
    v = mx(v, row_rotated<4>(v));
    v = mx(v, row_rotated<2>(v));
    v = mx(v, row_rotated<1>(v));
    return mx(v, __shfl_xor(v, 16, 64));
}

// pack_block's code: round(clamp(m / scale, -127, 127)) + 128, 128 for a
// zero scale (ties to even).
VS_DEV uint32_t b8_code(float m, float scale) {
    if (!(scale > 0.0f)) return 128u;
    return (uint32_t)(__builtin_rintf(clampf(m / scale, -127.0f, 127.0f)) + 128.0f);
}

VS_DEV float b8_value(uint32_t word, int j, float scale) {
    return ((float)((word >> (8 * j)) & 255u) - 128.0f) * scale;
}

// step_kernel_w4 (quant_kernels.rs:582-727) and the second moment before it
// (optim.rs:447-469).  Values of culled splats keep their coefficient and
// moment; a block without a value of a visible splat is left untouched; every
// other block is re-packed from the stepped moments.
//
// A workgroup owns 128 splats and so whole moment blocks.  Its first 128 lanes
// take a splat each: the second moment (v beta2 + grad_sq (1 - beta2) for
// splats with gradients, kept for culled ones; at the first step
// grad_sq (1 - beta2) for all), the step's denominator and its reciprocal, and
// the row's K*3 gradients into LDS.  Then half-waves take its moment blocks.
// Bound by issue, not by its 0.3 GB at 1M splats of degree 3: with each word's
// lane evaluating its row's basis and picking four products, and a division a
// value for the step, the code and the rounding, it took 173 us and the
// second moment's own pass 5; now 118 us in all.
template <int DEG>
__global__ void __launch_bounds__(SH_STEP_BLOCK) sh_step_kernel(ShStepArgs a) {
    constexpr uint32_t K = sh_count<DEG>();
    constexpr uint32_t RW = K * 3;                        // values per splat row
    constexpr bool WHOLE = RW % 4 == 0;                   // a word's four values are one row's
    constexpr uint32_t STRIDE = WHOLE ? RW + 4 : RW;      // LDS floats per row: 16-byte stores (or odd) meet no bank twice
    constexpr float CULLED = -1.0f;                       // no denominator is negative
    __shared__ __attribute__((aligned(16))) float s_grad[SH_STEP_ROWS * STRIDE];
    __shared__ __attribute__((aligned(16))) float s_lr[RW];
    __shared__ float s_den[SH_STEP_ROWS], s_rden[SH_STEP_ROWS];
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t row0 = blockIdx.x * SH_STEP_ROWS;
    for (uint32_t i = t; i < RW; i += SH_STEP_BLOCK) s_lr[i] = a.lr_scale[i] * a.lr;
    if (t < SH_STEP_ROWS) {
        const uint32_t g = row0 + t;
        float den = CULLED;
        if (g < a.num_splats) {
            const uint32_t gr = a.grad_rows[g];
            if (gr != 0u || a.first) {
                const float c2 = 1.0f - a.beta2;
                const float gsq = a.grad_sq[g];
                const float v = a.first ? gsq * c2 : a.variance[g] * a.beta2 + gsq * c2;
                a.variance[g] = v;
                if (gr != 0u) den = __builtin_sqrtf(v * a.inv2) + a.epsilon;
            }
            if (gr != 0u) {
                const float* cd = a.color_dir + (size_t)gr * 6;
                const float c[3] = {cd[0], cd[1], cd[2]};
                float y[K], gv[RW];
                sh_basis<DEG>(F3{cd[3], cd[4], cd[5]}, y);
#pragma unroll
                for (uint32_t i = 0; i < RW; ++i) gv[i] = y[i / 3u] * c[i % 3u];
                float* out = s_grad + t * STRIDE;
                if constexpr (WHOLE) {
#pragma unroll
                    for (uint32_t i = 0; i < RW; i += 4)
                        *reinterpret_cast<float4*>(out + i) = make_float4(gv[i], gv[i + 1], gv[i + 2], gv[i + 3]);
                } else {
#pragma unroll
                    for (uint32_t i = 0; i < RW; ++i) out[i] = gv[i];
                }
            }
        }
        s_den[t] = den;
        s_rden[t] = sh_recip(den);
    }
    __syncthreads();

    const float factor = 1.0f - a.beta1;
    const uint32_t n = a.num_values;
    for (uint32_t w = t; w < SH_STEP_ROWS * RW / 4; w += SH_STEP_BLOCK) {
        const uint32_t block = blockIdx.x * RW + w / B8_WORDS;     // the whole half-wave agrees
        if (block >= a.num_blocks) break;
        const uint32_t local = w * 4u, first = row0 * RW + local;
        const uint32_t row_a = local / RW, row_b = WHOLE ? row_a : (local + 3u) / RW;
        const float den_a = s_den[row_a], den_b = WHOLE ? den_a : s_den[row_b];
        const bool any = den_a != CULLED || den_b != CULLED;       // rows past the end are culled ones
        const uint64_t ballot = __ballot(any);
        if ((uint32_t)(ballot >> (lane & 32u)) == 0u) continue;    // half-wave uniform: no shuffle below mixes halves

        const uint32_t word = block * B8_WORDS + (w & 31u);
        const float old_scale = a.scales[block];
        const uint32_t old = a.codes[word];
        float m[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) m[j] = WHOLE || first + j < n ? b8_value(old, j, old_scale) : 0.0f;
        if (WHOLE && first >= n) m[0] = m[1] = m[2] = m[3] = 0.0f;

        if (any) {
            uint16_t* p = a.sh + first;
            uint16_t ph[4];
            const bool whole = WHOLE || first + 3u < n;            // some value is live, so a whole row's word is inside
            if (whole) {
                const uint2 q = *reinterpret_cast<const uint2*>(p);
                ph[0] = (uint16_t)(q.x & 0xFFFFu); ph[1] = (uint16_t)(q.x >> 16);
                ph[2] = (uint16_t)(q.y & 0xFFFFu); ph[3] = (uint16_t)(q.y >> 16);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) ph[j] = first + j < n ? p[j] : (uint16_t)0;
            }
            const uint32_t col_a = local - row_a * RW;
            float gv[4], lr[4];
            if constexpr (WHOLE) {
                const float4 g4 = *reinterpret_cast<const float4*>(s_grad + row_a * STRIDE + col_a);
                const float4 l4 = *reinterpret_cast<const float4*>(s_lr + col_a);
                gv[0] = g4.x; gv[1] = g4.y; gv[2] = g4.z; gv[3] = g4.w;
                lr[0] = l4.x; lr[1] = l4.y; lr[2] = l4.z; lr[3] = l4.w;
            }
            const float rden_a = s_rden[row_a], rden_b = WHOLE ? rden_a : s_rden[row_b];
            float num[4], den[4], ratio[4];
            bool on[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool on_a = WHOLE || col_a + j < RW;
                den[j] = on_a ? den_a : den_b;
                on[j] = WHOLE || den[j] != CULLED;
                if (!WHOLE) {
                    gv[j] = on[j] ? s_grad[local + j] : 0.0f;      // a culled row's gradients are not written
                    lr[j] = s_lr[on_a ? col_a + j : col_a + j - RW];
                }
                const float moment = m[j] * a.beta1 + gv[j] * factor;
                num[j] = moment * a.inv1;
                m[j] = on[j] ? moment : m[j];
                ratio[j] = sh_quotient(num[j], den[j], on_a ? rden_a : rden_b);
            }
            // Zeros and NaNs come out of the sequence as of the division, but for a -0 that
            // turns to +0 (no coefficient tells them apart); the rest outside the range divides.
            const uint32_t least = min(min((as_u(num[0]) << 1) - 1u, (as_u(num[1]) << 1) - 1u),
                                       min((as_u(num[2]) << 1) - 1u, (as_u(num[3]) << 1) - 1u));
            const float most = mx(mx(__builtin_fabsf(num[0]), __builtin_fabsf(num[1])),
                                  mx(__builtin_fabsf(num[2]), __builtin_fabsf(num[3])));
            if (!(least >= (as_u(0x1p-60f) << 1) - 1u && most <= 0x1p60f && sh_mid_range(den_a) && sh_mid_range(den_b))) {
#pragma unroll
                for (int j = 0; j < 4; ++j) ratio[j] = num[j] / den[j];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float delta = ratio[j] * lr[j];
                const uint16_t stepped = f2h(stochastic_half(h2f(ph[j]) - delta, first + j, a.round_seed));
                ph[j] = on[j] ? stepped : ph[j];
            }
            if (whole) {
                *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)ph[0] | ((uint32_t)ph[1] << 16),
                                                          (uint32_t)ph[2] | ((uint32_t)ph[3] << 16));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (first + j < n) p[j] = ph[j];
            }
        }
        const float top = mx(mx(__builtin_fabsf(m[0]), __builtin_fabsf(m[1])),
                             mx(__builtin_fabsf(m[2]), __builtin_fabsf(m[3])));
        const float scale = half_wave_max(top) / 127.0f;
        if ((lane & 31u) == 0u) a.scales[block] = scale;
        uint32_t packed = 0u;
        if (sh_mid_range(scale)) {
            // quotients small enough for a remainder to underflow all round to code 128
            const float r = sh_recip(scale);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                packed = __builtin_amdgcn_cvt_pk_u8_f32(
                    __builtin_rintf(clampf(sh_quotient(m[j], scale, r), -127.0f, 127.0f)) + 128.0f, j, packed);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) packed |= b8_code(m[j], scale) << (8 * j);
        }
        a.codes[word] = packed;
    }
}

// encode_kernel / pack_block (quant_kernels.rs:438-484): values past n are 0.
__global__ void __launch_bounds__(SH_STEP_BLOCK) b8_encode_kernel(const float* __restrict__ values, uint32_t n,
                                                                  uint32_t num_blocks, uint32_t* __restrict__ codes,
                                                                  float* __restrict__ scales) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t block = (blockIdx.x * SH_STEP_BLOCK + threadIdx.x) >> 5;
    if (block >= num_blocks) return;              // half-wave uniform
    const uint32_t word = block * B8_WORDS + (lane & 31u);
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = word * 4u + j < n ? values[word * 4u + j] : 0.0f;
    const float local = mx(mx(__builtin_fabsf(v[0]), __builtin_fabsf(v[1])), mx(__builtin_fabsf(v[2]), __builtin_fabsf(v[3])));
    const float scale = half_wave_max(local) / 127.0f;
    if ((lane & 31u) == 0u) scales[block] = scale;
    uint32_t packed = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) packed |= b8_code(v[j], scale) << (8 * j);
    codes[word] = packed;
}

// decode_kernel / unpack (quant_kernels.rs:486-498).
__global__ void b8_decode_kernel(const uint32_t* __restrict__ codes, const float* __restrict__ scales, uint32_t n,
                                 float* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = b8_value(codes[i / 4u], (int)(i % 4u), scales[i / B8_VALUES]);
}

// zero_moment_rows_kernel (quant_kernels.rs:911-925): each value of the
// listed rows gets the zero code 128; rows may share words, so the byte is
// cleared and set with two word atomics that touch only it.  Values past n
// are ignored.
__global__ void b8_zero_rows_kernel(uint32_t* __restrict__ codes, uint32_t n, const uint32_t* __restrict__ rows,
                                    uint32_t num_rows, uint32_t row_width) {
    const uint64_t pos = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (pos >= (uint64_t)num_rows * row_width) return;
    const uint64_t idx = (uint64_t)rows[pos / row_width] * row_width + pos % row_width;
    if (idx >= n) return;
    const uint32_t shift = (uint32_t)(idx % 4u) * 8u;
    atomicAnd(codes + idx / 4u, ~(255u << shift));
    atomicOr(codes + idx / 4u, 128u << shift);
}

hipError_t launch_sh_step(const ShStepArgs& a, hipStream_t s) {
    if (a.num_splats == 0) return hipSuccess;
    const uint32_t grid = (a.num_splats + SH_STEP_ROWS - 1) / SH_STEP_ROWS;
    switch (a.sh_degree) {
    case 0: sh_step_kernel<0><<<grid, SH_STEP_BLOCK, 0, s>>>(a); break;
    case 1: sh_step_kernel<1><<<grid, SH_STEP_BLOCK, 0, s>>>(a); break;
    case 2: sh_step_kernel<2><<<grid, SH_STEP_BLOCK, 0, s>>>(a); break;
    case 3: sh_step_kernel<3><<<grid, SH_STEP_BLOCK, 0, s>>>(a); break;
    default: sh_step_kernel<4><<<grid, SH_STEP_BLOCK, 0, s>>>(a); break;
    }
    return hipGetLastError();
}

hipError_t launch_b8_encode(const float* values, uint32_t n, uint32_t* codes, float* scales, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint32_t blocks = (n + B8_VALUES - 1) / B8_VALUES;
    b8_encode_kernel<<<(blocks + SH_STEP_BLOCK / 32 - 1) / (SH_STEP_BLOCK / 32), SH_STEP_BLOCK, 0, s>>>(
        values, n, blocks, codes, scales);
    return hipGetLastError();
}

hipError_t launch_b8_decode(const uint32_t* codes, const float* scales, uint32_t n, float* values, hipStream_t s) {
    if (n == 0) return hipSuccess;
    b8_decode_kernel<<<(n + 255) / 256, 256, 0, s>>>(codes, scales, n, values);
    return hipGetLastError();
}

hipError_t launch_b8_zero_rows(uint32_t* codes, uint32_t n, const uint32_t* rows, uint32_t num_rows,
                               uint32_t row_width, hipStream_t s) {
    const uint64_t total = (uint64_t)num_rows * row_width;
    if (total == 0) return hipSuccess;
    b8_zero_rows_kernel<<<(uint32_t)((total + 255) / 256), 256, 0, s>>>(codes, n, rows, num_rows, row_width);
    return hipGetLastError();
}

} // namespace vs
