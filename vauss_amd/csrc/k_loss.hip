// k_loss.hip -- the image loss after the render: L1 + SSIM over an [H,W,C]
// f32 prediction and RGBA8-packed ground truth, its per-tile partial sums,
// and its gradient.
//
// Restates crates/splat-train-loss/src/lib.rs: image_loss_forward_kernel
// (:238-478) and image_loss_backward_coeffs_kernel (:821-1020).  SSIM uses an
// 11-tap Gaussian window (sigma 1.5) applied separably with zero padding,
// C1 = 0.01^2, C2 = 0.03^2, clamped to [-1, 1]; the per-pixel loss is
// l1_w |p - g| + ssim_w SSIM (ssim_w negative for training), optionally
// times gt.a (mask), with g composited over a background when asked.  The
// forward also keeps, per pixel and channel, the partials of SSIM w.r.t. the
// blurred moments (<x>, <x^2>, <xy>), so the backward blurs chain x partial
// once instead of re-running the forward's blurs.
//
// Sums follow one fixed order everywhere (per tap distance d = 1..5 add
// (left + right) * w, then the centre; rows, then columns; tile sums by a
// halving tree), which the CPU restatement repeats bit for bit.  That order
// leaves 17 unfused operations per blurred value and direction, so both
// kernels are bound by VALU issue, not by memory, and are built to do nothing
// but those: one wavefront marches down a strip of 64 columns for one colour
// channel, blurs each input row once (taps from a row buffer in LDS that only
// this wavefront touches: no barrier), and keeps the last eleven row blurs in
// registers for the column blur, so no blurred value passes through LDS.  The
// three channels of a strip share a workgroup and, through its CU's cache,
// their pixels.  (One 256-lane workgroup per 16x16 tile, both blurs through
// LDS: 3840x2160 RGBA with mask and alpha, forward 394 and backward 284 us;
// this form 250 and 170.)
#include <algorithm>
#include "vs_device.h"
#include "vs_internal.h"

namespace vs {

// gauss_taps() (lib.rs:48-62) in f32: exp(-x^2 / 4.5) rounded to f32, divided
// by their f32 sum.
__device__ constexpr float LGW[6] = {0x1.0d957p-10f, 0x1.f1fe04p-8f, 0x1.26eb18p-5f, 0x1.bff1p-4f, 0x1.b43c4p-3f,
                                     0x1.106562p-2f};
constexpr float LOSS_C1 = 0.01f * 0.01f;
constexpr float LOSS_C2 = 0.03f * 0.03f;
constexpr float LOSS_INV_255 = 1.0f / 255.0f;
constexpr int LT = 16;              // tile edge of the partial sums
constexpr int LH = 5;               // window half width
constexpr int LTAPS = 2 * LH + 1;
constexpr int LW = 64;              // strip width: one column per lane
constexpr int LROW = LW + 2 * LH;   // a strip's input row
constexpr int LBLOCK = 3 * 64;      // one wavefront per colour channel

__device__ __forceinline__ float gt_byte(uint32_t v, uint32_t c) { return (float)((v >> (c * 8u)) & 0xffu) * LOSS_INV_255; }

template <bool COMPOSITE>
__device__ __forceinline__ float gt_eff(uint32_t v, uint32_t c, const LossArgs& a) {
    const float g = gt_byte(v, c);
    if constexpr (COMPOSITE) return g + (1.0f - gt_byte(v, 3)) * a.bg[c];
    return g;
}

// A row of `bytes` bytes at a uniform pointer as a buffer: lanes address it by
// a 32-bit byte offset (no 64-bit lane arithmetic), loads past its end give 0
// and stores past it are dropped, so a lane or a row outside the image needs
// no branch (ROW_OUT, or a row of no bytes).
using RowBuf = __amdgpu_buffer_rsrc_t;
constexpr uint32_t ROW_OUT = 0xFFFFFFF0u;
__device__ __forceinline__ RowBuf row_buf(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000);
}
__device__ __forceinline__ uint32_t row_u32(RowBuf r, uint32_t byte) { return __builtin_amdgcn_raw_buffer_load_b32(r, byte, 0, 0); }
__device__ __forceinline__ float row_f32(RowBuf r, uint32_t byte) { return as_f(row_u32(r, byte)); }
__device__ __forceinline__ void row_put(RowBuf r, uint32_t byte, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(as_u(v), r, byte, 0, 0);
}

// Orders a wavefront's own LDS stores before its later loads of other lanes'
// slots (LDS executes a wavefront's operations in order; this holds the
// compiler to it).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// 1 / b with the division's bits for 2^-100 <= |b| <= 2^100 (div_cr with
// a = 1, compared with the division at all such b); num * recip_cr(b) with one
// remainder correction is then num / b correctly rounded (Markstein), unless
// the remainder underflows.
__device__ __forceinline__ float recip_cr(float b) {
    const float r0 = __builtin_amdgcn_rcpf(b);
    const float r1 = __builtin_fmaf(__builtin_fmaf(-b, r0, 1.0f), r0, r0);
    return __builtin_fmaf(__builtin_fmaf(-b, r1, 1.0f), r1, r1);
}

// One tap pair of a blur: s += (left + right) * w.  FIRST starts the sum at
// +0; a sum of squares (SQ) cannot be -0, so its first term stands alone.
template <bool FIRST, bool SQ>
__device__ __forceinline__ void tap(float& s, float l, float r, float w) {
    const float t = (l + r) * w;
    s = FIRST ? (SQ ? t : 0.0f + t) : s + t;
}

template <int N>
__device__ __forceinline__ float row_ror(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xF, 0xF, false));
}

// Sum of a 16x16 tile's 256 values by the halving tree over row * 16 + column:
// lane l's column holds s[row * LW + l]; rows r and r + 8, + 4, + 2, + 1, then
// columns c and c + 8, + 4, + 2, + 1 (addition commutes and the halves repeat, so
// rotations within the tile's 16 lanes leave the tree's sum in each).
__device__ __forceinline__ float tile_tree(const float* s, uint32_t lane) {
    float v[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r] = s[r * LW + lane] + s[(r + 8) * LW + lane];
#pragma unroll
    for (int step = 4; step >= 1; step >>= 1)
#pragma unroll
        for (int r = 0; r < step; ++r) v[r] += v[r + step];
    float t = v[0];
    t += row_ror<8>(t);
    t += row_ror<4>(t);
    t += row_ror<2>(t);
    t += row_ror<1>(t);
    return t;
}

template <bool COMPOSITE, bool MASK, bool ALPHA>
__global__ void __launch_bounds__(LBLOCK) loss_fwd_kernel(LossArgs a, uint32_t strip) {
    __shared__ float4 s_row[3][2][LROW];             // x = pred, y = effective gt, x^2, y^2 of the current input row
    __shared__ float s_xy[3][2][LROW];               // x y
    __shared__ float s_lv[3][LT * LW];               // a tile row's loss values
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t w = a.img_w, h = a.img_h, cn = a.channels;
    const int x0 = (int)(blockIdx.x * LW);
    const uint32_t y0 = blockIdx.y * strip;
    const uint32_t rows_out = min(strip, h - y0);
    const uint32_t steps = rows_out + 2 * LH;
    const size_t plane = (size_t)h * w;
    const uint32_t px = (uint32_t)x0 + lane;
    const bool in = px < w;
    const uint32_t tiles_x = (w + LT - 1) / LT, T = tiles_x * ((h + LT - 1) / LT);
    float* s_mine = s_lv[c];

    // input row y0 - 5 + i: this lane's column x0 - 5 + lane, lanes below ten
    // also column x0 + 59 + lane; 0 outside the image
    const int ca = x0 - LH + (int)lane, cb = x0 + LW - LH + (int)lane;
    const bool in_a = ca >= 0 && ca < (int)w, in_b = lane < 2u * LH && cb < (int)w;
    const uint32_t la = in_a ? 4u * (uint32_t)ca : ROW_OUT, lb = in_b ? 4u * (uint32_t)cb : ROW_OUT;
    const uint32_t pla = in_a ? 4u * ((uint32_t)ca * cn + c) : ROW_OUT, plb = in_b ? 4u * ((uint32_t)cb * cn + c) : ROW_OUT;
    float pa, pb;
    uint32_t ga, gb;
    auto fetch = [&](uint32_t i) {
        const int y = (int)y0 - LH + (int)i;            // uniform
        const bool row_in = y >= 0 && y < (int)h;
        const size_t at = row_in ? (size_t)y * w : 0;
        const RowBuf pr = row_buf(a.pred + at * cn, row_in ? w * cn * 4u : 0u), gr = row_buf(a.gt + at, row_in ? w * 4u : 0u);
        pa = row_f32(pr, pla); pb = row_f32(pr, plb);
        ga = row_u32(gr, la); gb = row_u32(gr, lb);
    };
    fetch(0);

    float hx[LTAPS], hxx[LTAPS], hy[LTAPS], hyy[LTAPS], hxy[LTAPS];   // row blurs, input row i at slot i % 11
    float l1[LTAPS];                                                  // |pred - gt| at the lane's column
    for (uint32_t base = 0; base < steps; base += LTAPS) {
#pragma unroll
        for (int j = 0; j < LTAPS; ++j) {
            const uint32_t i = base + (uint32_t)j;
            if (i >= steps) break;                      // uniform
            float4* row = s_row[c][i & 1u];
            float* rxy = s_xy[c][i & 1u];
            const int yi = (int)y0 - LH + (int)i;
            const bool row_in = yi >= 0 && yi < (int)h;  // uniform
            // a background shows through a zero word, so compositing needs the outside zeroed
            auto effective = [&](uint32_t v, bool inside) {
                const float g = gt_eff<COMPOSITE>(v, c, a);
                return COMPOSITE && !(row_in && inside) ? 0.0f : g;
            };
            const float xa = pa, ya = effective(ga, in_a);
            row[lane] = make_float4(xa, ya, xa * xa, ya * ya);
            rxy[lane] = xa * ya;
            if (lane < 2u * LH) {
                const float xb = pb, yb = effective(gb, in_b);
                row[LW + lane] = make_float4(xb, yb, xb * xb, yb * yb);
                rxy[LW + lane] = xb * yb;
            }
            fetch(i + 1u);
            wave_lds_fence();
            {
                float sx, sxx, sy, syy, sxy;
#pragma unroll
                for (int d = 1; d <= LH; ++d) {
                    const float4 L = row[lane + LH - d], R = row[lane + LH + d];
                    const float lxy = rxy[lane + LH - d], rxy_ = rxy[lane + LH + d];
                    const float wd = LGW[5 - d];
                    if (d == 1) {
                        tap<true, false>(sx, L.x, R.x, wd);
                        tap<true, false>(sy, L.y, R.y, wd);
                        tap<true, true>(sxx, L.z, R.z, wd);
                        tap<true, true>(syy, L.w, R.w, wd);
                        tap<true, false>(sxy, lxy, rxy_, wd);
                    } else {
                        tap<false, false>(sx, L.x, R.x, wd);
                        tap<false, false>(sy, L.y, R.y, wd);
                        tap<false, true>(sxx, L.z, R.z, wd);
                        tap<false, true>(syy, L.w, R.w, wd);
                        tap<false, false>(sxy, lxy, rxy_, wd);
                    }
                }
                const float4 M = row[lane + LH];
                const float wc = LGW[5];
                hx[j] = sx + M.x * wc;
                hxx[j] = sxx + M.z * wc;
                hy[j] = sy + M.y * wc;
                hyy[j] = syy + M.w * wc;
                hxy[j] = sxy + rxy[lane + LH] * wc;
                l1[j] = __builtin_fabsf(M.x - M.y);
            }
            if (i < 2u * LH) continue;                  // uniform: the window is not full yet
            const uint32_t o = i - 2u * LH;             // output row of the strip
            const size_t pix = (size_t)(y0 + o) * w + px;
            auto column = [&](const float (&v)[LTAPS], bool sq) {
                float s;
#pragma unroll
                for (int d = 1; d <= LH; ++d) {
                    const float u = v[(j + LTAPS - LH - d) % LTAPS], l = v[(j + LTAPS - LH + d) % LTAPS];
                    if (d == 1) { if (sq) tap<true, true>(s, u, l, LGW[5 - d]); else tap<true, false>(s, u, l, LGW[5 - d]); }
                    else tap<false, false>(s, u, l, LGW[5 - d]);
                }
                return s + v[(j + LTAPS - LH) % LTAPS] * LGW[5];
            };
            const float mu1 = column(hx, false), m11 = column(hxx, true), mu2 = column(hy, false);
            const float m22 = column(hyy, true), m12 = column(hxy, false);
            float lv = 0.0f;
            if (in) {
                const float mu1_sq = mu1 * mu1, mu2_sq = mu2 * mu2;
                const float sigma1_sq = mx(0.0f, m11 - mu1_sq);
                const float sigma2_sq = mx(0.0f, m22 - mu2_sq);
                const float sigma12 = m12 - mu1 * mu2;
                const float A = mu1_sq + mu2_sq + LOSS_C1;
                const float B = sigma1_sq + sigma2_sq + LOSS_C2;
                const float c_top = 2.0f * mu1 * mu2 + LOSS_C1;
                const float d_top = 2.0f * sigma12 + LOSS_C2;
                const float num = c_top * d_top, ab = A * B;
                float q, inv_ab, inv_b;                 // num / ab, 1 / ab and 1 / B, each the division's bits
                if (ab <= 0x1p60f && __builtin_fabsf(num) >= 0x1p-40f) {
                    // A >= C1 and B >= C2 bound ab and B from below
                    inv_ab = recip_cr(ab);
                    inv_b = recip_cr(B);
                    const float q0 = num * inv_ab;
                    q = __builtin_fmaf(__builtin_fmaf(-ab, q0, num), inv_ab, q0);
                } else {
                    q = num / ab;
                    inv_ab = 1.0f / ab;
                    inv_b = 1.0f / B;
                }
                const float val = clampf(q, -1.0f, 1.0f);
                if (a.coeffs) {
                    const float cd = c_top * d_top * inv_ab;
                    const bool clamped = cd < -1.0f || cd > 1.0f;
                    float* co = a.coeffs + (size_t)c * 3 * plane + (size_t)(y0 + o) * w;     // uniform
                    row_put(row_buf(co, w * 4u), 4u * px, clamped ? 0.0f : 2.0f * inv_ab * (mu2 * (d_top - c_top) - mu1 * cd * (B - A)));
                    row_put(row_buf(co + plane, w * 4u), 4u * px, clamped ? 0.0f : -cd * inv_b);
                    row_put(row_buf(co + 2 * plane, w * 4u), 4u * px, clamped ? 0.0f : 2.0f * c_top * inv_ab);
                }
                lv = a.l1_weight * l1[(j + LTAPS - LH) % LTAPS] + a.ssim_weight * val;
                if constexpr (MASK) lv = lv * gt_byte(row_u32(row_buf(a.gt + (size_t)(y0 + o) * w, w * 4u), 4u * px), 3);
                if (a.loss_map) a.loss_map[pix * cn + c] = lv;
            }
            if (a.partials) {
                s_mine[(o % LT) * LW + lane] = lv;
                if (o % LT == LT - 1u || o + 1u == rows_out) {          // uniform: a tile row is complete
                    for (uint32_t r = o % LT + 1u; r < LT; ++r) s_mine[r * LW + lane] = 0.0f;
                    wave_lds_fence();
                    const float t = tile_tree(s_mine, lane);
                    const uint32_t tile_x = px / LT;
                    if (lane % LT == 0u && in)
                        a.partials[(size_t)c * T + (size_t)((y0 + o) / LT) * tiles_x + tile_x] = t * a.rgb_weight;
                    wave_lds_fence();
                }
            }
        }
    }
    if constexpr (ALPHA) {
        // lib.rs:266-285: |pred.a - gt.a| (times gt.a when masking), no blur;
        // the strip's tile rows are dealt to the three wavefronts
        for (uint32_t t0 = c * LT; t0 < rows_out; t0 += 3u * LT) {
#pragma unroll
            for (uint32_t r = 0; r < LT; ++r) {
                float v = 0.0f;
                if (in && t0 + r < rows_out) {
                    const size_t pix = (size_t)(y0 + t0 + r) * w + px;
                    const float g = gt_byte(a.gt[pix], 3);
                    v = __builtin_fabsf(a.pred[pix * cn + 3] - g);
                    if constexpr (MASK) v = v * g;
                    if (a.loss_map) a.loss_map[pix * cn + 3] = v;
                }
                s_mine[r * LW + lane] = v;
            }
            wave_lds_fence();
            if (a.partials) {
                const float t = tile_tree(s_mine, lane);
                if (lane % LT == 0u && in)
                    a.partials[(size_t)3 * T + (size_t)((y0 + t0) / LT) * tiles_x + px / LT] = t * a.alpha_weight;
            }
            wave_lds_fence();
        }
    }
}

template <bool COMPOSITE, bool MASK, bool ALPHA, bool SCALAR>
__global__ void __launch_bounds__(LBLOCK) loss_bwd_kernel(LossBwdArgs a, uint32_t strip) {
    __shared__ float2 s_row[3][2][LROW];             // chain x coefficients 0, 1 of the current input row
    __shared__ float s_row2[3][2][LROW];             // chain x coefficient 2
    __shared__ float s_out[LT][LW * 4];              // a tile row's gradients, channel-interleaved
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t w = a.img_w, h = a.img_h, cn = a.channels;
    const int x0 = (int)(blockIdx.x * LW);
    const uint32_t y0 = blockIdx.y * strip;
    const uint32_t rows_out = min(strip, h - y0);
    const uint32_t steps = rows_out + 2 * LH;
    const size_t plane = (size_t)h * w;
    const uint32_t px = (uint32_t)x0 + lane;
    const bool in = px < w;
    const uint32_t tiles_x = (w + LT - 1) / LT, T = tiles_x * ((h + LT - 1) / LT);

    // chain_at (lib.rs:141-159): the upstream gradient of a pixel's tile sum times its weight.
    const float dl0 = SCALAR ? a.dl[0] : 0.0f;
    auto chain_at = [&](uint32_t ch, uint32_t y, uint32_t x, float weight) {
        const float g = SCALAR ? dl0 : a.dl[(size_t)ch * T + (y / LT) * tiles_x + x / LT];
        return g * weight;
    };
    // the input row's values as loaded (0 outside the image), one row ahead;
    // they are scaled when stored to LDS
    const int ca = x0 - LH + (int)lane, cb = x0 + LW - LH + (int)lane;
    const bool in_a = ca >= 0 && ca < (int)w, in_b = lane < 2u * LH && cb < (int)w;
    const uint32_t la = in_a ? 4u * (uint32_t)ca : ROW_OUT, lb = in_b ? 4u * (uint32_t)cb : ROW_OUT;
    const uint32_t lx = in ? 4u * px : ROW_OUT, plx = in ? 4u * (px * cn + c) : ROW_OUT;
    const float* co = a.coeffs + (size_t)c * 3 * plane;
    float va[3], vb[3], ch_a = 0.0f, ch_b = 0.0f, p1 = 0.0f, p_alpha = 0.0f;
    uint32_t ma = 0u, mb = 0u, gv = 0u;
    auto fetch = [&](uint32_t i) {
        const int y = (int)y0 - LH + (int)i;            // uniform
        const bool row_in = y >= 0 && y < (int)h;
        const float* cr = co + (row_in ? (size_t)y * w : 0);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const RowBuf r = row_buf(cr + (size_t)k * plane, row_in ? w * 4u : 0u);
            va[k] = row_f32(r, la); vb[k] = row_f32(r, lb);
        }
        if constexpr (MASK) {
            const RowBuf r = row_buf(a.gt + (row_in ? (size_t)y * w : 0), row_in ? w * 4u : 0u);
            ma = row_u32(r, la); mb = row_u32(r, lb);
        }
        if constexpr (!SCALAR) {
            const uint32_t yc = (uint32_t)min(max(y, 0), (int)h - 1);
            ch_a = chain_at(c, yc, in_a ? (uint32_t)ca : 0u, a.rgb_weight);
            ch_b = chain_at(c, yc, in_b ? (uint32_t)cb : 0u, a.rgb_weight);
        }
        // the output row of that step
        const int yo = y - LH;
        const bool out_in = yo >= 0 && yo < (int)h;
        const size_t at = out_in ? (size_t)yo * w : 0;
        const RowBuf pr = row_buf(a.pred + at * cn, out_in ? w * cn * 4u : 0u);
        p1 = row_f32(pr, plx);
        if constexpr (ALPHA) p_alpha = row_f32(pr, in ? px * 16u + 12u : ROW_OUT);        // ALPHA only with four channels
        gv = row_u32(row_buf(a.gt + at, out_in ? w * 4u : 0u), lx);
    };
    fetch(0);

    float h0[LTAPS], h1[LTAPS], h2[LTAPS];           // row blurs, input row i at slot i % 11
    for (uint32_t base = 0; base < steps; base += LTAPS) {
#pragma unroll
        for (int j = 0; j < LTAPS; ++j) {
            const uint32_t i = base + (uint32_t)j;
            if (i >= steps) break;                      // uniform
            float2* row = s_row[c][i & 1u];
            float* row2 = s_row2[c][i & 1u];
            const int yi = (int)y0 - LH + (int)i;
            const bool row_in = yi >= 0 && yi < (int)h;  // uniform
            {
                float fa = SCALAR ? chain_at(c, 0u, 0u, a.rgb_weight) : ch_a, fb = SCALAR ? fa : ch_b;
                if constexpr (MASK) { fa = fa * gt_byte(ma, 3); fb = fb * gt_byte(mb, 3); }
                const bool za = row_in && in_a, zb = row_in && in_b;      // outside: 0 whatever the chain is
                row[lane] = make_float2(za ? va[0] * fa : 0.0f, za ? va[1] * fa : 0.0f);
                row2[lane] = za ? va[2] * fa : 0.0f;
                if (lane < 2u * LH) {
                    row[LW + lane] = make_float2(zb ? vb[0] * fb : 0.0f, zb ? vb[1] * fb : 0.0f);
                    row2[LW + lane] = zb ? vb[2] * fb : 0.0f;
                }
            }
            // this step's output pixel
            const uint32_t o = i - 2u * LH;
            const bool out_row = i >= 2u * LH;          // uniform
            const float po = p1, pao = p_alpha;
            const uint32_t go = gv;
            fetch(i + 1u);
            wave_lds_fence();
            {
                float s0, s1, s2;
#pragma unroll
                for (int d = 1; d <= LH; ++d) {
                    const float2 L = row[lane + LH - d], R = row[lane + LH + d];
                    const float l2 = row2[lane + LH - d], r2 = row2[lane + LH + d];
                    const float wd = LGW[5 - d];
                    if (d == 1) {
                        tap<true, false>(s0, L.x, R.x, wd);
                        tap<true, false>(s1, L.y, R.y, wd);
                        tap<true, false>(s2, l2, r2, wd);
                    } else {
                        tap<false, false>(s0, L.x, R.x, wd);
                        tap<false, false>(s1, L.y, R.y, wd);
                        tap<false, false>(s2, l2, r2, wd);
                    }
                }
                const float2 M = row[lane + LH];
                h0[j] = s0 + M.x * LGW[5];
                h1[j] = s1 + M.y * LGW[5];
                h2[j] = s2 + row2[lane + LH] * LGW[5];
            }
            if (!out_row) continue;
            auto column = [&](const float (&v)[LTAPS]) {
                float s;
#pragma unroll
                for (int d = 1; d <= LH; ++d) {
                    const float u = v[(j + LTAPS - LH - d) % LTAPS], l = v[(j + LTAPS - LH + d) % LTAPS];
                    if (d == 1) tap<true, false>(s, u, l, LGW[5 - d]); else tap<false, false>(s, u, l, LGW[5 - d]);
                }
                return s + v[(j + LTAPS - LH) % LTAPS] * LGW[5];
            };
            const float g0 = column(h0), g1 = column(h1), g2 = column(h2);
            const uint32_t r = o % LT;
            if (in) {
                const float ge = gt_eff<COMPOSITE>(go, c, a.fwd);
                const float ssim_grad = g0 + (2.0f * po) * g1 + ge * g2;
                const float diff = po - ge;
                const float sign = diff > 0.0f ? 1.0f : (diff < 0.0f ? -1.0f : 0.0f);
                float cc = chain_at(c, y0 + o, px, a.rgb_weight);
                if constexpr (MASK) cc = cc * gt_byte(go, 3);
                s_out[r][lane * cn + c] = a.fwd.ssim_weight * ssim_grad + a.fwd.l1_weight * sign * cc;
                if (c == 2u && cn == 4u) {
                    float ag = 0.0f;
                    if constexpr (ALPHA) {
                        const float gal = gt_byte(go, 3);
                        const float da = pao - gal;
                        const float sa = da > 0.0f ? 1.0f : (da < 0.0f ? -1.0f : 0.0f);
                        float chain = chain_at(3, y0 + o, px, a.alpha_weight);
                        if constexpr (MASK) chain = chain * gal;
                        ag = sa * chain;
                    }
                    s_out[r][lane * 4 + 3] = ag;
                }
            }
            if (r == LT - 1u || o + 1u == rows_out) {   // uniform over the workgroup: store the tile row's pixels
                __syncthreads();
                const uint32_t cols = min((uint32_t)LW, w - (uint32_t)x0), first = y0 + o - r;
                if (cn == 4u) {
                    for (uint32_t k = threadIdx.x; k < (r + 1u) * LW; k += LBLOCK) {
                        const uint32_t ry = k / LW, rx = k % LW;
                        if (rx < cols)
                            reinterpret_cast<float4*>(a.dl_dpred)[(size_t)(first + ry) * w + x0 + rx] =
                                *reinterpret_cast<const float4*>(&s_out[ry][rx * 4]);
                    }
                } else {
                    for (uint32_t ry = 0; ry <= r; ++ry)
                        for (uint32_t k = threadIdx.x; k < cols * 3u; k += LBLOCK)
                            a.dl_dpred[((size_t)(first + ry) * w + x0) * 3 + k] = s_out[ry][k];
                }
                __syncthreads();
            }
        }
    }
}

// The total of the weighted tile partials: one 1024-lane block, sixteen values
// (four 16-byte loads where the buffer allows) in flight per lane, then a
// wave64 butterfly and a 16-entry LDS sum.  The block is bound by the latency
// of its loads (97k partials of a 3840x2160 RGBA image: 24 us with four
// values in flight, 10 with sixteen).  The summation order is fixed but
// differs from the tile tree's; the total is a convenience (the partials are
// the exact outputs).
constexpr int TOTAL_BLOCK = 1024;
__global__ void __launch_bounds__(TOTAL_BLOCK) loss_total_kernel(const float* __restrict__ partials, uint32_t n,
                                                                 float* __restrict__ total) {
    __shared__ float s[TOTAL_BLOCK / 64];
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t i = 0;
    if (((uintptr_t)partials & 15u) == 0u) {
        const float4* p4 = reinterpret_cast<const float4*>(partials);
        const uint32_t n4 = n / 4u;
        uint32_t k = threadIdx.x;
        for (; k + 3u * TOTAL_BLOCK < n4; k += 4u * TOTAL_BLOCK) {
            float4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = p4[k + (uint32_t)u * TOTAL_BLOCK];
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[u] += (v[u].x + v[u].y) + (v[u].z + v[u].w);
        }
        for (; k < n4; k += TOTAL_BLOCK) { const float4 v = p4[k]; acc[0] += (v.x + v.y) + (v.z + v.w); }
        i = n4 * 4u;
    }
    for (i += threadIdx.x; i < n; i += TOTAL_BLOCK) acc[1] += partials[i];
    float v = (acc[0] + acc[1]) + (acc[2] + acc[3]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63u) == 0u) s[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
#pragma unroll
        for (int k = 0; k < TOTAL_BLOCK / 64; ++k) t += s[k];
        *total = t;
    }
}

// Rows a wavefront marches over, a multiple of the partials' tile.  Each strip
// blurs ten rows more than it writes, so strips are as long as keeps every
// SIMD at its four wavefronts in one round of workgroups: a second, partly
// filled round costs more than the extra rows of shorter strips.  Measured
// forward + backward us by strip: 3840x2160 16: 515, 64: 440, 128: 408;
// 1920x1080 16: 133, 32: 110, 64: 141; 1237x823 16: 86, 32: 102.
constexpr uint32_t LOSS_ROUND_WAVES = 4096;
static uint32_t loss_strip(uint32_t w, uint32_t h) {
    const uint32_t cols = 3u * ((w + LW - 1) / LW);
    const uint32_t strips = std::max(1u, LOSS_ROUND_WAVES / cols);
    const uint32_t rows = (h + strips - 1) / strips;
    return (rows + LT - 1) / LT * LT;
}

template <bool C, bool M, bool A>
static void launch_fwd3(const LossArgs& a, dim3 grid, uint32_t strip, hipStream_t s) {
    loss_fwd_kernel<C, M, A><<<grid, LBLOCK, 0, s>>>(a, strip);
}
hipError_t launch_loss_forward(const LossArgs& a, hipStream_t s) {
    const uint32_t strip = loss_strip(a.img_w, a.img_h);
    const dim3 grid((a.img_w + LW - 1) / LW, (a.img_h + strip - 1) / strip);
    const bool alpha = a.alpha_weight_cfg > 0.0f && a.channels == 4;
    const int sel = (a.composite ? 4 : 0) | (a.mask ? 2 : 0) | (alpha ? 1 : 0);
    switch (sel) {
    case 0: launch_fwd3<false, false, false>(a, grid, strip, s); break;
    case 1: launch_fwd3<false, false, true>(a, grid, strip, s); break;
    case 2: launch_fwd3<false, true, false>(a, grid, strip, s); break;
    case 3: launch_fwd3<false, true, true>(a, grid, strip, s); break;
    case 4: launch_fwd3<true, false, false>(a, grid, strip, s); break;
    case 5: launch_fwd3<true, false, true>(a, grid, strip, s); break;
    case 6: launch_fwd3<true, true, false>(a, grid, strip, s); break;
    default: launch_fwd3<true, true, true>(a, grid, strip, s); break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !a.total || !a.partials) return e;
    const uint32_t planes = alpha ? 4u : 3u;
    loss_total_kernel<<<1, TOTAL_BLOCK, 0, s>>>(a.partials, planes * ((a.img_w + LT - 1) / LT) * ((a.img_h + LT - 1) / LT), a.total);
    return hipGetLastError();
}

template <bool C, bool M, bool A>
static void launch_bwd3(const LossBwdArgs& a, dim3 grid, uint32_t strip, bool scalar, hipStream_t s) {
    if (scalar) loss_bwd_kernel<C, M, A, true><<<grid, LBLOCK, 0, s>>>(a, strip);
    else loss_bwd_kernel<C, M, A, false><<<grid, LBLOCK, 0, s>>>(a, strip);
}
hipError_t launch_loss_backward(const LossBwdArgs& a, bool scalar, hipStream_t s) {
    const uint32_t strip = loss_strip(a.img_w, a.img_h);
    const dim3 grid((a.img_w + LW - 1) / LW, (a.img_h + strip - 1) / strip);
    const bool alpha = a.fwd.alpha_weight_cfg > 0.0f && a.channels == 4;
    const int sel = (a.fwd.composite ? 4 : 0) | (a.fwd.mask ? 2 : 0) | (alpha ? 1 : 0);
    switch (sel) {
    case 0: launch_bwd3<false, false, false>(a, grid, strip, scalar, s); break;
    case 1: launch_bwd3<false, false, true>(a, grid, strip, scalar, s); break;
    case 2: launch_bwd3<false, true, false>(a, grid, strip, scalar, s); break;
    case 3: launch_bwd3<false, true, true>(a, grid, strip, scalar, s); break;
    case 4: launch_bwd3<true, false, false>(a, grid, strip, scalar, s); break;
    case 5: launch_bwd3<true, false, true>(a, grid, strip, scalar, s); break;
    case 6: launch_bwd3<true, true, false>(a, grid, strip, scalar, s); break;
    default: launch_bwd3<true, true, true>(a, grid, strip, scalar, s); break;
    }
    return hipGetLastError();
}

} // namespace vs
