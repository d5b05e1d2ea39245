// k_neural.hip -- backward of the compact neural appearance.
//
// Restates crates/splat-train-render/src/bwd/kernels/neural_backwards.rs
// (row_backward :141-283, neural_backwards_kernel :285-442) and the partial
// sum of bwd/render_bwd.rs:390-435.  Each wavefront owns a run of splats: rows
// without a colour gradient get zero outputs, the others queue up in id order
// and are taken 64 at a time, one per lane.  A row recomputes the decoder's
// activations, writes its row gradient [base (DC units), latents, 0] and the
// row's mean square, and adds its view-direction term to the mean gradient
// the projection backward wrote.  The decoder gradient is three products over
// rows, [16 x 64][64 x 32], [16 x 64][64 x 16] and [3 x 64][64 x 16] a step, on
// the f32 matrix instruction from rows staged in LDS; a wavefront writes one
// [816] partial, and one pass sums the partials per weight in f64 in a fixed
// order.  No float atomics, and the result does not depend on scheduling.
#include "vs_neural.h"
#include "vs_internal.h"

namespace vs {

// The kernel is bound by issue: a row's two passes through the decoder are
// 3,264 multiplies and adds that stay unfused (the row gradients have the
// restatement's bits).  A row's values stay in registers and the weights are
// scalar operands, so a step touches LDS only to turn rows into matrix
// operands: 7 reads and 4 matrix instructions per 4 rows, where products a
// lane and weight at a time read 80.  A wavefront is a workgroup with
// 13.6 KB of LDS, eleven to a CU, and waits for no other.  600k splats
// (1920x1080 view): 192 us in 128-lane workgroups with weights and rows
// in 64 KB of LDS (586 wavefronts for 1024 SIMDs), 83 us.
constexpr uint32_t NB_ROWS = 64;                // rows per step
constexpr uint32_t NB_STRIDE = 52;              // floats per staged row: 16-byte stores of 64 rows meet no bank twice
// Splats per wavefront: as many wavefronts as the chip holds (about 2,048 with
// eight a CU in flight), and no fewer than four blocks of 64 each, below which
// a step's lanes run empty and the partials outgrow what they sum.
constexpr uint32_t NB_WAVES = 2048, NB_MIN_CHUNK = 4 * NB_ROWS;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) float* ConstWeights;   // uniform reads become scalar loads

static uint32_t neural_bwd_chunk(uint32_t num_splats) {
    const uint32_t c = (uint32_t)(((uint64_t)num_splats + NB_WAVES * NB_ROWS - 1) / (NB_WAVES * NB_ROWS)) * NB_ROWS;
    return c < NB_MIN_CHUNK ? NB_MIN_CHUNK : c;
}

// Orders the wavefront's LDS stores and the other lanes' loads around it.
VS_DEV void nb_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// `weights` + offset as a pointer that the compiler takes for a new one, known
// only after `done`: a layer's rows are loaded where they are used, since the
// 816 weights do not fit the scalar registers and would be loaded ahead and
// kept (spilled) from one use to the next.
VS_DEV ConstWeights nb_weights(uintptr_t& weights, float& done, int offset) {
    asm volatile("" : "+s"(weights), "+v"(done));
    return (ConstWeights)weights + offset;
}

// What a row's backward leaves for the weight products.
struct NeuralRow {
    float x[NEURAL_INPUTS], h1[NEURAL_HIDDEN], h2[NEURAL_HIDDEN];
    float d1[NEURAL_HIDDEN], d2[NEURAL_HIDDEN], go[3];
};

// One row's backward (neural_backwards.rs:141-283).  Every sum adds its terms
// in input order from 0, as the forward's dot products do.
template <typename SHT>
VS_DEV void neural_row_bwd(const NeuralBwdArgs& a, uint32_t g, NeuralRow& R) {
    uintptr_t weights = reinterpret_cast<uintptr_t>(a.decoder);
    const SHT* row = static_cast<const SHT*>(a.rows) + (size_t)g * NEURAL_ROW;
    const float* t = a.transforms + (size_t)g * 10;
    const float* rg = a.v_combined + (size_t)g * 10;
    const vs_camera& u = a.cam;
    const F3 u_world = F3{t[0], t[1], t[2]} - F3{u.cam_pos[0], u.cam_pos[1], u.cam_pos[2]};
    const float u_len = length(u_world);
    const F3 dir = u_world * (1.0f / u_len);
#pragma unroll
    for (int i = 0; i < NEURAL_LATENTS; ++i) sincosf_c(sh_ld(row, 3 + i), R.x[2 * i], R.x[2 * i + 1]);
    direction_basis(R.x, dir, a.degree);
    // h1 = ReLU(W1 x), h2 = ReLU(W2 h1)
#pragma unroll
    for (int j = 0; j < NEURAL_HIDDEN; ++j) {
        const ConstWeights W = nb_weights(weights, j ? R.h1[j ? j - 1 : 0] : R.x[NEURAL_INPUTS - 1], NEURAL_W1 + j * NEURAL_INPUTS);
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < NEURAL_INPUTS; ++k) acc += W[k] * R.x[k];
        R.h1[j] = mx(acc, 0.0f);
    }
#pragma unroll
    for (int j = 0; j < NEURAL_HIDDEN; ++j) {
        const ConstWeights W = nb_weights(weights, j ? R.h2[j ? j - 1 : 0] : R.h1[NEURAL_HIDDEN - 1], NEURAL_W2 + j * NEURAL_HIDDEN);
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < NEURAL_HIDDEN; ++k) acc += W[k] * R.h1[k];
        R.h2[j] = mx(acc, 0.0f);
    }
    const ConstWeights W3 = nb_weights(weights, R.h2[NEURAL_HIDDEN - 1], NEURAL_W3);
    // o = W3 h2; colour = ReLU(C0 base + tanh(o) + 0.5)
    const float gc[3] = {rg[5], rg[6], rg[7]};
    float vrow[NEURAL_ROW];
    float sq = 0.0f;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        float o = 0.0f;
#pragma unroll
        for (int k = 0; k < NEURAL_HIDDEN; ++k) o += W3[c * NEURAL_HIDDEN + k] * R.h2[k];
        const float th = tanhf_c(o);
        const float base = sh_ld(row, c) * NEURAL_C0;
        const float gcol = (base + th + 0.5f > 0.0f) ? gc[c] : 0.0f;     // ReLU of the colour
        vrow[c] = gcol * NEURAL_C0;
        sq += (gcol * NEURAL_C0) * (gcol * NEURAL_C0);
        R.go[c] = gcol * (1.0f - th * th);
    }
    // d2 = [h2 > 0] W3^T go
#pragma unroll
    for (int k = 0; k < NEURAL_HIDDEN; ++k) {
        float s2 = 0.0f;
#pragma unroll
        for (int c = 0; c < 3; ++c) s2 += W3[c * NEURAL_HIDDEN + k] * R.go[c];
        R.d2[k] = (R.h2[k] > 0.0f) ? s2 : 0.0f;
    }
    // d1 = [h1 > 0] W2^T d2
#pragma unroll
    for (int k = 0; k < NEURAL_HIDDEN; ++k) R.d1[k] = 0.0f;
#pragma unroll
    for (int j = 0; j < NEURAL_HIDDEN; ++j) {
        const ConstWeights W = nb_weights(weights, j ? R.d1[NEURAL_HIDDEN - 1] : R.d2[NEURAL_HIDDEN - 1], NEURAL_W2 + j * NEURAL_HIDDEN);
#pragma unroll
        for (int k = 0; k < NEURAL_HIDDEN; ++k) R.d1[k] += W[k] * R.d2[j];
    }
#pragma unroll
    for (int k = 0; k < NEURAL_HIDDEN; ++k) R.d1[k] = (R.h1[k] > 0.0f) ? R.d1[k] : 0.0f;
    // dx = W1^T d1
    float dx[NEURAL_INPUTS];
#pragma unroll
    for (int k = 0; k < NEURAL_INPUTS; ++k) dx[k] = 0.0f;
#pragma unroll
    for (int j = 0; j < NEURAL_HIDDEN; ++j) {
        const ConstWeights W = nb_weights(weights, j ? dx[NEURAL_INPUTS - 1] : R.d1[NEURAL_HIDDEN - 1], NEURAL_W1 + j * NEURAL_INPUTS);
#pragma unroll
        for (int k = 0; k < NEURAL_INPUTS; ++k) dx[k] += W[k] * R.d1[j];
    }
#pragma unroll
    for (int i = 0; i < NEURAL_LATENTS; ++i) {           // latents through sin / cos
        const float gl = dx[2 * i] * R.x[2 * i + 1] - dx[2 * i + 1] * R.x[2 * i];
        vrow[3 + i] = gl;
        sq += gl * gl;
    }
    vrow[11] = 0.0f;
    if (a.v_rows) {
        float4* o4 = reinterpret_cast<float4*>(a.v_rows + (size_t)g * NEURAL_ROW);
        o4[0] = make_float4(vrow[0], vrow[1], vrow[2], vrow[3]);
        o4[1] = make_float4(vrow[4], vrow[5], vrow[6], vrow[7]);
        o4[2] = make_float4(vrow[8], vrow[9], vrow[10], vrow[11]);
    }
    if (a.v_rows_sq) a.v_rows_sq[g] = sq / (float)NEURAL_ROW;
    if (a.v_transforms) {
        const F3 g_dir = direction_basis_vjp(dx, dir, a.degree);
        const F3 vm = (g_dir - dir * dot(dir, g_dir)) * (1.0f / u_len);
        float* vt = a.v_transforms + (size_t)g * 10;
        vt[0] += vm.x;
        vt[1] += vm.y;
        vt[2] += vm.z;
    }
}

// Stages `count` values (a multiple of four) at column `at` of the lane's row.
VS_DEV void nb_stage(float* row, uint32_t at, const float* v, uint32_t count) {
#pragma unroll
    for (uint32_t i = 0; i < count; i += 4)
        *reinterpret_cast<float4*>(row + at + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
}

// One wavefront per `chunk` splats.
template <typename SHT>
__global__ void __launch_bounds__(NB_ROWS) neural_bwd_kernel(NeuralBwdArgs a, uint32_t chunk) {
    __shared__ __attribute__((aligned(16))) float s_rows[NB_ROWS * NB_STRIDE];
    __shared__ uint32_t s_queue[2 * NB_ROWS];
    const uint32_t lane = threadIdx.x;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const uint64_t begin = (uint64_t)blockIdx.x * chunk;
    const uint32_t end = (uint32_t)(begin + chunk < a.num_splats ? begin + chunk : a.num_splats);
    uint32_t pos = (uint32_t)begin, queued = 0;
    f32x4 w1a = {0.0f, 0.0f, 0.0f, 0.0f}, w1b = w1a, w2 = w1a, w3 = w1a;
    float* mine = s_rows + lane * NB_STRIDE;
    // operand element of this lane: row lane / 16 of a group of four, column lane % 16
    const uint32_t col = lane & 15u;
    const float* opnd = s_rows + (lane >> 4) * NB_STRIDE + col;
    const float* go_op = s_rows + (lane >> 4) * NB_STRIDE + 48 + (col < 3u ? col : 0u);
    while (true) {
        // Fill the queue to a step's rows (at most 63 stay from before).
        while (queued < NB_ROWS && pos < end) {
            const uint32_t g = pos + lane;
            bool act = false;
            if (g < end) {
                const float* rg = a.v_combined + (size_t)g * 10;
                act = rg[5] != 0.0f || rg[6] != 0.0f || rg[7] != 0.0f;
                if (!act) {
                    if (a.v_rows) {
                        float4* o4 = reinterpret_cast<float4*>(a.v_rows + (size_t)g * NEURAL_ROW);
                        o4[0] = o4[1] = o4[2] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    }
                    if (a.v_rows_sq) a.v_rows_sq[g] = 0.0f;
                }
            }
            const uint64_t m = __ballot(act);
            if (act) s_queue[queued + (uint32_t)__popcll(m & lt_mask)] = g;
            queued += (uint32_t)__popcll(m);
            pos += NB_ROWS;
        }
        if (queued == 0u) break;
        nb_fence();
        const uint32_t nrows = queued < NB_ROWS ? queued : NB_ROWS;
        const uint32_t g = s_queue[lane], next = s_queue[NB_ROWS + lane];
        NeuralRow R;
        if (lane < nrows) {
            neural_row_bwd<SHT>(a, g, R);
        } else {                                // rows that add +0 to every product
#pragma unroll
            for (int k = 0; k < NEURAL_INPUTS; ++k) R.x[k] = 0.0f;
#pragma unroll
            for (int k = 0; k < NEURAL_HIDDEN; ++k) R.h1[k] = R.h2[k] = R.d1[k] = R.d2[k] = 0.0f;
            R.go[0] = R.go[1] = R.go[2] = 0.0f;
        }
        nb_fence();
        queued -= nrows;
        if (lane < queued) s_queue[lane] = next;
        // A step's products start at 0 and are added to the running ones, so the sums stay pairwise by 64 rows.
        f32x4 p1a = {0.0f, 0.0f, 0.0f, 0.0f}, p1b = p1a, p2 = p1a, p3 = p1a;
        const float go[4] = {R.go[0], R.go[1], R.go[2], 0.0f};
        nb_stage(mine, 0, R.h1, NEURAL_HIDDEN);
        nb_stage(mine, 16, R.h2, NEURAL_HIDDEN);
        nb_stage(mine, 32, R.d2, NEURAL_HIDDEN);
        nb_stage(mine, 48, go, 4);
        nb_fence();
#pragma unroll 4
        for (uint32_t r = 0; r < NB_ROWS; r += 4) {      // dW2 = d2^T h1, dW3 = go^T h2
            const float* o = opnd + r * NB_STRIDE;
            const float gv = go_op[r * NB_STRIDE];
            p2 = __builtin_amdgcn_mfma_f32_16x16x4f32(o[32], o[0], p2, 0, 0, 0);
            p3 = __builtin_amdgcn_mfma_f32_16x16x4f32(col < 3u ? gv : 0.0f, o[16], p3, 0, 0, 0);
        }
        nb_fence();
        nb_stage(mine, 0, R.x, NEURAL_INPUTS);
        nb_stage(mine, 32, R.d1, NEURAL_HIDDEN);
        nb_fence();
#pragma unroll 4
        for (uint32_t r = 0; r < NB_ROWS; r += 4) {      // dW1 = d1^T x
            const float* o = opnd + r * NB_STRIDE;
            p1a = __builtin_amdgcn_mfma_f32_16x16x4f32(o[32], o[0], p1a, 0, 0, 0);
            p1b = __builtin_amdgcn_mfma_f32_16x16x4f32(o[32], o[16], p1b, 0, 0, 0);
        }
        nb_fence();
        w1a += p1a; w1b += p1b; w2 += p2; w3 += p3;
    }
    // Element i of an accumulator is row 4 (lane / 16) + i, column lane % 16.
    float* p = a.partials + (size_t)blockIdx.x * NEURAL_LEN;
    const uint32_t j0 = (lane >> 4) * 4u;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        p[NEURAL_W1 + (j0 + i) * NEURAL_INPUTS + col] = w1a[i];
        p[NEURAL_W1 + (j0 + i) * NEURAL_INPUTS + 16 + col] = w1b[i];
        p[NEURAL_W2 + (j0 + i) * NEURAL_HIDDEN + col] = w2[i];
        if (j0 + i < 3u) p[NEURAL_W3 + (j0 + i) * NEURAL_HIDDEN + col] = w3[i];
    }
}

// The [blocks, 816] partials summed per weight in f64: 16 weights per block (a
// 64-byte segment of each partial), 64 lanes per weight striding the partial
// rows, combined in a fixed order.  51 blocks with 64 chains a weight read
// 6 MB of partials in 6 us.
constexpr uint32_t NS_COLS = 16, NS_PARTS = 64;
__global__ void __launch_bounds__(NS_COLS * NS_PARTS) neural_sum_kernel(const float* __restrict__ partials,
                                                                        uint32_t nblocks, float* __restrict__ out) {
    __shared__ double s_part[NS_PARTS][NS_COLS];
    const uint32_t c = threadIdx.x % NS_COLS, part = threadIdx.x / NS_COLS;
    const uint32_t w = blockIdx.x * NS_COLS + c;
    static_assert(NEURAL_LEN % NS_COLS == 0, "every lane owns a weight");
    double acc = 0.0;
#pragma unroll 8
    for (uint32_t b = part; b < nblocks; b += NS_PARTS) acc += (double)partials[(size_t)b * NEURAL_LEN + w];
    s_part[part][c] = acc;
    __syncthreads();
    for (uint32_t half = NS_PARTS / 2; half > 0; half >>= 1) {
        if (part < half) s_part[part][c] += s_part[part + half][c];
        __syncthreads();
    }
    if (part == 0) out[w] = (float)s_part[0][c];
}

uint32_t neural_bwd_blocks(uint32_t num_splats) {
    const uint32_t chunk = neural_bwd_chunk(num_splats);
    const uint32_t b = (uint32_t)(((uint64_t)num_splats + chunk - 1) / chunk);
    return b < 1u ? 1u : b;
}

hipError_t launch_neural_bwd(const NeuralBwdArgs& a, hipStream_t s) {
    const uint32_t nb = neural_bwd_blocks(a.num_splats), chunk = neural_bwd_chunk(a.num_splats);
    if (a.half) neural_bwd_kernel<uint16_t><<<nb, NB_ROWS, 0, s>>>(a, chunk);
    else neural_bwd_kernel<float><<<nb, NB_ROWS, 0, s>>>(a, chunk);
    if (a.v_decoder) neural_sum_kernel<<<NEURAL_LEN / NS_COLS, NS_COLS * NS_PARTS, 0, s>>>(a.partials, nb, a.v_decoder);
    return hipGetLastError();
}

}  // namespace vs
