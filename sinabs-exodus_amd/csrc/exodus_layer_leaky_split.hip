// Backward kernel of the leaky layer for layers with few neurons and many steps: one lane per neuron and chunk of CKPT steps.
#include "exodus_layer.hpp"

namespace {

// layer_leaky_backward gives a neuron one lane, and a layer of a few thousand neurons is a few lone waves that walk the whole
// sequence at 96 ns per step.  Its recurrence is affine: with h what reaches a step from later ones, g_t = h + grad_out_t and
// h' = alpha g_t, a chunk of n steps maps h to P + alpha^n h.  So every chunk gets a lane, as in layer_lif_backward_split: it
// walks its chunk for P, the maps go through LDS, a lane folds those of the newer chunks and walks its chunk again with the
// operations of the one-lane kernel.  Longer sequences are walked in groups of chunks, what leaves a group waiting in LDS.
// grad_x and the sums agree with the one-lane kernel's to rounding: powers and fold are fp64, as 31 roundings of one sign in a^32
// would be ten times what a walk loses.
// A factor beyond [-1, 1], or values that are not finite, would not survive the fold (0 times infinity): a block that has any
// passes h through its chunks one after the other.
// One lane per neuron / this, us, with alpha gradient: (1, 2000, 64) 190 / 12.4, (64, 300, 10) 30.9 / 6.8, (32, 100, 512) 12.5 / 7.3,
// (12, 400, 1323) 41.9 / 26.7, (8, 1000, 2048) 100 / 39.5.  Its error against float64 is smaller than the walk's: 0.5 times for
// grad_x, 0.4 for the alpha gradient (1025 steps, factors of 0.6 to 0.999; a sum that starts anew in every chunk loses less).
// What bounds it: two chains of 32 steps per group of chunks and a trip to memory and back.
template <bool ALPHA, bool WITH_X, bool GO1>
__global__ void __launch_bounds__(SPLIT_LANES) layer_leaky_backward_split(const LeakySplitArgs q, const int64_t blocks_per_batch,
                                                                          const int neurons_log)
{
    typedef BufIO<1, false> IO;
    __shared__ float map_p[SPLIT_LANES], carry[SPLIT_NEURONS];
    __shared__ double map_q[SPLIT_LANES];
    __shared__ double parts[ALPHA ? SPLIT_LANES : 1];
    const int64_t T = q.T, M = q.M;
    const int tid = threadIdx.x, many = 1 << neurons_log, chunks = blockDim.x >> neurons_log;
    const int lane = tid & (many - 1), j = tid >> neurons_log;
    const int64_t b = blockIdx.x / blocks_per_batch, m0 = (blockIdx.x - b * blocks_per_batch) << neurons_log;
    // lanes past the end of the layer compute on the block's first neuron; their offsets lie beyond every resource
    const bool active = m0 + lane < M;
    const int64_t row = b * M + m0 + (active ? lane : 0), n_ck = (T + CKPT - 1) / CKPT;
    const unsigned step_bytes = static_cast<unsigned>(M) * 4u, row_bytes = static_cast<unsigned>(M - m0) * 4u;
    const float a = q.alpha[row], kept = __fsub_rn(1.0f, a), v0 = ALPHA ? q.v_init[row] : 0.f;
    const float g1 = GO1 ? q.grad_out[0] : 0.f;
    double a_full = a;                                           // a ^ CKPT
#pragma unroll
    for (int k = 1; k < CKPT; k *= 2) a_full *= a_full;
    const auto finite = [](float f) { return fabsf(f) < __builtin_inff(); };
    if (j == 0) carry[lane] = q.grad_v_last ? q.grad_v_last[row] : 0.f;
    TileSum acc;
    acc.clear();
    float h = 0.f;
    __syncthreads();

    for (int64_t group = (n_ck + chunks - 1) / chunks - 1; group >= 0; --group) {
        const int64_t tg = group * chunks * CKPT, t0 = tg + j * CKPT;
        const int len = static_cast<int>(T - t0 >= CKPT ? CKPT : (T > t0 ? T - t0 : 0));
        const unsigned steps = static_cast<unsigned>(T - tg < chunks * CKPT ? T - tg : chunks * CKPT);
        const unsigned bytes = (steps - 1) * step_bytes + row_bytes;   // below 2^31: the host keeps M below 2^19
        const int64_t at = (b * T + tg) * M + m0;
        const unsigned from = static_cast<unsigned>(j * CKPT);
        // the outputs of the step before: one step further back, and none before the first
        const unsigned back = tg > 0 ? 1u : 0u;
        const Rsrc rg = make_rsrc(GO1 ? nullptr : q.grad_out + at, bytes), rx = make_rsrc(WITH_X ? q.x + at : nullptr, bytes);
        const Rsrc ro = make_rsrc(ALPHA ? q.out + at - back * M : nullptr, bytes + back * step_bytes);
        float g[GO1 ? 1 : CKPT], o[ALPHA ? CKPT : 1], x[WITH_X ? CKPT : 1], gx[CKPT];
#pragma unroll
        for (int k = 0; k < CKPT; ++k) {
            const bool in = active && k < len;
            const unsigned off = in ? (from + k) * step_bytes + lane * 4u : BEYOND;
            if (!GO1) g[GO1 ? 0 : k] = IO::load(rg, off, 0);
            if (WITH_X) x[WITH_X ? k : 0] = IO::load(rx, off, 0);
            if (ALPHA) o[ALPHA ? k : 0] = IO::load(ro, in && from + k + back > 0 ? off + back * step_bytes - step_bytes : BEYOND, 0);
        }
        if (ALPHA && t0 == 0) o[0] = v0;

        // what leaves the chunk of an h that enters it
        const auto through = [&](float enters) {
#pragma unroll
            for (int kq = 0; kq < CKPT; ++kq) {
                const int k = CKPT - 1 - kq;
                const float out = __fmul_rn(__fadd_rn(enters, GO1 ? g1 : g[GO1 ? 0 : k]), a);
                enters = k < len ? out : enters;
            }
            return enters;
        };
        double power = a_full;
        if (len != CKPT) {
            power = 1.0;
            for (int k = 0; k < len; ++k) power *= a;
        }
        const float p = through(0.f);
        map_p[tid] = p;
        map_q[tid] = power;
        const bool tame = !active || (fabsf(a) <= 1.f && finite(p) && finite(carry[lane]));
        const bool wild = __syncthreads_or(!tame);
        h = carry[lane];
        if (!wild) {
            double enters = h;
            for (int c = chunks - 1; c > j; --c) enters = map_p[(c << neurons_log) + lane] + map_q[(c << neurons_log) + lane] * enters;
            h = static_cast<float>(enters);
        } else {
            __syncthreads();                                     // everybody has read the carry
            for (int c = chunks - 1; c >= 0; --c) {
                if (j == c) {
                    if (c < chunks - 1) h = map_p[tid + many];
                    map_p[tid] = through(h);
                }
                __syncthreads();
            }
        }

        // the walk of the one-lane kernel
#pragma unroll
        for (int kq = 0; kq < CKPT; ++kq) {
            const int k = CKPT - 1 - kq;
            if (k < len) {
                const float gt = __fadd_rn(h, GO1 ? g1 : g[GO1 ? 0 : k]);
                h = __fmul_rn(gt, a);
                float result = q.decay_early ? h : gt;
                if (ALPHA) {
                    acc.add(gt, o[ALPHA ? k : 0]);
                    if (WITH_X) {
                        const float xe = x[WITH_X ? k : 0];
                        if (q.decay_early) acc.add(gt, q.norm_input ? __fmul_rn(kept, xe) : xe);
                        if (q.norm_input) acc.sub(result, xe);
                    }
                }
                gx[k] = q.norm_input ? __fmul_rn(result, kept) : result;
            }
            if (ALPHA && k % 8 == 0) acc.fold();
        }
        const Rsrc rw = make_rsrc(q.grad_x + at, bytes);
#pragma unroll
        for (int k = 0; k < CKPT; ++k) IO::store(gx[k], rw, active && k < len ? (from + k) * step_bytes + lane * 4u : BEYOND, 0);
        __syncthreads();                                         // everybody has read the maps and the carry
        if (j == 0) carry[lane] = h;
        __syncthreads();
    }

    if (ALPHA) {
        parts[tid] = acc.total;
        __syncthreads();
    }
    if (j != 0 || !active) return;
    if (q.v_init_grad) q.v_init_grad[row] = h;
    if (ALPHA) {
        double sum = 0.0;
        for (int c = 0; c < chunks; ++c) sum += parts[(c << neurons_log) + lane];
        q.alpha_grad[row] = static_cast<float>(sum);
    }
}

template <bool ALPHA, bool WITH_X>
int launch(const LeakySplitArgs &a, bool uniform, int64_t B, hipStream_t s)
{
    const SplitShape shape = split_shape(B, a.T, a.M);
    if (shape.blocks_per_batch > 0x7fffffffLL / B) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(shape.blocks_per_batch * B)), block(shape.lanes);
    if (uniform)
        hipLaunchKernelGGL((layer_leaky_backward_split<ALPHA, WITH_X, true>), grid, block, 0, s, a, shape.blocks_per_batch,
                           shape.neurons_log);
    else
        hipLaunchKernelGGL((layer_leaky_backward_split<ALPHA, WITH_X, false>), grid, block, 0, s, a, shape.blocks_per_batch,
                           shape.neurons_log);
    return static_cast<int>(hipGetLastError());
}

}  // namespace

// Up to 16 384 neurons a call with a gradient per output is ahead at every length, level for 33 to 48 steps without alpha gradient.
// One lane / this, us, with alpha gradient and scalings, (8, t, 2048) 33 steps 7.6 / 6.1, 64 steps 9.7 / 6.4, 300 steps 44 / 18.6, 1000
// steps 138 / 47; without, 33 steps 5.0 / 5.0, 300 steps 21.2 / 10.7.  At 32 768 (16, t, 2048) 33 steps 6.1 / 6.4, 300 steps
// 34.8 / 29.4, 1000 steps 106 / 91; at 65 536 300 steps 43.4 / 51.5.  Blocks hold 16 neurons at least, but many samples of few neurons
// leave the one-lane kernel's waves as empty: (16384, 300, 1) 1187 / 212, (4096, 300, 4) 311 / 45, (1024, 33, 4) 16.9 / 6.8.
// A gradient of one value for all outputs leaves the one-lane kernel a tensor less to read, none without alpha gradient, and it is ahead
// there up to 96 steps, (8, t, 2048) 33 steps 3.8 / 4.8, 64 steps 4.5 / 5.0, 160 steps 6.7 / 6.4, and by up to 8 % at 300 steps of
// 8192 neurons and more, 9.5 / 9.9 (1000 steps 20.4 / 15.8); with alpha gradient up to 40 steps without scalings, 33 steps
// 5.1 / 6.0.  It takes this kernel all the same: the call then gives the bits of the one with that value written out.
constexpr int64_t LEAKY_SPLIT_MOST_NEURONS = 16384;
bool exodus_layer_leaky_split_applies(int64_t B, int64_t T, int64_t M)
{
    const int mode = exodus_layer_split_mode();
    if (mode == 0 || T <= CKPT || !exodus_layer_split_applies(M)) return false;
    return mode == 3 || B * M <= LEAKY_SPLIT_MOST_NEURONS;
}

int exodus_layer_leaky_split(const LeakySplitArgs &a, bool uniform, int64_t B, hipStream_t s)
{
    if (!a.alpha_grad) return launch<false, false>(a, uniform, B, s);
    return a.decay_early || a.norm_input ? launch<true, true>(a, uniform, B, s) : launch<true, false>(a, uniform, B, s);
}
