// Backward kernel of the spiking layer for layers with few neurons and many steps: one lane per neuron and chunk of CKPT
// steps.
#include "exodus_layer.hpp"

namespace {

// With one lane per neuron (exodus_layer_backward.hip) a layer of a few thousand neurons fills a fraction of the machine,
// and its run time is the length of one lane's chain: 120 to 150 ns per step.  Two facts allow cutting the chain into
// pieces: the chunks of CKPT steps can be rebuilt independently from their checkpoints, and the adjoint recurrences are
// affine once the forward values are known.  With a_t = s_t g_t and b_t = 1 - c s_t (and both gone where the potential was
// clamped)
//     lambda_t = a_t + b_t h_{t+1},   h_t = a_mem lambda_t,        h_T  = gradient on the final potential,
//     mu_t = hm_{t+1} + k lambda_t,   hm_t = a_syn mu_t,           hm_T = gradient on the final synaptic current,
// so a chunk maps what enters it from later steps to what leaves it:
//     h_out = A + B h_in,   hm_out = C + D h_in + U hm_in.
// A lane rebuilds its chunk, keeps (a, b, vpost, i) of every step, walks it once for (A, B, C, D, U), exchanges them through
// LDS, folds the maps of the newer chunks into its own (h_in, hm_in), and walks the chunk again with the operations of the
// one-lane kernel.  A block holds up to 32 chunks of 16 to 64 neurons (see launch); longer sequences are walked in groups
// of chunks, newest first, what leaves a group waiting in LDS for the next.  Results agree with the one-lane kernel's to
// rounding (h_in and hm_in are folded instead of walked), not bit for bit.
//
// B, D and U are products of 32 factors a_mem (1 - c s) or a_syn.  Where |1 - c s| stays above 16 (narrow surrogates) B
// leaves the floats' range, and infinity times an h_in of 0, or of 1e-30, says nothing about h_out.  A block with such a
// map passes h and hm through the group's chunks one after the other with the operations of the walk, which is right for
// every value: 39 us more per group of 32 chunks, (4, 2000, 512) 31 -> 109 against 276 with one lane per neuron.  The waves
// say so where they publish their maps, which costs other calls 0.1 to 0.4 us of 8 to 10 (a vote of the block on the folded
// values, one barrier more, 0.2 to 0.9).  Where all maps are finite an h_in that is no number is folded like any other:
// `stops` has it end at a clamped step as the walk does.
//
// What bounds it: the chain of 3 x 32 steps per group and one trip to memory and back, 9-11 us for up to 32 chunks on an
// otherwise idle machine ((32, 100, 512) 15.6 -> 9.8 us, (64, 300, 10) 16.1 -> 10.1 against a kernel that carried two numbers
// through one walk, with up to 1024 lanes of 128 registers; (4, 2000, 512) with synapses 302 -> 41 us against one lane per
// neuron).  512 lanes per block leave 256 registers per lane: the four values of 32 steps and all but 12 to 28 bytes of the
// rest, 132 to 156 with a synapse and state records, go into them.  Sums of a neuron's gradients are fp32 over 8 steps and
// fp64 beyond: against float64 their error is 0.7 to 0.8 times the one-lane kernel's, that of grad_x the same.
static_assert(CKPT == 32, "a chunk's clamped steps are bits of an unsigned, a_syn^CKPT is squared up, a group spans 2^10 steps");

// EXTRA: gradients on the state records; GO1: one value as the gradient of every spike (see the one-lane kernel)
template <bool SYN, int KIND, int CAPK, bool EXTRA, bool GO1>
__global__ void __launch_bounds__(SPLIT_LANES) layer_lif_backward_split(const SplitArgs q, const int64_t blocks_per_batch,
                                                                        const int neurons_log)
{
    constexpr bool FROM_TENSOR = KIND == EXODUS_SURR_TENSOR;
    typedef BufIO<1, false> IO;
    __shared__ float map_a[SPLIT_LANES], map_b[SPLIT_LANES];
    __shared__ float map_c[SYN ? SPLIT_LANES : 1], map_d[SYN ? SPLIT_LANES : 1], map_u[SYN ? SPLIT_LANES : 1];
    __shared__ unsigned char stops[SPLIT_LANES];   // 1: h_in ends inside the chunk, 2: it does not get into mu either
    __shared__ union {
        unsigned char of_wave[SPLIT_LANES / WAVE];
        uint64_t all;
    } wild;                                        // a map of the wave is not finite
    __shared__ float carry_h[SPLIT_NEURONS], carry_m[SPLIT_NEURONS];
    __shared__ double part_m[SPLIT_LANES], part_s[SYN ? SPLIT_LANES : 1];
    const LayerConsts &p = q.p;
    const int64_t T = q.T, M = q.M;
    const int tid = threadIdx.x, many = 1 << neurons_log;
    const int chunks = blockDim.x >> neurons_log;                // chunks of a group
    const int lane = tid & (many - 1), j = tid >> neurons_log;
    const int64_t b = blockIdx.x / blocks_per_batch;
    const int64_t m0 = (blockIdx.x - b * blocks_per_batch) << neurons_log;
    // lanes past the end of the layer compute on the block's first neuron; their offsets lie beyond every resource
    const bool active = m0 + lane < M;
    const int64_t row = b * M + m0 + (active ? lane : 0);
    const int64_t n_ck = (T + CKPT - 1) / CKPT;
    const unsigned step_bytes = static_cast<unsigned>(M) * 4u;
    const unsigned row_bytes = static_cast<unsigned>(M - m0) * 4u;

    Cap cc;
    cc.cap = p.cap;
    cc.one = p.cap >= 1u ? 1.f : 0.f;
    Neuron nr = {};
    neuron_load<SYN, CAPK>(nr, p, row);
    const float xg = (SYN && p.decay_early) ? nr.as : 1.0f;      // factor between mu and grad_x
    const SurrConst sk = surrogate_consts<KIND>(nr.th, q.p0, q.p1);
    const float g1 = GO1 ? q.grad_spikes[0] : 0.f;
    float u_full = nr.as;                                        // a_syn ^ CKPT
    if (SYN) {
#pragma unroll
        for (int k = 1; k < CKPT; k *= 2) u_full = __fmul_rn(u_full, u_full);
    }
    if (j == 0) {
        carry_h[lane] = q.grad_v_last ? q.grad_v_last[row] : 0.f;
        carry_m[lane] = (SYN && q.grad_i_last) ? q.grad_i_last[row] : 0.f;
    }
    TileSum acc_m, acc_n, acc_s;                                 // sums of lambda_t vpost_{t-1}, lambda_t i_t, mu i
    acc_m.clear();
    acc_n.clear();
    acc_s.clear();
    float h = 0.f, hm = 0.f;

    for (int64_t group = (n_ck + chunks - 1) / chunks - 1; group >= 0; --group) {
        const int64_t tg = group * chunks * CKPT;                // first step of the group
        const int64_t t0 = tg + j * CKPT;
        const int len = static_cast<int>(T - t0 >= CKPT ? CKPT : (T > t0 ? T - t0 : 0));
        const unsigned steps = static_cast<unsigned>(T - tg < chunks * CKPT ? T - tg : chunks * CKPT);
        const unsigned bytes = (steps - 1) * step_bytes + row_bytes;   // below 2^31: the host keeps M below 2^19
        const unsigned voff = (active && len > 0) ? static_cast<unsigned>(j * CKPT) * step_bytes + lane * 4u : BEYOND;
        const int64_t at = (b * T + tg) * M + m0;
        const bool whole = __builtin_amdgcn_ballot_w64(len != CKPT) == 0;   // all chunks of the wave are
        float xr[CKPT], gr[CKPT], br[CKPT], vp[CKPT];            // x then i; g, a, then grad_x; b; vpost
        float qv[EXTRA ? CKPT : 1], qi[(EXTRA && SYN) ? CKPT : 1];
        unsigned open = 0;                                       // steps whose potential was not clamped
        float vp0 = 0.f, i0 = 0.f;                               // vpost and i of the step before the chunk
        if (len > 0) {
            const int64_t ck = (b * n_ck + group * chunks + j) * M + m0 + (active ? lane : 0);
            vp0 = q.ckpt_v[ck];
            i0 = SYN ? q.ckpt_i[ck] : 0.f;
        }
        auto load = [&](auto guard) {
            constexpr bool GUARD = decltype(guard)::value;
            const Rsrc rx = make_rsrc(q.x + at, bytes), rg = make_rsrc(GO1 ? nullptr : q.grad_spikes + at, bytes);
            const Rsrc rs = make_rsrc(FROM_TENSOR ? q.surr + at : nullptr, bytes);
            const Rsrc rqv = make_rsrc(EXTRA ? q.grad_v_rec + at : nullptr, bytes);
            const Rsrc rqi = make_rsrc((EXTRA && SYN) ? q.grad_i_rec + at : nullptr, bytes);
#pragma unroll
            for (int k = 0; k < CKPT; ++k) {
                const unsigned vo = GUARD ? (k < len ? voff + k * step_bytes : BEYOND) : voff;
                const unsigned so = GUARD ? 0u : k * step_bytes;
                xr[k] = IO::load(rx, vo, so);
                gr[k] = GO1 ? g1 : IO::load(rg, vo, so);
                if (FROM_TENSOR) br[k] = IO::load(rs, vo, so);
                if (EXTRA) qv[k] = IO::load(rqv, vo, so);
                if (EXTRA && SYN) qi[k] = IO::load(rqi, vo, so);
            }
        };
        if (whole) load(std::false_type{}); else load(std::true_type{});

        // rebuild (the operations of the forward pass in its order) and turn every step into its (a, b)
        nr.vpost = vp0;
        nr.i = i0;
#pragma unroll
        for (int k = 0; k < CKPT; ++k) {
            const float v = neuron_advance<SYN>(nr, xr[k]);
            nr.vpost = __fsub_rn(v, reset_amount<CAPK>(v, nr, cc));
            const float sg = FROM_TENSOR ? br[k] : surrogate<KIND>(v, nr.th, q.inv_p0, sk);
            xr[k] = nr.i;
            vp[k] = nr.vpost;
            br[k] = __fsub_rn(1.0f, __fmul_rn(nr.c, sg));
            gr[k] = __fmul_rn(sg, gr[k]);
            if (EXTRA) gr[k] = __fadd_rn(gr[k], __fmul_rn(br[k], qv[EXTRA ? k : 0]));
            open |= v > nr.gate ? 1u << k : 0u;
        }
        // lambda of an open step, 0 of a clamped one (whatever it would have been)
        auto pass = [&](float l, int k) { return (open >> k) & 1u ? l : 0.f; };

        // the chunk's map (steps past the end of the sequence leave it alone)
        float hp = 0.f, hq = 1.f, mp = 0.f, mq = 0.f, mu_u = 1.f;
        auto map = [&](auto guard) {
            constexpr bool GUARD = decltype(guard)::value;
#pragma unroll
            for (int kq = 0; kq < CKPT; ++kq) {
                const int k = CKPT - 1 - kq;
                const bool in = !GUARD || k < len;
                const float lp = pass(__fadd_rn(gr[k], __fmul_rn(br[k], hp)), k), lq = pass(__fmul_rn(br[k], hq), k);
                hp = in ? __fmul_rn(nr.am, lp) : hp;
                hq = in ? __fmul_rn(nr.am, lq) : hq;
                if (SYN) {
                    float np = __fadd_rn(mp, __fmul_rn(nr.k, lp));
                    if (EXTRA) np = __fadd_rn(np, qi[(EXTRA && SYN) ? k : 0]);
                    mp = in ? __fmul_rn(nr.as, np) : mp;
                    mq = in ? __fmul_rn(nr.as, __fadd_rn(mq, __fmul_rn(nr.k, lq))) : mq;
                    if (GUARD) mu_u = in ? __fmul_rn(nr.as, mu_u) : mu_u;
                }
            }
            if (!GUARD) mu_u = u_full;
        };
        if (whole) map(std::false_type{}); else map(std::true_type{});
        map_a[tid] = hp;
        map_b[tid] = hq;
        if (SYN) {
            map_c[tid] = mp;
            map_d[tid] = mq;
            map_u[tid] = mu_u;
        }
        const unsigned inside = len >= CKPT ? ~0u : (1u << len) - 1u;
        stops[tid] = ((open & inside) != inside ? 1 : 0) | (len == 0 || !((open >> (len - 1)) & 1u) ? 2 : 0);
        const auto finite = [](float f) { return fabsf(f) < __builtin_inff(); };
        const bool tame = finite(hp) && finite(hq) && (!SYN || (finite(mp) && finite(mq) && finite(mu_u)));
        const bool some = __builtin_amdgcn_ballot_w64(active && !tame) != 0;
        if ((tid & (WAVE - 1)) == 0) wild.of_wave[tid / WAVE] = some ? 1 : 0;
        __syncthreads();
        // what enters this chunk from later steps
        h = carry_h[lane];
        hm = SYN ? carry_m[lane] : 0.f;
        for (int c = chunks - 1; c > j; --c) {
            const int at_c = (c << neurons_log) + lane;
            const int stop = stops[at_c];
            if (SYN) {
                hm = __fadd_rn(map_c[at_c], __fmul_rn(map_u[at_c], hm));
                if (!(stop & 2)) hm = __fadd_rn(hm, __fmul_rn(map_d[at_c], h));
            }
            h = stop & 1 ? map_a[at_c] : __fadd_rn(map_a[at_c], __fmul_rn(map_b[at_c], h));
        }
        if (wild.all << (64 - 8 * (blockDim.x / WAVE))) {        // some wave's byte: chunk after chunk, results in map_a, map_c
            __syncthreads();                                     // everybody has read the maps
            for (int c = chunks - 1; c >= 0; --c) {
                if (j == c) {
                    h = c == chunks - 1 ? carry_h[lane] : map_a[tid + many];
                    if (SYN) hm = c == chunks - 1 ? carry_m[lane] : map_c[tid + many];
                    float h_out = h, m_out = hm;
                    unsigned through = open;                     // opaque copies: 64 masks kept for this rare block would
                    int steps_in = len;                          // push those of the walks out of their registers
                    asm volatile("" : "+v"(through), "+v"(steps_in));
#pragma unroll
                    for (int kq = 0; kq < CKPT; ++kq) {
                        const int k = CKPT - 1 - kq;
                        const float l = (through >> k) & 1u ? __fadd_rn(gr[k], __fmul_rn(br[k], h_out)) : 0.f;
                        if (SYN) {
                            float mu = __fadd_rn(m_out, __fmul_rn(l, nr.k));
                            if (EXTRA) mu = __fadd_rn(mu, qi[(EXTRA && SYN) ? k : 0]);
                            m_out = k < steps_in ? __fmul_rn(nr.as, mu) : m_out;
                        }
                        h_out = k < steps_in ? __fmul_rn(nr.am, l) : h_out;
                    }
                    map_a[tid] = h_out;
                    if (SYN) map_c[tid] = m_out;
                }
                __syncthreads();
            }
        }

        // the walk of the one-lane kernel
        auto walk = [&](auto guard) {
            constexpr bool GUARD = decltype(guard)::value;
#pragma unroll
            for (int kq = 0; kq < CKPT; ++kq) {
                const int k = CKPT - 1 - kq;
                if (!GUARD || k < len) {
                    const float lam = pass(__fadd_rn(gr[k], __fmul_rn(br[k], h)), k);
                    h = __fmul_rn(nr.am, lam);
                    acc_m.add(lam, k > 0 ? vp[k > 0 ? k - 1 : 0] : vp0);
                    acc_n.add(lam, xr[k]);
                    const float du = __fmul_rn(lam, nr.k);
                    if (SYN) {
                        float mu = __fadd_rn(hm, du);
                        if (EXTRA) mu = __fadd_rn(mu, qi[(EXTRA && SYN) ? k : 0]);
                        hm = __fmul_rn(nr.as, mu);
                        acc_s.add(mu, p.decay_early ? xr[k] : (k > 0 ? xr[k > 0 ? k - 1 : 0] : i0));
                        gr[k] = __fmul_rn(mu, xg);
                    } else {
                        gr[k] = du;
                    }
                }
                if (k % 8 == 0) {                                // short fp32 sums: 3 additions in fp64 each
                    acc_m.fold();
                    acc_n.fold();
                    acc_s.fold();
                }
            }
            const Rsrc ro = make_rsrc(q.grad_x + at, bytes);
#pragma unroll
            for (int k = 0; k < CKPT; ++k)
                IO::store(gr[k], ro, GUARD ? (k < len ? voff + k * step_bytes : BEYOND) : voff, GUARD ? 0u : k * step_bytes);
        };
        if (whole) walk(std::false_type{}); else walk(std::true_type{});
        __syncthreads();                                         // everybody has read the maps and the carry
        if (j == 0) {
            carry_h[lane] = h;
            carry_m[lane] = hm;
        }
    }

    part_m[tid] = p.norm_input ? acc_m.total - acc_n.total : acc_m.total;
    if (SYN) part_s[tid] = acc_s.total;
    __syncthreads();
    if (j != 0 || !active) return;
    if (q.v_init_grad) q.v_init_grad[row] = h;
    if (SYN && q.i_init_grad) q.i_init_grad[row] = hm;
    double sum_m = 0.0, sum_s = 0.0;
    for (int c = 0; c < chunks; ++c) {
        sum_m += part_m[(c << neurons_log) + lane];
        if (SYN) sum_s += part_s[(c << neurons_log) + lane];
    }
    if (q.alpha_mem_grad) q.alpha_mem_grad[row] = static_cast<float>(sum_m);
    if (SYN && q.alpha_syn_grad)
        q.alpha_syn_grad[row] = static_cast<float>(p.decay_early ? sum_s / static_cast<double>(nr.as) : sum_s);
}

template <bool SYN, int KIND, int CAPK, bool EXTRA, bool GO1>
int launch(const SplitArgs &a, int64_t B, hipStream_t s)
{
    const SplitShape shape = split_shape(B, a.T, a.M);
    if (shape.blocks_per_batch > 0x7fffffffLL / B) return hipErrorInvalidValue;
    hipLaunchKernelGGL((layer_lif_backward_split<SYN, KIND, CAPK, EXTRA, GO1>), dim3(static_cast<unsigned>(shape.blocks_per_batch * B)),
                       dim3(shape.lanes), 0, s, a, shape.blocks_per_batch, shape.neurons_log);
    return static_cast<int>(hipGetLastError());
}

template <bool SYN, int KIND>
int dispatch(const SplitArgs &a, bool uniform, int64_t B, hipStream_t s)
{
    if (a.grad_v_rec) return launch<SYN, KIND, 0, true, false>(a, B, s);   // one general instance, as in the one-lane kernel
    if constexpr (KIND != EXODUS_SURR_TENSOR) {
        if (uniform) {
            if (a.p.cap == 1u) return launch<SYN, KIND, 1, false, true>(a, B, s);
            if (a.p.cap == 2u) return launch<SYN, KIND, 2, false, true>(a, B, s);
            return launch<SYN, KIND, 0, false, true>(a, B, s);
        }
    }
    if (a.p.cap == 1u) return launch<SYN, KIND, 1, false, false>(a, B, s);
    if (a.p.cap == 2u) return launch<SYN, KIND, 2, false, false>(a, B, s);
    return launch<SYN, KIND, 0, false, false>(a, B, s);
}

template <bool SYN>
int dispatch_kind(const SplitArgs &a, int kind, bool uniform, int64_t B, hipStream_t s)
{
    switch (kind) {
        case EXODUS_SURR_TENSOR: return dispatch<SYN, EXODUS_SURR_TENSOR>(a, uniform, B, s);
        case EXODUS_SURR_SINGLE_EXP: return dispatch<SYN, EXODUS_SURR_SINGLE_EXP>(a, uniform, B, s);
        case EXODUS_SURR_PERIODIC_EXP: return dispatch<SYN, EXODUS_SURR_PERIODIC_EXP>(a, uniform, B, s);
        case EXODUS_SURR_HEAVISIDE: return dispatch<SYN, EXODUS_SURR_HEAVISIDE>(a, uniform, B, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

int exodus_layer_backward_split(const SplitArgs &a, bool syn, int kind, bool uniform, int64_t B, hipStream_t s)
{
    return syn ? dispatch_kind<true>(a, kind, uniform, B, s) : dispatch_kind<false>(a, kind, uniform, B, s);
}
