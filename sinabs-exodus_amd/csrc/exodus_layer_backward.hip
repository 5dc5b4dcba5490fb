// Backward kernel of the spiking layer on its own (batch, time, neurons) layout, one lane per neuron walking the whole
// sequence, and the choice between it and the kernel for layers with few neurons (exodus_layer_backward_split.hip).
#include "exodus_layer.hpp"

namespace {

// ---------------------------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------------------------
// With lambda_t = dL/du_t (membrane adjoint) and mu_t = dL/di_t (synapse adjoint):
//   g_t      = s_t * grad_spikes_t              (at the last step the gradients of the final states
//                                                join in: see below)
//   lambda_t = nc_t (g_t + (a_mem - a_mem c s_t) lambda_{t+1})
//   mu_t     = a_syn mu_{t+1} + k lambda_t,     k = norm_input ? 1 - a_mem : 1
//   grad_x_t = decay_early ? a_syn mu_t : mu_t  (no synapse: grad_x_t = k lambda_t)
//   grad_alpha_mem = sum_t lambda_t vpost_{t-1} - (norm_input ? sum_t lambda_t i_t : 0)
//   grad_alpha_syn = decay_early ? (sum_t mu_t i_t) / a_syn : sum_t mu_t i_{t-1}
//   grad_v_init = a_mem lambda_0,  grad_i_init = a_syn mu_0
// The final potential handed out by the forward is vpost_{T-1} = v_{T-1} - c count_{T-1}; a gradient
// gv on it reaches v_{T-1} directly and the spike count with weight -c, a gradient on the final
// synaptic current adds to mu_{T-1}.
// KIND == EXODUS_SURR_TENSOR reads the surrogate derivative of every step from `surr` (a third
// streamed tensor, whose register buffer costs the kernel one wave per SIMD); the other kinds
// evaluate it from the rebuilt potential and ignore `surr`.
// EXTRA: gradients also arrive at the per-step state records of the forward (grad_v_rec on the potential
// after each reset, with synapse grad_i_rec on each synaptic current): two more streamed inputs.
// GO1: the gradient of the spikes is one value for every neuron and step (the gradient of a sum of the
// output, which autograd hands over as a broadcast scalar): `grad_spikes` then points at that one float and the
// kernel streams one tensor less (8 instead of 12 bytes per neuron-timestep).
template <bool SYN, int KIND, int CAPK, bool NT, bool EXTRA, bool GO1 = false>
__global__ void __launch_bounds__(BWD_BLOCK)
    __attribute__((amdgpu_waves_per_eu(
        (KIND == EXODUS_SURR_TENSOR || EXTRA) ? 2 : (GO1 ? EXODUS_LAYER_BWD_WAVES_G1 : EXODUS_LAYER_BWD_WAVES),
        (KIND == EXODUS_SURR_TENSOR || EXTRA) ? 2 : (GO1 ? EXODUS_LAYER_BWD_WAVES_G1 : EXODUS_LAYER_BWD_WAVES))))
layer_lif_backward(
    float *__restrict__ grad_x, float *__restrict__ alpha_mem_grad, float *__restrict__ alpha_syn_grad,
    float *__restrict__ v_init_grad, float *__restrict__ i_init_grad, const float *__restrict__ grad_spikes,
    const float *__restrict__ grad_v_last, const float *__restrict__ grad_i_last, const float *__restrict__ x,
    const float *__restrict__ surr, const float *__restrict__ grad_v_rec, const float *__restrict__ grad_i_rec,
    const float *__restrict__ ckpt_v, const float *__restrict__ ckpt_i, const LayerConsts p, const float p0,
    const float p1, const float inv_p0, const int64_t blocks_per_batch, const int64_t T, const int64_t M, const unsigned run)
{
    typedef BufIO<1, NT> IO;
    const unsigned block_of_layer = layer_block(run);
    const int64_t b = block_of_layer / blocks_per_batch;
    const int64_t m0 = static_cast<int64_t>(block_of_layer - b * blocks_per_batch) * blockDim.x;
    const unsigned lane_off = threadIdx.x;
    // lanes past the end of the layer walk the same loops and meet every barrier, but all memory
    // accesses and all arithmetic sit behind `active`
    const bool active = m0 + lane_off < M;
    const int64_t row = b * M + m0 + lane_off;
    const int64_t n_ck = (T + CKPT - 1) / CKPT;
    // block-uniform bases; lane and step offsets are added by the buffer instructions
    const float *xp = x + (b * T) * M + m0;
    const float *gp = GO1 ? nullptr : grad_spikes + (b * T) * M + m0;
    const float g1 = GO1 ? grad_spikes[0] : 0.f;
    float *op = grad_x + (b * T) * M + m0;
    constexpr bool FROM_TENSOR = KIND == EXODUS_SURR_TENSOR;
    const float *srp = FROM_TENSOR ? surr + (b * T) * M + m0 : nullptr;
    const float *qvp = EXTRA ? grad_v_rec + (b * T) * M + m0 : nullptr;
    const float *qip = (EXTRA && SYN) ? grad_i_rec + (b * T) * M + m0 : nullptr;
    const float *cvp = ckpt_v + (b * n_ck) * M + m0;
    const float *cip = SYN ? ckpt_i + (b * n_ck) * M + m0 : nullptr;
    const unsigned voff = lane_off * 4u;
    const unsigned step_bytes = static_cast<unsigned>(M) * 4u;

    Cap cc;
    cc.cap = p.cap;
    cc.one = p.cap >= 1u ? 1.f : 0.f;
    Neuron nr = {};
    if (active) neuron_load<SYN, CAPK>(nr, p, row);
    const float xg = (SYN && p.decay_early) ? nr.as : 1.0f;   // factor between mu and grad_x
    const bool pair_new = p.decay_early != 0;                  // the synapse sum pairs i_t with mu_t (else mu_{t+1})
    const SurrConst sk = surrogate_consts<KIND>(nr.th, p0, p1);

    // Running adjoints.  Besides lambda_{t+1} and mu_{t+1} themselves the walk carries what reaches the
    // step below them, h = a_mem lambda_{t+1} and hm = a_syn mu_{t+1}: a gradient arriving at the final
    // states is then nothing but their initial value (the final potential is vpost_{T-1}, whose
    // gradient enters v_{T-1} with the same factor 1 - c s_{T-1} as a_mem lambda_T would), and no step
    // needs a special case.
    float lam = 0.f, mu = 0.f;
    float h = (active && grad_v_last) ? grad_v_last[row] : 0.f;
    float hm = (active && SYN && grad_i_last) ? grad_i_last[row] : 0.f;
    TileSum acc_m, acc_n, acc_s;                               // sums of lambda_{t+1} vpost_t, lambda_t i_t, mu i
    acc_m.clear();
    acc_n.clear();
    acc_s.clear();

    // One block of CKPT steps: load, rebuild forward from the checkpoint, walk in reverse, store.
    // GUARD = the block may end before CKPT steps (only the newest block of a sequence can).
    auto block = [&](const int64_t j, auto guard) {
        constexpr bool GUARD = decltype(guard)::value;
        const int64_t t0 = j * CKPT;
        const int len = GUARD ? static_cast<int>(T - t0) : CKPT;
        float xr[CKPT], gr[GO1 ? 1 : CKPT], vr[CKPT], sr[FROM_TENSOR ? CKPT : 1];   // (GO1: results go where the inputs were)
        float qv[EXTRA ? CKPT : 1], qi[(EXTRA && SYN) ? CKPT : 1];
        __syncthreads();                                   // keeps the block's waves at the same step
        if (!active) return;
        {
            // always CKPT loads per tensor (steps past the end re-read the last step): a constant number
            // of loads in flight lets each use wait for its own load only
            const Rsrc rx = make_rsrc(xp + t0 * M), rg = make_rsrc(GO1 ? nullptr : gp + t0 * M);
            const Rsrc rs = make_rsrc(FROM_TENSOR ? srp + t0 * M : nullptr);
            const Rsrc rqv = make_rsrc(EXTRA ? qvp + t0 * M : nullptr);
            const Rsrc rqi = make_rsrc((EXTRA && SYN) ? qip + t0 * M : nullptr);
            const unsigned last = static_cast<unsigned>(len - 1);
#pragma unroll
            for (int k = 0; k < CKPT; ++k) {
                const unsigned so = (GUARD ? (k < last ? k : last) : k) * step_bytes;
                xr[k] = IO::load(rx, voff, so);
                if (!GO1) gr[GO1 ? 0 : k] = IO::load(rg, voff, so);
                if (FROM_TENSOR) sr[k] = IO::load(rs, voff, so);
                if (EXTRA) qv[k] = IO::load(rqv, voff, so);
                if (EXTRA && SYN) qi[k] = IO::load(rqi, voff, so);
            }
        }
        nr.vpost = NT ? ld_stream(cvp + j * M + lane_off) : cvp[j * M + lane_off];
        nr.i = SYN ? (NT ? ld_stream(cip + j * M + lane_off) : cip[j * M + lane_off]) : 0.f;

        // rebuild the block: vr[k] = pre-reset potential, xr[k] = synaptic current (the value that
        // was normalised and fed to the membrane; without synapse that is the input itself)
#pragma unroll
        for (int k = 0; k < CKPT; ++k)
            if (!GUARD || k < len) {
                const float v = neuron_advance<SYN>(nr, xr[k]);
                nr.vpost = __fsub_rn(v, reset_amount<CAPK>(v, nr, cc));
                vr[k] = v;
                xr[k] = nr.i;
            }

        // reverse walk
#pragma unroll
        for (int kq = 0; kq < CKPT; ++kq) {
            const int k = CKPT - 1 - kq;
            if (!GUARD || k < len) {
                float v = vr[k];
                const float cur_i = xr[k];
                // The longer surrogate is evaluated when its step is reached, not for all 32 steps ahead of the walk
                // (which the compiler otherwise does: 32 more live values, spilled to memory): the empty statement makes
                // this step's potential depend on the adjoint that the previous one has produced.
                if (KIND == EXODUS_SURR_PERIODIC_EXP) asm volatile("" : "+v"(v) : "v"(h));
                const float sg = FROM_TENSOR ? sr[FROM_TENSOR ? k : 0] : surrogate<KIND>(v, nr.th, inv_p0, sk);
                const float vpost = __fsub_rn(v, reset_amount<CAPK>(v, nr, cc));
                acc_m.add(lam, vpost);                          // lambda_{t+1} * vpost_t
                const float through = __fsub_rn(1.0f, __fmul_rn(nr.c, sg));   // d vpost_t / d v_t
                // a gradient on the recorded vpost_t joins what the next step sends down to vpost_t
                const float below = EXTRA ? __fadd_rn(h, qv[EXTRA ? k : 0]) : h;
                const float l = __fadd_rn(__fmul_rn(sg, GO1 ? g1 : gr[GO1 ? 0 : k]), __fmul_rn(through, below));
                lam = v > nr.gate ? l : 0.f;                      // clamped (or NaN) steps pass nothing on
                h = __fmul_rn(nr.am, lam);
                acc_n.add(lam, cur_i);                          // lambda_t * i_t
                const float du = __fmul_rn(lam, nr.k);
                if (SYN) {
                    const float mu_next = mu;
                    mu = __fadd_rn(hm, du);
                    if (EXTRA) mu = __fadd_rn(mu, qi[(EXTRA && SYN) ? k : 0]);
                    hm = __fmul_rn(nr.as, mu);
                    acc_s.add(pair_new ? mu : mu_next, cur_i);
                    (GO1 ? xr[k] : gr[GO1 ? 0 : k]) = __fmul_rn(mu, xg);
                } else {
                    (GO1 ? xr[k] : gr[GO1 ? 0 : k]) = du;
                }
            }
        }
        {
            const Rsrc ro = make_rsrc(op + t0 * M);
#pragma unroll
            for (int k = 0; k < CKPT; ++k)
                if (!GUARD || k < len) IO::store(GO1 ? xr[k] : gr[GO1 ? 0 : k], ro, voff, k * step_bytes);
        }
        acc_m.fold();
        acc_n.fold();
        acc_s.fold();
    };

    int64_t j = n_ck - 1;
    if (T - j * CKPT < CKPT) {
        block(j, std::true_type{});
        --j;
    }
    for (; j >= 0; --j) block(j, std::false_type{});

    if (!active) return;                                       // no barrier follows
    if (v_init_grad) v_init_grad[row] = h;
    if (SYN && i_init_grad) i_init_grad[row] = hm;
    if (alpha_mem_grad) {
        acc_m.add(lam, p.v_init[row]);
        acc_m.fold();
        alpha_mem_grad[row] = static_cast<float>(p.norm_input ? acc_m.total - acc_n.total : acc_m.total);
    }
    if (SYN && alpha_syn_grad) {
        if (p.decay_early) {
            acc_s.total = acc_s.total / static_cast<double>(nr.as);
        } else {
            acc_s.add(mu, p.i_init[row]);
            acc_s.fold();
        }
        alpha_syn_grad[row] = static_cast<float>(acc_s.total);
    }
}

// 0: never, 1: for layers that leave most of the machine idle (default), 2: layers of any size without synapse, with a
// surrogate evaluated in the kernel, no gradients on state records and at most SPLIT_PLAIN_CHUNKS chunks, and no others,
// 3: whenever the kernel applies
std::atomic<int> split_mode{1};
// batch * neurons up to which mode 1 splits: the most at which no form of the call loses by it.  The split kernel does half
// as much again and more in arithmetic and holds fewer waves.  One lane / split, us, at 16 384 neurons (8, t, 2048), without
// synapse, with one, with one and state records, with a surrogate tensor: 64 steps 15.1 / 11.6, 15.0 / 12.9, 15.3 / 13.6,
// 14.1 / 11.2 (launches among them); 300 steps 40 / 23, 43 / 26, 46 / 38, 41 / 24; 2000 steps 223 / 96, 247 / 109, 292 / 177,
// 234 / 136.  At 32 768 neurons: 15.2 / 11.5, 15.3 / 13.9, 16.7 / 19.2, 15.5 / 11.0; 43 / 38, 49 / 46, 53 / 68, 47 / 39;
// 233 / 186, 265 / 206, 319 / 339, 258 / 253.
constexpr int64_t SPLIT_MOST_NEURONS = 16384;
constexpr int64_t SPLIT_PLAIN_CHUNKS = 16;

template <bool SYN, int KIND, int CAPK>
int launch_bwd(float *grad_x, float *am_g, float *as_g, float *v0_g, float *i0_g, const float *grad_spikes,
               const float *gvl, const float *gil, const float *x, const float *surr, const float *gvr,
               const float *gir, const float *ckpt_v, const float *ckpt_i, const LayerConsts &p, float p0, float p1,
               bool uniform, int64_t B, int64_t T, int64_t M, hipStream_t s)
{
    const bool whole = uniform ? whole_lines(M, {grad_x, x}) : whole_lines(M, {grad_x, grad_spikes, x, surr, gvr, gir});
    const int lanes = backward_lanes(B, M, gvr || surr, whole);
    const int64_t blocks_per_batch = (M + lanes - 1) / lanes;
    if (blocks_per_batch > 0x7fffffffLL / B) return hipErrorInvalidValue;
    const int64_t blocks = blocks_per_batch * B;
    const unsigned run =
        uniform ? neighbours_per_xcd(blocks, M, {grad_x, x}) : neighbours_per_xcd(blocks, M, {grad_x, grad_spikes, x, surr, gvr, gir});
#define EXODUS_LAUNCH(CK, NT, EX, G1)                                                                              \
    hipLaunchKernelGGL((layer_lif_backward<SYN, KIND, CK, NT, EX, G1>), dim3(static_cast<unsigned>(blocks)),      \
                       dim3(lanes), 0, s, grad_x, am_g, as_g, v0_g, i0_g, grad_spikes, gvl, gil, x, surr, gvr, \
                       gir, ckpt_v, ckpt_i, p, p0, p1, p0 != 0.f ? 1.f / p0 : 0.f, blocks_per_batch, T, M, run)
    if (uniform) {
        // one value as the gradient of every spike: instances exist for the in-kernel surrogates, without
        // gradients on the state records
        if constexpr (KIND == EXODUS_SURR_TENSOR) {
            return hipErrorInvalidValue;
        } else {
            if (gvr) return hipErrorInvalidValue;
            if (whole) EXODUS_LAUNCH(CAPK, true, false, true);
            else EXODUS_LAUNCH(CAPK, false, false, true);
        }
    } else if (gvr) {
        // gradients on the state records: one general instance per surrogate kind
        EXODUS_LAUNCH(0, false, true, false);
    } else if (whole) {
        EXODUS_LAUNCH(CAPK, true, false, false);
    } else {
        EXODUS_LAUNCH(CAPK, false, false, false);
    }
#undef EXODUS_LAUNCH
    return static_cast<int>(hipGetLastError());
}

template <bool SYN, int KIND, class... A>
int dispatch_bwd_cap(unsigned cap, A... a)
{
    if (cap == 1u) return launch_bwd<SYN, KIND, 1>(a...);
    if (cap == 2u) return launch_bwd<SYN, KIND, 2>(a...);
    return launch_bwd<SYN, KIND, 0>(a...);
}

}  // namespace

int exodus_layer_split_mode() { return split_mode.load(std::memory_order_relaxed); }

// ---------------------------------------------------------------------------------------------
// Checkpoint memory of exodus_layer_lif_backward_from_input, the one entry point that must not
// allocate.  Every GPU the library runs on holds its own copy of this array, at its own address,
// until the process ends.  In host code the array's name is only a handle for hipGetSymbolAddress:
// kernels get the device address looked up below, never the name.
// ---------------------------------------------------------------------------------------------
constexpr int64_t SCRATCH_FLOATS = int64_t{1} << 24;           // 64 MiB
static __device__ __align__(256) float scratch[SCRATCH_FLOATS];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex scratch_lock;
float *scratch_of_device[MAX_DEVICES] = {};

// device address of `scratch` on the current device (looked up once per device)
int scratch_address(float **out)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return static_cast<int>(e);
    if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> hold(scratch_lock);
    if (!scratch_of_device[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return static_cast<int>(e);
        if (!ptr) return hipErrorInvalidSymbol;
        scratch_of_device[dev] = static_cast<float *>(ptr);
    }
    *out = scratch_of_device[dev];
    return hipSuccess;
}

}  // namespace

extern "C" {

#define EXODUS_API __attribute__((visibility("default")))

EXODUS_API int exodus_layer_lif_backward(float *grad_input, float *alpha_mem_grad, float *alpha_syn_grad,
                                         float *vmem_init_grad, float *isyn_init_grad, const float *grad_spikes,
                                         const float *grad_v_last, const float *grad_i_last, const float *input,
                                         const float *ckpt_v, const float *ckpt_i, const float *vmem_post_initial,
                                         const float *isyn_initial, const float *alpha_mem, const float *alpha_syn,
                                         const float *membr_subtract, const float *theta, const float *theta_low,
                                         int apply_theta_low, int max_num_spikes, int decay_early, int norm_input,
                                         int surrogate_kind, float surr_p0, float surr_p1, const float *surr,
                                         const float *grad_v_rec, const float *grad_i_rec, int grad_spikes_uniform,
                                         int64_t batch, int64_t t, int64_t neurons, void *stream)
{
    if (bad3(batch, t, neurons)) return hipErrorInvalidValue;
    if (batch == 0 || t == 0 || neurons == 0) return hipSuccess;
    if (too_wide(neurons)) return hipErrorInvalidValue;
    const bool syn = alpha_syn != nullptr;
    if (grad_spikes_uniform && (surrogate_kind == EXODUS_SURR_TENSOR || grad_v_rec || grad_i_rec))
        return hipErrorInvalidValue;
    if (!grad_input || !grad_spikes || !input || !ckpt_v || !alpha_mem || !membr_subtract || !theta ||
        (apply_theta_low && !theta_low) || (syn && !ckpt_i) || (surrogate_kind == EXODUS_SURR_TENSOR && !surr))
        return hipErrorInvalidValue;
    if (surrogate_kind != EXODUS_SURR_TENSOR) surr = nullptr;
    if (syn ? ((grad_v_rec != nullptr) != (grad_i_rec != nullptr)) : grad_i_rec != nullptr) return hipErrorInvalidValue;
    if (alpha_mem_grad && !vmem_post_initial) return hipErrorInvalidValue;
    if (syn && alpha_syn_grad && !decay_early && !isyn_initial) return hipErrorInvalidValue;
    LayerConsts p;
    p.v_init = vmem_post_initial;
    p.i_init = isyn_initial;
    p.alpha_mem = alpha_mem;
    p.alpha_syn = alpha_syn;
    p.c = membr_subtract;
    p.theta = theta;
    p.theta_low = theta_low;
    p.apply_low = apply_theta_low ? 1 : 0;
    p.decay_early = decay_early ? 1 : 0;
    p.norm_input = norm_input ? 1 : 0;
    p.cap = static_cast<unsigned>(max_num_spikes);
    p.rec_pre = 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // few neurons, many steps: one lane per chunk of 32 steps instead of one lane per neuron
    const int mode = exodus_layer_split_mode();
    const bool plain = !syn && surrogate_kind != EXODUS_SURR_TENSOR && !grad_v_rec && t <= SPLIT_PLAIN_CHUNKS * CKPT;
    if (t > CKPT && exodus_layer_split_applies(neurons) &&
        ((mode == 1 && batch * neurons <= SPLIT_MOST_NEURONS) || (mode == 2 && plain) || mode == 3))
        return exodus_layer_backward_split(
            SplitArgs{grad_input, alpha_mem_grad, alpha_syn_grad, vmem_init_grad, isyn_init_grad, grad_spikes, grad_v_last,
                      syn ? grad_i_last : nullptr, input, surr, grad_v_rec, grad_i_rec, ckpt_v, ckpt_i, p, surr_p0, surr_p1,
                      surr_p0 != 0.f ? 1.f / surr_p0 : 0.f, t, neurons}, syn, surrogate_kind, grad_spikes_uniform != 0, batch, s);
#define EXODUS_BWD(SYN, K)                                                                                        \
    return dispatch_bwd_cap<SYN, K>(p.cap, grad_input, alpha_mem_grad, alpha_syn_grad, vmem_init_grad,            \
                                    isyn_init_grad, grad_spikes, grad_v_last, grad_i_last, input, surr,           \
                                    grad_v_rec, grad_i_rec, ckpt_v, ckpt_i, p, surr_p0, surr_p1,                  \
                                    grad_spikes_uniform != 0, batch, t, neurons, s)
    switch (surrogate_kind) {
        case EXODUS_SURR_TENSOR: if (syn) EXODUS_BWD(true, EXODUS_SURR_TENSOR); EXODUS_BWD(false, EXODUS_SURR_TENSOR);
        case EXODUS_SURR_SINGLE_EXP: if (syn) EXODUS_BWD(true, EXODUS_SURR_SINGLE_EXP); EXODUS_BWD(false, EXODUS_SURR_SINGLE_EXP);
        case EXODUS_SURR_PERIODIC_EXP: if (syn) EXODUS_BWD(true, EXODUS_SURR_PERIODIC_EXP); EXODUS_BWD(false, EXODUS_SURR_PERIODIC_EXP);
        case EXODUS_SURR_HEAVISIDE: if (syn) EXODUS_BWD(true, EXODUS_SURR_HEAVISIDE); EXODUS_BWD(false, EXODUS_SURR_HEAVISIDE);
        default: return hipErrorInvalidValue;
    }
#undef EXODUS_BWD
}

EXODUS_API int exodus_layer_backward_time_split(int mode)
{
    const int before = split_mode.load(std::memory_order_relaxed);
    if (mode >= 0 && mode <= 3) split_mode.store(mode, std::memory_order_relaxed);
    return before;
}

EXODUS_API int64_t exodus_layer_scratch_floats(void) { return SCRATCH_FLOATS; }

EXODUS_API int exodus_layer_lif_backward_from_input(
    float *grad_input, float *alpha_mem_grad, float *alpha_syn_grad, float *vmem_init_grad, float *isyn_init_grad,
    const float *grad_spikes, const float *grad_v_last, const float *grad_i_last, const float *input,
    const float *vmem_post_initial, const float *isyn_initial, const float *alpha_mem, const float *alpha_syn,
    const float *membr_subtract, const float *theta, const float *theta_low, int apply_theta_low, int max_num_spikes,
    int decay_early, int norm_input, int surrogate_kind, float surr_p0, float surr_p1, const float *surr,
    const float *grad_v_rec, const float *grad_i_rec, int grad_spikes_uniform, int64_t batch, int64_t t,
    int64_t neurons, void *stream)
{
    if (bad3(batch, t, neurons)) return hipErrorInvalidValue;
    if (batch == 0 || t == 0 || neurons == 0) return hipSuccess;
    if (too_wide(neurons)) return hipErrorInvalidValue;
    const bool syn = alpha_syn != nullptr;
    if (!grad_input || !grad_spikes || !input || !vmem_post_initial || !alpha_mem || !membr_subtract || !theta ||
        (apply_theta_low && !theta_low) || (syn && !isyn_initial) ||
        (surrogate_kind == EXODUS_SURR_TENSOR && !surr) || surrogate_kind < EXODUS_SURR_TENSOR ||
        surrogate_kind > EXODUS_SURR_HEAVISIDE ||
        (grad_spikes_uniform && (surrogate_kind == EXODUS_SURR_TENSOR || grad_v_rec || grad_i_rec)))
        return hipErrorInvalidValue;
    if (syn ? ((grad_v_rec != nullptr) != (grad_i_rec != nullptr)) : grad_i_rec != nullptr) return hipErrorInvalidValue;
    // checkpoints of one batch element; the batch is walked in slices of as many elements as fit
    const int64_t n_ck = (t + CKPT - 1) / CKPT;
    if (n_ck > SCRATCH_FLOATS / neurons) return EXODUS_ERROR_SCRATCH_TOO_SMALL;
    const int64_t per_element = ((n_ck * neurons + 63) / 64) * 64;          // each tensor starts on a 256-byte boundary
    const int64_t fit = SCRATCH_FLOATS / (per_element * (syn ? 2 : 1));
    if (fit < 1) return EXODUS_ERROR_SCRATCH_TOO_SMALL;
    float *base = nullptr;
    if (const int rc = scratch_address(&base)) return rc;
    LayerConsts p;
    p.v_init = vmem_post_initial;
    p.i_init = isyn_initial;
    p.alpha_mem = alpha_mem;
    p.alpha_syn = alpha_syn;
    p.c = membr_subtract;
    p.theta = theta;
    p.theta_low = theta_low;
    p.apply_low = apply_theta_low ? 1 : 0;
    p.decay_early = decay_early ? 1 : 0;
    p.norm_input = norm_input ? 1 : 0;
    p.cap = static_cast<unsigned>(max_num_spikes);
    p.rec_pre = 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto at = [](auto *q, int64_t offset) { return q ? q + offset : q; };   // absent tensors stay absent
    for (int64_t b0 = 0; b0 < batch; b0 += fit) {
        const int64_t nb = batch - b0 < fit ? batch - b0 : fit;
        const int64_t el = b0 * t * neurons, row = b0 * neurons;             // offsets of this slice
        float *ckpt_v = base, *ckpt_i = syn ? base + fit * per_element : nullptr;
        // the checkpoints of a slice are laid out (nb, n_ck, neurons) without padding between elements
        LayerConsts q = p;
        q.v_init = at(p.v_init, row);
        q.i_init = at(p.i_init, row);
        q.alpha_mem = at(p.alpha_mem, row);
        q.alpha_syn = at(p.alpha_syn, row);
        q.c = at(p.c, row);
        q.theta = at(p.theta, row);
        q.theta_low = at(p.theta_low, row);
        const int rc = exodus_layer_checkpoints_only(ckpt_v, ckpt_i, input + el, q, syn, nb, t, neurons, s);
        if (rc) return rc;
        const int rb = exodus_layer_lif_backward(
            at(grad_input, el), at(alpha_mem_grad, row), at(alpha_syn_grad, row), at(vmem_init_grad, row),
            at(isyn_init_grad, row), grad_spikes_uniform ? grad_spikes : at(grad_spikes, el), at(grad_v_last, row),
            at(grad_i_last, row), input + el,
            ckpt_v, ckpt_i, q.v_init, q.i_init, q.alpha_mem, q.alpha_syn, q.c, q.theta, q.theta_low, apply_theta_low,
            max_num_spikes, decay_early, norm_input, surrogate_kind, surr_p0, surr_p1, at(surr, el), at(grad_v_rec, el),
            at(grad_i_rec, el), grad_spikes_uniform, nb, t, neurons, stream);
        if (rb) return rb;
    }
    return hipSuccess;
}

}  // extern "C"
