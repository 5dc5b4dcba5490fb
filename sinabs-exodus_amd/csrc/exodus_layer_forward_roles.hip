// Forward kernel of the spiking layer on its own (batch, time, neurons) layout for layers with few neurons: three or four waves
// share the work on 64 neurons.
#include "exodus_layer.hpp"

namespace {

// A layer of a few thousand neurons is a handful of waves with a SIMD each, and a step costs a lone wave the number of its
// instructions: 2.35 ns for a vector or scalar instruction, whether it depends on the one before or not, about 7 for a load or a
// store.  So the instructions of a step are dealt out to waves on SIMDs of their own, each working for the same 64 neurons: one
// loads the input and scales it, with a synapse one works out its current, one does what the spikes depend on and nothing else,
// one stores the counts and adds them up.  They hand each other stages of STAGE steps through LDS, a barrier per stage; those in
// the middle ask for a stage while they work on the one before.  The operations and their order are those of layer_lif_forward
// (exodus_layer.hip), so the bits are the same.
// One wave for everything / this, us: (4, 2000, 512) 81.2 / 46.1, with synapses 87.6 / 44.4, with synapses, a bound and at most
// two spikes 95.4 / 53.5, at most one spike 77.3 / 41.6; (64, 300, 10) 16.9 / 11.6; (32, 100, 512) 11.1 / 10.1; (8, 100, 256)
// 9.8 / 8.0.  A stage takes 0.31 us for the membrane's wave, 0.17 of which are its 72 instructions; what remains is the barrier,
// the way through LDS and the counts of two or more spikes, which are worked out again ("redo").
constexpr int STAGE = 16, QUADS = STAGE / 4;         // steps; four steps of a neuron lie together in LDS
constexpr int DEPTH = 4;                             // stages of input in flight: a stage takes a quarter of the memory's latency
static_assert(CKPT == 2 * STAGE, "a checkpoint in front of every even stage");

typedef f32x4 Stage[QUADS][WAVE];

template <bool SYN, int CAPK, bool LOW>
__global__ void __launch_bounds__((SYN ? 4 : 3) * WAVE) layer_lif_forward_roles(
    float *__restrict__ spikes, float *__restrict__ ckpt_v, float *__restrict__ ckpt_i, float *__restrict__ v_last,
    float *__restrict__ i_last, const Sums sums, const float *__restrict__ x, const LayerConsts p, const int64_t blocks_per_batch,
    const int64_t T, const int64_t M)
{
    typedef BufIO<1, false> IO;
    // between the waves: scaled inputs (with a synapse), currents into the membrane, counts.  Four slots where the reader may come
    // back to the stage it works on (the membrane's exact steps), two elsewhere.
    __shared__ Stage inputs[SYN ? 2 : 1], currents[4], counts[2];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const unsigned lane = threadIdx.x & (WAVE - 1);
    const int64_t b = blockIdx.x / blocks_per_batch, part_of_b = blockIdx.x - b * blocks_per_batch;
    const int64_t m0 = part_of_b * WAVE;
    // lanes past the end of the layer compute on the block's first neuron; their offsets lie beyond every resource
    const bool active = m0 + lane < M;
    const int64_t row = b * M + m0 + (active ? lane : 0);
    const unsigned voff = active ? lane * 4u : BEYOND;
    const unsigned step_bytes = static_cast<unsigned>(M) * 4u;     // STAGE steps stay below 2^31 bytes (the host sees to it)
    const unsigned row_bytes = static_cast<unsigned>(M - m0) * 4u;
    const int64_t n_ck = (T + CKPT - 1) / CKPT, stage_floats = STAGE * M, at = b * T * M + m0, at_ck = b * n_ck * M + m0;
    const int full = static_cast<int>(T / STAGE), rest = static_cast<int>(T - static_cast<int64_t>(full) * STAGE);
    const int stages = full + (rest ? 1 : 0);
    // In the tick (between two barriers) t the loading wave prepares stage t, the synapse's works on t - 2 and the membrane's on
    // t - LAST + 1, the last one stores stage t - LAST.  All waves meet `ticks` barriers.
    constexpr int SYNAPSE = 2, MEMBRANE = SYN ? 4 : 2, LAST = MEMBRANE + 1;
    const int ticks = (stages + LAST + DEPTH - 1) / DEPTH * DEPTH;
    // bytes from the first step of a stage to the end of its last one
    const auto bytes = [&](int stage) {
        const int len = stage < full ? STAGE : (stage == full ? rest : 0);
        return len > 0 ? (len - 1) * step_bytes + row_bytes : 0u;
    };
    const auto offsets = [&](unsigned(&off)[STAGE]) {              // all in the vector part: the range check is exact
#pragma unroll
        for (int u = 0; u < STAGE; ++u) off[u] = voff + u * step_bytes;
    };
    const auto idle = [](int from, int to) {
        for (int t = from; t < to; ++t) __syncthreads();
    };
    // A wave in the middle: from tick `lag` on stage after stage, work(values, stage, steps in it, GUARD); the stage to come is
    // read from `ring` meanwhile.
    const auto pipeline = [&](int lag, const auto &ring, auto &&keep, auto &&work) {
        constexpr int SLOTS = sizeof(ring) / sizeof(Stage);
        f32x4 a[QUADS], c[QUADS];
        const auto read = [&](f32x4(&to)[QUADS], int stage) {
#pragma unroll
            for (int k = 0; k < QUADS; ++k) to[k] = ring[stage & (SLOTS - 1)][k][lane];
            __builtin_amdgcn_sched_barrier(0);
        };
        idle(0, lag - 1);
        read(a, 0);
        __syncthreads();
        int s = 0;
        for (; s + 2 <= full; s += 2) {
            read(c, s + 1);
            keep(s / 2);
            work(a, s, STAGE, std::false_type{});
            __syncthreads();
            read(a, s + 2);
            work(c, s + 1, STAGE, std::false_type{});
            __syncthreads();
        }
#pragma unroll 1
        for (; s < stages; ++s) {                                  // a full one at most, and the rest
            read(c, s + 1);
            if (s % 2 == 0) keep(s / 2);
            work(a, s, s < full ? STAGE : rest, std::true_type{});
            __syncthreads();
#pragma unroll
            for (int k = 0; k < QUADS; ++k) a[k] = c[k];
        }
        idle(lag + stages, ticks);
    };
    const auto checkpoint = [&](float *to, float value, int64_t j) {
        IO::store(value, make_rsrc(to + (to ? at_ck + j * M : 0), to ? row_bytes : 0u), voff, 0);
    };
    Cap cc;
    cc.cap = p.cap;
    cc.one = p.cap >= 1u ? 1.f : 0.f;
    Neuron n = {};
    neuron_load<SYN, CAPK>(n, p, row);
    decays_load<SYN>(n, p, b, row - b * M, row, active && wave == 0);

    if (wave == 0) {
        float scale = SYN ? n.xs : n.k;
        asm volatile("" : "+v"(scale));                            // there before the loop
        unsigned off[STAGE];
        offsets(off);
        float in[DEPTH][STAGE];
        const float *from = x + at;
        const auto fetch = [&](float(&to)[STAGE], int stage) {
            const unsigned size = bytes(stage);
            const Rsrc r = make_rsrc(size ? from : x, size);
#pragma unroll
            for (int u = 0; u < STAGE; ++u) to[u] = IO::load(r, off[u], 0);
            __builtin_amdgcn_sched_barrier(0);
            from += stage_floats;
        };
#pragma unroll
        for (int q = 0; q < DEPTH; ++q) fetch(in[q], q);
        for (int t = 0; t < ticks; t += DEPTH) {
#pragma unroll
            for (int q = 0; q < DEPTH; ++q) {                      // (what lies past the end of the sequence is zeros)
                Stage &to = SYN ? inputs[q & 1] : currents[q];
#pragma unroll
                for (int k = 0; k < QUADS; ++k) {
                    f32x4 out;
#pragma unroll
                    for (int e = 0; e < 4; ++e) out[e] = __fmul_rn(SYN ? in[q][k * 4 + e] : scale, SYN ? scale : in[q][k * 4 + e]);
                    to[k][lane] = out;
                }
                fetch(in[q], t + q + DEPTH);
                __syncthreads();
            }
        }
    } else if (SYN && wave == 1) {
        n.i = p.i_init[row];
        settle(n);
        pipeline(SYNAPSE, inputs, [&](int64_t j) { checkpoint(ckpt_i, n.i, j); },
                 [&](const f32x4(&from)[QUADS], int stage, int len, auto guard) {
                     constexpr bool GUARD = decltype(guard)::value;
#pragma unroll
                     for (int k = 0; k < QUADS; ++k) {
                         f32x4 out;
#pragma unroll
                         for (int e = 0; e < 4; ++e) {
                             const float i = __fadd_rn(__fmul_rn(n.i, n.as), from[k][e]);
                             n.i = !GUARD || k * 4 + e < len ? i : n.i;
                             out[e] = __fmul_rn(n.k, n.i);
                         }
                         currents[stage & 3][k][lane] = out;
                     }
                 });
        if (i_last && active) i_last[row] = n.i;
    } else if (wave == (SYN ? 2 : 1)) {
        float scale, shift, redo;
        spike_line(scale, shift, redo, n, cc);
        n.vpost = p.v_init[row];
        settle(n);
        asm volatile("" : "+v"(scale), "+v"(shift), "+v"(redo));
        bool careful = false;                                      // exact steps to come; uniform over the wave
        const auto potential = [&](float u) {
            const float v = __fadd_rn(__fmul_rn(n.vpost, n.am), u);
            return LOW ? __builtin_elementwise_maximum(v, n.lo) : v;
        };
        // The exact steps, `top` and `redo` as in layer_lif_forward; the stage's currents are still in their slot.
        const auto exact = [&](int stage, int len) {
            float top = -__builtin_inff();
#pragma unroll 1
            for (int k = 0; k < QUADS; ++k) {
                const f32x4 u = currents[stage & 3][k][lane];
                f32x4 out;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = potential(u[e]), count = spike_count_fast<CAPK>(v, n, cc);
                    const bool in = k * 4 + e < len;
                    n.vpost = in ? __fsub_rn(v, __fmul_rn(count, n.c)) : n.vpost;
                    top = in ? fmaxf(top, v) : top;
                    out[e] = in ? count : 0.f;
                }
                counts[stage & 1][k][lane] = out;
            }
            careful = __builtin_amdgcn_ballot_w64(top >= redo) != 0;
        };
        pipeline(MEMBRANE, currents, [&](int64_t j) { checkpoint(ckpt_v, n.vpost, j); },
                 [&](const f32x4(&from)[QUADS], int stage, int len, auto guard) {
                     constexpr bool GUARD = decltype(guard)::value;
                     if (careful) {
                         exact(stage, len);
                         return;
                     }
                     const float before = n.vpost;
                     float top = -__builtin_inff();
#pragma unroll
                     for (int k = 0; k < QUADS; ++k) {
                         f32x4 out;
#pragma unroll
                         for (int e = 0; e < 4; ++e) {
                             const float v = potential(from[k][e]);
                             float count = saturate(__fmaf_rn(v, scale, shift));
                             if (CAPK == 2) count += saturate(__fmaf_rn(v, 0.5f * scale, shift));
                             const float after = __fmaf_rn(-count, n.c, v);
                             const bool in = !GUARD || k * 4 + e < len;
                             n.vpost = in ? after : n.vpost;
                             top = in ? fmaxf(top, v) : top;
                             out[e] = in ? count : 0.f;
                         }
                         counts[stage & 1][k][lane] = out;
                     }
                     if (__builtin_amdgcn_ballot_w64(top >= redo) != 0) {
                         n.vpost = before;
                         exact(stage, len);
                         careful = true;
                     }
                 });
        if (active) v_last[row] = n.vpost;
    } else {
        unsigned off[STAGE];
        offsets(off);
        double mine = 0.0;
        float *to = spikes + at;
        idle(0, LAST);
        for (int s = 0; s < stages; ++s) {
            const Rsrc r = make_rsrc(to, bytes(s));                // steps past the end lie past it
            float part = 0.f;                                      // exact: zeros past the end
#pragma unroll
            for (int k = 0; k < QUADS; ++k) {
                const f32x4 c = counts[s & 1][k][lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    IO::store(c[e], r, off[k * 4 + e], 0);
                    part += c[e];
                }
            }
            mine += static_cast<double>(part);
            to += stage_floats;
            __syncthreads();
        }
        idle(LAST + stages, ticks);
        if (sums.at) {
            mine = active ? mine : 0.0;
#pragma unroll
            for (int apart = WAVE / 2; apart > 0; apart >>= 1) mine += __shfl_xor(mine, apart, WAVE);
            if (lane == 0) {
                if (sums.slots) sums.at[blockIdx.x] = mine;        // one slot per block
                else if (mine != 0.0) atomicAdd(sums.at, mine);
            }
        }
    }
}

template <bool SYN, int CAPK>
int launch(float *spikes, float *ckpt_v, float *ckpt_i, float *v_last, float *i_last, const Sums &sums, const float *x,
           const LayerConsts &p, int64_t B, int64_t T, int64_t M, hipStream_t s)
{
    const int64_t blocks_per_batch = (M + WAVE - 1) / WAVE;
    const dim3 grid(static_cast<unsigned>(blocks_per_batch * B)), block((SYN ? 4 : 3) * WAVE);
    if (p.apply_low)
        hipLaunchKernelGGL((layer_lif_forward_roles<SYN, CAPK, true>), grid, block, 0, s, spikes, ckpt_v, ckpt_i, v_last, i_last,
                           sums, x, p, blocks_per_batch, T, M);
    else
        hipLaunchKernelGGL((layer_lif_forward_roles<SYN, CAPK, false>), grid, block, 0, s, spikes, ckpt_v, ckpt_i, v_last, i_last,
                           sums, x, p, blocks_per_batch, T, M);
    return static_cast<int>(hipGetLastError());
}

}  // namespace

// One block per compute unit at most, which leaves each wave a SIMD of its own, and more than one checkpoint interval: the first
// stages pass three to five barriers before anything is stored.  layer_lif_forward / this, us: 17 steps of (16, t, 1024), 256
// blocks, 6.6 / 7.8, 33 steps 7.9 / 7.9, 300 steps 20.0 / 15.4; 512 blocks (32, t, 1024) 33 steps 8.9 / 9.3, 300 steps
// 22.9 / 20.4, but (24, 250, 1323) with 504 blocks 21.0 / 21.9.
bool exodus_layer_forward_roles_apply(int64_t B, int64_t T, int64_t M)
{
    return T > CKPT && B * ((M + WAVE - 1) / WAVE) <= compute_units() && M < (int64_t{1} << 24) && T < (int64_t{1} << 30);
}

int exodus_layer_forward_roles(float *spikes, float *ckpt_v, float *ckpt_i, float *v_last, float *i_last, const Sums &sums,
                               const float *x, const LayerConsts &p, int64_t B, int64_t T, int64_t M, hipStream_t s)
{
    const auto run = [&](auto syn) {
        constexpr bool SYN = decltype(syn)::value;
        if (p.cap == 1u) return launch<SYN, 1>(spikes, ckpt_v, ckpt_i, v_last, i_last, sums, x, p, B, T, M, s);
        if (p.cap == 2u) return launch<SYN, 2>(spikes, ckpt_v, ckpt_i, v_last, i_last, sums, x, p, B, T, M, s);
        return launch<SYN, 0>(spikes, ckpt_v, ckpt_i, v_last, i_last, sums, x, p, B, T, M, s);
    };
    return p.alpha_syn ? run(std::true_type{}) : run(std::false_type{});
}
