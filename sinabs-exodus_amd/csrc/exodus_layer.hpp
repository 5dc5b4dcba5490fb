// Shared by the translation units of the layer-layout kernels (exodus_layer.hip: the forward pass and the leaky
// integrator; exodus_layer_backward.hip: the backward pass of the spiking layer): memory access, the per-neuron step
// and the host helpers of the dispatch.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <initializer_list>
#include <mutex>
#include <type_traits>

#include "exodus_common.hpp"

// One decay factor's time constant, where a forward kernel works the factors out itself (tau null: it does not).
struct Decay {
    const float *tau = nullptr;
    float *alpha = nullptr, *kept = nullptr;     // what it writes: the factors, and a copy of the constants
    int one = 0;                                 // one constant for all neurons
};

struct LayerConsts {
    const float *v_init, *i_init, *alpha_mem, *alpha_syn, *c, *theta, *theta_low;
    int apply_low, decay_early, norm_input;
    unsigned cap;
    int rec_pre;        // the potential record holds the value before the reset instead of after it
    Decay mem, syn;     // forward kernels only
};

// where a forward kernel puts what its blocks counted
struct Sums {
    double *at;          // null: no total wanted
    bool slots;          // one double per block's lanes neurons of a batch element, else one double in all
};

namespace {

#ifndef EXODUS_LAYER_BLOCK
#define EXODUS_LAYER_BLOCK 256        // lanes per block of the kernels that hold several neurons per lane
#endif
#ifndef EXODUS_LAYER_BWD_BLOCK
#define EXODUS_LAYER_BWD_BLOCK 256    // lanes per block of the spiking backward kernel (one neuron per lane)
#endif
#ifndef EXODUS_LEAKY_WAVES
#define EXODUS_LEAKY_WAVES 8          // waves per CU the leaky kernels want before a lane takes more than one neuron
#endif
#ifndef EXODUS_WHOLE_NEURONS
#define EXODUS_WHOLE_NEURONS 16       // neurons per step must be a multiple of this for the non-temporal kernel instances
#endif
#ifndef EXODUS_LAYER_BWD_WAVES
#define EXODUS_LAYER_BWD_WAVES 3      // resident waves per SIMD the backward kernel is compiled for
#endif
#ifndef EXODUS_LAYER_BWD_WAVES_G1
#define EXODUS_LAYER_BWD_WAVES_G1 3   // ... and its instances that stream one tensor less (one gradient value for all): a
                                      // fourth wave fits them only with spills and measures no faster
#endif
constexpr int CKPT = 32;                              // steps between checkpoints = length of a backward chunk
constexpr int fwd_unroll(int npl) { return npl == 1 ? 16 : 8; }   // forward steps per software-pipeline stage (divides CKPT / 2)
constexpr int BLOCK = EXODUS_LAYER_BLOCK;
constexpr int BWD_BLOCK = EXODUS_LAYER_BWD_BLOCK;

template <int NPL> struct Vec;
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <> struct Vec<1> { typedef float type; };
template <> struct Vec<2> { typedef f32x2 type; };
template <> struct Vec<4> { typedef f32x4 type; };

template <int NPL> __device__ __forceinline__ float lane_get(const typename Vec<NPL>::type &v, int e);
template <> __device__ __forceinline__ float lane_get<1>(const float &v, int) { return v; }
template <> __device__ __forceinline__ float lane_get<2>(const f32x2 &v, int e) { return v[e]; }
template <> __device__ __forceinline__ float lane_get<4>(const f32x4 &v, int e) { return v[e]; }
template <int NPL> __device__ __forceinline__ void lane_put(typename Vec<NPL>::type &v, int e, float x);
template <> __device__ __forceinline__ void lane_put<1>(float &v, int, float x) { v = x; }
template <> __device__ __forceinline__ void lane_put<2>(f32x2 &v, int e, float x) { v[e] = x; }
template <> __device__ __forceinline__ void lane_put<4>(f32x4 &v, int e, float x) { v[e] = x; }

// ---------------------------------------------------------------------------------------------
// memory access: raw buffer instructions
// ---------------------------------------------------------------------------------------------
// Every (batch, time, neurons) access of a block has the form
//     block-uniform base (SGPR pair inside a buffer resource)  +  step * neurons * 4 (SGPR)
//                                                              +  lane offset (one VGPR, loop-invariant)
// which is exactly what a buffer instruction adds up by itself, so no access needs vector
// arithmetic or 64-bit address registers.  The one-lane backward kernel guards every access by code
// and sets num_records to the maximum; the forward, the leaky and the split backward kernels give
// every resource its end and let the hardware's range check drop what lanes and steps past the end
// of the layer ask for (BEYOND below), so that no branch surrounds a load or a store.
typedef __amdgpu_buffer_rsrc_t Rsrc;
// Cache hint of the streamed accesses (bit 1 = non-temporal).  Streaming data that nobody reads twice
// is marked non-temporal, which measures a few percent faster; but when a step's neurons do not start
// and end on 64-byte sectors (neuron count not a multiple of 16, or a view at an odd offset) neighbouring
// waves and blocks share sectors, and a non-temporal line is dropped before the neighbour gets to it:
// reads from memory grow by a third and partial writes appear.  Such layers use NT = false.
// All kernels put a workgroup barrier in front of every group of loads (the waves of a block share no
// data; the barrier only keeps them at the same step): waves that ask for the two halves of a line at
// the same moment are served by one fetch, waves that have drifted apart are not (+10-15 % where lines
// are shared), and neighbouring pieces requested together also suit the memory better when nothing is
// shared (+1-2 %).
template <bool NT> struct Aux {
    static constexpr int load = (NT && EXODUS_NT_LOAD) ? 2 : 0;
    static constexpr int store = (NT && EXODUS_NT_STORE) ? 2 : 0;
};

__device__ __forceinline__ Rsrc make_rsrc(const float *base)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, -1, 0x00020000);
}

// The same with an end: accesses at `bytes` or beyond read zeros and store nothing.  BEYOND is such an offset for every
// resource of up to 2^31 bytes (16 steps of the widest layer), with any step offset below 2^31 added to it.
__device__ __forceinline__ Rsrc make_rsrc(const float *base, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, static_cast<int>(bytes), 0x00020000);
}
constexpr unsigned BEYOND = 0x80000000u;

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

template <int NPL, bool NT> struct BufIO;
template <bool NT> struct BufIO<1, NT> {
    static __device__ __forceinline__ float load(Rsrc r, unsigned voff, unsigned soff)
    {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, Aux<NT>::load));
    }
    static __device__ __forceinline__ void store(float v, Rsrc r, unsigned voff, unsigned soff)
    {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, Aux<NT>::store);
    }
};
template <bool NT> struct BufIO<2, NT> {
    static __device__ __forceinline__ f32x2 load(Rsrc r, unsigned voff, unsigned soff)
    {
        return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, Aux<NT>::load));
    }
    static __device__ __forceinline__ void store(f32x2 v, Rsrc r, unsigned voff, unsigned soff)
    {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, Aux<NT>::store);
    }
};
template <bool NT> struct BufIO<4, NT> {
    static __device__ __forceinline__ f32x4 load(Rsrc r, unsigned voff, unsigned soff)
    {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, Aux<NT>::load));
    }
    // A 16-byte store takes more than one pass to read its data registers.  The compiler keeps the
    // next instruction from overwriting them only when the store has no SGPR offset; with one, a
    // vector instruction that rewrites the data right behind the store corrupted the last lanes of
    // each group of 16 on gfx950 (seen as sporadic wrong outputs when two blocks shared a compute
    // unit).  So the step offset travels in the vector offset here and the scalar offset stays 0, and a
    // short wait that reads the data keeps every writer away until the store has taken it.
    static __device__ __forceinline__ void store(f32x4 v, Rsrc r, unsigned voff, unsigned soff)
    {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voff + soff, 0, Aux<NT>::store);
        asm volatile("s_nop 1" : : "v"(v));                    // the data registers stay untouched two more cycles
    }
};

// ---------------------------------------------------------------------------------------------
// one neuron
// ---------------------------------------------------------------------------------------------
// Per-neuron constants and running state.  The layer's options are folded into the constants so
// that the step itself has no option-dependent code: a factor that an option switches off is 1
// (multiplying by 1 is exact), a bound that is switched off is an infinity.
struct Neuron {
    float am, as;       // decay factors of membrane and synapse
    float k;            // factor on the current entering the membrane: 1 - alpha_mem (norm_input) or 1
    float xs;           // factor on the input entering the synapse: alpha_syn (decay_early) or 1
    float c, th;        // subtract value, threshold
    float c2;           // 2 * subtract value (exact), what two spikes take away
    float th2;          // 2 * threshold: from here on a second spike (NaN, so never, where th is not positive)
    float thd;          // from here on the spike count needs the quotient v / th (+inf if never)
    float lo;           // lower bound of the potential, -inf without one
    float gate;         // gradients pass where the potential lies above
    float vpost, i;     // potential after the reset of the previous step, synaptic current
};

// The values of a neuron are in their registers from here on (an empty statement that uses them all).
__device__ __forceinline__ void settle(Neuron &n)
{
    asm volatile("" : "+v"(n.am), "+v"(n.as), "+v"(n.k), "+v"(n.xs), "+v"(n.c), "+v"(n.th), "+v"(n.lo), "+v"(n.vpost), "+v"(n.i));
}

// spike-count cap as the kernels use it (block-uniform)
struct Cap {
    float one;          // min(cap, 1)
    unsigned cap;
};

// CAPK: 1 = at most one spike per step, 2 = at most two, 0 = any other cap (none, 0, >= 3)
template <bool SYN, int CAPK>
__device__ __forceinline__ void neuron_load(Neuron &n, const LayerConsts &p, int64_t row)
{
    n.am = p.alpha_mem[row];
    n.as = SYN ? p.alpha_syn[row] : 0.f;
    n.k = p.norm_input ? __fsub_rn(1.0f, n.am) : 1.0f;
    n.xs = (SYN && p.decay_early) ? n.as : 1.0f;
    n.c = p.c[row];
    n.c2 = __fadd_rn(n.c, n.c);
    n.th = p.theta[row];
    // For th > 0:  v >= th <=> RN(v/th) >= 1  and  v >= 2 th <=> RN(v/th) >= 2  (2 th is exact and no
    // float lies between its predecessor and the rounding boundary of the quotient), so counts up to
    // 2 need no division.  Everything else -- more than two spikes, or a threshold that is not
    // positive -- takes the quotient.
    // A subtract value whose double is beyond the floats' range goes there, too, so that count * c is exact below n.thd.
    const bool plain = n.th > 0.f && !(fabsf(n.c) > 0x1p126f);
    n.th2 = plain ? __fadd_rn(n.th, n.th) : __builtin_nanf("");
    n.thd = plain ? (CAPK == 0 ? n.th2 : __builtin_inff()) : n.th;
    n.lo = p.apply_low ? p.theta_low[row] : -__builtin_inff();
    // a bound that is no number bounds nothing and lets no gradient pass
    n.gate = n.lo != n.lo ? __builtin_inff() : n.lo;
    if (n.lo != n.lo) n.lo = -__builtin_inff();
}

// Advance synapse and membrane by one step, in the order the composed layer does it
// (input scaling, synapse, input normalisation, membrane, clamp):
//   xin = x * xs;  i = i * a_syn + xin   (SYN; otherwise i = x)
//   u = k * i;   v = vpost * a_mem + u;   v = max(v, lo)
// Returns the pre-reset potential v; n.i is advanced, n.vpost is left to the caller (it needs the
// spike count).
template <bool SYN>
__device__ __forceinline__ float neuron_advance(Neuron &n, float x)
{
    if (SYN) {
        const float xin = __fmul_rn(x, n.xs);
        n.i = __fadd_rn(__fmul_rn(n.i, n.as), xin);
    } else {
        n.i = x;
    }
    const float u = __fmul_rn(n.k, n.i);
    const float v = __fadd_rn(__fmul_rn(n.vpost, n.am), u);
    return __builtin_elementwise_maximum(v, n.lo);             // keeps a NaN potential, as v < lo ? lo : v does
}

// count = v >= th ? min(unsigned(v / th), cap) : 0   (IEEE division, truncation), in two parts:
// the count by comparisons, and the quotient for the rare potentials at or above n.thd (with CAPK == 0 that is where two
// spikes begin).
template <int CAPK>
__device__ __forceinline__ float count_by_compare(float v, const Neuron &n, const Cap &cc)
{
    const float count = v >= n.th ? (CAPK == 0 ? cc.one : 1.f) : 0.f;
    return CAPK == 2 && v >= n.th2 ? 2.f : count;
}

__device__ __forceinline__ float count_by_quotient(float v, const Neuron &n, const Cap &cc)
{
    const unsigned q = static_cast<unsigned>(__fdiv_rn(v, n.th));
    return static_cast<float>(q < cc.cap ? q : cc.cap);
}

template <int CAPK>
__device__ __forceinline__ float spike_count_fast(float v, const Neuron &n, const Cap &cc)
{
    float count = count_by_compare<CAPK>(v, n, cc);
    if (v >= n.thd) count = count_by_quotient(v, n, cc);
    return count;
}

// count * c, what the reset subtracts from the potential, for callers that do not need the count itself: with a cap
// of one or two spikes the product is 0, c or 2c (all exact), picked by the comparisons that would have picked the
// count -- the same bits as the multiplication, one instruction less.
template <int CAPK>
__device__ __forceinline__ float reset_amount(float v, const Neuron &n, const Cap &cc)
{
    if (CAPK == 0) return __fmul_rn(spike_count_fast<0>(v, n, cc), n.c);
    float taken = v >= n.th ? n.c : 0.f;
    if (CAPK == 2) taken = v >= n.th2 ? n.c2 : taken;
    if (v >= n.thd) taken = __fmul_rn(count_by_quotient(v, n, cc), n.c);   // thresholds that are not positive
    return taken;
}

__device__ __forceinline__ float decay_factor(float tau) { return expf(-__fdiv_rn(1.0f, tau)); }

// The decay factor of neuron m of batch element b in row `row`; `write`: this lane writes what the call is to leave behind.
// (A launch for it was 2.4 us on the device and 5 on the host, for calls that take 100.  A spiking layer does without it where the
// parameters are those of its last call: a step of an optimizer has them checked again, and the check wants the factors ahead.)
__device__ __forceinline__ float decay_of(const Decay &d, int64_t b, int64_t m, int64_t row, bool write)
{
    const float tau = d.tau[d.one ? 0 : m], alpha = decay_factor(tau);
    if (write) {
        d.alpha[row] = alpha;
        if (b == 0 && (!d.one || m == 0)) d.kept[m] = tau;
    }
    return alpha;
}

// neuron_load has read factors that are not there yet
template <bool SYN>
__device__ __forceinline__ void decays_load(Neuron &n, const LayerConsts &p, int64_t b, int64_t m, int64_t row, bool write)
{
    if (p.mem.tau) {
        n.am = decay_of(p.mem, b, m, row, write);
        n.k = p.norm_input ? __fsub_rn(1.0f, n.am) : 1.0f;
    }
    if (SYN && p.syn.tau) {
        n.as = decay_of(p.syn, b, m, row, write);
        n.xs = p.decay_early ? n.as : 1.0f;
    }
}

__device__ __forceinline__ float saturate(float x) { return fminf(fmaxf(x, 0.f), 1.f); }   // the clamp of the instruction before

// v >= th ? 1 : 0 as saturate(v * scale + shift), for thresholds between 2^-100 and 2^100.  scale is the power of two that
// takes th to [2^24, 2^25), or to 2^25 where th is a power of two itself: the float before th then lies 2 below it, th * scale
// is an even integer and shift = 2 - th * scale a float.  So v == th gives 2, the float before it 0, and the one rounding of
// the fused multiply-add cannot carry any other v to the wrong side (NaN saturates to 0, as the comparison fails for it).
// The threshold of two spikes, 2 th, takes half the scale and the same shift.  Any other neuron gets a line that is always 0
// and is done again from its threshold on (from every potential where 0 * c is no number).
__device__ __forceinline__ void spike_line(float &scale, float &shift, float &redo, const Neuron &n, const Cap &cc)
{
    const bool usable = n.th >= 0x1p-100f && n.th <= 0x1p100f && fabsf(n.c) <= 0x1p126f;
    const int bits = __float_as_int(n.th), exponent = (bits >> 23) - 127;
    const float up = __uint_as_float(static_cast<unsigned>(((bits & 0x7fffff) ? 24 : 25) - exponent + 127) << 23);
    scale = usable ? cc.one * up : 0.f;
    shift = usable ? cc.one * (2.f - n.th * up) : 0.f;
    redo = usable ? n.thd : (fabsf(n.c) < __builtin_inff() ? n.th : -__builtin_inff());
}

// compute units of the current device, asked for once per device
inline int compute_units()
{
    static std::atomic<int> known[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int cus = known[dev].load(std::memory_order_relaxed);
    if (cus > 0) return cus;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    known[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// Neurons per lane of the kernels that support several.  Wider lanes mean wider memory accesses but fewer lanes.
//   two: from `waves_per_cu` waves per compute unit on.  The spiking forward has a long dependent chain per step and wants 16
//        (with 16 / with 8, us: (16, 500, 49152) 588 / 613, (8, 1000, 66560) 861 / 954); the leaky kernels measure best from 8 on.
//   four: only where so many waves are left that memory is all that counts.  Two / four per lane, us, spiking and leaky
//        forward: 1 M neurons (32, 200, 32768) 319 / 333 and 299 / 314, with synapses (16, 1000, 65536) 1606 / 1624;
//        2 M (64, 300, 32768) 927 / 960 and 906 / 962; 4 M (32, 300, 131072) 1906 / 1868 and 1870 / 1870.  Where steps do not
//        fill whole sectors (`whole` false) neighbouring blocks share them, wider blocks share fewer, and four pay sooner:
//        1.1 M (64, 300, 17000) 584 / 602 and 563 / 576, 2 M (32, 400, 65528) 1452 / 1436 and 1416 / 1398.
// Where steps fill whole sectors a wider lane is taken only if its blocks spread over the compute units about as evenly as those
// of one neuron per lane: `even` is the share of lanes that have work while the units that got one block more than the others
// finish it (and that lie inside the layer).  Memory-bound blocks advance at one pace, so the other units stand idle by then.
// One / two, us, spiking and leaky forward, leaky backward: (64, 300, 12544), even 0.94 / 0.88, 375 / 394, 355 / 374 and
// 550 / 566; (40, 250, 11008), 0.96 / 0.84, 176 / 176 (13 waves per unit would be left: forced here), 163 / 174 and 252 / 263;
// where both are even (64, 300, 8192) 227 / 219, 211 / 204 and 322 / 314.  With shared sectors two stay ahead:
// (64, 300, 17000) 631 / 584.
// `align` is the common alignment (bytes) of all (batch, time, neurons) pointers involved.
inline int pick_neurons_per_lane(int64_t batch, int64_t neurons, unsigned align, int widest, int waves_per_cu, bool whole)
{
    const int cus = compute_units();
    const int64_t n = batch * neurons;
#ifdef EXODUS_FORCE_NPL
    if (EXODUS_FORCE_NPL <= widest) widest = EXODUS_FORCE_NPL;
#endif
    const auto even = [&](int npl) {
        const int64_t blocks = batch * ((neurons + BLOCK * npl - 1) / (BLOCK * npl)), rounds = (blocks + cus - 1) / cus;
        return static_cast<double>(n) / (static_cast<double>(rounds) * cus * BLOCK * npl);
    };
    for (int npl = widest; npl > 1; npl /= 2) {
        const int64_t lanes = static_cast<int64_t>(cus) * WAVE * (npl == 2 ? waves_per_cu : (whole ? 64 : 24));
        if (neurons % npl == 0 && align % (4u * npl) == 0 && n / npl >= lanes && (!whole || even(npl) >= even(1) - 0.03))
            return npl;
    }
    return 1;
}

// Lanes per block.  Four waves that keep each other at the same step suit memory (see the barriers); but up to a few waves per
// compute unit they only crowd on a few units, whose way to memory their accesses then share, while the others stand idle: one
// wave per block there, which also leaves no wave without a neuron.  `half_waves`: half waves per compute unit up to which.
inline int lanes_per_block(int64_t batch, int64_t neurons, int half_waves)
{
    return 2 * batch * ((neurons + WAVE - 1) / WAVE) <= half_waves * compute_units() ? WAVE : BLOCK;
}

// Forward and leaky kernels: two waves per compute unit.  256 / 64 lanes, us, spiking (at most one spike) and leaky forward, the
// same tensors again and again: (4, 2000, 512) 96.6 / 70.4 and 80.0 / 55.6, (64, 300, 10) 20.2 / 16.1 and 15.0 / 11.3,
// (24, 250, 1323) with 504 waves 20.9 / 20.2 and 15.7 / 16.7, (32, 250, 2048) with 1024 26.9 / 30.3 and 23.7 / 26.3; other
// tensors in every call, so that they come from memory: (24, 250, 1323) 26.9 / 25.8 and 25.9 / 24.8, (24, 1000, 1323)
// 86.0 / 82.2 and 83.3 / 79.9, (8, 500, 4090) with 512 waves 44.4 / 43.2 and 42.6 / 41.5, (32, 250, 1024) 20.1 / 18.5 and
// 19.3 / 17.3.
constexpr int FORWARD_HALF_WAVES = 4;
// The spiking forward that records both states moves four tensors.  Where its steps do not fill whole sectors (`whole` false) and
// blocks are neighbours in a step, blocks of one wave share more sectors than blocks of four, and only one and a half pay.
// 256 / 64, us, other tensors in every call: 512 waves (8, 500, 4090) 87 / 97, (64, 200, 500) 42.1 / 44.5, 504 (24, 1000, 1323)
// 168 / 189, (24, 250, 1323) 50.2 / 54.6, 500 (250, 200, 100) 38.0 / 40.2, 448 (7, 500, 4090) 85 / 89, 384 (6, 500, 4090)
// 83.2 / 82.2, (24, 300, 1000) 54.7 / 54.3; whole sectors, 512 (32, 250, 1024) 43.5 / 42.6; one wave per element (500, 200, 40)
// 44.1 / 37.1.
inline int forward_half_waves(int64_t neurons, bool both_records, bool whole)
{
    return both_records && !whole && neurons > WAVE ? 3 : FORWARD_HALF_WAVES;
}

// What a launch of a forward or leaky kernel looks like.  `widest` is 1 for a kernel that knows no other width.
struct LaunchShape {
    int npl, lanes;      // neurons per lane, lanes per block
};

inline LaunchShape launch_shape(int64_t batch, int64_t neurons, unsigned align, int widest, int waves_per_cu, bool whole,
                                int half_waves = FORWARD_HALF_WAVES)
{
    const int npl = pick_neurons_per_lane(batch, neurons, align, widest, waves_per_cu, whole);
    return {npl, npl == 1 ? lanes_per_block(batch, neurons, half_waves) : BLOCK};
}

constexpr int FORWARD_WAVES = 16;

// The one-lane backward: one wave per block up to four waves per compute unit.  256 lanes / 64, us, other tensors in every call,
// without and with a synapse: 504 waves (24, 250, 1323) 49.3 / 41.4 and 63.1 / 57.5, 1024 (32, 250, 2048) 54.0 / 46.3 and
// 67.1 / 64.4, (16, 500, 4096) 94.7 / 82.6 and 122 / 115; 2048 (the same tensors) (64, 300, 2048) 95 / 105 and
// (16, 300, 8192) 110 / 118.
// More tensors (gradients on state records, a surrogate tensor: `extra`) leave it at that where steps fill whole sectors: records
// and surrogate tensor, 1024 waves (32, 250, 2048) 62.4 / 60.3 and 61.4 / 59.3, with a synapse 88.9 / 88.3 and 76.7 / 73.8, though
// (16, 1000, 4096) 217 / 231 and 205 / 217.  Where blocks share sectors, three waves per unit: 768 (48, 300, 1000) 70.4 / 65.7 and
// 68.0 / 63.7, (12, 500, 4090) 113.3 / 109.6 and 108.6 / 107.1; 832 (13, 500, 4090) 115 / 119 and 110 / 119; 1024
// (16, 500, 4090) 129 / 144 and 123 / 142, (64, 1000, 1000) 241 / 265 and 238 / 265.  Without more tensors shared sectors leave
// it at four: 1024 (64, 300, 1000) 69.6 / 68.5 and 80.7 / 80.0, 960 (60, 300, 1000) 67.1 / 65.0 and 84.8 / 80.1, though without a
// synapse (16, 500, 4090) 105 / 113.
inline int backward_lanes(int64_t batch, int64_t neurons, bool extra, bool whole)
{
    return lanes_per_block(batch, neurons, extra && !whole ? 6 : 8) == WAVE ? WAVE : BWD_BLOCK;
}

inline unsigned common_alignment(std::initializer_list<const void *> ptrs)
{
    uintptr_t bits = 0;
    for (const void *q : ptrs) bits |= reinterpret_cast<uintptr_t>(q);   // null pointers do not constrain
    return static_cast<unsigned>(bits & 15u) == 0 ? 16u : ((bits & 7u) == 0 ? 8u : 4u);
}

// true when every step's neurons start and end on 64-byte sectors of memory for all the given tensors: then no
// sector is shared between waves and the streamed accesses can be marked non-temporal (with whole 128-byte lines
// and with whole sectors that measures 1-5 % faster than without the mark; with steps that start on 32-byte
// boundaries 10 % slower)
inline bool whole_lines(int64_t neurons, std::initializer_list<const void *> ptrs)
{
    uintptr_t bits = 0;
    for (const void *q : ptrs) bits |= reinterpret_cast<uintptr_t>(q);
    return (neurons % EXODUS_WHOLE_NEURONS) == 0 && (bits & (4u * EXODUS_WHOLE_NEURONS - 1u)) == 0;
}

// Blocks that are neighbours in a step, on one XCD.  The machine deals the blocks of a grid out to its eight XCDs one by one, each
// with an L2 of its own: the line that two neighbouring blocks share is then fetched twice and written in two parts.  Where steps
// do not fill whole lines of 128 bytes, runs of NEIGHBOURS blocks go to one XCD instead.  Before / after, us, forward and backward,
// other tensors in every call, spiking and leaky: (64, 300, 17000) 574 + 904 / 562 + 852 and 570 + 827 / 552 + 801, (64, 300, 4999)
// 198 + 280 / 182 + 266 and 191 + 264 / 174 + 245, (32, 400, 65533) 1616 + 2175 / 1491 + 2103 and 1489 + 2165 / 1409 + 2015,
// (8, 500, 4090) 34.4 + 67.7 / 32.5 + 65.2 and 34.3 + 53.0 / 29.0 + 51.7, (24, 250, 1323) 22.3 + 39.8 / 20.7 + 37.3 and
// 20.4 + 28.9 / 18.0 + 27.8; half lines shared, (64, 300, 4976) 165 + 258 / 163 + 254 and 160 + 237 / 157 + 232.  Runs of 8 and 16
// are level or up to 2 % behind, of 64 up to 5 %.  Whole lines stay as they are dealt: nothing is shared, and the XCDs then walk
// addresses further apart, (32, 300, 131072) 1879 + 2801 / 2023 + 2806, (64, 300, 12544) 370 + 558 / 369 + 559.
constexpr int NEIGHBOURS = 32, XCDS = 8;
inline unsigned neighbours_per_xcd(int64_t blocks, int64_t neurons, std::initializer_list<const void *> ptrs)
{
    uintptr_t bits = static_cast<uintptr_t>(neurons) * 4u;
    for (const void *q : ptrs) bits |= reinterpret_cast<uintptr_t>(q);
    if (bits % 128u == 0) return 1;
    const int64_t share = blocks / XCDS;                        // a small grid is one run for each XCD
    return share >= 2 * NEIGHBOURS ? NEIGHBOURS : (share > 1 ? static_cast<unsigned>(share) : 1u);
}

// The block of the layer that block blockIdx.x works on: XCDS runs of `run` blocks trade places so that each lies on one XCD; what
// is left at the end of the grid stays where it is (a permutation of the grid's blocks, the identity for run == 1).
__device__ __forceinline__ unsigned layer_block(unsigned run)
{
    const unsigned many = XCDS * run, start = blockIdx.x / many * many, at = blockIdx.x - start;
    return gridDim.x - start < many ? blockIdx.x : start + at % XCDS * run + at / XCDS;
}

constexpr int SPLIT_LANES = 512;
constexpr int SPLIT_CHUNKS = 32;           // most chunks of a group
constexpr int SPLIT_NEURONS = 64;          // most neurons of a block

// How the kernels that give every chunk of CKPT steps a lane of its own spread a layer: chunks of a group and neurons of a block.
struct SplitShape {
    int64_t blocks_per_batch;
    int neurons_log, lanes;
};

inline SplitShape split_shape(int64_t B, int64_t T, int64_t M)
{
    const int64_t n_ck = (T + CKPT - 1) / CKPT;
    // 256 registers per lane leave a compute unit eight waves, one block of more than four.  A launch of more such blocks than
    // there are compute units takes another round of them, so it takes smaller groups of chunks instead: 16 chunks of 32
    // neurons in the place of 32 of 16, and where that is too many blocks 8 of 32, two blocks to a compute unit.  Without /
    // with, us: 16 384 neurons 300 steps 26.8 / 21.9, 512 steps 31.0 / 25.4, with synapses 37.7 / 29.6, 2000 steps 171 / 107,
    // with state records 309 / 203, with a surrogate tensor 188 / 130; 10 240 neurons 300 steps 22.2 / 18.8; 8192 neurons
    // 1000 steps 41 / 30.  Where one round does, smaller groups only lengthen the chain: 8192 neurons 300 steps 12.5 / 15.8,
    // 4096 neurons 1000 steps with synapses 25.6 / 28.2.  (Up to 8 chunks of 64 neurons are one round for 16 384 neurons.)
    const auto blocks = [&](int log) { return ((M + (int64_t{1} << log) - 1) >> log) * B; };
    const int64_t cus = compute_units();
    int most = SPLIT_CHUNKS, widest = 6;
    if (n_ck > 16 && blocks(4) > cus) most = 16;
    if (n_ck > 8 && blocks(5) > cus) {
        most = 8;
        widest = 5;
    }
    const int64_t groups = (n_ck + most - 1) / most;
    const int chunks = static_cast<int>((n_ck + groups - 1) / groups);
    // as many neurons per block as its lanes hold, but no more than the layer has
    int neurons_log = 4;
    while (neurons_log < widest && (chunks << (neurons_log + 1)) <= SPLIT_LANES && (int64_t{1} << neurons_log) < M)
        ++neurons_log;
    const int64_t blocks_per_batch = (M + (int64_t{1} << neurons_log) - 1) >> neurons_log;
    const int lanes = ((chunks << neurons_log) + WAVE - 1) / WAVE * WAVE;
    return {blocks_per_batch, neurons_log, lanes};
}

inline bool bad3(int64_t b, int64_t t, int64_t m)
{
    if (b < 0 || t < 0 || m < 0) return true;
    if (b == 0 || t == 0 || m == 0) return false;
    if (b > INT64_MAX / t) return true;
    return (b * t) > INT64_MAX / m;
}

// step offsets inside a block of CKPT steps are 32-bit byte offsets
inline bool too_wide(int64_t neurons) { return neurons >= (int64_t{1} << 25); }

}  // namespace

// the forward pass again, keeping nothing but the checkpoints (exodus_layer.hip)
int exodus_layer_checkpoints_only(float *ckpt_v, float *ckpt_i, const float *x, const LayerConsts &p, bool syn, int64_t B,
                                  int64_t T, int64_t M, hipStream_t s);

// the forward pass with three or four waves for 64 neurons (exodus_layer_forward_roles.hip)
bool exodus_layer_forward_roles_apply(int64_t B, int64_t T, int64_t M);
int exodus_layer_forward_roles(float *spikes, float *ckpt_v, float *ckpt_i, float *v_last, float *i_last, const Sums &sums,
                               const float *x, const LayerConsts &p, int64_t B, int64_t T, int64_t M, hipStream_t s);

// the backward pass with one lane per neuron and chunk of CKPT steps (exodus_layer_backward_split.hip)
struct SplitArgs {
    float *grad_x, *alpha_mem_grad, *alpha_syn_grad, *v_init_grad, *i_init_grad;
    const float *grad_spikes, *grad_v_last, *grad_i_last, *x, *surr, *grad_v_rec, *grad_i_rec, *ckpt_v, *ckpt_i;
    LayerConsts p;
    float p0, p1, inv_p0;
    int64_t T, M;
};
// the backward pass of the leaky layer with one lane per neuron and chunk (exodus_layer_leaky_split.hip)
struct LeakySplitArgs {
    float *grad_x, *alpha_grad, *v_init_grad;
    const float *grad_out, *grad_v_last, *out, *x, *v_init, *alpha;
    int decay_early, norm_input;
    int64_t T, M;
};
bool exodus_layer_leaky_split_applies(int64_t B, int64_t T, int64_t M);
int exodus_layer_split_mode();             // what exodus_layer_backward_time_split has set
int exodus_layer_leaky_split(const LeakySplitArgs &a, bool uniform, int64_t B, hipStream_t s);

// the kernels keep the offsets of 32 chunks below 2^31 bytes
inline bool exodus_layer_split_applies(int64_t neurons) { return neurons < (int64_t{1} << 19); }
int exodus_layer_backward_split(const SplitArgs &a, bool syn, int kind, bool uniform, int64_t B, hipStream_t s);
