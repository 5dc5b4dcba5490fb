"""ctypes loader for ``libexodus_hip.so`` and thin tensor-level wrappers around its C ABI.

This module plays the role of the reference's ``exodus_cuda`` pybind module
(reference cuda/bindings.cu:362-373): same six functions, same argument order, plus the two
fused backward entry points.  Tensors must live on a HIP device, be ``float32`` and contiguous;
anything else raises, as the reference's ``CHECK_INPUT`` asserts do
(reference cuda/bindings.cu:7-10).  There is no CPU path: if the shared library is missing the
import of this module fails with an ``ImportError`` that says how to build it.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys
from typing import Optional

import torch  # must be imported before the library so both share one HIP runtime

from . import hbm

_HERE = os.path.dirname(os.path.abspath(__file__))
# EXODUS_HIP_LIBRARY may point at another build of the same ABI (e.g. one compiled with other flags)
LIB_PATH = os.environ.get("EXODUS_HIP_LIBRARY") or os.path.join(_HERE, "libexodus_hip.so")

SURR_TENSOR, SURR_SINGLE_EXP, SURR_PERIODIC_EXP, SURR_HEAVISIDE = 0, 1, 2, 3
ABI_VERSION = 8

_p = ctypes.c_void_p
_i64 = ctypes.c_int64
_int = ctypes.c_int
_f = ctypes.c_float

_SIGNATURES = {
    "exodus_hip_abi_version": ([], _int),
    "exodus_hip_error_string": ([_int], ctypes.c_char_p),
    "exodus_check_parameters": ([_p] * 5 + [_i64, _p], _int),
    "exodus_lif_forward": ([_p] * 8 + [_int, _int, _i64, _i64, _p], _int),
    "exodus_lif_backward": ([_p] * 6 + [_i64, _i64, _p], _int),
    "exodus_lif_backward_alpha": ([_p] * 8 + [_int, _i64, _i64, _p], _int),
    "exodus_leaky_forward": ([_p] * 4 + [_i64, _i64, _p], _int),
    "exodus_leaky_backward": ([_p] * 3 + [_i64, _i64, _p], _int),
    "exodus_leaky_backward_alpha": ([_p] * 5 + [_i64, _i64, _p], _int),
    "exodus_leaky_backward_fused": ([_p] * 7 + [_i64, _i64, _p], _int),
    "exodus_lif_backward_fused": ([_p] * 12 + [_int, _int, _int, _f, _f, _i64, _i64, _p], _int),
    "exodus_synlif_forward": ([_p] * 11 + [_int, _int, _int, _int, _i64, _i64, _p], _int),
    "exodus_synlif_backward": ([_p] * 17 + [_int, _int, _int, _int, _int, _f, _f, _i64, _i64, _p], _int),
    "exodus_spike_forward": ([_p, _p, _f, _f, _f, _f, _int, _int, _i64, _i64, _p], _int),
    "exodus_spike_backward": ([_p] * 4 + [_f, _f, _i64, _i64, _p], _int),
    "exodus_layer_checkpoint_interval": ([], _int),
    "exodus_layer_sum_slots": ([_i64, _i64], _i64),
    "exodus_layer_lif_forward": ([_p] * 16 + [_int, _int, _int, _int, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_lif_forward_total": ([_p] * 17 + [_int, _int, _int, _int, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_lif_forward_decays": ([_p] * 18 + [_int, _int, _int, _int, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_lif_backward": ([_p] * 18 + [_int, _int, _int, _int, _int, _f, _f, _p, _p, _p, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_backward_time_split": ([_int], _int),
    "exodus_layer_scratch_floats": ([], _i64),
    "exodus_layer_lif_backward_from_input": ([_p] * 16 + [_int, _int, _int, _int, _int, _f, _f, _p, _p, _p, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_leaky_forward": ([_p] * 6 + [_int, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_leaky_forward_total": ([_p] * 7 + [_int, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_leaky_forward_decays": ([_p] * 8 + [_int, _int, _i64, _i64, _i64, _p], _int),
    "exodus_layer_leaky_backward": ([_p] * 9 + [_int, _int, _int, _i64, _i64, _i64, _p], _int),
    "exodus_decay_expand": ([_p, _p, _p, _i64, _i64, _i64, _p], _int),
    "exodus_layer_launch_shape": ([_int, _i64, _i64, _p, _p], _int),
    "exodus_decay_work": ([_i64] * 3, _i64),
    "exodus_decay_grad": ([_p] * 4 + [_i64, _i64, _i64, _p], _int),
    "exodus_hbm_regions_create": ([_int, ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint64, _int, ctypes.c_uint64, _p], _int),
    "exodus_hbm_regions_destroy": ([_int], _int),
    "exodus_hbm_alloc_striped": ([ctypes.c_size_t, _int, _p], _p),
    "exodus_hbm_alloc_region0": ([ctypes.c_size_t, _int, _p], _p),
    "exodus_hbm_alloc_region1": ([ctypes.c_size_t, _int, _p], _p),
    "exodus_hbm_alloc_region2": ([ctypes.c_size_t, _int, _p], _p),
    "exodus_hbm_free": ([_p, ctypes.c_size_t, _int, _p], None),
    "exodus_hbm_usage": ([_int, _p, _p], _int),
}


def _load() -> ctypes.CDLL:
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            f"{LIB_PATH} not found. Build it with `python build_hip.py` in the package root "
            "(needs hipcc; cross-compiles for gfx950 without a GPU). There is no CPU fallback."
        )
    lib = ctypes.CDLL(LIB_PATH)
    missing = [name for name in _SIGNATURES if not hasattr(lib, name)]     # a library of the same version may be older
    if missing:
        raise ImportError(f"{LIB_PATH} is not a library of this package or an older one: it lacks {', '.join(missing)}")
    for name, (argtypes, restype) in _SIGNATURES.items():
        fn = getattr(lib, name)
        fn.argtypes = argtypes
        fn.restype = restype
    got = lib.exodus_hip_abi_version()
    if got != ABI_VERSION:
        raise ImportError(f"{LIB_PATH} has ABI version {got}, this package expects {ABI_VERSION}")
    return lib


lib = _load()


class ExodusHipError(RuntimeError):
    pass


def _check(status: int, what: str) -> None:
    if status != 0:
        msg = lib.exodus_hip_error_string(status)
        raise ExodusHipError(f"{what} failed: {msg.decode() if msg else status} (status {status})")


def _dev(x: torch.Tensor, name: str, like: Optional[torch.Tensor] = None) -> torch.Tensor:
    if not isinstance(x, torch.Tensor):
        raise TypeError(f"{name} must be a tensor")
    if not x.is_cuda:
        raise RuntimeError(f"{name} must be a tensor on a HIP device (got {x.device}); there is no CPU path")
    if x.dtype != torch.float32:
        raise RuntimeError(f"{name} must be float32 (got {x.dtype})")
    if not x.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")
    if like is not None and x.device != like.device:
        raise RuntimeError(f"{name} and the first tensor must be on the same device")
    return x


def _native_module():
    """The host side of the calls in native code, given this library's entry points."""
    running = f"torch {torch.__version__}, Python {sys.version_info[0]}.{sys.version_info[1]};"
    try:
        from . import _exodus_torch as native
        if native.built_for != running:        # torch's C++ interfaces change with its version
            raise ImportError(f"it was built for {native.built_for} this is {running}")
    except ImportError as err:
        raise ImportError(f"{os.path.join(_HERE, '_exodus_torch.so')} cannot be loaded ({err}). Build it with "
                          "`python build_hip.py` in the package root.") from err
    native.bind({name: ctypes.cast(getattr(lib, name), _p).value for name in _SIGNATURES}, _check, _place)
    return native


def _rows(x: torch.Tensor, name: str, n: int) -> torch.Tensor:
    if x.ndim != 1 or x.shape[0] != n:
        raise RuntimeError(f"{name} must have shape ({n},), got {tuple(x.shape)}")
    return x


def _mat(x: torch.Tensor, name: str, n: int, t: int) -> torch.Tensor:
    if x.ndim != 2 or x.shape[0] != n or x.shape[1] != t:
        raise RuntimeError(f"{name} must have shape ({n}, {t}), got {tuple(x.shape)}")
    return x


def _cap(spikes: int) -> int:
    """Most spikes per step as the C ABI takes it: an int whose bits are an unsigned number, -1 = no limit.  No count reaches a
    limit beyond 32 bits."""
    spikes = int(spikes)
    if spikes < 1 << 31:
        return spikes
    return spikes - (1 << 32) if spikes < 1 << 32 else -1


def _ptr(x: Optional[torch.Tensor]):
    return None if x is None else x.data_ptr()             # ctypes takes a plain integer for a void pointer


def _stream(x: torch.Tensor):
    return torch.cuda.current_stream(x.device).cuda_stream or None


class _NoGuard:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_GUARD = _NoGuard()


def _on_device_of(device: torch.device):
    """Device guard for a launch: ``device`` becomes current for the call -- which it nearly always is already, and
    then nothing needs switching."""
    return _NO_GUARD if torch.cuda.current_device() == device.index else torch.cuda.device(device)


def _place(like: torch.Tensor, shape: Optional[tuple] = None):
    """What allocates a call's results of up to the size of ``like`` (or of ``shape``): ``hbm.empty`` after ``hbm.enable()``
    (memory striped over the regions of HBM), None for the ordinary allocator."""
    if not isinstance(like, torch.Tensor):
        return None                            # refused by the call
    return hbm.empty if hbm.places(like.numel() if shape is None else math.prod(shape), like) else None


_native = _native_module()


def checkParameters(flags, alpha, alphaOther, theta, thetaLow) -> None:
    """Sets flags[0] where a decay factor lies outside [0, 1] and flags[1] where a threshold does not exceed its lower bound;
    the vectors (or None) have one length.  ``flags`` is a pinned int32 host tensor: read it once the stream has got here."""
    first = alpha if alpha is not None else thetaLow
    with _on_device_of(first.device):
        _check(lib.exodus_check_parameters(_ptr(flags), _ptr(alpha), _ptr(alphaOther), _ptr(theta), _ptr(thetaLow),
                                           first.numel(), _stream(first)), "exodus_check_parameters")


# ------------------------------------------------------------------------------------------
# the six functions of the reference extension, same names and argument order
# (an argument that a call does not use is not looked at, here and below: the native calls take tensors or None)
# ------------------------------------------------------------------------------------------

def lifForward(outputSpikes, vmem, input, vmemPostInitial, alpha, membrSubtract, theta, thetaLow,
               applyThetaLow: bool, maxNumSpikes: int) -> None:
    """reference cuda/bindings.cu:14-70; fills the caller-allocated ``outputSpikes`` and ``vmem``."""
    _native.lif_forward(outputSpikes, vmem, input, vmemPostInitial, alpha, membrSubtract, theta,
                        thetaLow if applyThetaLow else None, bool(applyThetaLow), _cap(maxNumSpikes))


def lifBackward(surr, outputGrad, notClipped, alpha, membrSubtract) -> torch.Tensor:
    """reference cuda/bindings.cu:72-110; ``membrSubtract`` is alpha times the subtract value."""
    _dev(surr, "surr")
    if surr.ndim != 2:
        raise RuntimeError("surr must be 2-D (rows, time)")
    n, t = surr.shape
    _mat(_dev(outputGrad, "outputGrad", surr), "outputGrad", n, t)
    _mat(_dev(notClipped, "notClipped", surr), "notClipped", n, t)
    _rows(_dev(alpha, "alpha", surr), "alpha", n)
    _rows(_dev(membrSubtract, "membrSubtract", surr), "membrSubtract", n)
    inputGrad = hbm.empty_like(surr)
    with _on_device_of(surr.device):
        _check(lib.exodus_lif_backward(_ptr(inputGrad), _ptr(surr), _ptr(outputGrad), _ptr(notClipped),
                                       _ptr(alpha), _ptr(membrSubtract), n, t, _stream(surr)),
               "exodus_lif_backward")
    return inputGrad


def lifBackwardAlpha(surr, outputGrad, vmemPost, vmemPostInitial, notClipped, alpha, membrSubtract,
                     gateInitial: bool = False) -> torch.Tensor:
    """reference cuda/bindings.cu:112-158.  ``gateInitial=False`` is the reference's arithmetic."""
    _dev(surr, "surr")
    if surr.ndim != 2:
        raise RuntimeError("surr must be 2-D (rows, time)")
    n, t = surr.shape
    for nm, x in (("outputGrad", outputGrad), ("vmemPost", vmemPost), ("notClipped", notClipped)):
        _mat(_dev(x, nm, surr), nm, n, t)
    for nm, x in (("vmemPostInitial", vmemPostInitial), ("alpha", alpha), ("membrSubtract", membrSubtract)):
        _rows(_dev(x, nm, surr), nm, n)
    alphaGrad = torch.zeros_like(alpha)
    with _on_device_of(surr.device):
        _check(lib.exodus_lif_backward_alpha(_ptr(alphaGrad), _ptr(surr), _ptr(outputGrad), _ptr(vmemPost),
                                             _ptr(vmemPostInitial), _ptr(notClipped), _ptr(alpha),
                                             _ptr(membrSubtract), int(bool(gateInitial)), n, t, _stream(surr)),
               "exodus_lif_backward_alpha")
    return alphaGrad


def leakyForward(input, vmemInitial, alpha, *, output=None) -> torch.Tensor:
    """reference cuda/bindings.cu:163-193.  ``output`` (not in the reference) is a preallocated result."""
    return _native.leaky_forward(input, vmemInitial, alpha, output, _place(input))


def leakyBackward(outputGrad, alpha) -> torch.Tensor:
    """reference cuda/bindings.cu:195-221."""
    _dev(outputGrad, "outputGrad")
    if outputGrad.ndim != 2:
        raise RuntimeError("outputGrad must be 2-D (rows, time)")
    n, t = outputGrad.shape
    _rows(_dev(alpha, "alpha", outputGrad), "alpha", n)
    inputGrad = hbm.empty_like(outputGrad)
    with _on_device_of(outputGrad.device):
        _check(lib.exodus_leaky_backward(_ptr(inputGrad), _ptr(outputGrad), _ptr(alpha), n, t,
                                         _stream(outputGrad)), "exodus_leaky_backward")
    return inputGrad


def leakyBackwardAlpha(outputGrad, output, vmemInitial, alpha) -> torch.Tensor:
    """reference cuda/bindings.cu:223-257."""
    _dev(outputGrad, "outputGrad")
    if outputGrad.ndim != 2:
        raise RuntimeError("outputGrad must be 2-D (rows, time)")
    n, t = outputGrad.shape
    _mat(_dev(output, "output", outputGrad), "output", n, t)
    _rows(_dev(vmemInitial, "vmemInitial", outputGrad), "vmemInitial", n)
    _rows(_dev(alpha, "alpha", outputGrad), "alpha", n)
    alphaGrad = torch.zeros_like(alpha)
    with _on_device_of(outputGrad.device):
        _check(lib.exodus_leaky_backward_alpha(_ptr(alphaGrad), _ptr(outputGrad), _ptr(output),
                                               _ptr(vmemInitial), _ptr(alpha), n, t, _stream(outputGrad)),
               "exodus_leaky_backward_alpha")
    return alphaGrad


def spikeForward(vmem, alpha: float, membrSubtract: float, theta: float, thetaLow: float, applyThetaLow: bool,
                 maxNumSpikes: int) -> torch.Tensor:
    """reference cuda/bindings.cu:262-290 (experimental): ``vmem`` (rows, time) is corrected in place
    for resets and lower bound, the spike raster is returned."""
    _dev(vmem, "vmem")
    if vmem.ndim != 2:
        raise RuntimeError("vmem must be 2-D (rows, time)")
    n, t = vmem.shape
    spikes = hbm.empty_like(vmem)
    with _on_device_of(vmem.device):
        _check(lib.exodus_spike_forward(_ptr(spikes), _ptr(vmem), float(alpha), float(membrSubtract), float(theta),
                                        float(thetaLow), int(bool(applyThetaLow)), _cap(maxNumSpikes), n, t,
                                        _stream(vmem)), "exodus_spike_forward")
    return spikes


def spikeBackward(surr, outputGrad, notClipped, alpha: float, membrSubtract: float) -> torch.Tensor:
    """reference cuda/bindings.cu:327-359 (experimental)."""
    _dev(surr, "surr")
    if surr.ndim != 2:
        raise RuntimeError("surr must be 2-D (rows, time)")
    n, t = surr.shape
    _mat(_dev(outputGrad, "outputGrad", surr), "outputGrad", n, t)
    _mat(_dev(notClipped, "notClipped", surr), "notClipped", n, t)
    inputGrad = hbm.empty_like(surr)
    with _on_device_of(surr.device):
        _check(lib.exodus_spike_backward(_ptr(inputGrad), _ptr(surr), _ptr(outputGrad), _ptr(notClipped),
                                         float(alpha), float(membrSubtract), n, t, _stream(surr)),
               "exodus_spike_backward")
    return inputGrad


# ------------------------------------------------------------------------------------------
# fused backward passes (what the autograd Functions use)
# ------------------------------------------------------------------------------------------

def leakyBackwardFused(outputGrad, alpha, output=None, vmemInitial=None, needAlphaGrad: bool = False,
                       inputGrad: Optional[torch.Tensor] = None):
    """One reverse pass: returns (inputGrad, alphaGrad | None, initGrad)."""
    if not needAlphaGrad:
        output = vmemInitial = None
    return _native.leaky_backward_fused(outputGrad, alpha, output, vmemInitial, bool(needAlphaGrad), inputGrad,
                                        _place(outputGrad))


def lifBackwardFused(gradSpikes, gradVmem, vmem, vmemPostInitial, alpha, membrSubtract, theta, thetaLow,
                     applyThetaLow: bool, maxNumSpikes: int, surrogateKind: int, surrP0: float = 0.0,
                     surrP1: float = 0.0, surr: Optional[torch.Tensor] = None, needAlphaGrad: bool = False,
                     inputGrad: Optional[torch.Tensor] = None):
    """One reverse pass over the saved membrane potential: returns (inputGrad, alphaGrad | None, initGrad).

    ``membrSubtract`` is the plain subtract value here (not pre-multiplied by alpha).
    """
    return _native.lif_backward_fused(gradSpikes, gradVmem, vmem, vmemPostInitial if needAlphaGrad else None, alpha,
                                      membrSubtract, theta, thetaLow if applyThetaLow else None, bool(applyThetaLow),
                                      _cap(maxNumSpikes), int(surrogateKind), float(surrP0), float(surrP1),
                                      surr if surrogateKind == SURR_TENSOR else None, bool(needAlphaGrad), inputGrad, _place(vmem))


def synLifForward(input, vmemPostInitial, isynInitial, alphaMem, alphaSyn, membrSubtract, theta, thetaLow,
                  applyThetaLow: bool, maxNumSpikes: int, decayEarly: bool, normInput: bool,
                  out: Optional[tuple] = None):
    """Fused synapse + membrane forward: returns (spikes, vmem, isyn), all (n, t)."""
    _dev(input, "input")
    if input.ndim != 2:
        raise RuntimeError("input must be 2-D (rows, time)")
    n, t = input.shape
    for nm, x in (("vmemPostInitial", vmemPostInitial), ("isynInitial", isynInitial), ("alphaMem", alphaMem),
                  ("alphaSyn", alphaSyn), ("membrSubtract", membrSubtract), ("theta", theta)):
        _rows(_dev(x, nm, input), nm, n)
    if applyThetaLow:
        _rows(_dev(thetaLow, "thetaLow", input), "thetaLow", n)
    else:
        thetaLow = None
    if out is None:
        out = (hbm.empty_like(input), hbm.empty_like(input), hbm.empty_like(input))
    spikes, vmem, isyn = out
    for nm, x in (("spikes", spikes), ("vmem", vmem), ("isyn", isyn)):
        _mat(_dev(x, nm, input), nm, n, t)
    with _on_device_of(input.device):
        _check(lib.exodus_synlif_forward(_ptr(spikes), _ptr(vmem), _ptr(isyn), _ptr(input), _ptr(vmemPostInitial),
                                         _ptr(isynInitial), _ptr(alphaMem), _ptr(alphaSyn), _ptr(membrSubtract),
                                         _ptr(theta), _ptr(thetaLow), int(bool(applyThetaLow)), _cap(maxNumSpikes),
                                         int(bool(decayEarly)), int(bool(normInput)), n, t, _stream(input)),
               "exodus_synlif_forward")
    return spikes, vmem, isyn


def synLifBackward(gradSpikes, gradVmem, gradIsyn, vmem, isyn, vmemPostInitial, isynInitial, alphaMem, alphaSyn,
                   membrSubtract, theta, thetaLow, applyThetaLow: bool, maxNumSpikes: int, decayEarly: bool,
                   normInput: bool, surrogateKind: int, surrP0: float, surrP1: float,
                   inputGrad: Optional[torch.Tensor] = None):
    """Fused reverse pass: returns (inputGrad, alphaMemGrad, alphaSynGrad, vmemInitGrad, isynInitGrad)."""
    _dev(vmem, "vmem")
    if vmem.ndim != 2:
        raise RuntimeError("vmem must be 2-D (rows, time)")
    n, t = vmem.shape
    _mat(_dev(gradSpikes, "gradSpikes", vmem), "gradSpikes", n, t)
    _mat(_dev(isyn, "isyn", vmem), "isyn", n, t)
    if (gradVmem is None) != (gradIsyn is None):
        raise RuntimeError("gradVmem and gradIsyn must be given together")
    if gradVmem is not None:
        _mat(_dev(gradVmem, "gradVmem", vmem), "gradVmem", n, t)
        _mat(_dev(gradIsyn, "gradIsyn", vmem), "gradIsyn", n, t)
    for nm, x in (("vmemPostInitial", vmemPostInitial), ("isynInitial", isynInitial), ("alphaMem", alphaMem),
                  ("alphaSyn", alphaSyn), ("membrSubtract", membrSubtract), ("theta", theta)):
        _rows(_dev(x, nm, vmem), nm, n)
    if applyThetaLow:
        _rows(_dev(thetaLow, "thetaLow", vmem), "thetaLow", n)
    else:
        thetaLow = None
    if inputGrad is None:
        inputGrad = hbm.empty_like(vmem)
    else:
        _mat(_dev(inputGrad, "inputGrad", vmem), "inputGrad", n, t)
    per_row = [torch.zeros_like(alphaMem) for _ in range(4)]
    with _on_device_of(vmem.device):
        _check(lib.exodus_synlif_backward(_ptr(inputGrad), *[_ptr(x) for x in per_row], _ptr(gradSpikes),
                                          _ptr(gradVmem), _ptr(gradIsyn), _ptr(vmem), _ptr(isyn),
                                          _ptr(vmemPostInitial), _ptr(isynInitial), _ptr(alphaMem), _ptr(alphaSyn),
                                          _ptr(membrSubtract), _ptr(theta), _ptr(thetaLow),
                                          int(bool(applyThetaLow)), _cap(maxNumSpikes), int(bool(decayEarly)),
                                          int(bool(normInput)), int(surrogateKind), float(surrP0), float(surrP1),
                                          n, t, _stream(vmem)), "exodus_synlif_backward")
    return (inputGrad, *per_row)


# ------------------------------------------------------------------------------------------
# layer-layout kernels: (batch, time, neurons) tensors, no transposition
# ------------------------------------------------------------------------------------------

# neurons per batch element the layer-layout entry points accept (they return invalid-value beyond)
LAYER_MAX_NEURONS = 1 << 25


_CHECKPOINT_INTERVAL = int(lib.exodus_layer_checkpoint_interval())


_LAYER_LIF_OUTPUTS = ("spikes", "v_last", "i_last", "ckpt_v", "ckpt_i", "v_rec", "i_rec", "spike_sum")


def checkpointInterval() -> int:
    return _CHECKPOINT_INTERVAL


def layerLifForward(input, vmemPostInitial, isynInitial, alphaMem, alphaSyn, membrSubtract, theta, thetaLow,
                    applyThetaLow: bool, maxNumSpikes: int, decayEarly: bool, normInput: bool,
                    wantCheckpoints: bool = True, wantRecords: bool = False, wantSpikeSum: bool = True,
                    outSpikes: Optional[torch.Tensor] = None, stateShape: Optional[tuple] = None,
                    wantPreReset: bool = False):
    """Returns dict(spikes, v_last, i_last, ckpt_v, ckpt_i, v_rec, i_rec, spike_sum); absent items are None.
    ``stateShape`` (product = batch*neurons) gives v_last / i_last that shape instead of a flat vector.
    ``wantRecords`` records potential (after the reset) and synaptic current of every step;
    ``wantPreReset`` records only the potential, before the reset (the surrogate function's argument)."""
    return dict(zip(_LAYER_LIF_OUTPUTS, _native.layer_lif_forward(
        input, vmemPostInitial, None if alphaSyn is None else isynInitial, alphaMem, alphaSyn, membrSubtract, theta,
        thetaLow if applyThetaLow else None, bool(applyThetaLow),
        _cap(maxNumSpikes), bool(decayEarly), bool(normInput), bool(wantCheckpoints), bool(wantRecords), bool(wantPreReset),
        bool(wantSpikeSum), outSpikes, stateShape, _place(input))))


def layerLif(input, alphaMem, alphaSyn, vmemPostInitial, isynInitial, tauMem, tauSyn, keptMem, keptSyn, theta, membrSubtract,
             thetaLow, surrogateKind: int, surrP0: float, surrP1: float, maxNumSpikes: int, decayEarly: bool, normInput: bool,
             records: bool, stateShape):
    """The pass of ``layerLifForward`` as a node of the autograd graph, for the surrogates that the kernels evaluate:
    (spikes, v_last, spike_sum, i_last | None, v_rec | None, i_rec | None).  ``input`` and the initial states may have any
    contiguous shape (``input`` (batch, time, ...)); spikes and records come in that of ``input``.  ``tauMem`` / ``tauSyn`` are
    time constants to be trained in the place of the decay factors; ``alphaMem`` / ``alphaSyn`` and ``keptMem`` / ``keptSyn`` are
    then what ``decayExpand`` made of them, or None: the forward kernel does it."""
    return _native.layer_lif(input, alphaMem, alphaSyn, vmemPostInitial, isynInitial, tauMem, tauSyn, keptMem, keptSyn, theta,
                             membrSubtract, thetaLow, surrogateKind, surrP0, surrP1, _cap(maxNumSpikes), bool(decayEarly),
                             bool(normInput), bool(records), stateShape, _place(input))[:6]


def layerLeaky(input, alpha, vmemInitial, tau, decayEarly: bool, normInput: bool, stateShape):
    """The pass of ``layerLeakyForward`` as a node of the autograd graph, (out, v_last, out_sum); shapes as for ``layerLif``,
    ``tau`` a time constant to be trained in the place of ``alpha`` (then None)."""
    return _native.layer_leaky(input, alpha, vmemInitial, tau, bool(decayEarly), bool(normInput), stateShape, _place(input))


# stamps(kept, values): a tuple with one entry per value, the entries of ``kept`` (an earlier result, or None) where a value is
# unchanged since, and ``kept`` itself where all are
stamps = _native.stamps


_SHAPES = ("forward", "forward records", "leaky forward", "leaky backward", "leaky backward alpha", "backward",
           "backward more")


def launchShape(kernel: str, batch: int, neurons: int) -> tuple:
    """(neurons per lane, lanes per block) of a layer kernel's launch: which of its variants a layer of this size gets."""
    npl, lanes = _int(), _int()
    _check(lib.exodus_layer_launch_shape(_SHAPES.index(kernel), batch, neurons, ctypes.byref(npl), ctypes.byref(lanes)),
           "exodus_layer_launch_shape")
    return npl.value, lanes.value


def decayExpand(tau, batch: int, neurons: int):
    """exp(-1 / tau) for every neuron of every batch element, (batch*neurons,), and a copy of ``tau`` for ``decayGrad``
    (the caller's may change until then); ``tau`` holds one value or ``neurons``."""
    return _native.decay_expand(tau, batch, neurons)


def decayGrad(gradAlpha, tau, batch: int, neurons: int):
    """Gradient of ``tau``, in its shape, from that of ``decayExpand(tau, batch, neurons)``."""
    return _native.decay_grad(gradAlpha, tau, batch, neurons)


def backwardTimeSplit(mode: int = -1) -> int:
    """How ``layerLifBackward`` and ``layerLeakyBackward`` treat layers with few neurons and many steps
    (``exodus_layer_backward_time_split``): 0 never splits the sequence over lanes, 1 (default) does for layers of up to 16 384
    neurons, 2 for spiking layers of any size without synapse, with an in-kernel surrogate, at most 512 steps and no gradients
    on state records (leaky ones as 1), 3 whenever the kernels apply; -1 only asks.  Returns the mode that was set before."""
    return int(lib.exodus_layer_backward_time_split(int(mode)))


def scratchFloats() -> int:
    """Floats of checkpoint memory the library holds per GPU for ``layerLifBackward(..., ckptV=None)``."""
    return int(lib.exodus_layer_scratch_floats())


def layerLifBackward(gradSpikes, gradVLast, gradILast, input, ckptV, ckptI, vmemPostInitial, isynInitial, alphaMem,
                     alphaSyn, membrSubtract, theta, thetaLow, applyThetaLow: bool, maxNumSpikes: int,
                     decayEarly: bool, normInput: bool, surrogateKind: int, surrP0: float, surrP1: float,
                     gradInput: Optional[torch.Tensor] = None, surr: Optional[torch.Tensor] = None,
                     gradVRec: Optional[torch.Tensor] = None, gradIRec: Optional[torch.Tensor] = None,
                     wantAlphaMemGrad: bool = True, wantAlphaSynGrad: bool = True, wantVInitGrad: bool = True,
                     wantIInitGrad: bool = True, gradUniform: bool = False):
    """Returns (gradInput, alphaMemGrad, alphaSynGrad | None, vInitGrad, iInitGrad | None); a per-neuron
    gradient that is not wanted is neither computed nor allocated and comes back as None.
    ``gradUniform``: ``gradSpikes`` is a one-element tensor whose value is the gradient of every spike (the
    gradient of a sum of the output); the kernel then reads one tensor less.  Only with an in-kernel
    surrogate and without ``gradVRec`` / ``gradIRec``.
    ``surrogateKind == SURR_TENSOR`` takes the spike function's derivative from ``surr`` (batch, time, neurons).
    ``gradVRec`` / ``gradIRec`` (batch, time, neurons) are gradients on the forward's state records; one that is
    missing while the other is given counts as zero.
    ``ckptV is None`` calls ``exodus_layer_lif_backward_from_input``: the library rebuilds the checkpoints in its
    own fixed device array (``scratchFloats()``) and allocates nothing; concurrent calls on one GPU must not overlap."""
    if alphaSyn is None:
        gradILast = ckptI = isynInitial = gradIRec = None
    if ckptV is None:
        ckptI = None
    if surrogateKind != SURR_TENSOR:
        surr = None
    return _native.layer_lif_backward(
        gradSpikes, gradVLast, gradILast, input, ckptV, ckptI, vmemPostInitial, isynInitial, alphaMem, alphaSyn, membrSubtract,
        theta, thetaLow if applyThetaLow else None, bool(applyThetaLow), _cap(maxNumSpikes), bool(decayEarly), bool(normInput), int(surrogateKind),
        float(surrP0), float(surrP1), gradInput, surr, gradVRec, gradIRec, bool(wantAlphaMemGrad), bool(wantAlphaSynGrad),
        bool(wantVInitGrad), bool(wantIInitGrad), bool(gradUniform), _place(input))


def layerLeakyForward(input, vmemInitial, alpha, decayEarly: bool, normInput: bool,
                      stateShape: Optional[tuple] = None, wantSum: bool = False):
    """Leaky-integrator layer on (batch, time, neurons): returns (out, v_last), or with ``wantSum``
    (out, v_last, out_sum) where out_sum is a float64 scalar holding the sum of all outputs."""
    res = _native.layer_leaky_forward(input, vmemInitial, alpha, bool(decayEarly), bool(normInput), stateShape, bool(wantSum),
                                      _place(input))
    return res if wantSum else res[:2]


def layerLeakyBackward(gradOut, gradVLast, out, input, vmemInitial, alpha, decayEarly: bool, normInput: bool,
                       needAlphaGrad: bool, shape: Optional[tuple] = None):
    """Returns (gradInput, alphaGrad | None, vInitGrad).  With ``shape`` = (batch, time, neurons), ``gradOut`` is a
    one-element tensor whose value is the gradient of every output (the gradient of a sum)."""
    if shape is not None:
        shape = tuple(int(v) for v in shape)
    if not needAlphaGrad:
        out = input = vmemInitial = None
    elif not (decayEarly or normInput):
        input = None
    return _native.layer_leaky_backward(gradOut, gradVLast, out, input, vmemInitial, alpha, bool(decayEarly), bool(normInput),
                                        bool(needAlphaGrad), shape, _place(gradOut, shape))
