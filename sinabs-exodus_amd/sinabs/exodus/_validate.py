"""Value checks on device-resident parameters.

The reference Functions test ``0 <= alpha <= 1`` and ``threshold > min_v_mem`` with ``.any()`` on
device tensors (reference sinabs/exodus/spike.py:183-191), which makes the host wait for the device
on every forward call.  Three modes, selected with ``set_mode``:

``"sync"`` (default)   the call that carries a violation raises the ``ValueError``, as in the reference; the host
                        waits for the flags alone, and the call's own kernel runs meanwhile;
``"deferred"``          the flags are copied to pinned host memory without waiting; a violation is
                        raised by a later call into this module (or by ``flush()``), so the host can
                        keep queueing work;
``"off"``               no checks.

While the current stream is capturing a HIP graph no check runs in any mode: the capture cannot wait
for the device, and a replay has no host code that could raise.
"""
from typing import List, Optional, Sequence

import torch

from . import _hip

_MODE = "sync"
_ALPHA_MSG = "'alpha' must be between 0 and 1."
_THRESHOLD_MSG = "`threshold` must be greater than `min_v_mem`."
_pending: List[tuple] = []          # (event, pinned flags, messages)


def set_mode(mode: str) -> None:
    global _MODE
    if mode not in ("sync", "deferred", "off"):
        raise ValueError("mode must be 'sync', 'deferred' or 'off'")
    flush()
    _MODE = mode


def get_mode() -> str:
    return _MODE


def _raise_if_flagged(flags: Sequence, messages: Sequence[str]) -> None:
    for flag, msg in zip(flags, messages):
        if flag:
            raise ValueError(msg)


def _poll(wait: bool) -> None:
    while _pending:
        event, host_flags, messages = _pending[0]
        if not wait and not event.query():
            return
        if wait:
            event.synchronize()
        _pending.pop(0)
        _raise_if_flagged(host_flags.tolist(), messages)


def flush() -> None:
    """Wait for all deferred checks and raise the first violation found."""
    _poll(wait=True)


class _Running:
    """Checks whose flags are on their way from the device to the host."""

    def __init__(self, event, flags, messages):
        self.event, self.flags, self.messages = event, flags, messages

    def finish(self) -> None:
        """Wait for the flags (not for what was launched after the checks) and raise what they say."""
        self.event.synchronize()
        _raise_if_flagged(self.flags.tolist(), self.messages)


class _Done:
    def finish(self) -> None:
        pass


_DONE = _Done()


def _one_kernel_checks(tensors) -> bool:
    """Whether the checks are one kernel: float32 vectors of one length next to each other on a GPU."""
    first = tensors[0]
    return (first.is_cuda and all(t.dtype == torch.float32 and t.device == first.device and t.is_contiguous()
                                  and t.shape == first.shape for t in tensors))


def check_parameters(alphas: Sequence[torch.Tensor], threshold: Optional[torch.Tensor] = None,
                     min_v_mem: Optional[torch.Tensor] = None, wait: bool = True):
    """``alphas``: decay factors that must lie in [0, 1]; ``threshold`` must exceed ``min_v_mem``.  ``wait=False``: what is
    launched between this call and ``finish()`` of its result runs while the host waits for the flags; ``finish()`` has to be
    called in any case (the flags' memory is given back then)."""
    running = _begin(alphas, threshold, min_v_mem)
    if not wait:
        return running
    running.finish()


def _begin(alphas, threshold, min_v_mem):
    if _MODE == "off":
        return _DONE
    if torch.cuda.is_available() and torch.cuda.is_current_stream_capturing():
        return _DONE    # a graph under capture can neither wait for the device nor raise on replay
    if _MODE == "deferred":
        _poll(wait=False)
    checked = list(alphas) + ([threshold, min_v_mem] if min_v_mem is not None else [])
    if not checked:
        return _DONE
    if len(alphas) <= 2 and _one_kernel_checks(checked):
        first = checked[0]
        host = torch.zeros(2, dtype=torch.int32, device="cpu", pin_memory=True)
        _hip.checkParameters(host, alphas[0] if alphas else None, alphas[1] if len(alphas) > 1 else None,
                             threshold if min_v_mem is not None else None, min_v_mem)
        messages = (_ALPHA_MSG, _THRESHOLD_MSG)
        event = torch.cuda.Event()
        event.record(torch.cuda.current_stream(first.device))
        if _MODE == "sync":
            return _Running(event, host, messages)
        _pending.append((event, host, messages))
        return _DONE
    flags = [((a < 0) | (a > 1)).any() for a in alphas]
    messages = [_ALPHA_MSG] * len(flags)
    if min_v_mem is not None:
        flags.append((threshold <= min_v_mem).any())
        messages.append(_THRESHOLD_MSG)
    stacked = torch.stack(flags)
    if _MODE == "sync" or not stacked.is_cuda:
        _raise_if_flagged(stacked.tolist(), messages)
        return _DONE
    host = torch.empty(stacked.shape, dtype=stacked.dtype, device="cpu", pin_memory=True)
    host.copy_(stacked, non_blocking=True)
    event = torch.cuda.Event()
    event.record(torch.cuda.current_stream(stacked.device))
    _pending.append((event, host, messages))
    return _DONE
