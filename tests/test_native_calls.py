"""The native host side of the kernel calls: what it refuses, which exceptions callers see, and calls from several threads on
several streams at once."""
import ctypes
import importlib.util
import os
import subprocess
import sys
import threading
import time

import pytest
import torch


def hip():
    from sinabs.exodus import _hip
    return _hip


def calls(x, r, two):
    """name -> call with the (batch, time, neurons) tensor x, the per-neuron vector r and the (rows, time) matrix two"""
    h = hip()
    return {
        "layerLifForward": lambda: h.layerLifForward(x, r, None, r, None, r, r, None, False, -1, True, True),
        "layerLifBackward": lambda: h.layerLifBackward(x, None, None, x, None, None, r, None, r, None, r, r, None, False, -1,
                                                       True, True, 1, 0.5, 1.0),
        "layerLeakyForward": lambda: h.layerLeakyForward(x, r, r, True, True),
        "layerLeakyBackward": lambda: h.layerLeakyBackward(x, None, x, x, r, r, True, True, True),
        "decayExpand": lambda: h.decayExpand(r, 1, 6),
        "decayGrad": lambda: h.decayGrad(r, r, 1, 6),
        "lifForward": lambda: h.lifForward(two, two, two, r, r, r, r, None, False, -1),
        "lifBackwardFused": lambda: h.lifBackwardFused(two, None, two, r, r, r, r, None, False, -1, 1),
        "leakyForward": lambda: h.leakyForward(two, r, r),
        "leakyBackwardFused": lambda: h.leakyBackwardFused(two, r, two, r, True),
    }


NAMES = ("layerLifForward", "layerLifBackward", "layerLeakyForward", "layerLeakyBackward", "decayExpand", "decayGrad",
         "lifForward", "lifBackwardFused", "leakyForward", "leakyBackwardFused")


@pytest.mark.parametrize("name", NAMES)
def test_tensors_that_are_not_on_the_gpu_and_things_that_are_no_tensors(name):
    with pytest.raises(RuntimeError, match="HIP device"):
        calls(torch.zeros(1, 4, 6), torch.zeros(6), torch.zeros(6, 4))[name]()
    with pytest.raises(TypeError):
        calls([0.0], [0.0], [0.0])[name]()


@pytest.mark.gpu
def test_arguments_that_a_call_does_not_use_may_be_anything():
    h, no = hip(), "nothing"
    x, r, two = torch.rand(1, 4, 6).cuda(), torch.rand(6).cuda() * 0.5 + 0.3, torch.rand(6, 4).cuda()
    ck = torch.rand(1, 1, 6).cuda()
    h.lifForward(two.clone(), two.clone(), two, r, r, r, r, no, False, -1)
    h.leakyBackwardFused(two, r, no, no, False)
    h.lifBackwardFused(two, None, two, no, r, r, r, no, False, -1, 1, surr=no)
    h.layerLifForward(x, r, no, r, None, r, r, no, False, -1, True, True)
    h.layerLifBackward(x, None, no, x, ck, no, r, no, r, None, r, r, no, False, -1, True, True, 1, 0.5, 1.0, surr=no, gradIRec=no)
    h.layerLifBackward(x, None, None, x, None, no, r, r, r, r, r, r, no, False, -1, True, True, 1, 0.5, 1.0)
    h.layerLeakyBackward(x, None, no, no, no, r, True, True, False)
    h.layerLeakyBackward(x, None, x, no, r, r, False, False, True)


@pytest.mark.parametrize("most,bits", [(-1, -1), (0, 0), (7, 7), (2 ** 31 - 1, 2 ** 31 - 1), (2 ** 31, -2 ** 31),
                                       (2 ** 32 - 2, -2), (2 ** 32 - 1, -1), (2 ** 32, -1), (2 ** 32 + 5, -1), (10 ** 20, -1)])
def test_spike_limits_of_any_size(most, bits):
    assert hip()._cap(most) == bits


@pytest.mark.gpu
@pytest.mark.parametrize("most", [2 ** 31, 2 ** 32, 2 ** 63, 10 ** 20])
def test_a_limit_that_no_count_reaches(most):
    import sinabs.exodus.layers as el
    from sinabs.exodus._compat import MaxSpike, MultiSpike
    x = (10.0 * torch.rand(2, 20, 30)).cuda()
    for native in (True, False):
        outs = []
        for spike_fn in (MultiSpike, MaxSpike(most)):
            layer = el.IAF(spike_fn=spike_fn).cuda()
            layer.native_layout = native
            outs.append(layer(x))
        assert outs[0].max() > 2 and torch.equal(*outs)


def test_library_of_another_version_is_refused():
    """Neither the Python nor the native half takes it, and the native half keeps the library it has."""
    h, native = hip(), hip()._native
    addresses = {name: ctypes.cast(getattr(h.lib, name), ctypes.c_void_p).value for name in h._SIGNATURES}
    other = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: h.ABI_VERSION - 1)
    wrong = {**{name: 0 for name in addresses}, "exodus_hip_abi_version": ctypes.cast(other, ctypes.c_void_p).value}
    with pytest.raises(ImportError, match=f"version {h.ABI_VERSION - 1}"):
        native.bind(wrong, h._check)
    native.bind(addresses, h._check)


def test_library_without_an_entry_point_is_named():
    probes = os.path.join(os.path.dirname(hip().__file__), "..", "..", "libexodus_bench_probes.so")
    got = subprocess.run([sys.executable, "-c", "import sinabs.exodus.layers"], capture_output=True, text=True,
                         env={**os.environ, "EXODUS_HIP_LIBRARY": os.path.abspath(probes),
                              "PYTHONPATH": os.path.join(os.path.dirname(hip().__file__), "..", "..")})
    assert got.returncode != 0 and "ImportError" in got.stderr and "exodus_check_parameters" in got.stderr, got.stderr


def builder():
    path = os.path.join(os.path.dirname(hip().__file__), "..", "..", "build_hip.py")
    spec = importlib.util.spec_from_file_location("build_hip_under_test", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def test_module_built_for_another_torch_is_refused_and_built_again(monkeypatch):
    build_hip, h = builder(), hip()
    assert h._native.built_for == build_hip.built_for()
    monkeypatch.setattr(build_hip.os.path, "getmtime", lambda path: 0.0)    # as if no source had changed
    assert build_hip.up_to_date()
    monkeypatch.setattr(torch, "__version__", "1.13.1")
    assert not build_hip.up_to_date()
    with pytest.raises(ImportError, match="torch 1.13.1.*[Bb]uild it"):
        h._native_module()


def test_build_failure_names_compiler_and_source(monkeypatch, tmp_path):
    build_hip = builder()
    broken = tmp_path / "broken.cpp"
    broken.write_text("#error on purpose\n")
    monkeypatch.setattr(build_hip, "SRCS", [])
    monkeypatch.setattr(build_hip, "TORCH_SRC", str(broken))
    for name in ("OUT", "PROBE_OUT", "TORCH_OUT"):
        monkeypatch.setattr(build_hip, name, str(tmp_path / name))
    with pytest.raises(RuntimeError, match=r"^g\+\+ failed compiling broken.cpp$"):
        build_hip.build()


@pytest.mark.gpu
@pytest.mark.parametrize("name", NAMES)
def test_wrong_types_shapes_and_strides(name):
    x, r, two = torch.rand(1, 4, 6).cuda(), torch.rand(6).cuda() * 0.5 + 0.3, torch.rand(6, 4).cuda()
    calls(x, r, two)[name]()
    with pytest.raises(RuntimeError, match=r"must be float32 \(got torch.float64\)"):
        calls(x.double(), r.double(), two.double())[name]()
    with pytest.raises(RuntimeError, match="contiguous"):
        calls(x.transpose(1, 2), r.repeat_interleave(2)[::2], two.t())[name]()
    if not name.startswith("decay"):
        with pytest.raises(RuntimeError, match=r"must have shape \(6,\), got \(7,\)"):
            calls(x, torch.rand(7).cuda(), two)[name]()
        with pytest.raises(RuntimeError, match="3-D|2-D"):
            calls(r, r, r)[name]()


@pytest.mark.gpu
def test_a_status_of_the_library_becomes_its_own_exception():
    h = hip()
    wide = torch.empty(1, 0, h.LAYER_MAX_NEURONS).cuda()
    r = torch.empty(h.LAYER_MAX_NEURONS).cuda()
    x = torch.zeros(1, 1, h.LAYER_MAX_NEURONS).cuda()
    assert h.layerLeakyForward(wide, r, r, False, False)[0].numel() == 0      # no step: nothing to refuse
    with pytest.raises(h.ExodusHipError, match="exodus_layer_leaky_forward_total failed"):
        h.layerLeakyForward(x, r, r, False, False)


@pytest.mark.gpu
@pytest.mark.parametrize("constant", [False, True])
def test_the_entry_point_that_failed_is_the_one_named(constant):
    h = hip()
    x, r = torch.zeros(1, 1, h.LAYER_MAX_NEURONS).cuda(), torch.ones(h.LAYER_MAX_NEURONS).cuda()
    tau, alpha = (torch.ones(1).cuda(), None) if constant else (None, r)
    form = "decays" if constant else "total"
    with pytest.raises(h.ExodusHipError, match=f"exodus_layer_leaky_forward_{form} failed"):
        h.layerLeaky(x, alpha, r, tau, False, False, (1, h.LAYER_MAX_NEURONS))
    with pytest.raises(h.ExodusHipError, match=f"exodus_layer_lif_forward_{form} failed"):
        h.layerLif(x, alpha, None, r, None, tau, None, None, None, r, r, None, 1, 0.5, 1.0, -1, False, False, False,
                   (1, h.LAYER_MAX_NEURONS))


@pytest.mark.gpu
def test_running_out_of_memory_is_torchs_exception():
    tau = torch.ones(1).cuda()
    with pytest.raises(torch.OutOfMemoryError):
        hip().decayExpand(tau, 1 << 40, 1)
    assert hip().decayExpand(tau, 4, 1)[0].shape == (4,)


@pytest.mark.gpu
def test_other_threads_run_while_an_allocation_waits():
    """The allocator at its limit gives cached memory back, for which it waits for the device: here for a kernel of half a second."""
    tau = torch.ones(1).cuda()
    began, ended = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    torch.cuda._sleep(1000)
    began.record()
    torch.cuda._sleep(10_000_000)
    ended.record()
    torch.cuda.synchronize()
    cycles = int(10_000_000 * 500 / began.elapsed_time(ended))
    torch.cuda.empty_cache()
    # memory that can be given back: a segment of its own, not a piece of one that something else still uses
    held, before = [], torch.cuda.memory_reserved()
    while torch.cuda.memory_reserved() == before:
        held.append(torch.empty(1 << 30, dtype=torch.uint8, device="cuda"))
    held.pop()
    gaps, stop = [], threading.Event()

    def tick():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.002)
            now = time.perf_counter()
            gaps.append(now - last)
            last = now

    other = threading.Thread(target=tick)
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (64 << 20)) / total)
    try:
        other.start()
        torch.cuda._sleep(cycles)
        start = time.perf_counter()
        with pytest.raises(torch.OutOfMemoryError):
            hip().decayExpand(tau, 1 << 31, 1)
        waited = time.perf_counter() - start
    finally:
        stop.set()
        other.join()
        torch.cuda.set_per_process_memory_fraction(1.0)
        torch.cuda.synchronize()
    assert waited > 0.2 and max(gaps) < waited / 2, (waited, max(gaps))


@pytest.mark.gpu
def test_threads_on_streams_of_their_own():
    import sinabs.exodus.layers as el
    want, got = {}, {}

    def step(k, into):
        g = torch.Generator(device="cuda").manual_seed(k)
        layer = el.LIF(tau_mem=10.0 + k, tau_syn=5.0).cuda()
        x = torch.empty(3 + k, 70, 50, device="cuda").normal_(0.5, 2.0, generator=g).requires_grad_(True)
        for _ in range(5):
            layer.reset_states()
            layer.zero_grad()
            x.grad = None
            out = layer(x)
            out.backward(torch.ones_like(out))
        torch.cuda.current_stream().synchronize()
        into[k] = (out.detach().cpu(), x.grad.cpu(), layer.tau_mem.grad.cpu())

    def on_stream(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            step(k, got)

    for k in range(4):
        step(k, want)
    threads = [threading.Thread(target=on_stream, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(4):
        for p, q in zip(want[k], got[k]):
            assert torch.equal(p, q)
