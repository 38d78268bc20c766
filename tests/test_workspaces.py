"""The host's account of split-K workspaces and their give-up reports, on the CPU:
buffers in host memory stand for the device's, a write to the word at the address a
buffer carries for the kernel's report. (The kernel's side: tests/test_gpu_fixup.py.)"""

from __future__ import annotations

import ctypes

import pytest
import torch

from ternel_amd import _lib, kernels

OFFSET = kernels._HOST_WORD_OFFSET
ERROR_WORD = 64 * 1024 - 4
CPU = torch.device("cpu")


@pytest.fixture
def host(monkeypatch):
    """The module's state emptied, with device calls replaced by host ones;
    ``host.stream`` and ``host.capturing`` are what the calls find."""

    class Host:
        stream, capturing = 7, False

    class Word(kernels._HostWord):
        def __init__(self) -> None:
            self.tensor = torch.zeros(1, dtype=torch.int32)
            self.word = ctypes.c_int.from_address(self.tensor.data_ptr())

    state = Host()
    for name, value in (("_WORKSPACES", {}), ("_RETIRED", []), ("_CAPTURED", set()), ("_FLAGS", {}),
                        ("_FLAG_WORDS", ()), ("_HostWord", Word)):
        monkeypatch.setattr(kernels, name, value)
    monkeypatch.setattr(kernels, "_device_index", lambda device: 0)
    monkeypatch.setattr(kernels, "_raw_stream", lambda index: state.stream)
    monkeypatch.setattr(kernels, "_new_buffer", lambda index, nbytes: torch.full((nbytes,), 255, dtype=torch.uint8))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state.capturing)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda index=None: None)
    return state


def give_up(buf: torch.Tensor) -> None:
    """What a kernel does: the error word, then the host word it finds in the buffer."""
    buf[ERROR_WORD:ERROR_WORD + 4].view(torch.int32).fill_(2)
    address = int(buf[OFFSET:OFFSET + 8].view(torch.int64).item())
    ctypes.c_int.from_address(address).value = 2


def error_word(buf: torch.Tensor) -> int:
    return int(buf[ERROR_WORD:ERROR_WORD + 4].view(torch.int32).item())


def clean(buf: torch.Tensor) -> bool:
    rest = buf.clone()
    rest[OFFSET:OFFSET + 8] = 0
    return not bool(rest.any())


def test_a_report_from_a_replaced_workspace_clears_every_buffer_of_its_stream(host) -> None:
    old = kernels.workspace(CPU, 1 << 22)
    host.capturing, host.stream = True, 8       # a capture borrows it
    assert kernels.workspace(CPU, 1 << 22) is old
    host.capturing, host.stream = False, 7
    new = kernels.workspace(CPU, 1 << 23)       # replaced, and still the graph's
    assert new is not old and kernels._RETIRED[0][1] is old
    host.stream = 9
    other = kernels.workspace(CPU, 1 << 22)
    for buf in (old, new, old):                 # reports again after each recovery
        give_up(buf)
        with pytest.raises(_lib.NativeError, match="bounded wait"):
            kernels._surface(0)
        assert clean(old) and clean(new) and clean(other)
        kernels._surface(0)                     # nothing left to report


def test_growth_keeps_a_report_that_no_call_has_raised(host) -> None:
    old = kernels.workspace(CPU, 1 << 22)
    give_up(old)
    new = kernels.workspace(CPU, 1 << 23)
    assert clean(new)
    with pytest.raises(_lib.NativeError, match="bounded wait"):
        kernels._surface(0)
    kernels._surface(0)


def test_a_report_is_kept_while_a_stream_captures(host) -> None:
    buf = kernels.workspace(CPU, 1 << 22)
    give_up(buf)
    host.capturing = True
    kernels._surface(0)
    assert error_word(buf) == 2
    host.capturing = False
    with pytest.raises(_lib.NativeError):
        kernels._surface(0)


def test_sizes_are_kept_per_device_that_plans_the_launch(monkeypatch) -> None:
    """The library plans on the current device: an answer given there is not
    used for a call made while another one is current."""

    class Library:
        def __getattr__(self, name):
            return lambda *sizes: 1000 * device + len(sizes)

    device = 0
    monkeypatch.setattr(_lib, "lib", lambda: Library())
    monkeypatch.setattr(kernels, "_plan_device", lambda: device)
    caches = (kernels._answer, kernels._linear_answers)
    for cache in caches:
        cache.cache_clear()
    try:
        calls = (lambda: kernels._matmul_bytes(2, 64, 128, 0, 0), lambda: kernels._gemm_bytes(2, 64, 128, 0, 0),
                 lambda: kernels._linear_plan(2, 64, 128, 0)[1],
                 lambda: kernels._swiglu_bytes(2, 64, 128, 0))
        first = [call() for call in calls]
        device = 1
        assert [call() for call in calls] == [1000 + value for value in first]
        device = 0
        assert [call() for call in calls] == first
    finally:
        for cache in caches:
            cache.cache_clear()
