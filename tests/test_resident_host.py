"""The host side of the resident-activation GEMM (qlx_linear_resident): its plan on both sides of the
kernel's size limits; and the counters of its and the other kernels' K slices. Nothing here reaches a GPU."""

import ctypes
import types

import pytest
import torch

from kernels import _lib

FORMATS = {"w4a16": (_lib.FMT_W4A16, 2), "w8a16": (_lib.FMT_W8A16, 1), "fp8": (_lib.FMT_FP8, 1),
           "int8g64": (_lib.FMT_REF8, 1), "int4g64": (_lib.FMT_REF4, 2)}  # format, codes a byte


def planned(fmt, m, n, k):
    plan = _lib.Plan()
    assert _lib.lib().qlx_plan_resident(fmt, _lib.MODE_BF16, m, n, k, plan) == 0
    return plan


@pytest.mark.parametrize("name", list(FORMATS))
def test_plan_takes_no_call_that_the_kernel_refuses(name):
    """At and around 2 GiB of weights a plan with slices is one that the call accepts: the error is
    then the misaligned weight's, which is looked at after every size."""
    fmt, per_byte = FORMATS[name]
    served = 0
    for k in (4096, 16384):
        edge = (1 << 31) * per_byte // k  # rows of 2 GiB
        for n in (151936, edge - 16, edge, edge + 16, 2 * edge):
            for m in (1, 5, 16, 33, 64):
                plan = planned(fmt, m, n, k)
                if plan.splits == 0:
                    continue
                served += 1
                plan.workspace = plan.tickets = 1 << 20
                rc = _lib.lib().qlx_linear_resident(fmt, 8, 16, 16, 16, 16, m, n, k, ctypes.byref(plan), None)
                assert rc == _lib.QLX_EINVAL and "16-byte boundaries" in _lib.last_error(), (name, m, n, k, _lib.last_error())
                assert n < edge, (name, m, n, k)
    assert served or name == "fp8"  # FP8 weights of over 64 MiB are left to another kernel


@pytest.fixture
def counters(monkeypatch):
    """The counters on CPU memory, their state put back afterwards; returns the capture of each stream."""
    captures = {}
    monkeypatch.setattr(_lib, "capture_id", lambda stream: captures.get(stream, 0), raising=False)
    monkeypatch.setattr(_lib, "_stream_tickets", {})
    monkeypatch.setattr(_lib, "_tickets", {})
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(synchronize=lambda: None))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(captures))
    return captures


def test_captured_calls_count_apart_from_every_other_call(counters):
    """A graph's replays may overlap eager calls and other graphs' replays, whatever stream each was
    captured on: one capture's calls on one stream share counters, no other calls do."""
    cpu = torch.device("cpu", 0)
    eager = _lib.stream_tickets(cpu, 16)
    seen = {eager}
    for capture in (1, 2):
        counters.update({16: capture, 32: capture})  # the same streams captured again, one forked to
        held = [_lib.stream_tickets(cpu, s) for s in (16, 32)]
        keep = list(_lib._local.counters.values())  # the graph's memory
        assert held == [_lib.stream_tickets(cpu, s) for s in (16, 32)]
        assert len(seen | set(held)) == len(seen) + 2
        seen |= set(held)
        counters.clear()
        assert _lib.stream_tickets(cpu, 16) == eager and not _lib._local.counters
        assert all(int(buf.abs().sum()) == 0 for buf in keep)


def test_a_capture_makes_no_counters_for_eager_calls(counters):
    """The first sliced call of a device may be a captured one; the eager calls' counters are made, and
    zeroed, by an eager call."""
    cpu = torch.device("cpu", 0)
    counters[16] = 7
    _lib.stream_tickets(cpu, 16)
    assert not _lib._stream_tickets
    counters.clear()
    _lib.stream_tickets(cpu, 16)
    assert len(_lib._stream_tickets) == 1


def test_streams_past_the_slots_share_none(counters):
    """Each stream counts apart from the 64 that hold a slot, and from its neighbours, also past them."""
    cpu = torch.device("cpu", 0)
    at = [_lib.stream_tickets(cpu, 16 * s) for s in range(1, _lib.STREAM_SLOTS + 9)]
    base = _lib._stream_tickets[0][0].data_ptr()
    size = 4 * _lib.STREAM_TICKETS
    assert sorted(at[:_lib.STREAM_SLOTS]) == [base + size * i for i in range(_lib.STREAM_SLOTS)]
    assert all(not base <= a < base + size * _lib.STREAM_SLOTS for a in at[_lib.STREAM_SLOTS:])
    assert all(a != b for a, b in zip(at[_lib.STREAM_SLOTS:], at[_lib.STREAM_SLOTS + 1:]))
    assert len(_lib._stream_tickets[0][1]) == _lib.STREAM_SLOTS
    assert at[:_lib.STREAM_SLOTS] == [_lib.stream_tickets(cpu, 16 * s) for s in range(1, _lib.STREAM_SLOTS + 1)]


def test_the_other_kernels_calls_count_apart_too(counters, monkeypatch):
    """tickets() of the decode and skinny kernels: by stream, a capture's own, more of them when asked."""
    cpu = torch.device("cpu", 0)

    def at(stream, count=160):
        monkeypatch.setattr(_lib, "stream", lambda device: stream)
        buf = _lib.tickets(cpu, count)
        assert buf.numel() >= count and not buf.any()
        return buf

    eager = [at(16 * s) for s in range(1, _lib.STREAM_SLOTS + 4)]
    assert len({b.data_ptr() for b in eager}) == len(eager) and len(_lib._tickets) == _lib.STREAM_SLOTS
    assert at(16) is eager[0] and at(16, 9496) is at(16, 9496) is not eager[0]
    counters.update({16: 3, 32: 3})
    held = [at(16), at(32), at(16)]
    assert held[0] is held[2] is not held[1] and all(b is not h for b in _lib._tickets.values() for h in held)
    counters.update({16: 4})
    assert at(16) is not held[0]
