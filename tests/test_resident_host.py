"""The host side of the resident-activation GEMM (qlx_linear_resident): its plan on both sides of the
kernel's size limits; and the counters of its and the other kernels' K slices. Nothing here reaches a GPU."""

import ctypes
import types

import pytest
import torch

from kernels import _lib, qlinear

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
    monkeypatch.setattr(_lib, "_local", _lib._Local())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(synchronize=lambda: None))
    return captures


CPU = torch.device("cpu", 0)
SIZE = 4 * _lib.STREAM_TICKETS


def in_slots(address):
    base = _lib._stream_tickets[0][0].data_ptr()
    return base <= address < base + SIZE * _lib.STREAM_SLOTS


def test_captured_calls_count_apart_from_every_other_call(counters):
    """A graph's replays may overlap eager calls and other graphs' replays, whatever stream each was
    captured on: one capture's calls on one stream share counters, no other calls do."""
    eager = _lib.stream_tickets(CPU, 16)
    seen = {eager}
    for capture in range(1, _lib.STREAM_SLOTS):  # from the middle on the slots are taken
        counters.update({16: capture, 32: capture})  # the same streams captured again, one forked to
        held = [_lib.stream_tickets(CPU, s) for s in (16, 32)]
        assert held == [_lib.stream_tickets(CPU, s) for s in (16, 32)] and held[0] != held[1]
        for a in held:
            assert not in_slots(a) or a not in seen
        if capture < _lib.STREAM_SLOTS // 2 - 1:
            assert in_slots(held[0]) and in_slots(held[1])
        seen |= set(held)
        counters.clear()
        assert _lib.stream_tickets(CPU, 16) == eager
    assert not in_slots(held[1]) and not _lib._stream_tickets[0][0].any()


def test_counters_outside_the_slots_are_the_captures_own(counters):
    """The first sliced call of a device may be a captured one: the slots are made, and zeroed, by an eager
    call, the captured calls' counters are zeroed in their capture and go with it."""
    held = []
    for capture in (7, 8):
        counters.update({16: capture, 32: capture})
        at = [_lib.stream_tickets(CPU, s) for s in (16, 32, 16, 32)]
        assert at[:2] == at[2:] and at[0] != at[1] and not _lib._stream_tickets
        held.append(list(_lib._local.counters.values()))
        assert [b.data_ptr() for b in held[-1]] == at[:2] and not any(b.any() for b in held[-1])
    assert len({b.data_ptr() for bufs in held for b in bufs}) == 4
    counters.clear()
    assert in_slots(_lib.stream_tickets(CPU, 16)) and not _lib._stream_tickets[0][0].any()
    assert not _lib._local.counters, "an ended capture's memory goes back to its pool"
    _lib.stream_tickets(CPU, 16, 9496)
    assert _lib._local.capture == 0 and all(b is not h for b in _lib._local.counters.values() for h in held[-1])


def test_streams_past_the_slots_share_none(counters):
    """Each stream counts apart from those that hold a slot, and from every other, also past them."""
    streams = [16 * s for s in range(1, _lib.STREAM_SLOTS + 9)]
    at = [_lib.stream_tickets(CPU, s) for s in streams]
    base = _lib._stream_tickets[0][0].data_ptr()
    assert sorted(at[:_lib.STREAM_SLOTS]) == [base + SIZE * i for i in range(_lib.STREAM_SLOTS)]
    assert len(set(at)) == len(at) and not any(in_slots(a) for a in at[_lib.STREAM_SLOTS:])
    assert len(_lib._stream_tickets[0][1]) == _lib.STREAM_SLOTS
    assert at == [_lib.stream_tickets(CPU, s) for s in streams]
    for s in range(1, 200):  # what lies outside the slots stays bounded
        _lib.stream_tickets(CPU, 16 * (s + 2 * _lib.STREAM_SLOTS))
    assert len(_lib._local.counters) <= 64


def test_the_other_kernels_calls_count_apart_too(counters, monkeypatch):
    """tickets() of the decode and skinny kernels: by stream, a capture's own, more of them when asked."""
    def at(stream, count=160):
        monkeypatch.setattr(_lib, "stream", lambda device: stream)
        return _lib.tickets(CPU, count)

    assert at(16) == at(16) == _lib.stream_tickets(CPU, 16) != at(32)
    wide = at(16, 9496)
    assert wide == at(16, 9496) and not in_slots(wide) and wide != at(32, 9496)
    assert _lib._local.counters[0, 16].numel() >= 9496
    eager = [at(16), at(32), wide]
    keep = list(_lib._local.counters.values())
    counters.update({16: 3, 32: 3})
    held = [at(16), at(32), at(16, 9496)]
    assert not set(held) & set(eager) and len(set(held)) == 3
    keep += _lib._local.counters.values()
    counters.update({16: 4})
    assert at(16) not in held and at(16, 9496) not in held and not any(b.any() for b in keep)


@pytest.mark.parametrize("name,n,k,ours,others", [
    # 8-bit weights over 64 MiB, and FP8 of one token
    ("fp8", 151936, 2560, (), (1, 2, 8, 16, 64)), ("w8a16", 151936, 2560, (33, 64), (1, 8, 16, 32)),
    # long runs: from 1024 tiles (FP8), past 1024 and 1536 (W8A16), between 1536 and 2048 (W4A16)
    ("fp8", 16368, 2560, (2, 8, 9, 32, 64), (1,)), ("fp8", 16384, 2560, (2, 8), (9, 16, 32, 33, 64)),
    ("w8a16", 16384, 2560, (1, 8, 9, 16, 17, 64), ()), ("w8a16", 16400, 2560, (1, 8, 17, 32, 64), (9, 16)),
    ("w8a16", 24576, 2048, (8, 17, 32, 33), (9, 16)), ("w8a16", 24592, 2048, (8, 33, 64), (9, 16, 17, 32)),
    ("w4a16", 24576, 2560, (1, 8, 9, 16, 32, 64), ()), ("w4a16", 24592, 2560, (1, 8, 33, 64), (9, 16, 17, 32)),
    ("w4a16", 32768, 2560, (1, 8, 33, 64), (9, 16, 17, 32)), ("w4a16", 32784, 2560, (1, 8, 9, 16, 32, 64), ()),
    ("w4a16", 65520, 2560, (1, 4, 9, 32), ()), ("w4a16", 65536, 2560, (5, 8, 9, 32, 64), (1, 4)),
    # runs of K slices
    ("fp8", 4080, 8192, (2, 4, 8), (1,)), ("fp8", 4096, 8192, (8,), (2, 4)), ("fp8", 8192, 8192, (), (2, 4, 8)),
    ("fp8", 10224, 6144, (9, 64), ()), ("fp8", 10240, 6144, (), (9, 16, 64)),
    ("w8a16", 28672, 5120, (33, 64), ()), ("w8a16", 28688, 5120, (), (33, 64)), ("w8a16", 28688, 2560, (33, 64), ()),
    ("w8a16", 28688, 1024, (), (33, 64)), ("w4a16", 65536, 5120, (16, 33), (17, 32)),
    ("w4a16", 4096, 9728, (4,), (1, 2)), ("w4a16", 8208, 9728, (1, 2, 4), ()),
    # the reference's formats, whose calls the decode kernel takes otherwise
    ("int8g64", 151936, 2560, (1, 8, 16, 64), ()), ("int4g64", 151936, 2560, (1, 8, 16, 64), ())])
def test_plan_leaves_the_calls_that_another_kernel_streams_faster(name, n, k, ours, others):
    """Both sides of each line of the dispatch."""
    for m in ours:
        assert planned(FORMATS[name][0], m, n, k).splits >= 1, (name, n, k, m)
    for m in others:
        assert planned(FORMATS[name][0], m, n, k).splits == 0, (name, n, k, m)


@pytest.mark.parametrize("fmt,m,has", [("fp8", 1, False), ("fp8", 8, True), ("w8a16", 1, True), ("w4a16", 64, True)])
def test_a_race_has_the_resident_gemm_where_its_plan_has_the_call(fmt, m, has):
    """A candidate named for a kernel is that kernel, not what serves the call without it."""
    from kernels import gemm
    weight = torch.zeros(2560, 512 if fmt == "w4a16" else 1024, dtype=torch.uint8)
    tiles = qlinear.Tiled(weight, torch.zeros(2560 * (8 if fmt == "w4a16" else 1), dtype=torch.bfloat16), 2560, 1024, fmt)
    assert has == any("resident" in c.label for c in gemm._north_candidates(m, [tiles], False))
    off = qlinear.Tiled(torch.zeros(weight.numel() + 8, dtype=torch.uint8)[8:], tiles.scale, 2560, 1024, fmt)
    assert off.weight.data_ptr() % 16 and not any("resident" in c.label for c in gemm._north_candidates(m, [off], False))


def test_plan_slices_is_the_planned_shape_fitted():
    """qlx_plan_slices: what make_plan and a fit of its workgroup shape give in turn."""
    from kernels import _linear
    for fmt in (_lib.FMT_REF8, _lib.FMT_REF4, _lib.FMT_W8A16):
        for n, k in ((512, 1024), (2560, 9728), (19456, 2560), (4096, 28672)):
            for m in (1, 8, 17, 64):
                for ask in (1, 4):
                    base = _linear.make_plan(fmt, _lib.MODE_PLANES, m, n, k)
                    want = _linear.splits_for(fmt, _lib.MODE_PLANES, m, n, k, (base.waves, base.kw, base.rw, ask), fit=True)
                    assert _lib.lib().qlx_plan_slices(fmt, _lib.MODE_PLANES, m, n, k, ask) == want
    assert _lib.lib().qlx_plan_slices(_lib.FMT_REF8, 0, 0, 512, 1024, 1) == _lib.QLX_EINVAL
