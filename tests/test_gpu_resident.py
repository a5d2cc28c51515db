"""The resident-activation GEMM (qlx_linear_resident): every format, at the edges of its launch --
token fragments and blocks (1 to 64 tokens), one tile to more tiles than workgroups, waves without
units, each K-slice count the shape takes, SwiGLU halves that are not whole tiles.

The comparison is with the decode kernel on the same weights (the same products summed in another order, so
outputs within one bf16 rounding step: 2^-7 of the value plus 2^-9 of the row's largest; SwiGLU, two
roundings more, 2^-6), and the oracle's dequantize-then-matmul at a rel-L2 of 1e-2. A
zero weight row gives exactly zero; fp32 planes summed in slice order are the reduced output."""

import functools

import numpy as np
import pytest
import torch

import oracle.qlinear_oracle as O
from kernels import _lib, _linear, cuda_fp8, qlinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FMTS = {"w4a16": _lib.FMT_W4A16, "w8a16": _lib.FMT_W8A16, "fp8": _lib.FMT_FP8, "int8g64": _lib.FMT_REF8,
        "int4g64": _lib.FMT_REF4}


def bits16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def make(fmt, n, k, seed):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16)
    w[0].zero_()
    bits = 4 if fmt in ("w4a16", "int4g64") else 8
    packed = cuda_fp8.quantize(w.to(DEV), bits=bits, fmt="ref" if fmt.endswith("g64") else fmt)
    return packed, cuda_fp8.prepare(packed)


def acts(m, k, seed):
    return torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(DEV)


def decode(fmt, x, p, swiglu):
    """The decode kernel's result on the same weights (explicit plan: no other kernel takes it)."""
    mode = _lib.MODE_SWIGLU if swiglu else _lib.MODE_BF16
    base = _linear.make_plan(FMTS[fmt], mode, x.shape[0], p.rows, p.k)
    cfg = (base.waves, base.kw, base.rw, base.splits)
    if fmt.endswith("g64"):
        return _linear.run(FMTS[fmt], "qlx_linear_ref", x, p.rows, p.k, (_lib.ptr(p.weight), _lib.ptr(p.scale), _lib.ptr(x)),
                           (p.bits, 1), mode=mode, config=cfg, fit=True)
    return qlinear.FORMATS[fmt][1](x, p.tiles, config=cfg, swiglu=swiglu)


def resident(fmt, x, p, splits, swiglu=False, planes=False, mode=None):
    xs = None
    if fmt == "fp8":
        x, xs = qlinear.quantize_fp8_activation(x)
    plan = _lib.Plan()
    plan.mode = mode or (_lib.MODE_PLANES if planes else (_lib.MODE_SWIGLU if swiglu else _lib.MODE_BF16))
    plan.splits = splits
    return qlinear.run_resident(plan, FMTS[fmt], p.weight, p.scale, x, xs, x.shape[0], p.rows, p.k)


def close(got, want, swiglu, what):
    got, want = got.float(), want.float()
    tol = (2.0 ** -6 if swiglu else 2.0 ** -7) * want.abs() + 2.0 ** -9 * want.abs().amax(dim=1, keepdim=True)
    assert bool(torch.isfinite(got).all()), what
    assert ((got - want).abs() > tol).sum().item() == 0, (what, (got - want).abs().max().item())


@pytest.mark.parametrize("fmt", list(FMTS))
@pytest.mark.parametrize("n,k,swiglu", [(16, 256, False), (48, 1024, True), (272, 2816, False), (2064, 3328, True),
                                        (4128, 512, False), (80, 9728, False)])
def test_resident_matches_decode_kernel(fmt, n, k, swiglu):
    packed, p = make(fmt, n, k, n + k)
    for m in (1, 2, 4, 5, 8, 9, 16, 17, 32, 33, 48, 64):
        x = acts(m, k, 100 + m)
        want = decode(fmt, x, p, swiglu)
        served = 0
        for s in (1, 2, 3, 5, 8):
            try:
                got = resident(fmt, x, p, s, swiglu)
            except ValueError:  # the slice does not fit the registers, or too few tiles for two token blocks
                continue
            served += 1
            print(f"resident {fmt} n={n} k={k} m={m} splits={s}", flush=True)
            close(got, want, swiglu, (fmt, n, k, m, s))
            assert torch.equal(got, resident(fmt, x, p, s, swiglu)), "deterministic"
            if not swiglu:
                assert not got[:, 0].float().abs().sum().item(), "a zero weight row gives zero"
        assert served or (m > 32 and n < 128), (fmt, n, k, m)
    assert all(int(buf.abs().sum()) == 0 for buf, _, _ in _lib._stream_tickets.values()), "tickets are left at zero"


@pytest.mark.parametrize("fmt", list(FMTS))
def test_resident_planes_and_oracle(fmt):
    n, k = 512, 2560
    packed, p = make(fmt, n, k, 5)
    for m in (3, 24, 64):
        print(f"resident planes {fmt} m={m}", flush=True)
        x = acts(m, k, m)
        for s in (1, 2, 4):
            got = resident(fmt, x, p, s)
            planes = resident(fmt, x, p, s, planes=True)
            acc = torch.zeros_like(planes[0])
            for plane in planes:
                acc += plane
            if fmt == "fp8":  # the token scale is part of a plane's values, the sum the same
                assert ((acc - got.float()).abs() <= 2.0 ** -8 * got.float().abs() + 1e-6).all()
            else:
                assert torch.equal(acc.to(torch.bfloat16), got), (fmt, m, s)
            one = resident(fmt, x, p, s, mode=_lib.MODE_SUM)
            assert one.shape == (1, m, n) and torch.equal(one[0], acc) and torch.equal(one[0].to(torch.bfloat16), got), (fmt, m, s)
        if fmt == "fp8":
            want = O.linear_fp8_w8a8(bits16(x), packed[0].view(torch.uint8).cpu().numpy(), bits16(packed[1])[:, None])
        else:
            want = O.linear_dequant(bits16(x), bits16(cuda_fp8.dequantize(packed)))
        assert O.rel_l2(resident(fmt, x, p, 1).float().cpu().numpy(), want) <= 1e-2


@pytest.mark.parametrize("fmt", list(FMTS))
def test_a_row_of_nan_or_inf_stays_in_its_row(fmt):
    """Rows are independent, also those that share a load (4 or 8 tokens) or a workgroup."""
    _, p = make(fmt, 256, 1024, 9)
    for m in (2, 4, 7, 20):
        print(f"resident nan row {fmt} m={m}", flush=True)
        x = acts(m, 1024, m)
        want = resident(fmt, x, p, 1)
        for bad in (float("nan"), float("inf")):
            y = x.clone()
            y[1, 3] = bad
            got = resident(fmt, y, p, 1)
            keep = [i for i in range(m) if i != 1]
            assert torch.equal(got[keep], want[keep]) and not bool(torch.isfinite(got[1, 1:]).all())


def test_operands_off_a_16_byte_boundary():
    """An activation that starts inside a larger buffer is read through a copy; a weight that does is
    left to the decode kernel."""
    _, p = make("w8a16", 256, 1024, 3)
    flat = torch.zeros(5 * 1024 + 3, dtype=torch.bfloat16, device=DEV)
    x = acts(5, 1024, 8)
    flat[3:] = x.reshape(-1)
    odd = flat[3:].view(5, 1024)
    assert odd.data_ptr() % 16
    assert torch.equal(cuda_fp8.matmul(odd, p), cuda_fp8.matmul(x, p))
    w = torch.zeros(p.weight.numel() + 8, dtype=torch.int8, device=DEV)
    w[8:] = p.weight.reshape(-1)
    t = qlinear.Tiled(w[8:].view(p.weight.shape), p.scale, p.rows, p.k, "w8a16")
    close(qlinear.linear_w8a16(x, t), cuda_fp8.matmul(x, p), False, "weight off the boundary")
    plan = qlinear.plan_resident(_lib.FMT_W8A16, 5, 256, 1024)
    with pytest.raises(ValueError):
        qlinear.run_resident(plan, _lib.FMT_W8A16, t.weight, t.scale, x, None, 5, 256, 1024)


def test_reference_format_planes_count():
    """cuda_fp8.splits names the planes matmul_partials returns, whichever kernel makes them; their
    sum is matmul's result."""
    for fmt in ("int8g64", "int4g64"):
        _, p = make(fmt, 2560, 9728, 6)
        for m in (1, 8, 33, 64):
            for config in ((4, 1), (8, 4)):
                x = acts(m, 9728, m)
                planes = cuda_fp8.matmul_partials(x, p, config)
                assert planes.shape[0] == cuda_fp8.splits(p, m, config), (fmt, m, config)
                acc = torch.zeros_like(planes[0])
                for plane in planes:
                    acc += plane
                assert torch.equal(acc.to(torch.bfloat16), cuda_fp8.matmul(x, p, config)), (fmt, m, config)


def test_graph_replays_equal_eager():
    _, p = make("int8g64", 2560, 4096, 4)
    x = acts(20, 4096, 1)
    eager = cuda_fp8.matmul(x, p)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = cuda_fp8.matmul(x, p)
    for seed in (1, 2, 3):
        x.copy_(acts(20, 4096, seed))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, cuda_fp8.matmul(x, p))
    assert eager.shape == out.shape


def test_calls_of_two_streams_count_apart():
    """K slices' tickets: a slot per stream, the same on the next call; overlapping calls' results are
    those of the calls one after the other."""
    fmt, m, n, k = "w8a16", 8, 2560, 9728
    ps = [make(fmt, n, k, seed)[1] for seed in (51, 52)]
    xs = [acts(m, k, seed) for seed in (53, 54)]
    want = [bits16(resident(fmt, x, p, 4)) for x, p in zip(xs, ps)]
    streams = [torch.cuda.Stream(DEV) for _ in range(2)]
    slots = [_lib.stream_tickets(torch.device(DEV), st.cuda_stream) for st in streams]
    assert abs(slots[0] - slots[1]) >= 4 * _lib.STREAM_TICKETS
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(8):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(resident(fmt, xs[i], ps[i], 4))
    torch.cuda.synchronize()
    assert slots == [_lib.stream_tickets(torch.device(DEV), st.cuda_stream) for st in streams]
    for i in range(2):
        for y in got[i]:
            assert (bits16(y) == want[i]).all()


def sliced(kernel, x, p):
    """A W8A16 call in K slices on one kernel."""
    if kernel == "resident":
        return resident("w8a16", x, p, 4)
    return qlinear.linear_w8a16(x, p.tiles, skinny=True) if kernel == "skinny" else \
        qlinear.linear_w8a16(x, p.tiles, config=(8, 8, 1, 4))


def captured(calls):
    """A graph of calls one after the other, on torch's own capture stream."""
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = [fn() for fn in calls]
    return graph, outs


@pytest.mark.parametrize("kernel", ["resident", "skinny", "decode"])
def test_replays_that_overlap_count_apart(kernel):
    """Graphs captured on one stream, replayed on two while the same calls run eagerly on a third: every
    result is that of the calls one after the other."""
    m, n, k = 8, 2560, 9728
    calls = [functools.partial(sliced, kernel, acts(m, k, seed + 3), make("w8a16", n, k, seed)[1]) for seed in (71, 72, 73)]
    want = [bits16(fn()) for fn in calls]
    graphs = [captured(calls) for _ in range(2)]
    streams = [torch.cuda.Stream(DEV) for _ in range(3)]
    for _ in range(4):
        for _, outs in graphs:
            for y in outs:
                y.zero_()
        torch.cuda.synchronize()
        eager = []
        for _ in range(4):
            for st, (graph, _) in zip(streams, graphs):
                with torch.cuda.stream(st):
                    graph.replay()
            with torch.cuda.stream(streams[2]):
                eager.append([fn() for fn in calls])
        torch.cuda.synchronize()
        for outs in [g[1] for g in graphs] + eager:
            for y, w in zip(outs, want):
                assert (bits16(y) == w).all()


def test_the_first_sliced_call_may_be_a_captured_one(monkeypatch):
    """Eager calls before the graph's first replay, and after it, find their own counters zeroed."""
    monkeypatch.setattr(_lib, "_stream_tickets", {})
    fmt, m, n, k = "w4a16", 4, 2560, 9728
    p, x = make(fmt, n, k, 81)[1], acts(m, k, 82)
    graph, (out,) = captured([lambda: resident(fmt, x, p, 3)])
    eager = bits16(resident(fmt, x, p, 3))
    close(resident(fmt, x, p, 3), decode(fmt, x, p, False), False, "eager before the replay")
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert (bits16(out) == eager).all() and (bits16(resident(fmt, x, p, 3)) == eager).all()
    assert all(int(buf.abs().sum()) == 0 for buf, _, _ in _lib._stream_tickets.values())


@pytest.mark.parametrize("fmt,k,splits", [("w4a16", 8448, 4), ("fp8", 3328, 6), ("int4g64", 8448, 4)])
def test_a_short_last_slice_of_one_token(fmt, k, splits):
    """A last K slice whose waves hold several units fewer than the others', the last of them at the end
    of the weight (one tile) and of the activation (one token)."""
    p = make(fmt, 16, k, 61)[1]
    x = acts(1, k, 62)
    close(resident(fmt, x, p, splits), decode(fmt, x, p, False), False, (fmt, k, splits))
