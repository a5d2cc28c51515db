"""Quantize and relayout kernels at the edges of their launch shapes: group lengths that take each
of the lane-segment, row-block and wave kernels, partial last blocks, special values. Bit-exact
against the oracle. The quotient that the integer quantizer computes from a reciprocal is compared
with IEEE division on the CPU, over every pair of mantissas it can see."""

from fractions import Fraction

import numpy as np
import pytest
import torch

import oracle.qlinear_oracle as O
from kernels import _lib

DEV = "cuda:0"


def bits16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def weight(n, k, seed):
    g = torch.Generator().manual_seed(seed)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16)
    w[0].zero_()
    w[1] = (torch.randn(k, generator=g) * 1e-9).to(torch.bfloat16)   # the fp16 scale underflows to 0
    w[2] = (torch.randn(k, generator=g) * 1e30).to(torch.bfloat16)   # the fp16 scale overflows
    w[3] = (torch.randint(-14, 15, (k,), generator=g) / 2).to(torch.bfloat16)  # codes on half-integers
    w[4, ::7] = float("nan")
    return w


@pytest.mark.gpu
@pytest.mark.parametrize("k,group", [(24, 8), (120, 40), (192, 64), (576, 72), (384, 128), (400, 200), (1024, 512),
                                     (1040, 520), (1024, 1024), (1032, 1032), (4096, 2048), (2056, 2056), (4096, 4096), (4104, 4104), (16384, 16384), (16392, 16392)])
@pytest.mark.parametrize("bits,scale,storage", [(8, "f16", "offset"), (8, "bf16", "signed"), (4, "f16", "offset"),
                                                (4, "bf16", "k32")])
def test_quantize_group_lengths(k, group, bits, scale, storage):
    print("quantize", k, group, bits, scale, storage, flush=True)
    n = 37
    w = weight(n, k, k + bits)
    code = "codes" if storage == "k32" else storage
    oq, os_, _ = O.quantize(np.where(np.isnan(w.float().numpy()), 0, bits16(w)).astype(np.uint16), group=group, bits=bits,
                            scale_dtype=scale, storage=code)
    oq = oq.copy()
    # a NaN never takes part in the maximum; its own code is 0 (the oracle runs without it)
    oq[np.isnan(w.float().numpy())] = 0
    if storage == "k32":
        oq = O.pack_int4_k32(oq)
    dt = torch.int32 if storage == "k32" else (torch.int8 if storage == "signed" else torch.uint8)
    q = torch.empty(n, k // 8 if storage == "k32" else k, dtype=dt, device=DEV)
    s = torch.empty(n, k // group, dtype=torch.bfloat16, device=DEV)
    wd = w.to(DEV)
    _lib.call("qlx_quantize_weight", _lib.ptr(wd), _lib.ptr(q), _lib.ptr(s), n, k, group, bits,
              _lib.SCALE_F16 if scale == "f16" else _lib.SCALE_BF16, 1,
              {"offset": _lib.STORE_OFFSET, "signed": _lib.STORE_SIGNED, "k32": _lib.STORE_K32}[storage],
              _lib.stream(wd.device))
    assert np.array_equal(bits16(s), os_.reshape(n, -1))
    assert np.array_equal(q.cpu().numpy(), oq)


@pytest.mark.gpu
@pytest.mark.parametrize("k,group", [(48, 8), (384, 128), (1040, 520), (2048, 1024), (1032, 1032), (2048, 2048), (2056, 2056),
                                     (9728, 9728), (16392, 16392)])
def test_quantize_fp8_group_lengths(k, group):
    print("quantize fp8", k, group, flush=True)
    w = weight(19, k, k)
    w[4].zero_()
    oq, os_ = O.fp8_quantize(bits16(w), group=group)
    wd = w.to(DEV)
    q = torch.empty(19, k, dtype=torch.uint8, device=DEV)
    s = torch.empty(19, k // group, dtype=torch.bfloat16, device=DEV)
    _lib.call("qlx_quantize_fp8_weight", _lib.ptr(wd), _lib.ptr(q), _lib.ptr(s), 19, k, group, _lib.stream(wd.device))
    assert np.array_equal(q.cpu().numpy(), oq) and np.array_equal(bits16(s), np.asarray(os_).reshape(19, -1))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", [(16, 128), (48, 384), (4112, 128)])
@pytest.mark.parametrize("bits,tiled", [(8, True), (8, False), (4, True)])
@pytest.mark.parametrize("skip", [0, 3])  # the source may start at any byte of a larger buffer
def test_prepare_reference_layouts(rows, k, bits, tiled, skip):
    print("prepare", rows, k, bits, tiled, skip, flush=True)
    rng = np.random.default_rng(rows + k)
    src = rng.integers(0, 256 if bits == 8 else 16, (rows, k), dtype=np.uint8)
    want = O.prepare_weight(src, bits=bits, tiled=tiled)
    flat = torch.zeros(rows * k + skip, dtype=torch.uint8)
    flat[skip:] = torch.from_numpy(src.reshape(-1))
    flat = flat.to(DEV)
    out = torch.empty(rows * (k // 2 if bits == 4 else k), dtype=torch.uint8, device=DEV)
    _lib.call("qlx_prepare_ref", _lib.ptr(flat[skip:]), _lib.ptr(out), rows, k, bits, int(tiled), _lib.stream(out.device))
    assert np.array_equal(out.cpu().numpy(), np.asarray(want).reshape(-1))


def test_quotient_by_reciprocal_rounds_as_division():
    """q0 = x y, r = fma(-q0, s, x), q = fma(r, y, q0) with y = 1 / s rounded, for every bf16 mantissa
    of x and every fp16 (so also every bf16 of 8 bits) mantissa of s: the IEEE quotient. Exponents
    only shift the result. (The doubles below hold every step but the last exactly; where its
    second rounding could matter, it is redone in whole numbers.)"""
    x = np.arange(128, 256, dtype=np.float64)[:, None]
    for mant in (np.arange(1024, 2048, dtype=np.float64)[None, :], np.arange(128, 256, dtype=np.float64)[None, :]):
        for xs in (x, 2 * x):  # quotients either side of 1
            s32, x32 = mant.astype(np.float32), xs.astype(np.float32)
            y = (np.float32(1) / s32).astype(np.float64)
            q0 = (xs * y).astype(np.float32).astype(np.float64)
            r = (xs - q0 * mant).astype(np.float32).astype(np.float64)
            assert np.array_equal(r, xs - q0 * mant), "the residual is exact"
            got = (r * y + q0).astype(np.float32)
            want = x32 / s32
            for i, j in np.argwhere(got != want):
                exact = Fraction(float(r[i, j])) * Fraction(float(y[0, j])) + Fraction(float(q0[i, j]))
                w = Fraction(float(want[i, j]))
                ulp = Fraction(float(np.spacing(want[i, j])))
                assert abs(exact - w) < ulp / 2, (i, j)
