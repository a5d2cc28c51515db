"""The per-row kernels -- residual + RMSNorm with its quantized forms, the FP8 activation quantizer,
head norm + RoPE + cache write -- at the edges of their launch shapes: rows of one chunk, of a partial
wave, of one and two chunks per thread, odd head counts; and values the hardware's bf16 pair
conversion rounds differently (NaN). Bit-exact against the oracle; a NaN's bits are compared as the
integer rounding leaves them (0x7FC0 beside the sign)."""

import numpy as np
import pytest
import torch

import oracle.attention_oracle as A
import oracle.qlinear_oracle as O
from kernels import add_rms_norm, norm, qkv_norm_rope_to_cache, qlinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def bits16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def rand(*shape, seed, std=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).to(torch.bfloat16)


def same(got, want):
    """Equal bits, NaNs up to their sign (a NaN made by an operation has the hardware's sign)."""
    got, want = bits16(got), np.asarray(want, dtype=np.uint16)
    nan = (want & 0x7FFF) > 0x7F80
    assert np.array_equal(got & 0x7FFF, np.where(nan, 0x7FC0, want & 0x7FFF))
    assert np.array_equal(got[~nan], want[~nan])


@pytest.mark.parametrize("n", [8, 12, 504, 512, 2560, 8192, 8200, 16384])
@pytest.mark.parametrize("special", [False, True])
def test_add_rms_norm_widths(n, special):
    print("add_rms_norm", n, special, flush=True)
    x, d, w = rand(5, n, seed=n), rand(5, n, seed=n + 1), rand(n, seed=n + 2)
    if special:
        x[1, n // 2], x[2, 1], d[3, 0] = float("nan"), float("inf"), float("-inf")
    with np.errstate(invalid="ignore", over="ignore"):
        r0, y0 = O.add_rms_norm(bits16(x), bits16(d), bits16(w), 1e-6)
        y1 = O.rms_norm(bits16(x), bits16(w), 1e-6)
    r, y = add_rms_norm(x.to(DEV), d.to(DEV), w.to(DEV), 1e-6)
    same(r, r0)
    same(y, y0)
    same(norm.rms_norm(x.to(DEV), w.to(DEV), 1e-6), y1)
    planes = torch.randn(5, 5, n, generator=torch.Generator().manual_seed(3)).to(torch.float32)
    r0, y0 = O.add_rms_norm_partials(bits16(x[:5]), planes.numpy(), bits16(w), 1e-6)
    r, y = norm.add_rms_norm_partials(x.to(DEV), planes.to(DEV), w.to(DEV), 1e-6)
    same(r, r0)
    same(y, y0)


@pytest.mark.parametrize("n", [8, 72, 2560, 8192, 8200, 16384])
def test_add_norm_quant_fp8_widths(n):
    print("add_norm_quant_fp8", n, flush=True)
    x, d, w = rand(3, n, seed=n), rand(3, n, seed=n + 5), rand(n, seed=n + 6)
    r0, y0 = O.add_rms_norm(bits16(x), bits16(d), bits16(w), 1e-6)
    q0, s0 = O.quantize_fp8_activation(y0)
    r, q, s, y = qlinear.add_norm_quant_fp8(x.to(DEV), d.to(DEV), w.to(DEV), 1e-6, keep_normed=True)
    assert np.array_equal(bits16(r), r0) and np.array_equal(bits16(y), y0)
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), q0) and np.array_equal(s.cpu().numpy(), s0)


@pytest.mark.parametrize("k", [8, 520, 2560, 8192, 8200, 9728, 16384, 16392])
def test_quantize_fp8_activation_widths(k):
    print("quantize_fp8_activation", k, flush=True)
    x = rand(4, k, seed=k, std=3.0)
    x[1].zero_()
    x[2, k - 1] = 300.0
    q, s = qlinear.quantize_fp8_activation(x.to(DEV))
    q0, s0 = O.quantize_fp8_activation(bits16(x))
    assert np.array_equal(q.view(torch.uint8).cpu().numpy(), q0) and np.array_equal(s.cpu().numpy(), s0)


def int8_heads(bits):
    """Codes and scales of bf16 heads as the kernel forms them: a NaN counts in no maximum and takes the code
    -127, as does an infinity over the infinite scale it makes, under which finite values take 0."""
    y = O.bf16_to_f32(bits)
    amax = np.where(np.isnan(y), np.float32(0), np.abs(y)).max(-1)
    scale = (np.maximum(amax, np.float32(1e-12)) / np.float32(127)).astype(np.float32)
    with np.errstate(invalid="ignore"):
        code = np.floor((y / scale[..., None]).astype(np.float32) + np.float32(0.5))
    return np.where(np.isnan(code), -127, np.clip(code, -127, 127)).astype(np.int8), scale


@pytest.mark.parametrize("n_q,n_kv", [(1, 1), (5, 3), (32, 8), (3, 0), (40, 10)])
@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("special", [False, True])
def test_rope_head_counts(n_q, n_kv, int8, special):
    """Heads share 16-lane groups and waves across the Q / K / V boundaries; a head of zeros; value and key
    heads with a NaN and with infinities, whose INT8 codes the oracle leaves open (int8_heads)."""
    print("rope", n_q, n_kv, int8, special, flush=True)
    rows, cap, pos = 3, 20, 17
    qkv = rand(rows, (n_q + 2 * n_kv) * 128, seed=n_q)
    qkv[0, :128] = 0
    if special:
        qkv[1, 3] = float("nan")
        qkv[1, -5] = float("nan")
        qkv[2, -9], qkv[2, -77] = float("inf"), float("-inf")
        if n_kv:
            qkv[0, n_q * 128 + 7] = float("inf")
            qkv[1, n_q * 128 + 70] = float("nan")
    qn, kn = rand(128, seed=1), rand(128, seed=2)
    ang = torch.randn(cap, 128, generator=torch.Generator().manual_seed(9))
    cos, sin = ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16)
    kv = max(n_kv, 1)
    kc = np.zeros((rows, kv, cap, 128), np.int8 if int8 else np.uint16)
    vc, ks, vs = kc.copy(), np.zeros((rows, kv, cap), np.float32), np.zeros((rows, kv, cap), np.float32)
    kw, vw = (np.zeros((rows, kv, 1, 128), np.uint16) for _ in range(2))
    with np.errstate(invalid="ignore", over="ignore"):
        q0 = A.qkv_norm_rope_to_cache(bits16(qkv), n_q, n_kv, bits16(qn), bits16(kn), bits16(cos), bits16(sin), [pos], 1, kc,
                                      vc, 1e-6, *((ks, vs) if int8 else (None, None)), kw, vw)
    if n_kv == 0:
        from kernels import q_norm_rope
        got = q_norm_rope(qkv.to(DEV), n_q, qn.to(DEV), cos.to(DEV), sin.to(DEV),
                          torch.tensor([pos], dtype=torch.int32, device=DEV), 1, 1e-6)
        return same(got, q0)
    dt = torch.int8 if int8 else torch.bfloat16
    kd, vd = (torch.zeros(rows, n_kv, cap, 128, dtype=dt, device=DEV) for _ in range(2))
    ksd, vsd = ((torch.zeros(rows, n_kv, cap, device=DEV) for _ in range(2)) if int8 else (None, None))
    got = qkv_norm_rope_to_cache(qkv.to(DEV), n_q, n_kv, qn.to(DEV), kn.to(DEV), cos.to(DEV), sin.to(DEV),
                                 torch.tensor([pos], dtype=torch.int32, device=DEV), 1, kd, vd, 1e-6, ksd, vsd)
    same(got, q0)
    if int8:
        for codes, scales, cache, factors, heads in ((kd, ksd, kc, ks, kw), (vd, vsd, vc, vs, vw)):
            want, factor = int8_heads(heads[:, :, 0])
            ok = ((heads[:, :, 0] & 0x7FFF) < 0x7F80).all(-1)
            assert ok.all() != special
            assert np.array_equal(want[ok], cache[:, :, pos][ok]) and np.array_equal(factor[ok], factors[..., pos][ok])
            assert np.array_equal(codes.cpu().numpy()[:, :, pos], want) and np.array_equal(scales.cpu().numpy()[..., pos], factor)
            assert not codes.cpu().numpy()[:, :, :pos].any() and not codes.cpu().numpy()[:, :, pos + 1:].any()
    else:
        same(kd, kc)
        same(vd, vc)
