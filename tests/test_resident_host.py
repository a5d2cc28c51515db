"""The host side of the resident-activation GEMM (qlx_linear_resident): its plan on both sides of the
kernel's size limits. Nothing here reaches a GPU."""

import ctypes

import pytest

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
