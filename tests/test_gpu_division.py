"""The divisions and square roots the kernels build from one approximate
instruction (qs_device.h: recip, quotient, sqrt_root): the property their proof needs over every mantissa, and the formats
against the oracle where a wave's divisions lie on both sides of the range in
which they are used."""

import ctypes

import numpy as np
import pytest
import torch

import oracle
from test_gpu_parity import dev  # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e", [-60, -36, -1, 0, 1, 36, 60])
def test_reciprocal_and_quotient_over_every_mantissa(qs, dev, e):  # noqa: F811
    lib = ctypes.CDLL(str(qs.LIB_PATH.parent / "libqs_calib.so"))
    lib.qs_calib_recip.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    out = torch.zeros(2, dtype=torch.int32, device=dev)
    assert lib.qs_calib_recip(e, out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    worst = out.cpu().numpy()[:1].view(np.float32)[0]
    # |1 - b recip(b)| < 2^-23 / m with 2^-18 to spare (the last 64 mantissas
    # apart, whose quotients are all compared)
    assert 0 < worst < 1 - 2.0**-18
    assert int(out[1]) == 0


@pytest.mark.parametrize("k", [-48, -40, -1, 0, 1, 50, 53])
def test_root_of_every_mantissa(qs, dev, k):  # noqa: F811
    lib = ctypes.CDLL(str(qs.LIB_PATH.parent / "libqs_calib.so"))
    lib.qs_calib_sqrt.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    out = torch.zeros(1, dtype=torch.int32, device=dev)
    assert lib.qs_calib_sqrt(k, out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    assert int(out[0]) == 0


@pytest.mark.parametrize("imat", [False, True])
@pytest.mark.parametrize("qtype", ["q2_k", "q3_k", "q4_k", "q5_k", "q6_k", "iq4_xs", "iq4_nl"])
def test_scales_across_the_division_range(qs, dev, qtype, imat):  # noqa: F811
    """Rows scaled by 2^-45 .. 2^45 and imatrix columns by 2^-70 .. 2^70, so
    that scales, mins and weighted sums fall inside and outside the range, in
    the same wave too; zero and constant blocks among them."""
    rng = np.random.default_rng(31)
    x = rng.standard_normal((46, 1024)).astype(np.float32)
    x *= np.exp2(np.arange(-45, 47, 2, dtype=np.float32))[:, None]
    x[3, 256:512] = 0
    x[5, :256] = x[5, 0]
    x[7:20, 512:] *= np.exp2(rng.integers(-40, 40, (13, 1)).astype(np.float32))
    x = x.astype(np.float32)
    xb = torch.from_numpy(x).to(torch.bfloat16).float().numpy()
    qw = None
    if imat:
        qw = (rng.lognormal(0, 1, 1024) * np.repeat(np.exp2(np.linspace(-70, 70, 32)), 32)).astype(np.float32)
    fn = qs.QUANT_TYPES[qtype].make_kernel(dev, None if qw is None else torch.from_numpy(qw))
    got = fn(torch.from_numpy(xb).to(dev)).cpu().numpy()
    assert np.array_equal(got, oracle.quantize(qtype, xb, qw))


def four_squares(n: int) -> list[int]:
    for a in range(int(n**0.5), 0, -1):
        for b in range(int((n - a * a) ** 0.5), -1, -1):
            r = n - a * a - b * b
            for c in range(int(r**0.5), -1, -1):
                d = int((r - c * c) ** 0.5)
                if a * a + b * b + c * c + d * d == n:
                    return [a, b, c, d]
    raise ValueError(n)


@pytest.mark.parametrize("n", [1, 2100, 4200])
def test_minimum_that_overflows(qs, dev, n):  # noqa: F811
    """A candidate whose minimum is +inf (sum_l2 sum_x overflows: weights of
    both signs that cancel in sum_w and sum_l, so D and the scale stay small) is
    fitted again with a minimum of 0 (kq_common.py:77-80) and can be accepted."""
    groups = [
        ([2.0, 0.5625, 1.46875, 1.140625, 1.796875, 0.890625, 0.8125, 0.609375, 0.46875, 1.296875], [1, -2, -2, 2, -2]),
        ([2.0, 0.09375, 0.53125, 0.125, 0.078125, 1.109375, 0.375, 0.15625, 1.828125, 0.296875], [2, -4, -2, 1, -2]),
        ([2.0, 0.125, 1.203125, 0.296875, 0.109375, 1.65625, 0.796875, 1.734375, 1.484375, 0.40625], [-1, -2, -1, -1, 4]),
    ]
    rng = np.random.default_rng(2)
    for values, signs in groups:
        # multiples of 2^7 elsewhere whose squares sum to 2^36: every root is 2^14 and
        # the group's weights are exact (and no other group of the wave is out of range)
        m = np.rint(rng.standard_normal(240) * 110).astype(np.int64)
        rest = 2**22 - int((m[:236] ** 2).sum())
        m[236:] = four_squares(rest)
        x = np.zeros((1, 256), np.float32)
        x[0, 16:] = m * 128
        x[0, :10] = values
        qw = np.full(256, 2.0**-14, np.float32)
        qw[:16] = 0
        qw[0:10:2] = np.asarray(signs) * 2.0**52
        qw[1:11:2] = -np.asarray(signs) * 2.0**52
        qw[10] = 2.0**-54
        fn = qs.QUANT_TYPES["q2_k"].make_kernel(dev, torch.from_numpy(qw))
        got = fn(torch.from_numpy(x).to(dev).repeat(n, 1)).cpu().numpy()
        assert (got == oracle.quantize("q2_k", x, qw)).all()
