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
