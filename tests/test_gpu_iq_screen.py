"""The IQ searches decide most lists from fused scores and send the close ones to
the reference's arithmetic: inputs whose scores lie close together, at every
spread of the weights, against the oracle."""

import numpy as np
import pytest
import torch

import oracle
from test_gpu_parity import dev  # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spread", [0.0, 1.0, 8.0])
@pytest.mark.parametrize("qtype", ["iq2_xxs", "iq2_xs", "iq2_s", "iq3_xxs", "iq3_s"])
def test_close_scores(qs, dev, qtype, spread):  # noqa: F811
    rng = np.random.default_rng(5)
    x = rng.standard_normal((48, 1024)).astype(np.float32) * np.float32(0.02)
    x[0:12] = np.sign(x[0:12]) * np.float32(0.02)              # one magnitude: ties up to rounding
    x[12:24] *= np.float32(1) + np.float32(2e-7) * rng.integers(0, 3, (12, 1024)).astype(np.float32)
    x[24:32] = np.round(x[24:32] * 100) / 100                  # few levels
    x[32:36] *= np.exp2(rng.integers(-30, 30, (4, 1024))).astype(np.float32)
    qw = np.exp(spread * rng.standard_normal(1024)).astype(np.float32)
    qw[5::16] = 0
    qw[512:544] = 0
    fn = qs.QUANT_TYPES[qtype].make_kernel(dev, torch.from_numpy(qw))
    got = fn(torch.from_numpy(x).to(dev)).cpu().numpy()
    assert np.array_equal(got, oracle.quantize(qtype, x, qw))


def _weights_case(case: str, rng, k: int) -> np.ndarray | None:
    qw = np.exp(rng.standard_normal(k)).astype(np.float32)
    if case == "none":
        return None
    if case == "constant":
        qw[:] = 1
    elif case == "tiny":
        # one weight per 8 values at 2^-12 .. 2^-22 of the others' (the distance
        # weights are roots of these): entries that differ in its value only lie
        # 2^-9 .. 2^-24 of sc^2 W apart: 1-3% of the lists within a factor of 8 of the
        # screen's 2^-18 on either side, none of the ordinary ones
        at = np.arange(0, k, 8) + rng.integers(0, 8, k // 8)
        qw[at] *= np.exp2(-2.0 * rng.uniform(12, 22, k // 8)).astype(np.float32)
    elif case == "zero-superblocks":
        qw[: k // 4][rng.random(k // 4) < 0.1] = 0             # a quarter of each row's superblocks
    elif case == "zero-column":
        qw[k // 2 + 37] = 0
    return qw


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("qtype,case", [
    (t, c) for t in ["iq2_xxs", "iq2_xs", "iq2_s", "iq3_xxs", "iq3_s"]
    for c in ["positive", "tiny", "zero-superblocks", "zero-column", "constant"] + ["none"] * t.startswith("iq3")])
def test_screened_and_exact_waves(qs, dev, qtype, case, dtype):  # noqa: F811
    """Waves that screen every list, waves that search every list exactly (ties
    known before the sweep) and both in one launch; a launch of few superblocks
    and, of the same rows, one of many."""
    rng = np.random.default_rng(11)
    rows, k = 9, 8192
    x = torch.from_numpy(rng.standard_normal((rows, k)).astype(np.float32) * np.float32(0.02))
    x[7:] = torch.round(x[7:] * 200) / 200                     # few levels: equal values, exact midpoints
    x = x.to(dtype)
    qw = _weights_case(case, rng, k)
    ref = oracle.quantize(qtype, x.float().numpy(), qw)
    fn = qs.QUANT_TYPES[qtype].make_kernel(dev, None if qw is None else torch.from_numpy(qw))
    assert np.array_equal(fn(x.to(dev)).cpu().numpy(), ref)
    many = 24                                                  # 6,912 superblocks
    got = fn(x.to(dev).repeat(many, 1)).cpu().numpy().reshape(many, *ref.shape)
    assert (got == ref).all()
