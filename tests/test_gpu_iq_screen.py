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
