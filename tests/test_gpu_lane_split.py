"""Calls of few superblocks take other variants of a kernel than calls of many
(several lanes per group); their bytes are the same, and the oracle's."""

import numpy as np
import pytest
import torch

import oracle
from test_gpu_parity import dev  # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu

# superblocks per call on both sides of every line of the dispatch, and one
# superblock, and counts that leave a wave partly empty
COUNTS = [1, 3, 255, 2048, 2049, 4096, 4097, 6144, 6145, 12288]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("imat", [False, True])
@pytest.mark.parametrize("qtype", ["q2_k", "q3_k", "q4_k", "q5_k", "iq4_xs"])
def test_variants_agree_over_the_dispatch(qs, dev, qtype, imat, dtype):  # noqa: F811
    gen = torch.Generator(device="cuda").manual_seed(17)
    rows = 12300
    x = torch.randn(rows, 256, generator=gen, device=dev) * 0.02
    x *= torch.exp(torch.randn(rows, 1, generator=gen, device=dev))
    x[5] = 0
    x[6] = 0.125
    x[7, :128] = 0
    x[8, 32:48] = x[8, 32]
    x[9] = x[9].abs()
    x[10:12] *= 1e-13
    x[12:14] *= 1e13 if dtype == torch.float32 else 1e4
    x[14, 100] = 3.0
    x = x.to(dtype)
    qw = torch.exp(torch.randn(256, generator=gen, device=dev)) if imat else None
    if imat:
        qw[::7] = 0
    fn = qs.QUANT_TYPES[qtype].make_kernel(dev, qw)
    whole = fn(x).cpu()
    ref = oracle.quantize(qtype, x[:600].float().cpu().numpy(), None if qw is None else qw.cpu().numpy())
    assert np.array_equal(whole[:600].numpy(), ref)
    for n in COUNTS:
        assert torch.equal(fn(x[:n]).cpu(), whole[:n]), n
        assert torch.equal(fn(x[rows - n:]).cpu(), whole[rows - n:]), n


@pytest.mark.parametrize("imat", [False, True])
@pytest.mark.parametrize("qtype", ["iq3_xxs", "iq3_s"])
def test_iq3_agrees_over_its_line(qs, dev, qtype, imat):  # noqa: F811
    """Few superblocks take the exact search alone: both sides of the line."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = (torch.randn(4200, 256, generator=gen, device=dev) * 0.02).to(torch.bfloat16)
    x[3] = 0
    x[4, 64:96] = x[4, 64]
    qw = torch.exp(torch.randn(256, generator=gen, device=dev)) if imat else None
    fn = qs.QUANT_TYPES[qtype].make_kernel(dev, qw)
    whole = fn(x).cpu()
    ref = oracle.quantize(qtype, x[:400].float().cpu().numpy(), None if qw is None else qw.cpu().numpy())
    assert np.array_equal(whole[:400].numpy(), ref)
    for n in (1, 3, 4095, 4096, 4097):
        assert torch.equal(fn(x[:n]).cpu(), whole[:n]), n
