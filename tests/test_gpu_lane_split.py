"""Calls of few superblocks take other variants of a kernel than calls of many
(several lanes per group); their bytes are the same, and the oracle's."""

import numpy as np
import pytest
import torch

import oracle
from golden_data import clean_blocks, nonfinite_case
from test_gpu_parity import NAN_SIGN_TYPES, SQRT_CASES, dev, ffn_like, nan_sign_cleared, to_device  # noqa: F401

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


SPLIT_TYPES = ["q2_k", "q3_k", "q4_k", "q5_k", "iq4_xs", "iq3_xxs", "iq3_s"]
# a call between every two lines of the dispatch (besides one of the rows as they are)
TOTALS = [3000, 5000, 9000, 13000]


def in_every_variant(call, x, n_rows, k):
    """call(rows) for the rows as they are and repeated into calls of TOTALS
    superblocks: (repeats, bytes as repeats x rows x row bytes)."""
    for total in [n_rows * k // 256, *TOTALS]:
        n = -(-total * 256 // (n_rows * k))
        got = call(x.repeat(n, 1)).cpu().numpy()
        yield n, got.reshape(n, n_rows, -1)


def edge_runs(imat: bool):
    """(what, f32 rows, imatrix)"""
    rng = np.random.default_rng(41)
    k = 2560
    q = rng.lognormal(0, 1, k).astype(np.float32) if imat else None
    x = (rng.standard_normal((8, k)) * 0.02).astype(np.float32)
    xn, qn, _ = nonfinite_case()
    yield "non-finite values", xn, qn if imat else None
    big = x.copy()
    big[0:2, :32] = 0
    big[0:2, 5] = 3.0e38
    big[2:4, 288:300] = 0
    big[2:4, 300] = -2.9e38
    big[4:6, 600] = 2.0e36
    big[6:8, 1004] = 3.3e38
    yield "values near FLT_MAX", big, q
    sparse = x * (rng.random(x.shape) < 0.1)
    sparse[4:, ::512] = x[4:, ::512]
    yield "mostly zero values", np.concatenate([sparse, x[:3]]).astype(np.float32), q
    scale = np.repeat([1e-13, 3e-15, 1.2e-15, 8e-16], 2)[:, None]
    yield "tiny values", (rng.standard_normal((8, k)) * scale).astype(np.float32), q
    if not imat:
        return
    small = (rng.standard_normal((8, k)) * 3e-4).astype(np.float32)
    yield "tiny imatrix", small, q * np.float32(1e-30)
    yield "huge imatrix", small, q * np.float32(1e34)
    for val in (np.inf, np.nan, -0.0):
        w = q.copy()
        w[rng.choice(k, 6, replace=False)] = val
        w[1024:1056] = np.float32(-0.0) if val == 0 else w[1024:1056]
        yield f"{val} columns", x, w


@pytest.mark.parametrize("imat", [False, True])
@pytest.mark.parametrize("qtype", SPLIT_TYPES)
def test_edge_values_in_every_variant(qs, dev, qtype, imat):  # noqa: F811
    for what, x, qw in edge_runs(imat):
        print(f"{qtype} imat={imat} {what}", flush=True)
        fn = qs.QUANT_TYPES[qtype].make_kernel(dev, None if qw is None else torch.from_numpy(qw))
        ref = oracle.quantize(qtype, x, qw)
        nb = ref.shape[1] * 256 // x.shape[1]
        clean = clean_blocks(x, 256)
        want = ref.reshape(-1, nb)
        for n, got in in_every_variant(fn, to_device(x, dev), *x.shape):
            got = got.reshape(n, -1, nb)
            assert (got == got[:1]).all(), (what, n)
            same = (got[0] == want).all(1)
            if qtype not in NAN_SIGN_TYPES:
                assert same.all(), (what, n)
            elif what == "non-finite values":
                assert same[clean].all(), (what, n)
            else:
                assert np.array_equal(nan_sign_cleared(got[0], nb), nan_sign_cleared(want, nb)), (what, n)


@pytest.mark.parametrize("mode", ["torch-cpu", "ieee", "torch-cpu-amd"])
@pytest.mark.parametrize("qtype,imat", [c for c in SQRT_CASES if c[0] in SPLIT_TYPES])
def test_square_root_modes_in_every_variant(qs, dev, mode, qtype, imat):  # noqa: F811
    import sqrt_hosts
    x, qw = ffn_like(24, 2560, seed=5)
    qw = qw if imat else None
    if mode == "ieee":
        oracle.use_ieee_sqrt(True)
    elif mode == "torch-cpu-amd":
        oracle.use_amd_host_sqrt(sqrt_hosts.amd_ulps())
    try:
        qs.set_sqrt_rounding(mode)
        ref = oracle.quantize(qtype, x, qw)
        fn = qs.QUANT_TYPES[qtype].make_kernel(dev, None if qw is None else torch.from_numpy(qw))
        for n, got in in_every_variant(fn, to_device(x, dev), *x.shape):
            assert (got == ref).all(), n
    finally:
        qs.set_sqrt_rounding("torch-cpu")
        oracle.use_ieee_sqrt(False)
        oracle.use_sqrt_table(None)


@pytest.mark.parametrize("qtype", SPLIT_TYPES)
def test_row_stride_and_output_offset_in_every_variant(qs, dev, qtype):  # noqa: F811
    """Rows in a wider tensor, packed to an address off every word boundary."""
    rows, k = 20, 1024
    x, qw = ffn_like(rows, k, seed=12)
    q = torch.from_numpy(qw).to(dev)
    ref = oracle.quantize(qtype, x, qw)

    def call(xs):
        wide = torch.zeros((xs.shape[0], k + 64), dtype=xs.dtype, device=dev)
        wide[:, :k] = xs
        buf = torch.zeros(xs.shape[0] * ref.shape[1] + 3, dtype=torch.uint8, device=dev)
        qs.quantize(int(qs.QUANT_TYPES[qtype].ggml_type), wide[:, :k], q, out=buf[1:-2])
        assert int(buf[0]) == 0 and buf[-2:].tolist() == [0, 0]
        return buf[1:-2]

    for n, got in in_every_variant(call, to_device(x, dev), rows, k):
        assert (got == ref).all(), n


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
