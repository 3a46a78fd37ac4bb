"""GPU parity of the fp8 W8A8 path (row quantization, weight prepack, MFMA
GEMM) against the CPU oracle; tolerance rel-err <= 2e-2 as the north star
states for fp8 (the oracle accumulates the decoded products in f64)."""
import numpy as np
import pytest
import torch

import oracle
from conftest import rel_err
from ubridge_amd import fp8, ops

pytestmark = pytest.mark.gpu


def test_quantize_rows_bit_exact(dev):
    x = torch.randn(37, 1000, generator=torch.Generator().manual_seed(1))
    x[3] = 0.0
    x[5, 7] = 1e-9
    q, s = fp8.quantize_rows(x.to(dev))
    oq, os_ = oracle.fp8_quantize_rows(x.numpy())
    assert np.array_equal(s.cpu().numpy(), os_)
    assert np.array_equal(q.cpu().numpy(), oq)
    # bf16 input
    xb = x.bfloat16()
    q2, s2 = fp8.quantize_rows(xb.to(dev))
    oq2, os2 = oracle.fp8_quantize_rows(xb.float().numpy())
    assert np.array_equal(q2.cpu().numpy(), oq2) and np.array_equal(s2.cpu().numpy(), os2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("R,C", [(1, 8), (3, 72), (5, 2048), (600, 2056), (2, 16384), (3, 28672),
                                 (2, 65544)])
def test_quantize_rows_units(dev, dtype, R, C):
    # rows of whole 16-byte units (the one-workgroup-per-row form: 1..8 units
    # per thread, partly filled, and longer than it takes) against the oracle:
    # zeros of both signs, infinities, NaN, midpoints between two codes, scales
    # where the row divides
    g = torch.Generator().manual_seed(R + C)
    x = torch.randn(R, C, generator=g) * torch.exp(2 * torch.randn(R, 1, generator=g))
    x[0, :8] = torch.tensor([0.0, -0.0, 17.0, -19.0, 2.0**-10, 3 * 2.0**-10, 448.0, -232.0])
    if R > 1:
        x[1] *= 1e-30
        x[R - 1, C - 1] = float("inf")
    x = x.to(dtype)
    q, s = fp8.quantize_rows(x.to(dev))
    want_q, want_s = oracle.fp8_quantize_rows(x.float().numpy())
    q, s = q.cpu().numpy(), s.cpu().numpy()
    assert np.array_equal(s, want_s)
    nan = (want_q & 0x7F) == 0x7F  # inf / inf: NaN, its sign is not fixed
    assert np.array_equal(q[~nan], want_q[~nan]) and np.all((q[nan] & 0x7F) == 0x7F)


@pytest.mark.parametrize("R,C", [(1023, 504), (1024, 504), (1024, 512), (4099, 128), (1025, 8)])
def test_quantize_rows_narrow(dev, R, C):
    # both sides of the rule for narrow rows (512 values, 1024 rows)
    x = torch.randn(R, C, generator=torch.Generator().manual_seed(R + C))
    x[R // 2] = 0.0
    for t in (torch.float32, torch.bfloat16):
        q, s = fp8.quantize_rows(x.to(t).to(dev))
        want_q, want_s = oracle.fp8_quantize_rows(x.to(t).float().numpy())
        assert np.array_equal(s.cpu().numpy(), want_s) and np.array_equal(q.cpu().numpy(), want_q)


@pytest.mark.parametrize("C", [8, 512])
def test_quantize_rows_many(dev, C):
    # more rows than a launch has workgroups of 256 threads (2^32 threads); the
    # rows with values against the oracle, zero rows: code 0, scale 1
    R = (1 << 24) + 5
    x = torch.zeros(R, C, dtype=torch.bfloat16, device=dev)
    rows = torch.tensor([0, 1, R // 2, (1 << 24) - 1, 1 << 24, R - 1], device=dev)
    v = torch.randn(rows.numel(), C, generator=torch.Generator().manual_seed(C)).bfloat16()
    x[rows] = v.to(dev)
    q, s = fp8.quantize_rows(x)
    want_q, want_s = oracle.fp8_quantize_rows(v.float().numpy())
    assert np.array_equal(q[rows].cpu().numpy(), want_q) and np.array_equal(s[rows].cpu().numpy(), want_s)
    rest = torch.ones(R, dtype=torch.bool, device=dev)
    rest[rows] = False
    assert bool((s[rest] == 1.0).all())
    q[rows] = 0
    assert not bool(q.any())


def test_prepack_transpose(dev):
    w = torch.randint(0, 256, (200, 72), dtype=torch.uint8, device=dev)
    assert torch.equal(fp8.prepack_weight(w), w.T.contiguous())


@pytest.fixture(params=[0, 1, 3, 2, 4],
                ids=["default", "hipblaslt", "own_bk128", "4_waves", "8_waves_bk64"])
def fp8_variant(request):
    # gemm_tile knob: 0 the default (up to 16 tokens the decode kernel, for K a
    # multiple of 128 up to 8192; else hipBLASLt's fp8 GEMM with row / column
    # scale vectors where it serves the shape, else the kernel of 3), 1 that
    # without the decode kernel, 3 the library's own kernel (128-byte K-steps
    # when K % 128 == 0, else 64-byte ones), 2 its 4-wavefront kernel, 4 the
    # 8-wavefront 64-byte one
    ops.tune_set("gemm_tile", request.param)
    yield request.param
    ops.tune_set("gemm_tile", 0)


@pytest.mark.parametrize("M,K,N", [(64, 256, 128), (130, 512, 200), (1, 128, 40), (257, 384, 384),
                                   (300, 64, 520), (40, 1216, 264)])
def test_fp8_gemm_vs_oracle(dev, fp8_variant, M, K, N):
    g = torch.Generator().manual_seed(M + K + N)
    a = torch.randn(M, K, generator=g)
    w = torch.randn(K, N, generator=g)
    aq, sa = oracle.fp8_quantize_rows(a.numpy())
    wq_t, sw = oracle.fp8_quantize_rows(w.numpy().T.copy())  # per output channel n
    wq = np.ascontiguousarray(wq_t.T)  # [K, N] as the config stores it
    w_nk = fp8.prepack_weight(torch.from_numpy(wq).to(dev))
    out = fp8.gemm(torch.from_numpy(aq).to(dev), torch.from_numpy(sa).to(dev), w_nk,
                   torch.from_numpy(sw).to(dev))
    want = oracle.fp8_gemm(aq, sa, wq, sw, M, K, N, nthreads=8)
    got = out.float().cpu().numpy()
    assert rel_err(got, oracle.bf16_to_f32(want)) < 2e-2
    # and against the unquantized product: fp8 quantization error is bounded
    assert rel_err(got, a.double().numpy() @ w.double().numpy()) < 8e-2


@pytest.mark.parametrize("K,N", [(128, 8), (384, 40), (1024, 16400), (1152, 520), (1920, 8200),
                                 (1152, 16400), (2048, 28688), (2176, 4099), (4096, 16400), (4224, 300),
                                 (8192, 4136)])
@pytest.mark.parametrize("M", [1, 7, 16])
def test_fp8_decode(dev, M, K, N):
    # up to 16 tokens: every step count / tile width of the decode kernel, K
    # with idle wavefronts, ragged N, more than one tile per workgroup
    _few_tokens(dev, M, K, N)


@pytest.mark.parametrize("knob,M,K,N", [(0, 16, 8320, 200), (0, 3, 14336, 264), (0, 5, 192, 72),
                                        (0, 16, 1088, 520), (1, 1, 128, 40), (1, 16, 4096, 264)])
def test_fp8_few_tokens_gemm(dev, knob, M, K, N):
    # up to 16 tokens outside the decode kernel's contract (K > 8192, K % 128)
    # or with the knob that leaves it out: the GEMM
    ops.tune_set("gemm_tile", knob)
    try:
        _few_tokens(dev, M, K, N)
    finally:
        ops.tune_set("gemm_tile", 0)


def _few_tokens(dev, M, K, N):
    g = torch.Generator(device=dev).manual_seed(M + K + N)
    aq, sa = fp8.quantize_rows(torch.randn(M, K, device=dev, generator=g))
    wq, sw = fp8.quantize_rows(torch.randn(N, K, device=dev, generator=g))
    guard = torch.full((M + 1, N), 3.0, device=dev, dtype=torch.bfloat16)
    out = fp8.gemm(aq, sa, wq, sw, out=guard[:M])
    dec = lambda q: q.view(torch.float8_e4m3fn).double()
    want = (dec(aq) * sa.double()[:, None]) @ (dec(wq) * sw.double()[:, None]).T.contiguous()
    # every output: one bf16 rounding (2^-9) of a sum whose f32 error is far below it
    err = (out.double() - want).abs()
    rms = want.square().mean().sqrt()
    assert bool((err <= 2.0**-8 * want.abs() + 1e-4 * rms).all()), (err / rms).max()
    assert bool((guard[M] == 3.0).all())


@pytest.mark.parametrize("M", [256, 4096])
def test_fp8_cfg5(dev, fp8_variant, M):
    # configs[4] shapes K=8192, N=28672; M = 4096 is the full config (16 row
    # tiles, so the XCD-grouped tile order is exercised), checked against the
    # f64 product of the decoded operands, globally and per 256-row band
    K, N = 8192, 28672
    gen = torch.Generator(device=dev).manual_seed(5)
    a = torch.randn(M, K, device=dev, generator=gen)
    w = torch.randn(K, N, device=dev, generator=gen)
    aq, sa = fp8.quantize_rows(a)
    wq_nk, sw = fp8.quantize_rows(w.T.contiguous())
    out = fp8.gemm(aq, sa, wq_nk, sw)
    dec = lambda q: q.view(torch.float8_e4m3fn).double()
    want = (dec(aq) * sa.double()[:, None]) @ (dec(wq_nk) * sw.double()[:, None]).T
    err = (torch.linalg.norm(out.double() - want) / torch.linalg.norm(want)).item()
    assert err < 2e-2, err
    band = [(torch.linalg.norm(out[i:i + 256].double() - want[i:i + 256]) /
             torch.linalg.norm(want[i:i + 256])).item() for i in range(0, M, 256)]
    assert max(band) < 2e-2, band
