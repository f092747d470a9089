"""Pointwise products (few rows, short K, thousands of unit-stride columns): one
and two blocks of rows, every K step count with ragged ends, column counts
around a wavefront's share, padded and unaligned rows, beta, both biases and
GELU with its pre-activation.  Against float64 products of the bf16-rounded
operands: FP32 accumulation over at most 64 terms, 64 * 2^-24 of sum |a b| plus
2^-23 of the other terms; GELU has slope below 1.13 and its tanh 2^-20."""
import numpy as np
import pytest

import namsa_amd._lib as L
from oracle import fno_oracle as F
from tests.test_gpu_corrector_kernels import bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,pad,off,beta,bias,gelu", [
    (1, 8192, 1, 0, 0, 0.0, 0, False), (32, 8193, 16, 0, 1, 0.0, 1, False), (33, 8200, 7, 3, 0, 1.0, 1, True),
    (64, 8255, 17, 1, 2, 0.5, 2, False), (2, 9000, 64, 0, 0, 0.0, 1, False), (32, 10007, 32, 2, 3, 1.0, 0, False),
    (64, 8192, 32, 0, 0, 0.0, 1, True), (31, 8449, 33, 5, 1, 0.0, 0, True), (64, 12288, 64, 0, 0, 2.0, 2, True)])
def test_pointwise_products(gpu, M, N, K, pad, off, beta, bias, gelu):
    import torch

    print(f"pointwise gemm M={M} N={N} K={K} pad={pad} off={off} beta={beta} bias={bias} gelu={gelu}", flush=True)
    rng = np.random.default_rng(N + K)
    s = N + pad
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal(off + K * s).astype(np.float32)
    C0 = rng.standard_normal(off + M * s).astype(np.float32)
    bv = rng.standard_normal(N if bias == 2 else M).astype(np.float32)
    Ad, Bd, Cd, bd = (torch.from_numpy(x.copy()).to(gpu) for x in (A, B, C0, bv))
    Pd = torch.zeros_like(Cd)
    L.call("namsa_gemm_bf16", L.ptr(Ad), 0, K, 1, L.ptr(Bd[off:]), 0, s, 1, L.ptr(Cd[off:]), 0, s, 1, M, N, K, 1, 1,
           np.float32(0.25), np.float32(beta), L.ptr(bd) if bias else None, bias, int(gelu), L.ptr(Pd[off:]) if gelu else None,
           L.stream_handle())
    rows = lambda x, n: x[off:off + n * s].reshape(n, s)   # noqa: E731
    a, b, c0 = bf16(A), bf16(rows(B, K)[:, :N]), rows(C0, M)[:, :N].astype(np.float64)
    add = beta * c0 + (bv[:, None] if bias == 1 else bv[None, :] if bias == 2 else 0.0)
    pre = 0.25 * (a @ b) + add
    bound = 64 * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 4 * 2.0 ** -23 * (np.abs(c0) * beta + np.abs(pre) + 4.0)
    got = rows(Cd.cpu().numpy(), M).astype(np.float64)
    if gelu:
        kept = rows(Pd.cpu().numpy(), M).astype(np.float64)
        assert (np.abs(kept[:, :N] - pre) <= bound).all() and (kept[:, N:] == 0).all()
        assert (np.abs(got[:, :N] - F.gelu(pre)) <= 1.13 * bound + 2.0 ** -20 * np.abs(pre)).all()
    else:
        assert (np.abs(got[:, :N] - pre) <= bound).all()
    assert np.array_equal(got[:, N:], rows(C0, M)[:, N:]) and np.array_equal(Cd[:off].cpu().numpy(), C0[:off])


@pytest.mark.parametrize("M,N", [(1, 2 ** 28), (2, 2 ** 27)])
def test_products_wider_than_the_pointwise_offsets(gpu, M, N):
    """Rows so long that a 32-bit offset of row 31 would wrap into row 0: K = 1,
    so each value is one product of two bf16 numbers, exact in float32."""
    import torch

    print(f"wide gemm M={M} N={N}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M)
    A = torch.randn((M, 1), device=gpu, generator=g).to(torch.bfloat16).float()
    B = torch.randn(N, device=gpu, generator=g).to(torch.bfloat16).float()
    C = torch.full((M, N), np.nan, device=gpu)
    L.call("namsa_gemm_bf16", L.ptr(A), 0, 1, 1, L.ptr(B), 0, N, 1, L.ptr(C), 0, N, 1, M, N, 1, 1, 1, np.float32(1.0),
           np.float32(0.0), None, 0, 0, None, L.stream_handle())
    for i in range(M):
        assert torch.equal(C[i], A[i] * B), i
