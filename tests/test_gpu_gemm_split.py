"""Split-K products with both operands contiguous along K (the corrector's
weight gradients): every combination of one and two 32-wide blocks with ragged
edges, K on both sides of a wavefront's step and a workgroup's share, rows and
pointers off 16 bytes, a zero-stride operand, batches and a strided C.  Against
float64 products of the bf16-rounded operands: FP32 accumulation, 2e-5 of the
norm of |A| |B|."""
import numpy as np
import pytest

import namsa_amd._lib as L
from tests.test_gpu_corrector_kernels import bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,batch,pad,off,zero", [
    (1, 1, 1, 1, 0, 0, False), (32, 32, 31, 1, 1, 1, False), (32, 32, 33, 2, 3, 2, False), (2, 64, 127, 1, 0, 0, False),
    (64, 1, 1000, 1, 0, 0, True), (33, 47, 129, 3, 2, 1, False), (64, 64, 4099, 1, 1, 3, False),
    (7, 32, 70001, 1, 0, 0, False), (32, 1, 40000, 2, 1, 0, True), (64, 33, 33000, 1, 0, 0, False)])
def test_split_products(gpu, M, N, K, batch, pad, off, zero):
    import torch

    print(f"split gemm M={M} N={N} K={K} batch={batch} pad={pad} off={off} zero stride={zero}", flush=True)
    rng = np.random.default_rng(K + M)
    sA, sB = K + pad, 0 if zero else K + pad
    A = rng.standard_normal(off + batch * M * sA + K).astype(np.float32)
    B = rng.standard_normal(off + batch * max(1, N * sB) + K).astype(np.float32)
    bA, bB = M * sA, N * sB
    sC = (1, M + 2)                                   # C stored column by column, padded
    C0 = rng.standard_normal(batch * N * (M + 2)).astype(np.float32)
    Ad, Bd, Cd = (torch.from_numpy(x).to(gpu) for x in (A, B, C0.copy()))
    L.call("namsa_gemm_bf16", L.ptr(Ad[off:]), bA, sA, 1, L.ptr(Bd[off:]), bB, 1, sB, L.ptr(Cd), N * (M + 2), *sC, M, N,
           K, batch, 3, np.float32(0.5), np.float32(0.0), None, 0, 0, None, L.stream_handle())
    got = Cd.cpu().numpy().astype(np.float64)
    touched = np.zeros(got.shape, bool)
    for b in range(batch):
        a = bf16(np.stack([A[off + b * bA + i * sA:][:K] for i in range(M)]))
        w = bf16(np.stack([B[off + b * bB + j * sB:][:K] for j in range(N)]))
        at = b * N * (M + 2) + np.arange(M)[:, None] * sC[0] + np.arange(N)[None, :] * sC[1]
        touched[at] = True
        err = np.linalg.norm(got[at] - C0[at] - 0.5 * (a @ w.T)) / np.linalg.norm(np.abs(a) @ np.abs(w).T)
        assert err < 2e-5, (b, err)
    assert np.array_equal(got[~touched], C0[~touched])


@pytest.mark.parametrize("M,N,n", [(1, 1, 1), (32, 32, 31), (8, 3, 127), (32, 7, 129), (32, 32, 70001)])
def test_weight_grad(gpu, M, N, n):
    """The product with its row sums, both added to what is there; the same bound."""
    import torch

    print(f"weight grad M={M} N={N} n={n}", flush=True)
    rng = np.random.default_rng(n)
    gy, x = (rng.standard_normal((k, n)).astype(np.float32) for k in (M, N))
    C0 = rng.standard_normal((M, N + 1)).astype(np.float32)
    gd, xd, W, b = (torch.from_numpy(v.copy()).to(gpu) for v in (gy, x, C0[:, :N], C0[:, N]))
    L.call("namsa_weight_grad", L.ptr(gd), L.ptr(xd), n, M, N, L.ptr(W), L.ptr(b), L.stream_handle())
    got = np.concatenate([W.cpu().numpy(), b.cpu().numpy()[:, None]], 1).astype(np.float64)
    a, w = bf16(gy), np.concatenate([bf16(x), np.ones((1, n))])
    err = np.linalg.norm(got - C0 - a @ w.T) / np.linalg.norm(np.abs(a) @ np.abs(w).T)
    assert err < 2e-5, err


def test_weight_grad_over_the_largest_k(gpu):
    """The last workgroup's share ends at 2^31 - 256: only the last 1000 values
    of one vector, taken as both operands, are not 0, so the sums are exact."""
    import torch

    n = 2 ** 31 - 256
    print(f"weight grad n={n}", flush=True)
    v = torch.zeros(n, device=gpu)
    v[-1000:] = 2.0
    out = torch.zeros(2, device=gpu)
    L.call("namsa_weight_grad", L.ptr(v), L.ptr(v), n, 1, 1, L.ptr(out), L.ptr(out[1:]), L.stream_handle())
    assert out.tolist() == [4000.0, 2000.0]
