"""namsa_integrate and namsa_norm2 at the edges of their launches: patterns of
a few pixels, planes and pointers off the 16-byte loads, one detector more than
a workgroup takes, counts on both sides of one workgroup per CU.  Products of
float32 values are exact in FP64, so only the n additions round: n 2^-53 of the
sum of absolute values."""
import numpy as np
import pytest

import namsa_amd._lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Ny,Nx,D,off", [(1, 1, 1, 1, 0), (2, 1, 3, 4, 0), (3, 64, 64, 5, 0), (3, 64, 64, 2, 1),
                                           (5, 33, 65, 9, 0), (257, 16, 20, 3, 0), (300, 31, 9, 6, 2),
                                           (64, 96, 96, 4, 0), (1, 256, 260, 8, 0)])
def test_integrate_matches_numpy(gpu, B, Ny, Nx, D, off):
    import torch

    print(f"integrate B={B} {Ny}x{Nx} detectors={D} offset={off}", flush=True)
    rng = np.random.default_rng(B + D)
    cb = rng.standard_normal((B, Ny, Nx)).astype(np.float32)
    det = rng.standard_normal((D, Ny, Nx)).astype(np.float32)
    flat = torch.zeros(B * Ny * Nx + off, dtype=torch.float32, device=gpu)
    flat[off:] = torch.from_numpy(cb.reshape(-1)).to(gpu)
    dd = torch.from_numpy(det).to(gpu)
    out = torch.full((B, D), np.nan, dtype=torch.float64, device=gpu)
    L.call("namsa_integrate", L.ptr(flat[off:]), B, Ny, Nx, L.ptr(dd), D, L.ptr(out), L.stream_handle())
    x, w = cb.reshape(B, -1).astype(np.float64), det.reshape(D, -1).astype(np.float64)
    bound = 2 * Ny * Nx * 2.0 ** -53 * (np.abs(x) @ np.abs(w).T)
    assert (np.abs(out.cpu().numpy() - x @ w.T) <= bound).all()


@pytest.mark.parametrize("n,off", [(1, 0), (1, 1), (2047, 0), (16384, 0), (16385, 1), (100001, 0), (1 << 18, 0)])
def test_norm2_matches_numpy(gpu, n, off):
    import torch

    print(f"norm2 n={n} offset={off}", flush=True)
    x = np.random.default_rng(n).standard_normal((n + off, 2)).astype(np.float32)
    xd = torch.view_as_complex(torch.from_numpy(x).to(gpu))
    out = torch.full((1,), np.nan, dtype=torch.float64, device=gpu)
    L.call("namsa_norm2", L.ptr(xd[off:]), n, L.ptr(out), L.stream_handle())
    ref = (x[off:].astype(np.float64) ** 2).sum()
    assert abs(float(out) - ref) <= 4 * n * 2.0 ** -53 * ref
