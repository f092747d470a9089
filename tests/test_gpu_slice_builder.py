"""The slice builder's two kernels at the edges of their tiles and chunks: the
projected potential against float32 sums in site order (the same additions in
the same order: equal bits), and the transmission against exp(i sigma V) of
them (2e-7: the float32 sine and cosine)."""
import numpy as np
import pytest

import namsa_amd._lib as L

pytestmark = pytest.mark.gpu


def _sums(tables, sites, offsets, Ny, Nx):
    nZ, Py, Px = tables.shape
    V = np.zeros((len(offsets) - 1, Ny, Nx), np.float32)
    lo = lambda c, p: np.rint(np.float32(c) - np.float32(p * 0.5)).astype(int)   # noqa: E731
    hi = lambda c, p: np.rint(np.float32(c) + np.float32(p * 0.5)).astype(int)   # noqa: E731
    for s in range(len(V)):
        for z, y, x in sites[offsets[s]:offsets[s + 1]]:
            if not 0 <= z < nZ:
                continue
            y0, x0 = lo(y, Py), lo(x, Px)
            r0, r1 = max(y0, 0), min(hi(y, Py), Ny, y0 + Py)
            c0, c1 = max(x0, 0), min(hi(x, Px), Nx, x0 + Px)
            if r0 < r1 and c0 < c1:
                V[s, r0:r1, c0:c1] += tables[z, r0 - y0:r1 - y0, c0 - x0:c1 - x0]
    return V


# (Ny, Nx, slices, sites, Py, Px): narrow launches (few 64 x 64 tiles) with site
# counts around the 256- and 1024-site chunks, then wide ones (1024 tiles or more)
@pytest.mark.parametrize("Ny,Nx,S,A,Py,Px", [(1, 1, 1, 3, 4, 4), (15, 17, 1, 1023, 6, 5), (16, 16, 1, 1025, 9, 8),
                                             (33, 65, 3, 770, 7, 12), (64, 64, 2, 513, 70, 80),
                                             (64, 64, 1024, 3000, 16, 17), (65, 63, 512, 2500, 9, 70),
                                             (129, 200, 100, 1200, 40, 6)])
def test_sums_in_site_order(gpu, Ny, Nx, S, A, Py, Px):
    import torch

    print(f"slice builder {Ny}x{Nx} S={S} A={A} tables {Py}x{Px}", flush=True)
    rng = np.random.default_rng(A)
    nZ = 3
    tables = rng.standard_normal((nZ, Py, Px)).astype(np.float32)
    sites = np.stack([rng.integers(-1, nZ + 1, A), rng.integers(-Py, Ny + Py, A), rng.integers(-Px, Nx + Px, A)],
                     axis=1).astype(np.int32)
    offsets = np.concatenate([[0], np.sort(rng.integers(0, A + 1, S - 1)), [A]]).astype(np.int32)
    ref = _sums(tables, sites, offsets, Ny, Nx)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)   # noqa: E731
    td, sd, od = dev(tables), dev(sites.reshape(-1)), dev(offsets)
    v = torch.full((S, Ny, Nx), np.nan, dtype=torch.float32, device=gpu)
    t = torch.empty((S, Ny, Nx), dtype=torch.complex64, device=gpu)
    L.call("namsa_build_potential", L.ptr(td), nZ, Py, Px, L.ptr(sd), L.ptr(od), S, Ny, Nx, L.ptr(v), L.stream_handle())
    L.call("namsa_build_slices", L.ptr(td), nZ, Py, Px, L.ptr(sd), L.ptr(od), S, Ny, Nx, np.float32(0.3), L.ptr(t),
           L.stream_handle())
    assert np.array_equal(v.cpu().numpy(), ref)
    ph = (ref * np.float32(0.3)).astype(np.float64)
    assert np.abs(t.cpu().numpy() - np.exp(1j * ph)).max() < 2e-7
