"""The Kirkland tables at the edges of their launch: one-pixel tables, sizes
that leave a workgroup part-filled, subsample counts on both sides of the
one-thread-per-subsample kernel, and a potential whose minimum is not in a
corner, against the FP64 oracle.  Both round an FP64 difference v - min v to
float32, v being a sum of terms known to about 1e-13 of themselves: at most
one float32 ulp apart, plus 1e-12 of the largest term before the shift."""
import numpy as np
import pytest

import namsa_amd._lib as L
from namsa_amd.msa import kirkland_params
from oracle import msa_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Py,Px,over", [(1, 1, 2), (2, 1, 2), (7, 9, 1), (9, 7, 3), (16, 16, 4), (5, 6, 5), (33, 31, 2)])
@pytest.mark.parametrize("ring", [False, True])
def test_tables_match_oracle(gpu, Py, Px, over, ring):
    import torch

    print(f"atomic tables {Py}x{Px} oversample {over} ring={ring}", flush=True)
    params = kirkland_params[np.array([6, 79]) - 1].copy()
    if ring:                     # a broad negative Gaussian: the minimum lies between centre and corner
        params[:, 2, 0], params[:, 3, 0] = -60.0, 30.0
    reach = 8.0
    ref = np.stack([O.atomic_table(p, (reach / (Py + 0.5), reach / (Px + 0.5)), reach, over) for p in params])
    assert ref.shape == (2, Py, Px)
    out = torch.full((2, Py, Px), np.nan, dtype=torch.float32, device=gpu)
    pd = torch.from_numpy(np.ascontiguousarray(params)).to(gpu)
    L.call("namsa_atomic_tables", L.ptr(pd), 2, Py, Px, reach, over, L.ptr(out), L.stream_handle())
    got = out.cpu().numpy().astype(np.float64)
    assert (got.reshape(2, -1).min(axis=1) == 0).all()
    # largest term of v: the Bessel sums and Gaussians at the centre
    pref = 4 * np.pi ** 2 * O.A0_BOHR * O.E_CHARGE
    term = pref * np.maximum(np.abs(params[:, 0]) * O.k0(O.BESSEL_EPS), np.abs(params[:, 2] / params[:, 3]) / 2).max(axis=1)
    bound = np.abs(ref) * 2.0 ** -23 + 1e-12 * term[:, None, None]
    assert (np.abs(got - ref) <= bound).all()
