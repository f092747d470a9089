"""Binning of the sites on the device against the host's site table, which
they equal exactly: atom counts on both sides of a workgroup's step, empty
slices, depths on the bounds, outside every slice, NaN and infinite, positions
an int cannot hold."""
import numpy as np
import pytest

from namsa_amd import MSAGPU, structures

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,dz,wild", [(2, 2.0, False), (63, 0.5, True), (16383, 2.0, False), (16385, 1.0, True),
                                       (30011, 0.7, True)])
def test_bins_match_host(gpu, A, dz, wild):
    print(f"bin sites A={A} dz={dz} wild={wild}", flush=True)
    rng = np.random.default_rng(A)
    xyz = rng.uniform(0.0, [20.0, 30.0, 41.0], (A, 3)).astype(np.float32)
    xyz[:2] = [0.0, 0.0, 0.0], [20.0, 30.0, 41.0]
    rec = structures.make_records(xyz, rng.choice([1, 6, 14, 79], A))
    sim = MSAGPU(100.0, 0.02, rec, sampling=np.array([128, 128]), debye_waller=False)
    sim.unique_Z = np.unique(sim.supercell_Z)
    sim.setup_device(0)
    at = sim.supercell_xyz
    at[2::5, 2] = np.floor(at[2::5, 2] / dz) * np.float32(dz)      # on a bound, or next to one
    if wild:
        at[3::50, 2] = rng.choice([np.nan, np.inf, -np.inf, -0.0, -3.0, 1e9], len(at[3::50])).astype(np.float32)
        at[4::50, 0] = rng.choice([np.nan, np.inf, -np.inf, -7.5, 3e12, -3e12], len(at[4::50])).astype(np.float32)
    with np.errstate(invalid="ignore"):
        sites, offsets = sim.site_table(dz)
    got, offs = sim._sites_device(dz)
    np.testing.assert_array_equal(offs.cpu().numpy(), offsets)
    assert got.numel() == 3 * A
    np.testing.assert_array_equal(got.cpu().numpy()[:sites.size].reshape(-1, 3), sites)
