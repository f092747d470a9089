"""The fused y transforms of the corrector's modes against the separate
products, which they equal bit for bit: H below, at and between the steps of 16
and 64 rows and the tiles of 32, channel counts of one to several samples."""
import numpy as np
import pytest

from namsa_amd import corrector as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,C,B", [(16, 32, 2), (17, 64, 1), (63, 32, 3), (170, 32, 5), (193, 8, 16), (512, 32, 2)])
def test_y_transforms_equal_separate_products(gpu, H, C, B):
    import torch
    print(f"y transforms H={H} C={C} B={B}", flush=True)
    net = K.FnoNet(H, 16, C=C)
    net._ensure_common(B)
    rng = np.random.default_rng(H + C)
    for t in (net.Z, net.Ys):
        t.copy_(torch.from_numpy(rng.standard_normal(tuple(t.shape)).astype(np.float32)))
    CB = C * B
    want, got = torch.full_like(net.Xs[0], np.nan), torch.full_like(net.Xs[0], np.nan)
    net._gemm(K._addr(net.Fy), (0, H, 1), K._addr(net.Z), (H * 32, 32, 1), K._addr(net.Pm), (1024, 32, 1), 32, 32, H,
              batch=CB)
    K.call("namsa_modes_combine", K.ptr(net.Pm), K.ptr(want), C, B, 16, net.st)
    net._y_forward(K.ptr(got), B)
    assert torch.isfinite(want).all() and torch.equal(got, want)
    want, got = torch.full_like(net.Zp, np.nan), net.Zp.fill_(np.nan)
    K.call("namsa_modes_expand", K.ptr(net.Ys), K.ptr(net.E), C, B, 16, net.st)
    net._gemm(K._addr(net.Fy), (0, 1, H), K._addr(net.E), (1024, 32, 1), K._addr(want), (H * 32, 32, 1), H, 32, 32,
              batch=CB)
    net._spectral_rows(K.ptr(net.Ys), B)
    assert torch.isfinite(want).all() and torch.equal(got, want)
