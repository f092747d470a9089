"""The corrector's row kernels in training against the separate products of
the same network: every activation and gradient bit for bit, since each sum
keeps its order (the weight gradients that atomics add up excepted)."""
import numpy as np
import pytest

from namsa_amd import corrector as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,cin,B", [
    (16, 16, 7, 1),      # one partial tile a row
    (37, 70, 3, 3),      # 111 rows: a workgroup with one idle wavefront; a last tile of 6 pixels
    (33, 96, 16, 2),     # whole tiles, every input channel the lift takes
    (170, 170, 7, 2),
])
def test_row_kernels_equal_separate_products(gpu, H, W, cin, B):
    import torch
    print(f"row kernels H={H} W={W} cin={cin} B={B}", flush=True)
    rng = np.random.default_rng(H + W)
    p = {k: rng.standard_normal(s) / np.sqrt(s[-1]) for k, s in K.FnoNet(H, W, cin=cin).shapes.items()}
    n = B * H * W
    u = torch.from_numpy(rng.standard_normal((cin, n)).astype(np.float32)).cuda()
    gout = torch.from_numpy(rng.standard_normal((2, n)).astype(np.float32)).cuda()
    got = []
    for rows in (True, False):
        net = K.FnoNet(H, W, cin=cin)
        net.load(p)
        if not rows:
            net.rows_ok = lambda B: False
        assert net.rows_ok(B) == rows
        net.ensure(B)
        for t in (*net.xs, *net.pre, net.ga, net.gb, net.Z, net.Zp, net.out, net.h, net.hpre):
            t.fill_(np.nan)
        net.u.copy_(u)
        net.gout.copy_(gout)
        net.forward(B)
        net.backward(B)
        torch.cuda.synchronize()
        got.append([*net.xs, *net.pre, net.out, net.ga, net.gb, net.Xs, net.gview("G").clone()])
    for i, (a, b) in enumerate(zip(*got)):
        assert torch.isfinite(b).all(), i
        assert torch.equal(a, b), i
