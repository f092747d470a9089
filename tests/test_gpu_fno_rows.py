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
            net.rows_ok = net.head_ok = lambda B: False
        assert net.rows_ok(B) == net.head_ok(B) == rows
        net.ensure(B)
        for t in (*net.xs, *net.pre, net.ga, net.gb, net.Z, net.Zp, net.out):
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


@pytest.mark.parametrize("n", [1, 31, 256, 1030, 9000, 66001])   # below a tile; a full one; ragged ends; several a wavefront
def test_head_equals_separate_products(gpu, n):
    """The head's outputs and input gradient bit for bit; its weight gradients
    against sums in 64 bits of the same bf16 operands, whose products FP32 holds
    exactly.  A sum of n terms, in any order, is within n 2^-23 of the sum of
    their sizes (2^-23: the matrix cores may truncate)."""
    import torch
    print(f"head n={n}", flush=True)
    got = []
    for fused in (True, False):
        net = K.FnoNet(16, 16)
        net.H, net.W = 1, n                         # the head sees pixels only
        net.load({k: np.random.default_rng(5).standard_normal(s) / np.sqrt(s[-1]) for k, s in net.shapes.items()})
        x = torch.from_numpy(np.random.default_rng(6).standard_normal((32, n)).astype(np.float32)).cuda()
        go = torch.from_numpy(np.random.default_rng(7).standard_normal((2, n)).astype(np.float32)).cuda()
        out, gx = torch.full((2, n), np.nan, device="cuda"), torch.full((32, n), np.nan, device="cuda")
        p, q, st = net._p, net._g, net.st
        if fused:
            K.call("namsa_fno_head", K.ptr(x), p("Q1"), p("bq1"), p("Q2"), p("bq2"), n, K.ptr(out), st)
            K.call("namsa_fno_head_backward", K.ptr(x), p("Q1"), p("bq1"), p("Q2"), K.ptr(go), n, K.ptr(gx), q("Q1"),
                   q("bq1"), q("Q2"), q("bq2"), st)
            grads = {k: net.gview(k).double().cpu() for k in ("Q1", "bq1", "Q2", "bq2")}
        else:
            h, pre, gh = (torch.empty((64, n), device="cuda") for _ in range(3))
            net._gemm(p("Q1"), (0, 32, 1), K.ptr(x), (0, n, 1), K.ptr(h), (0, n, 1), 64, n, 32, bias=p("bq1"),
                      bias_mode=1, gelu=True, P=K.ptr(pre))
            net._gemm(p("Q2"), (0, 64, 1), K.ptr(h), (0, n, 1), K.ptr(out), (0, n, 1), 2, n, 64, bias=p("bq2"),
                      bias_mode=1)
            net._gemm(p("Q2"), (0, 1, 64), K.ptr(go), (0, n, 1), K.ptr(gh), (0, n, 1), 64, n, 2)
            K.call("namsa_gelu_backward", K.ptr(gh), K.ptr(pre), 64 * n, st)
            net._gemm(p("Q1"), (0, 1, 32), K.ptr(gh), (0, n, 1), K.ptr(gx), (0, n, 1), 32, n, 64)
        torch.cuda.synchronize()
        got.append((out, gx))
    for a, b in zip(*got):
        assert torch.isfinite(b).all() and torch.equal(a, b)
    bf = lambda t: t.to(torch.bfloat16).double().cpu()
    one = torch.ones((1, n), dtype=torch.float64)
    terms = {"Q1": (bf(gh), bf(x)), "bq1": (bf(gh), one), "Q2": (bf(go), bf(h)), "bq2": (bf(go), one)}
    for k, (a, b) in terms.items():
        want, size = a @ b.T, a.abs() @ b.abs().T
        err = (grads[k].reshape(want.shape) - want).abs()
        assert (err <= n * 2.0 ** -23 * size).all(), (k, float((err / size).max()))


@pytest.mark.parametrize("H,W,cin,B", [(16, 385, 7, 1), (17, 800, 7, 1), (16, 768, 3, 2)])
def test_rows_wider_than_a_workgroup(gpu, H, W, cin, B):
    """More tiles a row than a workgroup's wavefronts hold: several runs a row
    (two, three uneven ones, two full ones), the row DFT carried from run to run."""
    test_row_kernels_equal_separate_products(gpu, H, W, cin, B)
