"""A probe's results do not depend on how many are run with it: the column
pass picks its strip width and images per workgroup from the batch, with the
same operations per column, so the CBEDs and exit waves of a batch equal those
of its probes run a few at a time, bit for bit, on thin runs and on runs thick
enough for the schedules that hold every twiddle."""
import numpy as np
import pytest

import namsa_amd._lib as L
from namsa_amd import autotune

pytestmark = pytest.mark.gpu

# batches on both sides of one narrow-strip task per CU, and of one image per
# workgroup; at 192 and 256 the whole batch fills a persistent launch evenly
BATCH = {128: 70, 192: 92, 256: 56, 384: 24, 512: 14, 768: 7, 1024: 9, 2048: 4}


@pytest.mark.parametrize("mode", [L.OUT_CBED, L.OUT_EXIT])
@pytest.mark.parametrize("thick", [False, True])
@pytest.mark.parametrize("N", sorted(BATCH))
def test_results_do_not_depend_on_the_batch(gpu, N, thick, mode):
    import torch

    B = BATCH[N]
    S = L.load().namsa_precise_slices(N) + 1 if thick else 2
    print(f"batch split N={N} B={B} S={S} mode={mode}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(N)
    lo, hi = autotune.default_band(N)
    unit = lambda *s: torch.polar(torch.ones(s, device=gpu), 0.5 * torch.randn(s, device=gpu, generator=g))   # noqa: E731
    psi_k = unit(N, N) / N
    t1 = unit(2, N, N)
    # the driver takes [S][N][N]; on thick runs every slice but two is 1
    t = torch.ones((S, N, N), dtype=torch.complex64, device=gpu)
    t[:2] = t1
    pm = unit(N, N)
    pm[:, :lo] = 0
    pm[:, hi:] = 0
    pos = 8.0 * torch.rand((B, 2), device=gpu, generator=g) - 4.0

    def run(i, b):
        ws = torch.empty((b, N, N), dtype=torch.complex64, device=gpu)
        cb = torch.empty((b, N, N), dtype=torch.float32, device=gpu)
        p = pos[i:i + b].contiguous()
        L.call("namsa_multislice", L.ptr(psi_k), L.ptr(p), b, N, N, np.float32(8.0), L.ptr(t), S, L.ptr(pm), lo, hi, b,
               mode, np.float32(1.0), L.ptr(ws), L.ptr(cb), None, 0, None, None, L.stream_handle())
        return torch.view_as_real(ws) if mode == L.OUT_EXIT else cb

    whole = run(0, B)
    assert bool(torch.isfinite(whole).all()) and float(whole.abs().max()) > 0
    i = 0
    for b in (1, 2, 3, 5, 8, 13, 21, 34):
        if i + b > B:
            break
        assert torch.equal(run(i, b), whole[i:i + b]), (N, i, b)
        i += b
