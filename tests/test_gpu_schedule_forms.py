"""The forms a column schedule takes by the launch's size agree."""
import numpy as np
import pytest

import namsa_amd._lib as L
from namsa_amd import autotune

pytestmark = pytest.mark.gpu


def _run(torch, dev, psi_k, pos, t, pm, band, kmax, mode):
    N, B = psi_k.shape[-1], len(pos)
    ws = torch.empty((B, N, N), dtype=torch.complex64, device=dev)
    cb = torch.empty((B, N, N), dtype=torch.float32, device=dev)
    L.call("namsa_multislice", L.ptr(psi_k), L.ptr(pos), B, N, N, np.float32(kmax), L.ptr(t), len(t), L.ptr(pm), *band,
           B, mode, np.float32(1.0), L.ptr(ws), L.ptr(cb), None, 0, None, None, L.stream_handle())
    return torch.view_as_real(ws) if mode == L.OUT_EXIT else cb


@pytest.mark.parametrize("N,name", [(192, "e12.r12.4.4.c16"), (256, "e8.r884.c8.pf")])
def test_readout_keeps_the_transform_of_the_slice_loop(gpu, N, name):
    """The default's readout has the radices of its passes: the CBEDs are those
    of the persistent schedule of the same transform, bit for bit."""
    import torch

    g = torch.Generator(device=gpu).manual_seed(N)
    unit = lambda *s: torch.polar(torch.ones(s, device=gpu), 0.5 * torch.randn(s, device=gpu, generator=g))   # noqa: E731
    psi_k, t, pm = unit(N, N) / N, unit(2, N, N), unit(N, N)
    pos = 8.0 * torch.rand((5, 2), device=gpu, generator=g) - 4.0
    keep = autotune.selected(N, 1)
    out = []
    try:
        for v in (keep, name):
            autotune.select(N, 1, v)
            out.append(_run(torch, gpu, psi_k, pos, t, pm, (0, N), 8.0, L.OUT_CBED))
    finally:
        autotune.select(N, 1, keep)
    assert torch.equal(*out)
