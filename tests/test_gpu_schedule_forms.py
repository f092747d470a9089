"""The forms a column schedule takes by the launch's size: narrow strips, the
persistent form, one or several images per workgroup.  Groups large enough that
the schedule's own form runs, against the FP64 oracle and, bit for bit, against
its probes run four at a time (narrow).  Four probe positions, repeated."""
import numpy as np
import pytest

import namsa_amd._lib as L
from namsa_amd import autotune
from tests.parity_util import rel_l2
from tests.test_gpu_schedules import _case

pytestmark = pytest.mark.gpu

# At 192^2 and 256^2 the persistent form holds about 110 and 70 images of the
# oracle case's band at a time (96 and 58 of the default band): these lie
# between one such set and two.
WIDE = {128: 48, 192: 150, 256: 90, 512: 8, 768: 4}
# Of the default band: one image per workgroup; several where a schedule takes them.
BATCHES = {128: (70, 300), 192: (110, 125, 150, 360, 400), 256: (64, 80, 200, 250), 384: (24, 64), 512: (14, 40),
           768: (7, 16), 1024: (9, 16, 24, 40), 2048: (4, 8)}


def _run(torch, dev, psi_k, pos, t, pm, band, kmax, mode):
    N, B = psi_k.shape[-1], len(pos)
    ws = torch.empty((B, N, N), dtype=torch.complex64, device=dev)
    cb = torch.empty((B, N, N), dtype=torch.float32, device=dev)
    L.call("namsa_multislice", L.ptr(psi_k), L.ptr(pos), B, N, N, np.float32(kmax), L.ptr(t), len(t), L.ptr(pm), *band,
           B, mode, np.float32(1.0), L.ptr(ws), L.ptr(cb), None, 0, None, None, L.stream_handle())
    return torch.view_as_real(ws) if mode == L.OUT_EXIT else cb


@pytest.mark.parametrize("N", sorted(WIDE))
def test_every_column_schedule_in_its_wide_form(gpu, N):
    """rel-L2 < 1e-5 against the oracle, FP32 rounding of eight transforms."""
    import torch

    psi_k, pos, t, pm, band, kmax, exit_ref, cbed_ref = _case(N, N + 1)
    c64 = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.complex64)).to(gpu)   # noqa: E731
    pk, td, pmd = c64(psi_k), c64(t), c64(pm)
    p = torch.from_numpy(np.resize(pos, (WIDE[N], 2))).to(gpu)
    keep = autotune.selected(N, 1)
    try:
        for name in autotune.schedules(N, 1):
            autotune.select(N, 1, name)
            print(f"N={N} B={WIDE[N]} column schedule={name}", flush=True)
            for mode, ref in ((L.OUT_EXIT, exit_ref), (L.OUT_CBED, cbed_ref)):
                got = _run(torch, gpu, pk, p, td, pmd, band, kmax, mode).cpu().numpy()
                got = got[..., 0] + 1j * got[..., 1] if mode == L.OUT_EXIT else got
                for i in (0, len(p) // 2, len(p) - 1):
                    e = rel_l2(got[i], ref[i % len(pos)])
                    assert e < 1e-5, (name, mode, i, e)
    finally:
        autotune.select(N, 1, keep)


@pytest.mark.parametrize("mode", [L.OUT_CBED, L.OUT_EXIT])
@pytest.mark.parametrize("N", sorted(BATCHES))
def test_forms_of_the_default_schedules_agree(gpu, N, mode):
    import torch

    g = torch.Generator(device=gpu).manual_seed(N + 1)
    unit = lambda *s: torch.polar(torch.ones(s, device=gpu), 0.5 * torch.randn(s, device=gpu, generator=g))   # noqa: E731
    band = lo, hi = autotune.default_band(N)
    psi_k, t, pm = unit(N, N) / N, unit(2, N, N), unit(N, N)
    pm[:, :lo] = 0
    pm[:, hi:] = 0
    pos = 8.0 * torch.rand((4, 2), device=gpu, generator=g) - 4.0
    few = _run(torch, gpu, psi_k, pos, t, pm, band, 8.0, mode)
    assert bool(torch.isfinite(few).all()) and float(few.abs().max()) > 0
    for B in BATCHES[N]:
        print(f"forms N={N} B={B} mode={mode}", flush=True)
        many = _run(torch, gpu, psi_k, pos.repeat((B + 3) // 4, 1)[:B].contiguous(), t, pm, band, 8.0, mode)
        for i in range(4):
            assert torch.equal(many[i::4], few[i].expand_as(many[i::4])), (B, i)


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
