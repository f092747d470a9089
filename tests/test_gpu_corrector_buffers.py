"""FnoNet.ensure holds every buffer of the training passes: none is allocated
by a pass (which a program may capture), and none that no pass of the network
reads or writes."""
import numpy as np
import pytest

from namsa_amd import corrector as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,m,Hq,cin", [(32, 16, 64, 7), (16, 8, 32, 7), (32, 16, 48, 7), (40, 8, 64, 5)])
def test_passes_allocate_nothing(gpu, C, m, Hq, cin):
    import torch
    H, W, B = 40, 50, 3
    print(f"buffers C={C} m={m} Hq={Hq} cin={cin}", flush=True)
    net = K.FnoNet(H, W, cin=cin, C=C, m=m, Hq=Hq)
    rng = np.random.default_rng(C + Hq)
    net.load({k: rng.standard_normal(s) / np.sqrt(s[-1]) for k, s in net.shapes.items()})
    net.ensure(B)
    net.u.copy_(torch.from_numpy(rng.standard_normal(tuple(net.u.shape)).astype(np.float32)))
    net.gout.copy_(torch.from_numpy(rng.standard_normal(tuple(net.gout.shape)).astype(np.float32)))
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]   # noqa: E731
    before = count()
    net.forward(B)
    net.forward(B - 1)
    net.forward(B)
    net.backward(B)
    assert count() == before
    assert bool(torch.isfinite(net.grad).all()) and float(net.grad.abs().max()) > 0
    general_head = (C, Hq) != (32, 64)
    assert (net.h is not None) == general_head
    assert (net.ones is not None) == (general_head or C > 32 or cin > 32)
