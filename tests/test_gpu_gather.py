"""A minibatch gathered in one launch against index_select, bit for bit: rows
of whole and of odd numbers of 16-byte words, scalars, repeated and reversed
rows, more than a workgroup's share a row; tensors it does not take fall back."""
import numpy as np
import pytest

from namsa_amd import corrector as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,idx", [((1,), [0]), ((7,), [3, 3, 0]), ((65, 67), [5, 4, 0, 5]),
                                       ((256, 256), list(range(5, -1, -1)))])
def test_gather_equals_index_select(gpu, shape, idx):
    import torch
    print(f"gather {shape} {idx}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(len(idx))
    real = torch.randn((6, *shape), device=gpu, generator=g)
    tensors = (torch.complex(real, -real), real, torch.arange(6, device=gpu, dtype=torch.int32), real[:, 0].contiguous(),
               torch.randn((7, 3), device=gpu, generator=g)[1:], real.double())
    for t in (tensors, (real.half(), real), (real.transpose(0, -1).contiguous().transpose(0, -1), real)):
        for a, b in zip(K._gather(t, idx), t):
            want = b.index_select(0, torch.as_tensor(idx, device=gpu))
            assert a.dtype == want.dtype and a.shape == want.shape and torch.equal(a, want)


@pytest.mark.parametrize("lazy", ["conj", "neg"])
def test_gather_resolves_lazy_views(gpu, lazy):
    """Views that torch marks as conjugated or negated instead of computing
    them are contiguous; their rows have the values, as index_select gives them."""
    import torch
    z = torch.randn((5, 6, 4), dtype=torch.complex64, device=gpu, generator=torch.Generator(device=gpu).manual_seed(1))
    view = z.conj() if lazy == "conj" else torch._neg_view(z.real.contiguous())
    assert view.is_contiguous() and (view.is_conj() or view.is_neg())
    got, = K._gather((view,), [4, 0, 2])
    want = view.index_select(0, torch.tensor([4, 0, 2], device=gpu))
    assert torch.equal(got, want) and float(want.abs().max()) > 0


def test_gather_leaves_other_devices_to_torch(gpu, monkeypatch):
    """The launch goes to the current device's stream: tensors of another
    device are left to index_select, which runs on theirs."""
    import torch
    t = torch.arange(12.0, device=gpu).reshape(4, 3)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: gpu.index + 1)
    monkeypatch.setattr(K, "call", lambda name, *a: pytest.fail(name))
    got, = K._gather((t,), [3, 1])
    assert got.tolist() == [[9.0, 10.0, 11.0], [3.0, 4.0, 5.0]]
