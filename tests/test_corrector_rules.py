"""The corrector's rules for its special training kernels, on the host: what
they are given is within what their entry points take, and batches that went
through before still do."""
from types import SimpleNamespace

import pytest

from namsa_amd import _lib as L
from namsa_amd import corrector as K


@pytest.mark.parametrize("H,W", [(170, 170), (1024, 16), (700, 31), (341, 32), (16, 16), (2048, 20), (512, 512)])
def test_rows_ok_keeps_to_the_row_kernels_limit(H, W):
    """The row kernels also index the row DFTs, 32 channels of 32 values a row,
    in 31 bits: the narrower windows' limit.  The entry point refuses what is past
    it (checked before any launch), the separate products take it."""
    most = (2 ** 31 - 1) // (128 * max(W, 32)) // H           # samples the entry point takes
    Wp = (W + 31) // 32 * 32
    one = L.C.c_void_p(4096)                                  # never followed
    for B in (1, most - 1, most, most + 1, 2 * most):
        net = SimpleNamespace(C=32, m=16, cin=7, H=H, W=W)
        assert K.FnoNet.rows_ok(net, B) == (B <= most), B
        if B > most:
            with pytest.raises(L.NamsaError, match="bad geometry"):
                L.call("namsa_fno_rows", one, 7, None, None, one, one, 0, one, 1.0, None, None, 1.0, B, H, W, Wp, one,
                       one, None)
