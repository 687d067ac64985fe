"""The subgrid-stress sample with the products transformed back only up to the LES cut, against the
closure oracle, over pairs of grids on both sides of the rule that picks it (scratch size), and with
NaN left in the scratch by an earlier call.  Bar 1e-6 (float32 outputs), as tests/test_gpu_closure.py."""
import numpy as np
import pytest

from conftest import rel
from test_gpu_closure import C

pytestmark = pytest.mark.gpu


# 64 -> 48 and 128 -> 96 keep the uncut path; 12 -> 8, 48 -> 16, 96 -> 64, 128 -> 64 are cut
@pytest.mark.parametrize("N,Nl", [(12, 8), (24, 16), (48, 16), (64, 24), (64, 48), (96, 64), (128, 64), (128, 96)])
def test_sample(nsg, oracle, N, Nl):
    uh = oracle.ic_k4(N, min(3.0, N / 8.0), 0.5, 500 + N)
    kc = max(2, Nl // 3)
    want_x, want_t = C.sgs_sample(uh, N, Nl, kc)[-2:]
    with nsg.Solver(N, nu=0.01) as dns, nsg.Solver(Nl, nu=0.01) as les:
        for bad in (False, True):
            if bad:
                nan = np.zeros(dns.spectral_shape, dtype=np.complex128)
                nan[1, 1, 1] = np.nan
                dns.set_state(nan)
                assert np.isnan(dns.realspace(0)).all()
            dns.set_state(uh)
            x, t = dns.sgs_sample(les, kc)
            assert rel(x.reshape(-1, 9), np.asarray(want_x).reshape(-1, 9)) < 1e-6
            assert rel(t.reshape(-1, 6), np.asarray(want_t).reshape(-1, 6)) < 1e-6
