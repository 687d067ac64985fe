"""The x and y passes leave the parts of their work arrays outside the 2/3 sphere's cylinder untouched:
whatever an earlier call left there must not reach a result, and what lies outside the sphere stays zero."""
import numpy as np
import pytest

from conftest import wavenumbers

pytestmark = pytest.mark.gpu


def poison(s):
    """fill the work arrays with NaN (the real-space fields of a NaN state pass through all of them)"""
    bad = np.zeros(s.spectral_shape, dtype=np.complex128)
    bad[1, 1, 1] = bad[0, 0, 0] = np.nan
    s.set_state(bad)
    for which in (0, 1):
        assert np.isnan(s.realspace(which)).all()


@pytest.mark.parametrize("precision", ["fp64", "fp32bulk"])
@pytest.mark.parametrize("N", [8, 12, 16, 24, 32, 48, 64, 96, 128, 256])
def test_nothing_outside_the_cut_is_read(nsg, oracle, N, precision):
    uh = oracle.ic_k4(N, min(2.0, N / 8.0), 0.5, 70 + N)
    kw = dict(nu=0.01, dt=1e-3, precision=precision, force_eps=0.1, force_kf=1.5)
    for sched in range(min(3, nsg.schedule_count(N) // 3)):
        got = []
        for bad in (False, True):
            with nsg.Solver(N, **kw) as s:
                s.set_schedule(sched)
                if bad:
                    poison(s)
                nl = s.rhs(uh)
                s.set_state(uh)
                s.step(2)
                got.append((nl, s.get_state()))
        for a, b in zip(*got):
            assert np.array_equal(a, b)
    kx, ky, kz = wavenumbers(N)
    out = kx * kx + ky * ky + kz * kz > (N // 3) ** 2
    assert not got[0][0][out].any() and not got[0][1][out].any()


@pytest.mark.parametrize("N", [12, 48, 96])
@pytest.mark.parametrize("scheme", ["rk5cn", "dp5"])
def test_dormand_prince_outside_the_cut(nsg, oracle, N, scheme):
    """the skipped blocks' error slots count as zero and the candidate state stays zero outside"""
    uh = oracle.ic_k4(N, 2.0, 0.5, 80 + N)
    got = []
    for bad in (False, True):
        with nsg.Solver(N, nu=0.01, dt=1e-3, scheme=scheme) as s:
            if bad:
                poison(s)
            s.set_state(uh)
            s.step(3)
            got.append((s.get_state(), s.dp_stats() if scheme == "dp5" else None))
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]
