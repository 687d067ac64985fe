"""Fused x/y passes (FFT schedule 0 up to 96^3) against the five separate passes (schedule 1): the same
steps, times and bookkeeping, whatever was called in between."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

# the two run the same sums with other radices: FP64 a few 1e-16 a step; FP32-bulk slopes differ by up to
# 1e-6 of a slope, which a step of dt moves by dt |slope| / |u| < 1e-2
TOL = {"fp64": 1e-13, "fp32bulk": 1e-7}


def run(nsg, uh, sched, steps, **kw):
    with nsg.Solver(uh.shape[0], **kw) as s:
        s.set_schedule(sched)
        s.set_state(uh)
        s.step(steps)
        return s.get_state(), s.time(), s.dp_stats() if kw.get("scheme") == "dp5" else None


@pytest.mark.parametrize("N", [8, 12, 16, 24, 32, 48, 64, 96])
@pytest.mark.parametrize("scheme,precision", [("rk4cn", "fp64"), ("rk4cn", "fp32bulk"), ("ifrk4", "fp64"), ("ifrk4", "fp32bulk"),
                                              ("rk5cn", "fp64"), ("rk5cn", "fp32bulk"), ("dp5", "fp64")])
def test_fused_against_separate(nsg, oracle, N, scheme, precision):
    uh = oracle.ic_k4(N, min(2.0, N / 8.0), 0.5, 300 + N)
    kw = dict(nu=0.01, dt=2e-3, scheme=scheme, precision=precision, force_eps=0.1, force_kf=min(2.5, N // 3))
    if scheme != "dp5":
        kw["cfl"] = 0.4
    a, ta, da = run(nsg, uh, 0, 3, **kw)
    b, tb, db = run(nsg, uh, 1, 3, **kw)
    assert rel(a, b) < TOL[precision]
    assert np.allclose(ta, tb, rtol=1e-6 if precision == "fp32bulk" else 1e-12, atol=0)
    if da:
        assert da[:2] == db[:2]  # (the error norm itself: tests/test_gpu_rk5.py, against the oracle)


@pytest.mark.parametrize("N", [8, 16, 32, 64])
@pytest.mark.parametrize("scheme", ["rk4cn", "ifrk4", "rk5cn"])
def test_fp32_values_of_the_five_passes(nsg, oracle, N, scheme):
    """FP32-bulk is fused only with the radices of the five passes (which profile() runs): equal FP32 values,
    so the state agrees to the rounding of its FP64 update (the forcing's shell sums have another order)"""
    uh = oracle.ic_k4(N, min(2.0, N / 8.0), 0.5, 400 + N)
    kw = dict(nu=0.01, dt=2e-3, scheme=scheme, precision="fp32bulk", force_eps=0.1, force_kf=min(2.5, N // 3), cfl=0.4)
    with nsg.Solver(N, **kw) as s, nsg.Solver(N, **kw) as ref:
        for x in (s, ref):
            x.set_state(uh)
        s.step(4)
        ref.profile(4)
        assert np.allclose(s.time(), ref.time(), rtol=1e-12, atol=0)
        assert rel(s.get_state(), ref.get_state()) < TOL["fp64"]


def test_calls_between_fused_steps(nsg, oracle):
    """the kz-major copy follows every other way of setting the state, and leaves the separate passes'
    own slopes alone"""
    N = 32
    uh = oracle.ic_k4(N, 2.0, 0.5, 7)
    other = oracle.ic_k4(N, 3.0, 0.4, 8)
    with nsg.Solver(N, nu=0.01, dt=1e-3) as s, nsg.Solver(N, nu=0.01, dt=1e-3) as ref:
        ref.set_schedule(1)
        for x in (s, ref):
            x.set_state(uh)
            x.step(2)
        assert rel(s.rhs(other), ref.rhs(other)) < 1e-13
        assert np.array_equal(s.rhs(other) != 0, ref.rhs(other) != 0)
        for x in (s, ref):
            x.step(1)
            x.set_state(other)
            x.step(2)
        s.set_schedule(1)  # and back to the separate passes
        s.step(1)
        s.set_schedule(0)
        s.step(1)
        ref.step(2)
        assert rel(s.get_state(), ref.get_state()) < 1e-13
        assert s.measures()[0].energy == pytest.approx(ref.measures()[0].energy, rel=1e-13)


def test_non_finite_state_is_reported(nsg):
    N = 16
    with nsg.Solver(N, nu=0.01, dt=1e-3) as s:
        bad = np.zeros(s.spectral_shape, dtype=np.complex128)
        bad[1, 2, 3] = np.nan
        s.set_state(bad)
        with pytest.raises(nsg.NSGError, match="non-finite"):
            s.step(1)
