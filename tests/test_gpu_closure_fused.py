"""The closure term through the fused small-box kernels (FFT schedule 0) against the separate transforms
(schedule 1): gradients, network input, stress spectra and term of the same state."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [16, 32, 48, 64, 96])
@pytest.mark.parametrize("precision,scheme", [("fp64", "rk4cn"), ("fp32bulk", "rk4cn"), ("fp64", "dp5")])
def test_closure_term_and_step(nsg, oracle, N, precision, scheme):
    uh = oracle.ic_k4(N, 2.0, 0.5, 400 + N)
    gain = np.linspace(0.5, 1.5, N // 3 + 1)
    got = []
    with nsg.Network(N, seed=3) as net:
        net.set_norm(1.8, [0.035] * 6)
        net.set_params(0.1 * net.get_params())
        for sched in (0, 1):
            with nsg.Solver(N, nu=0.01, dt=1e-3, precision=precision, scheme=scheme, force_eps=0.1) as s:
                s.set_schedule(sched)
                s.set_state(uh)
                s.attach_closure(net)
                a = s.closure_term()
                s.set_closure_gain(gain)
                b = s.closure_term()
                s.step(3)
                got.append((a, b, s.get_state()))
    (a0, b0, u0), (a1, b1, u1) = got
    # the network's input is rounded to bfloat16: one of 9 N^3 values within FP64 round-off of a tie
    # would move the term by about 2^-8 / sqrt(9 N^3) of itself; otherwise the chains agree to round-off
    bar = 2.0 ** -8 / np.sqrt(9.0 * N ** 3)
    assert rel(a0, a1) < bar and rel(b0, b1) < bar
    assert np.linalg.norm(a0) > 0 and rel(b0, a0) > 1e-2
    assert rel(u0, u1) < (1e-7 if precision == "fp32bulk" else 1e-9)
