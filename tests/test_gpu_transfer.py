"""Host copies through the pinned slots: every route (a kernel's own writes up to 64^3, chunks on the
calling thread, chunks on worker threads), several handles at once, arrays no chunk divides."""
import threading

import numpy as np
import pytest

from conftest import wavenumbers

pytestmark = pytest.mark.gpu


def masked(N, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((N, N, N // 2 + 1, 3)) + 1j * rng.standard_normal((N, N, N // 2 + 1, 3))
    kx, ky, kz = wavenumbers(N)
    keep = kx * kx + ky * ky + kz * kz <= (N // 3) ** 2
    return a, np.where(keep[..., None], a, 0)


@pytest.mark.parametrize("N", [8, 12, 64, 96, 128, 256])
def test_state_round_trip(nsg, N):
    raw, want = masked(N, N)
    with nsg.Solver(N) as s:
        for _ in range(2):
            s.set_state(raw)
            assert np.array_equal(s.get_state(), want)


def test_handles_on_several_threads(nsg):
    """six threads share the slots; each gets its own data back"""
    bad = []

    def work(i):
        N = (24, 64, 96, 128)[i % 4]
        raw, want = masked(N, 100 + i)
        with nsg.Solver(N) as s:
            for _ in range(6):
                s.set_state(raw)
                if not np.array_equal(s.get_state(), want):
                    bad.append(i)

    th = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


@pytest.mark.parametrize("N", [5, 37, 129])
def test_snapshot_upload(nsg, N):
    """a field whose increments identify every point's place (N^3 24 bytes: no multiple of a chunk)"""
    u = np.arange(N ** 3 * 3, dtype=np.float64).reshape(N, N, N, 3)
    with nsg.IncrementStats(N) as st:
        st.precompute(u)
        stats = st.results(ranges=False)[0]
    d = [u[1:, :, :, 0] - u[:-1, :, :, 0], u[:, 1:, :, 1] - u[:, :-1, :, 1], u[:, :, 1:, 2] - u[:, :, :-1, 2]]
    assert stats[0][0] == min(x.min() for x in d) and stats[0][1] == max(x.max() for x in d)
