"""Copies between host arrays and device tables (transfer.hip): every byte, at
the sizes where the plain copy gives way to pinned chunks and several threads,
and from several threads at once."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _round_trip(n, seed):
    from solvcon_amd import _lib as L
    from solvcon_amd.onedim import Euler1DCore
    c = Euler1DCore(ncoord=n, time_increment=1e-3)
    a = np.random.default_rng(seed).random((n, 3))
    b = np.zeros_like(a)
    L.check(L.lib().sc1d_upload(c._h, 2, L.dptr(a), a.size))
    L.check(L.lib().sc1d_download(c._h, 2, L.dptr(b), b.size))
    return np.array_equal(a, b)


# 24 bytes a point: 4 MiB is 174762.7 points (down), 32 MiB 1398101.3 (up);
# chunks of 2 MiB, up to four threads.
@pytest.mark.parametrize('n', [5, 87381, 174761, 174763, 174765, 262145,
                               349527, 700001, 1398101, 1398103, 1500001])
def test_round_trip(n):
    print('case: transfer', n, flush=True)
    assert _round_trip(n, n)


def test_round_trip_threads():
    # Ten copies at once: more than the pinned buffers serve.
    print('case: transfer, ten threads', flush=True)
    ok = [False] * 10

    def work(k):
        ok[k] = all(_round_trip(1400001 + 2 * k, 7 * k + r)
                    for r in range(2))
    th = [threading.Thread(target=work, args=(k,)) for k in range(10)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert all(ok)
