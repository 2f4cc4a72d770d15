"""Transfers of the C API through the client's pinned memory and past it: sizes around its limit of 512 KB, threads that share it."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMIT = (512 << 10) // 4


@pytest.fixture(scope="module")
def session():
    from metalhlo_amd import capi
    s = capi.Session()
    yield s
    s.close()


def _there_and_back(s, x):
    b = s.buffer(x, "f32")
    sent = x.copy()
    x.fill(0)                                             # the caller's memory is its own again
    y = s.to_numpy(b)
    s.lib.mhlo_buffer_destroy(b)
    return np.array_equal(y, sent)


@pytest.mark.parametrize("n", [1, 3, 4096, LIMIT - 1, LIMIT, LIMIT + 1, 3 * LIMIT])
def test_round_trip(session, n):
    for seed in range(3):
        assert _there_and_back(session, np.random.default_rng(seed + n).standard_normal(n).astype(np.float32))


def test_threads_share_the_memory(session):
    bad = []

    def work(i):
        rng = np.random.default_rng(i)
        for n in (LIMIT, 5, LIMIT + 7, 1000, LIMIT - 3) * 4:
            if not _there_and_back(session, rng.standard_normal(n).astype(np.float32)):
                bad.append((i, n))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
