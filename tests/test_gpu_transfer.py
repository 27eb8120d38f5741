"""Host arrays through the library's pinned chunks: sizes around the chunk,
slot and thread limits come back unchanged, also from several threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32


def _round_trip(mg, n, seed):
    M = np.random.default_rng(seed).standard_normal(3 * n).astype(F)
    with mg.Film(n, 1, 1, F(5e-9), F(5e-9), F(5e-9), demag=0) as f:
        for k in range(2):
            f.set_m(M)
            assert np.array_equal(f.get_m(), M)
            M = -M


# 12 bytes a cell: the runtime's copy and the first chunked one, an odd size, both sides of the threads' line, chunks
# that do not divide the array, more chunks than slots
@pytest.mark.parametrize("n", [1, 131071, 131072, 200001, 1048575, 1048576, 1500003, 3000001])
def test_round_trip(mg, n):
    _round_trip(mg, n, n)


def test_round_trips_of_several_threads(mg):
    errors = []

    def work(k):
        try:
            _round_trip(mg, 1100000 + 7 * k, k)
        except BaseException as e:
            errors.append(e)
    th = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors, errors[0]
