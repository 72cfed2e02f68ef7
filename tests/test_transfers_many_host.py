"""The packed transfer of many small results."""

import time

import numpy as np
import pytest

torch = pytest.importorskip("torch")


def test_time_grows_with_the_number_of_results():
    """Ten times the results take about ten times as long (a search of a list
    for each of them made it 60 times here)."""
    from py4dstem_amd.ptychography import download

    def best(n):
        tensors = [torch.full((2,), float(i)) for i in range(n)]
        times = []
        for _ in range(3):
            start = time.perf_counter()
            back = download(tensors)
            times.append(time.perf_counter() - start)
        assert all(np.array_equal(b, [i, i]) for i, b in enumerate(back))
        return min(times)

    best(10)
    assert best(30000) < 30 * best(3000)


def test_a_kept_result_holds_a_bounded_buffer():
    from py4dstem_amd import ptychography as P
    tensors = [torch.full((200, 300), float(i)) for i in range(150)] + [torch.zeros(0), torch.ones(3)]
    back = P.download(tensors)

    def held(a):
        while isinstance(a.base, np.ndarray):
            a = a.base
        return a.nbytes

    assert sum(a.nbytes for a in back) > 2 * 16 * 2 ** 20
    assert max(held(a) for a in back) <= 16 * 2 ** 20 + 8 * len(back)
    for a, t in zip(back, tensors):
        np.testing.assert_array_equal(a, t.numpy())
