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
