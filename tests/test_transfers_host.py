"""The packed transfers around a run keep every array's values, type and
shape: odd and empty sizes, results on both sides of the packing limit, and
results that own their memory.  Exact."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,shape,edge", [(0, (1, 1), (32, 32)), (3, (5, 7), (2, 32, 32)), (8, (362, 363), (64, 64))])
def test_packed_transfers_round_trip(n, shape, edge):
    from py4dstem_amd.ptychography import _PACK_BYTES, download, upload
    rng = np.random.default_rng(1)
    z = lambda s: (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)
    host = [rng.integers(0, 99, (max(n, 1), 11)).astype(np.int32), rng.standard_normal(max(n, 1)), None,
            (rng.random(shape) > 0.5).astype(np.uint8), z(edge)]
    dev = upload(torch.device("cpu"), host)
    for a, t in zip(host, dev):
        assert (a is None and t is None) or (np.array_equal(t.numpy(), a) and t.is_contiguous()
                                             and t.numpy().dtype == a.dtype)
    results = [torch.from_numpy(rng.standard_normal(n)), torch.from_numpy(z(shape)),
               torch.from_numpy(rng.standard_normal((shape[0], 3)).astype(np.float32)), torch.from_numpy(z(edge))]
    assert (results[1].numel() * 8 > _PACK_BYTES) == (shape[0] == 362)
    back = download(results)
    for t, a in zip(results, back):
        assert a.dtype == t.numpy().dtype and np.array_equal(a, t.numpy()) and a.flags.writeable
    back[3][...] = 0  # no two results share an element
    assert np.array_equal(back[0], results[0].numpy()) and np.array_equal(back[2], results[2].numpy())
