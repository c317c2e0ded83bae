"""GPU hashes at the edges of the 16-byte column loads: row counts around whole
vectors and block steps, columns that start between two vectors, every kind that
shares the kinds kernel at each way of widening 4-byte columns; against the oracle."""
import numpy as np
import pytest

import oracle
import vjoin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 1023, 1024, 1025, 2051])
@pytest.mark.parametrize("kw,nc,shift", [(8, 1, 0), (8, 3, 1), (4, 1, 1), (4, 2, 3), (4, 4, 2)])
@pytest.mark.parametrize("kind,bits,chunk", [("fnv", 64, 64), ("custom_mult_xor_hw", 64, 32), ("custom_add_hw", 32, 64),
                                             ("custom_n_mult_xor_shift", 64, 64)])
def test_row_counts_and_misaligned_columns(n, kw, nc, shift, kind, bits, chunk):
    import torch
    rng = np.random.default_rng(n * 100 + kw * 10 + nc)
    dt = np.uint32 if kw == 4 else np.uint64
    cols = [rng.integers(0, np.iinfo(dt).max, n + shift, dtype=dt, endpoint=True) for _ in range(nc)]
    dev = [torch.from_numpy(c.view(np.int32 if kw == 4 else np.int64)).cuda()[shift:] for c in cols]
    guard = torch.full((n + 2,), 77, dtype=torch.int32 if bits == 32 else torch.int64, device="cuda")
    vjoin.hash_table(dev, kind, bits, chunk, out=guard[1:n + 1])
    got = guard.cpu().numpy()
    assert got[0] == 77 and got[-1] == 77  # nothing written around the rows
    want = oracle.hash_rows(oracle.reference_rows([c[shift:] for c in cols]), kind, bits, chunk)
    assert np.array_equal(got[1:n + 1].view(np.uint32 if bits == 32 else np.uint64).astype(np.uint64), want)
