"""Edges of single kernels and dispatch branches, against the oracle, bit for bit."""
import numpy as np
import pytest

import gpu_index_test_amd as G
from oracle import oracle_lib as O
from tests.helpers import tiny_index_arrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [8, 13])
def test_bucket_lines_of_every_size(ctx, bits):
    """Buckets of 0 to 9 records, equal, adjacent and apart, up to the bucket's
    ends; every hash, its neighbours and the ends are looked up."""
    rng = np.random.default_rng(bits)
    low = 64 - bits - 9
    ents, keys = [], [0, 1, 2 ** 64 - 1]
    for top in range(2, 250):
        base = top << (64 - bits)
        n = top % 10
        fps = rng.choice([0, 1, 255, 256, 510, 511], size=n) if top % 3 else np.full(n, rng.integers(0, 512))
        hashes = [base | (int(f) << low) | int(rng.choice([0, 1, 2, 3, (1 << low) - 1])) for f in fps]
        ents += [(h, 1000 + 10 * i + top, (top % 5) << 8 | int(rng.integers(0, 60))) for i, h in enumerate(hashes)]
        keys += hashes + [h + 1 for h in hashes] + [h - 1 for h in hashes]
        keys += [base, base + 1, base | (511 << low), base | ((1 << (64 - bits)) - 1)]
    arr, starts = tiny_index_arrays(ents, bits)
    op = O.params_from_read_length(150)
    oidx = O.Index.wrap(arr, starts, bits, 30, op)
    idx = G.StrobemerIndex(None, G.IndexParameters.from_read_length(150))
    idx.upload(arr, starts, bits, 30)
    keys = np.array(keys, dtype=np.uint64)
    assert np.array_equal(idx.find_many(keys), np.array([oidx.find(int(k)) for k in keys], dtype=np.uint64))
    for part in np.array_split(keys, 40):
        q = np.zeros(len(part), dtype=O.QUERY_RANDSTROBE)
        q["hash"], q["start"] = part, np.arange(len(part)) * 2
        q["end"] = q["start"] + 20 + np.arange(len(part)) % 45
        fr, nams = G.find_nams(q, idx)
        efr, enams, _ = O.find_nams(oidx, q, canonical=True)
        assert np.float32(fr).tobytes() == np.float32(efr).tobytes()
        assert nams.tobytes() == enams.tobytes()
    idx.ctx.close()

