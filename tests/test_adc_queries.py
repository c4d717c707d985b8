"""The ADC scan of several queries at once, and of codes of at most 8 bytes,
against the oracle, bit for bit: query counts around the shared blocks of two
and four, code widths and alignments, candidate ids, and codes around the
grid's strides."""

import numpy as np
import pytest
import torch

from oracle import scan as oracle
from vectra_amd.index import scan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('m,stride', [(1, 8), (3, 8), (5, 16), (8, 8), (8, 24), (7, 7), (12, 16), (16, 16), (16, 32),
                                      (16, 24), (20, 32), (31, 32), (32, 32)])
@pytest.mark.parametrize('queries', [1, 2, 3, 4, 5, 9])
def test_several_queries_over_short_codes(queries, m, stride):
    rng = np.random.default_rng(queries * 100 + m)
    n = 2049 if queries % 2 else 1023
    tables = rng.random((queries, m * 256), dtype=np.float32) * 8
    tables[0, 3] = np.inf
    codes = rng.integers(0, 256, (n, stride), dtype=np.uint8)
    view = torch.from_numpy(codes).cuda()[:, :m]
    ids = rng.integers(0, n + 40, 777).astype(np.int32)  # some past the codes
    dev = torch.from_numpy(tables).cuda()
    for cand in (None, ids):
        print(f'adc: queries={queries} m={m} stride={stride} ids={cand is not None}', flush=True)
        got = scan.pq_adc_distances(dev, view, ids=None if cand is None else torch.from_numpy(cand).cuda())
        torch.cuda.synchronize()
        want = np.full((queries, n if cand is None else len(cand)), np.nan, np.float32)
        for q in range(queries):
            every = oracle.pq_adc(tables[q], np.ascontiguousarray(codes[:, :m]))
            want[q] = every if cand is None else np.where(cand < n, every[np.minimum(cand, n - 1)], np.nan)
        np.testing.assert_array_equal(got.cpu().numpy().view(np.uint32)[~np.isnan(want)], want.view(np.uint32)[~np.isnan(want)])
        assert np.array_equal(np.isnan(got.cpu().numpy()), np.isnan(want))


def test_a_shard_of_codes_over_several_grid_strides():
    rng = np.random.default_rng(2)
    tables = torch.from_numpy(rng.random((6, 8 * 256), dtype=np.float32)).cuda()
    codes = torch.from_numpy(rng.integers(0, 256, (1_500_001, 8), dtype=np.uint8)).cuda()
    got = scan.pq_adc_distances(tables, codes)
    alone = torch.cat([scan.pq_adc_distances(tables[i:i + 1], codes) for i in range(6)])
    torch.cuda.synchronize()
    assert torch.equal(got, alone)
