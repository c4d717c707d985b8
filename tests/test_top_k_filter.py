"""The filtered form of the k-nearest search (several queries over many
candidates): its results against the oracle and the one-workgroup form, bit
for bit, over query blocks, dimensions, candidate lists, ties, lists that run
over, and values its bounds cannot order; and which calls take it (host
only)."""

import ctypes

import numpy as np
import pytest
import torch

from oracle import scan as oracle
from tests.test_scan_capi import FAKE, _top_k_args
from vectra_amd.index import scan
from vectra_amd.kernels import _native


def _bytes(**over):
    fields = dict(num_queries=64, num_rows=100_000, dimension=128, row_stride=128, query_stride=128, k=10,
                  out_stride=512)
    fields.update(over)
    return _native.scan_library().vectra_scan_top_k_workspace_bytes(ctypes.byref(_top_k_args(**fields)))


def test_calls_that_keep_the_exact_forms():
    assert _bytes() > 0
    # One workgroup per query (no workspace): 64 queries or more.
    for over in (dict(num_rows=2048), dict(num_rows=4095), dict(k=513), dict(dimension=130, row_stride=132), dict(row_stride=129),
                 dict(rows=FAKE + 4), dict(dimension=260, row_stride=260, query_stride=260), dict(dimension=0)):
        assert _bytes(**over) == 0, over
    # The split form's workspace for a few queries (256 + queries * splits * k * 8).
    assert _bytes(num_queries=1) == 256 + 64 * 10 * 8
    assert _bytes(num_queries=3, k=100) == 256 + 3 * 16 * 100 * 8
    assert _bytes(num_queries=0) == 0
    # Small calls of a few queries: 11 x 4,096 pairs and 4 x 32,767.
    assert _bytes(num_queries=11, num_rows=4096) == 256 + 11 * 64 * 10 * 8
    assert _bytes(num_queries=4, num_rows=32_767) == 256 + 4 * 64 * 10 * 8
    assert _bytes(num_queries=12, num_rows=4096) > 100_000 < _bytes(num_queries=4, num_rows=32_768)
    # The filtered form's grows with the queries and stays modest.
    assert _bytes(num_queries=4) < 16 << 20 and _bytes(num_queries=1024, k=100) < 64 << 20


@pytest.mark.parametrize('n_q', [2000, 65_536, 100_000, 1_000_000, 20_000_000])
@pytest.mark.parametrize('k', [1, 10, 100, 512])
def test_the_workspace_of_many_queries_is_bounded(n_q, k):
    for rows in (8192, 100_000, 500_000):
        assert 0 < _bytes(num_queries=n_q, k=k, num_rows=rows) <= 64 << 20, rows


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _check(queries, rows, k, ids=None, against_oracle=True):
    q, r, i = _gpu(queries), _gpu(rows), None if ids is None else _gpu(ids.astype(np.int32))
    args, _keep, _d, _n = scan._top_k_args(q, r, k, i, None)  # pylint: disable=protected-access
    need = _native.scan_library().vectra_scan_top_k_workspace_bytes(ctypes.byref(args))
    groups = 256 + -(-queries.shape[0] // 64) * 64 * 4  # more than any split form of these calls needs
    assert need > groups, 'the filtered form is not taken'
    workspace = torch.randint(0, 256, (need,), dtype=torch.uint8, device='cuda')
    workspace[:256] = 0
    d, n = scan.nearest(q, r, k, i, workspace=workspace)
    d1, n1 = scan.nearest(q, r, k, i, form='single')
    torch.cuda.synchronize()
    assert not workspace[:256].any()
    assert torch.equal(n.view(torch.int32), n1.view(torch.int32))
    assert torch.equal(d.view(torch.int32), d1.view(torch.int32))
    if against_oracle:
        want_d, want_n = oracle.nearest(queries, rows, k, ids)
        np.testing.assert_array_equal(n.cpu().numpy(), want_n)
        np.testing.assert_array_equal(d.cpu().numpy().view(np.uint32), want_d.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize('n_q,n,dim,k', [(4, 33_000, 128, 10), (5, 26_215, 64, 1), (16, 4111, 4, 100), (17, 5000, 96, 37),
                                         (63, 6000, 100, 10), (64, 8192, 128, 512), (65, 9001, 256, 50),
                                         (130, 4200, 36, 100), (300, 4999, 132, 7)])
def test_filtered_search_against_the_oracle(n_q, n, dim, k):
    rng = np.random.default_rng(n + dim)
    _check(rng.standard_normal((n_q, dim)).astype(np.float32), rng.standard_normal((n, dim)).astype(np.float32), k)


@pytest.mark.gpu
@pytest.mark.parametrize('n_q,n,dim,k', [(64, 200_000, 128, 100), (9, 100_003, 64, 10), (1024, 12_500, 128, 100)])
def test_filtered_search_at_large_sizes(n_q, n, dim, k):
    rng = np.random.default_rng(n)
    _check(rng.standard_normal((n_q, dim)).astype(np.float32), rng.standard_normal((n, dim)).astype(np.float32), k,
           against_oracle=False)


@pytest.mark.gpu
@pytest.mark.parametrize('n_q,n,dim,k', [(3001, 20_000, 32, 512), (7000, 6500, 64, 400)])
def test_filtered_search_in_parts(n_q, n, dim, k):
    """More queries than the workspace's bound holds at once: two and four parts."""
    rng = np.random.default_rng(n_q)
    _check(rng.standard_normal((n_q, dim)).astype(np.float32), rng.standard_normal((n, dim)).astype(np.float32), k,
           against_oracle=False)


@pytest.mark.gpu
@pytest.mark.parametrize('dim', [64, 160])
def test_filtered_search_with_candidate_ids(dim):
    rng = np.random.default_rng(dim)
    rows = rng.standard_normal((3000, dim)).astype(np.float32)
    ids = rng.integers(0, 3100, 9000)  # repeats, and ids past the rows
    _check(rng.standard_normal((20, dim)).astype(np.float32), rows, 60, ids)
    _check(rng.standard_normal((13, dim)).astype(np.float32), rows, 10, np.full(5000, 3000))  # none valid


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['equal', 'two_values', 'clusters', 'offset', 'nan', 'inf', 'huge', 'tiny', 'nan_query',
                                  'zeros'])
def test_filtered_search_where_bounds_are_weak(kind):
    """Ties and clusters run lists over; a large common offset, NaN, infinite,
    overflowing and underflowing values leave bounds that order nothing."""
    rng = np.random.default_rng(3)
    n, dim = 8000, 128
    rows = rng.standard_normal((n, dim)).astype(np.float32)
    q = rng.standard_normal((12, dim)).astype(np.float32)
    if kind == 'equal':
        rows[:] = rows[0]
    elif kind == 'two_values':
        rows[::2], rows[1::2] = rows[0], rows[1]
    elif kind == 'clusters':  # runs of near-copies, the queries among them
        rows = (rows[np.arange(n) // 500] + 1e-3 * rows).astype(np.float32)
        q = (rows[rng.integers(0, n, 12)] + 1e-3).astype(np.float32)
    elif kind == 'offset':
        rows, q = rows + np.float32(300), q + np.float32(300)
    elif kind == 'nan':
        rows[rng.integers(0, n, 50), 3] = np.nan
        rows[7000:] = np.nan
    elif kind == 'inf':
        rows[::3, 5] = np.inf
        q[0, 5] = np.inf
    elif kind == 'huge':  # squares overflow; bf16 rounds 3.4e38 up to infinity
        rows[::2] *= np.float32(1e19)
        rows[5] = np.float32(3.4e38)
        q[1] *= np.float32(1e19)
    elif kind == 'tiny':  # squares underflow
        rows *= np.float32(1e-25)
        q *= np.float32(1e-25)
    elif kind == 'nan_query':
        q[2, 0] = np.nan
    elif kind == 'zeros':
        rows[:] = 0
        q[3] = 0
    print(f'weak bounds: {kind}', flush=True)
    with np.errstate(over='ignore', invalid='ignore', under='ignore'):
        _check(q, rows, 40)


@pytest.mark.gpu
@pytest.mark.parametrize('n_q,n,dim,k,shift', [(4, 33_000, 128, 10, 8), (65, 9001, 100, 50, 3), (20, 5000, 36, 37, 1e4),
                                               (17, 6000, 256, 10, 1e6), (200, 4111, 4, 100, -40)])
def test_filtered_search_about_a_centre(n_q, n, dim, k, shift):
    """Rows and queries far from the origin for their spread: bounds from the
    queries' mean, at shifts whose rounding is far above the spread too; a
    query that lies elsewhere, and rows that do."""
    rng = np.random.default_rng(n + dim)
    q = (rng.standard_normal((n_q, dim)) + shift).astype(np.float32)
    rows = (rng.standard_normal((n, dim)) + shift).astype(np.float32)
    _check(q, rows, k)
    q[n_q - 1] = -q[n_q - 1]
    rows[::5] -= np.float32(shift)
    _check(q, rows, k)
    _check(np.repeat(q[:1], n_q, axis=0), rows, k)


@pytest.mark.gpu
def test_a_smaller_workspace_takes_the_exact_forms():
    rng = np.random.default_rng(9)
    rows, q = _gpu(rng.standard_normal((20_000, 128)).astype(np.float32)), _gpu(
        rng.standard_normal((8, 128)).astype(np.float32))
    want = scan.nearest(q, rows, 20, form='single')
    for size in (256, 256 + 8 * 64 * 20 * 8, scan.workspace_bytes(q, rows, 20)):
        got = scan.nearest(q, rows, 20, workspace=torch.zeros(size, dtype=torch.uint8, device='cuda'))
        torch.cuda.synchronize()
        assert all(torch.equal(a.view(torch.int32), b.view(torch.int32)) for a, b in zip(got, want)), size


@pytest.mark.gpu
@pytest.mark.parametrize('k', [10, 200])
def test_lists_that_keep_their_smallest_keys(k):
    """The nearest candidates in one or two workgroups' shares: their lists run
    over, and what they left out is among the k nearest; equal keys of one node
    beyond a list's slots; equal distances of many nodes."""
    rng = np.random.default_rng(k)
    n, dim = 9000, 64
    q = rng.standard_normal((16, dim)).astype(np.float32)
    rows = rng.standard_normal((n, dim)).astype(np.float32)
    ahead = rows[np.argsort(((rows - q[3]) ** 2).sum(1))]
    for name, data, ids in (('sorted', ahead, None), ('reversed', ahead[::-1].copy(), None),
                            ('one_node', rows, np.full(6000, 7)), ('few_nodes', rows, rng.integers(0, 5, 6000)),
                            ('runs', rows[np.arange(n) // 300], None), ('runs_of_ids', rows, np.arange(9000) // 40)):
        print(name, k, flush=True)
        _check(q, data, k, ids)


def _times(q, rows, k):
    """Milliseconds of five calls, filtered and with one workgroup per query."""
    workspace = torch.zeros(scan.workspace_bytes(q, rows, k), dtype=torch.uint8, device='cuda')

    def time(**kw):
        best = float('inf')
        for _ in range(4):
            begin, end = torch.cuda.Event(True), torch.cuda.Event(True)
            begin.record()
            for _ in range(5):
                scan.nearest(q, rows, k, **kw)
            end.record()
            torch.cuda.synchronize()
            best = min(best, begin.elapsed_time(end))
        return best

    return time(workspace=workspace), time(form='single')


@pytest.mark.gpu
@pytest.mark.parametrize('kind', ['equal', 'two_values'])
def test_ties_cost_no_multiple_of_the_exact_search(kind):
    """Every list of every query runs over: without its smallest keys each
    query's candidates were computed again by one workgroup, five times the
    exact form's time in all."""
    gen = torch.Generator(device='cuda').manual_seed(1)
    rows = torch.randn(60_000, 128, generator=gen, device='cuda')
    q = torch.randn(64, 128, generator=gen, device='cuda')
    rows[:] = rows[:1] if kind == 'equal' else rows[:2].repeat(30_000, 1)
    filtered, exact = _times(q, rows, 100)
    print(f'{kind}: filtered {filtered:.3f} ms, exact {exact:.3f} ms', flush=True)
    assert filtered < 2.5 * exact


@pytest.mark.gpu
def test_a_shift_costs_less_than_the_exact_search():
    """Bounds from the origin let most pairs pass where rows and queries share
    an offset of 8 deviations an element: 1.2 ms against the exact form's 0.54."""
    gen = torch.Generator(device='cuda').manual_seed(1)
    rows = torch.randn(50_000, 96, generator=gen, device='cuda') + 8
    q = torch.randn(256, 96, generator=gen, device='cuda') + 8
    filtered, exact = _times(q, rows, 10)
    print(f'filtered {filtered:.3f} ms, exact {exact:.3f} ms', flush=True)
    assert filtered < exact
