"""Few query rows over more than one key tile: which kernel serves them (host
only), and the split stream kernel's results at the sizes where its tiles,
waves and merges meet (GPU, through the C ABI)."""

import pytest
import torch

from oracle import rbf as oracle
from tests.test_capi import _fake_args
from vectra_amd.kernels import capi


@pytest.mark.parametrize('dtype,dim', [(torch.bfloat16, 64), (torch.float16, 128), (torch.float32, 32),
                                       (torch.float32, 64), (torch.float32, 128)])
@pytest.mark.parametrize('n_k', [64, 65, 1000])
def test_every_head_width_streams_long_key_axes(dtype, dim, n_k):
    a = _fake_args(dtype=dtype, n_q=3, n_k=n_k, d=dim, dv=dim)
    assert capi.VARIANT_NAMES[capi.select_variant(a)] == 'stream'
    # Forms the kernel cannot address stay with the generic kernel.
    for name, value in (('k_stride', dim + 1), ('v_stride', -dim), ('k_stride', 1 << 30)):
        a = _fake_args(dtype=dtype, n_q=3, n_k=n_k, d=dim, dv=dim)
        getattr(a, name)[2] = value
        assert capi.VARIANT_NAMES[capi.select_variant(a)] == 'generic', (name, value)
    a = _fake_args(dtype=dtype, n_q=3, n_k=0, d=dim, dv=dim)
    assert capi.select_variant(a) > 0


# (batch, heads, n_q, n_k): 1 to 16 waves per row, rows that do not fill the
# last workgroup or the 8 XCDs, key counts around tiles of 4 to 64 keys.
SHAPES = [(1, 1, 1, 65), (1, 2, 1, 2048), (1, 3, 15, 129), (3, 7, 1, 127), (2, 5, 3, 1000), (700, 3, 1, 67),
          (2051, 1, 1, 96), (150, 2, 1, 513)]


@pytest.mark.gpu
@pytest.mark.parametrize('shape', SHAPES, ids=str)
@pytest.mark.parametrize('dtype,dim', [(torch.bfloat16, 16), (torch.bfloat16, 64), (torch.float16, 128),
                                       (torch.float32, 16), (torch.float32, 128)], ids=str)
def test_split_rows_against_the_float64_chain(shape, dtype, dim):
    batch, heads, n_q, n_k = shape
    gen = torch.Generator().manual_seed(n_k + dim)
    q, k, v = (torch.randn(batch, heads, n, dim, generator=gen).to(dtype) for n in (n_q, n_k, n_k))
    scale = (0.5 + torch.rand(1, heads, 1, 1, generator=gen)) / dim
    # Padding by -inf in most rows, by the type's lowest value in others (all
    # keys of the last batch entry: every key then weighs by its distance).
    counts = torch.randint(1, n_k + 1, (batch, 1, 1, 1), generator=gen)
    masked = torch.arange(n_k) >= counts
    lowest = (torch.arange(batch) % 3 == 1)[:, None, None, None]
    bias = torch.zeros(batch, 1, 1, n_k)
    bias = torch.where(masked & lowest, torch.finfo(torch.float32).min, bias)
    bias = torch.where(masked & ~lowest, float('-inf'), bias)
    bias[-1] = torch.finfo(torch.float32).min if batch > 1 else 0.0
    dev = [t.cuda() for t in (q, k, v, scale, bias)]
    out = torch.empty(batch, heads, n_q, dim, device='cuda')
    scale4, bias4 = capi.broadcast_operands(dev[0], dev[1], dev[3], dev[4])
    assert capi.VARIANT_NAMES[capi.select_variant(capi.make_args(*dev[:3], out, scale4, bias4))] == 'stream'
    got = capi.forward(*dev, out_dtype=torch.float32)
    torch.cuda.synchronize()
    # The distances enter a lowest-value bias below its last place, so that
    # row is the plain mean in 32 bits: 0 in the chain's bias gives it too.
    want_bias = bias.clone()
    want_scale = scale.expand(batch, heads, 1, 1).clone()
    if batch > 1:
        want_bias[-1] = 0.0
        want_scale[-1] = 0.0
    want = torch.from_numpy(oracle.direct_fp64(q, k, v, want_scale, want_bias))
    # Derived: the weights' exponents carry gamma (|q|^2 + |k|^2) ~ 3 of
    # 2^-24 each (sums of `dim` terms: a few units more), so every weight is
    # within ~2^-19 of itself and the weighted mean within that of max |v| ~ 5.
    torch.testing.assert_close(got.cpu().double(), want, rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
def test_split_rows_without_a_live_key_are_nan():
    q, k, v = (torch.randn(2, 2, n, 64, device='cuda').bfloat16() for n in (1, 300, 300))
    bias = torch.zeros(2, 1, 1, 300, device='cuda')
    bias[1] = float('-inf')
    out = torch.ops.vectra.rbf_attention(q, k, v, torch.tensor(0.01, device='cuda'), bias)
    torch.cuda.synchronize()
    assert bool(out[1].isnan().all()) and not bool(out[0].isnan().any())


@pytest.mark.gpu
@pytest.mark.parametrize('rows', [4, 4096])  # 16 waves and one wave per row
def test_split_rows_of_equal_keys_are_exact(rows):
    """Every weight is exactly 1, so sums and counts are whole numbers and each
    result is their exact quotient (a product with the rounded reciprocal of
    49 or 93 keys is not)."""
    off = []
    for n_k in (65, 93, 98, 123, 161, 186, 196, 333, 509):
        q = torch.ones(rows, 1, 1, 64, device='cuda')
        k = torch.ones(rows, 1, n_k, 64, device='cuda')
        v = torch.full((rows, 1, n_k, 64), 3.0, device='cuda')
        got = torch.ops.vectra.rbf_attention(q, k, v, torch.tensor(0.5, device='cuda'), None)
        torch.cuda.synchronize()
        if not bool((got == 3.0).all()):
            off.append(n_k)
    assert not off


def _milliseconds(call):
    best = float('inf')
    for _ in range(5):
        begin, end = torch.cuda.Event(True), torch.cuda.Event(True)
        begin.record()
        for _ in range(5):
            call()
        end.record()
        torch.cuda.synchronize()
        best = min(best, begin.elapsed_time(end))
    return best


@pytest.mark.gpu
def test_the_rows_of_a_plane_share_its_keys():
    """15 rows per plane against the same rows with a plane each, which reads 15
    times the bytes: in one order the rows find their tiles in the caches (0.45
    of the time; 0.73 where each walked them in an order of its own)."""
    gen = torch.Generator(device='cuda').manual_seed(0)
    q = torch.randn(30_000, 1, 1, 64, generator=gen, device='cuda')
    k, v = (torch.randn(30_000, 1, 300, 64, generator=gen, device='cuda') for _ in range(2))
    scale = torch.full((1, 1, 1, 1), 0.02, device='cuda')
    shared = _milliseconds(lambda: capi.forward(q.view(2000, 1, 15, 64), k[:2000], v[:2000], scale, variant='stream'))
    alone = _milliseconds(lambda: capi.forward(q, k, v, scale, variant='stream'))
    print(f'15 rows a plane {shared:.3f} ms, one {alone:.3f} ms', flush=True)
    assert shared < 0.6 * alone
