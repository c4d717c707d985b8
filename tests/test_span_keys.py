"""Long key axes of a few planes with a bias: the kernel whose waves share out the keys.

Sizes at the edges of its key pairs (32 keys), of its waves' rounds (16 pairs,
8 for 128-dim heads), of its query blocks (16 and 32 rows) and of the planes
that are staged whole instead; masks that leave waves without a key; large and
infinite biases and values.

Against float64 over the same 16-bit inputs.  The products and sums are fp32
and the weights hi + lo pairs of 16-bit floats (2^-17 relative at worst, per
weight of a weighted mean), the logits' rounding at most 2^-22 of |q|^2 +
|k|^2 terms below 40 before the exponential: under 1e-4 of the largest value
in all, which the tolerance states."""

import math

import pytest
import torch

from vectra_amd.kernels import capi

pytestmark = pytest.mark.gpu

# Blocks of 32 query rows over all planes: at most one per CU.
SHAPES = [
    # planes, n_q, n_k, dim
    (1, 1, 2000, 64), (2, 16, 609, 64), (1, 17, 1025, 64), (3, 33, 1024, 64), (1, 500, 3000, 64), (8, 700, 611, 64),
    (1, 31, 289, 128), (2, 16, 320, 128), (1, 257, 511, 128), (4, 1000, 1100, 128),
    (1, 16, 1025, 32), (2, 130, 1503, 32), (5, 900, 1537, 32), (1, 4096, 2049, 32), (1, 4097, 1100, 64),
    (8, 1024, 1100, 64), (8, 1000, 301, 128),
]


def _want(q, k, v, scale, bias):
    q, k, v = q.double(), k.double(), v.double()
    d2 = (q * q).sum(-1, keepdim=True) + (k * k).sum(-1)[:, :, None, :] - 2 * (q @ k.transpose(-1, -2))
    logits = -scale.double() * d2.clamp_min(0)
    if bias is not None:
        logits = logits + bias.double()
    return torch.softmax(logits, -1) @ v


def _run(q, k, v, scale, bias):
    dev = [None if t is None else t.cuda() for t in (q, k, v, scale, bias)]
    print(tuple(q.shape), tuple(k.shape), q.dtype, flush=True)
    return capi.forward(*dev, out_dtype=torch.float32, variant='tile').cpu()


def _inputs(planes, n_q, n_k, dim, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(1, planes, n, dim, generator=gen).to(dtype) for n in (n_q, n_k, n_k))
    scale = (0.5 + torch.rand(1, planes, 1, 1, generator=gen)) / dim
    return q, k, v, scale, gen


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16])
@pytest.mark.parametrize('masked', [False, True])
@pytest.mark.parametrize('planes,n_q,n_k,dim', SHAPES)
def test_sizes_at_the_edges(planes, n_q, n_k, dim, masked, dtype):
    q, k, v, scale, gen = _inputs(planes, n_q, n_k, dim, dtype)
    bias = torch.randn(1, planes, 1, n_k, generator=gen).to(dtype)  # a head's own
    if masked:  # most waves see masked keys only
        bias[..., torch.randperm(n_k, generator=gen)[: n_k // 2]] = -math.inf
        bias[..., : min(n_k - 3, 100)] = -math.inf
    torch.testing.assert_close(_run(q, k, v, scale, bias).double(), _want(q, k, v, scale, bias), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize('dim,n_k', [(64, 1200), (128, 700), (32, 1300)])
@pytest.mark.parametrize('kind', ['steps', 'one_key', 'all_masked', 'negative_scale', 'far', 'inf_value', 'nan_masked_key'])
def test_logits_and_values_at_the_limits(kind, dim, n_k):
    q, k, v, scale, _ = _inputs(2, 40, n_k, dim, torch.bfloat16, seed=1)
    bias = torch.zeros(1, 1, 1, n_k)
    if kind == 'steps':  # maxima that rise and fall by more than the shift's step along the axis
        bias = 25 * torch.sin(torch.arange(n_k) / 37.0).reshape(1, 1, 1, n_k)
    elif kind == 'one_key':
        bias[..., :] = -math.inf
        bias[..., n_k - 1] = -5.0
    elif kind == 'all_masked':
        bias[..., :] = -math.inf
    elif kind == 'negative_scale':
        scale = -0.2 * scale
    elif kind == 'far':  # weights far below 1: logits of about -1000
        q = q + 8.0
        k = k - 8.0
        scale = scale * 0 + 4.0 / dim
    elif kind == 'inf_value':
        v[..., 5, 3] = math.inf
    elif kind == 'nan_masked_key':
        k[..., 7, 0] = math.nan
        bias[..., 7] = -math.inf
    got = _run(q, k, v, scale, bias).double()
    if kind == 'all_masked' or kind == 'nan_masked_key':
        assert got.isnan().all()
        return
    if kind == 'negative_scale':
        d2 = ((q.double()[:, :, :, None] - k.double()[:, :, None]) ** 2).sum(-1)
        want = torch.softmax(-scale.double() * d2, -1) @ v.double()
    else:
        want = _want(q, k, v, scale, bias)
    if kind == 'inf_value':  # a weight's lo part may be zero or negative: inf or NaN, in that column alone
        assert not got[..., 3].isfinite().any()
        got, want = (torch.cat([t[..., :3], t[..., 4:]], -1) for t in (got, want))
    # 'far': |q|^2 + |k|^2 of 2 * 64 dim round to 2^-24 of it in the logits,
    # times 4 / dim and log2(e): 64 * 4 * 2 * 2^-22 = 1.2e-4 relative a weight.
    torch.testing.assert_close(got, want, rtol=1e-3 if kind == 'far' else 1e-4, atol=1e-3 if kind == 'far' else 1e-4)


def test_graph_replays_and_strided_rows():
    q, k, v, scale, _ = _inputs(2, 48, 1500, 64, torch.bfloat16, seed=2)
    q, k, v, scale = (t.cuda() for t in (q, k, v, scale))
    bias = torch.linspace(-3, 3, 1500, device='cuda').bfloat16()
    wide = torch.zeros(1, 2, 1500, 136, dtype=torch.bfloat16, device='cuda')
    wide[..., 64:128] = k
    ks = wide[..., 64:128]
    want = torch.ops.vectra.rbf_attention(q, k, v, scale, bias)
    assert torch.equal(torch.ops.vectra.rbf_attention(q, ks, v, scale, bias), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = torch.ops.vectra.rbf_attention(q, ks, v, scale, bias)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
