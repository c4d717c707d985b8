"""fp32 planes beyond one tile under key masks: 16-key blocks without a key
that counts are skipped, at the block, tile and wave-count boundaries (GPU,
through the C ABI)."""

import math

import pytest
import torch

from oracle import rbf as oracle
from vectra_amd.kernels import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n_q,n_k,dim', [(16, 17, 64), (65, 129, 16), (81, 130, 32), (100, 256, 32), (130, 65, 64),
                                         (257, 300, 64), (33, 97, 128), (300, 161, 128)])
def test_masked_fp32_planes_against_the_float64_chain(n_q, n_k, dim):
    g = torch.Generator().manual_seed(n_q * n_k)
    q, k, v = (torch.randn(3, 2, n, dim, generator=g) for n in (n_q, n_k, n_k))
    scale = (0.5 + torch.rand(1, 2, 1, 1, generator=g)) / dim
    bias = torch.zeros(3, 2, 1, n_k)
    bias[0, ..., n_k // 3:] = -math.inf              # a dead tail
    bias[1, ..., :n_k // 2] = -math.inf              # dead blocks first
    bias[2, 0, :, 1:] = -math.inf                    # one live key
    bias[2, 1] = torch.where(torch.arange(n_k) % 40 < 3, 0.0, -math.inf)
    dev = [t.cuda() for t in (q, k, v, scale, bias)]
    assert capi.select_variant(capi.make_args(*dev[:3], torch.empty_like(dev[0]),
                                              *capi.broadcast_operands(dev[0], dev[1], dev[3], dev[4]), 'mfma')) > 0
    print(f'fp32 masked: {n_q}x{n_k}x{dim}', flush=True)
    got = capi.forward(*dev, variant='mfma')
    torch.cuda.synchronize()
    want = torch.from_numpy(oracle.direct_fp64(q, k, v, scale, bias))
    # The expansion's rounding: gamma (|q|^2 + |k|^2) ~ 3 in sums of `dim` terms.
    torch.testing.assert_close(got.cpu().double(), want, rtol=1e-5, atol=1e-5)
    # The same masks as a finite bias no weight survives: bit for bit.
    kept = capi.forward(*dev[:4], torch.where(dev[4] == -math.inf, torch.tensor(-1e30, device='cuda'), dev[4]),
                        variant='mfma')
    assert torch.equal(kept, got)


def test_non_finite_rows_of_masked_fp32_keys_reach_the_output():
    q, k, v = (torch.randn(1, 3, n, 64) for n in (90, 200, 200))
    bias = torch.zeros(1, 1, 1, 200)
    bias[..., 100:] = -math.inf
    v[0, 0, 180, 7] = math.inf
    k[0, 1, 150, 3] = math.nan
    bias2 = torch.full((1, 3, 1, 200), -math.inf)
    bias2[:, :2] = bias
    out = capi.forward(q.cuda(), k.cuda(), v.cuda(), torch.tensor(0.01).cuda(), bias2.cuda(), variant='mfma').cpu()
    assert bool(out[0, 0, :, 7].isnan().all()) and int(out[0, 0].isnan().sum()) == 90
    assert bool(out[0, 1].isnan().all()) and bool(out[0, 2].isnan().all())


# Both sides of the rule on waves per workgroup for 65-80 rows and beyond, by
# planes and key count, at 256 compute units.
@pytest.mark.parametrize('planes,n_q,n_k,dim', [(150, 65, 90, 64), (160, 80, 90, 64), (330, 80, 130, 64), (520, 65, 130, 64),
                                                (520, 80, 170, 64), (160, 70, 70, 128), (520, 66, 40, 128), (150, 81, 100, 64),
                                                (160, 128, 100, 64), (330, 113, 70, 128)])
def test_many_masked_fp32_planes(planes, n_q, n_k, dim):
    print(planes, n_q, n_k, dim, flush=True)
    g = torch.Generator(device='cuda').manual_seed(planes + n_q)
    q, k, v = (torch.randn(planes, 1, n, dim, generator=g, device='cuda') for n in (n_q, n_k, n_k))
    scale = torch.full((1, 1, 1, 1), 0.9 / dim, device='cuda')
    counts = torch.randint(1, n_k + 1, (planes, 1, 1, 1), generator=g, device='cuda')
    bias = torch.zeros(planes, 1, 1, n_k, device='cuda')
    bias.masked_fill_(torch.arange(n_k, device='cuda') >= counts, -math.inf)
    got = capi.forward(q, k, v, scale, bias, variant='mfma')
    qd, kd, vd = (t[:, 0].double() for t in (q, k, v))
    d2 = (qd * qd).sum(-1)[..., None] + (kd * kd).sum(-1)[:, None] - 2 * (qd @ kd.transpose(1, 2).contiguous())
    want = torch.softmax(bias[:, 0].double() - scale.double().item() * d2, -1) @ vd
    torch.testing.assert_close(got[:, 0].double(), want, rtol=1e-5, atol=1e-5)
