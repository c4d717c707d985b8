"""The streamed-tile kernel at each number of query blocks per wave.

Enough planes that the key axis is streamed by work items (not shared out over
a workgroup's waves), with query counts one past a block or an item, with and
without a mask; a few planes against float64.  The weights are hi + lo pairs,
or one fp16 each where the item's own bound keeps the result within rtol 1e-3
and atol 1e-4 of the exact one, which is the tolerance here."""

import math

import pytest
import torch

from vectra_amd.kernels import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('masked', [False, True])
@pytest.mark.parametrize('planes,n_q,n_k,dim', [
    (300, 65, 1025, 64), (350, 129, 1100, 64), (300, 700, 1025, 64),
    (64, 257, 1300, 32), (300, 129, 1300, 32), (64, 257, 300, 128), (300, 129, 300, 128)])
def test_query_blocks_per_wave(planes, n_q, n_k, dim, masked):
    print(planes, n_q, n_k, dim, masked, flush=True)
    gen = torch.Generator(device='cuda').manual_seed(0)
    q, k, v = (torch.randn(planes, 1, n, dim, generator=gen, device='cuda').bfloat16() for n in (n_q, n_k, n_k))
    scale = torch.full((1, 1, 1, 1), 0.7 / dim, device='cuda')
    bias = None
    if masked:
        counts = torch.randint(1, n_k + 1, (planes, 1, 1, 1), generator=gen, device='cuda')
        bias = torch.zeros(planes, 1, 1, n_k, device='cuda')
        bias.masked_fill_(torch.arange(n_k, device='cuda') >= counts, -math.inf)
    got = capi.forward(q, k, v, scale, bias, out_dtype=torch.float32, variant='tile')
    for plane in (0, planes // 2, planes - 1):
        qd, kd, vd = (t[plane, 0].double() for t in (q, k, v))
        d2 = (qd * qd).sum(-1, keepdim=True) + (kd * kd).sum(-1) - 2 * (qd @ kd.T)
        logits = -scale.double().item() * d2
        if masked:
            logits = logits + bias[plane, 0].double()
        torch.testing.assert_close(got[plane, 0].double(), torch.softmax(logits, -1) @ vd, rtol=1e-3, atol=1e-4)
