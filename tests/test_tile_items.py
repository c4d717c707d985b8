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


def _long_axis(n_q, n_k, dim):
    """One batch entry on whose near rows one fp16 weight per key holds the
    contract, with row n_q // 2 far from every key: its group of rows (256 for
    64 dims, else 128) takes hi + lo weights as a whole."""
    gen = torch.Generator(device='cuda').manual_seed(n_q + dim)
    q, k = (0.5 * torch.randn(1, 1, n, dim, generator=gen, device='cuda') for n in (n_q, n_k))
    v = 0.25 * torch.randn(1, 1, n_k, dim, generator=gen, device='cuda')
    q[:, :, n_q // 2] += 4.0
    return [t.bfloat16() for t in (q, k, v)] + [torch.full((1, 1, 1, 1), 0.64 / dim, device='cuda')]


@pytest.mark.parametrize('n_q,n_k,dim', [(600, 2048, 64), (64, 1025, 64), (257, 1601, 64), (100, 1200, 64),
                                         (128, 1100, 64), (65, 1100, 64), (60, 1100, 32), (300, 2048, 32), (129, 1100, 32),
                                         (200, 1100, 128)])
@pytest.mark.parametrize('out_dtype', [torch.float32, torch.bfloat16], ids=str)
def test_rows_do_not_depend_on_the_planes_beside_them(n_q, n_k, dim, out_dtype):
    q, k, v, scale = _long_axis(n_q, n_k, dim)
    alone = capi.forward(q, k, v, scale, out_dtype=out_dtype, variant='tile')
    split = capi.forward(q, k, v, scale, out_dtype=torch.float32, variant='tile', split_weights=True)
    assert not alone.isnan().any()
    group = 256 if dim == 64 else 128
    first = n_q // 2 // group * group
    far = slice(first, min(first + group, n_q))
    if out_dtype == torch.float32:
        assert torch.equal(alone[:, :, far], split[:, :, far])
        assert n_q <= group or not torch.equal(alone, split), 'no group kept its fp16 weights'
    for planes in (3, 40, 150, 400, 700):
        print(planes, n_q, n_k, dim, flush=True)
        many = capi.forward(*(t.expand(planes, -1, -1, -1) for t in (q, k, v)), scale, out_dtype=out_dtype, variant='tile')
        assert torch.equal(many, alone.expand_as(many)), planes


def test_keys_padded_on_the_left_take_one_pass():
    """Where the first tiles are masked whole, the shift comes from the first
    that is not: a shift of 0 leaves these weight sums under fp16's range, and
    the planes took three passes (padded on the right: one)."""
    planes, n_q, n_k, dim = 256, 512, 1024, 64
    gen = torch.Generator(device='cuda').manual_seed(0)
    q, k, v = (torch.randn(planes, 1, n, dim, generator=gen, device='cuda').half() for n in (n_q, n_k, n_k))
    scale = torch.full((1, 1, 1, 1), 0.15, device='cuda')
    bias = torch.zeros(planes, 1, 1, n_k, device='cuda')
    bias[..., :200] = -math.inf

    def run(keys, values, mask):
        best = math.inf
        for _ in range(4):
            begin, end = torch.cuda.Event(True), torch.cuda.Event(True)
            begin.record()
            for _ in range(5):
                out = capi.forward(q, keys, values, scale, mask, out_dtype=torch.float32, variant='tile')
            end.record()
            torch.cuda.synchronize()
            best = min(best, begin.elapsed_time(end))
        return out, best

    left, left_ms = run(k, v, bias)
    right, right_ms = run(k.flip(2), v.flip(2), bias.flip(3))
    print(f'padded on the left {left_ms:.3f} ms, on the right {right_ms:.3f} ms', flush=True)
    # The shifts differ, and with them what fp16's last step of 2^-24 cuts from
    # 824 weights of a sum of at least 2^-3: up to 2^-22 of the sum each, as a
    # walk (four deviations of sqrt(824) 2^-22 / sqrt(3)) against |v| < 6.
    torch.testing.assert_close(left, right, rtol=0, atol=1e-4)
    assert left_ms < 1.6 * right_ms
