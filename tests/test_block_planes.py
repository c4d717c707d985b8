"""16-bit planes beyond one tile with a key bias or query counts that split
unevenly: planes staged whole in LDS (up to 160 KB: 288 to 1,024 keys by head
width) and streamed key tiles, at the sizes where the staging, the key pairs,
the waves and the work items end (GPU, through the C ABI)."""

import math

import pytest
import torch

from oracle import rbf as oracle
from vectra_amd.kernels import capi

pytestmark = pytest.mark.gpu

GATE = {'rtol': 1e-3, 'atol': 1e-4}
LOWEST = torch.finfo(torch.float32).min


def _inputs(batch, heads, n_q, n_k, dim, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(batch, n, heads, dim, generator=g).to(dtype).transpose(1, 2) for n in (n_q, n_k, n_k))
    scale = (0.5 + torch.rand(1, heads, 1, 1, generator=g)) / dim
    counts = torch.randint(1, n_k + 1, (batch, 1, 1, 1), generator=g)
    bias = torch.zeros(batch, 1, 1, n_k).masked_fill(torch.arange(n_k) >= counts, -math.inf)
    return q, k, v, scale, bias


def _run(q, k, v, scale, bias, variant='tile'):
    # Head-transposed views keep their strides on the device.
    dev = [t.transpose(1, 2).contiguous().cuda().transpose(1, 2) for t in (q, k, v)]
    got = capi.forward(*dev, scale.cuda(), None if bias is None else bias.cuda(), out_dtype=torch.float32,
                       variant=variant)
    torch.cuda.synchronize()
    return got.cpu().double()


# Keys are staged in pairs of 16.  64 dims: 608 keys fit (4 waves up to 128, 8 up
# to 288, 16 above); 32 dims: all up to 1,024; 128 dims: 288.  Longer planes stream.
@pytest.mark.parametrize('n_q,n_k,dim', [(16, 1, 64), (17, 31, 64), (33, 32, 64), (81, 33, 64), (100, 150, 64),
                                         (257, 257, 64), (65, 315, 64), (20, 608, 64), (130, 641, 64), (300, 1023, 64),
                                         (18, 81, 32), (129, 300, 32), (260, 1000, 32), (40, 1024, 32), (70, 1030, 32),
                                         (16, 40, 128), (90, 130, 128), (33, 288, 128), (140, 330, 128)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=str)
def test_masked_planes_against_the_float64_chain(n_q, n_k, dim, dtype):
    q, k, v, scale, bias = _inputs(2, 3, n_q, n_k, dim, dtype, n_q + n_k)
    print(f'masked planes: {n_q}x{n_k}x{dim} {dtype}', flush=True)
    want = torch.from_numpy(oracle.direct_fp64(q, k, v, scale, bias))
    torch.testing.assert_close(_run(q, k, v, scale, bias), want, **GATE)
    # Dead key pairs are skipped: a finite bias no weight survives keeps them.
    kept = torch.where(bias == -math.inf, torch.tensor(-1e30), bias)
    torch.testing.assert_close(_run(q, k, v, scale, kept), want, **GATE)


@pytest.mark.parametrize('n_k,dim', [(200, 64), (700, 64), (150, 32), (200, 128), (400, 128)])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=str)
@pytest.mark.parametrize('case', ['additive', 'large', 'rising', 'first_masked', 'negative_scale', 'far', 'lowest'])
def test_biases_that_move_the_shift(case, n_k, dim, dtype):
    """Weights shifted by the first keys' largest logits: biases around 0, far
    from 0, rising along the keys (the range check then fails and the exact
    passes run), with the first keys masked, gamma < 0, far points, and a mask
    of the type's lowest value."""
    q, k, v, scale, _ = _inputs(2, 2, 40, n_k, dim, dtype, n_k)
    g = torch.Generator().manual_seed(5)
    bias = torch.zeros(2, 2, 1, n_k)
    if case == 'additive':
        bias = torch.randn(2, 2, 1, n_k, generator=g)
    elif case == 'large':
        bias = 40 * torch.randn(2, 2, 1, n_k, generator=g)
    elif case == 'rising':
        bias = torch.linspace(-60, 60, n_k).expand(2, 2, 1, n_k)
    elif case == 'first_masked':
        bias[..., : n_k // 2] = -math.inf
    elif case == 'negative_scale':
        scale = -scale / 8
    elif case == 'far':
        q, k, scale = (3 * q.float()).to(dtype), (3 * k.float()).to(dtype), torch.full_like(scale, 0.3)
    elif case == 'lowest':
        bias[..., n_k // 3:] = LOWEST
    print(f'shift: {case} {n_k}x{dim} {dtype}', flush=True)
    want = torch.from_numpy(oracle.direct_fp64(q, k, v, scale, bias))
    got = _run(q, k, v, scale, bias.contiguous())
    generic = _run(q, k, v, scale, bias.contiguous(), 'generic')
    # Logits of hundreds carry 2^-24 of themselves into the weights: as far
    # from float64 as four times the general path is, where that is more.
    allow = GATE['atol'] + GATE['rtol'] * want.abs() + 4 * (generic - want).abs().amax()
    assert bool(((got - want).abs() <= allow).all())


@pytest.mark.parametrize('n_k,dim', [(200, 64), (700, 64), (100, 32)])
def test_planes_without_a_live_key_and_non_finite_masked_rows(n_k, dim):
    q, k, v, scale, bias = _inputs(3, 2, 50, n_k, dim, torch.bfloat16, 3)
    bias[:] = 0
    bias[1] = -math.inf            # no live key: NaN
    bias[2, ..., 40:] = -math.inf
    v[2, 0, n_k - 1, 5] = math.inf  # 0 times inf: that value dim is NaN
    k[2, 1, n_k - 2, 0] = math.nan  # a NaN distance: every row is NaN
    got = _run(q, k, v, scale, bias)
    assert bool(got[1].isnan().all()) and not bool(got[0].isnan().any())
    assert bool(got[2, 0, :, 5].isnan().all()) and int(got[2, 0].isnan().sum()) == 50
    assert bool(got[2, 1].isnan().all())


@pytest.mark.parametrize('n_q,n_k,dim,later', [(40, 257, 64, 200), (300, 300, 32, 299), (33, 150, 128, 40),  # staged whole
                                               (40, 1200, 64, 512), (20, 1500, 32, 1030), (50, 400, 128, 256)])  # shared out
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=str)
def test_what_the_split_drops_of_a_dominant_weight_drops_out(n_q, n_k, dim, later, dtype):
    """Two live keys, the later one 120 times the weight the shift is taken
    from: its hi + lo pair is 2^-17 off in bf16, and the sum it is divided by
    holds the same pair.  Left: the fp32 roundings of the products, sums, the
    reciprocal and its product (under 8 of 2^-24, the parts up to the values'
    largest), and the logits' 2^-20 in the lighter key's hundredth."""
    q, k, v, scale, _ = _inputs(2, 2, n_q, n_k, dim, dtype, 11)
    b = torch.full((1, 1, 1, n_k), -math.inf)
    b[..., 0], b[..., later] = 0.0, 4.8
    got = _run(q, k, v, scale / 8, b)
    want = torch.from_numpy(oracle.direct_fp64(q, k, v, scale / 8, b))
    print(n_q, n_k, dim, dtype, float((got - want).abs().max()), flush=True)
    torch.testing.assert_close(got, want, rtol=0, atol=8 * 2 ** -24 * float(v.float().abs().max()))


# A launch holds fewer than 2^32 threads: 2^22 workgroups of 16 waves, 2^24 of 4.
@pytest.mark.parametrize('planes,n_k', [((1 << 22) + 5, 640), ((1 << 24) + 3, 81)])
def test_more_planes_than_one_launch_holds(planes, n_k):
    print(planes, n_k, flush=True)
    q, k, v, scale = (t.contiguous().cuda() for t in _inputs(1, 1, 16, n_k, 32, torch.bfloat16, n_k)[:4])
    bias = torch.zeros(planes, 1, 1, 1, dtype=torch.bfloat16, device='cuda')
    bias[-1] = 1.0  # one value for all keys of a plane: no effect on its result
    one = capi.forward(q, k, v, scale, bias[:1].expand(1, 1, 1, n_k))
    out = torch.zeros(planes, 1, 16, 32, dtype=torch.bfloat16, device='cuda')
    capi.forward(*(t.expand(planes, 1, -1, -1) for t in (q, k, v)), scale, bias.expand(planes, 1, 1, n_k), out=out)
    torch.cuda.synchronize()
    assert torch.equal(out[:-1], one.expand(planes - 1, 1, 16, 32))
    torch.testing.assert_close(out[-1].float(), one[0].float(), rtol=2 ** -8, atol=1e-4)


# Many planes: one workgroup per plane (32 dims: 8 and 16 waves, 64 dims: 4, 8
# and 16, 128 dims: 8 and 16) whose waves take a second and a third query
# block; without a bias the longer ones are streamed.
@pytest.mark.parametrize('planes,n_q,n_k,dim', [(1100, 65, 100, 64), (1100, 129, 100, 64), (600, 129, 257, 64),
                                                (600, 257, 257, 64), (600, 257, 500, 64), (600, 513, 300, 64),
                                                (300, 250, 600, 64), (600, 129, 300, 32), (600, 257, 1000, 32),
                                                (1000, 100, 600, 32), (600, 129, 140, 128), (600, 257, 200, 128),
                                                (1000, 100, 180, 128)])
@pytest.mark.parametrize('masked', [False, True])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=str)
def test_many_planes_against_float64(planes, n_q, n_k, dim, masked, dtype):
    print(planes, n_q, n_k, dim, masked, dtype, flush=True)
    g = torch.Generator(device='cuda').manual_seed(n_q + n_k)
    q, k, v = (torch.randn(planes, 1, n, dim, generator=g, device='cuda').to(dtype) for n in (n_q, n_k, n_k))
    scale = torch.full((1, 1, 1, 1), 0.9 / dim, device='cuda')
    bias = torch.zeros(planes, 1, 1, n_k, device='cuda')
    if masked:
        counts = torch.randint(1, n_k + 1, (planes, 1, 1, 1), generator=g, device='cuda')
        bias.masked_fill_(torch.arange(n_k, device='cuda') >= counts, -math.inf)
    got = capi.forward(q, k, v, scale, bias if masked else None, out_dtype=torch.float32, variant='tile')
    for at in (slice(0, 1), slice(planes // 2, planes // 2 + 1), slice(planes - 1, planes)):
        qd, kd, vd = (t[at, 0].double() for t in (q, k, v))
        d2 = (qd * qd).sum(-1)[..., None] + (kd * kd).sum(-1)[:, None] - 2 * (qd @ kd.transpose(1, 2).contiguous())
        want = torch.softmax(bias[at, 0].double() - scale.double().item() * d2, -1) @ vd
        torch.testing.assert_close(got[at, 0].double(), want, **GATE)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float16], ids=str)
def test_planes_that_leave_cus_unequal_are_streamed(dtype):
    """1,000 planes, four workgroups on most CUs: streamed without a bias in 0.6
    of the time that the workgroups take with one of zeros."""
    g = torch.Generator(device='cuda').manual_seed(0)
    q, k, v = (torch.randn(1000, 1, n, 32, generator=g, device='cuda').to(dtype) for n in (100, 1000, 1000))
    scale = torch.full((1, 1, 1, 1), 0.03, device='cuda')
    times = {}
    for name, bias in (('none', None), ('zeros', torch.zeros(1, 1, 1, 1000, device='cuda'))):
        times[name] = math.inf
        for _ in range(5):
            begin, end = torch.cuda.Event(True), torch.cuda.Event(True)
            begin.record()
            for _ in range(5):
                capi.forward(q, k, v, scale, bias, variant='tile')
            end.record()
            torch.cuda.synchronize()
            times[name] = min(times[name], begin.elapsed_time(end))
    print(times, flush=True)
    assert times['none'] < 0.8 * times['zeros']
