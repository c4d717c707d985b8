"""Performance cases of the framework's two device paths.

* ``torch.ops.vectra.rbf_attention`` (kind 'attention'): one attention layer's
  call, in the shapes a price model and its relatives hand it.  Inputs are
  resident on the GPU, as they are inside a model's forward pass.
* ``vectra_amd.index.scan`` (kinds 'nearest' and 'pq'): the retrieval engine's
  exhaustive k-nearest search and its product-quantised scan over a resident
  shard.

An attention case gives the sizes, the element type, the layout of q, k and v
('contiguous': tensors of their own; 'fused': head-transposed views of one
qkv projection, as a self-attention layer makes them) and the smallest number
of valid keys of a batch entry (0: no mask).  Padded keys carry a -inf key
bias in the element type, [B, 1, 1, Nk].  Head widths are those of the
configurations and of larger models (16, 32, 64, 128).
"""

import math

import torch

from vectra_amd.index import scan
from vectra_amd.kernels import custom_ops  # noqa: F401  (registers the operator)

DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
PQ_CENTROIDS = 256


def _attention(name, batch, heads, n_q, n_k, dim, dtype, valid, layout='contiguous'):
    case = {'kind': 'attention', 'batch': batch, 'heads': heads, 'n_q': n_q, 'n_k': n_k, 'dim': dim, 'dtype': dtype,
            'valid': valid, 'layout': layout}
    return {'name': name, **case} if name else case


def _nearest(name, queries, rows, dim, k):
    case = {'kind': 'nearest', 'queries': queries, 'rows': rows, 'dim': dim, 'k': k}
    return {'name': name, **case} if name else case


def _pq(name, queries, codes, dim, subspaces):
    case = {'kind': 'pq', 'queries': queries, 'codes': codes, 'dim': dim, 'subspaces': subspaces}
    return {'name': name, **case} if name else case


def listed():
    return [
        # One pricing request: the subject attends to its comparables.  Launch latency.
        _attention('subject_one', 1, 8, 1, 64, 32, 'bf16', 8),
        # A full batch of requests, the serving configuration.
        _attention('subject_batch', 1024, 8, 1, 64, 32, 'bf16', 8),
        # Subjects against wide, ragged comparable sets with 64-dim heads.
        _attention('subject_wide', 64, 8, 1, 1000, 64, 'bf16', 200),
        # Self-attention over the subject and its 64 comparables, in training and serving types.
        _attention('set_bf16', 1024, 8, 65, 65, 32, 'bf16', 16),
        _attention('set_fp32', 1024, 8, 65, 65, 32, 'fp32', 16),
        # One attention site of the price model: fp16 blocks, views of the qkv projection.
        _attention('model_site', 1024, 8, 65, 65, 16, 'fp16', 9, 'fused'),
        # A block of a larger model: 64-dim heads over a few hundred padded tokens.
        _attention('block_bf16', 64, 8, 257, 257, 64, 'bf16', 64, 'fused'),
        # The same kind of block at full precision.
        _attention('block_fp32', 8, 8, 500, 500, 64, 'fp32', 100, 'fused'),
        # The long-key configuration: compute-bound, no mask.
        _attention('long_key', 16, 16, 4096, 4096, 64, 'bf16', 0),
        # One search request over the engine's exhaustive threshold of 2,048 rows.
        _nearest('nearest_request', 1, 2048, 128, 10),
        # A batch of searches over a shard that has outgrown it.
        _nearest('nearest_batch', 64, 200_000, 128, 100),
        # Product-quantised search: each query's tables, then its distances to a shard's codes.
        _pq('pq_shard', 8, 1_000_000, 128, 16),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    shape = rng.choice(['subject', 'set', 'block', 'long', 'nearest', 'pq'])
    if shape == 'subject':
        heads, dim = rng.choice([4, 8, 12]), rng.choice([16, 32, 32, 64, 64, 128])
        n_k = _log(rng, 16, 2048)
        # K and V of at most 64 million elements each (512 MB in fp32).
        batch = _log(rng, 1, max(1, min(1024, 64_000_000 // (heads * n_k * dim))))
        return _attention(None, batch, heads, 1, n_k, dim, rng.choice(['bf16', 'bf16', 'fp16', 'fp32']),
                          max(1, n_k // 8))
    if shape == 'set':
        n = rng.randint(17, 80)
        return _attention(None, _log(rng, 1, 1024), rng.choice([4, 8]), n, n, rng.choice([16, 32]),
                          rng.choice(['bf16', 'fp16', 'fp32']), max(1, n // 4), rng.choice(['contiguous', 'fused']))
    if shape == 'block':
        n, heads, dim = _log(rng, 81, 1023), rng.choice([4, 8, 12]), rng.choice([32, 64, 64, 128])
        dtype = rng.choice(['bf16', 'bf16', 'fp16', 'fp32'])
        # 35 GFLOP at most in 16 bits (a quarter of it in fp32).
        budget = 35e9 if dtype != 'fp32' else 9e9
        batch = _log(rng, 1, max(1, min(256, int(budget / (4 * heads * n * n * dim)))))
        return _attention(None, batch, heads, n, n, dim, dtype, max(1, n // 5), 'fused')
    if shape == 'long':
        dim = rng.choice([32, 64, 64, 128])
        n_q, n_k = _log(rng, 256, 4096), _log(rng, 1024, 4096)
        planes = max(1, min(256, int(1.0e12 / (4 * n_q * n_k * dim))))
        heads = rng.choice([1, 4, 8])
        batch = _log(rng, 1, max(1, planes // heads))
        return _attention(None, batch, heads, n_q, n_k, dim, rng.choice(['bf16', 'bf16', 'fp16']), 0)
    if shape == 'nearest':
        dim = rng.choice([64, 96, 100, 128, 128, 128, 256])
        queries = _log(rng, 1, 1024)
        rows = _log(rng, 1000, max(1001, min(500_000, 1_638_400_000 // (queries * dim))))
        return _nearest(None, queries, rows, dim, rng.choice([1, 10, 10, 50, 100]))
    subspaces = rng.choice([8, 16, 16, 32])
    queries = _log(rng, 1, 32)
    codes = _log(rng, 10_000, max(10_001, min(4_000_000, 160_000_000 // (queries * subspaces))))
    return _pq(None, queries, codes, 128, subspaces)


def prepare(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(int(seed))

    def randn(*size, dtype=torch.float32, std=1.0):
        return (torch.randn(*size, generator=gen, device='cuda') * std).to(dtype)

    if case['kind'] == 'nearest':
        queries, rows = randn(case['queries'], case['dim']), randn(case['rows'], case['dim'])
        # A search service keeps its workspace from one request to the next.
        need = scan.workspace_bytes(queries, rows, case['k'])
        workspace = torch.zeros(max(need, 1), dtype=torch.uint8, device='cuda')
        return {'kind': 'nearest', 'queries': queries, 'rows': rows, 'k': case['k'], 'workspace': workspace}
    if case['kind'] == 'pq':
        m, dim = case['subspaces'], case['dim']
        codebooks = randn(m, PQ_CENTROIDS, dim // m)
        codes = torch.randint(0, PQ_CENTROIDS, (case['codes'], m), generator=gen, device='cuda', dtype=torch.uint8)
        return {'kind': 'pq', 'queries': randn(case['queries'], dim), 'codebooks': codebooks, 'codes': codes,
                'subspaces': m}
    dtype = DTYPES[case['dtype']]
    b, h, d = case['batch'], case['heads'], case['dim']
    # Long unmasked key axes: the long-key configuration's distribution.
    long_axis = case['valid'] == 0
    if case['layout'] == 'fused':
        qkv = randn(b, case['n_q'], 3 * h * d, dtype=dtype)
        q, k, v = (t.view(b, case['n_q'], h, d).transpose(1, 2) for t in qkv.split(h * d, dim=-1))
    else:
        std = 0.5 if long_axis else 1.0
        q = randn(b, h, case['n_q'], d, dtype=dtype, std=std)
        k = randn(b, h, case['n_k'], d, dtype=dtype, std=std)
        v = randn(b, h, case['n_k'], d, dtype=dtype)
    unit = torch.rand(1, h, 1, 1, generator=gen, device='cuda')
    if long_axis:
        scale, bias = 0.005 + 0.045 * unit, None
    else:
        scale = (0.5 + unit) / d  # around the model's 1 / (2 sigma^2) .. 1 / sigma^2
        counts = torch.randint(case['valid'], case['n_k'] + 1, (b, 1, 1, 1), generator=gen, device='cuda')
        keys = torch.arange(case['n_k'], device='cuda')
        bias = torch.zeros(b, 1, 1, case['n_k'], dtype=dtype, device='cuda')
        bias.masked_fill_(keys >= counts, float('-inf'))
    return {'kind': 'attention', 'q': q, 'k': k, 'v': v, 'scale': scale, 'bias': bias}


def run(state):
    if state['kind'] == 'nearest':
        distances, nodes = scan.nearest(state['queries'], state['rows'], state['k'], workspace=state['workspace'])
        return {'distances': distances, 'nodes': nodes}
    if state['kind'] == 'pq':
        tables = scan.pq_distance_tables(state['queries'], state['codebooks'], state['subspaces'])
        return {'tables': tables, 'distances': scan.pq_adc_distances(tables, state['codes'])}
    return torch.ops.vectra.rbf_attention(state['q'], state['k'], state['v'], state['scale'], state['bias'])


def work(case):
    if case['kind'] == 'nearest':
        q, n, dim, k = case['queries'], case['rows'], case['dim'], case['k']
        return {'bytes': 4 * dim * (n + q) + 8 * q * k, 'flops': 3 * q * n * dim}
    if case['kind'] == 'pq':
        q, n, m, dim = case['queries'], case['codes'], case['subspaces'], case['dim']
        # Queries, codebooks and codes in; tables and distances out.
        return {'bytes': 4 * dim * (q + PQ_CENTROIDS) + n * m + 4 * q * m * PQ_CENTROIDS + 4 * q * n,
                'flops': 3 * q * PQ_CENTROIDS * dim + q * n * m}
    b, h, n_q, n_k, d = case['batch'], case['heads'], case['n_q'], case['n_k'], case['dim']
    size = 4 if case['dtype'] == 'fp32' else 2
    nbytes = b * h * d * size * 2 * (n_q + n_k) + 4 * h + (b * n_k * size if case['valid'] else 0)
    return {'bytes': nbytes, 'flops': 4 * b * h * n_q * n_k * d}


def tolerance(case):
    # The scans keep the reference's order of float operations: every bit is given.
    if case['kind'] != 'attention':
        return 'exact'
    # The output is rounded once to the element type (its step: 2^-8 of the
    # value in bf16, 2^-11 in fp16); fp32 sums carry the expansion's rounding.
    return {'bf16': {'rel': 6e-3, 'max': 2e-2}, 'fp16': {'rel': 1e-3, 'max': 4e-3},
            'fp32': {'rel': 4e-6, 'max': 1e-4}}[case['dtype']]


def exact(case, seed):
    """run()'s outputs in 64 bits, in plain torch."""
    state = prepare(case, seed)
    if case['kind'] == 'nearest':
        queries, rows = state['queries'].double(), state['rows'].double()
        best = torch.full((case['queries'], 0), 0.0, dtype=torch.float64, device='cuda')
        step = max(1, 20_000_000 // case['queries'])
        for start in range(0, case['rows'], step):
            part = torch.cdist(queries, rows[start:start + step], compute_mode='donot_use_mm_for_euclid_dist').square()
            best = torch.cat([best, part], 1).sort(1).values[:, :case['k']]
        if best.shape[1] < case['k']:
            pad = torch.full((case['queries'], case['k'] - best.shape[1]), math.inf, dtype=torch.float64, device='cuda')
            best = torch.cat([best, pad], 1)
        return {'distances': best, 'nodes': None}  # near ties: the order is that of the 32-bit distances
    if case['kind'] == 'pq':
        m = case['subspaces']
        sub = state['queries'].double().view(case['queries'], m, 1, -1)
        tables = (sub - state['codebooks'].double()).square().sum(-1)  # [q, m, 256]
        out = torch.zeros(case['queries'], case['codes'], dtype=torch.float64, device='cuda')
        for s in range(m):
            out += tables[:, s, :][:, state['codes'][:, s].long()]
        return {'tables': tables.reshape(case['queries'], -1), 'distances': out}
    q, k, v, scale, bias = (state[x] for x in ('q', 'k', 'v', 'scale', 'bias'))
    b, h = case['batch'], case['heads']
    out = torch.empty(*q.shape, dtype=torch.float64, device='cuda')
    step = max(1, 32_000_000 // (h * case['n_q'] * case['n_k']))
    for i in range(0, b, step):
        for j in range(0, h, h if step > 1 else 1):
            at = (slice(i, i + step), slice(j, j + (h if step > 1 else 1)))
            qf, kf, vf = (t[at].double().contiguous() for t in (q, k, v))
            dist = (qf.square().sum(-1, keepdim=True) + kf.square().sum(-1)[:, :, None, :]
                    - 2 * torch.matmul(qf, kf.transpose(-1, -2).contiguous())).clamp_(min=0)
            logits = -scale.double()[:, at[1]] * dist
            if bias is not None:
                logits = logits + bias[at[0]].double()
            out[at] = torch.matmul(torch.softmax(logits, -1), vf)
    return out
