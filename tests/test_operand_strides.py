"""The coefficient and the bias of vectra::rbf_attention are read in place,
whatever their broadcast form and strides.

Each form gives the same bits as the same values laid out in full
([B, H, 1, 1] and [B, H, 1, Nk], contiguous): only addresses differ."""

import pytest
import torch

from vectra_amd.kernels import custom_ops  # noqa: F401  (registers the operator)

B, H, NQ, NK, D = 2, 3, 5, 9, 16
DEVICES = ['cpu', pytest.param('cuda', marks=pytest.mark.gpu)]

SCALES = {
    'scalar': lambda x: x[0, 0],
    'one': lambda x: x[:1, 0],
    'per_head': lambda x: x[0, :H].reshape(H, 1, 1),
    'per_batch_column': lambda x: x[:B, 3].reshape(B, 1, 1, 1),  # stride 7 over the batch
    'transposed': lambda x: x[:H, :B].t()[:, :, None, None],
    'expanded': lambda x: x[:1, :H].expand(B, H)[:, :, None, None],
}
BIASES = {
    'none': None,
    'per_key': lambda x: x[0],
    'every_other': lambda x: x[:B, ::2][:, None, None, :],
    'per_head': lambda x: x[:B * H].reshape(B, H, 1, NK),
    'key_major': lambda x: x.t().contiguous().t()[:B][:, None, None, :],  # stride 8 over the keys
    'one_per_batch': lambda x: x[:B, :1][:, None, None, :],
    'flat': lambda x: x[0, 0].reshape(1, 1, 1, 1).expand(B, 1, 1, NK),
}


@pytest.mark.parametrize('device', DEVICES)
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16, torch.int32])
@pytest.mark.parametrize('bias_form', BIASES)
@pytest.mark.parametrize('scale_form', SCALES)
def test_every_broadcast_form_reads_the_same_values(scale_form, bias_form, dtype, device):
    gen = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(B, H, n, D, generator=gen).to(device) for n in (NQ, NK, NK))
    scale = SCALES[scale_form]((torch.rand(5, 7, generator=gen) * 2).to(dtype).to(device))
    bias = None
    if BIASES[bias_form] is not None:
        wide = (torch.randn(8, 2 * NK - (bias_form != 'every_other') * NK, generator=gen) * 3).to(dtype).to(device)
        bias = BIASES[bias_form](wide)
    got = torch.ops.vectra.rbf_attention(q, k, v, scale, bias)
    full = None if bias is None else bias.expand(B, bias.shape[1] if bias.dim() == 4 else 1, 1, NK).contiguous()
    want = torch.ops.vectra.rbf_attention(q, k, v, scale.expand(B, H, 1, 1).contiguous(), full)
    assert torch.equal(got, want)


@pytest.mark.parametrize('device', DEVICES)
@pytest.mark.parametrize('scale_shape,bias_shape', [
    ((2,), None), ((H + 1, 1, 1), None), ((1, 1, 1, 2), None), ((1, 1, 1, 1, 1), None),
    ((), (NK + 1,)), ((), (B + 1, 1, 1, NK)), ((), (1, H + 1, 1, NK)), ((), (1, 1, 1, 1, NK))])
def test_forms_that_do_not_broadcast_raise(scale_shape, bias_shape, device):
    q, k, v = (torch.zeros(B, H, n, D, device=device) for n in (NQ, NK, NK))
    bias = None if bias_shape is None else torch.zeros(bias_shape, device=device)
    with pytest.raises(RuntimeError):
        torch.ops.vectra.rbf_attention(q, k, v, torch.ones(scale_shape, device=device), bias)
