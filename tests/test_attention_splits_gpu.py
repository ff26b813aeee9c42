"""The generic attention (row-major values) over its key splits: the merge with
one workgroup per 16 dims, at one and more than one pass of 16 splits, and the
default's splits where the workspace holds fewer."""
import ctypes

import pytest
import torch

from fluxvla_amd import _lib
from fluxvla_amd import kernels as K

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _inputs(sq, sk, heads, hd):
    g = torch.Generator().manual_seed(sq + sk)
    q, k, v = (torch.randn(1, s, n, generator=g).to(BF16)
               for s, n in ((sq, heads * hd), (sk, hd), (sk, hd)))
    kg = torch.zeros(1, sk, dtype=torch.int32)
    kg[:, sk // 3:sk // 2] = 2**31 - 1          # hidden keys
    qg = torch.zeros(1, sq, dtype=torch.int32)
    s = torch.matmul(q.view(sq, heads, hd).float().transpose(0, 1),
                     k[0].float().t().contiguous()) * hd**-0.5
    s = s.masked_fill(kg[0] != 0, float('-inf'))
    ref = torch.matmul(torch.softmax(s, -1), v[0].float()).transpose(0, 1)
    return (t.cuda() for t in (q, k, v, kg, qg)), ref.reshape(1, sq, heads * hd)


def _check(o, ref):
    # bf16 probabilities and output: 2^-8 of the largest value, four of them
    err = (o.float().cpu() - ref).abs().max().item()
    assert err <= 4 * 2.0**-8 * ref.abs().max().item(), err


@pytest.mark.parametrize('splits', [0, 1, 2, 15, 16, 17, 20])
@pytest.mark.parametrize('sq,sk,heads,hd', [(50, 1281, 8, 256), (3, 1290, 1, 72)])
def test_splits(sq, sk, heads, hd, splits):
    (q, k, v, kg, qg), ref = _inputs(sq, sk, heads, hd)
    o = torch.zeros_like(q)
    K.mqa_attention(q, k, v, o, kgrp=kg, qgrp=qg, kv_splits=splits)
    _check(o, ref)


# the merge's builds of 4, 8 and 16 splits a pass, from their first to their last
@pytest.mark.parametrize('splits', [3, 4, 5, 8, 9])
@pytest.mark.parametrize('sq,sk,heads,hd', [(67, 4600, 2, 256), (70, 4600, 3, 72)])
def test_merge_builds(sq, sk, heads, hd, splits):
    (q, k, v, kg, qg), ref = _inputs(sq, sk, heads, hd)
    o = torch.zeros_like(q)
    K.mqa_attention(q, k, v, o, kgrp=kg, qgrp=qg, kv_splits=splits)
    _check(o, ref)


@pytest.mark.parametrize('keep', [0.0, 0.4, 1.0])
def test_default_splits_fit_the_workspace(keep):
    """With less workspace than the default plan wants, fewer splits."""
    sq, sk, heads, hd = 50, 866, 8, 256
    (q, k, v, kg, qg), ref = _inputs(sq, sk, heads, hd)
    o = torch.zeros_like(q)
    d = K.attention_desc(
        q, k, v, o, sq=sq, sk=sk, heads=heads, head_dim=hd,
        q_tok_stride=q.stride(1), q_head_stride=hd, k_tok_stride=k.stride(1),
        v_tok_stride=v.stride(1), o_tok_stride=o.stride(1), o_head_stride=hd,
        kgrp=kg, qgrp=qg)
    need = _lib.load().fvx_attention_workspace_bytes(ctypes.byref(d))
    assert need > 0
    d.workspace_bytes = int(need * keep)
    K.run_attention(d)
    _check(o, ref)


def test_more_splits_than_the_merge_addresses():
    """65100 key splits asked for: 4.3 GB of partials, more than 32-bit offsets reach."""
    sk, hd, splits = 65100 * 64, 256, 65100
    q = torch.zeros(1, 1, hd, dtype=BF16, device='cuda')
    k = torch.zeros(1, sk, hd, dtype=BF16, device='cuda')  # equal scores: the mean of v
    v = (torch.arange(sk, device='cuda') % 512 / 256.0).to(BF16)[None, :, None].expand(
        1, sk, hd).contiguous()
    o = torch.zeros_like(q)
    d = K.attention_desc(q, k, v, o, sq=1, sk=sk, heads=1, head_dim=hd, q_tok_stride=hd,
                         q_head_stride=hd, k_tok_stride=hd, v_tok_stride=hd,
                         o_tok_stride=hd, o_head_stride=hd, kv_splits=splits)
    need = _lib.load().fvx_attention_workspace_bytes(ctypes.byref(d))
    ws = torch.zeros(need, dtype=torch.uint8, device='cuda')
    d.workspace, d.workspace_bytes = ws.data_ptr(), need
    K.run_attention(d)
    # bf16 probabilities (exactly 1) and output: one rounding of the mean
    ref = v[0, :, 0].double().mean().item()
    assert (o.double() - ref).abs().max().item() <= 2.0**-8 * ref
