"""Unmasked attention with one query head per problem (the image encoder's), at
the sizes where its kernel's two builds begin and end, and at sizes and scales
that it leaves to the general kernel, against torch in fp32."""
import pytest
import torch

from fluxvla_amd import kernels as K

pytestmark = pytest.mark.gpu


# 64 rows per workgroup up to 256 blocks of 64 rows (one per CU) and for problems of up to
# 64 rows, else 128; one, an odd and an even number of key tiles, ragged rows
@pytest.mark.parametrize('n,sq,sk,hd', [
    (1, 1, 64, 8), (3, 65, 128, 72), (2, 200, 192, 80), (48, 256, 256, 72),
    (100, 130, 64, 40), (90, 257, 320, 72), (200, 130, 192, 80), (384, 256, 256, 72),
    (256, 64, 64, 72), (257, 1, 64, 72), (257, 64, 192, 72), (257, 65, 192, 72),
    # the general kernel: keys past the last whole tile
    (3, 100, 100, 72)])
def test_unmasked(n, sq, sk, hd):
    g = torch.Generator().manual_seed(n + sq + sk + hd)
    q, k, v = (torch.randn(n, s, hd, generator=g).to(torch.bfloat16).cuda()
               for s in (sq, sk, sk))
    q = q * 3  # a running maximum that moves
    o = torch.full((n, sq + 1, hd), 7.0, dtype=torch.bfloat16, device='cuda')
    for scale in (hd**-0.5, -0.1):  # (a negative scale: the general kernel)
        K.mqa_attention(q, k, v, o[:, :sq], scale=scale)
        s = torch.matmul(q.float(), k.float().transpose(1, 2).contiguous()) * scale
        ref = torch.matmul(torch.softmax(s, -1), v.float())
        # bf16 probabilities and output: 2^-8 of the largest value, four of them
        err = (o[:, :sq].float() - ref).abs().max().item()
        assert err <= 4 * 2.0**-8 * ref.abs().max().item(), (scale, err)
        assert (o[:, sq:] == 7).all()


# the general kernel (kv_splits = 2) over the same operands: K, V and O as column
# slices of wider rows, two problem strides, output rows of 8, 4 and 2 bytes'
# alignment (the last one stays with the general kernel)
@pytest.mark.parametrize('pad', [8, 4, 1])
def test_matches_the_general_kernel(pad):
    views, seq, heads, hd = 2, 192, 3, 72
    hid = heads * hd
    g = torch.Generator().manual_seed(pad)
    qkv = torch.randn(views * seq, 3 * hid + 16, generator=g).to(torch.bfloat16).cuda()
    outs = []
    for splits in (0, 2):
        o = torch.zeros(views * seq, hid + pad, dtype=torch.bfloat16, device='cuda')
        K.mha_packed_qkv(qkv, o[:, :hid], views, seq, heads, hd, kv_splits=splits)
        assert not o[:, hid:].any()
        outs.append(o[:, :hid].float())
    # bf16 probabilities and output on both sides: 2^-8 of the largest value each
    err = (outs[0] - outs[1]).abs().max().item()
    assert err <= 8 * 2.0**-8 * outs[1].abs().max().item(), err


# few rows and many keys: split keys and the merge with the default's workspace, the
# unsplit walk with none and with one range asked for
@pytest.mark.parametrize('ws,splits', [(None, 0), (0, 0), (None, 1)])
@pytest.mark.parametrize('n,sq,sk,hd', [(1, 64, 4096, 72), (4, 64, 1024, 72), (2, 7, 640, 80),
                                        (48, 64, 896, 40)])
def test_few_rows_many_keys(n, sq, sk, hd, ws, splits):
    g = torch.Generator().manual_seed(n + sq + sk + hd)
    q, k, v = (torch.randn(n, s, hd, generator=g).to(torch.bfloat16).cuda()
               for s in (sq, sk, sk))
    q = q * 3  # a running maximum that moves
    o = torch.full((n, sq + 1, hd), 7.0, dtype=torch.bfloat16, device='cuda')
    d = K.attention_desc(q, k, v, o, sq=sq, sk=sk, heads=1, head_dim=hd, n_problems=n,
                         q_tok_stride=hd, q_head_stride=hd, q_zs=(sq * hd, 0),
                         k_tok_stride=hd, k_zs=(sk * hd, 0), v_tok_stride=hd,
                         v_zs=(sk * hd, 0), o_tok_stride=hd, o_head_stride=hd,
                         o_zs=((sq + 1) * hd, 0), kv_splits=splits)
    if ws is not None:
        d.workspace, d.workspace_bytes = None, ws
    K.run_attention(d)
    s = torch.matmul(q.float(), k.float().transpose(1, 2).contiguous()) * hd**-0.5
    ref = torch.matmul(torch.softmax(s, -1), v.float())
    # bf16 probabilities and output: 2^-8 of the largest value, four of them
    err = (o[:, :sq].float() - ref).abs().max().item()
    assert err <= 4 * 2.0**-8 * ref.abs().max().item(), err
    assert (o[:, sq:] == 7).all()


def test_more_problems_than_one_grid_axis():
    """2^24 problems of one row, the general kernel's: 2^32 threads of the encoder's."""
    n, hd = 1 << 24, 8
    g = torch.Generator(device='cuda').manual_seed(5)
    q = torch.randn(n, 1, hd, generator=g, device='cuda').to(torch.bfloat16)
    k, v = torch.randn(2, 64, hd, generator=g, device='cuda').to(torch.bfloat16)
    o = torch.zeros_like(q)
    K.mqa_attention(q, k[None].expand(n, -1, -1), v[None].expand(n, -1, -1), o)
    s = torch.matmul(q[:, 0].float(), k.float().t()) * hd**-0.5
    ref = torch.matmul(torch.softmax(s, -1), v.float())
    # bf16 probabilities and output: 2^-8 of the largest value, four of them
    assert (o[:, 0].float() - ref).abs().max().item() <= 4 * 2.0**-8 * v.abs().max().item()
