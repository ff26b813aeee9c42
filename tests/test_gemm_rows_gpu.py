"""GEMMs with many rows: the tile order in blocks of rows (tile and wide kernels) at
sizes on both sides of a block, and every build of the one-round and two-group kernels
at a size that takes it (kernels_run), against torch in fp32."""
import pytest
import torch

from fluxvla_amd import kernels as K

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _rand(shape, seed, std=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(BF16)


def _close(got, ref):
    # bf16 output of fp32 accumulation: one bf16 rounding (2^-9 relative) on
    # values of about rms(ref), four of them at the largest element
    ref = ref.float()
    err = (got.float() - ref).abs().max().item()
    tol = 2.0**-7 * ref.abs().max().item()
    assert err <= tol, (err, tol)
    rel = ((got.float() - ref).norm() / ref.norm()).item()
    assert rel <= 4e-3, rel


# 64-row tiles in blocks of 16 (1024 rows): the tile kernel from 64 x 128 tiles past one
# round on (3137 rows; below, the one-round kernel), and where n is not a multiple of 8
@pytest.mark.parametrize('n,kernel', [(1284, 'tile 64x128'), (324, 'tile 64x64')])
@pytest.mark.parametrize('m', [1024, 1025, 1100, 2049, 2561])
def test_tile_row_blocks(m, n, kernel, kernels_run):
    x, w = _rand((m, 192), 1), _rand((n, 192), 2, 0.05)
    got = K.gemm(x.cuda(), w.cuda())
    _close(got.cpu(), x.float() @ w.float().t())
    assert kernels_run == [kernel]


@pytest.mark.parametrize('m', [1024, 1025, 1100, 2049, 3137])
def test_plain_row_blocks(m):
    n, k = 328, 192
    x, w = _rand((m, k), 1), _rand((n, k), 2, 0.05)
    got = K.gemm(x.cuda(), w.cuda())
    _close(got.cpu(), x.float() @ w.float().t())


@pytest.mark.parametrize('fp8', [False, True])
@pytest.mark.parametrize('m', [1024, 1030, 1300])
def test_geglu_row_blocks(m, fp8):
    n, k = 8192, 128  # 64 columns of tiles: the wide kernels from 4 tile rows on
    x = _rand((m, k), 3)
    wg, wu = _rand((n, k), 4, 0.05), _rand((n, k), 5, 0.05)
    if fp8:
        qg, qu = K.Fp8Weight.quantize(wg.cuda()), K.Fp8Weight.quantize(wu.cuda())
        got = K.gemm_geglu(x.cuda(), qg, qu)
        wg, wu = qg.dequantize().cpu(), qu.dequantize().cpu()
    else:
        got = K.gemm_geglu(x.cuda(), wg.cuda(), wu.cuda())
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    _close(got.cpu(), torch.nn.functional.gelu(g, approximate='tanh') * u)


# the wide kernel's tile rows in blocks of about 4 (1264, 2300 rows) and, with a short
# last tile row, in one block (1025, 1632, 2086)
# (and W8A8: activations that e4m3 holds exactly)
@pytest.mark.parametrize('fp8', [False, True])
@pytest.mark.parametrize('m', [1025, 1264, 1632, 2086, 2300])
def test_wide_row_blocks(m, fp8, kernels_run):
    n, k = 8200, 128
    x = torch.randint(-8, 9, (m, k), generator=torch.Generator().manual_seed(6)).to(BF16).cuda()
    wg, wu = _rand((n, k), 7, 0.01).cuda(), _rand((n, k), 8, 0.01).cuda()
    if fp8:
        qg, qu = (K.Fp8Weight.quantize(w, act='e4m3') for w in (wg, wu))
        got = K.gemm_geglu(x, qg, qu)
        wg, wu = qg.dequantize(), qu.dequantize()
    else:
        got = K.gemm_geglu(x, wg, wu)
    assert kernels_run == ['wide']
    g, u = x.float() @ wg.float().t(), x.float() @ wu.float().t()
    _close(got, torch.nn.functional.gelu(g, approximate='tanh') * u)


# gemm_pp_kernel: sizes at which the plan takes its tiles of 256 x 128, 256 x 192, 256 x
# 320 and 256 x 256, with rows and columns one past a tile and ragged, and K with a
# partial last slab (k % 64 != 0); all operands of the epilogue build.
PP = [(6145, 1152, 712), (2000, 4000, 776), (6150, 1160, 456), (4111, 4304, 584),
      (26000, 2048, 328), (6216, 2560, 712)]


@pytest.mark.parametrize('m,n,k', PP)
def test_pp_plain(m, n, k):
    x, w = _rand((m, k), 11), _rand((n, k), 12, 0.05)
    b, r, g = _rand((n,), 13), _rand((m, n), 14), _rand((m, n), 15)
    got = K.gemm(x.cuda(), w.cuda(), bias=b.cuda(), residual=r.cuda(),
                 gate=g.cuda(), act=2, rownorm_eps=1e-6)
    xf = x.cuda().float()
    xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)
    y = xf @ w.cuda().float().t() + b.cuda().float()
    y = torch.nn.functional.gelu(y, approximate='tanh')
    _close(got, y * g.cuda().float() + r.cuda().float())


# The same kernel with e4m3 weights (256 x 256 and 256 x 128 tiles; GeGLU 256 x
# 2 x 128): rows and columns one past a tile and ragged, K of one and more pairs
# of slabs; against the dequantized weights.
@pytest.mark.parametrize('rownorm', [False, True])
@pytest.mark.parametrize('m,n,k', [(6145, 1160, 1024), (2817, 2568, 2048), (6528, 2048, 2048),
                                   (8190, 2040, 640)])
def test_pp_fp8_plain(m, n, k, rownorm):
    x, r, b = _rand((m, k), 71).cuda(), _rand((m, n), 72).cuda(), _rand((n,), 73).cuda()
    w = K.Fp8Weight.quantize(_rand((n, k), 74, 0.05).cuda())
    ss = torch.full((K.ss_parts(n), m), -1.0, device='cuda')
    xf = x.float()
    if rownorm:
        xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)
    ref = xf @ w.dequantize().float().t()
    got = K.gemm(x, w, bias=b, residual=r, rownorm_eps=1e-6 if rownorm else None)
    _close(got, ref + b.float() + r.float())
    y = r.clone()
    K.gemm(x, w, out=y, residual=y, ss_out=ss, rownorm_eps=1e-6 if rownorm else None)
    _close(y, ref + r.float())
    pad = torch.nn.functional.pad(y.float().pow(2), (0, -n % 64))
    # 64 squares summed in fp32 in another order
    torch.testing.assert_close(ss, pad.view(m, -1, 64).sum(-1).t(), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize('handed', [False, True])
@pytest.mark.parametrize('m,n,k', [(257, 16384, 1024), (700, 16376, 2048), (1601, 4104, 1024)])
def test_pp_fp8_geglu(m, n, k, handed):
    x = _rand((m, k), 81).cuda()
    wg = K.Fp8Weight.quantize(_rand((n, k), 82, 0.05).cuda())
    wu = K.Fp8Weight.quantize(_rand((n, k), 83, 0.05).cuda())
    ss = x.float().pow(2).sum(1)[None].contiguous() if handed else None
    got = K.gemm_geglu(x, wg, wu, rownorm_eps=1e-6, ss_in=ss)
    xf = x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-6)
    g = torch.nn.functional.gelu(xf @ wg.dequantize().float().t(), approximate='tanh')
    _close(got, g * (xf @ wu.dequantize().float().t()))


# (the second GEMM, which takes them: the tile and the one-round kernel)
@pytest.mark.parametrize('m,n,k', [(6145, 1152, 712), (6528, 2560, 640),
                                   (3000, 4104, 520)])
def test_pp_row_sums_handed_on(m, n, k):
    x, w, w2 = _rand((m, k), 21), _rand((n, k), 22, 0.05), _rand((k, n), 23, 0.02)
    ss = torch.full((K.ss_parts(n), m), -1.0, device='cuda')
    res = _rand((m, n), 24).cuda()
    y = res.clone()
    K.gemm(x.cuda(), w.cuda(), out=y, residual=y, ss_out=ss)
    _close(y, x.cuda().float() @ w.cuda().float().t() + res.float())
    pad = torch.nn.functional.pad(y.float().pow(2), (0, -n % 64))
    blocks = pad.view(m, -1, 64).sum(-1).t()
    # 64 squares summed in fp32 in another order
    torch.testing.assert_close(ss, blocks, rtol=1e-5, atol=1e-5)
    z = K.gemm(y, w2.cuda(), rownorm_eps=1e-6, ss_in=ss)
    yf = y.float() * torch.rsqrt(y.float().pow(2).mean(-1, keepdim=True) + 1e-6)
    _close(z, yf @ w2.cuda().float().t())


@pytest.mark.parametrize('fp8', [False, True])
@pytest.mark.parametrize('transposed', [True, False])
# (bf16: gemm_pp_kernel's 256 x 256 and 256 x 320, then gemm_mid_kernel's 128 x 128, 64 x
# 128 and 64 x 64; e4m3: gemm_pp_kernel's 256 x 256, then the tile kernel)
@pytest.mark.parametrize('batch,seq,k', [(8, 777, 712), (31, 211, 520), (2, 500, 200),
                                         (8, 51, 136), (3, 47, 64)])
def test_qkv_rope(batch, seq, k, transposed, fp8):
    heads, hd = 8, 256
    m, n, T = batch * seq, 2560, (seq + 10) // 8 * 8 + 8
    if fp8:
        k = -(-k // 128) * 128  # whole blocks of 128
    x, w = _rand((m, k), 31).cuda(), _rand((n, k), 32, 0.05).cuda()
    if fp8:
        w = K.Fp8Weight.quantize(w)
    rope = K.rope_table(T, hd, device='cuda')
    pos = torch.arange(seq, dtype=torch.int32, device='cuda').repeat(batch)
    q = torch.zeros(m, heads * hd, dtype=BF16, device='cuda')
    kc = torch.zeros(batch, T, hd, dtype=BF16, device='cuda')
    vc = torch.zeros((batch, hd, T) if transposed else (batch, T, hd), dtype=BF16,
                     device='cuda')
    K.gemm_qkv_rope(x, w, rope, pos, q, kc.view(batch * T, hd),
                    vc if transposed else vc.view(batch * T, hd), heads, hd,
                    rownorm_eps=1e-6, row_group=seq, row_group_stride=T,
                    v_ld=T if transposed else None)
    xf = x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-6)
    y = xf @ (w.dequantize() if fp8 else w).float().t()
    c, s = rope[pos.long(), :, 0][:, None], rope[pos.long(), :, 1][:, None]
    p = y[:, :(heads + 1) * hd].view(m, heads + 1, hd // 2, 2)
    rot = torch.stack([p[..., 0] * c - p[..., 1] * s, p[..., 1] * c + p[..., 0] * s],
                      -1).view(m, -1)
    _close(q, rot[:, :heads * hd])
    _close(kc[:, :seq].reshape(m, hd), rot[:, heads * hd:])
    v = vc[:, :, :seq].transpose(1, 2) if transposed else vc[:, :seq]
    _close(v.reshape(m, hd), y[:, (heads + 1) * hd:])
    assert not kc[:, seq:].any()


# gemm_mid_kernel: tiles of 64 x 64 over two K groups and of 128 x 128, ragged rows and
# columns, an odd number of slabs (one K group a slab short) and a partial last slab
# (1024 x 1024, just past its rule: the tile kernel).
MID = [(65, 64, 64), (65, 1160, 72), (408, 1024, 136), (1024, 1024, 200),
       (70, 25608, 136), (769, 3456, 328), (2048, 2048, 64)]


@pytest.mark.parametrize('rownorm', [False, True])
@pytest.mark.parametrize('m,n,k', MID)
def test_mid_plain(m, n, k, rownorm):
    x, w = _rand((m, k), 41), _rand((n, k), 42, 0.05)
    b, r, g = _rand((n,), 43), _rand((m, n), 44), _rand((m, n), 45)
    got = K.gemm(x.cuda(), w.cuda(), bias=b.cuda(), residual=r.cuda(), act=1,
                 gate=g.cuda(), rownorm_eps=1e-6 if rownorm else None)
    xf = x.cuda().float()
    if rownorm:
        xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)
    y = torch.nn.functional.silu(xf @ w.cuda().float().t() + b.cuda().float())
    _close(got, y * g.cuda().float() + r.cuda().float())


@pytest.mark.parametrize('m,n,k', [(66, 72, 64), (816, 2048, 328), (1400, 2048, 264)])
def test_mid_row_sums(m, n, k):
    x, w, w2 = _rand((m, k), 51), _rand((n, k), 52, 0.05), _rand((2560, n), 53, 0.02)
    ss0 = x.float().pow(2).sum(1)[None].cuda()
    ss = torch.full((K.ss_parts(n), m), -1.0, device='cuda')
    y = _rand((m, n), 54).cuda()
    res = y.clone()
    K.gemm(x.cuda(), w.cuda(), out=y, residual=y, rownorm_eps=1e-6, ss_in=ss0,
           ss_out=ss)
    xf = x.cuda().float()
    xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)
    _close(y, xf @ w.cuda().float().t() + res.float())
    pad = torch.nn.functional.pad(y.float().pow(2), (0, -n % 64))
    # 64 squares summed in fp32 in another order
    torch.testing.assert_close(ss, pad.view(m, -1, 64).sum(-1).t(), rtol=1e-5, atol=1e-5)
    # more parts than the kernel keeps in registers
    z = K.gemm(y, w2.cuda(), rownorm_eps=1e-6, ss_in=ss)
    yf = y.float() * torch.rsqrt(y.float().pow(2).mean(-1, keepdim=True) + 1e-6)
    _close(z, yf @ w2.cuda().float().t())


@pytest.mark.parametrize('m,n,k', [(408, 4096, 200), (1281, 1480, 64), (129, 8200, 72)])
def test_mid_geglu(m, n, k):
    x, wg, wu = _rand((m, k), 61), _rand((n, k), 62, 0.1), _rand((n, k), 63, 0.1)
    got = K.gemm_geglu(x.cuda(), wg.cuda(), wu.cuda(), rownorm_eps=1e-6)
    xf = x.cuda().float()
    xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)
    g = torch.nn.functional.gelu(xf @ wg.cuda().float().t(), approximate='tanh')
    _close(got, g * (xf @ wu.cuda().float().t()))


# ---------------------------------------------------------------------------
# Every build of gemm_mid_kernel and gemm_pp_kernel, at a size where the plan takes it
# (asserted): ragged rows and columns, a partial last slab, and the row sums of the
# fused RMSNorm absent, taken in the K loop or handed over.
# ---------------------------------------------------------------------------
SUMS = [None, 'taken', 'handed']


def _norm(x, sums):
    """The kernel's arguments and the normalized rows."""
    if sums is None:
        return {}, x.float()
    xf = x.float()
    kw = {'rownorm_eps': 1e-6}
    if sums == 'handed':
        sq = torch.nn.functional.pad(xf.pow(2), (0, -x.shape[1] % 64))
        kw['ss_in'] = torch.stack(sq.view(x.shape[0], -1, 64).sum(-1).unbind(1))
    return kw, xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)


def _weight(n, k, seed, fp8):
    w = _rand((n, k), seed, 0.05).cuda()
    if not fp8:
        return w, w.float()
    q = K.Fp8Weight.quantize(w)
    return q, q.dequantize().float()


@pytest.mark.parametrize('sums', SUMS)
@pytest.mark.parametrize('kernel,fp8,m,n,k', [
    ('mid 64x64', False, 4000, 256, 200), ('mid 64x64', False, 67, 1096, 136),
    ('mid 128x128', False, 1401, 1992, 264), ('pp 128x256', False, 2070, 3632, 712),
    ('pp 256x128', False, 12001, 408, 712), ('pp 256x192', False, 14001, 408, 456),
    ('pp 256x256', False, 16385, 616, 456), ('pp 256x320', False, 16385, 824, 456),
    ('pp 256x128', True, 20001, 304, 512), ('pp 256x256', True, 12289, 824, 512)])
def test_plain_builds(kernel, fp8, m, n, k, sums, kernels_run):
    x, (w, wf) = _rand((m, k), 101).cuda(), _weight(n, k, 102, fp8)
    b, res = _rand((n,), 103).cuda(), _rand((m, n), 104).cuda()
    kw, xf = _norm(x, sums)
    ref = xf @ wf.t() + b.float() + res.float()
    _close(K.gemm(x, w, bias=b, residual=res, **kw), ref)
    if kernel.startswith('mid'):  # the general epilogue's builds
        pos = _rand((50, n), 105).cuda()
        ref = ref + pos.float()[torch.arange(m, device='cuda') % 50]
        _close(K.gemm(x, w, bias=b, residual=res, pos=pos, **kw), ref)
    assert set(kernels_run) == {kernel}


@pytest.mark.parametrize('sums', SUMS)
@pytest.mark.parametrize('kernel,fp8,m,n,k', [
    ('mid 64x128', False, 66, 72, 64), ('mid 64x128', False, 817, 2040, 328),
    ('mid 128x128', False, 1401, 1992, 264), ('pp 128x256', False, 2070, 3632, 456),
    ('pp 256x128', False, 14001, 408, 456), ('pp 256x256', False, 6338, 1552, 456),
    ('pp 256x128', True, 20001, 304, 512), ('pp 256x256', True, 12289, 824, 512)])
def test_hand_on_builds(kernel, fp8, m, n, k, sums, kernels_run):
    x, (w, wf) = _rand((m, k), 111).cuda(), _weight(n, k, 112, fp8)
    kw, xf = _norm(x, sums)
    mid = kernel.startswith('mid')
    for pos in (None, _rand((50, n), 114).cuda())[:1 + mid]:
        y = _rand((m, n), 113).cuda()
        ref = xf @ wf.t() + y.float()
        if pos is not None:
            ref = ref + pos.float()[torch.arange(m, device='cuda') % 50]
        ss = torch.full((K.ss_parts(n), m), -1.0, device='cuda')
        K.gemm(x, w, out=y, residual=y, ss_out=ss, pos=pos, **kw)
        _close(y, ref)
        pad = torch.nn.functional.pad(y.float().pow(2), (0, -n % 64))
        # 64 squares summed in fp32 in another order
        torch.testing.assert_close(ss, pad.view(m, -1, 64).sum(-1).t(), rtol=1e-5, atol=1e-5)
    assert set(kernels_run) == {kernel}


@pytest.mark.parametrize('sums', SUMS)
@pytest.mark.parametrize('kernel,fp8,m,heads,hd,k', [
    ('mid 64x64', False, 141, 8, 256, 64), ('mid 64x128', False, 409, 8, 256, 136),
    ('mid 128x128', False, 1001, 8, 256, 200), ('pp 128x256', False, 3137, 8, 256, 712),
    ('pp 256x128', False, 4786, 3, 256, 712), ('pp 256x192', False, 2652, 8, 256, 456),
    ('pp 256x256', False, 16385, 8, 64, 456), ('pp 256x320', False, 6435, 8, 256, 456),
    ('pp 256x128', True, 5853, 3, 256, 512), ('pp 256x256', True, 4301, 8, 256, 512)])
def test_qkv_builds(kernel, fp8, m, heads, hd, k, sums, kernels_run):
    n = (heads + 2) * hd
    x, (w, wf) = _rand((m, k), 121).cuda(), _weight(n, k, 122, fp8)
    kw, xf = _norm(x, sums)
    rope = K.rope_table(700, hd, device='cuda')
    pos = (torch.arange(m, device='cuda') % 699).int()
    q = torch.zeros(m, heads * hd, dtype=BF16, device='cuda')
    kc, vc = torch.zeros(2, m, hd, dtype=BF16, device='cuda')
    K.gemm_qkv_rope(x, w, rope, pos, q, kc, vc, heads, hd, **kw)
    assert kernels_run == [kernel]
    y = xf @ wf.t()
    c, s = rope[pos.long(), :, 0][:, None], rope[pos.long(), :, 1][:, None]
    p = y[:, :(heads + 1) * hd].view(m, heads + 1, hd // 2, 2)
    rot = torch.stack([p[..., 0] * c - p[..., 1] * s, p[..., 1] * c + p[..., 0] * s],
                      -1).view(m, -1)
    _close(q, rot[:, :heads * hd])
    _close(kc, rot[:, heads * hd:])
    _close(vc, y[:, (heads + 1) * hd:])


@pytest.mark.parametrize('sums', SUMS)
@pytest.mark.parametrize('kernel,fp8,m,n,k', [
    ('mid 128x128', False, 408, 4096, 200), ('mid 128x128', False, 1281, 1416, 64),
    ('mid 128x128', False, 129, 8184, 72), ('pp 256x256', True, 12289, 408, 512)])
def test_geglu_builds(kernel, fp8, m, n, k, sums, kernels_run):
    x, (wg, gf) = _rand((m, k), 131).cuda(), _weight(n, k, 132, fp8)
    wu, uf = _weight(n, k, 133, fp8)
    kw, xf = _norm(x, sums)
    got = K.gemm_geglu(x, wg, wu, **kw)
    assert kernels_run == [kernel]
    _close(got, torch.nn.functional.gelu(xf @ gf.t(), approximate='tanh') * (xf @ uf.t()))
