"""Which kernel, and how many key ranges, a call takes: the rules of the dispatch as
its queries show them (no GPU needed; 256 CUs are assumed without one)."""
import ctypes

import pytest

from fluxvla_amd import _lib


def _attn(rows, sk, head_dim, heads=1, problems=1, **kw):
    d = _lib.AttnDesc()
    d.q, d.k, d.v, d.o = 4096, 8192, 16384, 32768
    d.sq, d.sk, d.heads, d.head_dim, d.n_problems, d.zdiv = rows, sk, heads, head_dim, problems, 1
    d.q_tok_stride = d.o_tok_stride = heads * head_dim
    d.q_head_stride = d.o_head_stride = d.k_tok_stride = d.v_tok_stride = head_dim
    d.scale = head_dim**-0.5
    for k, v in kw.items():
        setattr(d, k, v)
    return d


def _splits(d):
    """Key ranges: the workspace holds 64 KiB of counters and the partials."""
    ws = _lib.load().fvx_attention_workspace_bytes(ctypes.byref(d))
    if not ws:
        return 1
    dims = 256 if d.head_dim > 80 else 80
    blocks = -(-d.sq * d.heads // 64) * d.n_problems
    return (ws - 65536) // (blocks * (64 * dims + 128) * 4)


# two tiles are split for up to 32 blocks of 64 rows, more tiles at every size
@pytest.mark.parametrize('rows,problems,sk,splits', [
    (50, 1, 64, 1), (50, 1, 65, 2), (50, 1, 128, 2), (256, 1, 128, 2), (257, 1, 128, 1),
    (50, 8, 128, 1), (50, 8, 129, 3), (100, 8, 100, 1), (100, 8, 192, 2), (50, 1, 866, 14)])
def test_row_major_head_dim_256(rows, problems, sk, splits):
    assert _splits(_attn(rows, sk, 256, heads=8, problems=problems)) == splits


# unmasked, one head: few blocks of 64 rows over many key tiles are split, short walks
# and problems that fill the CUs are not
@pytest.mark.parametrize('rows,problems,tiles,splits', [
    (64, 1, 8, 1), (64, 1, 9, 5), (64, 31, 9, 5), (64, 32, 9, 1), (64, 32, 10, 5),
    (64, 1, 64, 32), (1, 1, 64, 32), (64, 4, 16, 8), (64, 16, 8, 1),
    (256, 16, 4, 1), (64, 48, 11, 1), (64, 48, 14, 1), (64, 48, 16, 4), (64, 64, 20, 1), (64, 64, 32, 3),
    (64, 80, 96, 1), (256, 64, 64, 1)])
def test_unmasked_one_head(rows, problems, tiles, splits):
    assert _splits(_attn(rows, 64 * tiles, 72, problems=problems)) == splits
    # one range asked for: no workspace; two: theirs
    assert _splits(_attn(rows, 64 * tiles, 72, problems=problems, kv_splits=1)) == 1
    assert _splits(_attn(rows, 64 * tiles, 72, problems=problems, kv_splits=2)) == 2


def _gemm(m, n, k, mode=_lib.GEMM_PLAIN, fp8=False, **kw):
    p = 1 << 20
    d = _lib.GemmDesc()
    d.a, d.b, d.c, d.m, d.n, d.k, d.lda, d.ldb, d.ldc = p, p, p, m, n, k, k, k, n
    d.mode = mode
    if mode == _lib.GEMM_GEGLU:
        d.b2 = p
    if mode == _lib.GEMM_QKV_ROPE:
        d.head_dim, d.n_q_heads = 256, n // 256 - 2
        d.rope = d.positions = d.q_out = d.k_out = d.v_out = p
        d.ldq, d.ldk, d.ldv = max(1, d.n_q_heads) * 256, 256, 256
    if fp8:
        d.b_fp8, d.b_scale, d.b2_scale = 1, p, p
    for key, v in kw.items():
        setattr(d, key, v)
    return d


def _kernel(*args, **kw):
    return _lib.load().fvx_gemm_kernel(ctypes.byref(_gemm(*args, **kw))).decode()


@pytest.mark.parametrize('kernel,args', [
    ('skinny', (64, 1024, 1024)), ('mid 64x64', (65, 1024, 1024)),
    ('mid 128x128', (768, 3456, 1152)), ('pp 256x320', (6528, 2560, 2048)),
    ('tile 64x128', (768, 4308, 1152)), ('wide', (816, 16384, 2048, _lib.GEMM_GEGLU)),
    ('wide split', (816, 2048, 16384)), ('pp 256x256', (816, 16384, 2048, _lib.GEMM_GEGLU, True)),
    ('tile 64x128', (408, 4096, 1024, _lib.GEMM_GEGLU, True))])
def test_gemm_kernel_names(kernel, args):
    assert _kernel(*args) == kernel
    assert _lib.load().fvx_gemm_kernel(None) == b'none'


# few slabs: the two-group kernel from 176 tiles on (256 CUs)
@pytest.mark.parametrize('m,n,k,pp', [(1641, 4096, 432, False), (5582, 1280, 80, False),
                                      (6961, 1024, 272, False), (5309, 3456, 416, True),
                                      (1978, 4304, 136, True), (14235, 3456, 144, True),
                                      (1804, 3456, 1024, True)])
def test_two_group_kernel_at_short_k(m, n, k, pp):
    assert _kernel(m, n, k).startswith('pp') == pp
    assert not _kernel(m, n + 4, k).startswith('pp')  # (columns in eights)
