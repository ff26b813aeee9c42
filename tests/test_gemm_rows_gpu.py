"""GEMMs with many rows: the tile order in blocks of rows (tile and wide
kernels) at sizes on both sides of a block, against torch in fp32."""
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


# 64-row tiles in blocks of 16 (1024 rows), 256-row tiles in blocks of 4
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
