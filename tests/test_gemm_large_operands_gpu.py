"""GEMM epilogue operands of 2 GiB and more (residual, gate, Euler state, previous
chunk): a buffer view holds less than 2 GiB, so each workgroup reads them through
views that begin at its own first row.  Operands are column slices of one large
buffer; against torch in fp32."""
import pytest
import torch

from fluxvla_amd import kernels as K

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
GIB2 = 1 << 31


@pytest.fixture(scope='module')
def arena():
    t = torch.zeros(5 << 28, dtype=BF16, device='cuda')  # 2.5 GiB
    yield t
    del t
    torch.cuda.empty_cache()


def _slice(arena, rows, cols, ld, seed, dtype=BF16):
    """Random values in columns 0 .. cols - 1 of a [rows, ld] view of 2 GiB and more."""
    assert rows * ld * dtype.itemsize >= GIB2
    v = arena.view(dtype)[:rows * ld].view(rows, ld)[:, :cols]
    v.copy_(_rand((rows, cols), seed))
    return v


def _rand(shape, seed, std=1.0):
    g = torch.Generator(device='cuda').manual_seed(seed)
    return (torch.randn(*shape, generator=g, device='cuda') * std).to(BF16)


def _close(got, ref):
    # bf16 output of fp32 sums: one rounding, 2^-9 relative; twice that in the norm
    rel = ((got.float() - ref).norm() / ref.norm()).item()
    assert rel <= 4e-3, rel


# the plain epilogue (tile or two-group kernel, one-round kernel, split-K reduce
# behind the wide kernel) and the general one (a position table as well)
@pytest.mark.parametrize('pos', [False, True])
@pytest.mark.parametrize('operand', ['residual', 'gate'])
@pytest.mark.parametrize('m,n,k,ld', [(131100, 64, 64, 8200), (26000, 2048, 328, 41600),
                                      (4096, 64, 72, 300000), (300, 64, 8192, 4000000)])
def test_plain(arena, m, n, k, ld, operand, pos):
    x, w = _rand((m, k), 1), _rand((n, k), 2, 0.05)
    t = _slice(arena, m, n, ld, 3)
    ref = x.float() @ w.float().t()
    ref = ref + t.float() if operand == 'residual' else ref * t.float()
    kw = {operand: t}
    if pos:
        kw['pos'] = _rand((50, n), 4)
        ref = ref + kw['pos'].float()[torch.arange(m, device='cuda') % 50]
    _close(K.gemm(x, w, **kw), ref)


# output rows in groups of 47 of every 60: the residual's rows go with them
@pytest.mark.parametrize('gate_group', [1, 47])
def test_row_groups(arena, gate_group):
    groups, rg, stride, n, k, ld = 150, 47, 60, 72, 64, 130000
    m = groups * rg
    x, w = _rand((m, k), 5), _rand((n, k), 6, 0.05)
    res = _slice(arena, groups * stride, n, ld, 7)
    gate = _rand((m // gate_group, n), 8)
    out = torch.zeros(groups * stride, n, dtype=BF16, device='cuda')
    K.gemm(x, w, out=out, residual=res, gate=gate, gate_group=gate_group,
           row_group=rg, row_group_stride=stride)
    ref = x.float() @ w.float().t() * gate.float().repeat_interleave(gate_group, 0)
    pick = lambda t: t.unflatten(0, (groups, stride))[:, :rg].reshape(m, n).float()
    _close(pick(out), ref + pick(res))


def test_euler(arena):
    m, n, k, ld = 4096, 32, 64, 140000
    x, w = _rand((m, k), 9), _rand((n, k), 10, 0.05)
    xt = _slice(arena, m, n, ld, 11, torch.float32)
    x0 = xt.clone()
    prev = torch.randn(m, n, device='cuda')
    lk = torch.tensor([7], dtype=torch.int32, device='cuda')
    K.gemm_euler(x, w, None, xt, -0.1, rtc_lock=lk, rtc_period=50, rtc_prev=prev)
    ref = x0 - 0.1 * (x.float() @ w.float().t())
    locked = torch.arange(m, device='cuda') % 50 < 7
    ref[locked] = prev[locked]
    # fp32 sums of 64 products in another order
    torch.testing.assert_close(xt.contiguous(), ref, rtol=1e-5, atol=1e-5)
