"""Calls with more tiles or slices than one launch of large work-groups may have (2^32 threads along a grid dimension):
they run on a kernel, a tile or a grid that fits.  Inputs of some GiB, checked on the device at the first, the last and
random places; the input of a product overlaps itself (rows 4 or 8 elements apart) so that 2^28 rows of it fit."""
import ctypes as C

import pytest
import torch

from axiom_amd import capi
from oracle import axo
from tests import gpu_harness as gh

pytestmark = pytest.mark.gpu
F32, BF16 = axo.F32, axo.BF16


def places(n, count=2000):
    g = torch.Generator(device="cuda")
    g.manual_seed(n % 1000003)
    return torch.cat([torch.arange(64, device="cuda"), torch.arange(n - 64, n, device="cuda"), torch.randint(0, n, (count,), device="cuda", generator=g)])


@pytest.mark.parametrize("outer,axis,inner", [(17 << 20, 2, 8), ((1 << 24) + 40, 33, 8)])
def test_softmax_over_an_inner_axis_of_many_slices(outer, axis, inner):
    x = torch.empty(outer, axis, inner, dtype=torch.bfloat16, device="cuda").normal_()
    y = torch.empty_like(x)
    gh.sync()
    capi.check(capi.lib().axhip_softmax_axis(x.data_ptr(), BF16, outer, axis, inner, 0, y.data_ptr(), None))
    gh.sync()
    at = places(outer)
    want = torch.softmax(x[at].double(), 1)
    assert bool(((y[at].double() - want).abs() <= want * (2.0**-8 + 200 * 2.0**-23)).all())


def test_attention_of_many_slices():
    """One query row and one key per slice: the result is the value."""
    B, H, D = 131073, 64, 8
    q, k, v = (torch.empty(B, H, 1, D, dtype=torch.bfloat16, device="cuda").normal_() for _ in range(3))
    o = torch.zeros_like(v)
    p = capi.SdpaParams()
    p.dtype, p.batch, p.heads, p.seq_q, p.seq_kv, p.head_dim, p.scale = BF16, B, H, 1, 1, D, -1.0
    for strides in (p.q_strides, p.k_strides, p.v_strides, p.o_strides):
        strides[:] = gh.contiguous_strides(H, 1, D)
    gh.sync()
    capi.check(capi.lib().axhip_sdpa_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), None, C.byref(p), None))
    gh.sync()
    assert torch.equal(o, v)


@pytest.mark.parametrize("dt,m,n,k", [(F32, (1 << 27) + 16, 4, 32), (BF16, (1 << 28) + 32, 1, 64)], ids=["f32", "bf16"])
def test_products_of_many_row_tiles(dt, m, n, k):
    """x W^T of k exact terms (small whole numbers), rows of x overlapping."""
    kind, step = (torch.float32, 4) if dt == F32 else (torch.bfloat16, 8)
    x = torch.empty(m * step + k, dtype=kind, device="cuda").random_(-3, 4)
    w = torch.empty(n, k, dtype=kind, device="cuda").random_(0, 2)
    c = torch.zeros(m, n, dtype=kind, device="cuda")
    p = capi.GemmParams()
    p.dtype, p.trans_b, p.m, p.n, p.k, p.lda, p.ldb, p.ldc, p.batch = dt, 1, m, n, k, step, k, n, 1
    gh.sync()
    capi.check(capi.lib().axhip_gemm(x.data_ptr(), w.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    at = places(m)
    rows = x[at[:, None] * step + torch.arange(k, device="cuda")]
    want = (rows.double() @ w.double().t()).to(kind)
    assert torch.equal(c[at], want)


@pytest.mark.parametrize("m,n,trans_b", [(2, (1 << 29) + 41, 1), ((1 << 29) + 41, 3, 1), ((1 << 29) + 41, 4, 0), ((1 << 30) + 17, 1, 1)])
def test_fp32_products_of_more_tiles_than_a_launch_may_have(m, n, trans_b):
    """Long and narrow products of k exact terms, rows of the long operand overlapping: the strips have to go on in a or b, c,
    the bias and the residual (which is c)."""
    k, step = 32, 4
    a, lda = (torch.empty(m * step + k, device="cuda").random_(-3, 4), step) if m > n else (torch.empty(m, k, device="cuda").random_(-3, 4), k)
    b = (torch.empty(n * step + k, device="cuda").random_(0, 2) if n > m else torch.empty((n, k) if trans_b else (k, n), device="cuda").random_(0, 2))
    bias = torch.empty(n, device="cuda").random_(-5, 6)
    c = torch.empty(m, n, device="cuda").random_(-9, 10)
    p = capi.GemmParams()
    p.dtype, p.trans_b, p.m, p.n, p.k, p.lda, p.ldb, p.ldc, p.batch = F32, trans_b, m, n, k, lda, (step if n > m else k) if trans_b else n, n, 1
    p.bias, p.residual = bias.data_ptr(), c.data_ptr()
    at = torch.cat([places(max(m, n)), torch.arange((1 << 29) - 1024, 1 << 29, device="cuda")])  # (where the next strip starts, among them)
    kk = torch.arange(k, device="cuda")
    before = c[at] if m > n else c[:, at]
    if m > n:
        want = a[at[:, None] * step + kk] @ (b.t() if trans_b else b) + bias + before
    else:
        want = a @ b[at[:, None] * step + kk].t() + bias[at] + before
    gh.sync()
    torch.cuda.synchronize()
    capi.check(capi.lib().axhip_gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    assert torch.equal(c[at] if m > n else c[:, at], want)


@pytest.mark.parametrize("dt,k,trans_b", [(BF16, 16, 1), (BF16, 16, 0), (F32, 32, 1), (F32, 32, 0)], ids=["bf16-nt", "bf16-nn", "f32-nt", "f32-nn"])
def test_more_products_than_a_launch_may_have_tiles_for(dt, k, trans_b):
    """65535 products of one row and 16385 columns, 129 tiles each at the widest: whichever kernel runs needs several launches,
    which have to go on with the next product's a, b, c and residual.  b of product z is that of z - 1 a row (or column)
    further on; sums of k exact terms, all compared."""
    batch, n = 65535, 16385
    kind = torch.float32 if dt == F32 else torch.bfloat16
    a = torch.empty(batch, k, dtype=kind, device="cuda").random_(-2, 3)
    b = torch.empty((n + batch, k) if trans_b else (k, n + batch), dtype=kind, device="cuda").random_(-1, 2)
    bias, res = (torch.empty(s, dtype=kind, device="cuda").random_(-5, 6) for s in ((n,), (batch, n)))
    c = torch.full((batch, n), 99.0, dtype=kind, device="cuda")
    p = capi.GemmParams()
    p.dtype, p.trans_b, p.m, p.n, p.k, p.batch = dt, trans_b, 1, n, k, batch
    p.lda, p.ldb, p.ldc, p.stride_a, p.stride_b, p.stride_c = k, k if trans_b else n + batch, n, k, k if trans_b else 1, n
    p.bias, p.residual = bias.data_ptr(), res.data_ptr()
    gh.sync()
    torch.cuda.synchronize()
    capi.check(capi.lib().axhip_gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), C.byref(p), None))
    gh.sync()
    for z in range(0, batch, 1024):
        count = min(1024, batch - z)
        width = n + count - 1
        window = b[z : z + width].t() if trans_b else b[:, z : z + width]
        all_pairs = a[z : z + count].float() @ window.float()  # (product, column of the window)
        want = all_pairs.as_strided((count, n), (width + 1, 1)) + bias.float() + res[z : z + count].float()
        assert torch.equal(c[z : z + count].float(), want), z


@pytest.mark.parametrize("outer,a,b", [(1 << 21, 65, 65), ((1 << 24) + 300, 16, 17)])
def test_transposed_copy_of_many_small_slices(outer, a, b):
    """fp32 slices of several tiles (63 GiB in and out) and of one, of which there are more than a launch may have."""
    x = torch.empty(outer, a, b, device="cuda").random_(0, 1 << 20)
    y = torch.empty(outer, b, a, device="cuda")
    gh.sync()
    capi.check(capi.lib().axhip_strided_copy(x.data_ptr(), F32, y.data_ptr(), F32, 3, (C.c_int64 * 3)(outer, b, a), (C.c_int64 * 3)(a * b, 1, b), None))
    gh.sync()
    at = places(outer)
    assert torch.equal(y[at], x[at].transpose(1, 2))
