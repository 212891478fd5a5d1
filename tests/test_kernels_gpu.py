"""Each HIP kernel alone against its plain PyTorch counterpart (tests/kernel_refs.py),
at sizes other than the engine's tiny models: widths and vocabularies that are no
powers of two, several head sizes and group counts, ragged batches, pages out of order.
"""
import math
import types

import numpy as np
import pytest
import torch

import kernel_refs as R
from yalis_amd.engine.batch import SeqSpan, attention_tiles, attention_token_columns, build_host_batch, named_arrays

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from yalis_amd.ops.hip import HipOps

    return HipOps(DEV)


def rnd(shape, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype).to(DEV)


def device_cache(ops, kc, vc):
    """Pages written in the plain order -> what the kernels expect, on the GPU."""
    if ops.cache_tiled(kc.dtype, kc.shape[3], kc.shape[2]):
        kc, vc = R.tile_cache(kc.cpu(), vc.cpu())
    return kc.to(DEV), vc.to(DEV)


def plain_cache(ops, kc, vc):
    """Pages as the kernels keep them -> the plain order, on the CPU."""
    if ops.cache_tiled(kc.dtype, kc.shape[3], kc.shape[2]):
        return R.untile_cache(kc.cpu(), vc.cpu())
    return kc.cpu(), vc.cpu()


def close(got, want, atol, rtol=0.0):
    got = got.float().cpu()
    want = want.float().cpu()
    err = (got - want).abs()
    bound = atol + rtol * want.abs()
    assert torch.isfinite(got).all(), "kernel produced non-finite values"
    assert (err <= bound).all(), f"max err {err.max().item():.3e} (bound {bound.min().item():.3e})"


# ------------------------------------------------------------------------- embedding
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embed(ops, dtype):
    table = rnd((515, 192), dtype, 0)
    ids = torch.tensor([0, 514, 3, 3, 77, 200], dtype=torch.int32, device=DEV)
    got = ops.embed(ids, table)
    assert got.dtype == torch.float32
    assert torch.equal(got.cpu(), R.embed(ids.cpu(), table.cpu()))


# ------------------------------------------------------------------------------ norm
# (from 1,024 rows on a thread of the fast form holds two pieces of its row)
@pytest.mark.parametrize("width,rows", [(192, 7), (4096, 33), (1000, 3), (6144, 2), (3080, 1030), (72, 1025)])
@pytest.mark.parametrize("act", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16])
def test_add_rmsnorm(ops, width, rows, act, wdtype):
    res = rnd((rows, width), torch.float32, 1)
    res[0] *= 1e-4  # a near-zero row: eps matters
    delta = rnd((rows, width), act, 2)
    w = (1 + 0.1 * rnd((width,), torch.float32, 3)).to(wdtype)
    for eps, unit in ((1e-5, False), (1e-6, True)):
        for d in (delta, None):
            r_gpu = res.clone()
            r_ref = res.clone().cpu()
            got = ops.add_rmsnorm(r_gpu, d, w, eps, unit, act)
            want = R.add_rmsnorm(r_ref, None if d is None else d.cpu(), w.cpu(), eps, unit, torch.float32)
            close(r_gpu, r_ref, 1e-6)
            if act == torch.float32:
                close(got, want, 2e-5, 2e-5)
            else:
                close(got, want, 1e-3, 2**-8)


@pytest.mark.parametrize("width", [192, 4096, 1001])
@pytest.mark.parametrize("tdtype", [torch.float32, torch.bfloat16])
def test_add_rmsnorm_starts_from_embedding_rows(ops, width, tdtype):
    """The first norm gathers the embedding's rows itself: the residual it leaves and the
    normed rows are those of the embedding kernel followed by the norm."""
    table = rnd((515, width), tdtype, 70)
    ids = torch.tensor([0, 514, 3, 3, 77, 200, 1], dtype=torch.int32, device=DEV)
    w = rnd((width,), tdtype, 71) + 1
    res_a = ops.embed(ids, table)
    out_a = ops.add_rmsnorm(res_a, None, w, 1e-5, False, torch.bfloat16)
    res_b, rows = ops.embedded_rows(ids, table)
    res_b.fill_(float("nan"))  # never read
    out_b = ops.add_rmsnorm(res_b, rows, w, 1e-5, False, torch.bfloat16)
    assert torch.equal(res_a, res_b) and torch.equal(out_a, out_b)
    assert torch.equal(rows.gather(), res_a)


def test_gather_add_rmsnorm(ops):
    res = rnd((20, 320), torch.float32, 1)
    delta = rnd((20, 320), torch.bfloat16, 2)
    w = rnd((320,), torch.bfloat16, 3)
    rows = torch.tensor([19, 0, 7, 7], dtype=torch.int32, device=DEV)
    keep = res.clone()
    got = ops.gather_add_rmsnorm(res, delta, rows, w, 1e-5, False, torch.float32)
    want = R.gather_add_rmsnorm(keep.cpu(), delta.cpu(), rows.cpu(), w.cpu(), 1e-5, False, torch.float32)
    assert torch.equal(res, keep), "the gathered form must not change the residual"
    close(got, want, 2e-5, 2e-5)


# ------------------------------------------------------------------------------ gemm
@pytest.mark.parametrize("m,n,k", [(5, 37, 19), (70, 130, 100), (1, 515, 192), (64, 64, 64), (129, 65, 33)])
@pytest.mark.parametrize("xd,wd,od", [
    (torch.float32, torch.float32, torch.float32),
    (torch.bfloat16, torch.float32, torch.bfloat16),
    (torch.bfloat16, torch.bfloat16, torch.float32),
    (torch.float32, torch.bfloat16, torch.float32),
])
def test_gemm_fma(ops, m, n, k, xd, wd, od):
    x = rnd((m, k), xd, 4)
    w = rnd((n, k), wd, 5)
    got = ops.gemm_fma(x, w, od)
    want = x.double().cpu() @ w.double().cpu().T
    if od == torch.float32:
        close(got, want, 1e-5 * math.sqrt(k), 1e-5)
    else:
        close(got, want, 1e-3, 2**-8)


# rows and columns around a tile of 64 and the groups of 16 rows; K around the steps of 16, 32 and 64 and fewer
# steps than groups of waves (4); form 0 is the rule's own choice
@pytest.mark.parametrize("form", [0, 1, 2, 4])
@pytest.mark.parametrize("m,n,k", [(1, 16, 4), (2, 3072, 2048), (16, 17, 68), (17, 33, 1028), (33, 1, 20), (63, 65, 132), (64, 128, 64),
                                   (65, 63, 196), (129, 200, 96), (70, 6400, 36)])
@pytest.mark.parametrize("xd,wd,od", [
    (torch.float32, torch.float32, torch.float32),
    (torch.bfloat16, torch.float32, torch.bfloat16),
    (torch.float32, torch.bfloat16, torch.float32),
])
def test_float32_matrix_core_products(ops, form, m, n, k, xd, wd, od):
    x = rnd((m, k + 12), xd, 41)[:, 4: 4 + k]  # rows of their own stride, starting off 16 bytes for bfloat16
    w = rnd((n, k + 4), wd, 42)[:, :k]
    ops.force_float32_form(form)
    try:
        got = ops.gemm_fma(x, w, od)
    finally:
        ops.force_float32_form()
    want = x.double().cpu() @ w.double().cpu().T
    # float32 sums of k products of about 1: each of at most k / 16 + 16 additions in a row rounds the running sum, of about
    # sqrt(k), by 2^-24 of itself
    atol = math.sqrt(k) * math.sqrt(k / 16 + 16) * 2.0**-24 * 8
    close(got, want, atol, 2.0**-23 if od == torch.float32 else 2.0**-8)


# rows around tiles of 64, columns around waves' 32 and tiles of 128, K around steps of 32 and sums of 128, slices with a short last one and
# fewer made than asked for (5 of 6 pieces); 130 x 8 x 90,000: rows in three passes
@pytest.mark.parametrize("m,n,k,slices", [(33, 1, 4, 1), (64, 128, 36, 1), (65, 129, 128, 1), (1, 31, 132, 1), (129, 132, 132, 2), (63, 64, 640, 5),
                                          (127, 33, 1028, 1), (200, 260, 768, 5), (514, 260, 2048, 16), (130, 8, 90000, 1)])
def test_gemm_split(ops, m, n, k, slices):
    x = rnd((m, k + 8), torch.float32, 45)[:, 4: 4 + k]
    w = rnd((n, k + 4), torch.float32, 46)[:, :k]
    got = ops.gemm_split(x, w, slices)
    want = x.double().cpu() @ w.double().cpu().T
    # the running sum, of about sqrt(k), is rounded by 2^-24 of itself at each of k / 128 additions and some 16 of sums of 128 products and of
    # slices; what else is lost is 2^-7 of that
    close(got, want, math.sqrt(k) * math.sqrt(k / 128 + 16) * 2.0**-24 * 8, 2.0**-23)


@pytest.mark.parametrize("slices", [1, 2])
def test_gemm_split_of_numbers_at_the_limits(ops, slices):
    x, w = rnd((40, 256), torch.float32, 47), rnd((12, 256), torch.float32, 48)
    x[1] *= 1e-38  # subnormal numbers among them, and products that are
    x[2] = x[2].abs() * 1e36  # the products of this row
    w[1] = w[1].abs() * 1e30  # and this one grow beyond float32, and one another's signs hide none
    w[2] *= 1e-30
    x[3, 200], x[4, 9], w[3, 130] = math.inf, math.nan, -math.inf
    x[5] = 0
    got = ops.gemm_split(x, w, slices).cpu()
    want = x.double().cpu() @ w.double().cpu().T
    assert bool((got.isnan() == want.isnan()).all())
    big = want.abs() > 3.4028235e38
    assert bool((got.isinf() == big).all()) and bool((got[big].sign().double() == want[big].sign()).all())
    rest = ~(big | want.isnan())
    # 256 products, each at most the largest of its row and column, and sums below float32's smallest normal number to its last place
    scale = x.double().cpu().abs().nan_to_num(0, 0, 0).amax(1)[:, None] * w.double().cpu().abs().nan_to_num(0, 0, 0).amax(1)[None]
    bound = 16 * math.sqrt(256 / 128 + 16) * 2.0**-24 * 8 * scale + 2.0**-149 * 4
    assert bool(((got.double() - want).abs() <= bound)[rest].all())


# sums that are finite, but not when their operands are scaled: all of them, and those of one column; a short last piece of K
@pytest.mark.parametrize("k,slices", [(4096, 1), (4100, 1), (8192, 3), (2060, 1), (20, 1)])
def test_gemm_split_of_large_sums(ops, k, slices):
    x, w = rnd((70, k), torch.float32, 53), rnd((140, k), torch.float32, 54)
    for all_large in (True, False):
        a, b = x.clone(), w.clone()
        (a if all_large else b[7])[:] *= 2.0**90
        (b[7] if all_large else a[5])[:] *= 2.0**20
        want = a.double().cpu() @ b.double().cpu().T
        # in units of what a sum is large: 16 products are added one by one, the lanes' K / 1,024 sums of them (a lane's), and the lanes' in 6
        # steps, every addition rounded by at most 2^-24 of what it gives (on average half of that): in all of less than a sum's
        # size times sqrt(8 + K / 2,048 + 6) / 2; and the matrix cores' sums as above
        size = a.double().cpu().norm(dim=1)[:, None] * b.double().cpu().norm(dim=1)[None] / math.sqrt(k)
        off = ((ops.gemm_split(a, b, slices).double().cpu() - want) / size).square().mean().sqrt()
        assert off <= 1.5 * math.sqrt(14 + k / 2048) / 2 * 2.0**-24, off
        if k >= 2048:  # and it is what the float32 instructions give, or better
            ops.force_float32_form(4)
            try:
                other = ((ops.gemm_fma(a, b, torch.float32).double().cpu() - want) / size).square().mean().sqrt()
            finally:
                ops.force_float32_form()
            assert off <= 1.1 * other, (off, other)


def test_gemm_split_is_what_float32_products_of_many_rows_are(ops):
    for m, n, k, taken in [(33, 3072, 2048, True), (511, 2048, 8192, True), (64, 512, 512, False), (32, 3072, 2048, False)]:
        x, w = rnd((m, k), torch.float32, 49), rnd((n, k), torch.float32, 50)
        slices = ops._ask("yk_gemm_split_plan", m, n, k)
        assert bool(slices) == taken
        if taken:
            assert torch.equal(ops.gemm_fma(x, w, torch.float32), ops.gemm_split(x, w, slices))
    from yalis_amd.ops.hip import KernelError

    x, w = rnd((64, 256), torch.float32, 51), rnd((6, 256), torch.float32, 52)
    with pytest.raises(KernelError):
        ops.gemm_split(x, w, 2)  # rows of six columns are not for slices
    with pytest.raises(KernelError):
        ops.gemm_split(x, w, 3)


# one to four rows: a wave's one or two rows of the weight, K around its pieces of 256 and its 8 (4) in flight
@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k", [(1, 252), (5, 256), (9, 1028), (7, 2048), (6, 2052), (8191, 260), (8193, 1024), (8195, 1284),
                                 (3, 512), (5, 1800), (4095, 3844), (4097, 776), (4098, 1540)])
@pytest.mark.parametrize("xd,wd,od", [
    (torch.float32, torch.float32, torch.float32),
    (torch.bfloat16, torch.float32, torch.bfloat16),
    (torch.float32, torch.bfloat16, torch.float32),
])
def test_float32_products_of_up_to_four_rows(ops, m, n, k, xd, wd, od):
    x = rnd((m, k + 12), xd, 43)[:, 4: 4 + k]
    w = rnd((n, k + 4), wd, 44)[:, :k]
    got = ops.gemm_fma(x, w, od)
    want = x.double().cpu() @ w.double().cpu().T
    # a lane's four chains of at most k / 256 + 1 additions and eight more: the running sum, of about sqrt(k), is rounded
    # by 2^-24 of itself at each
    atol = math.sqrt(k) * math.sqrt(k / 256 + 9) * 2.0**-24 * 8
    close(got, want, atol, 2.0**-23 if od == torch.float32 else 2.0**-8)


# columns around a tile of 16, K around a chunk of 256 and a round of the eight waves (2,048), fewer chunks than waves
@pytest.mark.parametrize("m", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(16, 8), (48, 248), (32, 264), (64, 2048), (2064, 2056), (96, 4096), (16, 2304)])
def test_products_with_their_own_end(ops, m, n, k):
    """A few-row product with a bias or a gated pair in its launch: what the product and a kernel after it give,
    and the 64-bit result."""
    x = rnd((m, k + 16), torch.bfloat16, 45)[:, 8: 8 + k]  # rows of their own stride
    w = rnd((n, k + 8), torch.bfloat16, 46, scale=k**-0.5)[:, :k]
    bias = rnd((n,), torch.float32, 47)
    bf = torch.bfloat16
    exact = x.double() @ w.double().T
    # float32 sums of k products of about k^-1/2: the running sum, of at most about 4, is rounded by 2^-24 of itself at each
    # of k / 32 + 8 additions
    atol = 4 * math.sqrt(k / 32 + 8) * 2.0**-24 * 8
    close(ops.gemm_cols(x, w, torch.float32), exact.cpu(), atol, 1e-6)
    close(ops.gemm_cols(x, w, bf), exact.cpu(), atol, 2.0**-8)
    close(ops.gemm_cols(x, w, bf, bias=bias), (exact + bias.double()).cpu(), atol + 2.0**-8 * atol, 2.0**-8)
    close(ops.gemm_cols(x, w, bf, bias=bias.to(bf)), (exact + bias.to(bf).double()).cpu(), atol, 2.0**-8)
    prod = ops.gemm_cols(x, w, bf)  # rounded as the pairs take it
    for pair in ("silu", "gelu_tanh", ("clamped_swish", 1.5, 1.7)):
        assert torch.equal(ops.gemm_cols(x, w, bf, gated=pair), ops.gated_act(prod, pair, bf, group=8))


@pytest.mark.parametrize("n,k", [(1024, 520), (2048, 2048), (1024, 5632), (1500, 8192), (1024, 12288)])
def test_products_with_their_own_end_are_no_further_from_64_bits(ops, n, k):
    """The float32 sums that stay in one workgroup, against those of the K slices that such a product used to come as: over six
    seeds no further from the 64-bit result (8,192 entries and more a seed tell 2 % apart)."""
    far = [0.0, 0.0]
    for seed in range(6):
        x, w = rnd((8, k), torch.bfloat16, seed), rnd((n, k), torch.bfloat16, 100 + seed, scale=0.03)
        exact = x.double() @ w.double().T
        for i, form in enumerate((ops.gemm_mfma_skinny, ops.gemm_cols)):
            far[i] += ((form(x, w, torch.float32).double() - exact).norm() / exact.norm()).item()
    assert far[1] <= 1.02 * far[0], far


# both sides of every line of yk_gemm_cols_ok: rows of x, rows of w, elements, K
@pytest.mark.parametrize("m,n,k,whole,handed_on", [
    (1, 1024, 512, True, True), (8, 1024, 2048, True, True), (8, 1023, 2048, False, False), (9, 1024, 2048, True, False), (17, 1024, 2048, False, False),
    (8, 3168, 2048, True, True), (8, 3184, 2048, True, False), (8, 1536, 2304, True, True), (8, 1536, 2312, True, False), (8, 1024, 256, True, True),
    (8, 1024, 248, False, False), (8, 8192, 512, True, True), (8, 8208, 512, False, False), (8, 8208, 768, True, True), (8, 12304, 520, False, False),
    (8, 6352, 2048, True, False), (9, 6352, 2048, False, False), (9, 6344, 2048, True, False), (8, 6320, 2056, True, False), (8, 6336, 2056, False, False),
    (8, 17576, 2048, True, False), (8, 17584, 2048, False, False), (8, 16384, 1024, True, False), (8, 16400, 1024, False, False),
    (8, 1040, 8192, True, False), (8, 1040, 8200, False, False), (4, 1040, 8200, True, False), (12, 1040, 6152, True, False), (13, 1040, 6152, False, False),
    (16, 2112, 6144, True, False), (16, 2120, 6144, False, False),
    # beyond 6.5 M elements: a K of eight chunks, sides that are no square, rounds of the compute units, up to four rows and two
    (8, 4096, 2040, True, False), (8, 4096, 2048, True, True), (9, 4096, 2048, True, False), (8, 4096, 2728, True, True), (8, 4096, 2736, True, False),
    (8, 4096, 6136, False, False), (8, 4096, 6144, True, True), (8, 4096, 12288, True, True), (8, 4096, 12296, False, False), (9, 4096, 8192, False, False),
    (8, 3584, 8192, False, False), (8, 3600, 8192, True, True), (8, 4112, 8192, False, False), (8, 7168, 4096, False, False), (8, 7184, 4096, True, True),
    (8, 8192, 4096, True, True), (8, 8192, 4104, False, False), (8, 8208, 4096, False, False), (4, 2800, 8192, False, False), (4, 2816, 8192, True, True),
    (5, 2816, 8192, False, False), (4, 3072, 14336, True, True), (4, 3072, 14344, False, False), (4, 8192, 8200, False, False), (4, 8192, 12296, True, True),
    (4, 2048, 5632, True, True), (5, 2048, 5632, True, False), (4, 2048, 5640, True, False), (4, 2032, 5632, True, False),
    (2, 2048, 8192, True, True), (3, 2048, 8192, False, False), (2, 2048, 8200, False, False), (2, 1024, 4096, True, True), (2, 1024, 4104, True, False),
    (2, 14336, 2048, True, False), (2, 14352, 2048, True, True), (2, 16384, 2048, True, True), (3, 16384, 2048, True, False), (2, 16384, 2056, False, False),
])
def test_where_products_have_their_own_end(ops, m, n, k, whole, handed_on):
    """Which of the two forms a product takes, told by the order of its sums, and the same value as the other up to that."""
    x, w = rnd((m, k), torch.bfloat16, 51), rnd((n, k), torch.bfloat16, 52, scale=k**-0.5)
    f32 = torch.float32
    own, slices = (ops.gemm_cols(x, w, f32) if m <= 16 else None), ops.gemm_mfma_skinny(x, w, f32)
    exact = x.double() @ w.double().T
    # float32 sums of products of about k^-1/2, at most about 4: rounded by 2^-24 of that at each of up to k / 32 + 16 additions
    atol = 4 * math.sqrt(k / 32 + 16) * 2.0**-24 * 8
    close(slices, exact.cpu(), atol, 1e-6)
    if own is not None:
        close(own, slices.cpu(), 2 * atol, 2e-6)
        assert not torch.equal(own, slices)
    got, part = ops.linear(x, w, f32), ops.linear(x, w, f32, partial_ok=True)
    assert torch.equal(got, own if whole else slices)
    if handed_on:
        assert torch.equal(part, own)
    elif isinstance(part, torch.Tensor):  # one slice
        assert torch.equal(part, slices)
    else:
        close(part.reduce(), slices.cpu(), atol, 1e-6)  # (torch adds the slices in an order of its own)
    bias = rnd((n,), f32, 53)
    close(ops.linear(x, w, f32, bias=bias), (exact + bias.double()).cpu(), 2 * atol, 1e-6)
    if whole and handed_on and n % 16 == 0:
        # one form whatever becomes of the product
        assert torch.equal(ops.linear(x, w, f32, bias=bias), got + bias)
        bf = torch.bfloat16
        for act in ("silu", ("clamped_swish", 1.5, 1.7)):
            assert torch.equal(ops.gate_up_act(x, w, 8, act, bf), ops.gated_act(ops.linear(x, w, bf), act, bf, group=8))
    assert ops.lib.yk_gemm_cols_ok(8, 16384, 256, 0) and not ops.lib.yk_gemm_cols_ok(8, 16400, 256, 0)  # (one slice, and a kernel after it)
    ops.force_cols(1)
    try:
        assert torch.equal(ops.linear(x, w, f32), slices)
    finally:
        ops.force_cols()


def test_biased_products_refuse_what_others_refuse(ops):
    """Inputs and weights that are no rows end in the library's own error, with a bias and without one."""
    from yalis_amd.ops.hip import KernelError

    x, w, bias = rnd((4, 64), torch.bfloat16, 55), rnd((1024, 64), torch.bfloat16, 56), rnd((1024,), torch.bfloat16, 57)
    for b in (None, bias):
        for bad_x, bad_w in ((x[None], w), (x[0], w), (x, w[None]), (x, w[0]), (x[:, ::2], w[:, ::2]), (x[:, :32], w)):
            with pytest.raises(KernelError):
                ops.linear(bad_x, bad_w, torch.bfloat16, bias=b)
        with pytest.raises(KernelError):
            ops.linear(x, w, torch.bfloat16, bias=bias[:-1])


def test_products_with_their_own_end_at_any_width(ops):
    """Columns that are no multiple of 16, K that is no multiple of a chunk, and entries that are not finite in what lies around the
    operands: behind the K columns, before them and behind the last row."""
    for m, n, k in ((5, 33, 264), (16, 1, 8), (1, 47, 520), (9, 17, 2304)):
        xs, ws = rnd((m + 4, k + 24), torch.bfloat16, 48), rnd((n + 20, k + 24), torch.bfloat16, 49)
        for t, rows in ((xs, m), (ws, n)):
            t[:, :8] = float("nan")
            t[:, 8 + k:] = float("inf")
            t[rows:] = float("nan")
        x, w = xs[:m, 8: 8 + k], ws[:n, 8: 8 + k]
        got = ops.gemm_cols(x, w, torch.float32)
        # the running sum, of about sqrt(k), is rounded by 2^-24 of itself at each of k / 32 + 16 additions
        close(got, (x.double() @ w.double().T).cpu(), math.sqrt(k) * math.sqrt(k / 32 + 16) * 2.0**-24 * 8, 1e-6)
    with pytest.raises(Exception):
        ops.gemm_cols(rnd((17, 264), torch.bfloat16, 48), rnd((33, 264), torch.bfloat16, 49), torch.bfloat16)
    with pytest.raises(Exception):
        ops.gemm_cols(rnd((5, 264), torch.bfloat16, 48), rnd((33, 264), torch.bfloat16, 49), torch.bfloat16, gated="silu")

def test_gemm_fma_is_true_float32(ops):
    """Inputs that a reduced-precision matrix mode would truncate: 1 + 2^-12 has more
    mantissa bits than bfloat16 (8) or a 10-bit tensor-float mode keep, and every partial
    sum of its squares is still exact enough in float32."""
    k = 64
    x = torch.full((4, k), 1.0 + 2.0**-12, device=DEV)
    w = torch.full((8, k), 1.0 + 2.0**-12, device=DEV)
    got = ops.gemm_fma(x, w, torch.float32)
    want = k * (1.0 + 2.0**-12) ** 2  # 64.03125...; truncated inputs would give 64
    assert abs(got[0, 0].item() - want) < 2e-5


@pytest.mark.parametrize("m,n,k", [
    (1, 96, 64), (3, 515, 192), (16, 100, 200), (17, 64, 4096), (33, 130, 72), (64, 520, 328),
    (8, 4096, 4096), (100, 515, 192), (1, 16, 8),
])
@pytest.mark.parametrize("od", [torch.float32, torch.bfloat16])
def test_gemm_mfma_skinny(ops, m, n, k, od):
    x = rnd((m, k), torch.bfloat16, 6)
    w = rnd((n, k), torch.bfloat16, 7)
    got = ops.gemm_mfma_skinny(x, w, od)
    want = x.double().cpu() @ w.double().cpu().T
    if od == torch.float32:
        close(got, want, 2e-5 * math.sqrt(k), 1e-5)
    else:
        close(got, want, 1e-2, 2**-8)


@pytest.fixture
def forced(ops):
    """``forced(chunk=, waves=, slices=)`` forces the few-row product's plan for one test."""
    yield ops.force_skinny_plan
    ops.force_skinny_plan()


@pytest.mark.parametrize("chunk", [128, 256])
def test_gemm_mfma_skinny_chunk_lengths(ops, chunk, forced):
    """The few-row product walks K in chunks of 256 or 128, chosen by the length of a
    workgroup's slice; here each length is forced in turn on every row-tile count, on split
    and unsplit products, on K that is no multiple of the chunk, and on the fused activation."""
    forced(chunk=chunk)
    for m, n, k in [(8, 200, 4096), (3, 515, 200), (24, 130, 2056), (40, 96, 1000), (64, 520, 328), (100, 64, 4096)]:
        x = rnd((m, k), torch.bfloat16, 6)
        w = rnd((n, k), torch.bfloat16, 7)
        close(ops.gemm_mfma_skinny(x, w, torch.float32), x.double().cpu() @ w.double().cpu().T, 2e-5 * math.sqrt(k), 1e-5)
    for m, k, inter in [(8, 4096, 512), (30, 392, 200), (64, 1024, 264)]:
        x = rnd((m, k), torch.bfloat16, 30, 0.7)
        packed, group = ops.pack_gate_up(rnd((inter, k), torch.bfloat16, 31, 0.05), rnd((inter, k), torch.bfloat16, 32, 0.05))
        got = ops.gate_up_act(x, packed, group, "silu", torch.bfloat16)
        assert torch.equal(got, ops.gated_act(ops.linear(x, packed, torch.bfloat16), "silu", torch.bfloat16, group=group))


def test_gemm_mfma_skinny_eight_waves(ops, forced):
    """With more than 32 rows of x a workgroup may have eight waves (128 weight rows on one
    staged copy of x): the same sums in the same order as with four, so the same bits, on
    sizes that are no multiples of the workgroup's rows or of the chunk, split and unsplit,
    plain and with the activation in the epilogue.  Eight waves asked for with fewer rows of
    x are four."""
    for m, n, k in [(64, 200, 4096), (50, 515, 328), (40, 1040, 2056), (33, 96, 1000)]:
        x = rnd((m, k), torch.bfloat16, 6)
        w = rnd((n, k), torch.bfloat16, 7)
        for slices in (1, 3):
            forced(waves=4, slices=slices)
            four = ops.gemm_mfma_skinny(x, w, torch.float32)
            forced(waves=8, slices=slices)
            eight = ops.gemm_mfma_skinny(x, w, torch.float32)
            assert torch.equal(four, eight), (m, n, k, slices)
            close(eight, x.double().cpu() @ w.double().cpu().T, 2e-5 * math.sqrt(k), 1e-5)
    x = rnd((64, 1024), torch.bfloat16, 30, 0.7)
    packed, group = ops.pack_gate_up(rnd((264, 1024), torch.bfloat16, 31, 0.05), rnd((264, 1024), torch.bfloat16, 32, 0.05))
    forced(waves=8)
    got = ops.gate_up_act(x, packed, group, "silu", torch.bfloat16)
    assert torch.equal(got, ops.gated_act(ops.linear(x, packed, torch.bfloat16), "silu", torch.bfloat16, group=group))
    few = rnd((8, 1024), torch.bfloat16, 33)
    eight = ops.gemm_mfma_skinny(few, packed, torch.float32)
    forced(waves=4)
    assert torch.equal(eight, ops.gemm_mfma_skinny(few, packed, torch.float32))


def test_gemm_mfma_skinny_two_chunks_in_flight(ops, forced):
    """Long slices of K with 33 to 64 rows of x and eight waves walk in short chunks, two in
    flight per wave (a register set each, by turns): the same sums in the same order as one
    long chunk at a time, so the same bits; slices of an even and of an odd number of chunks,
    K no multiple of the chunk, the last slice shorter, one chunk only in a slice."""
    for m, n, k, slices in [(64, 200, 16384, 2), (48, 136, 4096 + 2600, 1), (33, 520, 3 * 4224 + 72, 3), (64, 96, 4352, 1), (40, 130, 4200, 1)]:
        x = rnd((m, k), torch.bfloat16, 6)
        w = rnd((n, k), torch.bfloat16, 7)
        forced(waves=8, slices=slices)
        two = ops.gemm_mfma_skinny(x, w, torch.float32)   # the rule's own choice for these slices
        forced(waves=8, slices=slices, chunk=256)
        one = ops.gemm_mfma_skinny(x, w, torch.float32)
        forced(waves=4, slices=slices, chunk=128)
        four = ops.gemm_mfma_skinny(x, w, torch.float32)
        assert torch.equal(two, one) and torch.equal(two, four), (m, n, k, slices)
        close(two, x.double().cpu() @ w.double().cpu().T, 2e-5 * math.sqrt(k), 1e-5)


@pytest.mark.parametrize("chunk", [128, 256])
@pytest.mark.parametrize("waves", [4, 8])
def test_gemm_mfma_skinny_wide_form(ops, forced, chunk, waves):
    """33 to 64 rows of x in the wide form (32 x 32 x 16 products, a wave owns 32 weight rows),
    forced here on every shape: sizes that are no multiples of a wave's 32 rows, of the chunk or
    of 64 rows of x, one-hot operands that name the element every lane must hold, split and
    unsplit, float32 and bfloat16 results, the activation in the epilogue (with a last tile
    that holds one gate/up pair only); by the library's own rule it is taken at an unsliced K of 8,192."""
    try:
        ops.wide_skinny_products(2)
        forced(chunk=chunk, waves=waves)
        for m, n, k in [(64, 200, 4096), (50, 515, 328), (40, 1040, 2056), (33, 96, 1000), (100, 72, 520)]:
            x = rnd((m, k), torch.bfloat16, 6)
            w = rnd((n, k), torch.bfloat16, 7)
            want = x.double().cpu() @ w.double().cpu().T
            for slices in (1, 3):
                forced(chunk=chunk, waves=waves, slices=slices)
                close(ops.gemm_mfma_skinny(x, w, torch.float32), want, 2e-5 * math.sqrt(k), 1e-5)
                part = ops.linear(x, w, torch.bfloat16, partial_ok=True)
                close(part.reduce() if hasattr(part, "reduce") else part, want, 2e-2, 2**-7)
            forced(chunk=chunk, waves=waves)
        m, n, k = 40, 48, 64
        for kk in (0, 7, 8, 15, 16, 40, 63):
            x = torch.zeros((m, k), dtype=torch.bfloat16, device=DEV)
            w = torch.zeros((n, k), dtype=torch.bfloat16, device=DEV)
            x[:, kk] = torch.arange(1, m + 1, dtype=torch.bfloat16)
            w[:, kk] = torch.arange(1, n + 1, dtype=torch.bfloat16) * 0.5
            got = ops.gemm_mfma_skinny(x, w, torch.float32).cpu()
            assert torch.equal(got, torch.outer(torch.arange(1, m + 1).float(), torch.arange(1, n + 1).float() * 0.5)), f"k={kk}"
        for inter in (264, 512, 40):  # 528, 1024 and 80 rows of gate/up: the last tile is half, none, half
            x = rnd((64, 1024), torch.bfloat16, 30, 0.7)
            packed, group = ops.pack_gate_up(rnd((inter, 1024), torch.bfloat16, 31, 0.05), rnd((inter, 1024), torch.bfloat16, 32, 0.05))
            got = ops.gate_up_act(x[:50], packed, group, "silu", torch.bfloat16)
            plain = ops.gated_act(ops.linear(x[:50], packed, torch.bfloat16), "silu", torch.bfloat16, group=group)
            assert torch.equal(got, plain), inter
            ops.wide_skinny_products(0)
            assert torch.equal(got, ops.gate_up_act(x[:50], packed, group, "silu", torch.bfloat16))
            ops.wide_skinny_products(2)
        ops.wide_skinny_products(1)
        forced()
        forced(slices=1)
        x, w = rnd((48, 8192), torch.bfloat16, 8, 0.3), rnd((136, 8192), torch.bfloat16, 9, 0.05)
        by_rule = ops.gemm_mfma_skinny(x, w, torch.float32)
        close(by_rule, x.double().cpu() @ w.double().cpu().T, 2e-5 * math.sqrt(8192), 1e-5)
        # with more than 48 rows of x the rule keeps two long chunks in flight per wave: the same
        # bits as one at a time (a forced chunk length), on a K of an odd number of chunks and a tail
        for m, k in ((64, 8192 + 256 + 72), (49, 8192)):
            x, w = rnd((m, k), torch.bfloat16, 8, 0.3), rnd((136, k), torch.bfloat16, 9, 0.05)
            forced(slices=1)
            two = ops.gemm_mfma_skinny(x, w, torch.float32)
            forced(slices=1, chunk=256)
            assert torch.equal(two, ops.gemm_mfma_skinny(x, w, torch.float32))
            close(two, x.double().cpu() @ w.double().cpu().T, 2e-5 * math.sqrt(k), 1e-5)
            packed, group = ops.pack_gate_up(rnd((72, k), torch.bfloat16, 31, 0.05), rnd((72, k), torch.bfloat16, 32, 0.05))
            forced()
            got = ops.gate_up_act(x, packed, group, "silu", torch.bfloat16)
            forced(chunk=256)
            assert torch.equal(got, ops.gate_up_act(x, packed, group, "silu", torch.bfloat16))
        forced()
    finally:
        ops.wide_skinny_products(1)


def _held(rows, cols, ld, seed):
    """Small whole numbers in bfloat16 rows ``ld`` apart, NaN in the gaps and behind the last row: products are exact, and a read too far shows."""
    g = torch.Generator().manual_seed(seed)
    buf = torch.full((rows + 3, ld), float("nan"), dtype=torch.bfloat16)
    buf[:rows, :cols] = torch.randint(-4, 5, (rows, cols), generator=g).to(torch.bfloat16)
    return buf.to(DEV)[:rows, :cols]


@pytest.mark.parametrize("form,least_k,sub", [(0, 192, 64), (1, 192, 64), (2, 256, 64), (3, 384, 128), (4, 256, 64)])
def test_gemm_block_forms(ops, form, least_k, sub):
    """Every form of the product in large tiles, bit for bit (sums of small whole numbers are exact in float32): tiles that hang over on
    either side, more tiles than a grid has workgroups, the shortest K, K cut into slices of which the last is shorter, rows with gaps."""
    from yalis_amd.ops.hip import KernelError, SplitSum

    for m, n, k in [(1, 8, least_k), (65, 200, least_k + sub), (255, 264, 2 * least_k), (300, 1032, 3 * least_k + sub), (129, 24, 1024), (700, 40008, least_k)]:
        x, w = _held(m, k, k + 8, 1), _held(n, k, k + 64, 2)
        want = x.float().cpu() @ w.float().cpu().T
        for slices in (1, 2, 3):
            per = -(-(k // sub) // slices)
            if k // sub - (slices - 1) * per <= least_k // sub - 1:
                with pytest.raises(KernelError, match="too short"):
                    ops.gemm_block(x, w, torch.bfloat16, form * 256 + slices)
                continue
            if slices == 1:
                assert torch.equal(ops.gemm_block(x, w, torch.float32, form * 256 + 1).cpu(), want), (m, n, k)
                assert torch.equal(ops.gemm_block(x, w, torch.bfloat16, form * 256 + 1).cpu(), want.to(torch.bfloat16)), (m, n, k)
            else:
                y = ops.gemm_block(x, w, torch.bfloat16, form * 256 + slices)
                assert isinstance(y, SplitSum) and y.n_splits == slices and y.out_dtype == torch.bfloat16
                assert torch.equal(y.tensor.sum(0).cpu(), want), (m, n, k, slices)
    with pytest.raises(KernelError, match="too short"):
        ops.gemm_block(_held(65, 64, 64, 1), _held(64, 64, 64, 2), torch.bfloat16, form * 256 + 1)


@pytest.mark.parametrize("form", [0, 2, 3, 4])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", ("clamped_swish", 7.0, 1.702)])
def test_gemm_block_gated(ops, form, activation):
    """Gated pairs in the product's end: the pairs of its own rounded product (one unit of bfloat16 apart at most, where the float32 values
    of the two activations straddle a rounding), for random gates, small and a thousand times as large, infinities and NaN as they come (every
    gate there is: below)."""
    for m, n, k in [(1, 16, 512), (130, 528, 512), (300, 1040, 640)]:
        x, w = rnd((m, k), torch.bfloat16, 3), rnd((n, k), torch.bfloat16, 4, 0.3)
        x[0, 0], x[m // 2, 3] = float("inf"), float("nan")
        if m > 1:
            x[m - 1] *= 1000.0
        gu = ops.gemm_block(x, w, torch.bfloat16, form * 256 + 1)
        want = ops.gated_act(gu, activation, torch.bfloat16, group=8).float()
        got = ops.gemm_block(x, w, torch.bfloat16, form * 256 + 1, gated=activation).float()
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        both_inf = torch.isinf(want) & (got == want)
        off = (got - want).abs()[~(torch.isnan(want) | both_inf)]
        assert bool((off <= 2**-7 * want.abs()[~(torch.isnan(want) | both_inf)] + 1e-37).all())


@pytest.mark.parametrize("plan", [2 * 256 + 2, 256 + 1])
def test_gate_up_act_where_the_forced_plan_has_no_pairs(ops, plan):
    x = rnd((130, 1024), torch.bfloat16, 14)
    w, group = ops.pack_gate_up(rnd((256, 1024), torch.bfloat16, 15, 0.05), rnd((256, 1024), torch.bfloat16, 16, 0.05))
    want = ops.gated_act(ops.linear(x, w, torch.bfloat16), "silu", torch.bfloat16, group=group)
    ops.force_block_plan(plan)
    try:
        got = ops.gate_up_act(x, w, group, "silu", torch.bfloat16)
    finally:
        ops.force_block_plan()
    close(got, want.double().cpu(), 2e-2, 2**-6)


@pytest.mark.parametrize("form", [0, 2, 3, 4])
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"] + [("clamped_swish", 7.0, s) for s in (-1.702, 0.0, 1.0, 1.25, 1.5, 1.6, 1.7, 1.702, 2.0)])
def test_gemm_block_gated_of_every_gate(ops, form, activation):
    """Every finite bfloat16 as a gate, and twice it (infinities among these): row i of x holds one 1 or 2 that picks element i of w's rows."""
    bits = torch.arange(1 << 16).view(128, 512)
    bits[(bits & 0x7F80) == 0x7F80] = 0  # (0 times what is no finite number would be no number in every row)
    gate = torch.zeros((512, 512), dtype=torch.bfloat16)
    gate[:, :128] = bits.to(torch.int16).view(torch.bfloat16).T
    up = torch.zeros_like(gate)
    up[:, :128] = torch.tensor([1.5, -3.0, 0.75, -1.0]).repeat(128)[:, None]
    x = torch.zeros((256, 512), dtype=torch.bfloat16)
    x[torch.arange(256), torch.arange(256) % 128] = torch.tensor([1.0, 2.0]).repeat_interleave(128).to(torch.bfloat16)
    w, group = ops.pack_gate_up(gate.to(DEV), up.to(DEV))
    gu = ops.gemm_block(x.to(DEV), w, torch.bfloat16, form * 256 + 1)
    seen, normal = gu.cpu().view(256, 64, 2, 8)[:128, :, 0].reshape(128, 512), gate[:, :128].T.abs() >= 2.0**-126  # (others may come as zeros)
    assert torch.equal(seen[normal], gate[:, :128].T[normal])
    want = ops.gated_act(gu, activation, torch.bfloat16, group=group).float()
    got = ops.gemm_block(x.to(DEV), w, torch.bfloat16, form * 256 + 1, gated=activation).float()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(torch.signbit(got) | got.isnan(), torch.signbit(want) | want.isnan())
    # a unit of bfloat16 where the float32 values straddle a rounding, at its smallest numbers one of 2^-133
    off = (got - want).abs()[torch.isfinite(want)]
    assert bool((off <= 2**-7 * want.abs()[torch.isfinite(want)] + 2.0**-133).all())


# every form, rows and columns around its tiles
@pytest.mark.parametrize("form", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["silu", "gelu_tanh", "relu2"])
@pytest.mark.parametrize("m,n,k", [(129, 264, 640), (300, 8, 384), (257, 520, 384)])
def test_linear_act_is_the_product_and_its_activation(ops, form, kind, m, n, k):
    x, w = rnd((m, k), torch.bfloat16, 61), rnd((n, k), torch.bfloat16, 62) * 0.1
    plan = form * 256 + 1
    want = ops.activation(ops.gemm_block(x, w, torch.bfloat16, plan), kind, torch.bfloat16)
    ops.force_block_plan(plan)
    try:
        got = ops.linear_act(x, w, kind, torch.bfloat16)
    finally:
        ops.force_block_plan()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # few rows, float32 and a view that starts off 16 bytes: the product, then the activation
    for a, b in ((x[:40], w), (x.float(), w.float()), (x[:, 4:], w[:, 4:])):
        old = ops.activation(ops.linear(a, b, a.dtype, partial_ok=True), kind, a.dtype)
        assert torch.equal(ops.linear_act(a, b, kind, a.dtype), old)


def test_gemm_block_is_what_linear_takes(ops):
    """Where ``linear`` and ``gate_up_act`` take the product in large tiles by themselves, and that they agree with the kernels for other sizes."""
    from yalis_amd.ops.hip import SplitSum

    x, w = rnd((999, 1024), torch.bfloat16, 5), rnd((3072, 1024), torch.bfloat16, 6, 0.05)
    want = x.double().cpu() @ w.double().cpu().T
    assert ops._block_plan(x, w, False) >= 0
    close(ops.linear(x, w, torch.bfloat16), want, 2e-2, 2**-7)
    close(ops.linear(x, w, torch.float32), want, 2e-5 * 32, 1e-5)
    bias = rnd((3072,), torch.bfloat16, 7)
    close(ops.linear(x, w, torch.bfloat16, bias=bias), want + bias.double().cpu(), 2e-2, 2**-7)
    xl, wl = rnd((300, 4096), torch.bfloat16, 8), rnd((1024, 4096), torch.bfloat16, 9, 0.05)
    y = ops.linear(xl, wl, torch.bfloat16, partial_ok=True)
    assert isinstance(y, SplitSum)
    close(y.reduce(), xl.double().cpu() @ wl.double().cpu().T, 2e-2, 2**-7)
    packed, group = ops.pack_gate_up(rnd((2048, 1024), torch.bfloat16, 10, 0.05), rnd((2048, 1024), torch.bfloat16, 11, 0.05))
    assert ops._block_plan(x, packed, False, gated=True) >= 0
    got = ops.gate_up_act(x, packed, group, "silu", torch.bfloat16)
    ops.force_block_plan(-2)
    try:
        assert ops._block_plan(x, packed, False, gated=True) < 0
        close(got, ops.gate_up_act(x, packed, group, "silu", torch.bfloat16).double().cpu(), 2e-2, 2**-6)
    finally:
        ops.force_block_plan()
    for m, n, k in [(64, 3072, 1024), (999, 3072, 1000), (999, 3073, 1024), (999, 3072, 64)]:  # too few rows, K no multiple of 64, odd columns, K too short
        assert ops._block_plan(torch.empty(m, k, device=DEV), torch.empty(n, k, device=DEV), True) < 0


# long matrices of 129 to 256 rows: cut along K by one kernel or the other, never the library's
@pytest.mark.parametrize("m,n,k,block", [(129, 8192, 28672, True), (256, 8192, 28672, True), (192, 6144, 16384 - 32, False), (256, 2048, 8192, False), (192, 3072, 8192, True)])
def test_linear_of_long_matrices(ops, m, n, k, block):
    x, w = rnd((m, k), torch.bfloat16, 12), rnd((n, k), torch.bfloat16, 13, 0.05)
    y = ops.linear(x, w, torch.bfloat16, partial_ok=True)
    assert y.n_splits > 1
    got = y.tensor.clone()
    other = ops.gemm_block(x, w, torch.bfloat16, ops._block_plan(x, w, True)) if block else ops.gemm_tile(x, w, torch.bfloat16, True)
    assert torch.equal(got, other.tensor)


def test_gemm_tile(ops):
    """The product in tiles of 128 x 128 for some dozens to a few hundred rows: sizes that are no
    multiples of the tile or of the step of 64 along K, one-hot operands, K cut into 1 to 8 slices
    (an odd number of steps in a slice, a last slice shorter than the others), float32 and
    bfloat16 results, slices kept for a consumer; and where ``linear`` takes it by itself."""
    from yalis_amd.ops.hip import SplitSum

    try:
        for m, n, k in [(65, 200, 4096), (128, 128, 64), (130, 515, 328), (256, 1040, 2056), (200, 96, 1000), (300, 136, 8192), (1, 8, 8)]:
            x = rnd((m, k), torch.bfloat16, 6)
            w = rnd((n, k), torch.bfloat16, 7)
            want = x.double().cpu() @ w.double().cpu().T
            for slices in (0, 1, 2, 3, 8):
                ops.force_tile_slices(slices)
                close(ops.gemm_tile(x, w, torch.float32), want, 2e-5 * math.sqrt(k), 1e-5)
                part = ops.gemm_tile(x, w, torch.bfloat16, partial_ok=True)
                if isinstance(part, SplitSum):
                    assert part.out_dtype == torch.bfloat16 and 1 < part.n_splits <= max(slices, 8)
                    close(part.reduce(), want, 2e-2, 2**-7)
                    res = rnd((m, n), torch.float32, 8)
                    got = ops.add_rmsnorm(res.clone(), part, torch.ones(n, device=DEV), 1e-5, False, torch.float32)
                    part = ops.gemm_tile(x, w, torch.bfloat16, partial_ok=True)
                    summed = part.tensor[0].clone()  # the consumers add the slices one after the other
                    for sl in range(1, part.n_splits):
                        summed += part.tensor[sl]
                    plain = ops.add_rmsnorm(res.clone(), summed.to(torch.bfloat16), torch.ones(n, device=DEV), 1e-5, False, torch.float32)
                    assert torch.equal(got, plain), "the slices' consumers round their sum as the product's output would have been"
                else:
                    close(part, want, 2e-2, 2**-7)
        ops.force_tile_slices(0)
        m, n, k = 150, 140, 128
        for kk in (0, 7, 8, 15, 16, 63, 64, 127):
            x = torch.zeros((m, k), dtype=torch.bfloat16, device=DEV)
            w = torch.zeros((n, k), dtype=torch.bfloat16, device=DEV)
            x[:, kk] = torch.arange(1, m + 1, dtype=torch.bfloat16)
            w[:, kk] = torch.arange(1, n + 1, dtype=torch.bfloat16) * 0.5
            got = ops.gemm_tile(x, w, torch.float32).cpu()
            assert torch.equal(got, torch.outer(torch.arange(1, m + 1).float(), torch.arange(1, n + 1).float() * 0.5)), f"k={kk}"
        # rows of x and w with gaps between them
        xs, wsrc = rnd((100, 4096 + 16), torch.bfloat16, 9), rnd((72, 4096 + 8), torch.bfloat16, 10)
        close(ops.gemm_tile(xs[:, :4096], wsrc[:, :4096], torch.float32), xs[:, :4096].double().cpu() @ wsrc[:, :4096].double().cpu().T, 2e-5 * 64, 1e-5)
        # a down projection of 65 to 256 rows is this kernel's by linear's own choice
        assert ops.long_matrix_tiles(128, 4096, 14336) and not ops.long_matrix_tiles(64, 4096, 14336)
        assert not ops.long_matrix_tiles(300, 4096, 14336) and not ops.long_matrix_tiles(128, 4096, 4096)
        x, w = rnd((100, 4096), torch.bfloat16, 11, 0.3), rnd((520, 4096), torch.bfloat16, 12, 0.05)
        y = ops.linear(x, w, torch.bfloat16, partial_ok=True)
        assert isinstance(y, SplitSum)
        close(y.reduce(), x.double().cpu() @ w.double().cpu().T, 2e-2, 2**-7)
        close(ops.linear(x, w, torch.bfloat16), x.double().cpu() @ w.double().cpu().T, 2e-2, 2**-7)
    finally:
        ops.force_tile_slices(0)


def test_forced_slice_counts_reach_the_consumers(ops, forced):
    """The number of K slices a product leaves behind is what the launch says it wrote, also
    when the plan is forced after the library was first asked about the shape."""
    from yalis_amd.ops.hip import SplitSum

    x, w = rnd((8, 4096), torch.bfloat16, 61), rnd((520, 4096), torch.bfloat16, 62)
    want = x.double().cpu() @ w.double().cpu().T
    auto = ops.linear(x, w, torch.bfloat16, partial_ok=True)
    for slices in (1, 3, 16):
        forced(slices=slices)
        y = ops.linear(x, w, torch.bfloat16, partial_ok=True)
        assert (y.n_splits if isinstance(y, SplitSum) else 1) == slices
        close(y.reduce() if isinstance(y, SplitSum) else y, want, 2e-2, 2**-7)
    forced()
    again = ops.linear(x, w, torch.bfloat16, partial_ok=True)
    assert (again.n_splits if isinstance(again, SplitSum) else 1) == (auto.n_splits if isinstance(auto, SplitSum) else 1)
    with pytest.raises(Exception, match="128 or 256"):
        forced(chunk=100)


def test_gemm_mfma_operand_order(ops):
    """One-hot operands name the element each lane must hold: y[m, n] = x[m, kx] * w[n, kx]
    for a single k picks out any mismatch between the two operands' k order."""
    m, n, k = 16, 16, 64
    for kk in (0, 7, 8, 31, 32, 63):
        x = torch.zeros((m, k), dtype=torch.bfloat16, device=DEV)
        w = torch.zeros((n, k), dtype=torch.bfloat16, device=DEV)
        x[:, kk] = torch.arange(1, m + 1, dtype=torch.bfloat16)
        w[:, kk] = torch.arange(1, n + 1, dtype=torch.bfloat16) * 0.5
        got = ops.gemm_mfma_skinny(x, w, torch.float32).cpu()
        want = torch.outer(torch.arange(1, m + 1).float(), torch.arange(1, n + 1).float() * 0.5)
        assert torch.equal(got, want), f"k={kk}"


def test_split_sums_feed_their_consumers(ops):
    """A few-row product may stay as unreduced K slices; norm, rotary + append and the
    gated activation add them up themselves, round the sum as the product's output would
    have been rounded, and so give the same bits as the reduced path."""
    from yalis_amd.ops.hip import SplitSum

    m, k = 5, 4096
    x = rnd((m, k), torch.bfloat16, 20, 0.5)
    w = rnd((256, k), torch.bfloat16, 21, 0.05)
    part = ops.linear(x, w, torch.bfloat16, partial_ok=True)
    assert isinstance(part, SplitSum) and part.n_splits > 1, "this shape was meant to split K"
    assert part.out_dtype == torch.bfloat16
    # (the slices live in the library's workspace until the next product; a copy of this test's
    # own can be fed to every consumer below)
    part = SplitSum(part.tensor.clone(), part.out_dtype)
    full = part.tensor.sum(0)
    assert (full.cpu() - (x.double().cpu() @ w.double().cpu().T).float()).abs().max() < 1e-3
    reduced = ops.linear(x, w, torch.bfloat16)  # the same slices, summed and rounded by the product
    assert torch.equal(part.reduce(), reduced.float())
    # norm
    res = rnd((m, 256), torch.float32, 22)
    nw = (1 + 0.1 * rnd((256,), torch.float32, 23)).to(torch.bfloat16)
    r1, r2 = res.clone(), res.clone()
    got = ops.add_rmsnorm(r1, part, nw, 1e-5, False, torch.bfloat16)
    want = ops.add_rmsnorm(r2, reduced, nw, 1e-5, False, torch.bfloat16)
    assert torch.equal(r1, r2) and torch.equal(got, want)
    close(r1, res.cpu() + full.cpu(), 1e-2, 2**-7)
    rows = torch.tensor([4, 0], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.gather_add_rmsnorm(res, part, rows, nw, 1e-5, False, torch.float32),
                       ops.gather_add_rmsnorm(res, reduced, rows, nw, 1e-5, False, torch.float32))
    # gated activation
    assert torch.equal(ops.gated_act(part, "silu", torch.bfloat16), ops.gated_act(reduced, "silu"))
    close(ops.gated_act(part, "silu", torch.float32), R.gated_act(reduced.float().cpu(), "silu"), 1e-5, 1e-5)
    # rotary + append: 2 query heads, 1 kv head of 64 -> 256 columns
    cos, sin = _tables(64, 100)
    positions = torch.tensor([3, 4, 50, 0, 99], dtype=torch.int32, device=DEV)
    slots = torch.tensor([5, 6, 40, 0, 63], dtype=torch.int32, device=DEV)
    kc = torch.zeros((4, 1, 16, 64), dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros((4, 1, 64, 16), dtype=torch.bfloat16, device=DEV)
    q = ops.rope_append(part, 2, 1, 64, positions, cos, sin, 64, False, kc, vc, slots, 16)
    assert q.shape == (m, 128) and q.dtype == torch.bfloat16
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    q2 = ops.rope_append(reduced.clone(), 2, 1, 64, positions, cos, sin, 64, False, kc2, vc2, slots, 16)
    assert torch.equal(q, q2[:, :128]) and torch.equal(kc, kc2) and torch.equal(vc, vc2)
    kr, vr = torch.zeros((4, 1, 16, 64)), torch.zeros((4, 1, 64, 16))
    ref2 = full.clone().cpu()
    R.rope_append(ref2, 2, 1, 64, positions.cpu(), cos.cpu(), sin.cpu(), 64, False, kr, vr, slots.cpu(), 16)
    close(q, ref2[:, :128], 1e-2, 2**-7)
    close(kc, kr, 1e-2, 2**-7)
    close(vc, vr, 1e-2, 2**-7)
    # slices of a product asked for in float32 are added without rounding
    part32 = ops.linear(x, w, torch.float32, partial_ok=True)
    assert isinstance(part32, SplitSum) and part32.out_dtype == torch.float32
    r3 = res.clone()
    ops.add_rmsnorm(r3, part32, nw, 1e-5, False, torch.bfloat16)
    close(r3, res.cpu() + full.cpu(), 2e-6, 2e-6)


@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("m,k,inter", [(1, 4096, 1024), (8, 512, 2048), (40, 320, 520), (64, 4096, 14336 // 4),
                                       (5, 8192, 64), (70, 256, 328), (9, 192, 100)])
def test_gate_up_act(ops, act, m, k, inter):
    """Both projections and the activation: as one kernel where the product has few rows and
    is not split over K, else product + activation kernel over the packed columns; the
    same bits either way, and the plain arithmetic on [gate; up] within rounding."""
    x = rnd((m, k), torch.bfloat16, 30, 0.7)
    wg = rnd((inter, k), torch.bfloat16, 31, 0.05)
    wu = rnd((inter, k), torch.bfloat16, 32, 0.05)
    packed, group = ops.pack_gate_up(wg, wu)
    assert group == (8 if inter % 8 == 0 else 0) and packed.shape == (2 * inter, k)
    got = ops.gate_up_act(x, packed, group, act, torch.bfloat16)
    assert got.shape == (m, inter)
    # product, then the activation kernel on the packed columns
    gu = ops.linear(x, packed, torch.bfloat16)
    two_steps = ops.gated_act(gu, act, torch.bfloat16, group=group)
    assert torch.equal(got, two_steps)
    gate = (x.double().cpu() @ wg.double().cpu().T).to(torch.bfloat16)
    up = (x.double().cpu() @ wu.double().cpu().T).to(torch.bfloat16)
    want = R.gated_act(torch.cat([gate, up], dim=1).float(), act)
    close(got, want, 3e-2, 2**-7)
    # float32 weights are never packed
    assert ops.pack_gate_up(wg.float(), wu.float())[1] == 0


def test_gated_act_grouped_columns(ops):
    gu = rnd((7, 2 * 72), torch.bfloat16, 33, 2.0)
    for group in (0, 4, 8, 24):
        close(ops.gated_act(gu, "silu", group=group), R.gated_act(gu.float().cpu(), "silu", group=group), 1e-2, 2**-7)
    part = rnd((3, 7, 2 * 72), torch.float32, 34, 1.0)
    from yalis_amd.ops.hip import SplitSum
    close(ops.gated_act(SplitSum(part, torch.bfloat16), "silu", torch.bfloat16, group=8),
          R.gated_act(part.sum(0).to(torch.bfloat16).float().cpu(), "silu", group=8), 1e-2, 2**-7)


def test_linear_dispatch(ops):
    x = rnd((200, 192), torch.bfloat16, 8)
    w = rnd((515, 192), torch.bfloat16, 9)
    want = x.double().cpu() @ w.double().cpu().T
    close(ops.linear(x, w, torch.bfloat16), want, 1e-2, 2**-7)
    close(ops.linear(x, w, torch.float32), want, 1e-4, 1e-5)
    close(ops.linear(x[:5], w, torch.bfloat16), want[:5], 1e-2, 2**-7)
    # 65 to 192 rows where the vendor library would have few tiles: the few-row kernel, in row tiles of 64
    assert ops.few_library_tiles(100, 515) and not ops.few_library_tiles(200, 515) and not ops.few_library_tiles(128, 28672)
    assert ops.few_library_tiles(128, 4096) and not ops.few_library_tiles(128, 6144) and not ops.few_library_tiles(160, 4096)
    for rows in (65, 100, 128, 192):
        close(ops.linear(x[:rows], w, torch.bfloat16), want[:rows], 1e-2, 2**-7)
        part = ops.linear(x[:rows], w, torch.bfloat16, partial_ok=True)
        close(part.reduce() if hasattr(part, "reduce") else part, want[:rows], 1e-2, 2**-7)
    wf = w.float()
    close(ops.linear(x, wf, torch.bfloat16), want, 1e-2, 2**-7)


@pytest.mark.parametrize("tuned", [False, True])
def test_library_product(ops, tuned):
    """The vendor library's product, called directly: rows of x and w with gaps between them,
    both result types, shapes that are timed when first met (up to 256 rows) and shapes that are
    not, and the same values again from the kept plan."""
    ops.tune_library_products(tuned)
    try:
        for seed, (m, n, k, pad) in enumerate(((70, 520, 200, 0), (200, 1032, 136, 8), (300, 264, 512, 16), (129, 4096, 256, 0))):
            # (other leading dimensions for the two settings, so that each makes plans of its own)
            pad += 8 if tuned else 0
            xs = rnd((m, k + pad), torch.bfloat16, 50 + seed)
            wsrc = rnd((n, k + pad), torch.bfloat16, 60 + seed)
            x, w = xs[:, :k], wsrc[:, :k]
            want = x.double().cpu() @ w.double().cpu().T
            first = ops.gemm_library(x, w, torch.bfloat16)
            close(first, want, 1e-2, 2**-7)
            assert torch.equal(first, ops.gemm_library(x, w, torch.bfloat16))
            close(ops.gemm_library(x, w, torch.float32), want, 1e-4, 1e-5)
    finally:
        ops.tune_library_products(False)
    from yalis_amd.ops.hip import KernelError

    with pytest.raises(KernelError, match="gemm_library"):
        ops.gemm_library(rnd((70, 64), torch.float32, 1), rnd((64, 64), torch.bfloat16, 2), torch.bfloat16)


# ---------------------------------------------------------------- rotary + cache append
def _tables(rotary_dim, positions, theta=10000.0):
    inv = 1.0 / (theta ** (torch.arange(0, rotary_dim, 2).float() / rotary_dim))
    ang = torch.outer(torch.arange(positions).float(), inv)
    return torch.cos(ang).to(DEV), torch.sin(ang).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("h,g,d,rd,inter", [(4, 2, 16, 16, False), (6, 3, 64, 64, False), (8, 1, 128, 64, True), (3, 3, 48, 32, False), (5, 0, 32, 32, False)])
def test_rope_append(ops, dtype, h, g, d, rd, inter):
    n, page, n_pages = 37, 16, 9
    qkv = rnd((n, (h + 2 * g) * d), dtype, 10)
    cos, sin = _tables(rd, 200)
    positions = torch.randint(0, 200, (n,), generator=torch.Generator().manual_seed(1), dtype=torch.int32).to(DEV)
    slots = torch.randperm(page * n_pages, generator=torch.Generator().manual_seed(2))[:n].to(torch.int32).to(DEV)
    kc = torch.zeros((n_pages, max(g, 1), page, d), dtype=dtype, device=DEV)
    vc = torch.zeros((n_pages, max(g, 1), d, page), dtype=dtype, device=DEV)
    kc_r, vc_r, qkv_r = kc.cpu().clone(), vc.cpu().clone(), qkv.cpu().clone()
    if g == 0:
        ops.rope_append(qkv, h, 0, d, positions, cos, sin, rd, inter, None, None, None, page)
        R.rope_append(qkv_r, h, 0, d, positions.cpu(), cos.cpu(), sin.cpu(), rd, inter, None, None, None, page)
    else:
        ops.rope_append(qkv, h, g, d, positions, cos, sin, rd, inter, kc, vc, slots, page)
        R.rope_append(qkv_r, h, g, d, positions.cpu(), cos.cpu(), sin.cpu(), rd, inter, kc_r, vc_r, slots.cpu(), page)
    tol = 1e-6 if dtype == torch.float32 else 2**-7
    close(qkv.view(n, -1, d)[:, :h], qkv_r.view(n, -1, d)[:, :h], tol, tol)
    if g:
        close(kc, kc_r, tol, tol)
        assert torch.equal(vc.cpu(), vc_r), "values are copied, not changed"


@pytest.mark.parametrize("h,g,d,rd,page", [(8, 2, 128, 128, 64), (6, 3, 64, 32, 16), (4, 4, 48, 48, 32), (5, 1, 80, 16, 16), (6, 3, 64, 32, 128)])
def test_rope_append_prompt_portions(ops, h, g, d, rd, page):
    """Many bfloat16 tokens: portions whose slots run on from a multiple of 8 (values stored
    as 16-byte pieces), portions that start anywhere, scattered single tokens, a token count
    that is no multiple of 8; everything else in the pages stays as it was."""
    u = 64  # slots are laid out in units of 64 whatever the page size
    n_pages = 12 * u // page
    runs = [(3 * u, 40), (7 * u + 5, 19), (0, u), (9 * u + 8, 11)]  # (first slot, tokens)
    slots, positions = [], []
    for first, count in runs:
        slots += list(range(first, first + count))
        positions += list(range(first % 50, first % 50 + count))
    scattered = [5 * u + 3, 2 * u + 9, 11 * u + 1]
    slots += scattered
    positions += [190, 0, 77]
    n = len(slots)
    assert n % 8 != 0 and len(set(slots)) == n
    qkv = rnd((n, (h + 2 * g) * d), torch.bfloat16, 40)
    cos, sin = _tables(rd, 200)
    positions = torch.tensor(positions, dtype=torch.int32, device=DEV)
    slots = torch.tensor(slots, dtype=torch.int32, device=DEV)
    kc_r, vc_r = rnd((n_pages, g, page, d), torch.bfloat16, 41).cpu(), rnd((n_pages, g, d, page), torch.bfloat16, 42).cpu()
    kc, vc = device_cache(ops, kc_r.clone(), vc_r.clone())
    qkv_r = qkv.cpu().clone()
    ops.rope_append(qkv, h, g, d, positions, cos, sin, rd, False, kc, vc, slots, page)
    R.rope_append(qkv_r, h, g, d, positions.cpu(), cos.cpu(), sin.cpu(), rd, False, kc_r, vc_r, slots.cpu(), page)
    close(qkv.view(n, -1, d)[:, :h], qkv_r.view(n, -1, d)[:, :h], 2**-7, 2**-7)
    kc_p, vc_p = plain_cache(ops, kc, vc)
    close(kc_p, kc_r, 2**-7, 2**-7)
    assert torch.equal(vc_p, vc_r), "values are copied, not changed"
    # the same rows one token at a time (the scalar kernel) give the same bits
    qkv1 = rnd((n, (h + 2 * g) * d), torch.bfloat16, 40)
    kc1, vc1 = device_cache(ops, rnd((n_pages, g, page, d), torch.bfloat16, 41), rnd((n_pages, g, d, page), torch.bfloat16, 42))
    for i in range(n):
        ops.rope_append(qkv1[i : i + 1], h, g, d, positions[i : i + 1], cos, sin, rd, False, kc1, vc1, slots[i : i + 1], page)
    assert torch.equal(qkv1.view(n, -1, d)[:, :h], qkv.view(n, -1, d)[:, :h]) and torch.equal(kc1, kc) and torch.equal(vc1, vc)


# ------------------------------------------------------------------------- attention
def _attention_case(ops, dtype, h, g, d, page, spans, window, seed, poison=True, n_pages=64, plan=None, long_plan=None, col_tiles=1, with_cols=False,
                    pool_pages=None):
    """spans: list of (cached tokens before the step, new tokens).  Builds pages in a
    shuffled order, fills cache for the earlier tokens, runs rope-free attention.
    pool_pages: the pages are the last n_pages of a pool of so many (never initialised below them)."""
    gen = torch.Generator().manual_seed(seed)
    order = torch.randperm(n_pages, generator=gen).tolist()
    kc = torch.zeros((n_pages, g, page, d), dtype=dtype)
    vc = torch.zeros((n_pages, g, d, page), dtype=dtype)
    if poison:
        kc.fill_(float("nan"))
        vc.fill_(float("nan"))
    seqs = []
    used = 0
    for cached, new in spans:
        total = cached + new
        n_p = -(-total // page)
        table = np.array(order[used : used + n_p], dtype=np.int32)
        used += n_p
        assert used <= n_pages
        k = torch.randn((total, g, d), generator=gen).to(dtype)
        v = torch.randn((total, g, d), generator=gen).to(dtype)
        for pos in range(total):
            kc[table[pos // page], :, pos % page, :] = k[pos]
            vc[table[pos // page], :, :, pos % page] = v[pos]
        seqs.append(SeqSpan(tokens=[0] * new, first_position=cached, block_tables=[table + (pool_pages - n_pages if pool_pages else 0)], state_slot=0))
    hb = build_host_batch(seqs, 1, page)
    tpt = ops.attention_tokens_per_tile(h, g)
    big = ops.attention_long_span_tile(h, g)
    big_c = ops.attention_long_span_tile(h, g, col_tiles)  # tokens of a long tile with col_tiles column tiles a wave
    arrays = named_arrays(hb, {"tiles": lambda b: attention_tiles(b, tpt, 1, big), "long_tiles": lambda b: attention_tiles(b, big_c, big + 1, longest_first=(seed % 2 == 0)),
                               "cols": lambda b: attention_token_columns(b, tpt, 1, big)})
    ctx = types.SimpleNamespace(
        arrays={k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in arrays.items()},
        max_ctx=hb.max_ctx,
    )
    ctx_cpu = types.SimpleNamespace(arrays={k: torch.from_numpy(np.ascontiguousarray(v)) for k, v in arrays.items()})
    n = hb.n_tokens
    q = (torch.randn((n, h * d), generator=gen) * 1.5).to(dtype)
    scale = 1.0 / math.sqrt(d)
    kc_d, vc_d = device_cache(ops, kc, vc)
    if pool_pages:
        pool_k = torch.empty((pool_pages,) + tuple(kc_d.shape[1:]), dtype=dtype, device=DEV)
        pool_v = torch.empty((pool_pages,) + tuple(vc_d.shape[1:]), dtype=dtype, device=DEV)
        pool_k[pool_pages - n_pages:] = kc_d
        pool_v[pool_pages - n_pages:] = vc_d
        kc_d, vc_d = pool_k, pool_v
    got = ops.attention(q.to(DEV), h, g, d, kc_d, vc_d, page, scale, window, ctx, 0, ctx.arrays["tiles"], ctx.arrays["long_tiles"], plan=plan, long_plan=long_plan, long_col_tiles=col_tiles,
                        token_cols=ctx.arrays["cols"] if with_cols else None)
    if pool_pages:
        return got, None  # (the plain implementation would need the pool on the host)
    want = R.attention(q.float(), h, g, d, kc.float(), vc.float(), page, scale, window, ctx_cpu, 0, None)
    return got, want


SPANS = [(0, 5), (17, 1), (0, 70), (63, 2), (100, 1), (31, 34), (0, 1)]


# enough (token, head)s for the form that makes four, two or one head a wave; windows that start inside a group of four keys
@pytest.mark.parametrize("h,g,d,page", [(48, 12, 16, 16), (40, 20, 80, 64), (45, 15, 32, 16), (40, 5, 256, 32)])
@pytest.mark.parametrize("window", [0, 3, 66])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_generic_many_tokens(ops, h, g, d, page, window, dtype):
    got, want = _attention_case(ops, dtype, h, g, d, page, SPANS, window, 19)
    if dtype == torch.float32:
        close(got, want, 2e-5, 1e-5)
    else:
        close(got, want, 1e-2, 2**-7)


# head sizes 64 and 128 in float32: tiles of 16 columns of 16, 8, 4, 2 and 1 heads, which tokens of several requests share; pages of a few slots
@pytest.mark.parametrize("h,g,d,page", [(48, 3, 64, 16), (40, 5, 128, 4), (48, 12, 64, 64), (72, 2, 128, 20), (40, 20, 64, 8), (45, 15, 128, 32)])
@pytest.mark.parametrize("window", [0, 3, 66])
def test_attention_float32_tiles(ops, h, g, d, page, window):
    got, want = _attention_case(ops, torch.float32, h, g, d, page, SPANS, window, 20, n_pages=160)
    close(got, want, 2e-5, 1e-5)


# a tile's requests shared out among workgroups (many requests of few tokens, one of them behind many keys): 16, 8 and 4 shares, tiles that hang over
@pytest.mark.parametrize("h,g,d,page", [(45, 15, 128, 32), (40, 20, 64, 8), (48, 12, 64, 64), (45, 15, 64, 20)])
@pytest.mark.parametrize("window", [0, 70])
def test_attention_float32_tiles_of_many_requests(ops, h, g, d, page, window):
    spans = [(260 + i if i % 9 == 0 else 7 * i % 40, 1 + (i % 5 == 4)) for i in range(90)]
    n = sum(new for _, new in spans)
    assert ops._ask("yk_attn_f32_form", n, h, g, len(spans), 1, max(a + b for a, b in spans), 0) == 2
    got, want = _attention_case(ops, torch.float32, h, g, d, page, spans, window, 22, n_pages=900)
    close(got, want, 2e-5, 1e-5)


@pytest.mark.parametrize("window", [0, 9])
def test_attention_float32_tiles_keep_later_values_from_earlier_tokens(ops, window):
    n, h, g, d, page, gen = 70, 64, 16, 64, 16, torch.Generator().manual_seed(21)
    q, keys, values = (torch.randn(s, generator=gen) for s in ((n, h, d), (n, g, d), (n, g, d)))
    values[10, :, 5], values[30, :, 7], values[69, 2] = math.inf, math.nan, -math.inf
    pages = -(-n // page)
    kc, vc = torch.zeros((pages, g, page, d)), torch.zeros((pages, g, d, page))
    for pos in range(n):
        kc[pos // page, :, pos % page], vc[pos // page, :, :, pos % page] = keys[pos], values[pos]
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ctx = types.SimpleNamespace(arrays={"positions": dev(list(range(n))), "token_seq": dev([0] * n), "block_table_g0": dev([list(range(pages))])}, max_ctx=n)
    got = ops.attention(q.view(n, -1).to(DEV), h, g, d, kc.to(DEV), vc.to(DEV), page, 0.125, window, ctx, 0, None).cpu().view(n, h, d)
    for t in range(n):
        first = max(0, t - window + 1) if window else 0
        k, v = (x[first: t + 1].double().repeat_interleave(h // g, 1) for x in (keys, values))
        want = torch.einsum("hk,khd->hd", (torch.einsum("hd,khd->hk", q[t].double(), k) * 0.125).softmax(-1), v)
        assert bool((got[t].isfinite() == want.isfinite()).all()), t
        at = want.isfinite()
        close(got[t][at], want[at], 2e-5, 1e-5)


# pages whose slots are no multiple of four, and pages that do not start at a multiple of 16 bytes; few and many (token, head)s
@pytest.mark.parametrize("h,g,d,page,shift", [(4, 2, 16, 6, 0), (6, 3, 48, 1, 0), (5, 5, 80, 18, 0), (48, 12, 16, 7, 0), (4, 1, 32, 32, 1), (48, 12, 16, 16, 3)])
@pytest.mark.parametrize("window", [0, 3, 66])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_generic_any_pages(ops, h, g, d, page, shift, window, dtype, monkeypatch):
    def shifted(t):
        room = torch.full((t.numel() + shift,), float("nan"), dtype=t.dtype, device=DEV)
        room[shift:] = t.reshape(-1).to(DEV)
        return room[shift:].view(t.shape)

    monkeypatch.setitem(globals(), "device_cache", lambda ops, kc, vc: (shifted(kc), shifted(vc)))
    got, want = _attention_case(ops, dtype, h, g, d, page, SPANS, window, 19, n_pages=400)
    if dtype == torch.float32:
        close(got, want, 2e-5, 1e-5)
    else:
        close(got, want, 1e-2, 2**-7)


# one key alone in its block: the last of 65, or the first that a window of 68 shows behind 131; forms of eight waves and of one
@pytest.mark.parametrize("h,g,n", [(4, 4, 2), (64, 16, 64), (63, 63, 66)])
@pytest.mark.parametrize("last,window,low", [(64, 0, 64), (130, 68, 63), (130, 0, 3)])
def test_attention_generic_where_a_block_scores_minus_infinity(ops, h, g, n, last, window, low):
    """A key whose product with the query overflows to -inf has weight 0, also where it is all that its block shows."""
    d, page, gen = 16, 16, torch.Generator().manual_seed(n)
    keys, values = torch.randn((last + 1, g, d), generator=gen), torch.randn((last + 1, g, d), generator=gen)
    keys[low] = -3e38
    pages = -(-(last + 1) // page)
    kc, vc = torch.zeros((pages, g, page, d)), torch.zeros((pages, g, d, page))
    for pos in range(last + 1):
        kc[pos // page, :, pos % page], vc[pos // page, :, :, pos % page] = keys[pos], values[pos]
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ctx = types.SimpleNamespace(arrays={"positions": dev([last] * n), "token_seq": dev([0] * n), "block_table_g0": dev([list(range(pages))])}, max_ctx=last + 1)
    q = torch.rand((n, h, d), generator=gen) + 0.5
    got = ops.attention(q.view(n, -1).to(DEV), h, g, d, kc.to(DEV), vc.to(DEV), page, 0.25, window, ctx, 0, None)
    first = max(0, last - window + 1) if window else 0
    s = torch.einsum("nhd,khd->nhk", q.double(), keys[first:].double().repeat_interleave(h // g, 1)) * 0.25
    want = torch.einsum("nhk,khd->nhd", s.softmax(-1), values[first:].double().repeat_interleave(h // g, 1))
    close(got, want.reshape(n, -1), 2e-5, 1e-5)


@pytest.mark.parametrize("h,g,d,page", [(4, 2, 16, 16), (4, 1, 32, 32), (6, 3, 48, 16), (5, 5, 80, 64), (2, 1, 256, 16)])
@pytest.mark.parametrize("window", [0, 24])
def test_attention_generic_f32(ops, h, g, d, page, window):
    got, want = _attention_case(ops, torch.float32, h, g, d, page, SPANS, window, seed=3)
    close(got, want, 2e-5, 1e-5)


@pytest.mark.parametrize("h,g,d,page", [(4, 2, 16, 16), (6, 3, 48, 32)])
def test_attention_generic_bf16(ops, h, g, d, page):
    got, want = _attention_case(ops, torch.bfloat16, h, g, d, page, SPANS, 0, seed=4)
    close(got, want, 1e-2, 2**-7)


@pytest.mark.parametrize("h,g,d,page", [
    (8, 2, 128, 64), (6, 3, 64, 16), (4, 4, 64, 32), (32, 1, 128, 16), (5, 1, 64, 48), (24, 8, 128, 64), (40, 2, 64, 16),
    (4, 4, 64, 128), (12, 3, 128, 192),
])
@pytest.mark.parametrize("window", [0, 40])
def test_attention_mfma(ops, h, g, d, page, window):
    got, want = _attention_case(ops, torch.bfloat16, h, g, d, page, SPANS, window, seed=5)
    close(got, want, 2e-2, 2**-6)


def test_attention_mfma_long_context_splits(ops):
    """Few waves and many keys: the launch splits the keys and merges the parts."""
    spans = [(1500, 1), (900, 3), (0, 2)]
    got, want = _attention_case(ops, torch.bfloat16, 8, 2, 128, 64, spans, 0, seed=6, n_pages=48)
    close(got, want, 2e-2, 2**-6)
    got, want = _attention_case(ops, torch.bfloat16, 8, 2, 128, 64, spans, 700, seed=6, n_pages=48)
    close(got, want, 2e-2, 2**-6)


@pytest.mark.parametrize("plan", [(1, 1), (4, 1), (1, 5), (4, 3), (4, 7)])
@pytest.mark.parametrize("d,page", [(64, 32), (128, 32), (64, 64), (128, 128)])
def test_attention_mfma_every_way_of_dividing_keys(ops, plan, d, page):
    """Keys divided among the waves of a workgroup, among workgroups, or both, give the
    same result; spans include ones with fewer key blocks than waves (idle waves hold
    an empty part) and windows that cut the first block.  Pages of 32 tokens are plain,
    those of 64 and 128 tiled."""
    spans = [(1500, 1), (900, 3), (0, 2), (63, 1), (64, 1), (200, 2)]
    for window in (0, 700, 33):
        got, want = _attention_case(ops, torch.bfloat16, 8, 2, d, page, spans, window, seed=16, n_pages=3072 // page + 6, plan=plan)
        close(got, want, 2e-2, 2**-6)


@pytest.mark.parametrize("plan", [(4, 2), (4, 5), (1, 3)])
@pytest.mark.parametrize("h,g,d,page", [(8, 2, 128, 64), (6, 3, 64, 32), (32, 8, 128, 64), (24, 8, 128, 64), (32, 1, 128, 32)])
def test_attention_splits_merged_by_the_product(ops, plan, h, g, d, page, monkeypatch):
    """A step of up to 16 tokens leaves its splits unmerged for the product that follows:
    merged on their own they are the attention's output, and the product fed by the splits
    gives the bits of the product fed by the merged tensor (tiles of 8, 4, 5 and 1 tokens;
    heads that need two chunks; a product that keeps its K slices, one that does not, and
    one whose K slices are too long, which merges first)."""
    import yalis_amd.ops.hip as hip_ops
    from yalis_amd.ops.hip import SplitAttention, SplitSum

    monkeypatch.setattr(hip_ops, "MERGE_IN_PRODUCT_MAX_TOKENS", 16)  # as far as the kernel goes, not as far as it pays
    spans = [(700, 1), (64, 2), (300, 1), (0, 3), (1500, 1), (63, 2)]
    plain, _ = _attention_case(ops, torch.bfloat16, h, g, d, page, spans, 0, seed=21, n_pages=2700 // page + 8, plan=plan)
    # (the unmerged splits live in the library's workspace until the next attention: made last)
    got, want = _attention_case(ops, torch.bfloat16, h, g, d, page, spans, 0, seed=21, n_pages=2700 // page + 8, plan=plan, with_cols=True)
    assert isinstance(got, SplitAttention) and got.n_splits == plan[1] and got.shape == (10, h * d)
    merged = got.merge()
    close(merged, want, 2e-2, 2**-6)
    assert torch.equal(plain, merged)
    fed = 0
    for n_out, out_dtype, partial_ok in ((h * d, torch.bfloat16, True), (515, torch.float32, False), (48, torch.bfloat16, True)):
        w = rnd((n_out, h * d), torch.bfloat16, 22)
        fed += bool(ops._ask("yk_gemm_skinny_from_attention_ok", 10, n_out, h * d))
        y = ops.linear(got, w, out_dtype, partial_ok=partial_ok)
        a = y.tensor.clone() if isinstance(y, SplitSum) else y.clone()
        y = ops.linear(merged, w, out_dtype, partial_ok=partial_ok)
        b = y.tensor if isinstance(y, SplitSum) else y
        assert a.shape == b.shape and torch.equal(a, b), (n_out, out_dtype)
        close(a.sum(0) if partial_ok and a.dim() == 3 else a, merged.double().cpu() @ w.double().cpu().T, 3e-2, 2**-6)
    assert fed >= 1, "no product here took the splits itself"
    # more than 16 tokens: merged by the attention itself
    got, want = _attention_case(ops, torch.bfloat16, h, g, d, page, spans + [(5, 9)], 0, seed=21, n_pages=2700 // page + 8, plan=plan, with_cols=True)
    assert isinstance(got, torch.Tensor)
    close(got, want, 2e-2, 2**-6)


def _bits(t):
    return t.contiguous().view(torch.int16)


def _rotary_inside_cases():
    shapes = [(32, 8, 128, 128, 64, False), (6, 2, 128, 128, 64, False), (6, 3, 64, 32, 16, False), (8, 1, 64, 64, 128, True),
              (32, 1, 128, 64, 32, False), (24, 8, 128, 128, 64, False), (4, 4, 64, 0, 64, False)]
    for shape in shapes:
        for slices in (1, 3):
            for plan in (None, (1, 1), (4, 1), (4, 3), (1, 4)):
                yield (*shape, slices, plan, 0)
    # a window: its edge inside the block that holds the token, in an earlier block, in a split
    # that another workgroup owns; pages below it given back
    for shape in shapes[:4] + shapes[6:]:
        for window in (24, 100):
            for slices, plan in ((1, None), (3, (4, 3)), (1, (1, 4)), (3, (4, 1))):
                yield (*shape, slices, plan, window)


@pytest.mark.parametrize("h,g,d,rd,page,inter,slices,plan,window", list(_rotary_inside_cases()))
def test_attention_rotates_and_appends_in_its_launch(ops, plan, slices, h, g, d, rd, page, inter, window):
    """A step of single tokens: rotary + append inside the attention launch give the bits of
    rotary + append followed by attention, in the output and in the pages, whether the
    projection comes as bfloat16 rows or as float32 K slices, however the keys are divided,
    with the token's own key first, last or in the middle of a block of 64 (the slot it goes to
    holds NaN before), in tiled and in plain pages; and both agree with the plain reference.
    With a window: contexts one short of it, equal to it and beyond, the pages that lie wholly
    below the window given back (-1 in the block table, NaN where they were), and the key just
    outside the window made large, so that a window off by one would let it take the output."""
    from yalis_amd.ops.hip import RopeInLaunch, SplitSum

    cached = [0, 1, 31, 32, 63, 64, 65, 700, 1500, 127, 190]
    if window:
        cached += [window - 1, window, window + 1]
    n = len(cached)
    gen = torch.Generator().manual_seed(31)
    n_pages = sum(-(-(c + 1) // page) for c in cached) + 3
    order = torch.randperm(n_pages, generator=gen).tolist()
    kc = torch.full((n_pages, g, page, d), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((n_pages, g, d, page), float("nan"), dtype=torch.bfloat16)
    seqs, used = [], 0
    for c in cached:
        n_p = -(-(c + 1) // page)
        table = np.array(order[used : used + n_p], dtype=np.int32)
        used += n_p
        k = torch.randn((c, g, d), generator=gen).to(torch.bfloat16)
        v = torch.randn((c, g, d), generator=gen).to(torch.bfloat16)
        first_seen = max(0, c - window + 1) if window else 0  # the oldest key the token at position c sees
        if window and first_seen > 0:
            k[first_seen - 1] *= 40.0  # just outside: were it seen, it would take half the heads' outputs
            table[: first_seen // page] = -1  # pages wholly below the window: given back, never filled
        for pos in range(c):
            if table[pos // page] >= 0:
                kc[table[pos // page], :, pos % page, :] = k[pos]
                vc[table[pos // page], :, :, pos % page] = v[pos]
        seqs.append(SeqSpan(tokens=[0], first_position=c, block_tables=[table], state_slot=0))
    hb = build_host_batch(seqs, 1, page)
    tpt, big = ops.attention_tokens_per_tile(h, g), ops.attention_long_span_tile(h, g)
    arrays = named_arrays(hb, {"tiles": lambda b: attention_tiles(b, tpt, 1, big), "cols": lambda b: attention_token_columns(b, tpt, 1, big)})
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in arrays.items()}
    ctx = types.SimpleNamespace(arrays=dev, max_ctx=hb.max_ctx, max_qlen=1)
    cols = (h + 2 * g) * d
    if slices == 1:
        raw = (torch.randn((n, cols), generator=gen) * 1.2).to(torch.bfloat16).to(DEV)
        give = lambda: raw.clone()
        summed = raw.float().cpu()
    else:
        parts = (torch.randn((slices, n, cols), generator=gen) * 0.7).to(DEV)
        give = lambda: SplitSum(parts.clone(), torch.bfloat16)
        summed = (parts[0] + parts[1] + parts[2]).to(torch.bfloat16).float().cpu()
    cos, sin = _tables(rd, 1600) if rd else (None, None)
    scale = 1.0 / math.sqrt(d)
    positions, slots = dev["positions"], dev["slots_g0"]
    # rotary + append, then attention
    kc_a, vc_a = device_cache(ops, kc.clone(), vc.clone())
    q = ops.rope_append(give(), h, g, d, positions, cos, sin, rd, inter, kc_a, vc_a, slots, page)
    out_a = ops.attention(q, h, g, d, kc_a, vc_a, page, scale, window, ctx, 0, dev["tiles"], plan=plan)
    # both in one launch
    kc_b, vc_b = device_cache(ops, kc.clone(), vc.clone())
    out_b = ops.attention(give(), h, g, d, kc_b, vc_b, page, scale, window, ctx, 0, dev["tiles"], plan=plan,
                          rope=RopeInLaunch(cos, sin, rd, inter, True))
    assert torch.isfinite(out_b.float()).all()
    assert torch.equal(_bits(out_a), _bits(out_b))
    assert torch.equal(_bits(kc_a), _bits(kc_b)) and torch.equal(_bits(vc_a), _bits(vc_b))
    # queries only, against pages that already hold the tokens' keys and values (a run entry
    # that reads another entry's cache)
    q_rows = give()
    q_rows = SplitSum(q_rows.tensor[:, :, : h * d].contiguous(), torch.bfloat16) if slices > 1 else q_rows[:, : h * d].contiguous()
    out_c = ops.attention(q_rows, h, g, d, kc_b, vc_b, page, scale, window, ctx, 0, dev["tiles"], plan=plan,
                          rope=RopeInLaunch(cos, sin, rd, inter, False))
    assert torch.equal(_bits(out_a), _bits(out_c))
    # the plain reference
    qkv_r = summed.clone()
    kc_r, vc_r = kc.float(), vc.float()
    cpu = {k: torch.from_numpy(np.ascontiguousarray(v)) for k, v in arrays.items()}
    R.rope_append(qkv_r, h, g, d, cpu["positions"], None if cos is None else cos.cpu(), None if sin is None else sin.cpu(), rd, inter, kc_r, vc_r, cpu["slots_g0"], page)
    kc_r, vc_r = kc_r.to(torch.bfloat16).float(), vc_r.to(torch.bfloat16).float()
    q_r = qkv_r.view(n, -1, d)[:, :h].reshape(n, h * d).to(torch.bfloat16).float()
    want = R.attention(q_r, h, g, d, kc_r, vc_r, page, scale, window, types.SimpleNamespace(arrays=cpu), 0, None)
    close(out_b, want, 2e-2, 2**-6)


def test_attention_with_rotary_inside_leaves_splits_for_the_product(ops):
    """One or two tokens whose keys are split across workgroups: the launch with rotary inside
    leaves its splits unmerged too, and merged they are the two-kernel path's output."""
    from yalis_amd.ops.hip import RopeInLaunch, SplitAttention

    h, g, d, page = 32, 8, 128, 64
    gen = torch.Generator().manual_seed(5)
    cached = [1100, 300]
    n_pages = 30
    kc = torch.randn((n_pages, g, page, d), generator=gen).to(torch.bfloat16)
    vc = torch.randn((n_pages, g, d, page), generator=gen).to(torch.bfloat16)
    tables = [np.arange(0, 18, dtype=np.int32), np.arange(20, 25, dtype=np.int32)]
    seqs = [SeqSpan(tokens=[0], first_position=c, block_tables=[t], state_slot=0) for c, t in zip(cached, tables)]
    hb = build_host_batch(seqs, 1, page)
    tpt, big = ops.attention_tokens_per_tile(h, g), ops.attention_long_span_tile(h, g)
    arrays = named_arrays(hb, {"tiles": lambda b: attention_tiles(b, tpt, 1, big), "cols": lambda b: attention_token_columns(b, tpt, 1, big)})
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in arrays.items()}
    ctx = types.SimpleNamespace(arrays=dev, max_ctx=hb.max_ctx, max_qlen=1)
    raw = torch.randn((2, (h + 2 * g) * d), generator=gen).to(torch.bfloat16).to(DEV)
    cos, sin = _tables(d, 1200)
    kc_a, vc_a = device_cache(ops, kc.clone(), vc.clone())
    q = ops.rope_append(raw.clone(), h, g, d, dev["positions"], cos, sin, d, False, kc_a, vc_a, dev["slots_g0"], page)
    out_a = ops.attention(q, h, g, d, kc_a, vc_a, page, 0.09, 0, ctx, 0, dev["tiles"], plan=(4, 4))
    kc_b, vc_b = device_cache(ops, kc.clone(), vc.clone())
    got = ops.attention(raw.clone(), h, g, d, kc_b, vc_b, page, 0.09, 0, ctx, 0, dev["tiles"], plan=(4, 4), token_cols=dev["cols"],
                        rope=RopeInLaunch(cos, sin, d, False, True))
    assert isinstance(got, SplitAttention)
    assert torch.equal(_bits(got.merge()), _bits(out_a)) and torch.equal(_bits(kc_a), _bits(kc_b)) and torch.equal(_bits(vc_a), _bits(vc_b))
    # refused for steps that hold more than single tokens
    ctx.max_qlen = 2
    with pytest.raises(Exception, match="single tokens"):
        ops.attention(raw.clone(), h, g, d, kc_b, vc_b, page, 0.09, 0, ctx, 0, dev["tiles"], rope=RopeInLaunch(cos, sin, d, False, True))


@pytest.mark.parametrize("col_tiles", [1, 2])
@pytest.mark.parametrize("splits", [1, 2, 5, 16])
@pytest.mark.parametrize("h,g,d,page", [(8, 2, 128, 64), (6, 3, 64, 16), (32, 1, 128, 32), (6, 2, 64, 128)])
def test_attention_long_spans_with_split_keys(ops, splits, h, g, d, page, col_tiles):
    """Portions of prompts against a long cached context, the keys split across workgroups
    and merged: spans that end a tile early, a window, more splits than some tiles have key
    blocks (empty parts); one and two column tiles per wave (tiles of twice the tokens)."""
    spans = [(900, 70), (0, 130), (1500, 33), (40, 100)]
    for window in (0, 300):
        got, want = _attention_case(ops, torch.bfloat16, h, g, d, page, spans, window, seed=18, n_pages=3000 // page + 8, long_plan=splits, col_tiles=col_tiles)
        close(got, want, 2e-2, 2**-6)


def test_attention_policies_keep_their_invariants():
    """What the launch policies must hold whatever their constants are: a plan has one or four
    waves and at least one split, never more waves than key blocks could feed; the long-span
    kernel gets one or two column tiles, and splits only as far as all workgroups stay on the
    GPU at once."""
    from yalis_amd.ops.hip import HipOps

    for groups in (1, 8, 64, 512, 5000):
        for key_blocks in (1, 2, 5, 16, 128, 2048):
            waves, splits = HipOps.attention_plan(groups, key_blocks)
            assert waves in (1, 4) and 1 <= splits <= 256
            assert key_blocks > 1 or (waves, splits) == (1, 1)
            assert waves * splits < 2 * 8 + key_blocks * 2
    for workgroups in (1, 8, 120, 256, 400, 1024, 5000):
        for fewest in (0, 512, 1024, 7000):
            assert HipOps.attention_long_col_tiles(workgroups, fewest) in (1, 2)
        for key_blocks in (1, 4, 20, 64, 400):
            for col_tiles in (1, 2):
                splits = HipOps.attention_long_splits(workgroups, key_blocks, col_tiles)
                assert 1 <= splits <= 16
                assert splits == 1 or (splits * workgroups <= (768 if col_tiles == 1 else 512) and key_blocks // splits >= 8)


@pytest.mark.parametrize("h,g,d,page", [(32, 8, 128, 64), (24, 8, 128, 64), (32, 8, 64, 64)])
def test_attention_gives_one_result_under_every_plan_its_policies_choose(ops, h, g, d, page):
    """The policies decide from the batch how the keys are divided (waves, splits, column tiles of
    the long-span kernel).  For workloads on which they decide differently, the result under the
    policy's own choice is, within rounding, the result with nothing divided and the plain
    reference's: retuning a policy can change speed only."""
    from yalis_amd.ops.hip import HipOps

    workloads = {
        "single tokens behind long contexts": [(2000, 1), (900, 1), (64, 1)],
        "a few tokens each": [(1500, 3), (0, 2), (700, 4)],
        "a portion behind a long cached context": [(1400, 200)],
        "a prompt from nothing": [(0, 300)],
        "portions beside single tokens": [(1100, 150), (600, 1), (0, 90), (1300, 1)],
    }
    seen = set()
    for what, spans in workloads.items():
        n_pages = sum(-(-(c + n) // page) for c, n in spans) + 2
        chosen, want = _attention_case(ops, torch.bfloat16, h, g, d, page, spans, 0, seed=30, n_pages=n_pages)
        undivided, _ = _attention_case(ops, torch.bfloat16, h, g, d, page, spans, 0, seed=30, n_pages=n_pages, plan=(1, 1), long_plan=1)
        two, _ = _attention_case(ops, torch.bfloat16, h, g, d, page, spans, 0, seed=30, n_pages=n_pages, col_tiles=2)
        close(chosen, want, 2e-2, 2**-6)
        close(undivided, want, 2e-2, 2**-6)
        close(two, want, 2e-2, 2**-6)
        # (the parts of a division are merged in float32 and rounded once: what a division can
        # change is the order of float32 sums, a unit of bfloat16 at most)
        close(chosen, undivided.float().cpu(), 2e-2, 2**-7)
        longest = max(c + n for c, n in spans)
        seen.add(HipOps.attention_plan(len(spans) * g, -(-longest // 64)))
    assert len(seen) > 1, "the workloads were meant to make the policy choose differently"


@pytest.mark.parametrize("dtype,h,g,d,page", [(torch.bfloat16, 32, 8, 128, 64), (torch.bfloat16, 6, 3, 64, 16), (torch.float32, 4, 2, 48, 32)])
def test_attention_in_a_pool_beyond_4_gib(ops, dtype, h, g, d, page):
    """Pages whose offsets in the pool do not fit 32 bits (a pool of more than 4 GiB of keys, and
    as much of values; more than 2^31 elements): the same bits as from the same pages at the
    start of a small pool, for single tokens, short and long spans, keys split and not."""
    free = torch.cuda.mem_get_info()[0]
    per_page = g * page * d * (2 if dtype == torch.bfloat16 else 4)
    pool_pages = (2**31 + 2**28) // (g * page * d)
    if free < 2.5 * pool_pages * per_page:
        pytest.skip("not enough free device memory for the pool")
    assert pool_pages * g * page * d > 2**31
    spans = [(0, 5), (17, 1), (0, 300), (63, 2), (700, 1), (31, 34), (200, 130)]
    for plan, long_plan in ((None, None), ((4, 3), 2)):
        small, want = _attention_case(ops, dtype, h, g, d, page, spans, 0, seed=5, plan=plan, long_plan=long_plan, n_pages=128)
        big, _ = _attention_case(ops, dtype, h, g, d, page, spans, 0, seed=5, plan=plan, long_plan=long_plan, n_pages=128, pool_pages=pool_pages)
        assert torch.equal(small, big)
        close(small, want, 2e-5 if dtype == torch.float32 else 2e-2, 0 if dtype == torch.float32 else 2**-7)
        torch.cuda.empty_cache()


def test_attention_far_key_stands_out(ops):
    """One far key gets a large score: if a kernel skipped or misplaced it, the output
    would be the average of the others instead of (almost exactly) that key's value."""
    h, g, d, page = 8, 2, 128, 64
    n_ctx = 777
    for dtype in (torch.bfloat16, torch.float32):
        gen = torch.Generator().manual_seed(11)
        kc = torch.zeros((16, g, page, d), dtype=dtype)
        vc = torch.zeros((16, g, d, page), dtype=dtype)
        table = np.arange(15, 15 - 13, -1).astype(np.int32)  # pages in reverse
        k = torch.randn((n_ctx, g, d), generator=gen) * 0.1
        v = torch.randn((n_ctx, g, d), generator=gen)
        far = 5  # an early key, hundreds of tokens back
        q = torch.randn((1, h * d), generator=gen) * 0.1
        k[far] = 0
        k[far, 0, :] = q.view(h, d)[1] * 200.0  # head 1 (group 0) loves key `far`
        for pos in range(n_ctx):
            kc[table[pos // page], :, pos % page, :] = k[pos].to(dtype)
            vc[table[pos // page], :, :, pos % page] = v[pos].to(dtype)
        span = SeqSpan(tokens=[0], first_position=n_ctx - 1, block_tables=[table], state_slot=0)
        hb = build_host_batch([span], 1, page)
        tpt = ops.attention_tokens_per_tile(h, g)
        arrays = named_arrays(hb, {"tiles": lambda b: attention_tiles(b, tpt)})
        ctx = types.SimpleNamespace(
            arrays={kk: torch.from_numpy(np.ascontiguousarray(vv)).to(DEV) for kk, vv in arrays.items()},
            max_ctx=hb.max_ctx,
        )
        kc_d, vc_d = device_cache(ops, kc, vc)
        got = ops.attention(q.to(dtype).to(DEV), h, g, d, kc_d, vc_d, page, 1.0 / math.sqrt(d), 0, ctx, 0, ctx.arrays["tiles"])
        head1 = got.view(h, d)[1].float().cpu()
        close(head1, v[far, 0].to(dtype).float(), 2e-2, 2**-6)


# ------------------------------------------------------------------------ activation
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
def test_gated_act(ops, dtype, act):
    gu = rnd((9, 2 * 328), dtype, 12, scale=3.0)
    got = ops.gated_act(gu, act)
    want = R.gated_act(gu.float().cpu(), act)
    if dtype == torch.float32:
        close(got, want, 1e-6, 1e-5)
    else:
        close(got, want, 1e-3, 2**-8)


# -------------------------------------------------------------------------- sampling
def test_argmax_lowest_index_on_ties(ops):
    logits = rnd((5, 1000), torch.float32, 13)
    logits[0, 17] = 50.0
    logits[0, 900] = 50.0
    logits[1, 999] = 60.0
    got = ops.argmax(logits).cpu()
    want = torch.argmax(logits.cpu(), dim=-1)
    assert got[0].item() == 17 and got[1].item() == 999
    assert torch.equal(got[2:].long(), want[2:])


def _sample(ops, logits, temperature, top_k, top_p, seed, draw, whole_row=False):
    rows = logits.shape[0]
    f = lambda v, dt: torch.full((rows,), v, dtype=dt, device=DEV)
    return ops.sample(
        logits, f(temperature, torch.float32), f(top_k, torch.int32), f(top_p, torch.float32),
        f(seed, torch.int32), torch.arange(draw, draw + rows, dtype=torch.int32, device=DEV), whole_row=whole_row,
    ).cpu()


def test_sample_matches_plain(ops):
    import plain_llama as P

    logits = rnd((1, 515), torch.float32, 14, scale=2.0)
    for temperature, top_k, top_p in [(0.7, 0, 1.0), (1.0, 5, 1.0), (1.3, 0, 0.8), (0.9, 50, 0.5), (0.0, 0, 1.0), (1.0, 1, 1.0), (1.0, 0, 0.0)]:
        for draw in range(20):
            got = _sample(ops, logits, temperature, top_k, top_p, 99, draw)[0].item()
            want = P.sample_token(logits[0].cpu(), temperature, top_k or None, top_p, 99, draw)
            assert got == want, (temperature, top_k, top_p, draw)


SAMPLE_SETTINGS = [(0.7, 0, 1.0), (1.0, 5, 1.0), (1.3, 0, 0.8), (0.9, 50, 0.5), (1.0, 1, 1.0), (1.0, 0, 0.0),
                   (0.8, 3000, 0.95), (1.0, 6000, 0.9), (2.0, 0, 0.999), (1.1, 700, 1.0), (0.6, 5000, 1.0)]


@pytest.mark.parametrize("vocab,kind", [(32003, "peaked"), (128256, "peaked"), (20000, "flat"), (9001, "ties")])
def test_sample_large_vocabulary_matches_plain(ops, vocab, kind):
    """Rows larger than the candidate store: peaked rows narrow down to a few tokens, a
    flat row under top_p alone and a row of thousands of equal logits fall back to the
    whole-row path; every way gives the plain implementation's token, and the forced
    whole-row path agrees."""
    import plain_llama as P

    gen = torch.Generator().manual_seed(vocab)
    if kind == "peaked":
        logits = torch.randn((1, vocab), generator=gen) * 3.0
    elif kind == "flat":
        logits = torch.randn((1, vocab), generator=gen) * 0.01
    else:
        logits = torch.randn((1, vocab), generator=gen).round()  # a handful of distinct values
    logits = logits.to(DEV)
    for temperature, top_k, top_p in SAMPLE_SETTINGS:
        if kind == "ties" and top_p < 1.0:
            # which of several equally likely tokens top_p keeps is left to the sort in the
            # reference (yalis/external/sampling.py:24); the kernel drops them together
            continue
        for draw in range(4):
            want = P.sample_token(logits[0].cpu(), temperature, top_k or None, top_p, 7, draw)
            got = _sample(ops, logits, temperature, top_k, top_p, 7, draw)[0].item()
            slow = _sample(ops, logits, temperature, top_k, top_p, 7, draw, whole_row=True)[0].item()
            assert got == want and slow == want, (kind, temperature, top_k, top_p, draw, got, slow, want)


@pytest.mark.parametrize("kind", ["peaked", "flat"])
def test_sample_divided_rows(ops, kind):
    """Rows of a large vocabulary are divided among workgroups: rows with different settings in
    one launch give the plain implementation's tokens, and each goes the way its settings
    say: greedy, a race over the row (plain temperature; top_p once its threshold is known),
    settled among the candidates (top_k), or left to one workgroup (more candidates than fit)."""
    import plain_llama as P

    vocab = 128256
    settings = [(0.0, 0, 1.0, 0), (1.0, 0, 1.0, 1), (1.0, 0, 0.8, 1), (1.0, 50, 1.0, 3), (0.7, 50, 0.8, 3),
                (2.0, 0, 0.9, 1), (1.0, 6000, 1.0, 4), (0.5, 1, 1.0, 3), (1.3, 0, 0.0, 1), (0.9, 3000, 0.95, 3)]
    gen = torch.Generator().manual_seed(77)
    logits = torch.randn((len(settings), vocab), generator=gen) * (3.0 if kind == "peaked" else 0.3)
    if kind == "peaked":
        logits[:, 1000:1040] += 9.0
    logits[1, 5] = float("-inf")  # a masked token: never drawn, and no part of the bins' extent
    dev = logits.to(DEV)
    col = lambda j, dt: torch.tensor([st[j] for st in settings], dtype=dt, device=DEV)
    seeds = torch.arange(len(settings), dtype=torch.int32, device=DEV) + 11
    for draw in range(3):
        draws = torch.full((len(settings),), draw, dtype=torch.int32, device=DEV)
        paths = torch.full((len(settings),), -1, dtype=torch.int32, device=DEV)
        got = ops.sample(dev, col(0, torch.float32), col(1, torch.int32), col(2, torch.float32), seeds, draws, paths=paths).cpu()
        assert paths.cpu().tolist() == [st[3] for st in settings]
        for i, (temperature, top_k, top_p, _) in enumerate(settings):
            want = P.sample_token(logits[i], temperature, top_k or None, top_p, 11 + i, draw)
            assert got[i].item() == want, (kind, i, settings[i], draw, got[i].item(), want)


@pytest.mark.parametrize("vocab", [8192, 8195, 16385, 128256, 131077])
def test_sample_small_top_k(ops, vocab):
    """Rows with a small top_k are settled among what stretches of the row hand on, with the word
    that all rows are such or without it: the tokens of the whole-row path, at the largest top_k
    that is settled so, one more, ties with the top_k-th, more ties than are handed on, and rows
    with masked logits, at lengths whose rows start off 16 bytes."""
    gen = torch.Generator().manual_seed(vocab)
    rows = 9
    logits = torch.randn((rows, vocab), generator=gen) * 2.5
    logits[1] = logits[1].round()  # hundreds of equal logits
    logits[2, ::2] = float("-inf")
    logits[3, : vocab - 3] = float("-inf")  # fewer finite logits than top_k
    logits[4] = 1.5  # all equal: more than are handed on
    logits[5, 100:140] += 9.0
    logits[6] -= 200.0
    logits[7] = torch.sort(logits[7]).values  # a thread's largest logits lie side by side
    dev = logits.to(DEV)
    seeds = torch.arange(rows, dtype=torch.int32, device=DEV) + 3
    for k, top_p, temperature in [(1, 1.0, 1.0), (50, 0.8, 0.7), (50, 1.0, 1.3), (128, 0.95, 1.0), (129, 0.95, 1.0), (5, 0.0, 1.0)]:
        full = lambda v, dt: torch.full((rows,), v, dtype=dt, device=DEV)
        t = full(temperature, torch.float32)
        t[8] = 0.0
        args = (dev, t, full(k, torch.int32), full(top_p, torch.float32), seeds, full(k, torch.int32))
        want = ops.sample(*args, whole_row=True).tolist()
        paths = full(-1, torch.int32)
        assert ops.sample(*args, most_top_k=k, paths=paths).tolist() == want, (k, top_p)
        assert paths[8].item() == 0 and paths[0].item() == 3
        assert ops.sample(*args).tolist() == want, (k, top_p)


def test_sample_small_top_k_of_masked_rows(ops):
    """Logits of minus infinity have no mass and are not handed on: rows of which stretches are masked, or hold fewer finite logits than
    top_k or than top_k threads, are settled as others are (path 3).  100,001 logits: seven stretches of about 14,300."""
    vocab = 100001
    gen = torch.Generator().manual_seed(3)
    base = torch.randn((9, vocab), generator=gen) * 2.5
    logits = torch.full_like(base, float("-inf"))
    keep = [slice(vocab // 2, vocab), slice(20000, 20700), slice(50000, 50130), slice(99990, vocab), slice(7, 8), slice(0, vocab, 160), slice(0, vocab, 1000)]
    for row, where in enumerate(keep):
        logits[row, where] = base[row, where]
    for q in range(4):  # about 60 threads with 16 logits each, more than a stretch hands on
        logits[7, 4096 * q: 4096 * q + 240] = base[7, 4096 * q: 4096 * q + 240]
    logits[8] = torch.sort(base[8]).values  # the largest side by side
    dev, rows = logits.to(DEV), 9
    seeds = torch.arange(rows, dtype=torch.int32, device=DEV) + 11
    full = lambda v, dt: torch.full((rows,), v, dtype=dt, device=DEV)
    for k, top_p, temperature in [(50, 0.8, 0.7), (50, 1.0, 1.3), (128, 0.95, 1.0), (1, 1.0, 1.0), (100, 0.0, 1.0)]:
        args = (dev, full(temperature, torch.float32), full(k, torch.int32), full(top_p, torch.float32), seeds, full(k, torch.int32))
        want = ops.sample(*args, whole_row=True).tolist()
        for word in (k, 0):
            paths = full(-1, torch.int32)
            assert ops.sample(*args, most_top_k=word, paths=paths).tolist() == want, (k, top_p, word)
            assert not word or paths.tolist() == [3] * rows, (k, word, paths.tolist())


def test_sample_small_top_k_with_ties(ops):
    """Ties with the top_k-th that a stretch may not hand on, that are no list any more (1,024) or do not fit (4,096) are settled in the
    same sums of integers, from the row itself; more than that is one workgroup's work (path 4)."""
    vocab = 100001
    gen = torch.Generator().manual_seed(4)
    logits = torch.randn((8, vocab), generator=gen) * 2.5
    logits[0, 3000:3600] = 20.0  # more than a stretch hands on
    logits[1, 3000:4024] = 20.0  # as many as the list holds, and one more
    logits[2, 3000:4025] = 20.0
    logits[3, 10000:14000] = 20.0
    logits[3, 50000:50040] = 21.0  # with some above them
    logits[4, ::25] = 20.0  # 4,001 over all stretches, none with more than it may hand on
    logits[5, ::20] = 20.0  # 5,001
    logits[6] = 1.5
    logits[7, 3000:3600] = 9.0
    logits[7, 60000:60049] += 30.0  # the 50th is tied
    dev, rows = logits.to(DEV), 8
    seeds = torch.arange(rows, dtype=torch.int32, device=DEV) + 5
    full = lambda v, dt: torch.full((rows,), v, dtype=dt, device=DEV)
    for k, top_p, temperature in [(50, 0.8, 0.7), (50, 1.0, 2.0), (128, 0.3, 1.0), (1, 1.0, 1.0), (30, 0.0, 1.0)]:
        args = (dev, full(temperature, torch.float32), full(k, torch.int32), full(top_p, torch.float32), seeds, full(k, torch.int32))
        want = ops.sample(*args, whole_row=True).tolist()
        for word in (k, 0):
            paths = full(-1, torch.int32)
            assert ops.sample(*args, most_top_k=word, paths=paths).tolist() == want, (k, top_p, word)
            assert not word or paths.tolist() == [3, 3, 3, 3, 3, 4, 4, 3], (k, word, paths.tolist())


@pytest.mark.parametrize("vocab,k", [(300000, 128), (300000, 50), (400003, 122), (400003, 123), (1000003, 49)])
def test_sample_small_top_k_of_many_stretches(ops, vocab, k):
    """More stretches than waves (19, 25, 62): a wave gathers several, and the largest top_k that is settled is 3,072 / stretches."""
    gen = torch.Generator().manual_seed(k)
    logits = torch.randn((3, vocab), generator=gen) * 2.5
    logits[1] = (logits[1] * 4).round() / 4  # ties in every stretch
    logits[2] = torch.sort(logits[2]).values
    dev = logits.to(DEV)
    full = lambda v, dt: torch.full((3,), v, dtype=dt, device=DEV)
    args = (dev, full(0.9, torch.float32), full(k, torch.int32), full(0.9, torch.float32), full(8, torch.int32), full(2, torch.int32))
    want = ops.sample(*args, whole_row=True).tolist()
    for word in (k, 0):
        paths = full(-1, torch.int32)
        assert ops.sample(*args, most_top_k=word, paths=paths).tolist() == want, word
        assert not word or paths.tolist() == [3, 3, 3]


def test_sample_temperature_that_is_no_number(ops):
    """NaN is neither greedy nor a temperature: no probability is a number then, no token wins the race, and the most likely one stays
    (with a small top_k too, whose rows otherwise take what their stretches hand on)."""
    logits = torch.randn((3, 40000), generator=torch.Generator().manual_seed(5))
    dev, want = logits.to(DEV), logits.argmax(-1).tolist()
    full = lambda v, dt: torch.full((3,), v, dtype=dt, device=DEV)
    t = full(0.7, torch.float32)
    t[1] = float("nan")
    for k, top_p in [(50, 1.0), (50, 0.8), (0, 1.0), (0, 0.8), (500, 0.9)]:
        args = (dev, t, full(k, torch.int32), full(top_p, torch.float32), full(7, torch.int32), full(1, torch.int32))
        alone = ops.sample(*args, whole_row=True).tolist()
        for word in {0, min(k, 128)}:
            got = ops.sample(*args, most_top_k=word).tolist()
            assert got[1] == want[1] and got == alone, (k, top_p, word, got, want)


def test_sample_rows_are_independent(ops):
    """Many rows with different settings in one launch give what each gives alone."""
    vocab = 50000
    logits = rnd((6, vocab), torch.float32, 41, scale=2.5)
    temperature = torch.tensor([0.0, 0.7, 1.0, 1.2, 0.9, 1.0], dtype=torch.float32, device=DEV)
    top_k = torch.tensor([0, 40, 0, 5000, 0, 1], dtype=torch.int32, device=DEV)
    top_p = torch.tensor([1.0, 0.9, 0.5, 1.0, 1.0, 0.3], dtype=torch.float32, device=DEV)
    seeds = torch.arange(6, dtype=torch.int32, device=DEV) + 100
    draws = torch.arange(6, dtype=torch.int32, device=DEV) * 3
    both = ops.sample(logits, temperature, top_k, top_p, seeds, draws).cpu()
    for i in range(6):
        alone = ops.sample(logits[i : i + 1].contiguous(), temperature[i : i + 1], top_k[i : i + 1], top_p[i : i + 1],
                           seeds[i : i + 1], draws[i : i + 1]).cpu()
        assert both[i].item() == alone[0].item()


def test_sample_frequencies(ops):
    """Draws follow softmax(logits / T): chi-square over many draws."""
    vocab, draws, temperature = 12, 20000, 0.8
    logits = torch.linspace(-2, 2, vocab, device=DEV).repeat(draws, 1).contiguous()
    got = _sample(ops, logits, temperature, 0, 1.0, 5, 0)
    counts = torch.bincount(got.long(), minlength=vocab).double()
    p = torch.softmax(logits[0].cpu().double() / temperature, dim=0)
    chi2 = ((counts - draws * p) ** 2 / (draws * p)).sum().item()
    assert chi2 < 40.0, chi2  # 11 degrees of freedom: 40 is beyond the 99.99th percentile


def test_tiled_pages_layout(ops):
    """Which pages are tiled, and that the description of the order which the tests work
    from is the one the kernels write: a token's key and value land where it says."""
    assert ops.cache_tiled(torch.bfloat16, 128, 64) and ops.cache_tiled(torch.bfloat16, 64, 192)
    assert not ops.cache_tiled(torch.float32, 128, 64) and not ops.cache_tiled(torch.bfloat16, 128, 32)
    assert not ops.cache_tiled(torch.bfloat16, 48, 64) and not ops.cache_tiled(torch.bfloat16, 256, 64)
    h, g, d, page = 2, 1, 64, 128
    cos, sin = _tables(d, 4)
    for slot in (0, 5, 37, 64, 127, 128 + 70):
        qkv = rnd((1, (h + 2 * g) * d), torch.bfloat16, slot)
        kc = torch.zeros((2, g, page, d), dtype=torch.bfloat16, device=DEV)
        vc = torch.zeros((2, g, d, page), dtype=torch.bfloat16, device=DEV)
        want_k, want_v = qkv[0, h * d : (h + 1) * d].clone(), qkv[0, (h + 1) * d :].clone()
        ops.rope_append(qkv, h, g, d, torch.zeros(1, dtype=torch.int32, device=DEV), cos, sin, d, False, kc, vc,
                        torch.tensor([slot], dtype=torch.int32, device=DEV), page)  # position 0: no rotation
        kp, vp = R.untile_cache(kc.cpu(), vc.cpu())
        assert torch.equal(kp[slot // page, 0, slot % page], want_k.cpu()) and kp.ne(0).sum() == want_k.ne(0).sum()
        assert torch.equal(vp[slot // page, 0, :, slot % page], want_v.cpu()) and vp.ne(0).sum() == want_v.ne(0).sum()


def test_machine_probes_run_and_refuse_bad_sizes(ops):
    """The benchmark's two probes: they leave their input and (for ordinary data) their sink
    alone, count their flops, and refuse sizes their kernels do not take."""
    from yalis_amd.ops.hip import KernelError

    data = rnd((1 << 16,), torch.float32, 0)
    before = data.clone()
    sink = torch.zeros(1, dtype=torch.float32, device=DEV)
    for workgroups in (1, 7, 300):
        ops.probe_stream_read(data, workgroups, sink, nontemporal=workgroups == 7)
    assert ops.probe_mfma_bf16(3, 32, sink) == 3 * 4 * 32 * 4 * 16384
    torch.cuda.synchronize()
    assert torch.equal(data, before) and sink.item() == 0.0
    with pytest.raises(KernelError):
        ops.probe_stream_read(data[1:4], 4, sink)  # neither aligned nor whole 16-byte pieces
    with pytest.raises(KernelError):
        ops.probe_mfma_bf16(3, 10, sink)
