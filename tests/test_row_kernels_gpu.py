"""Kernels of a step's rows (norms, activations, slices, few-row products, experts of few pairs, heads, recurrences) at sizes that do not fill their threads."""
import math

import pytest
import torch

import kernel_refs as R
from yalis_amd.ops.hip import HipOps, SplitSum

pytestmark = pytest.mark.gpu
_ops = {}


def ops():
    if "o" not in _ops:
        _ops["o"] = HipOps("cuda:0")
    return _ops["o"]


def close(got, want, tol):
    err = (got.double().cpu() - want.double()).abs().max().item() / want.double().abs().max().item()
    assert err <= tol, err


@pytest.mark.parametrize("n", [3, 1023, 1024])
@pytest.mark.parametrize("width", [4, 260, 516, 1028, 2052, 4092, 4096])
def test_norms_of_few_and_many_rows(n, width):
    """Float32 rows: a row's sum of squares is added in up to width / 64 + 10 roundings of 2^-24, halved by the root: 4e-6 holds
    for 4,096; both kernels write every column, and none of the next row's."""
    o, g = ops(), torch.Generator().manual_seed(width + n)
    res, br, other = (torch.randn(n, width, generator=g) for _ in range(3))
    w, w2 = torch.rand(width, generator=g) + 0.5, torch.rand(width, generator=g) + 0.5
    post, pre = (w, w2, 1e-5, True), (w2, None, 1e-6, False)
    dev = lambda c: tuple(t.cuda() if torch.is_tensor(t) else t for t in c)
    r_ref, r_dev = res.clone(), res.clone().cuda()
    want = R.sandwich_norm(r_ref, br, post, 0.3, pre, None, torch.float32)
    close(o.sandwich_norm(r_dev, br.cuda(), dev(post), 0.3, dev(pre), None, torch.float32), want, 4e-6)
    close(r_dev, r_ref, 4e-6)
    r_ref, r_dev = res.clone(), res.clone().cuda()
    want = R.sum_norm(r_ref, [(br, w, 1e-5), (other, w2, 1e-5)], 0.5, None, 2.0, w, 1e-5, True, torch.bfloat16)
    got = o.sum_norm(r_dev, [(br.cuda(), w.cuda(), 1e-5), (other.cuda(), w2.cuda(), 1e-5)], 0.5, None, 2.0, w.cuda(), 1e-5, True, torch.bfloat16)
    close(r_dev, r_ref, 4e-6)
    close(got, want, 2 ** -8)  # (the rounded copy: a rounding to bfloat16 may fall to the other side)


@pytest.mark.parametrize("kind", ["relu2", "silu", "gelu_tanh"])
@pytest.mark.parametrize("shape,shift", [((1, 4), 0), ((3, 1020), 0), ((3, 1021), 0), ((5, 1024), 1)])
def test_activation_in_pieces(kind, shape, shift):
    """Whole pieces, a count that is none and rows that are not aligned: within one rounding to bfloat16, NaN where the input is."""
    o, g = ops(), torch.Generator().manual_seed(shape[1])
    flat = torch.randn(shape[0] * shape[1] + shift, generator=g).to(torch.bfloat16)
    if kind != "relu2":  # (whose maximum with 0 drops it)
        flat[shift] = float("nan")
    x = flat.cuda()[shift:].view(shape)
    got, want = o.activation(x, kind, torch.bfloat16).cpu(), R.activation(flat[shift:].view(shape), kind, torch.bfloat16)
    assert torch.equal(got.isnan(), want.isnan())
    close(got.nan_to_num().float(), want.nan_to_num().float(), 2 ** -8)


@pytest.mark.parametrize("kind", ["relu2", "silu", "gelu_tanh"])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("columns", [1020, 1021])
@pytest.mark.parametrize("slices", [2, 8, 9, 10, 17])
def test_activation_of_slices(slices, columns, out_dtype, kind):
    """A product's slices, added eight at a time: one round, a full one, one and two more, two full ones, in whole pieces and in none; the
    sum is rounded to the product's type first.  The slices are added in their order, so only the activation's own roundings remain."""
    o, g = ops(), torch.Generator().manual_seed(slices)
    parts = torch.randn(slices, 3, columns, generator=g)
    total = parts[0]
    for p in parts[1:]:
        total = total + p
    want = R.activation(total.to(out_dtype), kind, out_dtype)
    got = o.activation(SplitSum(parts.cuda(), out_dtype), kind, out_dtype)
    close(got, want, 2e-6 if out_dtype == torch.float32 else 2 ** -8)


@pytest.mark.parametrize("n,width", [(3, 516), (2, 6148), (1030, 2052), (2, 10240)])  # one piece a thread, two, two of many rows, four
@pytest.mark.parametrize("top", [1, 2, 3, 8, 9])
def test_norm_add_of_expert_rows(n, width, top):
    """A branch and a token's expert rows together, more of either than are asked for at once: float32 sums in the reference's order, up to the
    rounding of the row's sum of squares (4e-6 as above)."""
    o, g = ops(), torch.Generator().manual_seed(width + top)
    res, src, e = torch.randn(n, width, generator=g), torch.randn(n, width, generator=g), torch.randn(n * top, width, generator=g)
    w = torch.rand(width, generator=g) + 0.5
    for branch in (src, None):
        r_ref, r_dev = res.clone(), res.clone().cuda()
        want = R.norm_add(r_ref, branch, w, 1e-5, True, torch.bfloat16, e, 0.3)
        got = o.norm_add(r_dev, None if branch is None else branch.cuda(), w.cuda(), 1e-5, True, torch.bfloat16, e.cuda(), 0.3)
        close(r_dev, r_ref, 4e-6)
        close(got.float(), want.float(), 2 ** -8)


def in_order(t, dtype):
    """The slices added one after another in float32 and rounded as a product of ``dtype`` would be."""
    total = torch.zeros_like(t[0])
    for one in t:
        total = total + one
    return total.to(dtype).float()


def same(got, want):
    return torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


CONSUMERS = {
    "add_rmsnorm": lambda o, res, d, w, rows: o.add_rmsnorm(res, d, w, 1e-5, True, torch.bfloat16),
    "gather_add_rmsnorm": lambda o, res, d, w, rows: o.gather_add_rmsnorm(res, d, rows, w, 1e-5, False, torch.float32),
    "rmsnorm": lambda o, res, d, w, rows: o.rmsnorm(d, w, 1e-5, False, torch.bfloat16),
    "norm_add": lambda o, res, d, w, rows: o.norm_add(res, d, w, 1e-5, True, torch.bfloat16),
    "sum_norm": lambda o, res, d, w, rows: o.sum_norm(res, [(d, w, 1e-5)], 0.5, w, 2.0, w, 1e-5, False, torch.bfloat16),
    "sum_norm second": lambda o, res, d, w, rows: o.sum_norm(res, [(res * 0.5, None, 1e-5), (d, w, 1e-5)], 0.5, None, 2.0, w, 1e-5, True, torch.bfloat16),
    "sandwich_norm": lambda o, res, d, w, rows: o.sandwich_norm(res, d, (w, w, 1e-5, True), 0.5, (w, None, 1e-5, False), None, torch.float32),
    "sandwich_norm rows": lambda o, res, d, w, rows: o.sandwich_norm(res, d, None, 1.0, (w, w, 1e-5, True), rows, torch.bfloat16),
    "activation": lambda o, res, d, w, rows: o.activation(d, "relu2", torch.float32),
    "gated_act": lambda o, res, d, w, rows: o.gated_act(d, "silu", torch.float32),
}


# rows that fill the chip (one piece a thread and two), rows of three and of four pieces
@pytest.mark.parametrize("consumer,n,width", [(c, n, w) for c in CONSUMERS for n, w in ((300, 1028), (1025, 1028), (1025, 256))]
                         + [(c, 2, w) for c in ("add_rmsnorm", "gather_add_rmsnorm", "rmsnorm", "norm_add") for w in (10244, 14340)]
                         + [(c, 2, 16384) for c in ("add_rmsnorm", "gather_add_rmsnorm", "rmsnorm")])
def test_slices_of_many_and_wide_rows(consumer, n, width):
    """As above where fewer slices are asked for at once: the bits of the sum itself."""
    o, g = ops(), torch.Generator(device="cuda").manual_seed(width + n)
    call, w = CONSUMERS[consumer], torch.rand(width, device="cuda", generator=g) + 0.5
    rows = torch.tensor([n - 1, 0, n // 2], dtype=torch.int32, device="cuda")
    for slices in (2, 3, 4, 5, 8, 9):
        t, res = torch.randn(slices, n, width, device="cuda", generator=g), torch.randn(n, width, device="cuda", generator=g)
        for dtype in (torch.float32, torch.bfloat16):
            first, second = res.clone(), res.clone()
            got, want = call(o, first, SplitSum(t, dtype), w, rows), call(o, second, in_order(t, dtype), w, rows)
            assert same(got, want) and same(first, second), slices


# rows and widths whose pieces of four end in a workgroup, a wave and a row; 64 rows take slices by rows, more of them by pieces; 6 and 258 the general kernel
@pytest.mark.parametrize("rows", [1, 3, 64, 65, 1027])
@pytest.mark.parametrize("inter,group", [(4, 0), (6, 0), (96, 4), (256, 0), (258, 0), (1020, 0), (1028, 4), (1028, 0), (3076, 0)])
def test_gated_pairs_of_any_rows(rows, inter, group):
    """The plain pairs of the slices' sum (float32 exp: 2e-6; rounded once: 2^-8), and the bits of that sum itself at any number of slices."""
    o, g = ops(), torch.Generator().manual_seed(rows + inter)
    for slices in (1, 2, 3, 8, 9):
        parts = torch.randn(slices, rows, 2 * inter, generator=g)
        for dtype in (torch.float32, torch.bfloat16):
            whole = in_order(parts, dtype)
            got = o.gated_act(SplitSum(parts.cuda(), dtype) if slices > 1 else whole.cuda(), "silu", dtype, group=group)
            assert torch.equal(got, o.gated_act(whole.cuda(), "silu", dtype, group=group))
            assert torch.equal(got, o.gated_act(whole.to(dtype).cuda(), "silu", dtype, group=group))
            close(got, R.gated_act_general(whole, "silu", dtype, group), 2e-6 if dtype == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("consumer", CONSUMERS)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,width", [(3, 4), (3, 516), (2, 4096), (2, 6148), (1025, 520)])  # one piece of a row a thread, two and four
def test_any_number_of_slices(consumer, dtype, n, width):
    """Slices go through registers in groups that depend on their number: the same bits as of the sum itself at every number,
    infinities and NaN of single slices included."""
    o, g = ops(), torch.Generator(device="cuda").manual_seed(width + n)
    call = CONSUMERS[consumer]
    w = torch.rand(width, device="cuda", generator=g) + 0.5
    rows = torch.tensor([n - 1, 0, n // 2], dtype=torch.int32, device="cuda")
    for slices in (2, 3, 4, 5, 8, 9, 12, 13, 16, 17, 20, 24, 25, 33):
        t = torch.randn(slices, n, width, device="cuda", generator=g)
        t[slices - 1, n - 1, width - 1] = float("inf") if slices % 2 else float("nan")
        t[:, 0, 0] = -0.0
        res = torch.randn(n, width, device="cuda", generator=g)
        res2, whole = res.clone(), in_order(t, dtype)
        got = call(o, res, SplitSum(t, dtype), w, rows)
        want = call(o, res2, whole, w, rows)
        assert same(got, want) and same(res, res2), slices


@pytest.mark.parametrize("h,g,d", [(8, 2, 128), (12, 4, 64), (20, 4, 64), (36, 2, 128)])  # 4, 3, 5 and 18 heads that share keys
@pytest.mark.parametrize("page", [48, 64, 192])
def test_decode_attention_with_slices_and_splits(h, g, d, page):
    """Single tokens behind contexts at the edges of half blocks, blocks and pages (sizes that are no powers of two among them), the slots
    behind them NaN: any number of slices of the projection gives the bits of its sum, and any number of splits, up to more
    than are merged at once, agrees with the plain reference within bfloat16's rounding of probabilities and values (2e-2, 2^-6 as elsewhere)."""
    import types

    o, gen = ops(), torch.Generator().manual_seed(page + h)
    cached = [0, 31, 32, 47, 48, 63, 64, 95, 96, 191, 192, 1000]
    n, width = len(cached), -(-1001 // page)
    pages = n * width
    kc, vc = torch.full((pages, g, page, d), float("nan")), torch.full((pages, g, d, page), float("nan"))
    table = torch.randperm(pages, generator=gen).int().view(n, width)
    for r, c in enumerate(cached):
        for p in range(c):
            kc[table[r, p // page], :, p % page] = torch.randn(g, d, generator=gen)
            vc[table[r, p // page], :, :, p % page] = torch.randn(g, d, generator=gen)
    kc, vc = kc.bfloat16(), vc.bfloat16()
    tiles = torch.tensor([[r, r, 1, c] for r, c in enumerate(cached)], dtype=torch.int32)
    arrays = {"block_table_g0": table, "positions": torch.tensor(cached, dtype=torch.int32), "token_seq": torch.arange(n, dtype=torch.int32)}
    ctx = types.SimpleNamespace(arrays={k: v.cuda() for k, v in arrays.items()}, max_ctx=1001, max_qlen=1)
    angle = torch.rand(1001, d // 2, generator=gen) * 6
    cos, sin = angle.cos(), angle.sin()
    from test_kernels_gpu import device_cache
    from yalis_amd.ops.hip import RopeInLaunch

    rope = RopeInLaunch(cos.cuda(), sin.cuda(), d, False, True)
    slots = torch.tensor([int(table[r, c // page]) * page + c % page for r, c in enumerate(cached)], dtype=torch.int32)
    for slices in (1, 2, 4, 7, 8, 9, 17):
        parts = torch.randn(slices, n, (h + 2 * g) * d, generator=gen) / math.sqrt(slices)
        rows = in_order(parts, torch.bfloat16)
        want = None
        for splits in (1, 2, 3, 7, 8, 9, 12):
            results = []
            for given in (SplitSum(parts.cuda(), torch.bfloat16), rows.bfloat16().cuda()):
                kd, vd = device_cache(o, kc.clone(), vc.clone())
                results.append(o.attention(given, h, g, d, kd, vd, page, d ** -0.5, 0, ctx, 0, tiles.cuda(), rope=rope, plan=(4, splits)).float())
            assert torch.equal(*results), (slices, splits)
            if want is None:
                q, kr, vr = rows.clone(), kc.float(), vc.float()
                R.rope_append(q, h, g, d, arrays["positions"], cos, sin, d, False, kr, vr, slots, page)
                want = R.attention(q[:, : h * d].bfloat16().float(), h, g, d, kr.bfloat16().float(), vr.bfloat16().float(), page, d ** -0.5, 0,
                                   types.SimpleNamespace(arrays=arrays), 0, None)
            err = (results[0].cpu() - want).abs()
            assert bool((err <= 2e-2 + 2 ** -6 * want.abs()).all()), (slices, splits, err.max().item())


# rows that fill a load of x and do not; K at a chunk, beyond one round of the waves, with remainders; 16 waves and eight; a last group of columns that is none
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(40, 8), (40, 256), (33, 2056), (48, 2304), (16, 6144), (40, 6400), (4112, 2312)])
def test_few_rows_in_one_workgroup_by_rows_of_x(m, n, k):
    """Each row of x against a row of ones but for one place far along K: a step that met another row's or another step's x would show."""
    o, g = ops(), torch.Generator().manual_seed(m + k)
    x, w = torch.randn(m, k, generator=g).bfloat16(), torch.randn(n, k, generator=g).bfloat16()
    wide = torch.full((m, k + 8), float("nan"), dtype=torch.bfloat16)  # rows further apart than they are long
    wide[:, :k] = x
    want = x.double() @ w.double().T
    got = o.gemm_cols(wide.cuda()[:, :k], w.cuda(), torch.float32)
    # float32 sums of k products of about 1: each addition rounds by 2^-24 of a sum of up to 4 sqrt(k)
    assert (got.cpu().double() - want).abs().max() <= 4 * math.sqrt(k) * 2.0 ** -24 * math.sqrt(k / 32 + 16) * 4
    one = torch.zeros(m, k, dtype=torch.bfloat16)
    for r in range(m):
        one[r, (r * 37 + k // 2) % k] = 1.0
    got = o.gemm_cols(one.cuda(), w.cuda(), torch.bfloat16).cpu()
    assert torch.equal(got, torch.stack([w[:, (r * 37 + k // 2) % k] for r in range(m)]))


def test_few_rows_far_apart():
    """Rows of x that reach over 2^31 elements: the bits of the same rows side by side, as a product, with a bias and with pairs."""
    o, g, bf = ops(), torch.Generator(device="cuda").manual_seed(3), torch.bfloat16
    m, n, k, apart = 3, 1024, 264, 2 ** 30 + 8
    wide = torch.empty(m, apart, dtype=bf, device="cuda")
    wide[:, :k] = torch.randn(m, k, device="cuda", generator=g)
    x, w, bias = wide[:, :k], torch.randn(n, k, device="cuda", generator=g).to(bf), torch.randn(n, device="cuda", generator=g)
    near = x.contiguous()
    for out in (torch.float32, bf):
        assert torch.equal(o.linear(x, w, out), o.linear(near, w, out)) and torch.equal(o.gemm_cols(x, w, out), o.gemm_cols(near, w, out))
        assert torch.equal(o.linear(x, w, out, bias=bias), o.linear(near, w, out, bias=bias))
    assert torch.equal(o.gate_up_act(x, w, 8, "silu", bf), o.gate_up_act(near, w, 8, "silu", bf))


@pytest.mark.parametrize("n,top,experts", [(1, 1, 2), (1, 4, 4), (4, 2, 16), (5, 3, 7), (16, 4, 32), (33, 1, 2), (64, 1, 2), (21, 3, 3)])
@pytest.mark.parametrize("hidden,ff", [(32, 32), (96, 64), (160, 288), (1056, 1024), (2048, 96)])  # fewer steps of 32 than waves, than are asked for ahead, more
def test_experts_of_few_pairs(n, top, experts, hidden, ff):
    """Pairs that find their own tiles: the plain arithmetic (bfloat16 rounds y: 2e-2 as for every path), each token's rows the bits that it
    has alone, whatever its neighbours choose (more than 16 of one expert among them), and a token of NaN changes no other's rows."""
    o, g = ops(), torch.Generator().manual_seed(n + hidden + experts)
    x = torch.randn(n, hidden, generator=g).bfloat16()
    ids = torch.randint(-2, 55, (n,), generator=g, dtype=torch.int32)  # (ids out of the table's range read its ends)
    table = torch.rand(50, experts, generator=g).argsort(-1)[:, :top].to(torch.int32).contiguous()
    wgu = (torch.randn(experts, 2, ff, hidden, generator=g) / hidden ** 0.5).bfloat16()
    wd = (torch.randn(experts, hidden, ff, generator=g) / ff ** 0.5).bfloat16()
    act = ("clamped_swish", 1.5, 1.702)
    dev = [t.cuda() for t in (x, ids, table, wgu, wd)]
    got = o.moe_experts(*dev, act).cpu()
    want = R.moe_experts(x, ids.clamp(0, 49), table, wgu, wd, act)
    assert (got - want).abs().max() <= 2e-2 * max(1.0, float(want.abs().max()))
    for t in {0, n // 2, n - 1}:
        alone = o.moe_experts(dev[0][t: t + 1], dev[1][t: t + 1], *dev[2:], act).cpu()
        assert torch.equal(alone, got[t * top: (t + 1) * top])
    # a choice per token, with a row of x per token and per pair, without a gate
    choice = table[ids.clamp(0, 49).long()].contiguous().cuda()
    assert torch.equal(o.moe_experts(dev[0], None, choice, dev[3], dev[4], act, input_per_token=True).cpu(), got)
    assert torch.equal(o.moe_experts(dev[0].repeat_interleave(top, 0), None, choice, dev[3], dev[4], act).cpu(), got)
    up = wgu[:, :1].contiguous()
    close(o.moe_experts(dev[0], dev[1], dev[2], up.cuda(), dev[4], "relu2").cpu(), R.moe_experts(x, ids.clamp(0, 49), table, up, wd, "relu2"), 2e-2)
    if n > 1:
        bad = dev[0].clone()
        bad[0] = float("nan")
        got2 = o.moe_experts(bad, *dev[1:], act).cpu()
        assert torch.equal(got2[top:], got[top:])  # (its own rows: the pair's clamps drop a NaN)


@pytest.mark.parametrize("steps", [1, 4, 5, 7, 8, 9, 13, 20, 28, 29, 33, 36, 61])  # of 32: one to four waves with some, one to sixteen a wave, last waves with fewer or none
def test_experts_of_few_pairs_at_any_depth(steps):
    """Both products at every remainder of what a wave asks for at once: the bits of the sorted pairs' form, which walks K two steps at a time."""
    o, g = ops(), torch.Generator(device="cuda").manual_seed(steps)
    n, top, experts, k = 12, 2, 5, 32 * steps
    for hidden, ff in ((k, 64), (64, k)):
        x = torch.randn(n, hidden, device="cuda", generator=g).bfloat16()
        table = torch.rand(n, experts, device="cuda", generator=g).argsort(-1)[:, :top].to(torch.int32).contiguous()
        ids = torch.arange(n, dtype=torch.int32, device="cuda")
        wgu = (torch.randn(experts, 2, ff, hidden, device="cuda", generator=g) / hidden ** 0.5).bfloat16()
        wd = (torch.randn(experts, hidden, ff, device="cuda", generator=g) / ff ** 0.5).bfloat16()
        got, ask = o.moe_experts(x, ids, table, wgu, wd, "silu"), o._ask
        o._ask = lambda name, *args: 0 if name == "yk_moe_few_pairs_ok" else ask(name, *args)
        try:
            assert torch.equal(got, o.moe_experts(x, ids, table, wgu, wd, "silu"))
        finally:
            del o._ask


# both sides of every line of yk_moe_few_pairs_ok: tokens, choices a token, experts, width, ff
@pytest.mark.parametrize("n,top,experts,hidden,ff,few", [
    (16, 2, 17, 4096, 1024, True), (16, 2, 16, 4096, 1024, False), (16, 2, 4, 4096, 1024, True), (16, 2, 5, 4096, 1024, False),
    (12, 2, 8, 4096, 992, True), (12, 2, 8, 4096, 1024, False), (25, 1, 8, 4096, 992, False), (16, 2, 8, 2048, 1024, True), (16, 2, 8, 2080, 1024, False), (32, 1, 2, 2048, 96, True), (33, 1, 9, 2048, 96, True),
    (33, 1, 8, 2048, 96, False), (33, 1, 9, 2080, 96, False), (64, 1, 2, 1024, 96, True), (64, 1, 15, 1056, 96, False), (64, 1, 16, 1056, 96, True),
    (65, 1, 33, 96, 96, False)])
def test_which_pairs_route_themselves(n, top, experts, hidden, ff, few):
    """The rule's answer, and the same bits in either form."""
    o, g = ops(), torch.Generator(device="cuda").manual_seed(n + hidden)
    x = torch.randn(n, hidden, device="cuda", generator=g).bfloat16()
    table = torch.rand(n, experts, device="cuda", generator=g).argsort(-1)[:, :top].to(torch.int32).contiguous()
    wgu = (torch.randn(experts, 2, ff, hidden, device="cuda", generator=g) / hidden ** 0.5).bfloat16()
    wd = (torch.randn(experts, hidden, ff, device="cuda", generator=g) / ff ** 0.5).bfloat16()
    assert bool(o._ask("yk_moe_few_pairs_ok", n * top, experts, hidden, ff, hidden)) == few
    forms, ask = [], o._ask
    try:
        for take in (0, int(n * top <= 64)):
            o._ask = lambda name, *args: take if name == "yk_moe_few_pairs_ok" else ask(name, *args)
            forms.append(o.moe_experts(x, None, table, wgu, wd, "silu", input_per_token=True))
    finally:
        del o._ask
    assert torch.equal(*forms) and torch.equal(forms[0], o.moe_experts(x, None, table, wgu, wd, "silu", input_per_token=True))


@pytest.mark.parametrize("dtype,n,top,experts", [(torch.bfloat16, 5, 2, 3), (torch.bfloat16, 40, 2, 16), (torch.bfloat16, 100, 1, 2), (torch.bfloat16, 200, 1, 2),
                                                 (torch.float32, 5, 2, 3)])  # pairs that route themselves, tiles of 16, 64 and 128 pairs, the general form
def test_experts_out_of_range_are_the_nearest(dtype, n, top, experts):
    """Numbers below zero and beyond the last expert in the table: the rows that the first and the last expert give, in the same bits."""
    o, g = ops(), torch.Generator().manual_seed(n)
    hidden, ff = 64, 96
    x = torch.randn(n, hidden, generator=g).to(dtype).cuda()
    ids = torch.randint(0, 30, (n,), generator=g, dtype=torch.int32).cuda()
    table = torch.randint(-3, experts + 4, (30, top), generator=g, dtype=torch.int32)
    table[0, 0], table[1, 0] = -2 ** 31, 2 ** 31 - 1
    wgu = (torch.randn(experts, 2, ff, hidden, generator=g) / hidden ** 0.5).to(dtype).cuda()
    wd = (torch.randn(experts, hidden, ff, generator=g) / ff ** 0.5).to(dtype).cuda()
    got = o.moe_experts(x, ids, table.cuda(), wgu, wd, "silu")
    assert torch.equal(got, o.moe_experts(x, ids, table.clamp(0, experts - 1).cuda(), wgu, wd, "silu"))


def test_more_experts_than_are_offered():
    """4,097 experts are refused, of however few pairs."""
    from yalis_amd.ops.hip import KernelError

    o, bf = ops(), torch.bfloat16
    for n in (2, 70):
        table = torch.zeros(n, 1, dtype=torch.int32, device="cuda")
        with pytest.raises(KernelError, match="4,096 experts"):
            o.moe_experts(torch.zeros(n, 32, dtype=bf, device="cuda"), None, table, torch.zeros(4097, 2, 32, 32, dtype=bf, device="cuda"),
                          torch.zeros(4097, 32, 32, dtype=bf, device="cuda"), "silu")


def _spans(spans, slots):
    from types import SimpleNamespace

    dev = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    starts = [sum(spans[:i]) for i in range(len(spans))]
    return SimpleNamespace(max_qlen=max(spans), arrays={"seq_qstart": dev(starts), "seq_qlen": dev(spans), "state_slots": dev(slots),
                                                        "token_seq": dev([i for i, s in enumerate(spans) for _ in range(s)])})


@pytest.mark.parametrize("dtype,w_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("spans", [[1], [1] * 9, [1] * 64, [2, 1, 5, 3], [1] * 65])
@pytest.mark.parametrize("channels,bias,act", [(8, True, None), (128, False, "silu"), (136, True, "silu"), (1160, True, None)])
def test_convolution_of_few_tokens(dtype, w_dtype, spans, channels, bias, act):
    """Two channels a thread against the sum in float64 (rounded once: 2^-8 of the largest in bfloat16, four products in float32), the state moved."""
    o, g = ops(), torch.Generator().manual_seed(channels + len(spans))
    n, slots = sum(spans), [len(spans) - i for i in range(len(spans))]
    x, w = torch.randn(n, channels + 8, generator=g).to(dtype)[:, :channels], torch.randn(channels, 4, generator=g).to(w_dtype)
    b = torch.randn(channels, generator=g).to(w_dtype) if bias else None
    state = torch.randn(len(spans) + 1, 3, channels, generator=g).to(dtype)
    want, kept, first = [], state.clone(), 0
    for slot, s in zip(slots, spans):
        rows = torch.cat([state[slot], x[first: first + s]])
        want += [sum(w[:, j].double() * rows[t + j].double() for j in range(4)) + (b.double() if bias else 0) for t in range(s)]
        kept[slot], first = rows[-3:], first + s
    want = torch.stack(want)
    want = torch.nn.functional.silu(want) if act else want
    st = state.cuda()
    wide = torch.zeros(n, channels + 8, dtype=dtype, device="cuda")
    wide[:, :channels] = x.cuda()
    got = o.causal_conv(wide[:, :channels], w.cuda(), b.cuda() if bias else None, st, _spans(spans, slots), act=act, move_state=True)
    close(got, want, 2.0 ** -8 if dtype == torch.bfloat16 else 1e-6)
    assert torch.equal(st.cpu(), kept)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 8, 9, 16, 17, 64])
@pytest.mark.parametrize("blocks,size", [(3, 32), (2, 160), (1, 256), (2, 288)])  # fewer steps of 32 than are asked for ahead, all, more
def test_gated_recurrence_of_few_tokens(n, blocks, size):
    """Single tokens against float64 from the same bfloat16 numbers: the products are summed in float32 (size roundings of 2^-24), the
    states then within 2e-5, the outputs rounded to bfloat16; the kept inputs exactly."""
    o, g, c = ops(), torch.Generator().manual_seed(n + size), blocks * size
    r = lambda *s: torch.randn(*s, generator=g).bfloat16()
    u, y, x, ba, bi, lam = r(n, c), r(n, c), r(n, c), r(c), r(c), r(c)
    wa, wi = ((torch.randn(blocks, size, size, generator=g) / size ** 0.5).bfloat16() for _ in range(2))
    S, kept = torch.randn(n + 1, c, generator=g), r(n + 1, 3, c)
    slots = list(range(n, 0, -1))
    product = lambda m, b: torch.einsum("nbk,bok->nbo", u.double().view(n, blocks, size), m.double()).reshape(n, c) + b.double()
    log_a = -8.0 * torch.nn.functional.softplus(lam.double()) * torch.sigmoid(product(wa, ba))
    want_S, want_kept = S.double(), kept.clone()
    want_S[slots] = torch.exp(log_a) * S.double()[slots] + torch.sqrt(-torch.expm1(2 * log_a)) * torch.sigmoid(product(wi, bi)) * u.double()
    want_kept[slots] = torch.cat([kept[slots][:, 1:], x[:, None]], 1)
    Sd, kd = S.cuda(), kept.cuda()
    t = lambda m: m.transpose(1, 2).contiguous().cuda()
    got = o.rglru(u.cuda(), y.cuda(), x.cuda(), t(wa), ba.cuda(), t(wi), bi.cuda(), lam.cuda(), 8.0, Sd, kd, 4, _spans([1] * n, slots), wa=wa.cuda(), wi=wi.cuda())
    close(Sd, want_S, 2e-5)
    close(got, want_S[slots] * torch.nn.functional.gelu(y.double(), approximate="tanh"), 2.0 ** -8)
    assert torch.equal(kd.cpu(), want_kept)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [3, 21])
@pytest.mark.parametrize("head_dim,value_dim,rotary,page,interleaved", [(2, 6, 2, 1, False), (66, 62, 34, 3, True), (128, 64, 128, 8, False), (130, 128, 64, 8, True),
                                                                        (256, 256, 256, 16, False)])
def test_projection_rows_at_the_ends_of_a_wave(dtype, n, head_dim, value_dim, rotary, page, interleaved):
    """Heads that end inside a lane's first piece, at a wave's end and in the last piece, pages of one token; then the same queries turned
    back and gated.  Float32: norms of up to 256 elements and two products a turn, 4e-6; bfloat16: rounded once or twice, 2^-7 of the largest."""
    from yalis_amd.parts.base import Rotation

    o, g, H, G = ops(), torch.Generator().manual_seed(head_dim + n), 3, 2
    qkv = torch.randn(n, H * head_dim + G * (head_dim + value_dim), generator=g).to(dtype)
    bias = torch.randn(qkv.shape[1], generator=g)
    positions = torch.randint(0, 40, (n,), generator=g, dtype=torch.int32)
    slots = torch.randperm(4 * page + n, generator=g)[:n].to(torch.int32)
    qn, kn = (torch.rand(head_dim, generator=g) + 0.5).to(dtype), (torch.rand(head_dim, generator=g) + 0.5).to(dtype)
    table = lambda width: [f(torch.arange(40.0)[:, None] * 100.0 ** (-torch.arange(width // 2) / (width // 2))) for f in (torch.cos, torch.sin)]
    rot, vrot = (Rotation(*table(w), w, inter) for w, inter in ((rotary, interleaved), (value_dim, not interleaved)))
    on = lambda r: Rotation(r.cos.cuda(), r.sin.cuda(), r.rotary_dim, r.interleaved)
    n_pages = (4 * page + n) // page + 1
    pages = lambda d: (torch.zeros(n_pages, G, page, head_dim, dtype=dtype, device=d), torch.zeros(n_pages, G, value_dim, page, dtype=dtype, device=d))
    (k, v), (kr, vr) = pages("cuda"), pages("cpu")
    got = o.qkv_prepare(qkv.cuda(), H, G, head_dim, value_dim, positions.cuda(), dtype, q_norm=qn.cuda(), k_norm=kn.cuda(), qk_eps=1e-6, rotation=on(rot),
                        value_norm_eps=1e-6, value_rotation=on(vrot), k_cache=k, v_cache=v, slots=slots.cuda(), page_size=page, bias=bias.cuda())
    want = R.qkv_prepare(qkv, H, G, head_dim, value_dim, positions, dtype, q_norm=qn, k_norm=kn, qk_eps=1e-6, rotation=rot, value_norm_eps=1e-6,
                         value_rotation=vrot, k_cache=kr, v_cache=vr, slots=slots, page_size=page, bias=bias)
    if o.masked_pages_tiled(dtype, head_dim, value_dim, page):
        k, v = R.untile_cache(k, v)
    tol = 4e-6 if dtype == torch.float32 else 2.0 ** -7
    for a, b in ((got, want), (k, kr), (v, vr)):
        close(a, b.to(a.dtype), tol)


@pytest.mark.parametrize("chunk", [1, 7, 8, 9, 64])
def test_gated_recurrence_of_ragged_chunks(chunk):
    """Chunks of less than, exactly and just over the tokens that are asked for at once, cut anywhere: against float64 token by token, 2e-5
    for the kept state (as above; a decay is at most 1, so errors do not grow along the span)."""
    o, g, blocks, size = ops(), torch.Generator().manual_seed(chunk), 2, 32
    spans, c = [33, 1, 40, 71], blocks * size
    n, slots = sum(spans), [3, 1, 4, 2]
    r = lambda *s: torch.randn(*s, generator=g).bfloat16()
    u, y, x, ba, bi, lam = r(n, c), r(n, c), r(n, c), r(c), r(c), r(c)
    wa, wi = ((torch.randn(blocks, size, size, generator=g) / size ** 0.5).bfloat16() for _ in range(2))
    S, kept = torch.randn(len(spans) + 1, c, generator=g), r(len(spans) + 1, 3, c)
    product = lambda m, b: torch.einsum("nbk,bok->nbo", u.double().view(n, blocks, size), m.double()).reshape(n, c) + b.double()
    log_a = -torch.nn.functional.softplus(lam.double()) * torch.sigmoid(product(wa, ba))
    b = torch.sqrt(-torch.expm1(2 * log_a)) * torch.sigmoid(product(wi, bi)) * u.double()
    want_S, want, want_kept, rows, first_chunk, first = S.double(), [], kept.clone(), [], [0], 0
    for i, (slot, length) in enumerate(zip(slots, spans)):
        for t in range(first, first + length):
            want_S[slot] = torch.exp(log_a[t]) * want_S[slot] + b[t]
            want.append(want_S[slot].clone())
        want_kept[slot] = torch.cat([kept[slot], x[first: first + length]])[-3:]
        rows += [(i, first + t, min(chunk, length - t)) for t in range(0, length, chunk)]
        first_chunk.append(len(rows))
        first += length
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    t, Sd, kd = (lambda m: m.transpose(1, 2).contiguous().cuda()), S.cuda(), kept.cuda()
    got = o.rglru(u.cuda(), y.cuda(), x.cuda(), t(wa), ba.cuda(), t(wi), bi.cuda(), lam.cuda(), 1.0, Sd, kd, 4, _spans(spans, slots), wa=wa.cuda(), wi=wi.cuda(),
                  chunks=dev(rows), seq_chunk0=dev(first_chunk))
    close(Sd, want_S, 2e-5)
    close(got, torch.stack(want) * torch.nn.functional.gelu(y.double(), approximate="tanh"), 2.0 ** -8)
    assert torch.equal(kd.cpu(), want_kept)
