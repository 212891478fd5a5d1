"""Per-head products of a handful of tokens by pairs of columns, against float64."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
_ops = {}


def ops():
    if "o" not in _ops:
        from yalis_amd.ops.hip import HipOps

        _ops["o"] = HipOps("cuda:0")
    return _ops["o"]


@pytest.mark.parametrize("n", [1, 7, 8, 9, 32, 33])
@pytest.mark.parametrize("in_dim,out_dim", [(1, 2), (31, 62), (32, 64), (33, 66), (256, 130), (257, 64), (1000, 48), (40, 33), (1500, 20)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_head_products_by_pairs(dtype, in_dim, out_dim, n):
    """Few elements (one column a thread), as many as slices and one more, one more and one less than a round of weights, columns that do not fill a tile, an odd number of
    columns and heads too long for the pairs' workspace (both one column a thread).  A sum of in_dim products in float32, by slices: within 8
    roundings (2^-24) of the sum of their sizes."""
    check(3, n, in_dim, out_dim, dtype)


@pytest.mark.parametrize("h,n", [(32, 8), (33, 8), (64, 8), (64, 16), (65, 16), (64, 9), (16, 32), (17, 32)])
@pytest.mark.parametrize("in_dim", [31, 32, 33, 47, 48, 63, 64, 65, 95, 96, 127, 128, 129])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_where_pairs_end(dtype, in_dim, h, n):
    """Both sides of the lines in input elements and in workgroups (a head's 512 columns are eight of them for every eight tokens)."""
    check(h, n, in_dim, 512, dtype)


def check(h, n, in_dim, out_dim, dtype):
    o = ops()
    g = torch.Generator().manual_seed(in_dim + n)
    x = torch.randn(n, h * in_dim, generator=g).to(dtype)
    w = torch.randn(h, in_dim, out_dim, generator=g).to(dtype)
    got = o.head_linear(x.cuda(), w.cuda(), h, in_dim, out_dim, torch.float32).cpu().double().view(n, h, out_dim)
    xs, ws = x.double().view(n, h, in_dim).transpose(0, 1).contiguous(), w.double()
    want, size = (torch.matmul(a, b).transpose(0, 1) for a, b in ((xs, ws), (xs.abs(), ws.abs())))
    assert ((got - want).abs() <= 8 * 2.0 ** -24 * size).all()


# 16 heads x 512 columns: 128 units of 16 tokens x 64 columns for every 16 tokens; one, two (from 1,792 units) and four (from 3,584, of 128 elements
# and more) token tiles a wave, with tokens around the end of a tile and of a wave's run
@pytest.mark.parametrize("n", [33, 48, 208, 209, 225, 432, 433, 449, 577])
@pytest.mark.parametrize("in_dim,out_dim", [(32, 512), (128, 496), (64, 528)])
@pytest.mark.parametrize("first", [True, False])
def test_head_products_of_many_tokens(first, in_dim, out_dim, n):
    """bfloat16 in and float32 out, or float32 in (as two bfloat16 parts) and gated bfloat16 out."""
    o = ops()
    h = 16
    g = torch.Generator().manual_seed(n + in_dim)
    xd, od = (torch.bfloat16, torch.float32) if first else (torch.float32, torch.bfloat16)
    x = torch.randn(n, h * in_dim, generator=g).to(xd)
    w = torch.randn(h, in_dim, out_dim, generator=g).to(torch.bfloat16)
    gate = None if first else torch.randn(n, 3 + h * out_dim, generator=g).to(torch.bfloat16)
    w_t = w.transpose(1, 2).contiguous().cuda()
    got = o.head_linear(x.cuda(), w.cuda(), h, in_dim, out_dim, od, w_t=w_t, gate=None if gate is None else gate.cuda(), gate_col=3,
                        gate_elems=out_dim).cpu().double().view(n, h, out_dim)
    xs, ws = x.double().view(n, h, in_dim).transpose(0, 1).contiguous(), w.double()
    want, size = (torch.matmul(a, b).transpose(0, 1) for a, b in ((xs, ws), (xs.abs(), ws.abs())))
    if gate is not None:
        s = torch.sigmoid(gate[:, 3:].double()).view(n, h, out_dim)
        want, size = want * s, size * s
    # in_dim / 32 + 32 additions in float32; a float32 input's two parts leave out 2^-17 of it; the gate's own roundings; the output's rounding
    tol = (in_dim / 32 + 32) * 2.0**-24 * size + (0 if first else 2.0**-17 * size + 2.0**-8 * want.abs() + 1e-6)
    assert ((got - want).abs() <= tol).all()


# one, two and four token tiles a wave (see above), the last wave's run cut short; columns that leave one workgroup a head, and nine
@pytest.mark.parametrize("h,n", [(16, 100), (16, 225), (16, 449), (16, 577), (32, 113), (130, 441)])
@pytest.mark.parametrize("in_dim,out_dim,tail", [(128, 512, 64), (128, 64, 8), (128, 528, 24)])
@pytest.mark.parametrize("interleaved", [False, True])
def test_head_products_of_many_tokens_with_a_turned_tail(interleaved, in_dim, out_dim, tail, h, n):
    """The tail behind every head's product, whose tokens and pairs are shared among a head's workgroups: all of it is turned, and
    nothing beside it is written."""
    o = ops()
    g = torch.Generator().manual_seed(n + tail)
    x = torch.randn(n, h * (in_dim + tail), generator=g).to(torch.bfloat16)
    w = (torch.randn(h, in_dim, out_dim, generator=g)).to(torch.bfloat16)
    angle = torch.randn(3 * n, tail // 2, generator=g)
    positions = torch.randperm(3 * n, generator=g)[:n].to(torch.int32)
    rotation = types.SimpleNamespace(rotary_dim=tail, cos=angle.cos().cuda(), sin=angle.sin().cuda(), interleaved=interleaved)
    got = o.head_linear(x.cuda(), w.cuda(), h, in_dim, out_dim, torch.float32, tail=tail, rotation=rotation, positions=positions.cuda(),
                        w_t=w.transpose(1, 2).contiguous().cuda()).cpu().double().view(n, h, out_dim + tail)
    heads = x.double().view(n, h, in_dim + tail)
    xs = heads[:, :, :in_dim].transpose(0, 1).contiguous()
    want, size = (torch.matmul(a, b).transpose(0, 1) for a, b in ((xs, w.double()), (xs.abs(), w.double().abs())))
    assert ((got[:, :, :out_dim] - want).abs() <= (in_dim / 32 + 32) * 2.0**-24 * size).all()
    t = heads[:, :, in_dim:]
    a, b = (t[..., 0::2], t[..., 1::2]) if interleaved else (t[..., : tail // 2], t[..., tail // 2:])
    c, s = (v[positions.long()].double()[:, None] for v in (angle.cos(), angle.sin()))
    u, v = a * c - b * s, b * c + a * s
    turned = torch.stack([u, v], -1).flatten(-2) if interleaved else torch.cat([u, v], -1)
    # one rounded product and one fused multiply-add
    assert ((got[:, :, out_dim:] - turned).abs() <= 2.0**-23 * (a.abs() + b.abs()).max()).all()


@pytest.mark.parametrize("n", [449, 897, 1793])  # one, two and four token tiles a wave
def test_head_products_of_many_tokens_with_a_gate_per_head(n):
    o = ops()
    h, in_dim, out_dim = 16, 512, 128
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, h * in_dim, generator=g)
    w = (torch.randn(h, in_dim, out_dim, generator=g)).to(torch.bfloat16)
    gate = torch.randn(n, 5 + h, generator=g).to(torch.bfloat16)
    got = o.head_linear(x.cuda(), w.cuda(), h, in_dim, out_dim, torch.bfloat16, w_t=w.transpose(1, 2).contiguous().cuda(), gate=gate.cuda(),
                        gate_col=5).cpu().double().view(n, h, out_dim)
    xs = x.double().view(n, h, in_dim).transpose(0, 1).contiguous()
    s = torch.sigmoid(gate[:, 5:].double())[..., None]
    want, size = (torch.matmul(a, b).transpose(0, 1) * s for a, b in ((xs, w.double()), (xs.abs(), w.double().abs())))
    tol = ((in_dim / 32 + 32) * 2.0**-24 + 2.0**-17) * size + 2.0**-8 * want.abs() + 1e-6
    assert ((got - want).abs() <= tol).all()
