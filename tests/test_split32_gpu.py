"""fp32 forward on split bf16 operands (stage 3, ``fa_s3_split``) against the fp64 oracle.

Sizes: both sides of every tile edge (32-row workgroups up to 128-row ones, partial last tiles of
32, 64 and 128 keys), each tile the rule can pick, GQA, strided views. Values: very different
magnitudes side by side, and everything that must leave the split path for the fp32 matrix
instructions (magnitudes from 2^60 on, nonzero ones below 2^-110, infinities).

The bar is the fp32 one of the other parity tests (|O err| <= 1e-5 + 1e-5 |ref|). With scaled V the
absolute part scales with V: every term of the error is proportional to it.
"""

import math

import numpy as np
import pytest
import torch

import fused_attn
from oracle.oracle import math_reference

pytestmark = pytest.mark.gpu


def _inputs(b, h, hkv, n, d, seed=0):
    gen = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(b, x, n, d, generator=gen).cuda() for x in (h, hkv, hkv))


def _check(q, k, v, causal, v_scale=1.0, atol=1e-5):
    o, lse = fused_attn.forward_stage(q, k, v, 3, is_causal=causal)
    ref, lse64 = math_reference(q, k, v, is_causal=causal)
    err = np.abs(o.double().cpu().numpy() - ref)
    assert np.isfinite(err).all()
    assert (err <= atol * v_scale + 1e-5 * np.abs(ref)).all(), err.max()
    # An fp32 sum of D products is off by at most D 2^-24 of its terms' magnitude, and so is an LSE
    # that one large score decides: 1e-3 alone would ask for less than half an ulp beyond 2^13.
    bound = 1e-3 + q.shape[-1] * 2.0 ** -24 * np.abs(lse64)
    assert (np.abs(lse.double().cpu().numpy() - lse64) <= bound).all()
    return o


@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("shape", [
    (1, 1, 1, 32, 64), (1, 2, 1, 96, 64), (1, 2, 2, 160, 64),       # BR 32 x BC 128
    (1, 2, 2, 32, 128), (1, 2, 1, 96, 128), (1, 2, 2, 352, 128),    # BR 64 x BC 64
    (3, 16, 4, 288, 64),                                            # BR 64 x BC 128
    (4, 16, 4, 288, 64), (4, 16, 8, 288, 128),              # BR 128 x BC 64 (causal 64 rows)
    (4, 24, 8, 352, 64),                                    # BR 64 x BC 128 in three rounds
    (2, 2, 1, 32, 128), (9, 32, 8, 96, 128),                        # one narrow tile per head
    (8, 32, 8, 352, 64), (8, 32, 8, 288, 128),                      # BR 128 x BC 32
], ids=lambda s: "B%d_H%d_Hkv%d_N%d_D%d" % s)
def test_tile_edges(shape, causal):
    _check(*_inputs(*shape), causal)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bc", [32, 64])
def test_forced_widths(d, bc):
    q, k, v = _inputs(1, 2, 2, 416, d, seed=1)
    fused_attn.set_debug_overrides(0, bc)
    try:
        _check(q, k, v, True)
    finally:
        fused_attn.set_debug_overrides(0, 0)


# Largest magnitude of a tensor at ordinary sizes, at the upper end of the split path's range, 2^60,
# and past it. q and k scale against each other, so that the scores keep the size of ordinary ones.
@pytest.mark.parametrize("top", [2.0 ** -7, 2.0 ** -6, 0.5, 2.0 ** 9 - 2.0 ** -14, 2.0 ** 9,
                                 2.0 ** 60 - 2.0 ** 36, 2.0 ** 60, 1e30], ids=lambda x: "%g" % x)
@pytest.mark.parametrize("which", ["q", "k", "v"])
def test_range_ends(which, top):
    q, k, v = _inputs(1, 2, 2, 192, 64, seed=2)

    def at(x):  # the tensor clipped to and scaled by its largest magnitude
        return x.clamp(-4, 4) / 4 * top

    scale = top / 4
    if which == "v":
        _check(q, k, at(v), True, v_scale=max(scale, 1e-30))
    elif which == "q":
        _check(at(q), k / scale, v, True)
    else:
        _check(q / scale, at(k), v, True)


@pytest.mark.parametrize("factor", [2e3, 1e19, 1e-36], ids=lambda x: "%g" % x)
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("tensor", [0, 1, 2], ids=["q", "k", "v"])
def test_one_row_of_another_size(tensor, d, factor):
    """One row of the last tile far larger than the rest, or outside the range, whose workgroups start
    over on the fp32 path after tiles of the split one. Everything that the row does not decide keeps
    the ordinary bar; the terms it has a part in add what fp32 leaves of them."""
    x = list(_inputs(1, 2, 2, 416, d, seed=3))
    x[tensor][0, 0, 401] *= factor
    if factor > 1e18 and tensor < 2:  # scores of ordinary size for the row, none for the others
        x[1 - tensor] /= factor
    q, k, v = x
    o, _ = fused_attn.forward_stage(q, k, v, 3)
    ref, _ = math_reference(q, k, v)
    bar = 1e-5 + 1e-5 * np.abs(ref)
    qd, kd, vd = (t[0, 0].double() for t in x)
    p = torch.softmax(qd @ kd.t().contiguous() / math.sqrt(d), dim=-1)
    if tensor == 2:
        # A sum of 416 products, each weight off by a few ulp of a score of size 4: 1e-6 of them.
        bar[0, 0] += 1e-6 * (p @ vd.abs()).cpu().numpy()
    elif factor == 2e3:
        # A score of D products is off by at most D 2^-24 of their magnitudes; it moves O by
        # p (1 - p) of that, times the spread of v.
        s_err = d * 2.0 ** -24 * (qd.abs() @ kd.abs().t().contiguous()) / math.sqrt(d)
        move = (s_err * p * (1 - p)).sum(dim=-1, keepdim=True) * 2 * vd.abs().max()
        bar[0, 0] += move.cpu().numpy()
    assert (np.abs(o.double().cpu().numpy() - ref) <= bar).all()


def test_zero_tiles_are_exact():
    q, k, v = _inputs(1, 2, 2, 256, 64, seed=4)
    z = torch.zeros_like(v)
    assert torch.equal(_check(q, k, z, True), z)
    o = _check(q, torch.zeros_like(k), v, False)  # flat rows: the mean of v
    assert (o - v.mean(dim=2, keepdim=True)).abs().max() <= 1e-6


def test_non_finite_inputs():
    """NaN and infinities reach the rows that see them and no other, as on the fp32 path; a key that is
    -inf in one entry scores -inf against positive queries and weighs nothing."""
    q, k, v = _inputs(1, 1, 1, 256, 64, seed=5)
    for bad in (math.nan, math.inf):
        n = v.clone()
        n[0, 0, 200, 3] = bad
        o, _ = fused_attn.forward_stage(q, k, n, 3, is_causal=True)
        fine = torch.isfinite(o[0, 0])
        assert not fine[200:, 3].any()          # rows that see key 200
        assert fine[:192].all()                 # rows of earlier 32-key blocks
        assert fine[:, [c for c in range(64) if c != 3]].all()
    n = k.clone()
    n[0, 0, 77, 5] = -math.inf
    qp = q.abs() + 1e-3
    o, _ = fused_attn.forward_stage(qp, n, v, 3)
    keep = [j for j in range(256) if j != 77]
    s = (qp[0, 0].double() @ k[0, 0, keep].double().t().contiguous()) / 8
    ref = torch.softmax(s, dim=-1) @ v[0, 0, keep].double()
    assert (o[0, 0].double() - ref).abs().max() <= 1e-5


def test_strided_views_match_dense():
    x = torch.randn(2, 224, 3, 4, 64, generator=torch.Generator().manual_seed(6)).cuda()
    q, k, v = (x[:, :, i].transpose(1, 2) for i in range(3))
    o = fused_attn.forward_strided(q, k, v, is_causal=True)
    assert torch.equal(o, fused_attn.forward(*(t.contiguous() for t in (q, k, v)), is_causal=True))


# Factors of q, k and v, together and against each other.
@pytest.mark.parametrize("factors", [(1e-3, 1e3, 1e-3), (300.0, 1 / 300, 300.0), (2e-6, 5e5, 1.0),
                                     (1.0, 1.0, 2e-9), (1.0, 1.0, 1e9), (1.0, 1.0, 4e-3)],
                         ids=lambda f: "q%g_k%g_v%g" % f)
@pytest.mark.parametrize("d", [64, 128])
def test_scaled_tensors(d, factors):
    q, k, v = (x * f for x, f in zip(_inputs(1, 4, 2, 416, d, seed=4), factors))
    _check(q, k, v, True, v_scale=factors[2])


# A scale so small that the scores' factor would leave fp32's range beside tiny q and k.
def test_tiny_scale():
    q, k, v = _inputs(1, 2, 2, 96, 64, seed=5)
    q, k = q * 1e-6, k * 1e-6
    o, lse = fused_attn.forward_stage(q, k, v, 3, is_causal=True, scale=1e-25)
    ref, lse64 = math_reference(q, k, v, is_causal=True, scale=1e-25)
    assert (np.abs(o.double().cpu().numpy() - ref) <= 1e-5 + 1e-5 * np.abs(ref)).all()
    assert np.abs(lse.double().cpu().numpy() - lse64).max() <= 1e-3


def _column_errors(o, ref):
    """Largest error of each output column over that column's largest value."""
    err = np.abs(o.double().cpu().numpy() - ref)
    return err.max(axis=(0, 1, 2)) / np.abs(ref).max(axis=(0, 1, 2))


# Values of very different magnitude side by side: an fp32 product keeps 24 bits of each operand
# whatever stands beside it, so every output is held to its own magnitude. The bar is the fp32 one,
# 1e-5 of it.
@pytest.mark.parametrize("small", [1e-3, 1e-6, 1e-10, 1e-25, 1e-36], ids=lambda x: "%g" % x)
@pytest.mark.parametrize("d", [64, 128])
def test_small_v_columns_beside_large_ones(d, small):
    q, k, v = _inputs(1, 2, 2, 288, d, seed=7)
    v[..., 5] *= small
    v[..., 9] *= 400.0
    o, _ = fused_attn.forward_stage(q, k, v, 3, is_causal=True)
    ref, _ = math_reference(q, k, v, is_causal=True)
    assert (_column_errors(o, ref) <= 1e-5).all()


@pytest.mark.parametrize("small", [1e-3, 1e-6, 1e-10, 1e-25, 1e-36], ids=lambda x: "%g" % x)
@pytest.mark.parametrize("d", [64, 128])
def test_small_first_rows_of_v(d, small):
    """The first causal rows depend on the first keys alone."""
    q, k, v = _inputs(1, 2, 2, 160, d, seed=8)
    v[:, :, :20] *= small
    o, _ = fused_attn.forward_stage(q, k, v, 3, is_causal=True)
    ref, _ = math_reference(q, k, v, is_causal=True)
    err = np.abs(o.double().cpu().numpy() - ref)[:, :, :20].max()
    assert err <= 1e-5 * np.abs(ref[:, :, :20]).max()


@pytest.mark.parametrize("spread", [1e3, 1e5, 1e8], ids=lambda x: "%g" % x)
@pytest.mark.parametrize("d", [64, 128])
def test_opposite_channel_scales(d, spread):
    """One channel of q is large where k's is small: its term of the scores is of ordinary size."""
    q, k, v = _inputs(1, 2, 2, 288, d, seed=9)
    q[..., 3] *= spread
    k[..., 3] /= spread
    q[..., 11] /= spread
    k[..., 11] *= spread
    _check(q, k, v, True)


def test_small_weights_on_large_values():
    """Outputs that one large value of small probability decides keep fp32's relative precision."""
    q, k, v = _inputs(1, 1, 1, 128, 64, seed=10)
    k[:, :, 70] = -6.0 * q.mean(dim=2) * 64.0 / (q.mean(dim=2) ** 2).sum() ** 0.5
    v[:, :, 70] = 1e6
    o, _ = fused_attn.forward_stage(q, k, v, 3)
    ref, _ = math_reference(q, k, v)
    p = torch.softmax(q[0, 0].double() @ k[0, 0].double().t().contiguous() / 8, dim=-1)
    # Per row: a score is off by up to D 2^-24 of its terms, and its weight by as much, relatively.
    terms = (q[0, 0].abs().double() @ k[0, 0].abs().double().t().contiguous() / 8).amax(dim=-1)
    bar = ((1e-6 + 64 * 2.0 ** -24 * terms)[:, None] * (p @ v[0, 0].abs().double())).cpu().numpy()
    assert (np.abs(o[0, 0].double().cpu().numpy() - ref[0, 0]) <= bar).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n,at", [(96, 64), (416, 224)])
def test_causal_rows_do_not_see_later_keys(d, n, at):
    """Bitwise: what later keys and rows hold changes nothing in the rows before them."""
    q, k, v = _inputs(1, 2, 2, n, d, seed=11)
    o, lse = fused_attn.forward_stage(q, k, v, 3, is_causal=True)
    for x, f in zip((q, k, v), (300.0, 1e-4, 3000.0)):
        x[:, :, at:] *= f
    o2, lse2 = fused_attn.forward_stage(q, k, v, 3, is_causal=True)
    assert torch.equal(o[:, :, :at], o2[:, :, :at]) and torch.equal(lse[:, :, :at], lse2[:, :, :at])
