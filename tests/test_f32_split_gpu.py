"""The float32 kernel whose products are products of bf16 parts (64 query rows a workgroup, steps of one 16-key tile, one or two sets of
waves that share out the keys), where its tiles, sets and rings of position rows can go wrong; and the other float32 kernel at the sizes that
the library no longer gives it."""
import math

import pytest
import torch

import test_f32_gpu as f32
from helpers import in_kernel, make_inputs
from turbodeberta_amd import _lib
from turbodeberta_amd.ops.flash_attention import flash_attention_with_disentangled
from turbodeberta_amd.ops.flash_attention_varlen import flash_attention_with_disentangled_varlen

pytestmark = pytest.mark.gpu
DIRECT, ONE_SET, TWO_SETS = _lib.TDB_FLAG_PERSISTENT, _lib.TDB_FLAG_RESIDENT, _lib.TDB_FLAG_PERSISTENT | _lib.TDB_FLAG_RESIDENT
# Products and sums of 32 bits on both sides, in other orders: a few units of 2^-24 of values of order 1 for each of some 64 to 300 terms.
BOUND = 2e-5


def _in_and_generic(flag, call):
    with in_kernel(flag):
        got = call(False)
    return got, call(True)


@pytest.mark.parametrize("flag", [ONE_SET, TWO_SETS])
@pytest.mark.parametrize("terms", [("pk", "pq"), ("pk",), ("pq",), ()])
@pytest.mark.parametrize("L", [1, 16, 17, 63, 64, 65, 96, 128, 129, 200, 273])      # one tile to 18: odd and even, rings once and three times around
def test_tiles_and_terms(flag, terms, L):
    d = {n: t.cuda() for n, t in make_inputs(L, 3, 2, L, 64, 32, 128).items()}
    lens = torch.tensor([L, max(1, L - 17), max(1, L // 3)], dtype=torch.int32, device="cuda")
    got, ref = _in_and_generic(flag, lambda g: flash_attention_with_disentangled(
        d["q"], d["k"], d["v"], None, None, False, f32.SCALE, 32, 128, seqlens_k=lens, force_generic=g, **{
            "pos_key_layer": d["pk"] if "pk" in terms else None, "pos_query_layer": d["pq"] if "pq" in terms else None}))
    assert (got - ref).abs().max() < BOUND
    assert all(not got[b, :, n:].any() for b, n in enumerate(lens.tolist()))


@pytest.mark.parametrize("flag", [DIRECT, ONE_SET, TWO_SETS])
@pytest.mark.parametrize("B", [7, 70])                                               # sorted by length up to 64 sequences
def test_packed_with_gaps(flag, B):
    lens = torch.randint(0, 150, (B,), generator=torch.Generator().manual_seed(B))
    cu = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)]).int()
    T = int(cu[-1]) + 40
    d = {n: t.cuda() for n, t in make_inputs(6, 1, 4, T, 64, 256, 512).items()}
    q, k, v = (d[n][0].transpose(0, 1).contiguous() for n in "qkv")
    cu = (cu + 20).cuda()                                                            # 20 rows before the first and behind the last
    got, ref = _in_and_generic(flag, lambda g: flash_attention_with_disentangled_varlen(
        q, k, v, None, None, cu, cu, 150, 150, False, f32.SCALE, 256, 512, pos_key_layer=d["pk"], pos_query_layer=d["pq"], force_generic=g))
    assert (got - ref).abs().max() < BOUND and not got[:20].any() and not got[T - 20:].any()


@pytest.mark.parametrize("L", [15, 17, 33, 64, 129, 161])
def test_direct_tile_edges(L):
    """32 query rows a workgroup."""
    with in_kernel(DIRECT):
        f32.test_tile_edges(40, 16, L)


@pytest.mark.parametrize("terms", [("c2p",), ("p2c",), ()])
def test_direct_term_subsets(terms):
    with in_kernel(DIRECT):
        f32.test_term_subsets(terms, 40, 16)


@pytest.mark.parametrize("where", ["query", "key", "value", "last_value", "c2p_row", "p2c_row", "score", "low_scores", "padding"])
def test_direct_nan_and_infinity(where):
    with in_kernel(DIRECT):
        f32.test_nan_and_infinity_reach_what_they_belong_to(where, 33, 16, 77)


@pytest.mark.parametrize("flag", [DIRECT, ONE_SET, TWO_SETS])
@pytest.mark.parametrize("where", ["query", "key", "value", "last_value", "c2p_row", "p2c_row", "score", "low_scores", "padding"])
def test_nan_and_infinity(flag, where):
    with in_kernel(flag):
        f32.test_nan_and_infinity_reach_what_they_belong_to(where, 2, 2, 130)


@pytest.mark.parametrize("flag", [ONE_SET, TWO_SETS])
@pytest.mark.parametrize("L", [65, 273])                                             # a wave without queries, and the second set's keys
@pytest.mark.parametrize("where", ["value", "last_value", "c2p_row", "p2c_row", "score"])
def test_rows_computed_again(flag, where, L):
    with in_kernel(flag):
        f32.test_nan_and_infinity_reach_what_they_belong_to(where, 2, 2, L)


@pytest.mark.parametrize("flag", [ONE_SET, TWO_SETS])
def test_results_beside_an_infinity_keep_their_bits(flag):
    """A query that is NaN and values that are infinite change their own row and column, also in the tile that is computed again."""
    d = {n: t.cuda() for n, t in make_inputs(7, 1, 2, 150, 64, 256, 512).items()}
    run = lambda: flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, f32.SCALE, 256, 512, pos_key_layer=d["pk"], pos_query_layer=d["pq"])
    with in_kernel(flag):
        clean = run()
        d["q"][0, 0, 37, 5], d["v"][0, 1, 20, 9] = math.nan, math.inf
        got = run()
    own = torch.zeros_like(clean, dtype=torch.bool)
    own[0, 0, 37], own[0, 1, :, 9] = True, True
    assert got[0, 0, 37].isnan().all() and (got[0, 1, :, 9] == math.inf).all()
    assert torch.equal(got[~own], clean[~own])


@pytest.mark.parametrize("flag", [ONE_SET, TWO_SETS])
@pytest.mark.parametrize("scale", [0.0, -0.3, 40.0])
def test_any_scale(flag, scale):
    """A score is scaled before its maximum is taken, and rounded as the maximum is: no scale makes a probability larger than 1."""
    d = {n: t.cuda() for n, t in make_inputs(1, 2, 2, 100, 64, 256, 512).items()}
    got, ref = _in_and_generic(flag, lambda g: flash_attention_with_disentangled(
        d["q"], d["k"], d["v"], None, None, False, scale, 256, 512, pos_key_layer=d["pk"], pos_query_layer=d["pq"], force_generic=g))
    # scores of some 25 |scale|, each off by a few units of 2^-24 of itself in either kernel
    assert (got - ref).abs().max() < BOUND * (1 + 25 * abs(scale))


@pytest.mark.parametrize("flag", [ONE_SET, TWO_SETS])
@pytest.mark.parametrize("size", [1e-25, 1e30])
def test_size_of_values(flag, size):
    """Parts keep the exponent: small and large values are as exact as others."""
    d = {n: t.cuda() for n, t in make_inputs(2, 1, 2, 90, 64, 256, 512).items()}
    d["v"] *= size
    got, ref = _in_and_generic(flag, lambda g: flash_attention_with_disentangled(
        d["q"], d["k"], d["v"], None, None, False, f32.SCALE, 256, 512, pos_key_layer=d["pk"], pos_query_layer=d["pq"], force_generic=g))
    assert (got - ref).abs().max() < BOUND * size


def _exact(d, L, scale):
    """The definition in 64 bits."""
    x = {n: t.double() for n, t in d.items()}
    delta = torch.from_numpy(_lib.delta_table(L, 256, 512).astype("int64")).cuda()
    at = delta[(torch.arange(L)[:, None] - torch.arange(L)[None] + L - 1).cuda()].expand(*x["q"].shape[:2], L, L)
    s = x["q"] @ x["k"].transpose(-1, -2).contiguous() + (x["q"] @ x["pk"].transpose(-1, -2).contiguous()[None]).gather(3, at)
    s = s + (x["k"] @ x["pq"].transpose(-1, -2).contiguous()[None]).gather(3, at.transpose(-1, -2)).transpose(-1, -2)
    return torch.softmax(s * scale, -1) @ x["v"]


@pytest.mark.parametrize("flag", [DIRECT, ONE_SET, TWO_SETS])
@pytest.mark.parametrize("sizes", [dict(v=1e-33), dict(v=1e-36), dict(v=2e-38), dict(v=1e36), dict(q=1e-36, k=1e36, pk=1e36, pq=1e-36), dict(q=1e36, k=1e-36, pk=1e-36, pq=1e36),
                                   dict(k=1e-36, pq=1e36, pk=0), dict(q=1e-36, pk=1e36, k=1), dict(q=1e-18, k=1e-18, pk=1e-18, pq=1e-18, scale=1e36)],
                         ids=lambda s: "-".join(f"{n}={x:g}" for n, x in s.items()))
def test_error_at_any_size(flag, sizes):
    """Where the last part of an operand is too small for its type, the result is as exact as elsewhere: sums of 64 products and 150 weighted
    values in 32 bits, 1.2e-7 to 2.4e-7 of their size for values of order 1."""
    d = {n: t.cuda() for n, t in make_inputs(8, 1, 2, 150, 64, 256, 512).items()}
    for n in d:
        d[n] *= sizes.get(n, 1)
    d["v"][..., 60:] = 0
    scale = f32.SCALE * sizes.get("scale", 1)
    exact = _exact(d, 150, scale)
    with in_kernel(flag):
        out = flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, scale, 256, 512, pos_key_layer=d["pk"], pos_query_layer=d["pq"])
    err = float((out.double() - exact).norm() / exact.norm())
    print(f"{sizes}: {err:.2e}")
    assert err < 1e-6 and not out[..., 60:].any()


@pytest.mark.parametrize("flag", [ONE_SET, TWO_SETS])
def test_strided_rows_and_shared_tables(flag):
    """Rows of a wider array, and a table of equal rows (stride 0) as an expanded tensor has it."""
    d = {n: t.cuda() for n, t in make_inputs(3, 2, 3, 80, 64, 256, 512).items()}
    wide = torch.zeros(2, 80, 3, 5, 64, device="cuda")
    for i, n in enumerate("qkv"):
        wide[:, :, :, i] = d[n].permute(0, 2, 1, 3)
    q, k, v = (wide[:, :, :, i].permute(0, 2, 1, 3) for i in range(3))
    pk = d["pk"][:, :1].expand(-1, 512, -1)
    got, ref = _in_and_generic(flag, lambda g: flash_attention_with_disentangled(
        q, k, v, None, None, False, f32.SCALE, 256, 512, pos_key_layer=pk, pos_query_layer=d["pq"], force_generic=g))
    assert (got - ref).abs().max() < BOUND


def test_error_against_64_bits_is_no_larger():
    """Small products first: sums of parts are more exact than float32 products one after another."""
    d = {n: t.cuda() for n, t in make_inputs(4, 2, 4, 300, 64, 256, 512).items()}
    exact = _exact(d, 300, f32.SCALE)
    err = {}
    for flag in (DIRECT, ONE_SET, TWO_SETS):
        with in_kernel(flag):
            out = flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, f32.SCALE, 256, 512, pos_key_layer=d["pk"], pos_query_layer=d["pq"])
        err[flag] = float((out.double() - exact).norm() / exact.norm())
    assert err[ONE_SET] <= err[DIRECT] and err[TWO_SETS] <= err[DIRECT] and err[DIRECT] < 1e-6, err
    assert math.isfinite(err[ONE_SET])
