"""The 16-bit kernel for short sequences (up to 128 tokens, 160 in large launches) at the edges of its units (32 query rows a wave, 64 keys a
step), against the vector-ALU kernel and bit for bit against the kernels for texts of any length."""
import math

import pytest
import torch

from helpers import assert_close_bf16, in_kernel, make_inputs, oracle_fixed
from turbodeberta_amd import _lib
from turbodeberta_amd.ops.flash_attention import flash_attention_with_disentangled
from turbodeberta_amd.ops.flash_attention_varlen import flash_attention_with_disentangled_varlen

pytestmark = pytest.mark.gpu
SCALE = 1.0 / math.sqrt(192)


def _packed(lens, dtype, terms=("c2p", "p2c"), H=3, seed=0):
    cu = torch.cat([torch.zeros(1, dtype=torch.long), torch.tensor(lens).cumsum(0)]).int().cuda()
    d = {n: t.cuda() for n, t in make_inputs(seed, 1, H, max(1, sum(lens)), 64, 256, 512, dtype).items()}
    q, k, v = (d[n][0].transpose(0, 1).contiguous() for n in "qkv")

    def run(longest, **kw):
        return flash_attention_with_disentangled_varlen(q, k, v, None, None, cu, cu, longest, longest, False, SCALE, 256, 512,
                                                        pos_key_layer=d["pk"] if "c2p" in terms else None,
                                                        pos_query_layer=d["pq"] if "p2c" in terms else None, **kw)
    return run


def _same_in_the_others(got, run, *args):
    for flag in (_lib.TDB_FLAG_PERSISTENT, _lib.TDB_FLAG_RESIDENT):
        with in_kernel(flag):
            assert torch.equal(got, run(*args)), flag


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L", [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128])
def test_fixed_edges(L, dtype):
    d = {n: t.cuda() for n, t in make_inputs(L, 2, 3, L, 64, 256, 512, dtype).items()}
    got, ref = (flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, SCALE, 256, 512, pos_key_layer=d["pk"],
                                                  pos_query_layer=d["pq"], force_generic=f) for f in (False, True))
    assert_close_bf16(got, ref, f"L={L}")


@pytest.mark.parametrize("terms", [("c2p", "p2c"), ("c2p",), ("p2c",), ()])
@pytest.mark.parametrize("lens", [[1], [30, 2, 33, 64], [16, 40] * 32, [5, 0, 96, 31, 70] * 20, [128, 1, 65, 100] * 25, [3, 9, 17] * 60],
                         ids=["one", "four", "64_with_single_tiles", "100", "100_to_128", "180_tiny"])
def test_packed_same_bits_as_the_other_kernels(lens, terms):
    run = _packed(lens, torch.bfloat16, terms)
    got = run(max(lens))
    _same_in_the_others(got, run, 161)      # (a maximum that the short kernel does not take)
    assert_close_bf16(got, run(max(lens), force_generic=True), str(terms))


@pytest.mark.parametrize("B,L", [(3, 50), (64, 64), (90, 128), (1, 128)])
def test_lengths_and_padding(B, L):
    d = {n: t.cuda() for n, t in make_inputs(B, B, 4, L, 64, 256, 512, torch.bfloat16).items()}
    lens = torch.randint(0, L + 1, (B,), generator=torch.Generator().manual_seed(B)).int()
    lens[0] = 0 if B > 1 else 40
    got, ref = (flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, SCALE, 256, 512, pos_key_layer=d["pk"],
                                                  pos_query_layer=d["pq"], seqlens_k=lens.cuda(), force_generic=f) for f in (False, True))
    assert_close_bf16(got, ref, f"{B} x {L}")
    assert all(not got[b, :, n:].any() for b, n in enumerate(lens.tolist()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("where", ["query", "key", "value", "last_value", "c2p_row", "p2c_row", "padding", "strip"])
@pytest.mark.parametrize("L", [29, 50, 128])
def test_nan_and_infinity_reach_what_they_belong_to(where, L, dtype):
    """As in the definition: a key that is NaN leaves no query of its sequence a number, a position row that is NaN none that
    meets it, a value its own columns; padding is not read."""
    nan, inf = float("nan"), float("inf")
    d, lens, tables, strips = make_inputs(5, 2, 2, L, 64, 256, 512, dtype), None, ("pk", "pq"), [None, None]
    if where == "query":
        d["q"][1, 0, 3, 7] = nan
    elif where == "key":
        d["k"][1, 1, L - 1, 0] = nan
    elif where == "value":
        d["v"][0, 1, 5, 9] = nan
    elif where == "last_value":
        d["v"][0, 0, L - 1, 2], d["v"][1, 1, L - 1, 63] = inf, -inf
    elif where == "c2p_row":
        d["pk"][1, 256 + 20, 4] = nan
    elif where == "p2c_row":
        d["pq"][0, 256 - 20, 60] = nan
    elif where == "padding":
        lens = d["lengths"] = torch.full((2,), L - 20, dtype=torch.int32)
    ref = oracle_fixed(d, 256, 512)
    if where == "padding":
        for n in "qkv":
            d[n][:, :, L - 20:] = nan
    elif where == "strip":
        tables, strips = (), [(x.float() @ t.float().transpose(-1, -2)[None]).to(dtype) for x, t in ((d["q"], d["pk"]), (d["k"], d["pq"]))]
        strips[0][0, 0, 3, 256 + 2] = nan           # query 3 meets it at key 1
        strips[1][1, 1, 4, 256 - 3] = nan           # key 4 at query 1
        ref[0, 0, 3] = ref[1, 1, 1] = nan
    g = lambda t: None if t is None else t.cuda()
    got = flash_attention_with_disentangled(g(d["q"]), g(d["k"]), g(d["v"]), *map(g, strips), False, SCALE, 256, 512, seqlens_k=g(lens),
                                            pos_key_layer=g(d["pk"]) if tables else None, pos_query_layer=g(d["pq"]) if tables else None).float().cpu()
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    assert ref.isnan().any() == (where not in ("last_value", "padding"))
    number = ref.isfinite()
    assert_close_bf16(got[number], ref[number], where)


def test_rows_follow_their_own_maximum():
    # scores that grow along the keys raise the running maximum of some rows only: same bits in all kernels
    d = {n: t.cuda() for n, t in make_inputs(1, 2, 3, 128, 64, 256, 512, torch.bfloat16).items()}
    d["k"] *= torch.linspace(0.1, 12, 128, device="cuda")[None, None, :, None]
    d["q"] *= torch.linspace(0.1, 3, 128, device="cuda")[None, None, :, None]
    pos = dict(pos_key_layer=d["pk"], pos_query_layer=d["pq"])
    got = flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, SCALE, 256, 512, **pos)
    wide = [torch.cat([d[n], d[n][:, :, :1]], 2) for n in "qkv"]                   # one row more, masked by its length
    lens = torch.tensor([128, 128], dtype=torch.int32, device="cuda")
    _same_in_the_others(got, lambda: flash_attention_with_disentangled(*wide, None, None, False, SCALE, 256, 512, seqlens_k=lens, **pos)[:, :, :128])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cu,longest", [([0, 20, 50], 30), ([3, 20, 50], 30), ([0, 20, 50], 12), ([0, 200, 230], 200), ([0, 200, 205], 150),
                                        ([5] + list(range(5, 230, 3)), 3), ([0], 4)])
def test_rows_outside_every_sequence_are_zeros(cu, longest, dtype):
    T = 260
    d = {n: t.cuda() for n, t in make_inputs(9, 1, 3, T, 64, 256, 512, dtype).items()}
    q, k, v = (d[n][0].transpose(0, 1).contiguous() for n in "qkv")
    c = torch.tensor(cu, dtype=torch.int32, device="cuda")
    junk = torch.full((64 << 20,), float("nan"), device="cuda")           # what a fresh allocation finds
    del junk
    run = lambda **kw: flash_attention_with_disentangled_varlen(q, k, v, None, None, c, c, longest, longest, False, SCALE, 256, 512,
                                                                pos_key_layer=d["pk"], pos_query_layer=d["pq"], **kw)
    out, ref = run(), run(force_generic=True)
    inside = torch.zeros(T, dtype=torch.bool)
    for a, b in zip(cu, cu[1:]):
        inside[a:min(b, a + longest)] = True
    assert not out[~inside.cuda()].any() and not ref[~inside.cuda()].any()
    assert_close_bf16(out, ref)


@pytest.mark.parametrize("terms", [("c2p", "p2c"), ("c2p",), ("p2c",)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,L,buckets", [(2, 1, 256), (3, 32, 256), (2, 33, 16), (70, 65, 256), (2, 96, 16), (40, 128, 256)])
def test_strips(B, L, buckets, dtype, terms):
    """Strips of random values, packed, full and padded: against the vector-ALU kernel, and packed bit for bit against the
    persistent kernel."""
    d = {n: t.cuda() for n, t in make_inputs(L, B, 3, L, 64, 256, 512, dtype).items()}
    g = torch.Generator(device="cuda").manual_seed(L)
    strip = [torch.randn(B, 3, L, 2 * buckets, device="cuda", generator=g).to(dtype) if t in terms else None for t in ("c2p", "p2c")]
    lens = torch.randint(0, L + 1, (B,), generator=torch.Generator().manual_seed(B)).int()
    lens[0] = L
    for kw in ({}, {"seqlens_k": lens.cuda()}):
        got, ref = (flash_attention_with_disentangled(d["q"], d["k"], d["v"], *strip, False, SCALE, buckets, 512, force_generic=f, **kw) for f in (False, True))
        assert_close_bf16(got, ref, f"{B} x {L}")
    rows = lambda t: torch.cat([t[b, :, :n].transpose(0, 1) for b, n in enumerate(lens.tolist())]).contiguous() if t is not None else None
    cu = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)]).int().cuda()
    a, b = (flash_attention_with_disentangled_varlen(*(rows(d[n]) for n in "qkv"), *(rows(s) for s in strip), cu, cu, n, n, False, SCALE, buckets, 512)
            for n in (L, 161))
    assert torch.equal(a, b)
    assert all(torch.equal(a[cu[i]:cu[i + 1]].transpose(0, 1), got_b) for i, got_b in
               ((i, flash_attention_with_disentangled(d["q"], d["k"], d["v"], *strip, False, SCALE, buckets, 512, seqlens_k=lens.cuda())[i, :, :lens[i]]) for i in (0, B - 1)))


@pytest.mark.parametrize("terms", [("c2p", "p2c"), ("c2p",), ("p2c",)])
@pytest.mark.parametrize("lens", [[129] * 70, [160] * 64, [160, 5, 129, 96, 0, 33] * 50], ids=["129", "160", "mixed"])
def test_five_query_tiles(lens, terms):
    run = _packed(lens, torch.bfloat16, terms)
    got = run(max(lens))
    _same_in_the_others(got, run, 161)      # (a maximum that the short kernel does not take)
    assert_close_bf16(got, run(max(lens), force_generic=True), str(terms))


@pytest.mark.parametrize("B,L,ragged", [(50, 129, False), (50, 160, False), (110, 160, True)])
def test_five_query_tiles_fixed(B, L, ragged):
    d = {n: t.cuda() for n, t in make_inputs(B, B, 3, L, 64, 256, 512, torch.float16).items()}
    lens = torch.randint(0, L + 1, (B,), generator=torch.Generator().manual_seed(B)).int().cuda() if ragged else None
    got, ref = (flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, SCALE, 256, 512, pos_key_layer=d["pk"],
                                                  pos_query_layer=d["pq"], seqlens_k=lens, force_generic=f) for f in (False, True))
    assert_close_bf16(got, ref, f"{B} x {L}")
