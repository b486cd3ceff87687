"""The 16-bit kernel with resident position tables at the edges of its tiles (16 or 32 query rows a wave, four or eight waves, 64 keys a
step) and of its deals: made to take every launch here, against the vector-ALU kernel and bit for bit against the persistent kernel, made
to take the same launch, whichever the library chooses, and the sequences alone."""
import math

import pytest
import torch

from helpers import assert_close_bf16, in_kernel, make_inputs
from turbodeberta_amd import _lib
from turbodeberta_amd.ops.flash_attention import flash_attention_with_disentangled
from turbodeberta_amd.ops.flash_attention_varlen import flash_attention_with_disentangled_varlen

pytestmark = pytest.mark.gpu
SCALE = 1.0 / math.sqrt(192)
BOTH = ("pk", "pq")


def _fixed(d, terms=BOTH, rows=slice(None), upto=None, buckets=256, **kw):
    q, k, v = (d[n][rows, :, :upto] for n in "qkv")
    return flash_attention_with_disentangled(q, k, v, None, None, False, SCALE, buckets, 512, pos_key_layer=d["pk"] if "pk" in terms else None,
                                             pos_query_layer=d["pq"] if "pq" in terms else None, **kw)


def _inputs(B, H, L, dtype, buckets=256):
    return {n: t.cuda() for n, t in make_inputs(L, B, H, L, 64, buckets, 512, dtype).items()}


def _same_in_each(run, name):
    """The result in the resident kernel, after a look at the other routes."""
    with in_kernel(_lib.TDB_FLAG_RESIDENT):
        got = run()
    with in_kernel(_lib.TDB_FLAG_PERSISTENT):
        assert torch.equal(got, run()), f"{name}: persistent kernel"
    assert torch.equal(got, run()), f"{name}: the library's choice"
    return got


@pytest.mark.parametrize("terms", [BOTH, ("pk",), ("pq",), ()])
@pytest.mark.parametrize("B,H,L,dtype,buckets", [
    (1, 3, 161, torch.bfloat16, 256), (2, 12, 193, torch.float16, 16), (1, 12, 512, torch.bfloat16, 256),       # half tiles of 16-row units
    (8, 12, 513, torch.float16, 256),                                                                           # a tile a workgroup
    (16, 12, 257, torch.bfloat16, 256), (33, 12, 289, torch.bfloat16, 32), (70, 3, 500, torch.float16, 256),    # runs of half tiles
    (9, 16, 320, torch.bfloat16, 256), (1, 1, 700, torch.float16, 256), (2, 64, 385, torch.bfloat16, 16),       # a head a group: of 16, 256, 4
    (3, 12, 1537, torch.bfloat16, 256), (2, 16, 1601, torch.float16, 256),                                      # far steps in 32 bits
])
def test_equal_lengths(B, H, L, dtype, buckets, terms):
    d = _inputs(B, H, L, dtype, buckets)
    print(f"[case] {B} x {H} x {L}", flush=True)
    got = _same_in_each(lambda: _fixed(d, terms, buckets=buckets), "equal")
    assert_close_bf16(got, _fixed(d, terms, buckets=buckets, force_generic=True), f"{B} x {L}")
    with in_kernel(_lib.TDB_FLAG_RESIDENT):
        assert torch.equal(got[B - 1:], _fixed(d, terms, rows=slice(B - 1, B), buckets=buckets))
        for limit in (8, 40):
            try:
                _lib.set_workgroup_limit(limit)
                assert torch.equal(got, _fixed(d, terms, buckets=buckets)), limit
            finally:
                _lib.set_workgroup_limit(0)


@pytest.mark.parametrize("terms", [BOTH, ("pk",), ("pq",)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,L,buckets,max_rel", [
    (1, 2, 1536, 8, 4096), (8, 12, 1537, 16, 4096), (2, 12, 2500, 8, 2048),        # wide buckets: far steps of one table row after another
    (1, 3, 1700, 16, 64), (9, 12, 1536, 4, 16),                                     # one run of near steps, also within a single step
])
def test_far_and_near_steps_in_turn(B, H, L, buckets, max_rel, dtype, terms):
    d = {n: t.cuda() for n, t in make_inputs(L + buckets, B, H, L, 64, buckets, max_rel, dtype).items()}
    kw = {"pos_key_layer": d["pk"] if "pk" in terms else None, "pos_query_layer": d["pq"] if "pq" in terms else None}
    print(f"[case] {B} x {H} x {L}, {buckets} buckets to {max_rel}", flush=True)
    run = lambda **more: flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, SCALE, buckets, max_rel, **kw, **more)
    assert_close_bf16(_same_in_each(run, "far and near"), run(force_generic=True), f"{L}, {buckets} buckets")


LENS = {
    "few": [256, 1, 0, 130], "rounds_of_halves": [511, 64, 300] * 3, "64": list(range(4, 516, 8)), "65_in_two": [500] * 60 + [1, 33, 0, 129, 256],
    "last_round_split": [512] * 43 + [129] * 3, "ends": [289] * 50, "long": [1600, 900, 64, 1537, 1, 1300, 2000, 1100],
    "wholes_by_halves": [1100] * 7, "longest_by_halves": [2000, 1732, 1464, 1196, 928, 660], "less_than_a_round": [800, 532, 264],
    "rounds_far_apart": list(range(640, 210, -11)),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name,H", [(n, 12) for n in LENS] + [(n, h) for n in ("few", "64", "wholes_by_halves", "longest_by_halves") for h in (1, 16)])
def test_different_lengths(name, H, dtype):
    lens = LENS[name]
    L = max(lens)
    d = _inputs(len(lens), H, L, dtype)
    n = torch.tensor(lens, dtype=torch.int32, device="cuda")
    print(f"[case] {name}, {H} heads", flush=True)
    padded = _same_in_each(lambda: _fixed(d, seqlens_k=n), "padded")
    assert_close_bf16(padded, _fixed(d, seqlens_k=n, force_generic=True), name)
    # packed, as views of one projection, and with rows behind the last sequence: zeros there
    cu = torch.cat([torch.zeros(1, dtype=torch.int32, device="cuda"), n.cumsum(0).int()])
    rows = torch.cat([torch.stack([d[x][b, :, :m].transpose(0, 1) for x in "qkv"], 1) for b, m in enumerate(lens)] + [torch.full((9, 3, H, 64), float("nan"), device="cuda").to(dtype)])
    packed = _same_in_each(lambda: flash_attention_with_disentangled_varlen(*rows.unbind(1), None, None, cu, cu, L, L, False, SCALE, 256, 512,
                                                                            pos_key_layer=d["pk"], pos_query_layer=d["pq"]), "packed")
    assert not packed[sum(lens):].any()
    for b, m in enumerate(lens):
        assert torch.equal(packed[cu[b]:cu[b + 1]].transpose(0, 1), padded[b, :, :m]) and not padded[b, :, m:].any(), b
    if L < 1536:                    # (above, the longest decides how far steps are computed)
        for b in {0, len(lens) // 2, len(lens) - 1}:
            if lens[b]:
                assert torch.equal(_fixed(d, rows=slice(b, b + 1), upto=lens[b])[0], padded[b, :, :lens[b]]), b


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,L,buckets", [(1, 200, 256), (16, 300, 16), (2, 1600, 256)])
@pytest.mark.parametrize("where", ["q", "k", "v", "pk", "pq"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_values_that_are_not_finite(B, L, buckets, where, value, dtype):
    d = _inputs(B, 12, L, dtype, buckets)
    d[where][(B - 1, 1, L - 3, 5) if where in "qkv" else (1, buckets + 3, 5)] = value
    with in_kernel(_lib.TDB_FLAG_RESIDENT):
        got = _fixed(d, buckets=buckets)
    ref = _fixed(d, buckets=buckets, force_generic=True)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    number = ref.isfinite()
    assert_close_bf16(got[number], ref[number], where)
