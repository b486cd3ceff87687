"""float32 calls at the edges of the matrix-core kernels' tiles, against the vector-ALU kernel, in whichever kernel the library chooses: small
ones in the one that has 16 queries or 32 per workgroup and deals keys to four waves in blocks of two 16-key tiles, larger ones mostly in the one whose
products are of bf16 parts (tests/test_f32_split_gpu.py runs both by name)."""
import math

import pytest
import torch

from helpers import assert_close_fp32, make_inputs, oracle_fixed
from turbodeberta_amd.ops.flash_attention import flash_attention_with_disentangled
from turbodeberta_amd.ops.flash_attention_varlen import flash_attention_with_disentangled_varlen

pytestmark = pytest.mark.gpu
SCALE = 1.0 / math.sqrt(192)


def _both(d, terms=("c2p", "p2c"), lens=None):
    kw = dict(pos_key_layer=d["pk"] if "c2p" in terms else None, pos_query_layer=d["pq"] if "p2c" in terms else None, seqlens_k=lens)
    return [flash_attention_with_disentangled(d["q"], d["k"], d["v"], None, None, False, SCALE, 256, 512, force_generic=f, **kw)
            for f in (False, True)]


@pytest.mark.parametrize("B,H", [(1, 2), (40, 16)])          # 16 query rows per workgroup, and 32 or bf16 parts
@pytest.mark.parametrize("L", [1, 15, 16, 17, 33, 64, 127, 129, 161])
def test_tile_edges(B, H, L):
    d = {n: t.cuda() for n, t in make_inputs(L, B, H, L, 64, 256, 512).items()}
    got, ref = _both(d)
    assert_close_fp32(got, ref, f"L={L}")
    if B == 1:
        cpu = {n: t.cpu() for n, t in d.items()}
        assert_close_fp32(got, oracle_fixed(cpu, 256, 512), f"L={L} oracle")


NAN, INF = float("nan"), float("inf")


@pytest.mark.parametrize("where", ["query", "key", "value", "last_value", "c2p_row", "p2c_row", "score", "low_scores", "padding"])
@pytest.mark.parametrize("B,H,L", [(2, 2, 50), (2, 2, 130), (33, 16, 77)])
def test_nan_and_infinity_reach_what_they_belong_to(where, B, H, L):
    """As in the definition: a key that is NaN leaves no query of its sequence a number, a position row that is NaN none that
    meets it, a value its own columns; scores of -infinity (a whole block of them too) weigh nothing; padding is not read."""
    d = make_inputs(5, B, H, L, 64, 256, 512)
    lens = None
    if where == "query":
        d["q"][1, 0, 3, 7] = NAN
    elif where == "key":
        d["k"][1, 1, L - 1, 0] = NAN
    elif where == "value":
        d["v"][0, 1, 5, 9] = NAN
    elif where == "last_value":
        d["v"][0, 0, L - 1, 2], d["v"][1, 1, L - 1, 63] = INF, -INF
    elif where == "c2p_row":
        d["pk"][1, 256 + 20, 4] = NAN
    elif where == "p2c_row":
        d["pq"][0, 256 - 30, 60] = NAN
    elif where == "score":
        d["q"][0, 0, 2] = d["k"][0, 0, 4] = 3e19
    elif where == "low_scores":
        d["q"], d["pk"], d["pq"] = d["q"].abs(), d["pk"] * 0, d["pq"] * 0
        d["k"][:, :, :L - 9] = d["k"][0, 1] = -3e38             # (0, 1): no key left, NaN
    elif where == "padding":
        lens = torch.full((B,), L - 20, dtype=torch.int32)
        d["lengths"] = lens
    ref = oracle_fixed(d, 256, 512)
    if where == "padding":
        for n in "qkv":
            d[n][:, :, L - 20:] = NAN
    got = _both({n: t.cuda() for n, t in d.items()}, lens=None if lens is None else lens.cuda())[0].cpu()
    assert torch.equal(got.isnan(), ref.isnan()) and ref.isnan().any() == (where not in ("last_value", "padding"))
    torch.testing.assert_close(got, ref, rtol=1e-4, atol=1e-4, equal_nan=True)


@pytest.mark.parametrize("terms", [("c2p",), ("p2c",), ()])
@pytest.mark.parametrize("B,H", [(1, 2), (40, 16)])
def test_term_subsets(terms, B, H):
    d = {n: t.cuda() for n, t in make_inputs(3, B, H, 77, 64, 256, 512).items()}
    assert_close_fp32(*_both(d, terms), what=str(terms))


@pytest.mark.parametrize("terms", [("c2p", "p2c"), ("c2p",), ("p2c",)])
@pytest.mark.parametrize("B,H", [(2, 2), (33, 16)])
def test_strips(terms, B, H):
    d = {n: t.cuda() for n, t in make_inputs(4, B, H, 45, 64, 256, 512).items()}
    g = torch.Generator(device="cuda").manual_seed(1)
    strip = [torch.randn(B, H, 45, 512, device="cuda", generator=g) if t in terms else None for t in ("c2p", "p2c")]
    lens = torch.randint(1, 46, (B,), device="cuda", generator=g).int()
    got, ref = (flash_attention_with_disentangled(d["q"], d["k"], d["v"], *strip, False, SCALE, 256, 512, seqlens_k=lens, force_generic=f)
                for f in (False, True))
    assert_close_fp32(got, ref, str(terms))


@pytest.mark.parametrize("B", [5, 64, 65])                   # sorted by length up to 64 sequences
def test_lengths_and_padding(B):
    L = 100
    d = {n: t.cuda() for n, t in make_inputs(5, B, 3, L, 64, 256, 512).items()}
    lens = torch.randint(0, L + 1, (B,), generator=torch.Generator().manual_seed(2)).int()
    lens[0], lens[1], lens[2] = 0, L, 1
    got, ref = _both(d, lens=lens.cuda())
    assert_close_fp32(got, ref, f"B={B}")
    assert all(not got[b, :, n:].any() for b, n in enumerate(lens.tolist()))


@pytest.mark.parametrize("B", [7, 64, 70])
def test_packed(B):
    lens = torch.randint(0, 90, (B,), generator=torch.Generator().manual_seed(3))
    cu = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)]).int().cuda()
    d = {n: t.cuda() for n, t in make_inputs(6, 1, 4, int(lens.sum()), 64, 256, 512).items()}
    q, k, v = (d[n][0].transpose(0, 1).contiguous() for n in "qkv")
    got, ref = (flash_attention_with_disentangled_varlen(q, k, v, None, None, cu, cu, 90, 90, False, SCALE, 256, 512,
                                                         pos_key_layer=d["pk"], pos_query_layer=d["pq"], force_generic=f)
                for f in (False, True))
    assert_close_fp32(got, ref, f"B={B}")


@pytest.mark.parametrize("terms", [("c2p", "p2c"), ("c2p",), ("p2c",), ()])
@pytest.mark.parametrize("B,L", [(2, 1), (2, 16), (2, 33), (2, 64), (90, 17), (90, 64)])
def test_single_key_tiles(B, L, terms):
    """Up to 64 tokens a wave has one key tile; both query tile heights."""
    d = {n: t.cuda() for n, t in make_inputs(L, B, 6, L, 64, 256, 512).items()}
    assert_close_fp32(*_both(d, terms), what=f"{B} x {L} {terms}")
