"""The float32 matrix-core kernel where the key tiles of a sequence do not fill the last round of its waves (blocks of two tiles, then
single ones), for 16 and 32 query rows a workgroup, against the vector-ALU kernel."""
import math

import pytest
import torch

from helpers import make_inputs
from turbodeberta_amd.ops.flash_attention import flash_attention_with_disentangled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("terms", [("pk", "pq"), ("pk",), ("pq",), ()])
@pytest.mark.parametrize("B", [1, 16])
def test_every_number_of_key_tiles(B, terms):
    L = 273                                         # up to 18 tiles: no round, one and two of eight, and each rest
    d = {n: t.cuda() for n, t in make_inputs(B, B, 4, L, 64, 32, 512, torch.float32).items()}
    for first in range(16, 272, 16 * B):
        lens = torch.tensor([min(first + 16 * b + (b % 3), L) for b in range(B)], dtype=torch.int32, device="cuda")
        for upto in ([int(lens[0])] if B == 1 else [L, 80]):
            q, k, v = (d[n][:, :, :upto] for n in "qkv")
            got, ref = (flash_attention_with_disentangled(q, k, v, None, None, False, 1.0 / math.sqrt(192), 32, 512, seqlens_k=lens.clamp(max=upto), force_generic=f,
                                                          pos_key_layer=d["pk"] if "pk" in terms else None, pos_query_layer=d["pq"] if "pq" in terms else None)
                        for f in (False, True))
            # both round each product once; sums of 64 to 273 of them in another order: a few units of 2^-24 of values of order 1
            assert (got - ref).abs().max() < 2e-5, (first, upto)
