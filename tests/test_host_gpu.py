"""The operators' native front: it takes every well-formed call and gives what the Python path gives, and leaves the
rest to that path."""
import math

import pytest
import torch

from helpers import make_inputs
from turbodeberta_amd import _lib
from turbodeberta_amd.ops import flash_attention as fa
from turbodeberta_amd.ops import flash_attention_varlen as fv

pytestmark = pytest.mark.gpu
SCALE = 1.0 / math.sqrt(192)


def _call(seed=0, B=2, H=3, L=70, dtype=torch.bfloat16):
    d = {n: t.cuda() for n, t in make_inputs(seed, B, H, L, 64, 256, 512, dtype).items()}
    fixed = [d["q"], d["k"], d["v"], None, None, False, SCALE, 256, 512, d["pk"], d["pq"], None, False]
    return d, fixed


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["tables", "tables4d", "lengths", "strips", "views", "default_scale", "no_position"])
def test_fixed_front_equals_python_path(form, dtype):
    d, a = _call(dtype=dtype)
    if form == "tables4d":
        a[9], a[10] = d["pk"][None], d["pq"][None]
    elif form == "lengths":
        a[11] = torch.tensor([70, 13], dtype=torch.int32, device="cuda")
    elif form == "strips":
        a[3], a[4] = (torch.matmul(x, t.transpose(-1, -2).contiguous()) for x, t in ((d["q"], d["pk"]), (d["k"], d["pq"])))
        a[9] = a[10] = None
    elif form == "views":
        qkv = torch.stack([t.transpose(1, 2) for t in a[:3]], 2).contiguous()
        a[:3] = qkv.permute(2, 0, 3, 1, 4).unbind(0)
    elif form == "default_scale":
        a[6] = None
    elif form == "no_position":
        a[9] = a[10] = None
    ref = fa.prepare(*a[:9], pos_key_layer=a[9], pos_query_layer=a[10], seqlens_k=a[11]).launch()
    out = _lib.host().fixed(*a)
    assert out is not None and out.stride() == ref.stride() and torch.equal(out, ref)


def test_varlen_front_equals_python_path():
    d, _ = _call(B=1, L=140)
    q, k, v = (d[n][0].transpose(0, 1).contiguous() for n in "qkv")
    cu = torch.tensor([0, 40, 40, 131], dtype=torch.int32, device="cuda")      # 9 rows belong to nobody: zeros
    a = [q, k, v, None, None, cu, cu, 91, 91, False, SCALE, 256, 512, d["pk"], d["pq"], False, True]
    ref = fv.prepare(*a[:13], pos_key_layer=d["pk"], pos_query_layer=d["pq"]).launch()
    out = _lib.host().varlen(*a)
    assert out is not None and torch.equal(out, ref) and not out[131:].any()


@pytest.mark.parametrize("odd", ["last_dim", "causal", "grad", "dtype", "length", "table", "lens64", "empty"])
def test_calls_left_to_the_python_path(odd):
    d, a = _call()
    if odd == "last_dim":
        a[0] = d["q"].transpose(-1, -2).contiguous().transpose(-1, -2)
    elif odd == "causal":
        a[5] = True
    elif odd == "grad":
        a[0] = d["q"].clone().requires_grad_()
    elif odd == "dtype":
        a[1] = d["k"].half()
    elif odd == "length":
        a[1] = d["k"][:, :, :69]
    elif odd == "table":
        a[9] = d["pk"][:, :500]
    elif odd == "lens64":
        a[11] = torch.tensor([70, 13], device="cuda")
    elif odd == "empty":
        a[:3] = [t[:0] for t in a[:3]]
    assert _lib.host().fixed(*a) is None


@pytest.mark.parametrize("form", ["tables", "lengths", "strips", "packed"])
def test_traced_operators_replay_on_other_inputs(form):
    """A trace holds the call and not its result."""
    def call(q, k, v, pk, pq, n):
        if form == "packed":
            rows = lambda t: t[0].transpose(0, 1)
            return fv.flash_attention_with_disentangled_varlen(rows(q), rows(k), rows(v), None, None, n, n, 70, 70, False, SCALE, 256, 512,
                                                               pos_key_layer=pk, pos_query_layer=pq)
        strips, tables = (None, None), dict(pos_key_layer=pk, pos_query_layer=pq)
        if form == "strips":
            strips, tables = (torch.matmul(x, t.transpose(-1, -2).contiguous()) for x, t in ((q, pk), (k, pq))), {}
        return fa.flash_attention_with_disentangled(q, k, v, *strips, False, SCALE, 256, 512, seqlens_k=n if form == "lengths" else None, **tables)

    def inputs(seed, split):
        d, _ = _call(seed)
        n = [0, split, 70] if form == "packed" else [70, split]
        return d["q"], d["k"], d["v"], d["pk"], d["pq"], torch.tensor(n, dtype=torch.int32, device="cuda")

    call(*inputs(0, 30))                        # (the front takes the call from here on: it has its position table)
    traced = torch.jit.trace(call, inputs(0, 30), check_trace=False)
    for seed, split in [(1, 30), (2, 9)]:
        a = inputs(seed, split)
        assert torch.equal(traced(*a), call(*a))


def test_compute_units_are_the_devices():
    units = torch.cuda.get_device_properties(0).multi_processor_count
    assert _lib.load().tdb_compute_units(0) == _lib.load().tdb_compute_units(-1) == units
    assert _lib.load().tdb_enc_small_splits(768) == min(8, units * 16 // 768)
