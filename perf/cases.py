"""The work that users of this package have it do, as cases that can be timed.

A case is a dict of plain values; ``prepare`` makes what a program has in hand before the call, ``run`` makes the call
through the public entry points: the two attention operators (position terms as per-head tables, or as the strips of
the reference's own signature) and the patched Hugging Face model.  All of them are forward only, as the operators are.
Shapes are those of the DeBERTa-v2/v3 family: head_dim 64, 256 position buckets, relative positions up to 512."""
import math

import numpy as np
import torch

from turbodeberta_amd import _lib
from turbodeberta_amd.ops.flash_attention import flash_attention_with_disentangled
from turbodeberta_amd.ops.flash_attention_varlen import flash_attention_with_disentangled_varlen

D, BUCKETS, MAX_REL, SPAN = 64, 256, 512, 256
SCALE = 1.0 / math.sqrt(3 * D)
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
VOCAB = 128100


def listed():
    return [
        # One short text, answered as it comes in: nothing but latency.
        {"name": "one_text", "kind": "fixed", "dtype": "bf16", "batch": 1, "heads": 12, "lo": 29, "hi": 29, "layout": "qkv"},
        # A small batch in float32, the type that Hugging Face loads checkpoints in.
        {"name": "small_batch_fp32", "kind": "fixed", "dtype": "fp32", "batch": 2, "heads": 12, "lo": 128, "hi": 128, "layout": "qkv"},
        # A padded batch of documents in float32 (question answering windows are 384 tokens long).
        {"name": "documents_fp32", "kind": "fixed", "dtype": "fp32", "batch": 8, "heads": 12, "lo": 96, "hi": 384, "layout": "qkv"},
        # An ordinary classification batch, unpadded, in float16, with q, k, v as contiguous tensors of their own.
        {"name": "classify_fp16", "kind": "fixed", "dtype": "fp16", "batch": 8, "heads": 16, "lo": 250, "hi": 250, "layout": "bhld"},
        # The benchmark's padded batch.
        {"name": "padded_b32_512", "kind": "fixed", "dtype": "bf16", "batch": 32, "heads": 12, "lo": 384, "hi": 512, "layout": "qkv"},
        # The benchmark's packed batch.
        {"name": "packed_64", "kind": "varlen", "dtype": "bf16", "batch": 64, "heads": 12, "lo": 16, "hi": 512, "layout": "qkv"},
        # Many short texts packed together: an indexing or reranking service.
        {"name": "packed_300_short", "kind": "varlen", "dtype": "bf16", "batch": 300, "heads": 12, "lo": 4, "hi": 96, "layout": "qkv"},
        # Long documents, all of one length.
        {"name": "long_b4_4096", "kind": "fixed", "dtype": "bf16", "batch": 4, "heads": 12, "lo": 4096, "hi": 4096, "layout": "qkv"},
        # Long documents of different lengths, packed.
        {"name": "long_packed_8", "kind": "varlen", "dtype": "bf16", "batch": 8, "heads": 12, "lo": 1024, "hi": 4096, "layout": "qkv"},
        # A caller of the reference's signature, who has computed the position strips.
        {"name": "strips_b32_512", "kind": "strips", "dtype": "bf16", "batch": 32, "heads": 12, "lo": 512, "hi": 512, "layout": "bhld"},
        # One text through a whole base-sized model: a request to a serving process.
        {"name": "model_one_text", "kind": "model", "dtype": "bf16", "batch": 1, "heads": 12, "layers": 12, "lo": 48, "hi": 48},
        # A padded batch through a whole large-sized model.
        {"name": "model_large_b16", "kind": "model", "dtype": "bf16", "batch": 16, "heads": 16, "layers": 24, "lo": 64, "hi": 512},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    family = rng.choice(["fixed", "fixed", "fixed", "varlen", "varlen", "varlen", "long", "long", "strips", "fp32", "fp32", "model"])
    heads = rng.choice([12, 12, 16])
    half = rng.choice(["bf16", "bf16", "fp16"])
    layout = rng.choice(["qkv", "qkv", "bhld"])
    if family == "model":
        hi = _log_int(rng, 16, 512)
        batch = _log_int(rng, 1, min(32, 8192 // hi))
        lo = hi if batch == 1 else max(1, int(hi * rng.uniform(0.1, 1.0)))
        return {"kind": "model", "dtype": half, "batch": batch, "heads": heads, "layers": rng.choice([6, 12]), "lo": lo, "hi": hi}
    if family == "long":
        hi = rng.randint(600, 4096)
        batch = rng.randint(1, max(1, min(8, 16384 // hi)))
        kind = rng.choice(["fixed", "varlen"])
        lo = rng.randint(hi // 4, hi) if kind == "varlen" else hi
        return {"kind": kind, "dtype": half, "batch": batch, "heads": 12, "lo": lo, "hi": hi, "layout": layout}
    if family == "strips":
        hi = _log_int(rng, 16, 512)
        batch = _log_int(rng, 1, min(32, 16384 // hi))
        return {"kind": "strips", "dtype": half, "batch": batch, "heads": 12, "lo": rng.choice([hi, max(1, hi // 2)]), "hi": hi, "layout": layout}
    if family == "fp32":
        hi = _log_int(rng, 16, 512)
        batch = _log_int(rng, 1, max(1, min(32, 4096 // hi)))
        lo = rng.choice([hi, max(1, int(hi * rng.uniform(0.1, 1.0)))])
        return {"kind": rng.choice(["fixed", "fixed", "varlen", "strips"]), "dtype": "fp32", "batch": batch, "heads": heads, "lo": lo, "hi": hi, "layout": layout}
    hi = _log_int(rng, 8, 512)
    lo = rng.choice([hi, max(1, int(hi * rng.uniform(0.03, 1.0)))])
    if family == "varlen":
        batch = _log_int(rng, 1, min(320, 24576 // hi))
    else:
        batch = _log_int(rng, 1, min(64, 16384 // hi))
    return {"kind": family, "dtype": half, "batch": batch, "heads": heads, "lo": lo, "hi": hi, "layout": layout}


def _lengths(case, seed=None):
    """Evenly spread over [lo, hi], both ends among them; the seed only says in which order they come."""
    n = case["batch"]
    lens = np.round(np.linspace(case["hi"], case["lo"], n)).astype(np.int64)
    return lens if seed is None else np.random.RandomState(seed).permutation(lens)


def _projected(case, g, shape, dtype):
    """Values as a projection gives them: N(0, 1) hidden states times N(0, 0.02^2) weights."""
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x * (0.02 * math.sqrt(D * case["heads"]))).to(dtype)


def prepare(case, seed):
    if case["kind"] == "model":
        return _prepare_model(case, seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype, H, B, L = DTYPES[case["dtype"]], case["heads"], case["batch"], case["hi"]
    lens = _lengths(case, seed)
    ragged = case["lo"] != case["hi"]
    pk, pq = _projected(case, g, (H, 2 * SPAN, D), dtype), _projected(case, g, (H, 2 * SPAN, D), dtype)
    s = {"kind": case["kind"], "pk": pk, "pq": pq, "q_pos": None, "k_pos": None}
    if case["kind"] == "varlen":
        T = int(lens.sum())
        if case["layout"] == "qkv":      # views of one projection's output
            s["q"], s["k"], s["v"] = _projected(case, g, (T, 3, H, D), dtype).unbind(1)
        else:
            s["q"], s["k"], s["v"] = (_projected(case, g, (T, H, D), dtype) for _ in range(3))
        s["cu"] = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
        s["longest"] = int(lens.max())
        return s
    if case["layout"] == "qkv":
        s["q"], s["k"], s["v"] = _projected(case, g, (B, L, 3, H, D), dtype).permute(2, 0, 3, 1, 4).unbind(0)
    else:
        s["q"], s["k"], s["v"] = (_projected(case, g, (B, H, L, D), dtype) for _ in range(3))
    s["lens"] = torch.from_numpy(lens.astype(np.int32)).cuda() if ragged else None
    if case["kind"] == "strips":
        s["q_pos"] = torch.matmul(s["q"].contiguous(), pk.transpose(-1, -2).contiguous())
        s["k_pos"] = torch.matmul(s["k"].contiguous(), pq.transpose(-1, -2).contiguous())
        s["pk"] = s["pq"] = None
    return s


def _prepare_model(case, seed):
    from transformers import DebertaV2Config, DebertaV2Model
    from turbodeberta_amd.model import patch_model
    hidden = 64 * case["heads"]
    config = DebertaV2Config(vocab_size=VOCAB, hidden_size=hidden, num_hidden_layers=case["layers"],
                             num_attention_heads=case["heads"], intermediate_size=4 * hidden, hidden_dropout_prob=0.0,
                             attention_probs_dropout_prob=0.0, max_position_embeddings=512, type_vocab_size=0,
                             relative_attention=True, position_buckets=BUCKETS, max_relative_positions=MAX_REL,
                             share_att_key=True, pos_att_type=["c2p", "p2c"], norm_rel_ebd="layer_norm",
                             position_biased_input=False, layer_norm_eps=1e-7, initializer_range=0.02)
    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = DebertaV2Model(config)
    model = patch_model(model.to(DTYPES[case["dtype"]]).eval())
    rs = np.random.RandomState(seed)
    lens = _lengths(case, seed)
    ids = rs.randint(1, VOCAB, size=(case["batch"], case["hi"]))
    ids[np.arange(case["hi"])[None] >= lens[:, None]] = 0
    return {"kind": "model", "model": model, "ids": torch.from_numpy(ids).cuda()}


def run(state):
    if state["kind"] == "model":
        with torch.no_grad():            # every batch brings a mask of its own: id 0 is padding
            ids = state["ids"]
            return state["model"](input_ids=ids, attention_mask=ids.ne(0).long()).last_hidden_state
    if state["kind"] == "varlen":
        return flash_attention_with_disentangled_varlen(
            state["q"], state["k"], state["v"], None, None, state["cu"], state["cu"], state["longest"], state["longest"],
            False, SCALE, BUCKETS, MAX_REL, pos_key_layer=state["pk"], pos_query_layer=state["pq"])
    return flash_attention_with_disentangled(
        state["q"], state["k"], state["v"], state["q_pos"], state["k_pos"], False, SCALE, BUCKETS, MAX_REL,
        pos_key_layer=state["pk"], pos_query_layer=state["pq"], seqlens_k=state["lens"])


def work(case):
    """Matrix products and bytes of one pass, without the padding: per head and sequence of l tokens 4 l l D for the
    scores and values, 4 l W D for the two position terms (W = relative positions that occur); a caller of the strips has
    done the latter.  q, k, v in and o out, and the tables, or the columns of the strips that some pair addresses."""
    lens, H, size = _lengths(case), case["heads"], 4 if case["dtype"] == "fp32" else 2
    tokens = float(lens.sum())
    flops = bytes_ = 0.0
    columns = {}
    for l in (int(x) for x in lens):
        flops += 4.0 * l * l * D
        if case["kind"] == "strips":
            if l not in columns:
                delta = _lib.delta_table(l, BUCKETS, MAX_REL).astype(np.int64)
                columns[l] = float((delta[l - 1:] - delta[:l] + 1).sum())
            bytes_ += 2.0 * size * H * columns[l]
        else:
            flops += 4.0 * l * min(2 * SPAN, 2 * l - 1) * D
    flops *= H
    if case["kind"] == "model":
        hidden = 64 * H
        weights = 12.0 * hidden * hidden
        return {"flops": case["layers"] * (flops + 2.0 * tokens * weights),
                "bytes": size * (case["layers"] * (weights + 4.0 * SPAN * hidden) + 2.0 * tokens * hidden)}
    if case["kind"] != "varlen":         # padded rows of the output are written as well
        bytes_ += size * (case["batch"] * case["hi"] - tokens) * H * D
    if case["kind"] != "strips":
        bytes_ += 2.0 * size * H * min(2 * SPAN, 2 * case["hi"] - 1) * D
    return {"flops": flops, "bytes": bytes_ + 4.0 * size * tokens * H * D}


def tolerance(case):
    """float32: sums of 64 products and of up to 512 weighted values.  16 bits: the probabilities, the position terms and
    the result are each rounded once.  A model rounds its hidden states some six times in each layer."""
    if case["kind"] == "model":
        return {"rel": 2e-2 if case["dtype"] == "bf16" else 3e-3}
    return {"rel": {"fp32": 1e-5, "bf16": 1e-2, "fp16": 2e-3}[case["dtype"]]}
