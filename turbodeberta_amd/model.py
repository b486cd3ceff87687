"""Hugging Face DeBERTa-v2/v3 modules with the attention core running on the fused MI355X kernel.

Class names follow TurboDeBERTa's ``model.py`` (``FlashDisentangledSelfAttention``,
``FlashDebertaV2Attention/Layer/Encoder/Model``).  Submodule and parameter names are Hugging Face's,
so a stock DeBERTa-v2/v3 ``state_dict`` loads unchanged; ``patch_model`` switches an already built
(e.g. ``from_pretrained``) model over in place.

What differs from the reference glue (model.py:34-186):
* no ``[B, H, L, 2*span]`` strips: the per-head projections of the relative embeddings go to the
  kernel, which contracts them on the matrix cores (``pos_key_layer`` / ``pos_query_layer``);
* q, k, v are passed as strided ``[B, H, L, D]`` views of the projection outputs -- no
  ``permute().contiguous()`` (model.py:70-78), and the output is written token-major so the final
  ``[B, L, H*D]`` is a view;
* padding is handled by per-sequence lengths inside the fixed-length kernel: no un-pad / re-pad
  gathers (model.py:138-183) and no host synchronisation (model.py:55-63, padding.py:82);
* the position index is Hugging Face's for both terms (modeling_deberta_v2.py:318, :336-343);
* in eval mode, work that does not depend on the input is done once instead of once per call: the
  per-head position tables (a function of the layer's weights and the shared relative embeddings
  only; the reference recomputes both strip GEMMs every call, model.py:94-110) and the
  concatenated Q/K/V weight of the single fused projection GEMM; the valid lengths are computed by
  the first layer that sees a mask and reused by the others (the reference recomputes them, with
  a host synchronisation, in every layer: model.py:55-63);
* in eval mode the encoder keeps a batch with padding packed from the embeddings to the last layer:
  projections, LayerNorms and feed-forward blocks run on ``[valid_tokens, hidden]`` and the packed
  attention kernel is called with views of the projection output, so padded positions cost
  nothing anywhere.  The reference packs and re-pads around the attention call of every layer
  (model.py:138-183); here there is one gather after the embeddings, one scatter at the end and one
  host synchronisation (the number of valid tokens) per forward.
"""
from __future__ import annotations

import math
import weakref
from typing import Optional

import torch
from torch import nn
from torch.utils._device import DeviceContext
from transformers.activations import GELUActivation
from transformers.modeling_outputs import BaseModelOutput
from transformers.models.deberta_v2.modeling_deberta_v2 import (
    DebertaV2Attention,
    DebertaV2Embeddings,
    DebertaV2Encoder,
    DebertaV2ForMaskedLM,
    DebertaV2ForMultipleChoice,
    DebertaV2ForQuestionAnswering,
    DebertaV2ForSequenceClassification,
    DebertaV2ForTokenClassification,
    DebertaV2Intermediate,
    DebertaV2Layer,
    DebertaV2Model,
    DebertaV2Output,
    DebertaV2SelfOutput,
    DisentangledSelfAttention,
)

from . import _lib
from .ops._launch import delta_lut
from .ops.flash_attention import flash_attention_with_disentangled
from .ops.flash_attention_varlen import flash_attention_with_disentangled_varlen
from .padding import index_first_axis, key_padding_mask, pad_input


def _versions(*tensors):
    """Identity of a set of live tensors (parameters) for cache keys: object, storage address and in-place
    modification counter.  Only meaningful for tensors that stay alive between the calls that compare keys."""
    return tuple((id(t), t.data_ptr(), t._version, t.dtype, t.device) if t is not None else None for t in tensors)


def _version_of(t):
    """In-place modification counter of a tensor, or None where there is none to read (inference tensors do not
    track one and raise on access)."""
    try:
        return t._version
    except (RuntimeError, AttributeError):
        return None


def _lasting(t):
    """Whether what is computed now from ``t`` may be kept for later calls: under graph capture it holds nothing before the
    graph is replayed."""
    return not (t.is_cuda and torch.cuda.is_current_stream_capturing())


class _MaskInfo:
    """What the fused paths need to know about an attention mask: ``lengths`` int32 ``[B]`` on the device,
    ``total``, the number of valid tokens (a host int; ``None`` when the caller declared the lengths without it), the
    running sum ``cu`` of the lengths (or None: not computed yet), the ``stream`` on which that sum has been queued (None: it
    is there), whether every nonzero entry is 1 (None: unknown) and whether the caller declared all this."""
    __slots__ = ("lengths", "total", "cu", "ones", "declared", "stream")

    def __init__(self, lengths, total, cu=None, ones=None, declared=False):
        self.lengths, self.total, self.cu, self.ones, self.declared, self.stream = lengths, total, cu, ones, declared, None


def _mask_info(attention_mask, ids=None, vocab=0):
    """Valid lengths of a batch whose mask is **right padded** (valid tokens first), verified: the kernels take
    per-sequence lengths, so a mask with holes or left padding cannot be expressed and raises ``ValueError`` instead
    of attending to the wrong tokens.  A 3-D / 4-D mask must be the outer product ``m_i * m_j`` Hugging Face's
    encoder builds (modeling_deberta_v2.py:601-608), or one row ``[.., 1, L]`` that broadcasts over the queries, and the
    same for every head; other shapes raise ``ValueError`` in ``key_padding_mask``.  The check costs one host synchronisation per mask object;
    the result is attached to the tensor, so the layers of an encoder, which all receive the same mask object
    (modeling_deberta_v2.py:651-660), share it.  (A mask without a modification counter -- an inference tensor --
    is trusted not to be modified in place between calls.)  Under ``torch.jit.trace`` nothing is attached or taken from an
    earlier call: to the tracer such lengths are constants, and a replay on another mask would go by the first one's.

    With ``ids`` (of the mask's shape), a valid token whose id does not lie in ``[0, vocab)`` raises ``IndexError`` where the
    mask is measured by the one kernel, which then reads the ids as well."""
    version = _version_of(attention_mask)
    tracing = torch.jit.is_tracing()
    cached = getattr(attention_mask, "_tdb_info", None)
    if cached is not None and cached[0] == version and (cached[1].declared or not tracing):
        if not cached[1].declared and attention_mask.is_cuda:        # (they live as long as the mask, whose owner does not know them)
            cached[1].lengths.record_stream(torch.cuda.current_stream(attention_mask.device))
        return cached[1]
    scan = _lib.host().scan_mask(attention_mask, ids, vocab) if attention_mask.is_cuda and attention_mask.dim() == 2 else None
    if scan is not None:                                             # one kernel, one synchronisation
        lengths, cu, ok_host, total, ones, known = scan
        if not known:
            raise IndexError(f"input_ids: the ids of valid tokens must lie in [0, {vocab})")
    else:
        cu = ones = None
        valid = key_padding_mask(attention_mask) != 0                               # [B, L]
        L = valid.shape[-1]
        lengths = valid.sum(dim=-1, dtype=torch.int32)
        ok = (valid == (torch.arange(L, device=valid.device)[None, :] < lengths[:, None])).all()
        if attention_mask.dim() == 4 and attention_mask.shape[1] > 1:
            ok = ok & ((attention_mask != 0) == (attention_mask[:, :1] != 0)).all()      # one length per sequence: no per-head masks
        if attention_mask.dim() > 2 and attention_mask.shape[-2] == L and L > 1:
            full = attention_mask if attention_mask.dim() == 3 else attention_mask[:, 0]
            ok = ok & ((full != 0) == (valid[:, :, None] & valid[:, None, :])).all()
        ok_host, total = torch.stack([ok.to(torch.int64), lengths.sum(dtype=torch.int64)]).tolist()   # the one synchronisation
    if not ok_host:
        raise ValueError("attention_mask must be right padded (valid tokens first, no holes) and, if 3-D or 4-D, the "
                         "outer product of a key-padding mask with itself (or one broadcast row of it), equal for all "
                         "heads: the fused attention takes per-sequence lengths.  Use the eager Hugging Face modules for "
                         "other masks.")
    info = _MaskInfo(lengths, int(total), cu, ones)
    if tracing:
        return info
    try:
        attention_mask._tdb_info = (version, info)
    except AttributeError:      # tensor subclasses without a __dict__
        pass
    return info


def declare_right_padded(attention_mask, lengths, total=None):
    """Opt out of the mask inspection: the caller vouches that ``attention_mask`` is right padded with ``lengths``
    (int32 ``[B]`` on the mask's device) valid tokens per sequence.  The facts are attached to the mask tensor the way
    ``_mask_info`` caches its own findings, so every fused module that receives this mask object uses them and none
    synchronises with the host: a forward on such a mask can be captured into a HIP graph.  ``total`` (a host int, the
    sum of the lengths) additionally lets the encoder pack the batch; without it the encoder keeps the padded layout,
    because the packed token count sizes host-side allocations.  Nothing is verified: wrong lengths, or a total that is
    not their sum, give wrong results.  (The mask's entries are taken to be 0 and 1.)  Returns the mask."""
    if lengths.dtype != torch.int32 or lengths.dim() != 1 or lengths.shape[0] != attention_mask.shape[0]:
        raise ValueError("lengths must be an int32 tensor with one entry per sequence of the mask")
    if lengths.device != attention_mask.device:
        raise ValueError("lengths must live on the mask's device")
    attention_mask._tdb_info = (_version_of(attention_mask), _MaskInfo(lengths, None if total is None else int(total), ones=True, declared=True))
    return attention_mask


def _boundaries(info):
    """int32 ``[B+1]`` running sum of the lengths, with a leading 0.  Kept for later calls on the same stream."""
    n, tracing = info.lengths, torch.jit.is_tracing()
    stream = torch.cuda.current_stream(n.device).cuda_stream if n.is_cuda else None
    if info.cu is not None and not tracing and info.stream in (None, stream):
        return info.cu
    cu = torch.nn.functional.pad(torch.cumsum(n, dim=0, dtype=torch.int32), (1, 0))
    if not tracing and _lasting(n):
        info.cu, info.stream = cu, stream
    return cu


def _packing_of(info, batch, seqlen, device):
    """``(indices, cu_seqlens)`` of a verified right-padded batch without a further synchronisation: positions of the
    valid tokens in the flattened ``[B*L]`` batch, int32 boundaries with a leading 0.  (Under ``torch.jit.trace`` their
    number is found again in every replay.)"""
    cu = _boundaries(info)
    if torch.jit.is_tracing():
        valid = torch.arange(seqlen, device=device)[None, :] < info.lengths[:, None]
        return torch.nonzero(valid.flatten()).flatten(), cu
    token, starts = torch.arange(info.total, device=device), cu.long()
    seq = torch.searchsorted(starts[1:], token, right=True).clamp_(max=batch - 1)
    return (token - starts[seq] + seq * seqlen).clamp_(0, batch * seqlen - 1), cu     # (a caller's lengths may not fit)


class FlashDisentangledSelfAttention(DisentangledSelfAttention):
    """``DisentangledSelfAttention`` (modeling_deberta_v2.py:137-345) with the score / softmax / value
    product replaced by one kernel launch.  Same constructor, parameters and ``forward`` signature.

    Masks: sequences must be right-padded (valid tokens first), which is what the DeBERTa tokenizers
    produce; the valid length of each sequence is taken from the mask, and a mask of any other shape
    (holes, left padding, a 3-D / 4-D mask that is not ``m_i * m_j``) raises ``ValueError`` -- checked
    once per mask object, with one host synchronisation.  Rows of padded query tokens
    are returned as zeros (the eager module gives them a meaningless uniform average,
    modeling_deberta_v2.py:256-259); downstream layers mask them anyway.
    ``output_attentions=True`` needs the probability matrix, which the fused kernel never forms: that
    call is served by the eager parent class."""

    def forward(self, hidden_states, attention_mask, output_attentions=False, query_states=None,
                relative_pos=None, rel_embeddings=None):
        if output_attentions:
            return super().forward(hidden_states, attention_mask, output_attentions, query_states,
                                   relative_pos, rel_embeddings)
        if query_states is None:
            query_states = hidden_states
        B, L, _ = hidden_states.shape
        H, D = self.num_attention_heads, self.attention_head_size
        if query_states.shape[1] != L:
            raise ValueError("self-attention only: query_states and hidden_states must have one length")

        frozen = not self.training and not torch.is_grad_enabled()       # nothing below can change between calls
        if frozen and query_states is hidden_states:
            # one projection GEMM; q, k, v are views into its [B, L, 3, H, D] output (token stride 3*H*D)
            w, b = self._fused_qkv()
            qkv = nn.functional.linear(hidden_states, w, b).view(B, L, 3, H, D)
            q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
        else:
            heads = lambda x: x.view(B, L, H, D).permute(0, 2, 1, 3)      # [B, H, L, D] view, token-major storage
            q = heads(self.query_proj(query_states))
            k = heads(self.key_proj(hidden_states))
            v = heads(self.value_proj(hidden_states))

        pos_key, pos_query, sm_scale, buckets, max_rel = self._position_terms(rel_embeddings, hidden_states.dtype,
                                                                              frozen)
        seqlens = _mask_info(attention_mask).lengths if attention_mask is not None else None
        out = flash_attention_with_disentangled(q, k, v, None, None, False, sm_scale, buckets, max_rel,
                                                pos_key_layer=pos_key, pos_query_layer=pos_query,
                                                seqlens_k=seqlens)
        # out has q's strides: [B, H, L, D] view of token-major storage
        return (out.permute(0, 2, 1, 3).reshape(B, L, H * D), None)

    def forward_packed(self, hidden_states, cu_seqlens, max_seqlen, rel_embeddings=None):
        """Eval-mode forward on packed tokens: ``hidden_states [T, hidden]`` holds the valid tokens of all
        sequences back to back, ``cu_seqlens`` int32 ``[B+1]`` their boundaries.  Returns ``[T, H*D]``.
        The counterpart of the reference's packed branch (model.py:138-183) without its per-layer gathers."""
        T = hidden_states.shape[0]
        H, D = self.num_attention_heads, self.attention_head_size
        w, b = self._fused_qkv()
        qkv = nn.functional.linear(hidden_states, w, b).view(T, 3, H, D)
        pos_key, pos_query, sm_scale, buckets, max_rel = self._position_terms(rel_embeddings, hidden_states.dtype, True)
        out = flash_attention_with_disentangled_varlen(qkv[:, 0], qkv[:, 1], qkv[:, 2], None, None, cu_seqlens,
                                                       cu_seqlens, max_seqlen, max_seqlen, False, sm_scale, buckets,
                                                       max_rel, pos_key_layer=pos_key, pos_query_layer=pos_query,
                                                       zero_output=False)      # the packing comes from the verified mask
        return out.reshape(T, H * D)

    def _position_terms(self, rel_embeddings, dtype, frozen):
        """``(pos_key, pos_query, sm_scale, position_buckets, max_relative_positions)`` of one call."""
        scale_factor = 1
        pos_key = pos_query = None
        buckets = max_rel = 0
        if self.relative_attention:
            scale_factor += int("c2p" in self.pos_att_type) + int("p2c" in self.pos_att_type)
            buckets, max_rel = self.position_buckets, self.max_relative_positions
            if frozen:
                pos_key, pos_query = self._position_tables(rel_embeddings, dtype)
            else:
                rel = self.pos_dropout(rel_embeddings)[0:2 * self.pos_ebd_size]                 # HF:295
                pos_key, pos_query = self._project_tables(rel)
        return pos_key, pos_query, 1.0 / math.sqrt(self.attention_head_size * scale_factor), buckets, max_rel   # HF:120-121, :243

    def _project_tables(self, rel):
        """Per-head projections of the relative embeddings, ``[H, 2*span, D]`` views (modeling_deberta_v2.py:296-312)."""
        H, D = self.num_attention_heads, self.attention_head_size
        table = lambda proj: proj(rel).view(rel.shape[0], H, D).permute(1, 0, 2)
        pos_key = pos_query = None
        if "c2p" in self.pos_att_type:
            pos_key = table(self.key_proj if self.share_att_key else self.pos_key_proj)
        if "p2c" in self.pos_att_type:
            pos_query = table(self.query_proj if self.share_att_key else self.pos_query_proj)
        return pos_key, pos_query

    def _position_tables(self, rel_embeddings, dtype):
        """Eval-mode cache of ``_project_tables``: recomputed only when the relative embeddings or the
        projection weights have been modified (or moved / cast)."""
        kp = self.key_proj if self.share_att_key else getattr(self, "pos_key_proj", None)
        qp = self.query_proj if self.share_att_key else getattr(self, "pos_query_proj", None)
        # Identity of the relative embeddings: the encoder's layer-normed copy is a temporary, whose address says
        # nothing (it can be reused by a later, different tensor); FlashDebertaV2Encoder tags what it hands out with
        # the identity of its sources.  A parameter speaks for itself.  Anything else is not cached.
        source = getattr(rel_embeddings, "_tdb_source", None)
        if source is None and isinstance(rel_embeddings, nn.Parameter):
            source = _versions(rel_embeddings)
        if source is None:
            return self._project_tables(rel_embeddings[0:2 * self.pos_ebd_size])
        key = (source, _versions(*(t for m in (kp, qp) if m is not None for t in (m.weight, m.bias))), dtype)
        cached = self.__dict__.get("_tdb_tables")
        if cached is None or cached[0] != key:
            rel = rel_embeddings[0:2 * self.pos_ebd_size]                # dropout is the identity in eval mode
            cached = (key, self._project_tables(rel))
            if _lasting(rel):
                self.__dict__["_tdb_tables"] = cached
        return cached[1]

    def _fused_qkv(self):
        """Eval-mode cache of the concatenated ``[3*H*D, hidden]`` projection weight (and bias)."""
        mods = (self.query_proj, self.key_proj, self.value_proj)
        key = _versions(*(t for m in mods for t in (m.weight, m.bias)))
        cached = self.__dict__.get("_tdb_qkv")
        if cached is None or cached[0] != key:
            w = torch.cat([m.weight for m in mods], dim=0)
            b = torch.cat([m.bias for m in mods], dim=0) if all(m.bias is not None for m in mods) else None
            if b is None and any(m.bias is not None for m in mods):
                b = torch.cat([m.bias if m.bias is not None else m.weight.new_zeros(m.weight.shape[0]) for m in mods])
            cached = (key, (w, b))
            if _lasting(w):
                self.__dict__["_tdb_qkv"] = cached
        return cached[1]


class FlashDebertaV2Attention(DebertaV2Attention):
    def __init__(self, config):
        super().__init__(config)
        self.self = FlashDisentangledSelfAttention(config)


class FlashDebertaV2Layer(DebertaV2Layer):
    def __init__(self, config):
        super().__init__(config)
        self.attention = FlashDebertaV2Attention(config)


class FlashDebertaV2Encoder(DebertaV2Encoder):
    """``DebertaV2Encoder`` (modeling_deberta_v2.py:565-686) over ``FlashDebertaV2Layer``.

    In eval mode under ``torch.no_grad()`` a batch that contains padding runs **packed**: the valid tokens
    are gathered once, every layer works on ``[valid_tokens, hidden]`` (``forward_packed`` of the attention
    module, then Hugging Face's own output / feed-forward submodules, which are shape agnostic), and the
    result is scattered back to ``[B, L, hidden]`` with zeros at padded positions.  Verifying the mask and
    counting the valid tokens is the only host synchronisation of the forward.  Everything else -- training,
    gradients, ``output_attentions``, ``query_states``, CPU tensors, batches without padding -- takes the
    parent's loop over the (fused, padded) layers.  Masks must be right padded in either path (see
    ``FlashDisentangledSelfAttention``); others raise ``ValueError``.

    ``pack_sequences = False`` switches the packed path off."""

    pack_sequences = True

    def __init__(self, config):
        super().__init__(config)
        self.layer = nn.ModuleList([FlashDebertaV2Layer(config) for _ in range(config.num_hidden_layers)])

    def get_rel_embedding(self):
        """As the parent (modeling_deberta_v2.py:593-597); in eval mode under ``no_grad`` the (layer-normed) result is
        computed once per state of its sources and tagged with their identity, which the attention modules key
        their position-table caches on."""
        if self.training or torch.is_grad_enabled() or not self.relative_attention:
            return super().get_rel_embedding()
        sources = [self.rel_embeddings.weight]
        if "layer_norm" in self.norm_rel_ebd:
            sources += [self.LayerNorm.weight, self.LayerNorm.bias]
        key = _versions(*sources)
        cached = self.__dict__.get("_tdb_rel")
        if cached is None or cached[0] != key:
            rel = super().get_rel_embedding()
            if rel is self.rel_embeddings.weight:
                rel = rel.detach()           # a tensor of its own to carry the tag (shares the storage)
            rel._tdb_source = key
            cached = (key, rel)
            if _lasting(rel):
                self.__dict__["_tdb_rel"] = cached
        return cached[1]

    def forward(self, hidden_states, attention_mask, output_hidden_states=True, output_attentions=False,
                query_states=None, relative_pos=None, return_dict=True, intermediate_states=True):
        """As the parent (modeling_deberta_v2.py:634-695).  ``intermediate_states=False`` (an argument of this class
        only) says that of the hidden states the caller reads just the first and the last: the packed path then
        leaves the layers in between out of the returned tuple instead of scattering each back to ``[B, L, hidden]``."""
        fused = (not output_attentions and torch.is_tensor(hidden_states)
                 and all(isinstance(l.attention.self, FlashDisentangledSelfAttention) for l in self.layer))
        packable = (fused and self.pack_sequences and not self.training and not torch.is_grad_enabled()
                    and query_states is None and hidden_states.is_cuda and attention_mask.dim() in (2, 3, 4))
        if packable:
            B, L, _ = hidden_states.shape
            info = _mask_info(attention_mask)                                # the one host synchronisation
            packable = info.total is not None and info.total < B * L      # (no total: declared by the caller)
            if packable:
                indices, cu_seqlens = _packing_of(info, B, L, hidden_states.device)
        if not packable:
            if fused and relative_pos is None and self.relative_attention:
                relative_pos = hidden_states.new_empty(0)    # fused layers never read the [L, L] matrix: do not build it
            return super().forward(hidden_states, attention_mask, output_hidden_states, output_attentions,
                                   query_states, relative_pos, return_dict)

        keep_all = output_hidden_states and intermediate_states
        padded = lambda t: pad_input(t, indices, B, L)
        all_hidden_states = (hidden_states,) if output_hidden_states else None
        rel_embeddings = self.get_rel_embedding()
        x = index_first_axis(hidden_states.reshape(B * L, -1), indices)
        for i, layer in enumerate(self.layer):
            attn = layer.attention
            attended = attn.output(attn.self.forward_packed(x, cu_seqlens, L, rel_embeddings), x)     # HF:368-378
            x = layer.output(layer.intermediate(attended), attended)                                   # HF:431-432
            if i == 0 and self.conv is not None:                                                       # HF:666-667
                x = index_first_axis(self.conv(hidden_states, padded(x), key_padding_mask(attention_mask).long())
                                     .reshape(B * L, -1), indices)
            if keep_all and i + 1 < len(self.layer):
                all_hidden_states = all_hidden_states + (padded(x),)
        output_states = padded(x)
        if output_hidden_states:
            all_hidden_states = all_hidden_states + (output_states,)
        if not return_dict:
            return tuple(v for v in [output_states, all_hidden_states, None] if v is not None)
        return BaseModelOutput(last_hidden_state=output_states, hidden_states=all_hidden_states, attentions=None)


# Plans of the native encoder loop, by model (kept outside the modules: a plan can be neither copied nor pickled).  False: the
# model's structure is not one the loop knows.
_PLANS = weakref.WeakKeyDictionary()


def _native_plan(model):
    """The plan of ``model`` for the native loop from token ids to the last hidden state (csrc/host_encoder.cpp), or None:
    the plan of an earlier call if the module tree is still what it was, else a new one."""
    host = _lib.host()
    plan = _PLANS.get(model)
    if plan is False or torch.nn.modules.module._has_any_global_hook():
        return None
    if plan is not None and host.plan_ok(plan, model):
        return plan
    if not _known_structure(model):
        _PLANS[model] = False
        return None
    _PLANS.pop(model, None)
    plan = host.begin_plan(model) if _stock_methods() else None
    if plan is None:                             # a module in training mode, a hook, a forward of its own, ...
        return None
    emb, enc = model.embeddings, model.encoder
    table = emb.word_embeddings.weight
    rel = enc.get_rel_embedding()
    layers = []
    for layer in enc.layer:
        att, so, mid, out = layer.attention.self, layer.attention.output, layer.intermediate.dense, layer.output
        wqkv, bqkv = att._fused_qkv()
        pos_key, pos_query, scale, buckets, max_rel = att._position_terms(rel, table.dtype, True)
        layers.append((wqkv, bqkv, pos_key, pos_query, so.dense.weight, so.dense.bias, so.LayerNorm.weight, so.LayerNorm.bias,
                       mid.weight, mid.bias, out.dense.weight, out.dense.bias, out.LayerNorm.weight, out.LayerNorm.bias,
                       float(so.LayerNorm.eps), float(out.LayerNorm.eps)))
    tensors = [t for l in layers for t in l[:14] if t is not None] + [table, emb.LayerNorm.weight, emb.LayerNorm.bias]
    if any(t.dtype != table.dtype or t.device != table.device or t.data_ptr() % 16 or not (t.is_contiguous() or t.dim() == 3) for t in tensors):
        return None
    if not host.complete_plan(plan, model, layers, (table, emb.LayerNorm.weight, emb.LayerNorm.bias, float(emb.LayerNorm.eps)),
                              att.num_attention_heads, att.attention_head_size, scale, buckets, max_rel):
        return None
    if _lasting(table):
        if table.is_cuda:
            torch.cuda.current_stream(table.device).synchronize()    # later calls may come on other streams
        _PLANS[model] = plan
    return plan


# What the native loop takes to be the same in all attention modules
_PER_MODEL = ("num_attention_heads", "attention_head_size", "pos_att_type", "relative_attention", "position_buckets", "max_relative_positions")


def _known_structure(model):
    """Whether the modules below ``model`` compute what the native loop computes: stock DeBERTa-v2/v3 layers with the fused
    attention, exact GELU, no convolution, embeddings that are a table and a LayerNorm, and in the places of the dropouts
    dropouts, which the loop leaves out."""
    emb, enc = model.embeddings, model.encoder
    dropout = lambda m: type(m._modules.get("dropout")) is nn.Dropout
    plain = lambda m, *names: all(type(getattr(m, n)) is nn.Linear and getattr(m, n).bias is not None for n in names)
    norm = lambda m: type(m) is nn.LayerNorm and m.weight is not None and m.bias is not None
    if not (type(emb) is DebertaV2Embeddings and type(emb.word_embeddings) is nn.Embedding and emb.word_embeddings.max_norm is None
            and not emb.position_biased_input and emb.token_type_embeddings is None and emb.embed_proj is None and norm(emb.LayerNorm) and dropout(emb)
            and type(enc) is FlashDebertaV2Encoder and enc.conv is None and len(enc.layer) > 0):
        return False
    hidden = emb.word_embeddings.weight.shape[1]
    if hidden % 8 or hidden > 4096 or emb.word_embeddings.weight.dtype not in (torch.float32, torch.bfloat16, torch.float16):
        return False
    first = None                                 # (attention, feed-forward) of the first layer
    for layer in enc.layer:
        if not (type(layer) in (DebertaV2Layer, FlashDebertaV2Layer) and type(layer.attention) in (DebertaV2Attention, FlashDebertaV2Attention)):
            return False
        att, so, mid, out = layer.attention.self, layer.attention.output, layer.intermediate, layer.output
        first = first or (att, mid)
        if not (type(att) is FlashDisentangledSelfAttention and type(so) is DebertaV2SelfOutput and type(mid) is DebertaV2Intermediate
                and type(out) is DebertaV2Output and type(mid.intermediate_act_fn) is GELUActivation
                and mid.intermediate_act_fn.act is nn.functional.gelu
                and dropout(att) and dropout(so) and dropout(out) and type(att._modules.get("pos_dropout")) in (nn.Dropout, type(None))):
            return False
        if not (plain(att, "query_proj", "key_proj", "value_proj") and plain(so, "dense") and plain(out, "dense") and plain(mid, "dense")
                and norm(so.LayerNorm) and norm(out.LayerNorm) and att.num_attention_heads * att.attention_head_size == hidden == out.dense.out_features
                and mid.dense.out_features == first[1].dense.out_features
                and all(getattr(att, n, None) == getattr(first[0], n, None) for n in _PER_MODEL)):
            return False
    return True


# The methods that the native loop was written for, as their classes' own files define them; where one has been replaced on
# its class the modules are run.  (What happens to them later, or on an instance, the snapshot of a plan sees.)
_LOOP_TYPES = (nn.Linear, nn.LayerNorm, nn.Embedding, nn.Dropout, GELUActivation, DebertaV2Embeddings, DebertaV2Attention, DebertaV2SelfOutput,
               DebertaV2Intermediate, DebertaV2Output, DebertaV2Layer, FlashDebertaV2Attention, FlashDebertaV2Layer,
               FlashDisentangledSelfAttention, FlashDebertaV2Encoder)


def _own(cls, name):
    """The class's method of this name (None: it has none), or an object that is nobody's method where another module put
    it there."""
    owner = next((c for c in cls.__mro__ if name in vars(c)), None)
    f = owner and vars(owner)[name]
    return f if f is None or (f.__module__ == owner.__module__ and not hasattr(f, "__wrapped__")) else object()


_STOCK = [(cls, name, _own(cls, name)) for cls in _LOOP_TYPES for name in ("forward", "__call__", "forward_packed", "get_rel_embedding")]


def _stock_methods():
    return all(getattr(cls, name, None) is method for cls, name, method in _STOCK)


def _observed():
    """Whether somebody watches the operations of this thread, or changes them: a tracer, a dispatch mode, a function mode
    other than a default device."""
    return _lib.host().observed() or any(type(torch._C._get_function_stack_at(i)) is not DeviceContext
                                         for i in range(torch._C._len_torch_function_stack()))


class FlashDebertaV2Model(DebertaV2Model):
    def __init__(self, config):
        super().__init__(config)
        self.encoder = FlashDebertaV2Encoder(config)
        self.post_init()

    def forward(self, input_ids=None, attention_mask=None, token_type_ids=None, position_ids=None,
                inputs_embeds=None, output_attentions=None, output_hidden_states=None, return_dict=None, **kwargs):
        """As the parent (modeling_deberta_v2.py:711-793), which always asks the encoder for every layer's output and
        then uses the last one (modeling_deberta_v2.py:760-768).  When the caller did not ask for the hidden states
        (and no ``z_steps`` pass needs the last but one), the encoder is told so through its ``intermediate_states``
        argument, so that the packed path does not scatter every layer's result back to ``[B, L, hidden]`` for
        nothing.  Nothing is stored on the modules: concurrent calls on one model do not see each other's flags.

        Ids outside the vocabulary: where the native loop runs and a mask is measured (the first call with a mask object) a
        valid token's id raises ``IndexError``; without a mask, with one that has been measured before or that the caller has
        declared, nothing is read back and every token of that id's sequence comes back as NaN.  The other paths are
        PyTorch's embedding, whose kernel aborts the process."""
        cfg = self.config
        want_hidden = output_hidden_states if output_hidden_states is not None else cfg.output_hidden_states
        if want_hidden or self.z_steps > 1 or kwargs:
            return super().forward(input_ids=input_ids, attention_mask=attention_mask, token_type_ids=token_type_ids,
                                   position_ids=position_ids, inputs_embeds=inputs_embeds,
                                   output_attentions=output_attentions, output_hidden_states=output_hidden_states,
                                   return_dict=return_dict, **kwargs)
        output_attentions = output_attentions if output_attentions is not None else cfg.output_attentions
        return_dict = return_dict if return_dict is not None else cfg.return_dict
        if (input_ids is None) == (inputs_embeds is None):
            raise ValueError("You have to specify exactly one of input_ids and inputs_embeds")
        given = input_ids if input_ids is not None else inputs_embeds[..., 0]
        if input_ids is not None:
            self.warn_if_padding_and_no_attention_mask(input_ids, attention_mask)
            if not output_attentions:
                last = self._forward_native(input_ids, attention_mask)
                if last is not None:
                    return BaseModelOutput(last_hidden_state=last, hidden_states=None, attentions=None) if return_dict else (last,)
        if attention_mask is None:
            attention_mask = torch.ones(given.shape, device=given.device)
        if token_type_ids is None:
            token_type_ids = torch.zeros(given.shape, dtype=torch.long, device=given.device)
        embedded = self.embeddings(input_ids=input_ids, token_type_ids=token_type_ids, position_ids=position_ids,
                                   mask=attention_mask, inputs_embeds=inputs_embeds)
        encoded = self.encoder(embedded, attention_mask, output_hidden_states=True, output_attentions=output_attentions,
                               return_dict=return_dict, intermediate_states=False)
        sequence_output = encoded[1][-1]
        if not return_dict:
            return (sequence_output,) + tuple(encoded[2:])
        return BaseModelOutput(last_hidden_state=sequence_output, hidden_states=None, attentions=encoded.attentions)


    def _forward_native(self, input_ids, attention_mask):
        """The last hidden state through the native loop, or None where the modules have to be run: with gradients, in
        training mode, under autocast, a compiler, a tracer or a mode that watches the operations, with hooks, for masks other
        than 2-D ones of zeros and ones.  As in the packed encoder, padded positions come back as zeros."""
        if (self.training or torch.is_grad_enabled() or not input_ids.is_cuda or input_ids.dim() != 2 or not input_ids.numel()
                or not getattr(self.encoder, "pack_sequences", False) or torch.is_autocast_enabled() or torch.compiler.is_compiling()
                or _observed()):
            return None
        B, L = input_ids.shape
        if attention_mask is not None and (attention_mask.shape != input_ids.shape or attention_mask.device != input_ids.device):
            return None
        plan = _native_plan(self)
        if plan is None:
            return None
        cu, total = None, B * L
        if attention_mask is not None:
            info = _mask_info(attention_mask, input_ids, self.embeddings.word_embeddings.weight.shape[0])    # the one host synchronisation
            if not info.total or not info.ones:
                return None
            if info.total < B * L:
                cu, total = _boundaries(info), info.total
        enc = self.encoder
        if enc.relative_attention:
            delta_lut(input_ids.device, L, enc.layer[0].attention.self.position_buckets, enc.layer[0].attention.self.max_relative_positions)
        return _lib.host().encode(plan, input_ids, cu, total)


class _FusedHead:
    """Task models with the reference's class names (model.py:244-314).  The Hugging Face parent builds the whole
    model -- so parameter names, weight tying and initialisation are exactly Hugging Face's and stock checkpoints
    load with ``from_pretrained`` -- and the attention / encoder / model classes inside are then switched to the fused
    ones.  (The reference's own constructors call ``DebertaV2PreTrainedModel().__init__(config)`` on a fresh,
    argument-less instance and cannot be instantiated.)"""

    def __init__(self, config):
        super().__init__(config)
        patch_model(self)


class FlashDebertaV2ForMaskedLM(_FusedHead, DebertaV2ForMaskedLM):
    pass


class FlashDebertaV2ForSequenceClassification(_FusedHead, DebertaV2ForSequenceClassification):
    pass


class FlashDebertaV2ForTokenClassification(_FusedHead, DebertaV2ForTokenClassification):
    pass


class FlashDebertaV2ForQuestionAnswering(_FusedHead, DebertaV2ForQuestionAnswering):
    pass


class FlashDebertaV2ForMultipleChoice(_FusedHead, DebertaV2ForMultipleChoice):
    pass


def patch_model(model: nn.Module) -> nn.Module:
    """Switch every ``DisentangledSelfAttention`` inside ``model`` (any DeBERTa-v2/v3 model or task head,
    e.g. one loaded with ``from_pretrained``) to the fused kernel, in place.  Parameters are untouched."""
    swaps = {DisentangledSelfAttention: FlashDisentangledSelfAttention, DebertaV2Encoder: FlashDebertaV2Encoder,
             DebertaV2Model: FlashDebertaV2Model}        # none of them adds parameters or constructor state
    for module in model.modules():
        if type(module) in swaps:
            module.__class__ = swaps[type(module)]
    return model
