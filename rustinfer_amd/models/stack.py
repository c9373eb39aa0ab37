"""A decoding step of a whole Llama stack as one launch (csrc/decode_stack.hip).

A model whose layers are all the same plain kind (pre-norm, grouped attention over all earlier keys with a rotation over
whole heads, SwiGLU), in bfloat16 with second copies of all its weights in tile order, is described once, when it is
loaded, by a table of its weights on the device; a step of up to eight rows of one token each, all of whose logits are
wanted, then runs as that one kernel.  Every other step, and every other model, goes part by part.
"""
from __future__ import annotations

import struct
from typing import Optional

import torch

from ..parts.attention import PagedAttention
from ..parts.block import PreNormBlock
from ..parts.embed import Embedding, LMHead
from ..parts.mlp import SwiGLUMLP
from ..parts.norm import RMSNorm
from ..parts.rope import RotaryEmbedding


class DecodeStack:
    def __init__(self, model, rt):
        """For a model that ``describes`` allows."""
        # (no reference to the model, which holds this: an engine that is let go is freed at once)
        self.rt, self.layers, self.hidden_size, self.vocab_size = rt, len(model.schedule), model.hidden_size, model.vocab_size
        self.embedding = model.embed.weight
        blocks = [model.layers[c.layer] for c in model.schedule]
        first = blocks[0]
        self.H, self.Hkv, self.hd = first.mixer.num_heads, first.mixer.num_kv_heads, first.mixer.head_dim
        self.ff, self.scale, self.rope = first.ffn.intermediate_size, first.mixer.scale, first.mixer.pos_enc
        weights = [w for b in blocks for w in (b.mixer.qkv_fused, b.mixer.o.weight_tiled, b.ffn.gate_up.weight_tiled, b.ffn.down.weight_tiled)]
        norms = [n for b in blocks for n in (b.mixer_norm, b.ffn_norm)] + [model.final_norm]
        weights.append(model.lm_head.weight_tiled)
        addresses = [t.data_ptr() for t in weights + [n.weight for n in norms]]
        table = struct.pack(f"<{len(addresses)}Q{len(norms)}d", *addresses, *(n.eps for n in norms))
        self.table = torch.frombuffer(bytearray(table), dtype=torch.int64).to(rt.device)
        self._held = weights + [n.weight for n in norms]       # (the table holds addresses: the tensors stay as long as it does)
        self._taken = rt.weights_taken                         # (and are the parts' own as long as none of them takes another)
        self.norm_dtype = model.final_norm.weight.dtype
        self.scratch_bytes = rt.ops.decode_stack_scratch(len(blocks), model.hidden_size, self.ff, self.H, self.Hkv, self.hd)

    @staticmethod
    def describes(model, rt) -> bool:
        """Whether every layer, the embedding, the head and the run order are of the one kind the kernel knows."""
        if rt.dtype != torch.bfloat16 or not hasattr(rt.ops, "decode_stack") or not model.schedule or model.stream_parts:
            return False
        if any(c.layer != i or c.cache != i or not c.write or c.enter is not None for i, c in enumerate(model.schedule)) \
                or len(model.schedule) != len(model.layers):
            return False
        e, head, norms = model.embed, model.lm_head, [model.final_norm]
        if type(e) is not Embedding or e.norm is not None or e.scale != 1.0 or e.weight.dtype != torch.bfloat16 or not e.weight.is_contiguous():
            return False
        if type(head) is not LMHead or head.logit_scale != 1.0 or head.softcap > 0.0 or head.weight_tiled is None:
            return False
        first = model.layers[0]
        for b in model.layers:
            if type(b) is not PreNormBlock or type(b.mixer) is not PagedAttention or type(b.ffn) is not SwiGLUMLP or b.mixer_shift is not None:
                return False
            m, f, m0 = b.mixer, b.ffn, getattr(first, "mixer", None)
            if m.window or not m.own_kv or m.qk_transform is not None or m.qkv_fused is None or f.delta_dtype is not None \
                    or any(w is None for w in (m.o.weight_tiled, f.gate_up.weight_tiled, f.down.weight_tiled)):
                return False
            if (m.num_heads, m.num_kv_heads, m.head_dim, m.scale, f.intermediate_size) != \
                    (m0.num_heads, m0.num_kv_heads, m0.head_dim, m0.scale, first.ffn.intermediate_size) or m.pos_enc is not m0.pos_enc:
                return False
            norms += [b.mixer_norm, b.ffn_norm]
        if any(type(n) is not RMSNorm or not n.plain_rms or n.weight.dtype != model.final_norm.weight.dtype or not n.weight.is_contiguous()
               or n.weight.dtype not in (torch.float32, torch.bfloat16) for n in norms):
            return False
        rope = first.mixer.pos_enc
        if type(rope) is not RotaryEmbedding or rope.rot_dim != first.mixer.head_dim or any(type(p) is not RotaryEmbedding for p in model.position_encodings):
            return False
        return rt.ops.decode_stack_takes(1, model.hidden_size, first.ffn.intermediate_size, first.mixer.num_heads, first.mixer.num_kv_heads,
                                         first.mixer.head_dim, 16, model.vocab_size)

    def takes(self, ctx, caches) -> bool:
        """Whether the weights are those that were loaded, and the step is of single tokens, all wanted, over one group of caches that holds a layer's after the other, not so many keys that the
        parts are faster, and there is a control block for it."""
        T = ctx.num_tokens
        if self.rt.weights_taken != self._taken:
            return False
        if ctx.max_q_len != 1 or ctx.num_want != T or not getattr(ctx, "want_all_in_order", False) or ctx.num_rows < T:
            return False
        groups = getattr(caches, "groups", None)
        if not groups or len(groups) != 1 or len(groups[0].cache_ids) != self.layers:
            return False
        ops = self.rt.ops
        if not ops.decode_stack_pays(T, self.hd, ctx.max_kv_len):
            return False
        return ops.decode_stack_takes(T, self.hidden_size, self.ff, self.H, self.Hkv, self.hd, groups[0].page_size, self.vocab_size) \
            and ops.decode_stack_control(ctx.workspace) is not None

    def forward(self, ctx, caches) -> torch.Tensor:
        g = caches.groups[0]
        logits = ctx.workspace.get("model.logits", ctx.num_tokens, self.vocab_size, torch.float32)
        scratch = ctx.workspace.get("model.stack", self.scratch_bytes // 256, 256, torch.uint8)
        cos, sin, _ = self.rope.rotary()
        self.rt.ops.decode_stack(self.table, self.layers, ctx, self.embedding, self.ff, self.H, self.Hkv, self.hd, cos, sin, g.k_pool, g.v_pool,
                                 ctx.block_tables[g.index], g.page_size, self.scale, self.norm_dtype, scratch, logits)
        return logits


def decode_stack(model, rt) -> Optional[DecodeStack]:
    """The description of ``model`` for the one-launch step, or None."""
    return DecodeStack(model, rt) if DecodeStack.describes(model, rt) else None
