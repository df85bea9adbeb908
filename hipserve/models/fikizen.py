"""Fikizen: a pre-norm layer-list decoder (``config.FikizenConfig``) on the hipserve op set.

    x <- x + mixer(norm1(x));   x <- x + ff(norm2(x))   (the second only where the layer has a feed-forward)

with the mixer one of ``models/mixers.py``: windowed sink attention with a per-head output
gate, a gated delta rule, or sink attention and a generalized delta rule side by side. A
layer may use another layer's weights; every layer RUN still has a paged cache and / or
state tensors of its own. The logits pass ``cap * tanh(. / cap)``.

The residual stream lives in 32-bit floats for every dtype; each residual update and the
norm that follows it are one fused op (``scaled_add_group_rmsnorm`` with one group), or part
of the products around them where the step has few rows. Per engine step the model sees the flat token rows of all scheduled sequences (prompt portions
and single decode tokens alike); attention reads and writes the paged cache through the
step's block tables, the recurrences their sequences' state slots.
"""
from __future__ import annotations

import torch

from .layer_list import LayerListModel


class FikizenModel(LayerListModel):
    def __init__(self, *args, **kwargs):
        super().__init__(*args, **kwargs)
        for lw in self.layers:
            for m in (lw.mixer, lw.mlp) if lw is not None else ():
                if m is not None:
                    m.takes_parts = True   # of the residual update below

    # ---------------------------------------------------------------- forward
    def forward(self, ids: torch.Tensor, meta, kv_caches) -> torch.Tensor:
        ops, cfg = self.ops, self.cfg
        T, H = ids.shape[0], cfg.hidden_size
        state = meta.state
        if meta.id_src is not None:  # decode lookahead: row i's id is the previous step's sample tok[src[i]]
            src, tok = meta.id_src
            ids = torch.where(src >= 0, tok.index_select(0, src.clamp(min=0)), ids)
        residual = torch.empty(T, H, device=ids.device, dtype=torch.float32)
        h = torch.empty(T, H, device=ids.device, dtype=self.dtype)
        first = self.layers[self.runs[0][0]].norm1 if self.runs else self.final_norm
        # the first norm reads the embedding table itself
        ops.scaled_add_group_rmsnorm(h, residual, first, 1, cfg.norm_eps, table=self.embed, ids=ids.long().contiguous())
        # steps of a few rows: a sublayer's last product may take the update and the next norm with it (not the last: ``forward`` returns
        # a tensor)
        fused = self.capture is None
        for r, (i, _, _) in enumerate(self.runs):
            lw = self.layers[i]
            last = r + 1 == len(self.runs)
            nxt = self.final_norm if last else self.layers[self.runs[r + 1][0]].norm1
            after = nxt if lw.mlp is None else lw.norm2   # the norm after the mixer
            h = lw.mixer.forward(h, meta, kv_caches[r], state[r] if state is not None else None,
                                 (residual, after, cfg.norm_eps) if fused and not (last and lw.mlp is None) else None)
            if torch.is_tensor(h):
                h = ops.scaled_add_group_rmsnorm(torch.empty(T, H, device=ids.device, dtype=self.dtype), residual, after, 1, cfg.norm_eps, h)
            if lw.mlp is not None:
                h = lw.mlp.forward(h, (residual, nxt, cfg.norm_eps) if fused and not last else None)
                if torch.is_tensor(h):
                    h = ops.scaled_add_group_rmsnorm(torch.empty(T, H, device=ids.device, dtype=self.dtype), residual, nxt, 1, cfg.norm_eps, h)
            if self.capture is not None:
                self.capture.append(residual.clone())
        return h

    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        """32-bit logits = cap * tanh(head . hidden / cap)."""
        cap = self.cfg.logit_softcap
        return self.ops.linear(hidden, self.lm_head, out_f32=True, **({"act": "softcap", "c0": cap} if cap > 0 else {}))
