"""Kanotar: a decoder-only LM of latent-attention layers.

Every layer has its own sizes, sliding window and feed-forward; a layer
may read an earlier layer's cached latents instead of having its own.
There are no positions in the attention. Each sublayer is normed on both
sides (x += norm(f(norm(x)))) and the residual stream is fp32, so the
step is a chain of products joined by one fused norm-add-norm launch per
sublayer.
"""

from __future__ import annotations

import torch
from torch.nn.modules import module

from .. import ops
from .blocks import ClampedGlu, LatentAttention
from .layered import LayeredCache, LayeredModel


_LINEAR = ops.linear


def _shared(part) -> dict:
    """Arguments with which a sublayer leaves the sum over shares of K to the
    norm behind it; none where a hook sees its output, it has other forms, or
    ops.linear has been replaced and is to see every product."""
    return ({"linear": ops.linear_parts}
            if type(part) in (ClampedGlu, LatentAttention)
            and "forward" not in part.__dict__ and ops.linear is _LINEAR
            and not (part._forward_hooks or module._global_forward_hooks)
            else {})


def _forms(part) -> dict:
    """The forms of a sublayer's products that a norm follows: _shared, and where
    a hook sees the output the same sums, joined, so that watching changes no
    result. Nothing sees the product that a mixer's own norms follow."""
    forms = _shared(part)
    if (not forms and type(part) in (ClampedGlu, LatentAttention)
            and "forward" not in part.__dict__ and ops.linear is _LINEAR):
        forms = {"linear": ops.linear_joined}
    if forms and type(part) is LatentAttention:
        forms["down"] = ops.linear_parts
    return forms


class KanotarModel(LayeredModel):
    layer_norms = ("norm1", "norm1b")
    mlp_norms = ("norm2", "norm2b")

    @torch.no_grad()
    def forward_step(self, batch, cache: LayeredCache,
                     trace: list | None = None) -> torch.Tensor:
        W, eps = self.dims.hidden_size, self.dims.norm_eps
        h, x = ops.embed_norm(batch.tokens, self.tok_emb,
                              self.layers[0].norm1, W, eps)
        for i, layer in enumerate(self.layers):
            after = (self.layers[i + 1].norm1 if i + 1 < len(self.layers)
                     else self.final_norm)
            y = layer.mixer(h, batch, cache.layers[i],
                            **_forms(layer.mixer))
            if layer.mlp is None:
                h = ops.post_norm_add(y, x, layer.norm1b, after, W, eps)
            else:
                h = ops.post_norm_add(y, x, layer.norm1b, layer.norm2, W,
                                      eps)
                h = ops.post_norm_add(layer.mlp(h, **_forms(layer.mlp)), x,
                                      layer.norm2b, after, W, eps)
            if trace is not None:
                trace.append(x[:, :W].clone())
        return h
