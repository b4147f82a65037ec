"""Arrangements of a layer's parts.

``pre_norm``: ``h = x + mixer(norm1(x)); y = h + ffn(norm2(h))``
(crates/burn-lm-llama/src/nn/transformer.rs:241-256).  Each add happens inside the next norm's
kernel on the float32 residual stream, so a block takes the pending ``delta`` of the block
before it and hands on its own.

In steps of few tokens the norm has no kernel of its own either, where its neighbours can do its work: the last product of the
sublayer in front of it adds itself to the residual and leaves ``h * gamma`` with the rows' sums of squares, and the first product
behind it scales its own sums (``Product``, ``Unscaled``)."""
from __future__ import annotations

from .base import Block, Product, speaks_for


class Seam:
    """A sublayer, the norm behind it and the sublayer behind that, where the norm's work can be done by the products of the two: the
    parts speak for what they would do apart (a part from outside that brings its own forward or norm is called by that, also one that
    came or was patched after the model was bound)."""

    def __init__(self, front, norm, back):
        self.front, self.norm, self.back = front, norm, back

    @classmethod
    def between(cls, front, norm, back):
        seam = cls(front, norm, back)
        return seam if seam.stands(front, norm, back) else None

    def stands(self, front, norm, back):
        """Whether these parts are the seam's, and still speak for themselves."""
        return (front is self.front and norm is self.norm and back is self.back
                and speaks_for(front, "forward_product", "forward", "output", "forward_after_norm") and speaks_for(norm, "joining", "add_norm")
                and speaks_for(back, "takes_unscaled", "forward", "forward_after_norm", "project", "forward_product")
                and hasattr(front, "rt") and hasattr(front.rt, "join_takes")
                and (not hasattr(type(front.rt), "linear") or speaks_for(front.rt, "join", "linear", "gated_linear")))

    def takes(self, step):
        # a step that will be recorded chooses by its recording's size, like every form of a result
        tokens = max(step.n_tokens, (getattr(step, "bucket", None) or (0,))[0])
        return self.front.rt.join_takes(tokens, self.front.last_weight()) and self.back.takes_unscaled(tokens)

    def run(self, h, product):
        rt = self.front.rt
        if not rt.join_reads(product.x, product.w):       # rows from outside, in a form that only the plain products take
            return self.norm.add_norm(h, rt.linear(product.x, product.w, partials=True))
        return rt.join(product, h, *self.norm.joining())


class PreNormBlock(Block):
    roles = {"mixer_norm": "norm", "mixer": "mixer", "ffn_norm": "norm", "feed_forward": "feed_forward"}
    inside = None          # the Seam between mixer and feed-forward

    def bound(self):
        self.inside = Seam.between(self.mixer, self.ffn_norm, self.feed_forward)

    def parts_to(self, after):
        """The last part of this block, and the norm and the part that the block behind it begins with; None where one of the two
        blocks is written otherwise."""
        blocks = all(isinstance(b, PreNormBlock) and speaks_for(b, "forward_to", "forward") for b in (self, after))
        return (self.feed_forward, after.mixer_norm, after.mixer) if blocks else None

    def seam_to(self, after):
        """The Seam between this block and the one behind it, or None."""
        parts = self.parts_to(after)
        return None if parts is None else Seam.between(*parts)

    def forward(self, h, delta, step, view):
        return self.forward_to(h, delta, step, view, None, None)

    def forward_to(self, h, delta, step, view, before, after):
        """forward between two seams: a delta that is a Product is run with the seam before, and the result comes as a Product
        for the seam after, which holds in this step (or is None)."""
        x = before.run(h, delta) if isinstance(delta, Product) else self.mixer_norm.add_norm(h, delta)
        if self.inside is not None and self.inside.takes(step) and self.inside.stands(self.mixer, self.ffn_norm, self.feed_forward):
            x = self.inside.run(h, self.mixer.forward_product(x, step, view))
        else:
            a = self.mixer.forward(x, step, view)
            if after is None:
                return self.feed_forward.forward_after_norm(h, a, self.ffn_norm, step)
            x = self.ffn_norm.add_norm(h, a)
        return self.feed_forward.forward(x, step) if after is None else self.feed_forward.forward_product(x, step)
