"""A pre-norm layer whose sublayers join the residual behind gates.

``n1 = norm1(x)``; ``x <- x + m * mixer(n1) * sigmoid(W_1 n1 + b_1)``; ``n2 = norm2(x)``;
``x <- x + m * feed_forward(n2) * sigmoid(W_2 n2 + b_2)``: each gate is projected from the very rows its sublayer
reads, and ``m`` is one residual multiplier for the model.  The gate's projection runs beside the sublayer; the
gating, the add into the float32 residual and the next norm are one kernel (the norm takes a ``Gated`` delta), so a
block takes the pending gated result of the block before it and hands on its own."""
from __future__ import annotations

from .base import Block, Gated, Part, TensorSpec


class ResidualGate(Part):
    """The gates of a layer.  params: width, mult (default 1), roles (the sublayers that have a gate; default mixer and
    feed_forward).  names: per role ``<role>`` ([width, width]) and ``<role>_bias`` ([width])."""
    graph_safe = True

    def _roles(self):
        return tuple(self.params.get("roles", ("mixer", "feed_forward")))

    def tensor_specs(self):
        d = self.params["width"]
        specs = {}
        for r in self._roles():
            specs[self.names[r]] = TensorSpec((d, d))
            specs[self.names[r + "_bias"]] = TensorSpec((d,))
        return specs

    def bind(self, tensors, rt):
        self.rt = rt
        self.mult = float(self.params.get("mult", 1.0))
        self.weights = {r: rt.weight(tensors[self.names[r]]) for r in self._roles()}
        self.biases = {r: tensors[self.names[r + "_bias"]].float().contiguous() for r in self._roles()}
        self.beside = set()       # the sublayers whose own weights hold their gate's: weights has a view of them

    def run_beside(self, role, sublayer):
        """The sublayer's first product takes the gate's where it can."""
        if role in self.weights and type(self).gated is ResidualGate.gated and hasattr(sublayer, "take_beside"):
            taken = sublayer.take_beside(self.weights[role])
            if taken is not None:
                self.weights[role] = taken
                self.beside.add(role)

    def _own(self):
        return [w.w for r, w in self.weights.items() if r not in self.beside]

    def step_bytes(self, rows):
        return sum(w.numel() * w.element_size() for w in self._own()) + sum(4 * b.numel() for b in self.biases.values())

    def step_flops(self, rows):
        return 2 * rows * sum(w.numel() for w in self._own())

    def gated(self, role, x, y, z=None):
        """The sublayer's result y (of the rows x it read) with its gate (z: its product where it is formed already), for the next
        norm's add."""
        return Gated(y, self.rt.linear(x, self.weights[role]) if z is None else z, self.biases[role], self.mult)


class _Gated(Block):
    """Where a sublayer can, its gate's projection is part of its own first product, or runs beside it."""

    def bound(self):
        for role in ("mixer", "feed_forward"):
            if role in self.roles and hasattr(self.gate, "run_beside"):
                self.gate.run_beside(role, self._parts[role])

    def run(self, role, x, *step):
        part = self._parts[role]
        if role in getattr(self.gate, "beside", ()):
            y, z = part.forward_beside(x, *step)
            return self.gate.gated(role, x, y, z)
        return self.gate.gated(role, x, part.forward(x, *step))


class GatedPreNormBlock(_Gated):
    roles = {"mixer_norm": "norm", "mixer": "mixer", "ffn_norm": "norm", "feed_forward": "feed_forward",
             "gate": "connection"}

    def forward(self, h, delta, step, view):
        x = self.mixer_norm.add_norm(h, delta)
        a = self.run("mixer", x, step, view)
        x = self.ffn_norm.add_norm(h, a)
        return self.run("feed_forward", x, step)


class GatedPreNormMixerBlock(_Gated):
    """The same without a feed-forward."""
    roles = {"mixer_norm": "norm", "mixer": "mixer", "gate": "connection"}

    def forward(self, h, delta, step, view):
        x = self.mixer_norm.add_norm(h, delta)
        return self.run("mixer", x, step, view)
