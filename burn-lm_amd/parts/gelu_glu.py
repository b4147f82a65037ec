"""Dense gated feed-forward with the tanh form of GELU: ``W_down (gelu_tanh(W_gate x) * (W_up x))`` without biases,
``gelu_tanh(z) = z/2 (1 + tanh(sqrt(2/pi) (z + 0.044715 z^3)))``.  Gate and up run as one product on the stacked
weight; the activation and the product are float32, in the epilogue of the hand-written products (few rows, and
prompts of the sizes the runtime gives to its tiled kernel) and in a kernel of their own behind the library's product."""
from __future__ import annotations

import torch

from .base import FeedForward, TensorSpec, forward_goes_beside


class GeluGLU(FeedForward):
    """params: width, inner.  names: gate, up, down."""
    graph_safe = True

    def tensor_specs(self):
        d, i = self.params["width"], self.params["inner"]
        return {self.names["gate"]: TensorSpec((i, d)), self.names["up"]: TensorSpec((i, d)),
                self.names["down"]: TensorSpec((d, i))}

    def bind(self, tensors, rt):
        self.rt = rt
        g, u = tensors[self.names["gate"]], tensors[self.names["up"]]
        if g.dtype != u.dtype:
            g, u = g.float(), u.float()
        self.w_gate_up, self.w_beside = rt.weight(torch.cat([g, u], dim=0), gated=True), None
        self.w_down = rt.weight(tensors[self.names["down"]])
        self.inner = self.params["inner"]

    def take_beside(self, weight):
        """The other weight as a view of what now holds its rows behind gate's and up's (forward_beside), or None."""
        own = self.w_gate_up
        if not forward_goes_beside(self) or own.dtype != weight.dtype or own.shape[1] != weight.shape[1] or weight.gated or weight.shape[0] % 8:
            return None
        self.stacked = torch.cat([own.w, weight.w], dim=0)        # each of the two is a stretch of it
        self.w_gate_up = self.rt.weight(self.stacked[:own.shape[0]], gated=True)
        self.w_beside = self.rt.weight(self.stacked[own.shape[0]:])
        return self.w_beside

    def _weights(self):
        return [w for w in (self.w_gate_up, self.w_down, self.w_beside) if w is not None]

    def step_bytes(self, rows):
        return sum(w.w.numel() * w.w.element_size() for w in self._weights())

    def step_flops(self, rows):
        return 2 * rows * sum(w.w.numel() for w in self._weights())

    def forward(self, x, step):
        rt = self.rt
        return rt.linear(rt.gated_linear(x, self.w_gate_up, activation="gelu_tanh"), self.w_down, partials=True)

    def forward_beside(self, x, step):
        """(forward's result, the other product's)."""
        act, z = self.rt.gated_linear_beside(x, self.w_gate_up, self.w_beside, self.stacked, "gelu_tanh")
        return self.rt.linear(act, self.w_down, partials=True), z
