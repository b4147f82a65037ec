"""Mixture of experts: ``experts`` small SwiGLU feed-forwards without biases, of which every token uses the ``top``
with the largest router logits ``W_router x + b``, weighted by the softmax over the chosen logits only; a shared
expert of the same form may run for every token, times ``sigmoid(W_sg x)`` (one number per token).

The router's logits, the choice and the weights are float32.  In steps of few rows all experts run as ONE stacked product:
their gate and up projections are the rows of one matrix, their down projections the columns of another, and every expert's
gated activations are multiplied by the token's weight for that expert (zero for experts it did not choose)
before the one down projection, which so adds the chosen experts' outputs up (up to 64 rows in the gate/up product's own
epilogue, ``ops.gemv_experts``).  That computes every expert for
every token, and reads the same weights as a batch that uses every expert.

In steps of many rows of experts without clamps and without a shared one, every token goes through its own experts only
(``ops.moe_grouped``; see ``_grouped`` for where): lists of every expert's tokens are made on the device, and the launches'
sizes come from the number of rows alone.  Either way a token's result does not depend on which tokens share its step
(beyond the number of rows), and no step shape depends on the routing, so steps replay from recorded graphs."""
from __future__ import annotations

import torch

from .base import FeedForward, TensorSpec, Term

# From how many rows on, and at how many times fewer products (tiles' padding counted, half a tile for each expert), every
# token runs through its own experts only.  Measured, us for the whole feed-forward behind the router, all experts / own ones
# (experts, chosen, inner, width): 16, 4, 512, 2048 at 256 rows 59.6 / 54.6, 512 rows 67.7 / 55.5, 2,048 rows 178 / 112, 8,192
# rows 612 / 336; 128, 8, 128, 1024 at 256 rows 50.7 / 68.6, 512 rows 75.6 / 73.0, 2,048 rows 226 / 99; 16, 2, 256, 2048 at 512
# rows 46.4 / 46.7, 2,048 rows 95 / 58.  With less than half the products saved nothing is won: 4, 2, 1024, 1024 (1.9 times
# fewer) at 4,096 rows 112.6 / 107.5, and a plane more for the next norm; 4, 3, 512, 1024 (1.3 times) 65.4 / 79.6.
GROUPED_MIN_ROWS = 512
GROUPED_MIN_GAIN = 2
GROUPED_TILE = 256
# The grouped form's planes and activations take top * (4 width + 2 inner) bytes a row, the stacked form's gates, ups and activations
# 6 * experts * inner: beyond this many bytes only where they are no more, so that no step needs more memory than the stacked form did.
GROUPED_FREE_BYTES = 1 << 30

class RoutedExperts(FeedForward):
    """params: width, experts, top, expert_inner, shared_inner (0: no shared expert).
    names: router, router_bias, e<i>.gate / e<i>.up / e<i>.down for every expert, and with a shared expert
    shared.gate, shared.up, shared.down, shared.sg."""
    graph_safe = True
    clamped = False

    def tensor_specs(self):
        p, n = self.params, self.names
        d, E, f, s = p["width"], p["experts"], p["expert_inner"], int(p.get("shared_inner", 0))
        specs = {n["router"]: TensorSpec((E, d)), n["router_bias"]: TensorSpec((E,))}
        for e in range(E):
            specs[n[f"e{e}.gate"]] = TensorSpec((f, d))
            specs[n[f"e{e}.up"]] = TensorSpec((f, d))
            specs[n[f"e{e}.down"]] = TensorSpec((d, f))
        if s:
            specs.update({n["shared.gate"]: TensorSpec((s, d)), n["shared.up"]: TensorSpec((s, d)),
                          n["shared.down"]: TensorSpec((d, s)), n["shared.sg"]: TensorSpec((1, d))})
        return specs

    def bind(self, tensors, rt):
        self.rt = rt
        p, n = self.params, self.names
        self.E, self.top, self.f, self.s = p["experts"], p["top"], p["expert_inner"], int(p.get("shared_inner", 0))
        if not 1 <= self.top <= self.E:
            raise ValueError(f"top = {self.top} of {self.E} experts")
        t = lambda name: tensors[n[name]]
        gates = [t(f"e{e}.gate") for e in range(self.E)] + ([t("shared.gate")] if self.s else [])
        ups = [t(f"e{e}.up") for e in range(self.E)] + ([t("shared.up")] if self.s else [])
        downs = [t(f"e{e}.down") for e in range(self.E)] + ([t("shared.down")] if self.s else [])
        ws = gates + ups + downs
        if len({w.dtype for w in ws}) != 1:
            gates, ups, downs = ([w.float() for w in group] for group in (gates, ups, downs))
        self.inner = self.E * self.f + self.s
        self.w_gate_up = self._stacked(gates, ups)
        self.w_down = rt.weight(torch.cat(downs, dim=1).contiguous())
        router = [t("router")] + ([t("shared.sg")] if self.s else [])
        if len({w.dtype for w in router}) != 1:
            router = [w.float() for w in router]
        rows = sum(w.shape[0] for w in router)
        pad = (-rows) % 16
        if pad:
            router.append(torch.zeros(pad, router[0].shape[1], dtype=router[0].dtype, device=router[0].device))
        self.w_router = rt.weight(torch.cat(router, dim=0))
        self.router_bias = t("router_bias").float().contiguous()

    def _stacked(self, gates, ups):
        """All experts' gates and ups as one matrix.  In pairs where the product of few rows takes the gating and the experts' weights into
        its epilogue (eight neighbouring pairs belong to one expert there)."""
        w = torch.cat(gates + ups, dim=0)
        pairs = self.rt.dtype == w.dtype == torch.bfloat16 and not self.clamped and self.f % 8 == 0 and self.s % 8 == 0
        return self.rt.weight(w, gated=pairs)

    def step_bytes(self, rows):
        return sum(w.w.numel() * w.w.element_size() for w in (self.w_gate_up, self.w_down, self.w_router))

    def step_flops(self, rows):
        return self._expert_flops(rows) + 2 * rows * self.w_router.w.numel()

    def _expert_flops(self, rows):
        flops = 2 * rows * (self.w_gate_up.w.numel() + self.w_down.w.numel())
        return flops * self.top // self.E if self._grouped(rows) else flops

    def route(self, x):
        """float32 [tokens, experts + 1]: every expert's weight for every token (zero if not chosen), and the shared
        expert's gate."""
        rt = self.rt
        logits = rt.linear(x, self.w_router, out_dtype=torch.float32)
        weights = torch.empty(x.shape[0], self.E + 1, dtype=torch.float32, device=x.device)
        return rt.ops.moe_route(logits, self.router_bias, self.E, self.top, self.E if self.s else -1, weights)

    def _mix(self, x, weights, step):
        """The experts' results for [tokens, width] by the weights of `route`, without clamps."""
        rt, ops = self.rt, self.rt.ops
        if self._runs_grouped(x, step):
            return ops.moe_grouped(x, self.w_gate_up.w, self.w_down.w, weights, self.E, self.top)
        if rt.experts_take(x, self.w_gate_up):
            act = torch.empty(x.shape[0], self.inner, dtype=x.dtype, device=x.device)
            return rt.linear(ops.gemv_experts(x, self.w_gate_up.packed, act, self.E, self.f, weights=weights), self.w_down, partials=True)
        gu = rt.linear(x, self.w_gate_up)
        act = torch.empty(x.shape[0], self.inner, dtype=gu.dtype, device=x.device)
        return rt.linear(ops.moe_gate(gu, weights, act, self.E, self.f), self.w_down, partials=True)

    def _runs_grouped(self, x, step):
        bucket = getattr(step, "bucket", None)
        return self._grouped(bucket[0] if bucket else x.shape[0]) and x.is_contiguous() and x.data_ptr() % 16 == 0

    def _grouped(self, T):
        """Whether in a step of T rows (of a recorded shape: the bucket's) every token goes through its own experts only (rather than all through all)."""
        ops, gu, down = self.rt.ops, self.w_gate_up.w, self.w_down.w
        D = gu.shape[1]
        return (self.rt.dtype == gu.dtype == down.dtype == torch.bfloat16 and self.s == 0 and not self.clamped and T >= GROUPED_MIN_ROWS
                and self.f % ops.MOE_GROUPED_STEP == 0 and D % ops.MOE_GROUPED_STEP == 0
                and self.E <= ops.MOE_GROUPED_EXPERTS and self.top <= ops.MOE_GROUPED_TOP and self.top <= self.E
                and max(gu.numel(), T * D, T * self.top) < 2 ** 30
                and T * self.top * (4 * D + 2 * self.f) <= max(GROUPED_FREE_BYTES, 6 * T * self.E * self.f)
                and T * self.E >= GROUPED_MIN_GAIN * (T * self.top + GROUPED_TILE // 2 * self.E))

    def forward(self, x, step):
        return self._mix(x, self.route(x), step)


class GroupedRoutedExperts(RoutedExperts):
    """The same experts behind another router: the scores are the softmax of ``W_router x`` over all experts;
    the choice goes by ``score + correction`` (a stored vector), only among the experts of the ``keep`` best of
    ``groups`` equal groups of neighbouring experts (a group ranks by its largest corrected score); the ``top`` chosen
    experts' weights are their scores (without the correction) over the sum of the chosen scores.  The last
    ``identity`` of the router's outputs belong to experts without tensors that hand their input on unchanged; they
    count like the others in softmax, groups and choice, and their share of the result is ``weight * x``.

    Variants by parameter: scores that are each expert's own sigmoid (``score="sigmoid"``); weights that are the chosen
    scores as they are (``renormalize=False``); clamped experts (``form="clamped"``) whose weight is on their input: an
    expert reads ``w x``, ``g = min(W_gate (w x), limit)``, ``u = clamp(W_up (w x), -limit, limit)`` and gives
    ``W_down (g sigmoid(alpha g) (u + 1))``; with them a shared expert of the same form, with a limit of its own, that runs
    for every token unweighted.  The share on the input goes through the stacked product as a factor on its results.

    params: width, experts (those with tensors), identity (default 0), top, groups (default 1), keep (default 1),
    expert_inner, correction (whether the checkpoint has one; default True), score ("softmax", the default, or "sigmoid"),
    renormalize (default True), form ("silu", the default, or "clamped"; then limit, alpha (default 1.702), shared_inner
    (default 0: no shared expert), shared_limit).
    names: router [experts + identity, width], correction [experts + identity], e<i>.gate / e<i>.up / e<i>.down, and with a
    shared expert shared.gate / shared.up / shared.down."""

    def _counts(self):
        p = self.params
        E, I = int(p["experts"]), int(p.get("identity", 0))
        groups, keep = int(p.get("groups", 1)), int(p.get("keep", 1))
        if E < 1 or I < 0 or groups < 1 or (E + I) % groups or not 1 <= keep <= groups:
            raise ValueError(f"grouped experts: {E} + {I} experts do not form {groups} equal groups of which {keep} stay")
        if not 1 <= p["top"] <= keep * ((E + I) // groups):
            raise ValueError(f"grouped experts: top = {p['top']} is more than {keep} groups of {(E + I) // groups} hold")
        form = p.get("form", "silu")
        if form not in ("silu", "clamped") or (form == "silu" and p.get("shared_inner")):
            raise ValueError(f"grouped experts: form {form!r} unknown (silu, clamped), or a shared expert that is not clamped")
        return E, I, groups, keep

    def tensor_specs(self):
        p, n = self.params, self.names
        d, f = p["width"], p["expert_inner"]
        E, I, _, _ = self._counts()
        specs = {n["router"]: TensorSpec((E + I, d))}
        if p.get("correction", True):
            specs[n["correction"]] = TensorSpec((E + I,))
        for e in range(E):
            specs[n[f"e{e}.gate"]] = TensorSpec((f, d))
            specs[n[f"e{e}.up"]] = TensorSpec((f, d))
            specs[n[f"e{e}.down"]] = TensorSpec((d, f))
        s = int(p.get("shared_inner", 0))
        if s:
            specs.update({n["shared.gate"]: TensorSpec((s, d)), n["shared.up"]: TensorSpec((s, d)), n["shared.down"]: TensorSpec((d, s))})
        return specs

    def bind(self, tensors, rt):
        self.rt = rt
        p, n = self.params, self.names
        self.E, self.I, self.groups, self.keep = self._counts()
        self.top, self.f, self.s = int(p["top"]), p["expert_inner"], int(p.get("shared_inner", 0))
        self.score, self.renormalize = p.get("score", "softmax"), bool(p.get("renormalize", True))
        self.clamped = p.get("form", "silu") == "clamped"
        if self.clamped:
            self.limit, self.alpha = float(p["limit"]), float(p.get("alpha", 1.702))
            self.shared_limit = float(p["shared_limit"]) if self.s else None
        t = lambda name: tensors[n[name]]
        blocks = [f"e{e}." for e in range(self.E)] + (["shared."] if self.s else [])
        gates, ups, downs = ([t(b + r) for b in blocks] for r in ("gate", "up", "down"))
        if len({w.dtype for w in gates + ups + downs}) != 1:
            gates, ups, downs = ([w.float() for w in group] for group in (gates, ups, downs))
        self.inner = self.E * self.f + self.s
        self.w_gate_up = self._stacked(gates, ups)
        self.w_down = rt.weight(torch.cat(downs, dim=1).contiguous())
        router = t("router")
        pad = (-router.shape[0]) % 16
        if pad:
            router = torch.cat([router, torch.zeros(pad, router.shape[1], dtype=router.dtype, device=router.device)], dim=0)
        self.w_router = rt.weight(router.contiguous())
        self.correction = t("correction").float().contiguous() if p.get("correction", True) else None

    def route(self, x):
        """float32 [tokens, experts + 1]: every expert's weight for every token (zero if not chosen), and behind them
        the weight of the token's pass-through experts together."""
        rt = self.rt
        logits = rt.linear(x, self.w_router, out_dtype=torch.float32)
        weights = torch.empty(x.shape[0], self.E + 1, dtype=torch.float32, device=x.device)
        return rt.ops.moe_route_grouped(logits, self.correction, self.E, self.I, self.groups, self.keep, self.top, weights,
                                        score=self.score, renormalize=self.renormalize)

    def forward_terms(self, x, step):
        rt = self.rt
        weights = self.route(x)
        if self.clamped:
            gu = rt.linear(x, self.w_gate_up)
            act = torch.empty(x.shape[0], self.inner, dtype=gu.dtype, device=x.device)
            rt.ops.moe_gate_clamped(gu, weights, act, self.E, self.f, self.limit, self.alpha, self.shared_limit)
            terms = [Term(rt.linear(act, self.w_down, partials=True))]
        else:
            terms = [Term(self._mix(x, weights, step))]
        if self.I:
            terms.append(Term(x, 1.0, weights[:, self.E]))
        return terms

    def forward(self, x, step):
        terms = self.forward_terms(x, step)
        if len(terms) == 1:
            return terms[0].y
        out = torch.zeros(1, x.shape[0], x.shape[1], dtype=torch.float32, device=x.device)
        self.rt.ops.scaled_add(out[0], [(t.y, None, t.row) for t in terms])
        return out


class TableExperts(RoutedExperts):
    """The same experts without a router: a stored table ``[vocab, top]`` names every token id's experts (the
    entries of a row differ), each with the weight ``1 / top``.  The step's token ids are read on the device, also those
    that a decode step's host has not seen yet.

    params: width, vocab, experts, top, expert_inner.  names: table, e<i>.gate / e<i>.up / e<i>.down."""

    def tensor_specs(self):
        p, n = self.params, self.names
        d, f = p["width"], p["expert_inner"]
        specs = {n["table"]: TensorSpec((p["vocab"], p["top"]), "int")}
        for e in range(p["experts"]):
            specs[n[f"e{e}.gate"]] = TensorSpec((f, d))
            specs[n[f"e{e}.up"]] = TensorSpec((f, d))
            specs[n[f"e{e}.down"]] = TensorSpec((d, f))
        return specs

    def bind(self, tensors, rt):
        self.rt = rt
        p, n = self.params, self.names
        self.E, self.top, self.f, self.s = p["experts"], p["top"], p["expert_inner"], 0
        if not 1 <= self.top <= self.E:
            raise ValueError(f"top = {self.top} of {self.E} experts")
        self.table = tensors[n["table"]].contiguous()
        if int(self.table.min()) < 0 or int(self.table.max()) >= self.E:
            raise ValueError(f"the table {n['table']} names experts outside 0 .. {self.E - 1}")
        gates, ups, downs = ([tensors[n[f"e{e}.{r}"]] for e in range(self.E)] for r in ("gate", "up", "down"))
        if len({w.dtype for w in gates + ups + downs}) != 1:
            gates, ups, downs = ([w.float() for w in group] for group in (gates, ups, downs))
        self.inner = self.E * self.f
        self.w_gate_up = self._stacked(gates, ups)
        self.w_down = rt.weight(torch.cat(downs, dim=1).contiguous())

    def step_bytes(self, rows):
        return sum(w.w.numel() * w.w.element_size() for w in (self.w_gate_up, self.w_down)) + 4 * self.top * rows

    def step_flops(self, rows):
        return self._expert_flops(rows)

    def _by_table(self, x):
        """Whether the product of the gates and ups looks the experts up itself."""
        ops = self.rt.ops
        return x.shape[0] <= ops.EXPERT_TABLE_ROWS and self.top <= ops.EXPERT_TABLE_TOP and self.rt.experts_take(x, self.w_gate_up)

    def forward(self, x, step):
        rt = self.rt
        if self._by_table(x):
            act = torch.empty(x.shape[0], self.inner, dtype=x.dtype, device=x.device)
            rt.ops.gemv_experts(x, self.w_gate_up.packed, act, self.E, self.f, table=self.table, ids=step.token_ids, token_source=step.token_source)
            return rt.linear(act, self.w_down, partials=True)
        if self._runs_grouped(x, step):
            return rt.ops.moe_grouped(x, self.w_gate_up.w, self.w_down.w, None, self.E, self.top, table=self.table, ids=step.token_ids,
                                      token_source=step.token_source)
        weights = torch.empty(x.shape[0], self.E + 1, dtype=torch.float32, device=x.device)
        rt.ops.moe_table(self.table, step.token_ids, weights, self.E, step.token_source)
        return self._mix(x, weights, step)
