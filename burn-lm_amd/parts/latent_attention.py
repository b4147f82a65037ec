"""Attention whose keys and values are expanded from one low-rank latent per token (latent attention).

``q = W_q x`` per head as ``[dim plain lanes | rot_dim lanes turned by position]``; ``W_dkv x`` gives the latent
``c`` (kv_rank lanes, RMS-normed with a weight) and one turned key part shared by all heads (rot_dim lanes).
A head's plain key is ``W_uk c`` and its value ``W_uv c``; score = (q_plain . k_plain + q_rot . k_rot) * scale,
causal softmax, output projection over the concatenated heads.  Only ``[c | k_rot]`` is cached: the scores are
computed as ``(W_uk^T q_plain) . c`` and the values applied as ``W_uv (sum_j p_j c_j)``, which is the same
function, so the cache holds one row of kv_rank + rot_dim lanes per token for all heads and no value pages.  Longer
prompts in bfloat16 expand the keys and values of the rows they see instead (see ``expands``).
Rotation: lane i of the first ``rot_dims`` turned lanes pairs with lane i + rot_dims/2 (``pairing="half"``, the
default), or lane 2i with lane 2i + 1 (``pairing="adjacent"``).

Variants by parameter: queries through a latent of their own (``q_rank``): ``c_q = rmsnorm(W_dq x)`` with a stored
weight, ``q = W_uq c_q``; a layer that borrows (``borrows=True``) has no ``W_dkv``: it reads the rows
``[c | k_rot]`` that an earlier layer keeps, as cached, and expands them with its own ``W_uk`` and ``W_uv``; a sliding
window (``window``: position i sees j while ``0 <= i - j < window``); a softmax sink (``sink``: the denominator also holds
``exp(sink_h)``, a learned logit per head, not scaled, without row or value); an output gate (``gate``: the concatenated
heads are multiplied element by element by ``sigmoid(W_g x)`` of the mixer's own input, whose rows run with the other
projections of that input)."""
from __future__ import annotations

import os

import torch

from .base import KVNeed, Mixer, TensorSpec

DECODE_BLOCKS_PER_UNIT = 2     # blocks of four (token, head) wavefronts the split decode aims for per compute unit
# Prompts expand keys and values from this many new tokens per sequence on (us of the whole mixer at width 2048, R = 512, 16
# heads of 128 + 64 / 128, absorbed / expanded: 32 tokens 92 / 70, behind 1,000 others 357 / 73; 64: 79 / 68; 512: 238 / 89; 2,048:
# 735 / 151 with a window of 1,024, 971 / 155 without; four sequences of 128: 132 / 85), while the rows that the page tables can
# name are at most so many, or so many times the step's tokens (the workspaces hold a key and a value per head for each: 8 KB a
# row at 16 heads of 128 lanes).
EXPAND_MIN_NEW = 32
EXPAND_MAX_ROWS = (16384, 4)
# For a shape that is recorded the bucket's sizes count, against half as many tokens and twice as many rows: sequences and
# pages are rounded up there, each by less than two times and to powers of two, so every step within the plain bounds stays
# within these (us of a whole step of two such mixers, absorbed / expanded: 16 sequences of 16 new tokens behind 1,000 others 2,466
# / 1,251, 4 of 2 behind 1,000 1,271 / 756, 5 of 20 behind 3,500 1,666 / 1,040, one of 64 behind 20,000 2,516 / 1,896).
EXPAND_BUCKET_SLACK = 2
EXPAND_MAX_BLOCKS = 65535      # sequences, and pages of one: the launch has a block row for each
MFMA_MAX_PIECES = 64           # most pieces the matrix-core decode cuts a sequence's half pages into



def most_pieces(tiles, rank, compute_units):
    """Into how many pieces the half pages of a decode step's tiles of 16 (token, head) pairs are cut at most.  A block of four wavefronts waits
    out a half page's trip from memory with nothing else to do, so short pieces are what shortens the step: up to a block for every unit of
    the chip, and from a block for every fourth unit on up to four pieces (16 heads, 512 + 64 lanes, us: 8 sequences of 1,125 tokens 32
    pieces 16.5, all 36 half pages 19.0; 16 of 600 tokens, 16 / 19 pieces 17.3 / 19.3; 64 of 600, 4 / 8 / 15 pieces 33.2 / 37.2 / 42.3; 128
    of 600, 2 / 4 / 7 pieces 58.7 / 53.6 / 59.6).  Of narrow latents, whose half pages are few loads, four blocks for every unit (8 heads, 128 +
    64 lanes, 24 sequences of 2,500 tokens 10 / 42 pieces 22.1 / 17.9, a wavefront to a piece before 18.4; 40 of 6,000 tokens 6 / 25 68.4 /
    41.0, 45.9; 64 of 1,125 4 / 16 24.9 / 20.8, 23.1; 4 heads, 64 + 32 lanes, 40 of 2,500 tokens 6 / 25 23.3 / 16.3, 17.4).  Wide ones
    of long sequences would take twice as many as they are given (256 + 64 lanes, 40 of 2,500 tokens 6 / 12 / 25 46.0 / 36.1 / 39.1, before 51.7)."""
    most = 4 * compute_units // tiles
    return min(MFMA_MAX_PIECES, most if rank < 256 else max(compute_units // tiles, min(4, most)))


class LatentAttention(Mixer):
    """params: width, heads, dim, rot_dim, vdim, kv_rank, scale, rot_dims, eps, position (the rotary table's
    owner, given by the model builder), pairing ("half", the default, or "adjacent"), q_rank (0, the default: queries
    projected directly; else the size of the queries' latent), borrows (default False), window (default 0: every earlier
    row), cache_window (what the cache keeps: the largest window of this layer and of those that borrow from it; default
    window), sink and gate (whether the layer has them; default False).
    names: q (or dq, dq_norm, uq with a query latent), uk, uv, o, unless the layer borrows dkv, dkv_norm, and sink, g
    where it has them."""
    graph_safe = True

    def tensor_specs(self):
        p, n = self.params, self.names
        d, H, dn, dr, dv, R = p["width"], p["heads"], p["dim"], p["rot_dim"], p["vdim"], p["kv_rank"]
        specs = {n["uk"]: TensorSpec((H * dn, R)), n["uv"]: TensorSpec((H * dv, R)), n["o"]: TensorSpec((d, H * dv))}
        qr = int(p.get("q_rank", 0))
        if qr:
            specs.update({n["dq"]: TensorSpec((qr, d)), n["dq_norm"]: TensorSpec((qr,)),
                          n["uq"]: TensorSpec((H * (dn + dr), qr))})
        else:
            specs[n["q"]] = TensorSpec((H * (dn + dr), d))
        if not p.get("borrows"):
            specs.update({n["dkv"]: TensorSpec((R + dr, d)), n["dkv_norm"]: TensorSpec((R,))})
        if p.get("sink"):
            specs[n["sink"]] = TensorSpec((H,))
        if p.get("gate"):
            specs[n["g"]] = TensorSpec((H * dv, d))
        return specs

    def cache_need(self):
        """One row [latent | turned key part] per token for all heads.  Where the matrix-core attention runs
        (bfloat16, sizes it is built for) the latent is kept a second time, transposed, as the value pages."""
        p = self.params
        window = int(p.get("cache_window", p.get("window", 0)))
        if getattr(self, "use_mfma", False):
            return KVNeed(1, p["kv_rank"] + p["rot_dim"], window, value_dim=p["kv_rank"])
        return KVNeed(1, p["kv_rank"] + p["rot_dim"], window, no_values=True)

    def bind(self, tensors, rt):
        self.rt = rt
        p, n = self.params, self.names
        self.H, self.dn, self.dr, self.dv, self.R = p["heads"], p["dim"], p["rot_dim"], p["vdim"], p["kv_rank"]
        self.scale, self.eps, self.rot = float(p["scale"]), float(p["eps"]), int(p["rot_dims"])
        if self.rot % 2 or not 0 <= self.rot <= self.dr:
            raise ValueError(f"{self.rot} turning lanes do not fit a turned part of {self.dr} lanes")
        self.position = p["position"]
        pairing = p.get("pairing", "half")
        if pairing not in ("half", "adjacent"):
            raise ValueError(f"latent attention: pairing={pairing!r} unknown (half, adjacent)")
        self.adjacent, self.borrows, self.q_rank = pairing == "adjacent", bool(p.get("borrows")), int(p.get("q_rank", 0))
        self.window = int(p.get("window", 0))
        self.sinks = tensors[n["sink"]].float().contiguous() if p.get("sink") else None
        self.gated = bool(p.get("gate"))
        ws = [tensors[n["dq"] if self.q_rank else n["q"]]] + ([] if self.borrows else [tensors[n["dkv"]]]) \
            + ([tensors[n["g"]]] if self.gated else [])
        if len({w.dtype for w in ws}) != 1:
            ws = [w.float() for w in ws]
        self.n_q = ws[0].shape[0]
        starts, stacked, at = [], [], 0      # every projection's columns start at a multiple of eight
        for w in ws:
            if at % 8:
                stacked.append(torch.zeros(8 - at % 8, w.shape[1], dtype=w.dtype, device=w.device))
                at += 8 - at % 8
            starts.append(at)
            stacked.append(w)
            at += w.shape[0]
        self.down_at = starts[1] if not self.borrows else 0
        self.down_n = 0 if self.borrows else self.R + self.dr
        self.gate_at = starts[-1] if self.gated else 0
        self.w_in, self.beside_at = rt.weight(torch.cat(stacked, dim=0)), None
        # (a reading layer writes no rows and has no weight for their norm; the kernel's check wants one of its size)
        self.norm_w = torch.ones(self.R, dtype=torch.float32, device=rt.device) if self.borrows \
            else tensors[n["dkv_norm"]].float().contiguous()
        if self.q_rank:
            self.q_norm_w = tensors[n["dq_norm"]].float().contiguous()
            self.w_uq = rt.weight(tensors[n["uq"]])
        H, dn, dv, R = self.H, self.dn, self.dv, self.R
        self.w_uk_t = tensors[n["uk"]].view(H, dn, R).transpose(1, 2).contiguous()   # [H, R, dn]: q_plain -> latent lanes
        self.w_uv = tensors[n["uv"]].view(H, dv, R).contiguous()
        self.w_o = rt.weight(tensors[n["o"]])
        rt.ops.latent_attn_init(rt.device)
        self.use_mfma = (os.environ.get("BURN_LM_AMD_LATENT_MFMA") != "0" and self.scale > 0 and self.w_uk_t.dtype == torch.bfloat16
                         and rt.ops.latent_attn_mfma_supported(rt.dtype, R, self.dr))

        self.can_expand = (self.use_mfma and self.w_uv.dtype == torch.bfloat16
                           and rt.ops.latent_prompt_supported(rt.dtype, R, dn, self.dr, dv))
        # [H * dn, R]: latents -> plain keys, a second layout of w_uk_t that only the expanded form reads
        self.w_uk = tensors[n["uk"]].contiguous() if self.can_expand else None
        if self.can_expand:
            rt.ops.latent_prompt_init(rt.device)
            # (a view into a larger tensor may start anywhere; the kernels read 16 bytes at a time)
            self.w_uk, self.w_uv = (w.clone() if w.data_ptr() % 16 else w for w in (self.w_uk, self.w_uv))

    def expands(self, step, q, view):
        """Whether the step's keys and values are expanded per head instead of absorbing the projections into queries and
        results: 2 R (dn + dv) operations per row and head once, against 2 (2 R + dr - dn - dr - dv) fewer per query and row."""
        bucket = getattr(step, "bucket", None)
        tokens, seqs, longest = bucket or (step.n_tokens, step.n_seqs, step.max_len_after)
        slack = EXPAND_BUCKET_SLACK if bucket else 1
        rows = seqs * -(-longest // 64) * 64
        return (self.can_expand and step.max_new > 1 and view.v.numel() > 0 and view.page_size == 64
                and tokens * slack >= EXPAND_MIN_NEW * seqs and rows <= max(slack * EXPAND_MAX_ROWS[0], EXPAND_MAX_ROWS[1] * tokens)
                and seqs <= EXPAND_MAX_BLOCKS and -(-longest // 64) <= EXPAND_MAX_BLOCKS and q.stride(0) % 8 == 0 and q.data_ptr() % 16 == 0)

    def _matrices(self):
        return [self.w_in.w, self.w_o.w, self.w_uk_t, self.w_uv] + ([self.w_uq.w] if self.q_rank else [])

    def step_bytes(self, rows):
        return sum(w.numel() * w.element_size() for w in self._matrices())

    def step_flops(self, rows):
        return 2 * rows * sum(w.numel() for w in self._matrices())

    def mixing_flops(self, past, new):
        """The smaller of the two forms' operations.  (The expansion of the new rows takes what step_flops counts for their products
        with W_uk and W_uv.)"""
        absorbed = 2 * self.H * (2 * self.R + self.dr) * self._pairs(past, new)
        return min(absorbed, self.expanded_flops(past, new) - self._expansion(new)) if self.can_expand else absorbed

    def expanded_flops(self, past, new):
        """Of attend_expanded: the expansion of every row that a new token sees, scores over dim + rot_dim lanes and weighted values
        over vdim lanes per (query, visible row, head)."""
        rows = new + (min(past, self.window - 1) if self.window else past)
        return self._expansion(rows) + 2 * self.H * (self.dn + self.dr + self.dv) * self._pairs(past, new)

    def _expansion(self, rows):
        return 2 * self.R * self.H * (self.dn + self.dv) * rows

    def _pairs(self, past, new):
        return sum(min(past + t + 1, self.window) for t in range(new)) if self.window else new * past + new * (new + 1) // 2

    def forward(self, x, step, view):
        return self._forward(x, step, view)[0]

    def forward_beside(self, x, step, view):
        y, qd = self._forward(x, step, view)
        return y, qd[:, self.beside_at:]

    def _forward(self, x, step, view):
        qd, q, gate = self._inputs(x)
        if self.expands(step, q, view):
            return self._finish(self.attend_expanded(self._turn(qd, q, step, view), step, view), gate), qd
        return self.output(self.attend(self._absorb(qd, q, step, view), step, view), gate), qd

    def project_expanded(self, x, step, view):
        """The plain queries and their turned lanes, for attend_expanded, with the step's rows in the cache afterwards; None, with nothing
        written, where the step runs in the absorbed form."""
        qd, q, _ = self._inputs(x)
        return self._turn(qd, q, step, view) if self.expands(step, q, view) else None

    def project(self, x, step, view):
        """The absorbed queries [tokens, heads, kv_rank + rot_dim] of the step's tokens; their latents and turned key
        parts are in the cache afterwards."""
        qd, q, _ = self._inputs(x)
        return self._absorb(qd, q, step, view)

    def _inputs(self, x):
        """The stacked projection's rows, the queries before any turning, and the output gate's columns (None without a gate)."""
        rt = self.rt
        qd = rt.linear(x, self.w_in)                         # [T, H (dn + dr) or q_rank | R + dr]
        q = qd[:, :self.n_q]
        if self.q_rank:
            cq = rt.ops.rmsnorm_rows(q, self.q_norm_w, self.eps, torch.empty(x.shape[0], self.q_rank, dtype=qd.dtype, device=x.device))
            q = rt.linear(cq, self.w_uq)
        return qd, q, (qd[:, self.gate_at:self.gate_at + self.H * self.dv] if self.gated else None)

    def _write(self, qd, q, turned, step, view, vcache):
        """The turned query lanes into turned ([tokens, heads, kv_rank + rot_dim] or [.., rot_dim]), the step's rows into the cache."""
        if self.borrows == bool(view.store):
            raise ValueError("a layer with a down-projection keeps its own rows, a borrowing layer reads another's")
        down = None if self.borrows else qd[:, self.down_at:self.down_at + self.down_n]
        self.rt.ops.latent_write(down, q, self.norm_w, self.eps, self.position.table, self.rot, turned, view.k, step,
                                 view.block_table(step), view.page_size, self.H, self.dn, self.R, self.dr, write_kv=view.store,
                                 vcache=vcache if view.store else None, adjacent=self.adjacent)

    def _absorb(self, qd, q, step, view):
        rt, H, dn, dr, R, T = self.rt, self.H, self.dn, self.dr, self.R, q.shape[0]
        mfma = self.use_mfma and view.v.numel() > 0 and view.page_size == 64
        qabs = torch.empty(T, H, R + dr, dtype=rt.dtype if mfma else torch.float32, device=q.device)
        self._write(qd, q, qabs, step, view, view.v if mfma else None)
        rt.ops.head_project(q, dn + dr, self.w_uk_t, qabs.view(T, H * (R + dr)), R + dr)
        return qabs

    def _turn(self, qd, q, step, view):
        turned = torch.empty(q.shape[0], self.H, self.dr, dtype=self.rt.dtype, device=q.device)
        self._write(qd, q, turned, step, view, view.v)
        return q, turned

    def attend_expanded(self, queries, step, view):
        """Every (token, head)'s weighted sum of the values it sees -> [tokens, heads * vdim], keys and values expanded per head."""
        q, turned = queries
        rt, H = self.rt, self.H
        o = torch.empty(q.shape[0], H * self.dv, dtype=rt.dtype, device=q.device)
        return rt.ops.latent_prompt(q, turned, o, view.k, self.w_uk, self.w_uv.view(H * self.dv, self.R), step, view.block_table(step),
                                    -(-step.max_len_after // 64), H, self.R, self.dn, self.dr, self.dv, self.scale, window=self.window,
                                    sinks=self.sinks)

    def attend(self, qabs, step, view):
        """Every (token, head)'s weighted sum of the latents it sees -> float32 [tokens, heads, kv_rank]."""
        rt, ops = self.rt, self.rt.ops
        H, dr, R = self.H, self.dr, self.R
        T = qabs.shape[0]
        olat = torch.empty(T, H, R, dtype=torch.float32, device=qabs.device)
        n_splits = 1
        seen = min(step.max_len_after, self.window) if self.window else step.max_len_after
        if qabs.dtype == torch.bfloat16:        # the matrix-core form: one wavefront per 16 (token, head) pairs
            if step.max_new == 1:
                halves = (seen + 31) // 32 + (1 if seen < step.max_len_after else 0)     # a window may begin inside a half page
                n_splits = max(1, min(halves, most_pieces(step.n_seqs * ((H + 15) // 16), R, rt.compute_units),
                                      ops.latent_attn_mfma_max_splits(step.n_seqs, 1, H, R)))
            return ops.latent_attn_mfma(qabs, olat, view.k, view.v, step, view.block_table(step), view.page_size, H, R,
                                        dr, self.scale, n_splits, window=self.window, sinks=self.sinks)
        if step.max_new == 1:
            chunks = (seen + 63) // 64
            blocks = (T * H + 3) // 4
            n_splits = max(1, min(chunks, (DECODE_BLOCKS_PER_UNIT * rt.compute_units) // blocks,
                                  ops.latent_attn_max_splits(T, H, R)))
        return ops.latent_attn(qabs, olat, view.k, step, view.block_table(step), view.page_size, H, R, dr, self.scale,
                               n_splits, window=self.window, sinks=self.sinks)

    def output(self, olat, gate=None):
        rt = self.rt
        T = olat.shape[0]
        o = torch.empty(T, self.H * self.dv, dtype=rt.dtype, device=olat.device)
        rt.ops.head_project(olat.view(T, self.H * self.R), self.R, self.w_uv, o, self.dv)
        return self._finish(o, gate)

    def _finish(self, o, gate):
        if gate is not None:
            self.rt.ops.sigmoid_gate(o, gate)
        return self.rt.linear(o, self.w_o, partials=True)
