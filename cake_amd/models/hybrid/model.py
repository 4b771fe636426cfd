"""Hybrid decoder model: embedding -> layer runs -> final norm -> head.

One step function serves prompts, decoding and mixtures of sequences (:meth:`HybridModel.step`):
the tokens of all sequences are packed back to back, every projection is one matrix product
over the packed rows, and only the mixers look at which row belongs to which sequence and
position.  A parallel layer is three stages — norm + input projections, mixer, output projections
+ residual — because its two sublayers read one norm and are summed (:mod:`.weights`); a serial
layer has its feed-forward (:mod:`.feedforward`) behind them.

* prompt rows: MFMA GEMMs (ops/gemm.py; the feed-forward's activation and the scaled residual
  sum in their epilogues), prompt kernels of the mixers (ops/mixers.py, ops/latent.py); of up to 64
  rows all projections of a layer are one product by sections where that gains (gemm.sections);
* one token of one sequence, 16-bit: three launches per parallel layer run
  (:meth:`decode_layers`, the body of the captured decode graph, models/decoder.py);
* one token of several sequences: the GEMMs over the batch, the mixers' decode kernels;
* f32: the same kernels in their 32-bit form; the plain products are the vendor's 32-bit GEMM.
"""
from __future__ import annotations

import contextlib
from dataclasses import dataclass
from functools import partial
from pathlib import Path

import torch

from ...ops import gemm as G
from ...ops import latent as LA
from ...ops import mixers as M
from ...ops._lib import upload
from ..base import StepEntry
from .config import AttentionMixer, HybridConfig, LatentMixer, from_path
from .state import StatePool
from .weights import LayerWeights, ModelWeights

# key splits of a decode-attention launch by live length: (up to this many tokens, splits)
SPLITS = ((256, 1), (1024, 8), (4096, 16), (1 << 30, 32))
# the latent kernels' for the same buckets: a workgroup takes one 64-key tile while there are
# splits for all of them
LATENT_SPLITS = {n: min(M.MAX_SPLIT, -(-lim // 64)) for lim, n in SPLITS}
MERGE_BYTES = 3 << 19   # of split sums that the value expansion of a sequence alone reads


def latent_alone(nsplit: int, sh: LA.LatentShape) -> tuple[int, int]:
    """(splits, tile) of a sequence alone: of short contexts 32-key tiles, unless their sums are as much to read as the
    tiles (128 heads of rank 512 over 40 / 150 / 250 keys 12.4 / 13.9 / 15.3 us, 13.0 / 14.3 / 14.5 in 64-key tiles; 64 heads
    11.2 / 12.3 / 12.7, 12.1 / 13.0 / 13.2)."""
    return (8, 32) if nsplit == 1 and 4 * sh.part_floats(1, 8) <= MERGE_BYTES else (LATENT_SPLITS[nsplit], 64)


def latent_splits(nsplit: int, rows: M.Rows, heads: int, per_cu: int = 1) -> int:
    """Splits of a step's sequences: no more workgroups at the longest one's length than CUs, since the value expansion
    reads every split's sums (16 heads of 24 sequences at 600 / 3000 keys 38.6 us in 16 splits / 70.4 in 32, 30.5 / 44.4 in
    8; 32 heads of 13 at 1000 45.4 in 16, 30.4 in 8; 32 heads of 2 at 3000 24.4 in 32, 25.1 in 16, 31.1 in 8).  While splits
    hold four tiles and more, as many as CUs with `per_cu` each hold, and a tenth of the longest's keys counts nothing
    (128 heads of rank 256 of 3 at 30000 142.9 in 8, 94.9 in 16, of rank 512 of one at 30000 and 12 at 100 146 in 16, 120
    in 32; of rank 256 of 2 at 3000, two tiles a split, 21.8 in 16, 25.0 in 32)."""
    keys = [p0 + n for _, n, p0, _ in rows.host]
    most, total, groups = max(keys), sum(keys), -(-heads // 16)
    # as many sequences of the longest one's length
    n = min(LATENT_SPLITS[nsplit], 1 << max(1, 256 // (-(-total // most) * groups)).bit_length() - 1)
    room = 256 * per_cu // (-(-(10 * total - most) // (10 * most)) * groups)
    while 2 * n <= min(LATENT_SPLITS[nsplit], room) and -(-most // (2 * n)) > 192:
        n *= 2
    return n


# Rows of a step from which on the last run's unread ones are left out (:meth:`HybridModel._last_rows`);
# fewer go through the products of few rows, which read the weights once either way
LAST_LEAST = 65
# ... and rows times weights of that layer, of all experts: the wanted rows are launches of their own, some 55 us
# of host time a step.  Nine runs of 61 million weights each at 100 / 200 / 260 / 500 rows 1039 / 1062 / 1145 / 1415
# us, 986 / 1056 / 1170 / 1457 with all rows (one call on an idle GPU at 128 / 200 / 260 1166 / 1204 / 1311, 1130 /
# 1241 / 1342); of 218 million at 65 rows 1524, 1542; of 532 million, most of them 64 experts', at 65 2232, 2406.
LAST_WORK = 12e9
GEN_SLOT = 0  # the generator's own sequence


def _splits(tk: int) -> int:
    return next(n for lim, n in SPLITS if tk <= lim)


@dataclass
class DecodeState:
    """Device buffers of the captured batch-1 decode step (stable addresses)."""
    x0: torch.Tensor       # embedding row, [Wp] f32
    xe: torch.Tensor       # the same, normed (designs that norm it)
    xa: torch.Tensor       # residual rows: a looped pass is entered from one into the other
    xb: torch.Tensor
    proj: torch.Tensor     # [max n_raw] f32
    act: torch.Tensor      # per layer: [mixer output | feed-forward], storage dtype
    lat_q: torch.Tensor    # latent attention: queries (f32), queries in the latent space
    lat_qa: torch.Tensor
    ff: torch.Tensor       # serial feed-forwards: activations, router logits, chosen experts
    route: torch.Tensor
    sel: torch.Tensor
    part: torch.Tensor
    ticket: torch.Tensor
    pos: torch.Tensor
    seq_slot: torch.Tensor
    tok: torch.Tensor
    hist: torch.Tensor
    hist_len: torch.Tensor
    slot: torch.Tensor     # token-selection key (argmax / draw)
    thr: torch.Tensor
    sel_ticket: torch.Tensor
    logits: torch.Tensor


class HybridModel:
    backend = "hip"
    all_local = True
    session = 0

    def __init__(self, cfg: HybridConfig, head: ModelWeights, layers: list[LayerWeights], device,
                 dtype, max_seq: int, slots: int = 2):
        self.cfg, self.head, self.layers = cfg, head, layers
        self.device, self.dtype = torch.device(device), dtype
        if self.device.type != "cuda":
            raise ValueError("the hybrid designs run on the GPU only")
        self.max_seq = max_seq
        self.runs = cfg.runs()
        self.W, self.Wp = cfg.hidden_size, cfg.width_padded
        self.pool = StatePool(cfg, self.device, dtype, max(2, slots), max_seq)
        self.pool.length[GEN_SLOT] = 0
        self._rot: dict = {}
        self._none = torch.zeros(2, device=self.device)
        self._bufs: DecodeState | None = None    # the captured decoder's
        self._eager: DecodeState | None = None   # single-token steps of any sequence
        self._nsplit: int | None = None
        # decode attention's split partials and arrival tickets (zeroed once, re-armed by the
        # kernel); grown for the largest batch seen
        self._part = self._ticket = None

    # ------------------------------------------------------------------ construction
    @classmethod
    def load(cls, model_dir: str | Path, device, dtype, max_seq: int, slots: int = 2):
        from ...utils.safetensors_io import ShardedCheckpoint
        cfg = from_path(model_dir)
        return cls.build(cfg, ShardedCheckpoint(model_dir).get, device, dtype, max_seq, slots)

    @classmethod
    def build(cls, cfg: HybridConfig, get, device, dtype, max_seq: int, slots: int = 2):
        own = {i: LayerWeights.load(get, i, cfg, device, dtype)
               for i, L in enumerate(cfg.layers) if L.weights_of is None}
        layers = [own[cfg.weights_layer(i)] for i in range(len(cfg.layers))]
        return cls(cfg, ModelWeights.load(get, cfg, device, dtype), layers, device, dtype, max_seq,
                   slots)

    # ------------------------------------------------------------------ pieces
    def _rotation(self, m: AttentionMixer | LatentMixer) -> torch.Tensor:
        """[S, dims] f32 (cos, sin) pairs of every cache position, computed in double."""
        if m.rot is None or m.rot.dims < 2:
            return self._none
        t = self._rot.get(m.rot)
        if t is None:
            n = m.rot.dims // 2
            f = torch.tensor(m.rot.frequencies(), dtype=torch.float64)
            a = torch.arange(self.pool.S, dtype=torch.float64)[:, None] * f
            t = torch.stack([a.cos(), a.sin()], -1).reshape(self.pool.S, 2 * n)
            t = (t * m.rot.magnitude()).float()
            t = self._rot[m.rot] = t.to(self.device).contiguous()
        return t

    def norm_rows(self, x, w32, rows=None, scale=None, dtype=None, where=None) -> torch.Tensor:
        """The model's norm of residual rows (of rows[r], times scale[r]; or each to the rows
        where[r])."""
        n = x.shape[0] if rows is None and where is None else (rows if where is None else where).numel()
        h = torch.empty((n, self.Wp), device=self.device, dtype=dtype or self.dtype)
        M.norm(x, w32, self.cfg.norm_offset, self.cfg.eps, self.W, h, rows=rows,
               ln=self.cfg.layer_norm, scale=scale, where=where)
        return h

    def product(self, x, w, out):
        """out = x w^T (out: storage dtype, or f32)."""
        if self.dtype == torch.float32:
            torch.mm(x, w.t(), out=out) if out.is_contiguous() else out.copy_(torch.mm(x, w.t()))
        elif out.dtype == torch.float32:
            G.linear(x, w, epi="store32", resid=out)
        else:
            G.linear(x, w, out=out)
        return out

    def product_add(self, x, w, y, alpha: float, bias=None):
        """y[:, :N] += alpha (x w^T + bias) (f32)."""
        y = y[:, :w.shape[0]]
        if self.dtype == torch.float32:
            t = torch.mm(x, w.t()) if bias is None else torch.addmm(bias, x, w.t())
            y.add_(t, alpha=alpha)
        else:
            G.linear(x, w, bias, epi="resid32", resid=y, alpha=alpha)

    def add_norm(self, x, w, y, alpha: float, norm32, bias=None):
        """:meth:`product_add`, and the norm of the new rows by norm32 where one launch does both (None: it
        is left to what reads them): of few rows the product stops at its slabs and the norm sums them."""
        W, cfg = w.shape[0], self.cfg
        form = None if norm32 is None or self.dtype == torch.float32 or W != self.Wp or \
            W > G.SLAB_NORM_MAX else G.slab_form(x.shape[0], W, x.shape[1], "resid32")
        if form is None:
            self.product_add(x, w, y, alpha, bias)
            return None
        h = torch.empty((x.shape[0], W), device=self.device, dtype=self.dtype)
        G.slab_norm(*G.slabs(x, w, form), y, norm32, cfg.eps, h, bias=bias, alpha=alpha,
                    offset=cfg.norm_offset, ln=cfg.layer_norm)
        return h

    def product_act(self, x, w, out, act: str = "gelu", bias=None):
        """out = activation(x w^T + bias)."""
        if self.dtype == torch.float32:
            M.act(act, torch.mm(x, w.t()), out, bias)
        else:
            G.linear(x, w, bias, epi=act, out=out)

    def _split_ws(self, B: int):
        """(partials, tickets) of decode attention for a batch of B sequences."""
        shapes = [s for s in self.pool.shapes if not s.recurrent]
        need = max((s.part_floats(B, n) for s in shapes for n in
                    ((max(LATENT_SPLITS.values()),) if isinstance(s, LA.LatentShape)
                     else (max(n for _, n in SPLITS),))), default=1)
        tick = max((B * s.tiles for s in shapes), default=1)
        if self._part is None or self._part.numel() < need or self._ticket.numel() < tick:
            self._part = torch.zeros(need, device=self.device, dtype=torch.float32)
            self._ticket = torch.zeros(tick, device=self.device, dtype=torch.int32)
        return self._part, self._ticket

    # ------------------------------------------------------------------ packed rows
    def _layer_rows(self, run, x, h, rows: M.Rows, nsplit: int, observe, next_norm):
        """One layer run of x; h: the norm of x if it is there.  Returns the norm by next_norm (None: of
        no use) of the new x if it is there."""
        L, w = self.cfg.layers[run.layer], self.layers[run.layer]
        m, N, cfg = L.mixer, rows.N, self.cfg
        decode = rows.max_len == 1
        h = self.norm_rows(x, w.norm32) if h is None else h
        new = torch.empty if w.mix_cols == w.shape.out_cols and w.ff % 8 == 0 else torch.zeros
        mix = new((N, w.out_cols), device=self.device, dtype=self.dtype)
        # the mixers' decode kernels read f32 projections, as the fused step leaves them; a latent
        # is normed before anything else reads it
        pdt = torch.float32 if decode or isinstance(m, LatentMixer) else self.dtype
        ncol = w.n_raw if decode else w.n_main
        proj = torch.empty((N, M.pad_to(ncol, 8)), device=self.device, dtype=pdt)
        ab = None if decode or not w.n_ab else \
            torch.empty((N, w.n_ab), device=self.device, dtype=torch.float32)
        up = mix[:, w.mix_cols:w.mix_cols + w.ff]
        n16, part = (0, proj[:, :ncol]) if pdt == torch.float32 else (w.n_main, ab)
        if not (w.ff and self.dtype != torch.float32 and
                G.sections(h, w.w_in, n16, w.n_raw, proj[:, :ncol], part, up)):
            if w.ff:
                self.product_act(h, w.w_in[w.n_raw:], up)
            self.product(h, w.w_in[:ncol], proj[:, :ncol])
            if ab is not None:
                self.product(h, w.w_in[w.n_main:w.n_raw], ab)
        a, b = self.pool.bufs[run.index]
        if isinstance(m, LatentMixer):
            self._latent_rows(m, w, proj, rows, a, mix, latent_splits(nsplit, rows, w.shape.heads,
                                                                            LA.decode_per_cu(w.shape, self.dtype)))
        elif isinstance(m, AttentionMixer):
            cs = self._rotation(m)
            if decode:
                part, ticket = self._split_ws(rows.B)
                M.attn_decode(w.shape, proj, rows.pos, rows.slot, cs, m.qk_norm, m.sink, m.gated,
                              cfg.eps, m.scale, a, b, mix, nsplit, part, ticket)
            else:
                qn = torch.empty((N, m.heads, w.shape.DP), device=self.device, dtype=self.dtype)
                M.attn_prep(w.shape, proj, rows, cs, m.qk_norm, cfg.eps, qn, a, b)
                gate = proj[:, w.shape.qkv_cols:w.n_main] if m.gated else None
                M.attn_prompt(w.shape, qn, a, b, rows, gate, mix, m.scale, m.sink)
        elif decode:
            M.delta_decode(w.shape, proj, proj[:, w.n_main:w.n_raw], rows.pos, rows.slot, cfg.eps,
                           **w.consts, state=a, ring=b, out=mix)
        else:
            M.delta_prompt(w.shape, proj, ab, rows, cfg.eps, **w.consts, state=a, ring=b, out=mix)
        h = self.add_norm(mix, w.w_out, x, cfg.residual_mult,
                          next_norm if w.post is None else w.post.norm32)
        if w.post is not None:
            h = w.post.rows(self, x, h, next_norm)
        if observe is not None:
            observe(x[:, :self.W])
        return h

    def _last_rows(self, run, x, h, rows: M.Rows, nsplit: int, sel) -> torch.Tensor:
        """The last run of a prompt of which only the rows sel (one of a sequence at most) are read: all
        rows leave keys and values or the state; what follows is that of one token per sequence, at the
        place of its row.  The cache is the same whichever rows are wanted; keys and values are a product of
        their own here, so against a step that takes all rows through they may differ by the order of its
        sums, a rounding.  Returns the wanted rows."""
        L, w, cfg = self.cfg.layers[run.layer], self.layers[run.layer], self.cfg
        m, N, n, dev = L.mixer, rows.N, sel.numel(), self.device
        h = self.norm_rows(x, w.norm32) if h is None else h
        x1, h1 = x.index_select(0, sel), h.index_select(0, sel)
        pos, slot = rows.pos.index_select(0, sel), rows.slot.index_select(0, sel)
        mix = torch.zeros((n, w.out_cols), device=dev, dtype=self.dtype)
        up = mix[:, w.mix_cols:w.mix_cols + w.ff]
        a, b = self.pool.bufs[run.index]
        one = None   # the wanted rows' projections
        if isinstance(m, AttentionMixer):
            q, kv = w.shape.q_cols, w.shape.qkv_cols
            q -= q % 8   # whole pieces of the rows
            proj = torch.empty((N, M.pad_to(kv, 8)), device=dev, dtype=self.dtype)
            self.product(h, w.w_in[q:kv], proj[:, q:kv])
            M.attn_prep(w.shape, proj, rows, self._rotation(m), m.qk_norm, cfg.eps, None, a, b)
            one = torch.empty((n, M.pad_to(w.n_raw, 8)), device=dev, dtype=torch.float32)[:, :w.n_raw]
        if not (w.ff and one is not None and G.sections(h1, w.w_in, 0, w.n_raw, None, one, up)):
            if w.ff:
                self.product_act(h1, w.w_in[w.n_raw:], up)
            if one is not None:
                self.product(h1, w.w_in[:w.n_raw], one)
        if isinstance(m, AttentionMixer):
            # (not the steps' own: a captured step may run meanwhile)
            part = torch.empty(w.shape.part_floats(n, nsplit), device=dev, dtype=torch.float32)
            ticket = torch.zeros(n * w.shape.tiles, device=dev, dtype=torch.int32)
            M.attn_decode(w.shape, one, pos, slot, self._rotation(m), m.qk_norm, m.sink, m.gated,
                          cfg.eps, m.scale, a, b, mix, nsplit, part, ticket, held=True)
        elif isinstance(m, LatentMixer):
            sh, c, cs = w.shape, w.consts, self._rotation(m)
            splits = latent_splits(nsplit, rows, sh.heads, LA.decode_per_cu(sh, self.dtype))
            proj = torch.empty((N, w.n_main), device=dev, dtype=torch.float32)
            self.product(h, w.w_in[:w.n_main], proj)
            cq = torch.empty((N, sh.QP), device=dev, dtype=self.dtype)
            LA.prep(sh, proj, rows, cs, cfg.eps, c["q_norm32"], c["kv_norm"], cq, a)
            part = torch.empty(sh.part_floats(n, splits), device=dev, dtype=torch.float32)
            self._latent_tokens(m, w, cq.index_select(0, sel), pos, slot, a, mix, splits, part)
        else:
            proj = torch.empty((N, M.pad_to(w.n_main, 8)), device=dev, dtype=self.dtype)[:, :w.n_main]
            ab = torch.empty((N, w.n_ab), device=dev, dtype=torch.float32)
            self.product(h, w.w_in[:w.n_main], proj)
            self.product(h, w.w_in[w.n_main:w.n_raw], ab)
            out = torch.empty((N, w.mix_cols), device=dev, dtype=self.dtype)
            M.delta_prompt(w.shape, proj, ab, rows, cfg.eps, **w.consts, state=a, ring=b, out=out)
            cols = w.shape.out_cols
            mix[:, :cols] = out[:, :cols].index_select(0, sel)
        h1 = self.add_norm(mix, w.w_out, x1, cfg.residual_mult, None if w.post is None else w.post.norm32)
        if w.post is not None:
            w.post.rows(self, x1, h1)
        return x1

    def _latent_tokens(self, m: LatentMixer, w, cq, pos, slot, cache, mix, nsplit: int, part) -> None:
        """Latent attention of one token per sequence, whose cache rows are there: cq [B, QP] their
        normed query latents."""
        sh, c, N = w.shape, w.consts, cq.shape[0]
        q = torch.empty((N, sh.q_cols), device=self.device, dtype=torch.float32)
        self.product(cq, c["uq"], q)
        qa = torch.empty((N, sh.heads, sh.LD), device=self.device, dtype=self.dtype)
        LA.absorb(sh, q, c["uk_t"], pos, slot, self._rotation(m), self.cfg.eps, c["kv_norm"], cache, qa)
        LA.decode(sh, qa, pos, slot, cache, m.scale, nsplit, part)
        LA.out(sh, part, pos, c["uv"], nsplit, mix)

    def _latent_rows(self, m: LatentMixer, w, proj, rows: M.Rows, cache, mix, nsplit: int) -> None:
        """Latent attention of projected rows into mix[:, :H vdim]."""
        sh, c, N, dev = w.shape, w.consts, rows.N, self.device
        cs = self._rotation(m)
        cq = torch.empty((N, sh.QP), device=dev, dtype=self.dtype)
        LA.prep(sh, proj, rows, cs, self.cfg.eps, c["q_norm32"], c["kv_norm"], cq, cache)
        if rows.max_len == 1:   # on the latent rows themselves
            part, _ = self._split_ws(N)
            self._latent_tokens(m, w, cq, rows.pos, rows.slot, cache, mix, nsplit, part)
            return
        q = torch.empty((N, sh.q_cols), device=dev, dtype=self.dtype)
        self.product(cq, c["uq"], q)
        # keys and transposed values of every live position, from the cache
        live = [cache[s, :M.pad_to(p0 + n, 64), :sh.RP] for _, n, p0, s in rows.host]
        lat = live[0] if len(live) == 1 else torch.cat(live)
        k = torch.empty((rows.n_keys, sh.heads * sh.dimP), device=dev, dtype=self.dtype)
        vt = torch.empty((sh.heads * sh.DVP, rows.n_keys), device=dev, dtype=self.dtype)
        self.product(lat, c["uk"], k)
        self.product(c["uv"], lat, vt)
        LA.prompt(sh, q, k, vt, rows, cs, cache, mix, m.scale)

    def _forward_rows(self, rows: M.Rows, observe=None, sel=None) -> torch.Tensor:
        """Residual rows [N, Wp] f32 after every layer run, of the rows sel alone if given."""
        N, head = rows.N, self.head
        x = torch.empty((N, self.Wp), device=self.device, dtype=torch.float32)
        x0 = torch.empty_like(x) if self.cfg.loop is not None else None
        M.embed(head.embed, rows.tok, x, x0)
        if self.cfg.embed_norm:
            x = self.norm_rows(x, head.embed_norm, dtype=torch.float32)
            if x0 is not None:
                x0.copy_(x)
        nsplit = _splits(max(p0 + n for _, n, p0, _ in rows.host))
        h = None
        for run, after in zip(self.runs, [*self.runs[1:], None]):
            if run.enter is not None:
                pair = torch.empty((N, head.loop_in.shape[1]), device=self.device,
                                   dtype=self.dtype)
                y = torch.empty_like(x)
                M.loop_rows(x, x0, head.loop_step[run.enter], self.W, pair, y)
                h = self.add_norm(pair, head.loop_in, y, 1.0, self.layers[run.layer].norm32)
                x = y
            if after is None and sel is not None:
                return self._last_rows(run, x, h, rows, nsplit, sel)
            # the last rows are gathered before their norm, an entered pass reads them as they are
            next_norm = None if after is None or after.enter is not None else \
                self.layers[after.layer].norm32
            h = self._layer_rows(run, x, h, rows, nsplit, observe, next_norm)
        return x

    def _logits(self, x, sel) -> torch.Tensor:
        """Logits [n, V] f32 of the residual rows sel [n] (None: of all)."""
        n = x.shape[0] if sel is None else sel.numel()
        out = torch.empty((n, self.cfg.vocab_size), device=self.device, dtype=torch.float32)
        if n:
            self.product(self.norm_rows(x, self.head.norm32, rows=sel), self.head.lm_head, out)
        return out

    def _reads_few(self, rows: M.Rows, entries, observe) -> bool:
        """Whether the last run's results are read at few rows, one of a sequence (:meth:`_last_rows`)."""
        n = sum(len(e.want) for e in entries)
        w = self.layers[self.runs[-1].layer]
        weights = w.w_in.numel() + w.w_out.numel() + (0 if w.post is None else w.post.weights)
        return observe is None and self.dtype != torch.float32 and rows.max_len > 1 and \
            rows.N >= LAST_LEAST and rows.N * weights >= LAST_WORK and \
            0 < n <= min(G.ROWS_MAX, rows.N // 4) and all(len(e.want) <= 1 for e in entries)

    # ------------------------------------------------------------------ steps
    def open_sequence(self) -> int:
        return self.pool.open()

    def close_sequence(self, sid: int) -> None:
        self.pool.close(sid)

    @torch.no_grad()
    def step(self, entries: list[StepEntry], observe=None) -> list[torch.Tensor]:
        """Feed each sequence its next tokens as one batch; logits [len(want), V] per entry.
        ``observe`` is called with the packed residual rows after every layer run."""
        if len({e.seq for e in entries}) != len(entries):
            raise ValueError("a sequence appears twice in one step")
        V = self.cfg.vocab_size
        for e in entries:
            if not e.tokens or not all(0 <= t < V for t in e.tokens) or \
                    not all(0 <= w < len(e.tokens) for w in e.want):
                raise ValueError("step: tokens or wanted places out of range")
            if self.pool.length[e.seq] + len(e.tokens) > self.max_seq:
                raise ValueError(f"sequence {e.seq} exceeds max_seq {self.max_seq}")
        seqs = [(e.seq, self.pool.reserve(e.seq, len(e.tokens)), e.tokens) for e in entries]
        if len(seqs) == 1 and len(entries[0].tokens) == 1 and self.dtype != torch.float32 \
                and observe is None:
            slot, pos, (tok,) = seqs[0]
            if self._eager is None:  # not the captured decoder's: its step state lives on
                self._eager = self._decode_buffers()
            b = self._eager
            b.tok.fill_(tok)
            b.pos.fill_(pos)
            b.seq_slot.fill_(slot)
            self.decode_embed(b)
            with self.decode_eager(pos):
                x = self.decode_layers(b, range(len(self.runs)))
            sel = torch.zeros(len(entries[0].want), dtype=torch.int32, device=self.device)
            return [self._logits(x.view(1, -1), sel)]
        rows = M.Rows.pack(seqs, self.device)
        take = [h[0] + w for h, e in zip(rows.host, entries) for w in e.want]
        sel = upload(take, torch.int32, self.device)
        if self._reads_few(rows, entries, observe):
            logits = self._logits(self._forward_rows(rows, None, sel), None)
        else:
            logits = self._logits(self._forward_rows(rows, observe), sel)
        return list(logits.split([len(e.want) for e in entries]))

    # ------------------------------------------------------------------ generator interface
    def reset(self) -> None:
        self.pool.length[GEN_SLOT] = 0

    def forward(self, tokens: list[int], pos0: int) -> torch.Tensor:
        """Logits (f32 [V]) of the last of `tokens`, fed at positions pos0.. of the
        generator's sequence."""
        self.pool.length[GEN_SLOT] = pos0
        return self.step([StepEntry(GEN_SLOT, list(tokens), [len(tokens) - 1])])[0][0]

    # ------------------------------------------------------------------ decode hooks
    @property
    def device_decode(self) -> bool:
        """Tokens can run as the fused step of a captured graph (16-bit weights)."""
        return self.dtype != torch.float32

    @property
    def decode_version(self) -> int:
        """Changes when captured graphs no longer fit the model's buffers."""
        return self.pool.version

    @property
    def num_decode_layers(self) -> int:
        return len(self.runs)

    def decode_buffers(self) -> DecodeState:
        if self._bufs is None:
            self._bufs = self._decode_buffers()
        return self._bufs

    def _decode_buffers(self) -> DecodeState:
        f, i32 = torch.float32, torch.int32
        z = partial(torch.zeros, device=self.device)
        part, ticket = self._split_ws(1)
        lat = [w.shape for w in self.layers if isinstance(w.shape, LA.LatentShape)]
        post = [w.post for w in self.layers if w.post is not None]

        def most(sizes):
            return max(sizes, default=0)
        return DecodeState(
            lat_q=z(most(s.q_cols for s in lat), dtype=f),
            lat_qa=z(most(s.heads * s.LD for s in lat), dtype=self.dtype),
            ff=z(most(p.act_elems for p in post), dtype=self.dtype),
            route=z(most(p.experts for p in post), dtype=f),
            sel=z(most(p.top for p in post), dtype=i32),
            x0=z(self.Wp, dtype=f), xe=z(self.Wp, dtype=f), xa=z(self.Wp, dtype=f), xb=z(self.Wp, dtype=f),
            proj=z(max(w.n_raw for w in self.layers), dtype=f),
            act=z((len(self.layers), max(w.out_cols for w in self.layers)), dtype=self.dtype),
            part=part, ticket=ticket, pos=z(1, dtype=i32), seq_slot=z(1, dtype=i32),
            tok=z(1, dtype=i32), hist=z(self.max_seq, dtype=i32), hist_len=z(1, dtype=i32),
            slot=z(1, dtype=torch.int64), thr=z(1, dtype=i32), sel_ticket=z(1, dtype=i32),
            logits=z(self.cfg.vocab_size, dtype=f))

    def decode_state(self, b: DecodeState) -> list[torch.Tensor]:
        return [b.tok, b.pos, b.hist_len, b.x0, *self.pool.recurrent(GEN_SLOT)]

    def decode_embed(self, b: DecodeState) -> None:
        M.embed(self.head.embed, b.tok, b.x0)

    def decode_layers(self, b: DecodeState, layers) -> torch.Tensor:
        """Layer runs of one token at device position b.pos of slot b.seq_slot (16-bit weights;
        graph-capturable); returns the residual row.  The first run of a step reads b.x0."""
        cfg = self.cfg
        x = x0 = b.xe if cfg.embed_norm else b.x0
        nsplit = self._nsplit or max(n for _, n in SPLITS)
        for r in layers:
            run = self.runs[r]
            if r == 0 and cfg.embed_norm:
                M.norm(b.x0.view(1, -1), self.head.embed_norm, cfg.norm_offset, cfg.eps, self.W,
                       b.xe.view(1, -1), ln=cfg.layer_norm)
            L, w = cfg.layers[run.layer], self.layers[run.layer]
            m = L.mixer
            if run.enter is not None:
                y = b.xb if x is b.xa else b.xa
                M.loop_in(x, x0, self.head.loop_step[run.enter], self.head.loop_in, self.W, y)
                x = y
            mix = b.act[run.layer, :w.out_cols]
            # the up rows go beside the mixer, which leaves most of the chip idle
            rows, up = w.w_in, None
            if w.ff and M.gains_by_up_rows(w.shape, w.ff, rows.shape[1]):
                rows = w.w_in[:w.n_raw]
                up = M.UpRows(x, w.norm, cfg.eps, cfg.norm_offset, cfg.layer_norm, self.W,
                              w.w_in[w.n_raw:], mix[w.mix_cols:])
            M.layer_in(x, w.norm, cfg.eps, cfg.norm_offset, self.W, rows, w.n_raw, b.proj,
                       mix[w.mix_cols:], ln=cfg.layer_norm)
            ka, kb = self.pool.bufs[run.index]
            proj = b.proj[:w.n_raw].view(1, -1)
            if isinstance(m, LatentMixer):
                self._latent_decode(m, w, b, proj, ka, mix.view(1, -1), *latent_alone(nsplit, w.shape))
            elif isinstance(m, AttentionMixer):
                M.attn_decode(w.shape, proj, b.pos, b.seq_slot, self._rotation(m), m.qk_norm,
                              m.sink, m.gated, cfg.eps, m.scale, ka, kb, mix.view(1, -1), nsplit,
                              b.part, b.ticket, up)
            else:
                M.delta_decode(w.shape, proj, proj[:, w.n_main:], b.pos, b.seq_slot, cfg.eps,
                               **w.consts, state=ka, ring=kb, out=mix.view(1, -1), up=up)
            y = b.xa if x is x0 else x
            M.layer_out(mix, w.w_out, cfg.residual_mult, x, y)
            x = y
            if w.post is not None:
                w.post.decode(self, b, x)
        self._last = x
        return x

    def _latent_decode(self, m: LatentMixer, w, b: DecodeState, proj, cache, mix,
                       nsplit: int, tile: int) -> None:
        """Latent attention of one token: query expansion (norm in the prologue), query into the
        latent space + cache row, attention over the latent rows, merge + value expansion."""
        sh, c, eps = w.shape, w.consts, self.cfg.eps
        q = b.lat_q[:sh.q_cols]
        M.layer_in(b.proj[:sh.QP], c["q_norm"], eps, 0.0, sh.q_rank, c["uq"], sh.q_cols, q)
        qa = b.lat_qa[:sh.heads * sh.LD]
        LA.absorb(sh, q.view(1, -1), c["uk_t"], b.pos, b.seq_slot, self._rotation(m), eps,
                  c["kv_norm"], cache, qa, proj=proj)
        LA.decode(sh, qa, b.pos, b.seq_slot, cache, m.scale, nsplit, b.part, tile)
        LA.out(sh, b.part, b.pos, c["uv"], nsplit, mix, tile)

    def decode_head(self, b: DecodeState) -> None:
        from ...ops import hip as K
        h = self.head
        K.norm_gemv_f32_off(self._last, h.norm, self.cfg.eps, self.cfg.norm_offset, self.W,
                            h.lm_head, b.logits, ln=self.cfg.layer_norm)

    def decode_head_select(self, b: DecodeState, last_n: int, penalty: float) -> None:
        from ...ops import hip as K
        h = self.head
        K.head_select_off(self._last, h.norm, self.cfg.eps, self.cfg.norm_offset, self.W,
                          h.lm_head, b.logits, b.hist, b.hist_len, last_n, penalty, b.slot,
                          b.sel_ticket, b.tok, b.pos, h.embed, b.x0,
                          ln=self.cfg.layer_norm)

    @contextlib.contextmanager
    def _split_scope(self, n: int):
        prev, self._nsplit = self._nsplit, n
        try:
            yield
        finally:
            self._nsplit = prev

    def decode_buckets(self) -> list:
        top = _splits(self.max_seq)
        return [(n, partial(self._split_scope, n)) for _, n in SPLITS if n <= top]

    def decode_need(self, tk: int) -> int:
        return _splits(tk)

    def decode_eager(self, pos: int):
        return self._split_scope(_splits(pos + 1))

    def decode_check(self, b: DecodeState) -> None:
        """Nothing to check: no launch of a step waits on another workgroup."""

    def prefill_logits(self, prompt: list[int], out: torch.Tensor) -> None:
        self.reset()
        out.copy_(self.forward(prompt, 0))
