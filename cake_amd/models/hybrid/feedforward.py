"""Feed-forwards of serial layers: dense, and routed experts.

Each class has its checkpoint layout (:func:`tensor_shapes`), its weights for the kernels, a form
for packed rows (``rows``) and one for a single 16-bit token (``decode``, graph-capturable).  Both
add to the residual row they read; the norm in front is theirs.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch

from ...ops import experts as X
from ...ops import mixers as M
from ...ops.mixers import pad_to
from .config import DenseMlp, ExpertsMlp
from .tensors import padded


def tensor_shapes(m: DenseMlp | ExpertsMlp, W: int) -> dict[str, tuple]:
    if m.kind == "dense":
        out = {"up": (m.ff, W), "down": (W, m.ff)}
        if m.bias:
            out.update({"up.b": (m.ff,), "down.b": (W,)})
        return out
    out = {"router": (m.experts, W)}
    for e in range(m.experts):
        out.update({f"e{e}.up": (m.ff, W), f"e{e}.down": (W, m.ff)})
    return out


def load(m: DenseMlp | ExpertsMlp, t, prefix: str, cfg, device, dtype):
    """t(name, dtype) -> tensor on the device; prefix names the layer."""
    norm32 = padded(t(prefix + "norm2", torch.float32), cfg.width_padded)
    p = prefix + "mlp."
    cls = DenseFf if m.kind == "dense" else ExpertsFf
    return cls.load(m, t, p, norm32, cfg.width_padded, dtype)


def columns(ff: int) -> int:
    """Columns of the activations and of the down weights' rows: whole 128-byte lines where that adds
    little.  Rows that start amid a line cost a product's pieces of them a second line (64 experts 4096
    x 3616, down product of 3 / 16 / 192 rows each 332 / 347 / 524 us, with 3648 columns 284 / 325 /
    458); the columns past the size are zeros that the up and the down products read too."""
    whole = pad_to(ff, 64)
    return whole if whole - ff <= ff // 32 else pad_to(ff, 8)


@dataclass
class DenseFf:
    act: str
    norm: torch.Tensor           # [Wp] storage type
    norm32: torch.Tensor
    up: torch.Tensor             # [FP, Wp], rows past the size zero
    down: torch.Tensor           # [W, FP]
    up_b: torch.Tensor | None    # [FP]
    down_b: torch.Tensor | None  # [W]

    @classmethod
    def load(cls, m: DenseMlp, t, p: str, norm32, Wp: int, dtype) -> "DenseFf":
        FP = columns(m.ff)
        return cls(m.act, norm32.to(dtype), norm32,
                   padded(padded(t(p + "up"), FP, dim=0), Wp, dim=1),
                   padded(t(p + "down"), FP, dim=1),
                   padded(t(p + "up.b"), FP) if m.bias else None,
                   t(p + "down.b").contiguous() if m.bias else None)

    @property
    def act_elems(self) -> int:
        return self.up.shape[0]

    experts = top = 0

    def rows(self, model, x: torch.Tensor, h=None, next_norm=None):
        """h: the norm of x if it is there; returns the norm by next_norm of the new x if it is."""
        h = model.norm_rows(x, self.norm32) if h is None else h
        a = torch.empty((x.shape[0], self.up.shape[0]), device=x.device, dtype=model.dtype)
        model.product_act(h, self.up, a, self.act, self.up_b)
        if next_norm is not None:
            return model.add_norm(a, self.down, x, model.cfg.residual_mult, next_norm, self.down_b)
        model.product_add(a, self.down, x, model.cfg.residual_mult, self.down_b)
        return None

    def decode(self, model, b, x: torch.Tensor) -> None:
        cfg = model.cfg
        a = b.ff[:self.up.shape[0]]
        M.layer_in(x, self.norm, cfg.eps, cfg.norm_offset, model.W, self.up, 0, None, a,
                   ln=cfg.layer_norm, kind=self.act, bias=self.up_b)
        M.layer_out(a, self.down, cfg.residual_mult, x, x, bias=self.down_b)


@dataclass
class ExpertsFf:
    act: str
    top: int
    norm: torch.Tensor           # [Wp] storage type
    norm32: torch.Tensor
    router: torch.Tensor         # [E, Wp]
    up: torch.Tensor             # [E, FP, Wp], rows past the size zero
    down: torch.Tensor           # [E, W, FP]

    @classmethod
    def load(cls, m: ExpertsMlp, t, p: str, norm32, Wp: int, dtype) -> "ExpertsFf":
        FP = columns(m.ff)
        up, down = None, None
        for e in range(m.experts):   # one expert at a time: no second copy of all of them
            u, d = t(f"{p}e{e}.up"), t(f"{p}e{e}.down")
            if up is None:
                up = u.new_zeros((m.experts, FP, Wp))
                down = d.new_zeros((m.experts, d.shape[0], FP))
            up[e, :m.ff, :u.shape[1]] = u
            down[e, :, :m.ff] = d
        return cls(m.act, m.top, norm32.to(dtype), norm32, padded(t(p + "router"), Wp, dim=1), up,
                   down)

    @property
    def experts(self) -> int:
        return self.router.shape[0]

    @property
    def act_elems(self) -> int:
        return self.top * self.up.shape[1]

    def rows(self, model, x: torch.Tensor, h=None, next_norm=None):
        """Router over all rows, then the chosen experts as grouped products over rows sorted by
        expert; a row is normed, scaled by its score and rounded once on its way there.  h: the norm of
        x if it is there; returns the norm by next_norm of the new x if it is."""
        N, M_ = x.shape[0], x.shape[0] * self.top
        E, FP, Wp = self.up.shape
        logits = torch.empty((N, pad_to(E, 4)), device=x.device, dtype=torch.float32)[:, :E]
        model.product(model.norm_rows(x, self.norm32) if h is None else h, self.router, logits)
        p = X.route_plan(logits, self.top, model.dtype, FP * Wp, FP)
        h = model.norm_rows(x, self.norm32, where=p.where, scale=p.scale)
        a = torch.empty((M_, FP), device=x.device, dtype=model.dtype)
        X.product(h, self.up, p, a, self.act)
        W = self.down.shape[1]
        y = torch.empty((M_, pad_to(W, 8)), device=x.device, dtype=model.dtype)
        X.product(a, self.down, p, y[:, :W])
        cfg = model.cfg
        if next_norm is None or model.dtype == torch.float32 or W != x.shape[1] or W > X.SUM_NORM_MAX:
            X.gather_sum(y, p, W, cfg.residual_mult, x)
            return None
        h = torch.empty_like(x, dtype=model.dtype)
        X.gather_sum_norm(y, p, W, cfg.residual_mult, x, next_norm, cfg.norm_offset, cfg.eps, cfg.layer_norm, h)
        return h

    def decode(self, model, b, x: torch.Tensor) -> None:
        cfg = model.cfg
        M.layer_in(x, self.norm, cfg.eps, cfg.norm_offset, model.W, self.router, self.experts,
                   b.route, ln=cfg.layer_norm)
        a = b.ff[:self.act_elems]
        X.up(x, self.norm, cfg.eps, cfg.norm_offset, cfg.layer_norm, model.W, b.route, self.top,
             self.up, self.act, a, b.sel)
        X.down(a, b.sel, self.top, self.down, cfg.residual_mult, x, x)
