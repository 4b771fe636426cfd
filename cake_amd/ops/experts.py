"""Torch-tensor wrappers of the routed-expert kernels (csrc/kernels/mixer_experts.hip and the
grouped GEMM); shapes, dtypes and strides are validated on the host before every launch."""
from __future__ import annotations

import math
from dataclasses import dataclass

import torch

from . import gemm as G
from ._lib import check
from .mixers import ACTS, DT, _lib, _mat, _stream, _vec

MAX_EXPERTS = 1024
MAX_TOP = 32
SUM_NORM_MAX = 8192   # columns of a row that gather_sum_norm holds
PLAN_ENTRIES = 1024   # of a plan that makes its rows' choice
BM32 = 32   # row tile of the f32 grouped product


def _routing(E: int, top: int):
    if not (0 < E <= MAX_EXPERTS and 0 < top <= min(MAX_TOP, E)):
        raise ValueError(f"unsupported routing: {top} of {E} experts")


def route(logits, top: int):
    """Router logits [N, E] f32 -> (expert ids int32 [N, top], sigmoid scores f32 [N, top])."""
    N, E = logits.shape
    _routing(E, top)
    lp, ldl = _mat(logits, "logits", torch.float32, N, E)
    ids = torch.empty((N, top), device=logits.device, dtype=torch.int32)
    score = torch.empty((N, top), device=logits.device, dtype=torch.float32)
    check(_lib().cake_expert_route(lp, max(ldl, E), N, E, top, ids.data_ptr(), score.data_ptr(),
                                   _stream()), "expert_route")
    return ids, score


@dataclass
class Plan:
    """(token, choice) entries sorted by expert, and the row tiles of the grouped products."""
    scale: torch.Tensor   # [M] score of every sorted row
    where: torch.Tensor   # [N, top] sorted row of every entry
    tiles: torch.Tensor   # [n + 1, 4], the last entry their number and height
    cfg: int              # grouped GEMM configuration (16-bit types)

    @property
    def row(self) -> torch.Tensor:
        """[M] token of every sorted row."""
        N, top = self.where.shape
        token = torch.arange(N, dtype=torch.int32, device=self.where.device).repeat_interleave(top)
        return torch.empty_like(token).scatter_(0, self.where.flatten().long(), token)


def _plan(N: int, top: int, E: int, dev, dtype, weight: int, up: int, launch) -> Plan:
    """launch(BM, up, wide, scale, where, tiles, number of tiles) fills the plan."""
    M = N * top
    up = up or math.isqrt(weight or 1 << 22)
    wide = max(1, (weight or 1 << 22) // up)
    cfg = G.grouped_cfg(M, E, torch.cuda.is_current_stream_capturing(), weight, wide)
    bm = BM32 if dtype == torch.float32 else G.GROUPED_CFGS[cfg]   # the least, of a height yet to choose
    n = M // bm + min(E, M)
    i32 = torch.empty(M + 4 * (n + 1) + 4, device=dev, dtype=torch.int32)
    where = i32[:M].view(N, top)
    at = M + -M % 4   # tiles are read whole, 16 bytes each
    tiles = i32[at:at + 4 * (n + 1)].view(n + 1, 4)
    scale = torch.empty(M, device=dev, dtype=torch.float32)
    launch(0 if dtype != torch.float32 and cfg == G.BY_LIST else bm, up, wide,
           scale.data_ptr(), where.data_ptr(), tiles.data_ptr(), n, _stream())
    return Plan(scale, where, tiles, cfg)


def plan(ids, score, E: int, dtype, weight: int = 0, up: int = 0) -> Plan:
    """Rows sorted by expert, and their tiles; weight: elements of an expert's matrix, up: columns of
    its up product (0: a square matrix)."""
    N, top = ids.shape
    _routing(E, top)
    ip, sp = _vec(ids, "ids", torch.int32, N * top), _vec(score, "score", torch.float32, N * top)
    return _plan(N, top, E, ids.device, dtype, weight, up, lambda bm, up, wide, *out: check(
        _lib().cake_expert_plan(ip, sp, N, top, E, bm, up, wide, *out), "expert_plan"))


def route_plan(logits, top: int, dtype, weight: int = 0, up: int = 0) -> Plan:
    """:func:`route` and :func:`plan`; of a few rows in one launch: while a wave has a row, or two
    short ones, that one workgroup is no slower than many."""
    N, E = logits.shape
    _routing(E, top)
    if not 0 < N <= (32 if E <= 64 else 16) or N * top > PLAN_ENTRIES:
        return plan(*route(logits, top), E, dtype, weight, up)
    lp, ldl = _mat(logits, "logits", torch.float32, N, E)
    return _plan(N, top, E, logits.device, dtype, weight, up, lambda bm, up, wide, *out: check(
        _lib().cake_expert_route_plan(lp, max(ldl, E), N, top, E, bm, up, wide, *out), "expert_route_plan"))


def product(x, w, p: Plan, out, act: str | None = None):
    """out[r] = act(x[r] w[expert of sorted row r]^T); w [E, N, K]."""
    E, N, K = w.shape
    if x.dtype != torch.float32:
        return G.grouped(x, w, p.tiles, p.cfg, out, epi=act or "store")
    M = p.where.numel()
    xp, ldx = _mat(x, "x", torch.float32, M, K)
    op, ldo = _mat(out, "out", torch.float32, M, N)
    check(_lib().cake_expert_gemm32(xp, ldx, _vec(w, "w", torch.float32), K, N * K,
                                    p.tiles.data_ptr(), p.tiles.shape[0] - 1, N, K,
                                    -1 if act is None else ACTS[act], op, max(ldo, N), _stream()),
          "expert_gemm32")
    return out


def gather_sum(y, p: Plan, width: int, alpha: float, x):
    """x[n, :width] += alpha * sum over the token's choices of their rows of y."""
    N, top = p.where.shape
    yp, ldy = _mat(y, "y", y.dtype, N * top, width)
    xp, ldx = _mat(x, "x", torch.float32, N, width)
    check(_lib().cake_expert_sum(DT[y.dtype], yp, ldy, p.where.data_ptr(), N, top, int(width),
                                 float(alpha), xp, max(ldx, width), _stream()), "expert_sum")


def gather_sum_norm(y, p: Plan, width: int, alpha: float, x, w, offset: float, eps: float, ln: bool, out):
    """:func:`gather_sum` of 16-bit rows up to 8192 wide (a multiple of 4), and out [N, width] = the norm
    of the new rows (ln: layer norm) times (offset + w [width] f32)."""
    N, top = p.where.shape
    yp, ldy = _mat(y, "y", y.dtype, N * top, width)
    xp, ldx = _mat(x, "x", torch.float32, N, width)
    op, ldo = _mat(out, "out", y.dtype, N, width)
    check(_lib().cake_expert_sum_norm(
        DT[y.dtype], yp, ldy, p.where.data_ptr(), N, top, int(width), float(alpha), xp, max(ldx, width),
        _vec(w, "w", torch.float32, width), float(offset), float(eps), int(ln), op, max(ldo, width), _stream()),
        "expert_sum_norm")


def up(resid, norm_w, eps: float, offset: float, ln: bool, width: int, logits, top: int, w,
       act: str, out, sel):
    """One token: norm, choice by the router logits [E], out [top, FP] = act(score_k W_up[k] x);
    the chosen experts go to sel.  w [E, FP, K] 16-bit."""
    E, FP, K = w.shape
    _routing(E, top)
    check(_lib().cake_expert_up(
        DT[w.dtype], _vec(resid, "resid", torch.float32, K), _vec(norm_w, "norm_w", w.dtype, K),
        float(eps), float(offset), int(ln), int(width), _vec(logits, "logits", torch.float32, E), E,
        top, _vec(w, "w", w.dtype), K, FP, ACTS[act], _vec(out, "out", w.dtype, top * FP),
        _vec(sel, "sel", torch.int32, top), _stream()), "expert_up")


def down(a, sel, top: int, w, alpha: float, x, y):
    """One token: y = x + alpha sum_k W_down[sel_k] a_k; w [E, W, FP] 16-bit, y may be x."""
    E, W, FP = w.shape
    check(_lib().cake_expert_down(
        DT[w.dtype], _vec(a, "a", w.dtype, top * FP), _vec(sel, "sel", torch.int32, top), top,
        _vec(w, "w", w.dtype), E, FP, W, float(alpha), _vec(x, "x", torch.float32, W),
        _vec(y, "y", torch.float32, W), _stream()), "expert_down")
