"""A run of Llama blocks over several rows as one native call (csrc/driver/block_rows.cpp).

:func:`block_rows` checks the tensors and plans the four products once for the whole run, by the
rules of :func:`gemm.linear`; it returns False, with nothing launched, for what only the separate
calls take (a library plan, sizes or layouts outside the kernels' fast forms)."""
from __future__ import annotations

import ctypes as C

import torch

from . import gemm as G
from ._lib import check, current_stream, kernels

P, I, F = C.c_void_p, C.c_int, C.c_float


class _Form(C.Structure):
    _fields_ = [("kind", I), ("cfg", I), ("splits", I), ("slabs", I)]


class _Run(C.Structure):
    _fields_ = [(n, P) for n in ("blocks", "hidden", "x", "qkv", "att", "act", "inv_freq", "zeros",
                                 "ws", "slabs", "rows_ws", "tick")] + \
               [(n, _Form) for n in ("qkv_form", "o_form", "gu_form", "down_form", "kv_form", "q1_form",
                                     "o1_form", "gu1_form", "down1_form")] + \
               [(n, I) for n in ("n", "dt", "T", "H", "I", "nh", "nkv", "hd", "S", "pos0", "tail", "few",
                              "few1")] + \
               [("eps", F), ("scale", F)]


def _forms(products, capturing: bool):
    """(kind, cfg, splits) of each (rows, Nv, K, epi, summed), as gemm.linear chooses them or, of those
    that a sum of slabs may follow, as gemm.slab_form does; the floats that the tile plans' slabs need,
    and those of the products that leave them.  None if one of them is the library GEMM's.  A product may be
    None: it has no form."""
    forms, floats, left = [], 0, 0
    for p in products:
        if p is None:
            forms.append(_Form())
            continue
        T, Nv, K, epi, summed = p
        gated = epi == "swiglu"
        big = max(T, Nv) * K * 2 >= 0x7fffffff
        slab = G.slab_form(T, Nv, K, epi, big) if summed else None
        if slab is not None:
            left = max(left, slab[2] * T * Nv)
            forms.append(_Form(*slab, 1))
            continue
        kind = G.rows_kind(T, Nv, K, gated) if (T, Nv, K, epi) not in G._plans else 0
        if kind == 2 and capturing:
            kind = 0
        cfg, splits = 0, 1
        if not kind:
            cfg, splits = G.resolve(T, Nv, K, epi, big)
            if cfg == G.LIB:
                return None, 0, 0
            if splits > 1:
                floats = max(floats, int(G._lib().cake_gemm_ws_floats(
                    cfg, splits, T, Nv // 2 if gated else Nv, K, int(gated))))
        forms.append(_Form(kind, cfg, splits, 0))
    return forms, floats, left


# A prompt of fewer rows goes through the last block whole: its products read the weights once either way
# and the one row's are a launch more (nine blocks of 1B / 8B / 70B, whole and with one row at the end: 45
# rows 540 / 978 / 2700 us, 544 / 984 / 2699; 80 rows 645 / 1240 / 3328, 642 / 1233 / 3271; 512 rows 1111 /
# 2496 / 7538, 1071 / 2354 / 7023).
TAIL_LEAST = 65
# ... and rows times weights of a block: the tail is five launches more on fewer rows.  Three blocks, whole and with one
# row at the end: 12.8 million weights (1024 wide) at 80 / 200 / 400 rows 128 / 154 / 189 us, 132 / 155 / 184 (one call on an
# idle GPU 176 / 202 / 239, 184 / 206 / 236); 24 million at 80 / 200 146 / 184, 148 / 178 (195 / 233, 205 / 235); 60 million
# at 65 212, 189 (253, 247).
TAIL_WORK = 3.5e9


def takes_tail(T: int, tail: int, weights: int) -> bool:
    """Whether only the tail's rows go through the products behind the last block's keys and values."""
    return 0 < tail * 4 <= T and T >= TAIL_LEAST and T * weights >= TAIL_WORK


def block_rows(hidden: torch.Tensor, blocks: list, slots: list[int], k: torch.Tensor,
               v: torch.Tensor, inv_freq: torch.Tensor, cfg, pos0: int, scale: float,
               tail: int = 0) -> bool:
    """hidden [T, H] f32 through `blocks` in place; k, v [layers, nkv, S, hd], block i's rows at
    slots[i].  tail: only so many of the last rows of the result are wanted (0: all)."""
    T, H = hidden.shape
    nh, nkv, hd = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    inter, S, dt = cfg.intermediate_size, k.shape[2], k.dtype
    nq, nqkv = nh * hd, (nh + 2 * nkv) * hd
    if dt not in G._DT or T < 1 or nh % nkv or hd % 8 or hd > 256 or H % 8 or inter % 16 or \
            not hidden.is_cuda or not hidden.is_contiguous() or hidden.data_ptr() % 16 or \
            not (k.is_contiguous() and v.is_contiguous()) or k.shape != v.shape or \
            v.dtype != dt or tuple(k.shape[1:]) != (nkv, S, hd) or pos0 < 0 or pos0 + T > S or \
            tuple(inv_freq.shape) != (hd // 2,) or inv_freq.dtype != torch.float32 or \
            not inv_freq.is_contiguous():
        return False
    shapes = ((H,), (nqkv, H), (H, nq), (H,), (2 * inter, H), (H, inter))
    kp, vp, step = k.data_ptr(), v.data_ptr(), nkv * S * hd * 2
    table = (P * (8 * len(blocks)))()
    for i, (b, s) in enumerate(zip(blocks, slots)):
        if not 0 <= s < k.shape[0]:
            return False
        ptrs = []
        for t, shape in zip((b.ln1, b.wqkv, b.wo, b.ln2, b.wgu, b.wd), shapes):
            p = t.data_ptr()
            if t.shape != shape or t.dtype != dt or not t.is_contiguous() or not t.is_cuda or \
                    p % 16:
                return False
            ptrs.append(p)
        table[8 * i:8 * i + 8] = [*ptrs, kp + s * step, vp + s * step]
    capturing = torch.cuda.is_current_stream_capturing()
    adds = H <= G.SLAB_NORM_MAX
    nk = nkv * hd
    if not blocks or not takes_tail(T, tail, nqkv * H + H * nq + 3 * inter * H):
        tail = 0

    few, few1 = G.few_pair(T, H, nq, inter), G.few_pair(tail, H, nq, inter)

    def behind(rows, few):   # the products behind the attention
        pair = (None, None) if few else ((rows, H, nq, "resid32", adds), (rows, 2 * inter, H, "swiglu", False))
        return (*pair, (rows, H, inter, "resid32", adds))
    forms, floats, left = _forms(((T, nqkv, H, "store", True), *behind(T, few)) + (() if not tail else (
        (T, 2 * nk, H, "store", False), (tail, nq, H, "store", False), *behind(tail, few1))), capturing)
    if forms is None:
        return False
    if not tail:
        forms += [_Form()] * 5
    dev, st = hidden.device, current_stream()
    x = torch.empty((T, H), device=dev, dtype=dt)
    qkv = torch.empty((T, nqkv), device=dev, dtype=dt)
    att = torch.empty((T, nq), device=dev, dtype=dt)
    act = torch.empty((T, inter), device=dev, dtype=dt)
    ws = G._workspace(dev, floats) if floats else None
    slabs = torch.empty(left, device=dev, dtype=torch.float32) if left else None
    rows_ws = tick = None
    if any(f.kind == 2 and not f.slabs for f in forms):
        rows_ws, tick = G._rows_state(dev, min(T, G.ROWS_MAX), st)
    elif any(f.splits > 1 and f.cfg in G.FOUR_WAVE and not f.slabs for f in forms):
        tick = G._counters(dev, st)
    ptr = [None if t is None else t.data_ptr() for t in (
        hidden, x, qkv, att, act, inv_freq, G._zeros16(dev), ws, slabs, rows_ws, tick)]
    run = _Run(C.addressof(table), *ptr, *forms, len(blocks), G._DT[dt], T, H, inter, nh, nkv, hd, S,
               int(pos0), int(tail), int(few), int(few1), float(cfg.rms_norm_eps), float(scale))
    check(kernels().cake_block_rows(C.addressof(run), st), "block_rows")
    return True
