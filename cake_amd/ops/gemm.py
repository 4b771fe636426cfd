"""Host side of the MFMA GEMM (csrc/kernels/gemm.hip): y = x W^T + fused epilogue.

Every T > 1 linear on the device path goes through :func:`linear`: Llama prefill
q|k|v, o (+residual), gate|up (+SwiGLU), down (+residual); every SD UNet / VAE /
CLIP projection (+bias, +residual, +GEGLU).  Shapes and strides are validated
on the host before launch; there is no library fallback.

Tile choice: products of up to 64 rows take forms of their own (gemm.hip rows_kind); from 65 rows
on, and where a captured graph keeps those out, :func:`resolve` asks the kernel library's fitted
estimate, which a measured entry of the very size (gemm_tuned.json) or a pinned plan
(:func:`set_plan`) goes before.
"""
from __future__ import annotations

import ctypes as C
import threading

import torch

from ._lib import check, current_stream, kernels, library

EPI = {"store": 0, "resid32": 1, "add16": 2, "swiglu": 3, "geglu": 4, "store32": 6, "silu": 7,
       "quick_gelu": 8, "gelu": 9, "relu2": 10}
_DT = {torch.bfloat16: 0, torch.float16: 1}
# (BM, BN) of the kernel's tile configurations (gemm.hip CAKE_GEMM_CFGS)
CFG_TILES = {0: (128, 128), 1: (64, 128), 2: (256, 128), 3: (128, 256), 4: (64, 64),
             5: (256, 256), 6: (256, 128), 7: (128, 128), 8: (128, 128), 11: (256, 256),
             12: (64, 128), 13: (64, 64), 14: (64, 160), 15: (64, 160), 16: (128, 160),
             17: (128, 160), 18: (64, 160), 19: (128, 160), 20: (256, 256), 21: (256, 256),
             22: (256, 256), 23: (256, 192),
             24: (128, 256), 25: (256, 256), 26: (256, 192), 27: (128, 256), 28: (128, 128),
             29: (128, 192), 30: (96, 256), 31: (160, 256), 32: (192, 192), 33: (224, 192),
             34: (192, 256), 35: (224, 256), 36: (160, 192), 37: (160, 128), 38: (224, 128)}
_SLOTS = {0: 2, 1: 2, 2: 1, 3: 1, 4: 4, 5: 1, 6: 1, 7: 1, 8: 2, 11: 1, 12: 2, 13: 2,
          14: 2, 15: 2, 16: 1, 17: 1, 18: 1, 19: 1, 20: 1, 21: 1, 22: 1, 23: 1, 24: 1, 25: 1, 26: 1, 27: 1,
          **dict.fromkeys(range(28, 39), 1)}  # WGs/CU
# 80-column wave tiles (two waves across the 160 columns): no gated epilogue
NO_GATED = {14, 17, 18, 19}
# register-staged / four-wave 256x256 (gemm_rs.h, gemm_4w.h): whole 64-element k steps only
K64_ONLY = set(range(21, 39))
FOUR_WAVE = set(range(22, 39))   # split k in pieces of a tile (gemm_4w.h)
# relative per-tile throughput (measured per-config sweep,
# profiles/r2_gemm_sweep_agpr.jsonl): the AGPR-accumulator 128x128 tile (0) for most
# shapes, the 8-wave 256x256 tile (11) where its tiles fill the chip, 64-wide tiles
# (1, 4) for short M
_EFF = {0: 1.0, 1: 0.8, 2: 0.8, 3: 0.8, 4: 0.7, 5: 1.2, 6: 0.95, 7: 0.9, 8: 0.9, 11: 1.1,
        12: 0.8, 13: 0.7, 14: 0.8, 15: 0.7, 16: 0.9, 17: 0.9, 18: 0.8, 19: 0.9, 20: 1.2, 21: 1.3, 22: 1.3, 23: 1.3, 24: 1.2, 25: 1.3, 26: 1.3, 27: 1.2,
        **dict.fromkeys(range(28, 39), 1.2)}
NUM_CUS = 256
# plan cfg of the library GEMM (hipBLASLt, csrc/driver/blaslt.cpp), kept as the A/B arm of
# scripts/bench_gemm_lib.py: off the default path (table entries naming it are read only
# under CAKE_GEMM_LIB=1, or when a caller passes cfg=LIB); epilogues it can carry: plain
# store, f32 store / accumulate (beta 1), and SwiGLU as library GEMM + silu_mul_rows
LIB = -1
LIB_EPIS = ("store", "resid32", "store32", "swiglu")
_LIB_WS_BYTES = 32 << 20
_bound = False
_plans: dict = {}
_ws: dict = {}            # (device, stream) -> split-K slabs, newest last
_ticks: dict = {}         # (device, stream) -> arrival counters, newest last
_graph_ticks: dict = {}   # (device, stream) -> (capture, counters) of its latest capture
_lock = threading.RLock()
_zeros: dict = {}


def _lib():
    """The GEMM library (libcake_gemm.so)."""
    global _bound
    lib = library("gemm")
    if not _bound:
        P, I, L = C.c_void_p, C.c_int, C.c_longlong
        lib.cake_gemm_scaled.argtypes = [I, I, I, I, P, L, P, L, P, L, P, P, L, P, P, P, I, I, I,
                                         C.c_float, P]
        lib.cake_gemm_scaled.restype = I
        lib.cake_gemm_ticks.argtypes = []
        lib.cake_gemm_ticks.restype = I
        lib.cake_stream_capture.argtypes = [P]
        lib.cake_stream_capture.restype = L
        lib.cake_gemm_ws_floats.argtypes = [I, I, I, I, I, I]
        lib.cake_gemm_ws_floats.restype = L
        lib.cake_gemm_grouped.argtypes = [I, I, I, P, L, P, L, L, P, L, P, I, P, I, I, P]
        lib.cake_gemm_grouped.restype = I
        lib.cake_gemm_plan.argtypes = [I, L, I, I, I, P, P]
        lib.cake_gemm_plan.restype = I
        lib.cake_gemm_rows_kind.argtypes = [I, L, I, I]
        lib.cake_gemm_rows_kind.restype = I
        lib.cake_gemm_rows_ws_floats.argtypes = [I]
        lib.cake_gemm_rows_ws_floats.restype = L
        lib.cake_gemm_rows_ticks.argtypes = []
        lib.cake_gemm_rows_ticks.restype = I
        lib.cake_gemm_rows.argtypes = [I, I, I, P, L, P, L, P, L, P, P, L, P, P, P, I, I, I,
                                       C.c_float, P]
        lib.cake_gemm_rows.restype = I
        lib.cake_gemm_slab_plan.argtypes = [I, L, I, I, I, P, P, P]
        lib.cake_gemm_slab_plan.restype = I
        lib.cake_gemm_slabs.argtypes = [I, I, I, I, P, L, P, L, P, P, I, I, I, P]
        lib.cake_gemm_slabs.restype = I
        lib.cake_slab_norm.argtypes = [I, P, I, P, L, P, C.c_float, P, I, C.c_float, C.c_float, I, I,
                                       I, P, L, P]
        lib.cake_slab_norm.restype = I
        lib.cake_slab_rope.argtypes = [I, P, I, P, I, I, I, I, I, P, I, I, P, P, P]
        lib.cake_slab_rope.restype = I
        lib.cake_slab_attn.argtypes = [I, P, I, P, L, I, I, I, I, P, I, P, P, C.c_float, P]
        lib.cake_slab_attn.restype = I
        lib.cake_gemm_few_pair.argtypes = [I, I, I, L]
        lib.cake_gemm_few_pair.restype = I
        lib.cake_gemm_few_add.argtypes = [I, P, L, P, L, P, L, I, I, I, P]
        lib.cake_gemm_few_add.restype = I
        lib.cake_gemm_few_gated.argtypes = [I, P, L, P, C.c_float, P, L, P, L, I, I, I, P]
        lib.cake_gemm_few_gated.restype = I
        lib.cake_gemm_sections_gain.argtypes = [I, I, I, I, I]
        lib.cake_gemm_sections_gain.restype = I
        lib.cake_gemm_rows_sections.argtypes = [I, P, L, P, L, P, L, P, L, P, L, I, I, P, P, P, I, I,
                                                I, P]
        lib.cake_gemm_rows_sections.restype = I
        lib.cake_gemm_rows_grouped.argtypes = [I, I, P, L, P, L, L, P, L, P, I, P, P, P, I, I, P]
        lib.cake_gemm_rows_grouped.restype = I
        _bound = True
    return lib


def _lib_blaslt():
    """The library GEMM's entry point (csrc/driver/blaslt.cpp, in libcake_kernels.so)."""
    fn = kernels().cake_blaslt_gemm
    if fn.argtypes is None:
        P, I, L = C.c_void_p, C.c_int, C.c_longlong
        fn.argtypes = [I, I, P, L, P, L, P, L, I, I, I, P, C.c_size_t, P]
        fn.restype = I
    return fn


def _zeros16(dev) -> torch.Tensor:
    z = _zeros.get(dev)
    if z is None:
        z = _zeros[dev] = torch.zeros(64, dtype=torch.int32, device=dev)
    return z


def _newest(table: dict, key, value) -> None:
    """table[key] = value, of the 16 newest streams (memory of the others is freed in the order of
    its own stream)."""
    table.pop(key, None)
    while len(table) >= 16:
        table.pop(next(iter(table)))
    table[key] = value


def _workspace(dev, numel: int) -> torch.Tensor:
    """Split-K slabs of one launch on the current stream: the stream's own (launches on two streams
    may run side by side).  Under capture the graph's own, of its memory pool: graphs share a
    capture stream and may be replayed side by side."""
    if torch.cuda.is_current_stream_capturing():
        return torch.empty(numel, dtype=torch.float32, device=dev)
    key = (dev, torch.cuda.current_stream(dev).cuda_stream)
    w = _ws.get(key)
    if w is None or w.numel() < numel or len(_ws) >= 16:
        with _lock:
            if w is None or w.numel() < numel:
                w = torch.empty(max(numel, 1 << 20), dtype=torch.float32, device=dev)
            _newest(_ws, key, w)
    return w


ROWS_MAX = 64   # rows that the products of few rows take at most
_rows_kinds: dict = {}
_rows_floats: dict = {}   # rows -> workspace floats of the stream form


def rows_kind(M: int, Nv: int, K: int, gated: bool) -> int:
    """Form of a product of M rows (gemm.hip rows_kind): 0 tile kernels, 1 direct, 2 stream."""
    if M > ROWS_MAX:
        return 0
    key = (M, Nv, K, gated)
    kind = _rows_kinds.get(key)
    if kind is None:
        kind = _rows_kinds[key] = int(_lib().cake_gemm_rows_kind(M, Nv, K, int(gated)))
    return kind


SLAB_NORM_MAX = 8192   # columns of a row that slab_norm holds
_slab_forms: dict = {}


def slab_form(M: int, N: int, K: int, epi: str, big: bool = False):
    """(kind, cfg, parts) of a product that leaves its sums in `parts` slabs or fewer for the launch
    behind it (gemm.hip cake_gemm_slab_plan), or None: the product as :func:`linear` runs it with `epi`,
    a launch of its own behind it.  Pinned plans run as pinned, the library's as its own.  A measured
    plan is one of a product alone: with what follows, slabs take 0.83 of its time (46 sizes of the table,
    32 .. 2048 rows, 0.40 to 0.99)."""
    if (M, N, K, epi) in _plans or N % 4 or K % 8:
        return None
    key = (M, N, K, epi, big)
    f = _slab_forms.get(key, 0)
    if f == 0:
        if len(_slab_forms) >= 65536:
            _slab_forms.clear()
        k, c, p = C.c_int(0), C.c_int(0), C.c_int(1)
        on = (rows_kind(M, N, K, False) or resolve(M, N, K, epi, big)[0] != LIB) and \
            _lib().cake_gemm_slab_plan(M, N, K, EPI[epi], int(big), C.addressof(k), C.addressof(c),
                                       C.addressof(p))
        f = _slab_forms[key] = (k.value, c.value, p.value) if on else None
    return f


def few_pair(M: int, H: int, K: int, inter: int) -> bool:
    """Whether a block's output product (rows of K to H, added to the residual rows) and its gated product of the
    normed rows (H to `inter`) run as :func:`few_add` and :func:`few_gated` (gemm_few.hip); pinned plans run as pinned,
    the library's as its own."""
    both = ((M, H, K, "resid32"), (M, 2 * inter, H, "swiglu"))
    return not any(p in _plans for p in both) and bool(_lib().cake_gemm_few_pair(M, H, K, inter)) and \
        all(rows_kind(m, n, k, e == "swiglu") or resolve(m, n, k, e)[0] != LIB for m, n, k, e in both)


def few_add(x: torch.Tensor, w: torch.Tensor, resid: torch.Tensor) -> None:
    """resid [M, N] f32 += x [M, K] w^T of up to eight rows."""
    (M, K), N = x.shape, w.shape[0]
    if x.dtype not in _DT or w.dtype != x.dtype or resid.dtype != torch.float32 or w.shape[1] != K or \
            tuple(resid.shape) != (M, N) or x.stride(1) != 1 or w.stride(1) != 1 or resid.stride(1) != 1:
        raise ValueError("few_add: 16-bit rows and weights, f32 sums of their shapes expected")
    check(_lib().cake_gemm_few_add(_DT[x.dtype], x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0),
                                   resid.data_ptr(), resid.stride(0), M, N, K, current_stream()), "few_add")


def few_gated(h: torch.Tensor, ln: torch.Tensor, eps: float, w: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    """out [M, N] = silu(x w[:N]^T) (x w[N:]^T), x the RMS norm of h [M, K] f32 with weights ln, of up to eight rows."""
    (M, K), N = h.shape, w.shape[0] // 2
    if w.dtype not in _DT or ln.dtype != w.dtype or out.dtype != w.dtype or h.dtype != torch.float32 or \
            tuple(w.shape) != (2 * N, K) or tuple(ln.shape) != (K,) or tuple(out.shape) != (M, N) or \
            h.stride(1) != 1 or w.stride(1) != 1 or out.stride(1) != 1 or not ln.is_contiguous():
        raise ValueError("few_gated: f32 rows, 16-bit weights and output of their shapes expected")
    check(_lib().cake_gemm_few_gated(_DT[w.dtype], h.data_ptr(), h.stride(0), ln.data_ptr(), float(eps),
                                     w.data_ptr(), w.stride(0), out.data_ptr(), out.stride(0), M, N, K,
                                     current_stream()), "few_gated")
    return out


def _counters(dev, st: int) -> torch.Tensor:
    """Arrival counters of a launch on stream `st`, the current one: zero between launches.
    Launches of one stream run one after the other and share them; launches that may run side by
    side never do.  A captured graph may run beside any stream, so its counters are its own: memory
    of its pool, cleared by a fill at the head of every replay, as long-lived as the graph, and no more than
    tiles in pieces need: the stream form stays out of graphs."""
    if not torch.cuda.is_current_stream_capturing():
        return _stream_counters(dev, st)
    capture = _lib().cake_stream_capture(st)
    if capture <= 0:
        raise RuntimeError("gemm: the capture of the current stream is not to be told")
    with _lock:
        have = _graph_ticks.get((dev, st))
        if have is None or have[0] != capture:
            have = (capture, torch.zeros(_lib().cake_gemm_ticks(), dtype=torch.int32, device=dev))
            _newest(_graph_ticks, (dev, st), have)
        return have[1]


def _stream_counters(dev, st: int) -> torch.Tensor:
    """:func:`_counters` outside of captures."""
    t = _ticks.get((dev, st))
    if t is None or len(_ticks) >= 16:
        with _lock:
            if t is None:
                t = torch.zeros(_n_ticks(), dtype=torch.int32, device=dev)
            _newest(_ticks, (dev, st), t)
    return t


def _n_ticks() -> int:
    return max(_lib().cake_gemm_rows_ticks(), _lib().cake_gemm_ticks())


def _rows_state(dev, M: int, st: int):
    """(workspace, counters) of one launch of the stream form, which graphs do not hold."""
    n = _rows_floats.get(M)
    if n is None:
        n = _rows_floats[M] = int(_lib().cake_gemm_rows_ws_floats(M))
    return torch.empty(n, dtype=torch.float32, device=dev), _stream_counters(dev, st)


def _load_tuned() -> list:
    """Measured best (cfg, split-K) per model shape (gemm_tuned.json, written by
    scripts/gemm_tune_table.py from a bench_gemm.py --sweep on an MI355X)."""
    import json
    import os
    p = os.environ.get("CAKE_GEMM_TABLE") or os.path.join(
        os.path.dirname(os.path.abspath(__file__)), "gemm_tuned.json")
    lib_ok = os.environ.get("CAKE_GEMM_LIB") == "1"
    try:
        with open(p) as f:
            return [e for e in json.load(f)["entries"]
                    if e["cfg"] in CFG_TILES
                    or (lib_ok and e["cfg"] == LIB and e["epi"] in LIB_EPIS)]
    except (OSError, ValueError, KeyError):
        return []


_TUNED = _load_tuned()


def _near_splits(splits: int, m_near: int, M: int) -> int:
    """Split-K of a measured neighbour scaled to this M (the split fills the grid the
    neighbour's M left short: twice the rows, half the splits), a power of two >= 1."""
    s = splits * m_near // max(M, 1)
    p = 1
    while p * 2 <= s:
        p *= 2
    return p


def _tuned(M: int, Nv: int, K: int, epi: str):
    """Exact measured shape, else the same (Nv, K, epilogue) measured at the nearest M
    within 2x (its tile config, split-K scaled to this M)."""
    near = None
    for e in _TUNED:
        if e["Nv"] != Nv or e["K"] != K or e["epi"] != epi:
            continue
        if e["M"] == M:
            return e["cfg"], e["splits"]
        r = max(M, e["M"]) / min(M, e["M"])
        if r <= 2 and (near is None or r < near[0]):
            near = (r, e)
    if near is None:
        return None
    e = near[1]
    return e["cfg"], (1 if e["cfg"] == LIB else _near_splits(e["splits"], e["M"], M))


def set_plan(M: int, N: int, K: int, epi: str, cfg: int, splits: int) -> None:
    """Pin the tile configuration / split-K of one shape (measured tuning)."""
    _plans[(M, N, K, epi)] = (cfg, splits)


def plan(M: int, Nv: int, K: int, epi: str = "store") -> tuple[int, int]:
    """(cfg, splits) by the measured table and its neighbours (Nv = weight rows read): the split
    of a call that names its tile; :func:`resolve` plans the others."""
    p = _plans.get((M, Nv, K, epi))
    if p is not None:
        return p
    p = _tuned(M, Nv, K, epi)
    return p if p is not None else _cost_plan(M, Nv, K)


def resolve(M: int, Nv: int, K: int, epi: str, big: bool = False,
            mfma_only: bool = False) -> tuple[int, int]:
    """(cfg, splits) that :func:`linear` runs: a pinned plan, the measured one of this very size
    unless the kernel library's estimate puts it well behind, else the estimate's best
    (gemm.hip cake_gemm_plan, shared with the native engines).  big: an operand of 2 GB or more;
    mfma_only: as if no plan named the library GEMM."""
    p = _plans.get((M, Nv, K, epi))
    if p is not None and not (mfma_only and p[0] == LIB):
        return p
    key = (M, Nv, K, epi, big, mfma_only)
    p = _resolved.get(key)
    if p is None:
        if len(_resolved) >= 65536:   # as many sizes as a long-lived server meets
            _resolved.clear()
        e = next((e for e in _TUNED if e["M"] == M and e["Nv"] == Nv and e["K"] == K
                  and e["epi"] == epi and not (mfma_only and e["cfg"] == LIB)), None)
        cfg, sp = C.c_int(-1 if e is None else e["cfg"]), C.c_int(1 if e is None else e["splits"])
        if cfg.value == LIB and e is not None:
            p = (LIB, 1)
        else:
            check(_lib().cake_gemm_plan(M, Nv, K, EPI[epi], int(big), C.addressof(cfg),
                                        C.addressof(sp)), "gemm_plan")
            p = (cfg.value, sp.value)
        _resolved[key] = p
    return p


_resolved: dict = {}


def _cost_plan(M: int, Nv: int, K: int) -> tuple[int, int]:
    """The MFMA kernel's (cfg, splits) by the cost model."""
    best = None
    ksteps = -(-K // 64)
    cands = (1, 4, 0) if M <= 64 else (0, 1, 4, 5)
    # the four-wave 256x256 tile where it can run (whole 64-element k steps, operands under
    # 2 GB); unsplit (its split-2 form is the shape-specific remainder pair)
    four = M > 64 and K % 64 == 0 and M * K * 2 < 2 ** 31 and Nv * K * 2 < 2 ** 31
    if four:
        cands = cands + (22,)
    for cfg in cands:
        bm, bn = CFG_TILES[cfg]
        tiles = -(-M // bm) * -(-Nv // bn)
        for splits in (1, 2, 4, 8, 16):
            if splits > 1 and (cfg == 22 or ksteps // splits < 4 or
                               tiles * splits > 2 * NUM_CUS * _SLOTS[cfg]):
                continue
            waves = -(-tiles * splits // (NUM_CUS * _SLOTS[cfg]))
            cost = waves * _SLOTS[cfg] * bm * bn * (-(-ksteps // splits)) / _EFF[cfg]
            cost += (splits > 1) * M * Nv * splits * 0.1   # slab round trip + finalize
            if best is None or cost < best[0]:
                best = (cost, cfg, splits)
    return best[1], best[2]


def _rows_view(t: torch.Tensor, name: str) -> tuple[torch.Tensor, int]:
    """[..., C] tensor with unit column stride -> ([R, C] VIEW of it, row stride)."""
    if t.dim() < 2:
        t = t.view(1, -1)
    if t.stride(-1) != 1:
        raise ValueError(f"{name}: needs unit column stride")
    if t.dim() > 2:
        try:
            t2 = t.view(-1, t.shape[-1])   # never a copy: outputs are written through it
        except RuntimeError:
            raise ValueError(f"{name}: leading dims do not flatten to one row stride") from None
    else:
        t2 = t
    if t2.dim() == 2 and t2.shape[0] > 1 and t2.stride(0) < t2.shape[1]:
        raise ValueError(f"{name}: overlapping rows")
    return t2, (t2.stride(0) if t2.shape[0] > 1 else t2.shape[1])


def linear(x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None, *,
           epi: str = "store", out: torch.Tensor | None = None,
           resid: torch.Tensor | None = None, cfg: int | None = None,
           splits: int | None = None, alpha: float = 1.0) -> torch.Tensor:
    """y = epilogue(x @ w.T) on MFMA.

    x [..., K] (16-bit, unit column stride, any row stride that is a multiple of
    8); w [N, K] ([2F, K] for the gated epilogues: rows [0, F) gate/h, [F, 2F)
    up/gate).  Epilogues:
      store   -> out [..., N] = y (+ bias)
      resid32 -> resid (f32 [..., N]) += alpha * (y (+ bias)); returns resid
      add16   -> out = y (+ bias) + resid (16-bit [..., N])
      swiglu  -> out [..., F] = silu(y_gate) * y_up
      geglu   -> out [..., F] = (y_h + b_h) * gelu_tanh(y_gate + b_gate)
      store32 -> resid (f32 [..., N], any row stride) = alpha * (y (+ bias)); returns resid
      silu    -> out = silu(y (+ bias))
      quick_gelu / gelu -> out = act(y (+ bias)) (CLIP MLP: x*sigmoid(1.702x) / erf GELU)
      relu2   -> out = max(y (+ bias), 0)^2
    """
    if epi not in EPI:
        raise ValueError(f"unknown epilogue {epi}")
    if not (x.is_cuda and w.is_cuda) or x.dtype not in _DT or w.dtype != x.dtype:
        raise TypeError("gemm.linear: 16-bit device tensors of one dtype expected")
    lead = x.shape[:-1]
    K = x.shape[-1]
    if x.dim() > 2 and x.stride(-1) == 1:
        try:
            x.view(-1, K)
        except RuntimeError:
            x = x.contiguous()
    x2, lda = _rows_view(x, "x")
    M = x2.shape[0]
    if w.dim() != 2 or w.shape[1] != K or w.stride(1) != 1:
        raise ValueError(f"gemm.linear: weight {tuple(w.shape)} does not match K={K}")
    ldb = w.stride(0)
    gated = epi in ("swiglu", "geglu")
    Nv = w.shape[0]
    if gated and Nv % 32:
        raise ValueError("gated epilogue needs 2F weight rows with F % 16 == 0")
    N = Nv // 2 if gated else Nv
    if K % 8 or lda % 8 or ldb % 8 or x2.data_ptr() % 16 or w.data_ptr() % 16:
        raise ValueError("gemm.linear: K, row strides must be multiples of 8 and bases 16-byte "
                         "aligned")
    if bias is not None:
        if not (bias.is_cuda and bias.dtype == x.dtype and bias.is_contiguous()
                and bias.numel() == Nv):
            raise ValueError(f"gemm.linear: bias must be a contiguous {x.dtype} [{Nv}] tensor")
    ldr = 0
    rptr = None
    if epi in ("resid32", "store32"):
        if resid is None or resid.dtype != torch.float32 or not resid.is_cuda:
            raise ValueError(f"{epi} needs an f32 device output/residual")
        r2, ldr = _rows_view(resid, "resid")
        if tuple(r2.shape) != (M, N):
            raise ValueError(f"resid shape {tuple(resid.shape)} != {(M, N)}")
        rptr = r2.data_ptr()
    elif epi == "add16":
        if resid is None or resid.dtype != x.dtype or not resid.is_cuda:
            raise ValueError("add16 needs a 16-bit device residual")
        r2, ldr = _rows_view(resid, "resid")
        if tuple(r2.shape) != (M, N):
            raise ValueError(f"resid shape {tuple(resid.shape)} != {(M, N)}")
        rptr = r2.data_ptr()
    if epi in ("resid32", "store32"):
        out2, ldc, cptr = None, 0, None
    else:
        if out is None:
            out = torch.empty(*lead, N, device=x.device, dtype=x.dtype)
        if out.dtype != x.dtype or not out.is_cuda:
            raise ValueError("out dtype/device mismatch")
        out2, ldc = _rows_view(out, "out")
        if tuple(out2.shape) != (M, N):
            raise ValueError(f"out shape {tuple(out.shape)} != {(M, N)}")
        cptr = out2.data_ptr()
    f32_out = epi in ("resid32", "store32")
    if M == 0:
        return resid if f32_out else out
    if alpha != 1.0 and not f32_out:
        raise ValueError(f"{epi} takes no alpha")
    if cfg is None and splits is None and M <= ROWS_MAX and (M, Nv, K, epi) not in _plans:
        kind = rows_kind(M, Nv, K, gated)
        if kind == 2 and torch.cuda.is_current_stream_capturing():
            kind = 0
        if kind:
            st = current_stream()
            ws, tick = _rows_state(x.device, M, st) if kind == 2 else (None, None)
            check(_lib().cake_gemm_rows(
                _DT[x.dtype], EPI[epi], kind, x2.data_ptr(), lda, w.data_ptr(), ldb, cptr, ldc,
                None if bias is None else bias.data_ptr(), rptr, ldr,
                None if ws is None else ws.data_ptr(), None if tick is None else tick.data_ptr(),
                _zeros16(x.device).data_ptr(), M, N, K, float(alpha), st), "gemm_rows")
            return resid if f32_out else out
    s0 = 1
    big = max((M - 1) * lda + K, (Nv - 1) * ldb + K) * 2 >= 0x7fffffff
    if cfg is None:
        cfg, s0 = resolve(M, Nv, K, epi, big)
    elif splits is None:
        s0 = plan(M, Nv, K, epi)[1]
    lib_ok = epi != "swiglu" or (ldc == N and N % 8 == 0 and out2.data_ptr() % 16 == 0)
    if cfg == LIB and bias is None and epi in LIB_EPIS and lib_ok and alpha == 1.0:
        _lib_gemm(x2, lda, w, ldb, epi, out2, ldc, r2 if f32_out else None, ldr, M, N, K)
        return resid if f32_out else out
    if cfg == LIB:  # an epilogue / bias / strided output the library form does not carry
        cfg, s0 = resolve(M, Nv, K, epi, big, mfma_only=True)
    splits = s0 if splits is None else max(1, int(splits))
    # the kernel library sizes it (pieces of a tile need their slabs only)
    st = current_stream()
    tick = _counters(x.device, st) if splits > 1 and cfg in FOUR_WAVE else None
    ws = _workspace(x.device, int(_lib().cake_gemm_ws_floats(
        int(cfg), int(splits), M, N, K, 1 if Nv != N else 0))) if splits > 1 else None
    check(_lib().cake_gemm_scaled(
        _DT[x.dtype], EPI[epi], int(cfg), int(splits), x2.data_ptr(), lda, w.data_ptr(), ldb, cptr,
        ldc, None if bias is None else bias.data_ptr(), rptr, ldr,
        None if ws is None else ws.data_ptr(), None if tick is None else tick.data_ptr(),
        _zeros16(x.device).data_ptr(), M, N, K, float(alpha), st), "gemm")
    return resid if f32_out else out


def sections(x: torch.Tensor, w: torch.Tensor, n1: int, n2: int, out16, out32, act) -> bool:
    """x [M, K] w [N, K]^T of few rows as one launch: columns [0, n1) to out16 (storage type), [n1, n2)
    to out32 (f32), the others through the erf GELU to act; matrices with row strides, None where a
    section is empty.  False, with nothing launched, where the stream form is not the product's, the products
    are better off by themselves (gemm.hip cake_gemm_sections_gain) or the plan of one is pinned."""
    (M, K), N = x.shape, w.shape[0]
    if _plans and any((M, n, K, e) in _plans for n, e in
                      ((n1, "store"), (n2 - n1, "store32"), (N - n2, "gelu"))):
        return False
    if M > ROWS_MAX or x.dtype not in _DT or n1 % 4 or n2 % 4 or K % 8 or \
            rows_kind(M, N, K, False) != 2 or not _lib().cake_gemm_sections_gain(M, n1, n2, N, K) or \
            torch.cuda.is_current_stream_capturing():
        return False
    ptrs, lds = [], []
    for t, n, dt in ((out16, n1, x.dtype), (out32, n2 - n1, torch.float32), (act, N - n2, x.dtype)):
        if n == 0:
            ptrs.append(None)
            lds.append(0)
            continue
        if t.dtype != dt or tuple(t.shape) != (M, n) or t.stride(1) != 1:
            raise ValueError(f"sections: {dt} [{M}, {n}] expected")
        ptrs.append(t.data_ptr())
        lds.append(t.stride(0) if M > 1 else n)
    if x.stride(1) != 1 or w.stride(1) != 1 or w.shape[1] != K or w.dtype != x.dtype:
        raise ValueError("sections: matrices of one 16-bit type expected")
    lda = x.stride(0) if M > 1 else K
    if lda % 8 or w.stride(0) % 8 or any((p or 0) % 16 for p in (x.data_ptr(), w.data_ptr(), *ptrs)):
        return False
    st = current_stream()
    ws, tick = _rows_state(x.device, M, st)
    check(_lib().cake_gemm_rows_sections(
        _DT[x.dtype], x.data_ptr(), lda, w.data_ptr(), w.stride(0), ptrs[0], lds[0], ptrs[1], lds[1], ptrs[2],
        lds[2], n1, n2, ws.data_ptr(), tick.data_ptr(), _zeros16(x.device).data_ptr(), M, N, K, st),
        "gemm_rows_sections")
    return True


def slabs(x: torch.Tensor, w: torch.Tensor, form) -> tuple[torch.Tensor, int]:
    """x [M, K] w [N, K]^T as f32 slabs [n, M, N] of a workspace, form of :func:`slab_form`: (slabs, n)
    for :func:`slab_norm` or :func:`slab_rope`."""
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1] or x.stride(1) != 1 or \
            w.stride(1) != 1 or x.dtype not in _DT or w.dtype != x.dtype or not (x.is_cuda and w.is_cuda):
        raise TypeError("gemm.slabs: 16-bit device matrices of one dtype expected")
    (M, K), N = x.shape, w.shape[0]
    lda = x.stride(0) if M > 1 else K
    if lda < K or lda % 8 or w.stride(0) % 8 or x.data_ptr() % 16 or w.data_ptr() % 16:
        raise ValueError("gemm.slabs: rows of a multiple of 8 on 16-byte boundaries")
    kind, cfg, parts = form
    ws = torch.empty(parts * M * N, device=x.device, dtype=torch.float32)
    n = _lib().cake_gemm_slabs(_DT[x.dtype], kind, cfg, parts, x.data_ptr(), lda, w.data_ptr(), w.stride(0),
                               ws.data_ptr(), _zeros16(x.device).data_ptr(), M, N, K, current_stream())
    check(max(0, -n), "gemm_slabs")
    return ws, n


def slab_norm(ws, n: int, x: torch.Tensor, w, eps: float, out, *, bias=None, alpha: float = 1.0,
              offset: float = 0.0, ln: bool = False) -> None:
    """x [M, >= N] f32 [:, :N] += alpha (the sum of n slabs + bias [N]); then, with w [N] (f32 or the
    storage type), out [M, N] = the RMS norm (ln: layer norm) of that times (offset + w).  n 0: of x as
    it is.  out None: 16-bit type of w, no norm."""
    N = (w if out is None else out).shape[-1]
    M, t = x.shape[0], w if out is None else out
    if x.dtype != torch.float32 or x.stride(1) != 1 or t.dtype not in _DT or not x.is_cuda or \
            x.shape[1] < N or (n and ws.numel() < n * M * N) or (bias is not None and (
                bias.dtype != t.dtype or bias.numel() != N or not bias.is_contiguous())):
        raise ValueError("slab_norm: f32 rows, 16-bit output and bias expected")
    ld = 0
    if out is not None:
        ld = out.stride(0) if M > 1 else N
        if out.shape[0] != M or out.stride(1) != 1 or w.numel() < N or not w.is_contiguous() or \
                w.dtype not in (torch.float32, out.dtype):
            raise ValueError("slab_norm: norm weights of the output's columns expected")
    check(_lib().cake_slab_norm(
        _DT[t.dtype], ws.data_ptr() if n else None, n, x.data_ptr(), x.stride(0) if M > 1 else x.shape[1],
        None if bias is None else bias.data_ptr(), float(alpha), None if out is None else w.data_ptr(),
        int(w.dtype == torch.float32), float(offset), float(eps), int(ln), M, N,
        None if out is None else out.data_ptr(), ld, current_stream()), "slab_norm")


def slab_rope(ws, n: int, q: torch.Tensor, heads: int, inv_freq, pos0: int, kc, vc) -> None:
    """hip.rope_kv of rows that are sums of n slabs [T, (heads + 2 nkv) hd]: rotated queries to q
    [T, >= heads hd], keys and values to rows pos0 .. of kc, vc [nkv, S, hd]."""
    T, (nkv, S, hd) = q.shape[0], kc.shape
    if q.dtype not in _DT or kc.dtype != q.dtype or vc.dtype != q.dtype or q.stride(1) != 1 or \
            q.shape[1] < heads * hd or not (kc.is_contiguous() and vc.is_contiguous()) or \
            vc.shape != kc.shape or ws.numel() < n * T * (heads + 2 * nkv) * hd or \
            inv_freq.dtype != torch.float32 or inv_freq.numel() != hd // 2:
        raise ValueError("slab_rope: 16-bit rows and caches of one dtype expected")
    check(_lib().cake_slab_rope(_DT[q.dtype], ws.data_ptr(), n, q.data_ptr(),
                                q.stride(0) if T > 1 else q.shape[1], T, heads, nkv, hd, inv_freq.data_ptr(),
                                int(pos0), S, kc.data_ptr(), vc.data_ptr(), current_stream()), "slab_rope")


def slab_attn_ok(T: int, pos0: int, hd: int) -> bool:
    """Rows that :func:`slab_attn` takes: a prompt's first ones."""
    return pos0 == 0 and T <= ROWS_MAX and hd in (64, 128)


def slab_attn(ws, n: int, out: torch.Tensor, heads: int, inv_freq, kc, vc, scale: float) -> None:
    """:func:`slab_rope` of a prompt's first rows (position 0 on), and their causal attention to out
    [T, >= heads hd]."""
    T, (nkv, S, hd) = out.shape[0], kc.shape
    if out.dtype not in _DT or kc.dtype != out.dtype or vc.dtype != out.dtype or out.stride(1) != 1 or \
            out.shape[1] < heads * hd or not (kc.is_contiguous() and vc.is_contiguous()) or \
            vc.shape != kc.shape or ws.numel() < n * T * (heads + 2 * nkv) * hd or \
            inv_freq.dtype != torch.float32 or inv_freq.numel() != hd // 2:
        raise ValueError("slab_attn: 16-bit rows and caches of one dtype expected")
    check(_lib().cake_slab_attn(_DT[out.dtype], ws.data_ptr(), n, out.data_ptr(),
                                out.stride(0) if T > 1 else out.shape[1], T, heads, nkv, hd,
                                inv_freq.data_ptr(), S, kc.data_ptr(), vc.data_ptr(), float(scale),
                                current_stream()), "slab_attn")


# tile configuration of a grouped product -> its rows (ROWS: the stream form; BY_LIST: 128 to 256,
# as the last entry of the tile list says: chosen on the device from the groups' sizes)
ROWS, BY_LIST = 32, 6
GROUPED_CFGS = {0: 128, 1: 160, 2: 192, 3: 224, 4: 64, 5: 256, BY_LIST: 128, ROWS: 16}


def grouped_cfg(rows: int, groups: int, capturing: bool = False, weight: int = 0, width: int = 0) -> int:
    """Tile configuration for `rows` sorted rows over `groups` weight groups of `weight` elements each
    (0: small), `width` columns of the rows (0: few)."""
    mean = rows / groups
    if mean <= 4 and not capturing:   # the stream form's counters stay out of graphs
        return ROWS
    if width > 1024:
        # up and down product, us in the stream form and at 64 / 128 rows a tile (gemm_ws.h's), by rows an expert: 64 of 3648 x
        # 4096 4 564 / 627 / 560, 8 595 / 656 / 584, 16 881 / 674 / 600, 48 2067 / 766 / 656; of 1856 x 2048 4 156 / 197 / 154, 8
        # 164 / 208 / 160, 16 243 / 212 / 164; 128 of 768 x 2048 8 135 / 183 / 158, 12 154 / 185 / 159, 16 215 / 189 / 162; 8 of
        # 2048 x 4096 8 55 / 91 / 71, 16 80 / 91 / 71; 32 of 1024 x 2048 8 50 / 67 / 60, 12 67 / 68 / 60
        if mean <= 8 and not capturing and groups * weight < 220_000_000:
            return ROWS
        return 0 if mean < 64 else BY_LIST
    # rows of up to 1024 columns are on 64-row tiles or gemm_4w.h's: the smaller make twice the workgroups.  One product at 14
    # rows, 64 / 128 rows a tile, by millions of weights in all: 17 14.4 / 17.6 (8 of 1024 x 2048 24.4 /
    # 29.3), 34 18.5 / 20.3, 101 47.6 / 50.1, 215 equal, 268 128.6 / 128.2
    big = groups * weight >= 200_000_000
    if mean < (12 if big else 24):
        return 4
    return 0 if mean < 64 else BY_LIST


def grouped(x: torch.Tensor, w: torch.Tensor, tiles: torch.Tensor, cfg: int, out: torch.Tensor,
            epi: str = "store") -> torch.Tensor:
    """out[r] = act(x[r] @ w[g].T) for the rows of every tile of `tiles` (int32 [n + 1, 4] on the
    device: weight group, first row, rows, 0; the last entry is the number of tiles in use and, for
    BY_LIST, their height), each within x's rows and at most the configuration's row count.  x [R, K], w [groups, N, K] and
    out [R, N] 16-bit; epi: store or one of the activations."""
    if epi not in ("store", "silu", "quick_gelu", "gelu", "relu2") or cfg not in GROUPED_CFGS:
        raise ValueError(f"grouped: epilogue {epi}, configuration {cfg}")
    if x.dtype not in _DT or not (x.dtype == w.dtype == out.dtype) or not x.is_cuda or \
            w.dim() != 3 or not w.is_contiguous():
        raise TypeError("grouped: 16-bit device tensors of one dtype, contiguous weights")
    x2, lda = _rows_view(x, "x")
    o2, ldc = _rows_view(out, "out")
    _, N, K = w.shape
    if x2.shape[1] != K or tuple(o2.shape) != (x2.shape[0], N) or K % 8 or lda % 8 or \
            x2.data_ptr() % 16 or w.data_ptr() % 16:
        raise ValueError(f"grouped: x {tuple(x.shape)}, w {tuple(w.shape)}, out {tuple(out.shape)}")
    if tiles.dtype != torch.int32 or not tiles.is_contiguous() or tiles.dim() != 2 or \
            tiles.shape[0] < 2 or tiles.shape[1] != 4 or not tiles.is_cuda or tiles.data_ptr() % 16:
        raise ValueError("grouped: tiles must be a contiguous int32 [n + 1, 4] device tensor")
    if cfg == ROWS and torch.cuda.is_current_stream_capturing():
        cfg = 4   # rows planned before the capture: the 64-row tile takes the same tile list
    if cfg == ROWS:
        st = current_stream()
        ws, tick = _rows_state(x.device, 16, st)
        check(_lib().cake_gemm_rows_grouped(
            _DT[x.dtype], EPI[epi], x2.data_ptr(), lda, w.data_ptr(), K, N * K, o2.data_ptr(), ldc,
            tiles.data_ptr(), tiles.shape[0] - 1, ws.data_ptr(), tick.data_ptr(),
            _zeros16(x.device).data_ptr(), N, K, st), "gemm_rows_grouped")
        return out
    check(_lib().cake_gemm_grouped(
        _DT[x.dtype], EPI[epi], int(cfg), x2.data_ptr(), lda, w.data_ptr(), K, N * K,
        o2.data_ptr(), ldc, tiles.data_ptr(), tiles.shape[0] - 1, _zeros16(x.device).data_ptr(), N, K,
        current_stream()), "gemm_grouped")
    return out


def _lib_gemm(x2, lda, w, ldb, epi, out2, ldc, r2, ldr, M, N, K) -> None:
    """The library GEMM (hipBLASLt) for a plan that names it.  Its workspace is one buffer
    per (device, stream), so library GEMMs on two streams never share one."""
    dev = x2.device
    st = current_stream()
    ws = _lib_ws.get((dev, st))
    if ws is None:
        ws = _lib_ws[(dev, st)] = torch.empty(_LIB_WS_BYTES, dtype=torch.uint8, device=dev)
    dt = _DT[x2.dtype]

    def run(mode, cptr, ld, n):
        check(_lib_blaslt()(dt, mode, x2.data_ptr(), lda, w.data_ptr(), ldb, cptr, ld,
                                      M, n, K, ws.data_ptr(), _LIB_WS_BYTES, st), "blaslt gemm")
    if epi == "store":
        run(0, out2.data_ptr(), ldc, N)
    elif epi in ("store32", "resid32"):
        run(1 if epi == "store32" else 2, r2.data_ptr(), ldr, N)
    else:  # swiglu: [M, 2N] library product (cached scratch), then silu(gate) * up
        gu = _lib_gu.get((dev, st, x2.dtype))
        if gu is None or gu.numel() < M * 2 * N:
            gu = _lib_gu[(dev, st, x2.dtype)] = torch.empty(M * 2 * N, device=dev,
                                                            dtype=x2.dtype)
        run(0, gu.data_ptr(), 2 * N, 2 * N)
        check(kernels().cake_silu_mul_rows(dt, gu.data_ptr(), M, N, out2.data_ptr(), st),
              "silu_mul_rows")


_lib_ws: dict = {}
_lib_gu: dict = {}
