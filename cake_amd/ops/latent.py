"""Torch-tensor wrappers of the latent-attention kernels (csrc/kernels/mixer_latent.hip); shapes,
dtypes and strides are validated on the host before every launch."""
from __future__ import annotations

from dataclasses import dataclass

import torch

from ._lib import check
from .mixers import DT, MAX_HEAD, MAX_SPLIT, Rows, _check_rows, _lib, _mat, _stream, _vec, pad_to

MAX_RANK = 1024   # largest cached latent the kernels hold
MAX_ROT = 128


@dataclass(frozen=True)
class LatentShape:
    heads: int
    dim: int          # unrotated query / key size of a head
    rot_dim: int
    vdim: int
    q_rank: int
    kv_rank: int
    rot_pairs: int
    recurrent = False
    tiles = 1         # no arrival tickets

    def __post_init__(self):
        if self.heads < 1 or self.dim < 1 or self.q_rank < 1 or not 0 < self.kv_rank <= MAX_RANK or \
                not 0 <= self.rot_dim <= MAX_ROT or 2 * self.rot_pairs > self.rot_dim or \
                self.DP > MAX_HEAD or not 0 < self.vdim <= MAX_HEAD:
            raise ValueError(f"unsupported latent attention shape {self}")

    # padded sizes: every part starts on 16 bytes in every storage type
    @property
    def QP(self) -> int:
        return pad_to(self.q_rank, 8)

    @property
    def RP(self) -> int:
        return pad_to(self.kv_rank, 16)

    @property
    def rotP(self) -> int:
        return pad_to(self.rot_dim, 8)

    @property
    def dimP(self) -> int:
        return pad_to(self.dim, 8)

    @property
    def LD(self) -> int:
        """Cache row: latent | rotated key part | zeros."""
        return pad_to(self.RP + self.rotP, 32)

    @property
    def DP(self) -> int:
        return pad_to(self.dimP + self.rotP, 32)

    @property
    def DVP(self) -> int:
        return pad_to(self.vdim, 16)

    @property
    def in_cols(self) -> int:
        """Projected columns of a row: query latent | latent | rotated key part."""
        return self.QP + self.RP + self.rotP

    @property
    def q_cols(self) -> int:
        return self.heads * (self.dimP + self.rotP)

    @property
    def out_cols(self) -> int:
        return self.heads * self.vdim

    def part_floats(self, B: int, nsplit: int) -> int:
        return B * self.heads * nsplit * (self.RP + 4)


def _cache(sh: LatentShape, cache, dtype):
    """cache [slots, S, LD] -> (pointer, slots, S)."""
    if cache.dim() != 3 or cache.shape[2] != sh.LD or cache.shape[1] % 64:
        raise ValueError(f"cache shape {tuple(cache.shape)} does not fit {sh}")
    return _vec(cache, "cache", dtype), cache.shape[0], cache.shape[1]


def _rotation(sh: LatentShape, cs, S: int):
    if sh.rot_pairs and (cs.shape[0] < S or cs.shape[1] != 2 * sh.rot_pairs):
        raise ValueError("rotation table does not cover the cache")
    return _vec(cs, "cs", torch.float32)


def prep(sh: LatentShape, proj, rows: Rows, cs, eps: float, q_norm, kv_norm, cq, cache):
    """Projected rows [N, in_cols] f32 -> cq [N, QP] (the normed query latent) and the rows' cache
    entries (normed latent, rotated key part).  Norm weights q_norm [QP] and kv_norm [RP], zeros
    past the sizes."""
    cp, slots, S = _cache(sh, cache, cq.dtype)
    _check_rows(rows, S, slots)
    pp, ldp = _mat(proj, "proj", torch.float32, rows.N, sh.in_cols)
    f = torch.float32
    check(_lib().cake_latent_prep(
        DT[cq.dtype], pp, ldp, rows.N, sh.q_rank, sh.QP, sh.kv_rank, sh.RP, sh.rot_dim, sh.LD,
        sh.rot_pairs, float(eps), _vec(q_norm, "q_norm", f, sh.QP),
        _vec(kv_norm, "kv_norm", f, sh.RP), _rotation(sh, cs, S), rows.pos.data_ptr(),
        rows.slot.data_ptr(), _vec(cq, "cq", cq.dtype, rows.N * sh.QP), cp, cache.stride(0),
        _stream()), "latent_prep")


def prompt(sh: LatentShape, q, k, vt, rows: Rows, cs, cache, out, scale: float):
    """Causal attention of packed rows: q [N, q_cols] (not rotated yet), k [n_keys, H dimP] and vt
    [H DVP, n_keys] of the sequences' live positions (packed as rows.key0), out [N, >= H vdim]."""
    cp, slots, S = _cache(sh, cache, q.dtype)
    _check_rows(rows, S, slots)
    qp, ldq = _mat(q, "q", q.dtype, rows.N, sh.q_cols)
    kp, ldk = _mat(k, "k", q.dtype, rows.n_keys, sh.heads * sh.dimP)
    vp, ldv = _mat(vt, "vt", q.dtype, sh.heads * sh.DVP, rows.n_keys)
    op, ldo = _mat(out, "out", q.dtype, rows.N, sh.out_cols)
    if (qp | kp | vp) % 16:
        raise ValueError("latent prompt: operands on 16-byte boundaries")
    check(_lib().cake_latent_flash(
        DT[q.dtype], qp, ldq, kp, ldk, vp, ldv, _vec(rows.key0, "key0", torch.int32, rows.B), cp,
        cache.stride(0), sh.LD, sh.RP, _vec(rows.seq, "seq", torch.int32, 4 * rows.B), rows.B,
        rows.max_len, _rotation(sh, cs, S), sh.rot_pairs, sh.heads, sh.dimP, sh.rotP, sh.vdim,
        sh.DP, sh.DVP, float(scale), op, ldo, _stream()), "latent_flash")


def absorb(sh: LatentShape, q, uk_t, pos, slot, cs, eps: float, kv_norm, cache, qa, proj=None):
    """One token per sequence: q [B, q_cols] f32 -> qa [B, H, LD], the queries against cache rows
    (uk_t [H, kv_rank, dimP]).  With proj [B, in_cols] f32 the tokens' cache rows are written too.
    The caller keeps pos inside the cache."""
    B = q.shape[0]
    cp, _, S = _cache(sh, cache, qa.dtype)
    qp, ldq = _mat(q, "q", torch.float32, B, sh.q_cols)
    pp, ldp = (None, 0) if proj is None else _mat(proj, "proj", torch.float32, B, sh.in_cols)
    check(_lib().cake_latent_absorb(
        DT[qa.dtype], qp, max(ldq, sh.q_cols),
        _vec(uk_t, "uk_t", qa.dtype, sh.heads * sh.kv_rank * sh.dimP), B, sh.heads, sh.dimP,
        sh.rotP, int(proj is not None), pp, ldp, sh.QP, sh.kv_rank, sh.RP, sh.rot_dim, sh.LD,
        sh.rot_pairs, float(eps), _vec(kv_norm, "kv_norm", torch.float32, sh.RP),
        _rotation(sh, cs, S), _vec(pos, "pos", torch.int32, B), _vec(slot, "slot", torch.int32, B),
        cp, cache.stride(0), _vec(qa, "qa", qa.dtype, B * sh.heads * sh.LD), _stream()),
        "latent_absorb")


def decode_per_cu(sh: LatentShape, dtype) -> int:
    """Workgroups of :func:`decode` in 64-key tiles that a CU's LDS holds (mixer_latent.hip launch_latent_decode)."""
    f32 = dtype == torch.float32
    size, piece = (4, 4) if f32 else (2, 8)
    tile = (32 if f32 else 64) // (2 if sh.RP > 512 or sh.LD > 640 else 1)
    return max(1, 160 * 1024 // (((tile + 16) * (sh.LD + piece) + 16 * (tile + piece)) * size))


def decode(sh: LatentShape, qa, pos, slot, cache, scale: float, nsplit: int, part, tile: int = 64):
    """Attention of one token per sequence over its cache rows 0 .. pos, split over the keys in whole tiles
    of 32 or 64; the splits' sums go to part."""
    B = pos.shape[0]
    cp, _, _ = _cache(sh, cache, qa.dtype)
    if not 1 <= nsplit <= MAX_SPLIT:
        raise ValueError(f"nsplit {nsplit} outside 1..{MAX_SPLIT}")
    check(_lib().cake_latent_decode(
        DT[qa.dtype], _vec(qa, "qa", qa.dtype, B * sh.heads * sh.LD), cp, cache.stride(0),
        _vec(pos, "pos", torch.int32, B), _vec(slot, "slot", torch.int32, B), B, sh.heads, sh.LD,
        sh.RP, int(nsplit), int(tile), float(scale),
        _vec(part, "part", torch.float32, sh.part_floats(B, nsplit)), _stream()), "latent_decode")


def out(sh: LatentShape, part, pos, uv, nsplit: int, y, tile: int = 64):
    """y [B, >= H vdim] = the value expansion uv [H, DVP, RP] of the merged splits."""
    B = pos.shape[0]
    yp, ldy = _mat(y, "y", y.dtype, B, sh.out_cols)
    check(_lib().cake_latent_out(
        DT[y.dtype], _vec(part, "part", torch.float32, sh.part_floats(B, nsplit)),
        _vec(pos, "pos", torch.int32, B), _vec(uv, "uv", y.dtype, sh.heads * sh.DVP * sh.RP), B,
        sh.heads, sh.vdim, sh.DVP, sh.RP, int(nsplit), int(tile), yp, max(ldy, sh.out_cols), _stream()),
        "latent_out")
