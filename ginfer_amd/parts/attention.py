"""Attention over the paged cache: grouped queries, rotary positions, all keys or a window."""
import math

import torch

from ..kernels import autotune, ops
from ..kernels.tuning import TUNING
from ..weights.loader import WeightSpec
from .base import Part, KVCacheSpec
from .linear import linear, linear_into_norm
from .registry import register_mixer


def _library_then_rotation_is_faster(rows, in_features, out_features):
    """The fused projection kernel cannot split K over workgroups (its epilogue needs whole sums), and each of its workgroups reads
    all rows: from 17 rows and some K on, and with more columns and rows than that, the BLAS library's product followed by the
    rotation kernel is faster (the figures stand beside the thresholds)."""
    if rows > TUNING.fused_qkv_up_to_rows and in_features >= TUNING.fused_qkv_unless_in_features:
        return True
    return (rows > TUNING.fused_qkv_wide_up_to_rows and out_features > TUNING.fused_qkv_wide_out_features
            and in_features >= TUNING.fused_qkv_wide_in_features)


def _projection_in_parts(rows, in_features, out_features):
    """Into how many parts of K the q|k|v product is split where the fused kernel does not take the rotation (part of a head, or a
    head size that is no multiple of 32), its parts to be added by the rotation kernel; 0: not this way, by sizes alone."""
    T = TUNING
    if (not T.qkv_in_parts_from_rows <= rows <= ops.SKINNY_MAX_ROWS or in_features >= T.qkv_in_parts_unless_in_features
            or out_features > T.qkv_in_parts_most_out_features):
        return 0
    parts = min(T.qkv_in_parts_most, 8, in_features // T.qkv_in_parts_min_k)
    return parts if parts >= 2 else 0


def _projection_way(x, w_qkv, head_dim, rotary_dim):
    """("fused",), ("parts", n) or ("library",): how rows x become q, k and v where their product is not dealt evenly to the chip."""
    if x.shape[0] > ops.SKINNY_MAX_ROWS:        # neither of the others takes them; such steps are launched kernel by kernel
        return ("library",)
    fused_ok = ops.qkv_rope_skinny_supported(x, w_qkv, head_dim, rotary_dim)
    return _other_way(x.shape[0], x.shape[1], w_qkv.shape[0], fused_ok, not fused_ok and _parts_supported(x, w_qkv, head_dim, rotary_dim))


def _parts_supported(x, w_qkv, head_dim, rotary_dim):
    return (not isinstance(x, ops.ScaledRows) and ops.gemm_skinny_supported(x, w_qkv) and (rotary_dim // 2) % 4 == 0
            and (head_dim - rotary_dim) % 4 == 0 and head_dim % 4 == 0)


def _other_way(rows, in_features, out_features, fused_ok, parts_ok):
    if fused_ok:
        return ("library",) if _library_then_rotation_is_faster(rows, in_features, out_features) else ("fused",)
    parts = _projection_in_parts(rows, in_features, out_features) if parts_ok else 0
    return ("parts", parts) if parts else ("library",)


def _dealing_is_slower(plan, rows, in_features, out_features):
    """Whether the other ways are faster than q|k|v over tiles dealt evenly to the chip by `plan`, by sizes alone (the measurements stand
    beside the thresholds)."""
    T = TUNING
    if rows <= T.qkv_spread_up_to_rows:
        return False
    _, m_tiles, groups = plan
    _, _, room_a, room_w, _ = ops.spread_share(plan, rows, out_features)
    padded = room_a * room_w * m_tiles * groups / (rows * out_features)
    if room_a >= T.qkv_spread_tall_tile:
        return m_tiles > 2 or padded > T.qkv_spread_tall_padded
    if (in_features % 128 or room_w < T.qkv_spread_wide_tile or in_features < T.qkv_spread_long_k
            or out_features * in_features <= T.qkv_spread_many_weights):
        return False
    if m_tiles == 3:
        return in_features >= T.qkv_spread_longer_k and rows > T.qkv_spread_longer_k_up_to_rows
    return m_tiles > 3 and padded > T.qkv_spread_wide_padded


def projection_choice(x, w_qkv, has_bias, num_heads, num_kv_heads, head_dim, rotary_dim):
    """(the way that rows x become q, k and v, the tuner's key for it or None): ("spread", plan) over tiles dealt evenly to the chip, where
    they hold the product and are the faster, or one of _projection_way's."""
    plan = ops.qkv_spread_plan(x, w_qkv, head_dim, rotary_dim)
    key = None
    if plan and autotune.active():
        fused_ok = ops.qkv_rope_skinny_supported(x, w_qkv, head_dim, rotary_dim)
        key = ("qkv", autotune.rows_class(x.shape[0]), w_qkv.shape[0], x.shape[1], has_bias, num_heads, num_kv_heads, head_dim, rotary_dim,
               fused_ok, not fused_ok and _parts_supported(x, w_qkv, head_dim, rotary_dim))
    if plan and not _dealing_is_slower(plan, *x.shape, w_qkv.shape[0]):
        return ("spread", plan), key
    return _projection_way(x, w_qkv, head_dim, rotary_dim), key


def project(way, x, w, bias, positions, cos, sin, slot_mapping, k_pages, v_pages, num_heads, num_kv_heads, head_dim, write_kv):
    """q|k|v of rows x: q rotated (the columns behind it are the kernel's own), k and v in their pages."""
    place = (positions, cos, sin, slot_mapping, k_pages, v_pages, num_heads, num_kv_heads, head_dim)
    if way[0] == "fused":
        # few rows (decode): projection, rotation and cache write in one kernel
        return ops.qkv_rope_skinny(x, w, bias, *place, write_kv=write_kv)
    if way[0] == "spread":
        # more rows: the same, over tiles that are dealt evenly to the chip (by the rows that come, where a plan stands for a class of them)
        return ops.qkv_spread(x, w, bias, *place, write_kv=write_kv, plan=way[1] if len(way) > 1 else None)
    if way[0] == "parts":
        # the product with K split over workgroups (every workgroup then reads a share of the rows only), its 32-bit
        # parts added up by the kernel that rotates and writes the cache
        sums = ops.gemm_skinny(x, w, None, out_dtype=torch.float32, nt=2, grid_splits=way[1])
        return ops.rope_kv_from_parts(sums, bias, *place, write_kv=write_kv)
    qkv = linear(x, w, bias)
    ops.rope_kv_write(qkv, *place, write_kv=write_kv)
    return qkv


def projection_candidates(key):
    """Every way to do the projection of an autotune key; the one that runs by the rules first."""
    _, rows, out_features, in_features, _, _, _, _, _, fused_ok, parts_ok = key
    spread, other = ("spread",), _other_way(rows, in_features, out_features, fused_ok, parts_ok)
    slower = _dealing_is_slower(ops.spread_few_columns(rows, out_features, in_features)[1], rows, in_features, out_features)
    ways = [other, spread] if slower else [spread, other]
    for way in (("fused",) if fused_ok else None, ("library",)):
        if way and way not in ways:
            ways.append(way)
    return ways


def _projection_timing(key, operands, device):
    """For the tuner: random rows, tokens of one request side by side in pages of 16."""
    _, rows, _, in_features, _, nh, nkv, hd, rotary_dim = key[:9]
    x = (torch.randn((rows, in_features), device=device) * 0.5).to(torch.bfloat16)
    positions, slots = torch.zeros(rows, dtype=torch.int32, device=device), torch.arange(rows, device=device)
    cos, sin = torch.ones((1, rotary_dim // 2), device=device), torch.zeros((1, rotary_dim // 2), device=device)
    k_pages = torch.zeros((-(-rows // 16), nkv, 16, hd), dtype=torch.bfloat16, device=device)
    v_pages = torch.zeros((-(-rows // 16), nkv, hd, 16), dtype=torch.bfloat16, device=device)
    return lambda way, i: project(way, x, *operands[i], positions, cos, sin, slots, k_pages, v_pages, nh, nkv, hd, True)


autotune.register_kind("qkv", projection_candidates, _projection_timing)


@register_mixer("attention")
class Attention(Part):
    """q/k/v projections (one fused product over the stacked weights; results equal the three separate
    ones of ginfer/core/layer/transformer/attention.cc:61-63), rotation of q and k and the cache write
    (:69-72, :32-33), attention over the request's pages (:34), output projection (:80-81).
    score scale 1/sqrt(head_dim) unless `scale` is given; `window` None attends to all earlier keys."""

    capturable = True
    takes_scaled_rows = True
    folds_norm = True

    def __init__(self, hidden_size, num_heads, num_kv_heads, head_dim, qkv_bias, out_bias, window, position,
                 scale, dtype, device):
        if num_heads % num_kv_heads:
            raise ValueError("num_heads %d is not a multiple of num_kv_heads %d" % (num_heads, num_kv_heads))
        if not 0 < head_dim <= 256:
            raise ValueError("head_dim %d is not supported: the attention kernels take head sizes up to 256 "
                             "(the matrix-core kernels multiples of 16, the general kernel the others)" % head_dim)
        self.hidden_size, self.nh, self.nkv, self.hd = hidden_size, num_heads, num_kv_heads, head_dim
        self.qkv_bias, self.out_bias = bool(qkv_bias), bool(out_bias)
        self.window = int(window) if window else None
        self.position = position
        self.scale = float(scale) if scale is not None else 1.0 / math.sqrt(head_dim)
        self.dtype, self.device = dtype, device
        self.w_qkv = self.b_qkv = self.w_o = self.b_o = None

    def cache_spec(self):
        return KVCacheSpec(self.nkv, self.hd, self.window)

    def weight_specs(self):
        H, q, kv = self.hidden_size, self.nh * self.hd, self.nkv * self.hd
        specs = {"q_proj.weight": WeightSpec((q, H)), "k_proj.weight": WeightSpec((kv, H)),
                 "v_proj.weight": WeightSpec((kv, H)), "o_proj.weight": WeightSpec((H, q))}
        if self.qkv_bias:
            specs.update({"q_proj.bias": WeightSpec((q,)), "k_proj.bias": WeightSpec((kv,)),
                          "v_proj.bias": WeightSpec((kv,))})
        if self.out_bias:
            specs["o_proj.bias"] = WeightSpec((H,))
        return specs

    def bind_weights(self, t):
        self.w_qkv = torch.cat([t["q_proj.weight"], t["k_proj.weight"], t["v_proj.weight"]], dim=0).contiguous()
        self.b_qkv = (torch.cat([t["q_proj.bias"], t["k_proj.bias"], t["v_proj.bias"]], dim=0).contiguous()
                      if self.qkv_bias else None)
        self.w_o = t["o_proj.weight"]
        self.b_o = t.get("o_proj.bias") if self.out_bias else None

    def kernel_modules(self):
        mods = ["rope_kv", "attention_generic", "gemm"]
        if self.dtype == torch.bfloat16:
            mods += ["gemm_skinny", "gemm_tiles"]
            if self.hd in ops.MFMA_HEAD_DIMS:
                mods += [("attention_mfma", {"HEAD_DIM": self.hd})]
        return mods

    def forward(self, x, step, cache, into_norm=None):
        """into_norm = (residual, norm): where the output projection's kernel can, the result is added to the
        residual here and the rows of `norm` come back as ops.ScaledRows; else the result comes back as ever."""
        cos, sin = self.position.tables()
        way, key = projection_choice(x, self.w_qkv, self.b_qkv is not None, self.nh, self.nkv, self.hd, self.position.rotary_dim)
        if key is not None:
            way = autotune.choose(key, (self.w_qkv, self.b_qkv)) or way
        qkv = project(way, x, self.w_qkv, self.b_qkv, step.positions, cos, sin, cache.slot_mapping, cache.k_pages, cache.v_pages,
                      self.nh, self.nkv, self.hd, cache.owner)
        a = ops.paged_attention(qkv, cache.k_pages, cache.v_pages, cache.block_table, step, self.nh, self.nkv,
                                self.hd, self.scale, self.window)
        if into_norm is not None:
            folded = linear_into_norm(a, self.w_o, self.b_o, *into_norm)
            if folded is not None:
                return folded
        return linear(a, self.w_o, self.b_o, parts_ok=True)
