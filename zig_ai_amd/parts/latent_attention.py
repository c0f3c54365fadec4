"""Attention over one small latent vector a token, as a part (mixer ``latent_attention``).

Per token, with ``h`` the mixer's input:

  c_q = rmsnorm(Wdq h) * q_norm                     the query latent, ``q_rank`` wide
  q_i = Wuq c_q                                     per head [head_dim unrotated | rotated_dim rotated]
  [c' | k_r] = Wdkv h;  c = rmsnorm(c') * kv_norm   the latent, ``kv_rank`` wide; ``k_r`` (not
                                                    normed) is one rotated key part for all heads
  k_i = Wuk_i c,  v_i = Wuv_i c                     every head's keys and values
  s_ij = (q_i,n . k_j,i + rot(q_i,r) . rot(k_r,j)) * softmax_scale,  j <= i
  o_i = sum_j softmax(s_i, with exp(sink_i) in the denominator)_j v_j,i
  y   = Wo (o * sigmoid(Wg h))                      ``gate="element"``: a number an element of
                                                    o; ``"head"``: a number a head; None: none

Only ``[c | rot(k_r)]`` is cached, one plane of ``kv_rank + rotated_dim`` elements a token.  Where
many new tokens see the same rows (``forming_pays``) every head's keys and values are formed from the
visible rows and attended to (``csrc/latent_expanded.hip``).  Elsewhere
they are not: ``Wuk_i^T q_i,n`` is taken instead (the score against ``c``
is the same number) and ``Wuv_i`` is applied to ``sum_j p_j c_j``, so the attention kernel sees
one key/value head whose value is a prefix of its key (``csrc/latent.hip``).  bfloat16 rows of
16-byte pieces run on the matrix cores (work items of 64 rows; a step that only decodes takes the
kernel whose four waves share 16 rows, its contexts cut into ranges), everything else the
general kernel.

All sizes and constants come from ``params``: ``hidden_size, num_heads, head_dim,
rotated_dim`` (0: no positions), ``value_dim, kv_rank, q_rank, softmax_scale`` (None:
``(head_dim + rotated_dim)^-1/2``), ``norm_eps, sink`` (true: a tensor ``sink [num_heads]``),
``gate`` and ``position`` (a nested rotary spec whose ``head_dim`` is ``rotated_dim``; its
``rotary_dim`` may be smaller: the other elements of the rotated part pass unchanged; its
``magnitude`` multiplies what it turns, in queries and keys).  ``makes_rows`` (true): with false
the layer has no ``Wdkv`` and reads the rows that another layer caches: its run-order entry
shares that layer's cache entry (``LayerCall.cache``, ``writes_cache=False``).
"""

from __future__ import annotations

import math
from typing import Any, Dict, Mapping, Optional

import torch

from ..kernels import ops
from .attention import plan_split
from .base import Mixer, PagedNeed, Runtime, TensorRule, lookup, register_mixer
from .feed_forward import fuse_rows, pad_rows


LATENT_SPLIT_TARGET = 1024    # workgroups to reach by cutting contexts into ranges
LATENT_SPLIT_KEYS = 128       # keys of a range at least
LATENT_SPLIT_BYTES = 32 << 20  # the most that the ranges' partial results may take


def plan_latent_split(groups: int, max_keys: int, target: int = LATENT_SPLIT_TARGET, tile: int = 64):
    """(keys per range, number of ranges) for one launch of the matrix-core kernels: a function
    of the batch shape and of the longest context only.  As many ranges as reach ``target``
    workgroups, of at least ``LATENT_SPLIT_KEYS`` keys each, in whole multiples of ``tile``: the kernels of one
    and four waves take 32 keys at a time, so short ranges pay; the one of eight waves takes 128."""
    if groups >= target or max_keys <= 2 * LATENT_SPLIT_KEYS:
        return 0, 1
    nsplit = min(target // groups, max_keys // LATENT_SPLIT_KEYS, 64)
    if nsplit <= 1:
        return 0, 1
    keys = ((max_keys + nsplit - 1) // nsplit + tile - 1) // tile * tile
    nsplit = (max_keys + keys - 1) // keys
    return (keys, nsplit) if nsplit > 1 else (0, 1)


# The kernel that takes single tokens' keys 128 at a time (``ops.latent_range_fits``) has one workgroup a compute
# unit at latents of 512 (two at 128), and a second round of them costs more than longer ranges.  Us with
# ranges of 128, 256 and 512 keys, 16 heads, R = 512 with 64 rotated: 8 requests at 2,050 keys 18.5, 19.8, 25.5, at
# 8,000 42, 29, 30; 32 at 2,000 36, 26, 29; 64 at 1,200 46, 39, 32; R = 128 with 32: 64 at 2,000 19.0, 15.7, 17.1.
# 129 to 255 groups get a range each, which leaves compute units idle, but cuts them only gain where contexts are long
# and three ranges fill two rounds well: in one, two and three ranges 130 requests at 1,000 keys 42, 59, 53, at 2,000
# 88, 105, 91, at 4,000 171, 193, 151, 200 at 4,000 191, 215, 223; 20 requests of 128 heads at 4,000 118, 132, 102.
LATENT_RANGE_TARGET, LATENT_RANGE_TARGET_SMALL, LATENT_RANGE_TILE = 256, 512, 128


FORMING_ROWS_A_TOKEN = 16      # visible rows a new token, at most
FORMING_BYTES = 256 << 20      # the most that formed keys and values may take


def forming_pays(step, bytes_a_row: int) -> bool:
    """Whether a step's keys and values are formed: every request brings a portion, and a visible row is
    seen by enough new tokens.  Us a layer folded and formed (16 heads, R = 512 with 64 rotated), by visible rows a new
    token.  1: one prompt of 64 32 and 15, 512 61 and 26, 1,777 145 and 61, 4,096 523 and 145; 4 tokens of 8 requests each 31 and
    13.  8 to 9: 128 tokens behind 900 cached ones 51 and 39, 64 of 8 requests each behind 512 65 and 54.  13: 512 behind
    6,000 348 and 158.  17: 128 behind 2,048 135 and 64, 64 behind 1,024 50 and 40, 64 of 8 each behind 1,024 91 and 81, 2 of 32
    each behind 32 27 and 23.  25: 128 behind 3,072 185 and 81, but 64 behind 1,536 50 and 55, 2 of 32 each behind 48 28 and
    31.  33: 512 behind 16,384 836 and 390, 64 of 8 each behind 2,048 140 and 144.  The line lies where all gain: beyond it
    few tokens lose, whose folded kernel cuts contexts into ranges.  Single tokens share their rows with nobody."""
    return step.fewest_tokens > 1 and step.visible_rows <= FORMING_ROWS_A_TOKEN * step.n_tokens \
        and step.visible_rows * bytes_a_row <= FORMING_BYTES


FORMING_BLOCK = 256      # rows


def forming_block(rows: int) -> int:
    """What ``rows`` are rounded up to a multiple of: an eighth of the power of two at or above them."""
    return max(FORMING_BLOCK, 1 << max((rows - 1).bit_length() - 3, 0))


def forming_rows(rows: int, outputs: int, kv_rank: int) -> int:
    """The rows that the forming product is asked for: ``rows``, which is any sum of contexts, or more.  The GEMM
    library plans every row count that it meets, and times its candidates for every block of them (10 to 60 ms), so
    it meets few: beyond ``FORMING_BLOCK`` its multiples, from eight of them on four to an octave
    (``LatentAttention.warm_up`` runs them ahead).  Pieces of 2,048 rows each would be fewer still, but take 49 us for
    6,512 rows of 16 heads where one product takes 33 (K = 512), for 32,768 225 and 129.  A count that this package's
    kernel takes is left as it is."""
    if rows <= FORMING_BLOCK or ops.half_plan(rows, outputs, kv_rank, False)[0]:
        return rows
    block = forming_block(rows)
    return -(-rows // block) * block


class LatentAttention(Mixer):
    kind = "latent_attention"
    graph_safe = True
    takes_normed_rows = True      # ``x`` is only ever handed to ``ops.linear``
    kernel_sources = ("gemm", "gemm_rows64", "latent", "latent_expanded", "norm", "activation")

    @staticmethod
    def _sizes(params):
        return tuple(int(params[k]) for k in ("hidden_size", "num_heads", "head_dim", "value_dim",
                                              "kv_rank", "q_rank")) \
            + (int(params.get("rotated_dim") or 0),)

    @classmethod
    def tensor_rules(cls, params: Mapping[str, Any]) -> Dict[str, TensorRule]:
        H, nh, d, dv, R, Rq, dr = cls._sizes(params)
        rules = {"q_down.weight": TensorRule(((Rq, H),)),
                 "q_norm.weight": TensorRule(((Rq,),), role="norm"),
                 "q_up.weight": TensorRule(((nh * (d + dr), Rq),)),
                 "k_up.weight": TensorRule(((nh * d, R),)),
                 "v_up.weight": TensorRule(((nh * dv, R),)),
                 "out_proj.weight": TensorRule(((H, nh * dv),))}
        if params.get("makes_rows", True):
            rules["kv_down.weight"] = TensorRule(((R + dr, H),))
            rules["kv_norm.weight"] = TensorRule(((R,),), role="norm")
        if params.get("sink"):
            rules["sink"] = TensorRule(((nh,),), role="bias")
        if params.get("gate") == "head":
            rules["gate_proj.weight"] = TensorRule(((nh, H),))
        elif params.get("gate") == "element":
            rules["gate_proj.weight"] = TensorRule(((nh * dv, H),))
        return rules

    @classmethod
    def cache_need(cls, params: Mapping[str, Any]):
        _, _, _, _, R, _, dr = cls._sizes(params)
        return PagedNeed(((1, R + dr),))

    def __init__(self, params, tensors, runtime: Runtime):
        super().__init__(params, tensors, runtime)
        H, nh, d, dv, R, Rq, dr = self._sizes(params)
        self.num_heads, self.head_dim, self.value_dim = nh, d, dv
        self.kv_rank, self.q_rank, self.rotated_dim = R, Rq, dr
        self.width = R + dr                    # cached elements a token
        if params.get("gate") not in (None, "head", "element"):
            raise ValueError(f"gate must be None, 'head' or 'element', got {params.get('gate')!r}")
        self.gate = params.get("gate")
        if self.width > ops.LATENT_MAX_WIDTH or R > ops.LATENT_MAX_RANK:
            raise ValueError(f"a latent of {R} with {dr} rotated elements: the kernels take rows up "
                             f"to {ops.LATENT_MAX_WIDTH} and latents up to {ops.LATENT_MAX_RANK}")
        scale = params.get("softmax_scale")
        self.scale = float(scale) if scale is not None else 1.0 / math.sqrt(d + dr)
        self.eps = float(params.get("norm_eps", 0.0))
        self.sink = tensors["sink"] if params.get("sink") else None
        pos = params.get("position")
        self.position = None
        self.rot_dims, self.adjacent, self.inv_freq, self.magnitude = 0, False, None, 1.0
        if dr:
            if pos is None:
                raise ValueError("a rotated part needs a position encoding")
            self.position = lookup("position", pos.kind)(pos.params, {}, runtime)
            if not getattr(self.position, "fused_rotation", False) or self.position.head_dim != dr:
                raise ValueError("the rotated part takes a rotary encoding of its own width")
            self.rot_dims = self.position.rotary_dim
            self.adjacent = self.position.pairing == "adjacent"
            self.inv_freq = self.position.inv_freq
            self.magnitude = float(self.position.magnitude)
        elif pos is not None:
            raise ValueError("a position encoding needs a rotated part")
        # the opening product: query latent | latent and rotated key part | gate, each
        # starting on a 16-byte boundary
        self.makes_rows = bool(params.get("makes_rows", True))
        pieces = [pad_rows(tensors["q_down.weight"])]
        self.c_col = pieces[0].shape[0]
        if self.makes_rows:
            pieces.append(pad_rows(tensors["kv_down.weight"]))
        self.gate_col = sum(p.shape[0] for p in pieces)
        if self.gate is not None:
            pieces.append(pad_rows(tensors["gate_proj.weight"]))
        self.w_open = ops.projection_weight(fuse_rows(*pieces))
        self.q_norm = tensors["q_norm.weight"]
        self.kv_norm = tensors["kv_norm.weight"] if self.makes_rows else None
        self.w_q_up = ops.projection_weight(tensors["q_up.weight"])
        self.w_out = ops.projection_weight(tensors["out_proj.weight"])
        # per head: Wuk^T as [R, d] (folds into the query), Wuv as [dv, R] (expands the result)
        k_up = tensors["k_up.weight"].view(nh, d, R).transpose(1, 2).contiguous()
        v_up = tensors["v_up.weight"].view(nh, dv, R).contiguous()
        # all heads' Wuk, then all heads' Wuv, where keys and values may be formed
        self.w_form = None
        if ops.latent_expanded_fits(runtime.dtype, d, dr, dv, R) and k_up.dtype == v_up.dtype == torch.bfloat16:
            self.w_form = fuse_rows(tensors["k_up.weight"], tensors["v_up.weight"])
            v_up = self.w_form[nh * d:].view(nh, dv, R)
        # (the matrix-core form reads 16-byte pieces of its rows)
        if k_up.dtype == torch.bfloat16 and (d % 8 or (d + dr) % 8):
            k_up = k_up.float()
        if v_up.dtype == torch.bfloat16 and R % 8:
            v_up = v_up.float()
        self.k_fold, self.v_expand = k_up, v_up
        # bfloat16 rows of 16-byte pieces run on the matrix cores, in work items of 64 rows
        self.mfma = ops.latent_mfma_fits(runtime.dtype, self.width, R)
        most = ops.LATENT_MFMA_ROWS if self.mfma else ops.LATENT_MAX_ROWS
        self.rows_per_item = max(1, most // min(nh, most))
        self.item_granularities = [self.rows_per_item]
        if self.w_form is not None:
            self.item_granularities.append((ops.LATENT_EXPANDED_ROWS, 2))
            ops.check_projection_weight(self.w_form, "latent attention w_form")
        for w, what in ((self.w_open, "w_open"), (self.w_q_up, "w_q_up"), (self.w_out, "w_out")):
            ops.check_projection_weight(w, "latent attention " + what)

    def forward(self, x, step, cache):
        nh, d, dv, R, dr = self.num_heads, self.head_dim, self.value_dim, self.kv_rank, self.rotated_dim
        T = x.shape[0]
        tune = self.runtime.tune
        plane = cache.planes[0]
        if cache.writes and not self.makes_rows:
            raise ValueError("a latent attention without rows of its own reads another layer's "
                             "cache: its run-order entry must not write")
        down = ops.linear(x, self.w_open, tune=tune)
        cq = ops.latent_prepare(down, 0, self.q_rank, self.c_col, R, dr, self.q_norm, self.kv_norm,
                                self.eps, step.positions, step.slot_mapping[cache.group],
                                self.inv_freq, self.rot_dims, self.adjacent,
                                plane if cache.writes else None, self.magnitude)
        q = ops.linear(cq, self.w_q_up, tune=tune).view(T, nh, d + dr)
        if self.w_form is not None and not step.recordable and forming_pays(step, 2 * nh * (d + dv)):
            a = self._formed(q, down, plane, step, cache)
            return ops.linear(a.view(T, nh * dv), self.w_out, partial_ok=self.partial_ok, tune=tune)
        qf = self._folded(q, step)
        item_seq, item_row0, item_count, n_items = step.attention_items(self.rows_per_item)
        waves = 0
        if self.mfma:
            # a step that only decodes: a wave a workgroup, heads in chunks of 16
            waves = 1 if step.n_tokens == step.n_seqs else 4
            groups = n_items * (-(-nh // (16 * waves)))
            if waves == 1 and ops.latent_range_fits(self.width, R, plane.shape[2]):
                keys, nsplit = plan_latent_split(groups, step.max_keys, LATENT_RANGE_TARGET if R > 256 else
                                                 LATENT_RANGE_TARGET_SMALL, LATENT_RANGE_TILE)
            else:
                keys, nsplit = plan_latent_split(groups, step.max_keys)
            # (the ranges' partial results are 32-bit rows of the latent's width: no cut where
            # they would be larger than the step is worth)
            if T * nh * nsplit * R * 4 > LATENT_SPLIT_BYTES:
                keys, nsplit = 0, 1
        else:
            keys, nsplit = plan_split(n_items, 1, step.max_keys)
        o = ops.latent_attention(qf, plane, R, step.block_tables[cache.group], step.positions,
                                 item_seq, item_row0, item_count, n_items, self.scale, self.sink,
                                 keys, nsplit, waves)
        # every head's result expanded by its Wuv, times the gate
        a = ops.head_linear(o, 0, self.v_expand, gate=down if self.gate else None,
                            gate_col=self.gate_col, gate_mode=self.gate)
        if getattr(step, "taps", None) is not None:
            step.taps["q"] = qf.clone()
            step.taps["o"] = a.clone()
        return ops.linear(a.view(T, nh * dv), self.w_out, partial_ok=self.partial_ok, tune=tune)

    def warm_up(self, step_tokens):
        if self.w_form is None:
            return
        outputs, counts = self.w_form.shape[0], [FORMING_BLOCK]
        most = min(FORMING_ROWS_A_TOKEN * step_tokens, FORMING_BYTES // (2 * outputs))
        while counts[-1] < most:
            counts.append(counts[-1] + forming_block(counts[-1] + 1))
        # (values as steps have them: on zeros other candidates win)
        latent = self.w_form.new_empty((counts[-1], self.kv_rank))
        latent.normal_(generator=torch.Generator(device=latent.device))
        for rows in counts:
            if not ops.half_plan(rows, outputs, self.kv_rank, False)[0]:
                ops.linear(latent[:rows], self.w_form, tune=self.runtime.tune)

    def _folded(self, q, step):
        """The folded queries [Wuk^T q_n | rot(q_r)]."""
        return ops.latent_fold(q, self.k_fold, self.rotated_dim, step.positions, self.inv_freq, self.rot_dims,
                               self.adjacent, self.magnitude)

    def _formed(self, q, down, plane, step, cache):
        """The heads' gated results over formed keys and values."""
        if getattr(step, "taps", None) is not None:
            step.taps["q"] = self._folded(q, step)      # (what the other steps leave)
        rows = forming_rows(step.visible_rows, self.w_form.shape[0], self.kv_rank)
        latent, rot = ops.latent_open_rows(
            q, self.head_dim, self.rotated_dim, step.positions, self.inv_freq, self.rot_dims, self.adjacent,
            self.magnitude, plane, self.kv_rank, step.block_tables[cache.group], step.seq_start, step.ctx_len,
            rows)
        kv = ops.linear(latent, self.w_form, tune=self.runtime.tune)
        a = ops.latent_expanded(q, kv, rot, step.positions, step.attention_items(ops.LATENT_EXPANDED_ROWS, 2),
                                step.seq_start, step.ctx_len, self.scale, self.sink, down if self.gate else None,
                                self.gate_col, self.gate)
        if getattr(step, "taps", None) is not None:
            step.taps["o"] = a.clone()
        return a


register_mixer(LatentAttention.kind, LatentAttention)
