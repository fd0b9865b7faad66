"""PaLM-style parallel attention + MLP block on the gfx950 kernels.

Public surface of the reference's gpt_fast/gpt_parallel_TP.py (`GPTParallel` :136-192,
`ParallelTransformerBlock` :195-229): one RMSNorm and one fused projection `wqkv1` per layer,
y = w2(silu(g) * u) + wo(attention), x = y + x.  As in the dense family, a semi-compiled shard
that is not rank 0 carries no residual (:205-206)."""
import torch
import torch.nn as nn
from torch import Tensor

from . import _hip
from ._model import GPTBase, Workspace
from .config import REGISTRIES, ModelArgs, find_multiple  # noqa: F401
from .utils import FuseAttentionMLP, RMSNorm, all_reduce_func

transformer_configs = REGISTRIES["parallel"]


class ParallelTransformerBlock(nn.Module):
    def __init__(self, config: ModelArgs) -> None:
        super().__init__()
        self.attention = FuseAttentionMLP(config)
        self.attention_norm = RMSNorm(config.dim, config.norm_eps)
        self.semi_compiled_model = config.semi_compiled_model
        self.keeps_residual = not (config.semi_compiled_model and config.tp_rank != 0)

    def forward(self, x: Tensor, input_pos: Tensor, freqs_cis: Tensor, mask: Tensor) -> Tensor:
        x = x.contiguous()
        y = self.attention(self.attention_norm(x), freqs_cis, mask, input_pos)
        y = all_reduce_func(y, clone=False)[0]
        return _hip.add(y, x, torch.empty_like(y)) if self.keeps_residual else y

    def extra_repr(self) -> str:
        return f"semi_compiled = {self.semi_compiled_model}"


class GPTParallel(GPTBase):
    family = "parallel"
    band_rows_from = 1   # six launches per block instead of nine also pay for a single row (5.6 -> 5.0 ms, 70B shard)

    def __init__(self, config):
        super().__init__(config)
        self._parts_pay = {}   # (rows, of a decode step): see _in_parts

    def _make_block(self, config, layer_idx):
        return ParallelTransformerBlock(config)

    def _fused_width(self) -> int:
        return super()._fused_width() + 2 * self.config.ffn_local

    def _pair_bytes(self, B):
        if B > _hip.BANDS_TO or hasattr(self.layers[0].attention.wqkv1, "scales"):
            return ()
        return (_hip.beside_product_bytes(B, 2 * self.config.ffn_local, self.config.dim),)

    def _products(self, B, S):
        nqkv = GPTBase._fused_width(self)
        for rows, N, K, pair in super()._products(B, S):
            yield rows, N, K, pair
            if N == self._fused_width() and (S == 1 and B <= 64 or self._in_parts(B, S)):   # (its two parts)
                yield rows, nqkv, K, False
                yield rows, N - nqkv, K, True

    def _run_layers(self, ws: Workspace, pos: Tensor):
        cfg = self.config
        nqkv = (cfg.n_head_local + 2 * cfg.n_kv_local) * cfg.head_dim
        att0 = self.layers[0].attention
        if not any(hasattr(m, "scales") for m in (att0.wqkv1, att0.wo, att0.w2)):
            if ws.S == 1 and self.band_rows_from <= ws.B <= 64:
                return self._run_layers_decode(ws, pos, nqkv)
            if self._in_parts(ws.B, ws.S):
                return self._run_layers_prompt(ws, pos, nqkv)
        for blk in self.layers:
            att = blk.attention
            _hip.add_rmsnorm(ws.x, None, None, blk.attention_norm.weight, None, ws.xn, cfg.norm_eps)
            self._attention(ws, blk, pos, att.wqkv1, ws.a)   # ws.qkv holds [q | k | v | u | g]
            _hip.module_linear_swiglu(ws.qkv[:, nqkv:], att.w2, ws.m, ws.act, ws.sums)
            _hip.add(ws.m, ws.a, ws.m)                               # w2(...) + wo(...)
            if blk.keeps_residual:
                _hip.add(ws.m, ws.x, ws.x)                           # y + x
            else:
                ws.x.copy_(ws.m)
        return None, None

    # Rows (of a prompt, or a decode batch above 64) whose fused input weight is two products with their output passes, eight launches for
    # eleven and no passes over the products' rows: up to 32, from parts_from on, and up to parts_to where the products' costs say that
    # they take no longer than one and what it leaves out: 8 us of passes, and 6 more for the launches of a prompt, which come one by one and take
    # about 110 us per block, where one product takes up to 50 (the other half of such a block is no longer).
    # us, one / two, one library, shapes of 8B, 1B, the 70B rank shard and Llama 3.2 3B.  A decode step's graph: 70 sequences 5198 / 4771,
    # 1273 / 1306, 6884 / 7018, 3070 / 3300, 160 sequences 5902 / 5759, 1520 / 1582, 8649 / 8529, 4044 / 4134; only 8B's is two.  A prompt as it is
    # called: 30 tokens 4390 / 4234, 1722 / 1602, 7725 / 7046, 3022 / 2772, 64 tokens 4437 / 3808, 1880 / 1769, 8468 / 7801, 3216 / 2920, 150 tokens
    # 5375 / 5259, 1786 / 1579, 8655 / 8417, 3071 / 3195; above 32 all but 3B's are two, though 1B's take 3 to 5 % longer on the device (64 tokens
    # 1092 / 1148) and the shard's up to 3.  Shapes that the line was not drawn from, of 6 and 12 layers: 70B 64 tokens 2161 / 1973, 160 sequences
    # 2954 / 2749, 7B 40 tokens 1542 / 1314, 150 tokens 1886 / 1954 (one), the 405B rank shard 64 tokens 1118 / 1163 (one), 20 tokens 1217 / 1238
    # (two).  190 tokens of 8B 5493 / 5618, 400 7397 / 7483; from 4096 rows on 2 to 5 % less (4 x 1100 52681 / 51065, 8782 / 8459, 69048 / 68578,
    # 25597 / 24814), but 4 x 1250 of the 70B shard 77036 / 78132; in between either, by up to 5 %.
    parts_to, parts_from = 160, 4096
    passes_us, launches_us, short_us = 8.0, 6.0, 50.0

    def _in_parts(self, B: int, S: int) -> bool:
        rows = B * S
        if not 4 < rows <= self.parts_to:
            return rows >= self.parts_from
        if rows <= _hip.BANDS_TO:
            return True
        if (rows, S == 1) not in self._parts_pay:
            dim, fused, nqkv = self.config.dim, self._fused_width(), GPTBase._fused_width(self)
            one = _hip.linear_plan_us(rows, fused, dim)
            two = _hip.linear_plan_us(rows, nqkv, dim) + _hip.linear_plan_us(rows, fused - nqkv, dim, True)
            launches = self.launches_us if S > 1 and one <= self.short_us else 0.0
            self._parts_pay[rows, S == 1] = two - one <= self.passes_us + launches
        return self._parts_pay[rows, S == 1]

    def _run_layers_prompt(self, ws: Workspace, pos: Tensor, nqkv: int):
        """Prompts (and decode batches above 64): the rows of the fused input weight as two products, whose output passes rotate and cache, and
        apply the activation; y + x with the next norm.  Eight launches for the eleven of one product and passes over its rows."""
        cfg = self.config
        Hq, Hkv, hd = cfg.n_head_local, cfg.n_kv_local, cfg.head_dim
        pending = None
        for blk in self.layers:
            att, kv = blk.attention, blk.attention.kv_cache
            _hip.add_rmsnorm(ws.x, pending, None, blk.attention_norm.weight, None if pending is None else ws.x, ws.xn, cfg.norm_eps)
            w = att.wqkv1.weight
            _hip.linear_rope_kv(ws.xn, w[:nqkv], ws.qkv[:, :nqkv], self.freqs_cis, pos, kv.k_cache, kv.v_cache, ws.B, ws.S, Hq, Hkv, hd, ws.sums)
            self._attention(ws, blk, pos, None, ws.a, roped=True)
            _hip.linear_swiglu_out(ws.xn, w[nqkv:], ws.act, ws.h, ws.sums)
            _hip.linear(ws.act, att.w2.weight, ws.m, scratch=ws.sums)
            _hip.add(ws.m, ws.a, ws.m)                               # w2(...) + wo(...)
            pending = ws.m
            if not blk.keeps_residual:
                ws.x.copy_(ws.m)
                pending = None
        return pending, None

    def _run_layers_decode(self, ws: Workspace, pos: Tensor, nqkv: int):
        """Decode step through the weight-streaming bands.  The rows of the fused input weight are two projections
        of the same input: [q | k | v], rotated and cached on the way out, and [up | gate], stored as silu(gate) * up
        -- the second independent of the attention, whose launch it shares: up to 16 sequences as bands (lr_attn_decode_beside),
        above that as a product with partial sums (lr_attn_decode_beside_product; 8B, us per step, bands and an attention of its
        own before it: 20 sequences 4330 -> 4020, 32 4810 -> 4520; 48 4640 -> 4140).  wo and w2 share a launch.  Up to 16
        sequences that launch also updates the residual and leaves the next block its rows undivided (linear_resid): three
        launches per block instead of nine; above, and in the last block, y + x is left to the next norm launch (x + y: the same
        sum), six.  Above 32 sequences q/k/v, wo and w2 too are products of their own, with partial sums."""
        cfg = self.config
        Hq, Hkv, hd = cfg.n_head_local, cfg.n_kv_local, cfg.head_dim
        q = ws.qkv[:, :nqkv]
        pending, xn, xu = None, ws.xn, ws.xn
        products = ws.tickets is not None   # from 17 sequences on, where the library has the grid for the shape
        for blk, after in zip(self.layers, [*self.layers[1:], None]):
            att, kv = blk.attention, blk.attention.kv_cache
            if xn is ws.xn:
                _hip.add_rmsnorm(ws.x, pending, None, blk.attention_norm.weight, None if pending is None else ws.x, ws.xn,
                                 cfg.norm_eps)
            w = att.wqkv1.weight
            qkv = (xn, w[:nqkv], q, _hip.rope_kv_epilogue(self.freqs_cis, pos, kv.k_cache, kv.v_cache, Hq, Hkv, hd))
            up_gate = (xu, w[nqkv:], ws.act, _hip.EPI_SWIGLU)
            if ws.B > self.band_rows_to:
                _hip.linear_rope_kv(ws.xn, w[:nqkv], q, self.freqs_cis, pos, kv.k_cache, kv.v_cache, ws.B, 1, Hq, Hkv, hd, ws.sums)
                products = products and _hip.attn_decode_beside_product(q, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, Hq, Hkv, hd,
                                                                        ws.tickets, ws.xn, w[nqkv:], ws.act, ws.sums)
                if not products:
                    _hip.linear_swiglu_out(ws.xn, w[nqkv:], ws.act, sums=ws.sums)
                    _hip.attn_decode(q, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, Hq, Hkv, hd)
                _hip.linear(ws.y, att.wo.weight, ws.a, scratch=ws.sums)
                _hip.linear(ws.act, att.w2.weight, ws.m, scratch=ws.sums)
            elif ws.B <= 16:
                _hip.linear_multi(qkv)
                if not _hip.attn_decode_beside(q, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, Hq, Hkv, hd, up_gate,
                                               ws.tickets):
                    _hip.linear_multi(up_gate)
                    _hip.attn_decode(q, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, Hq, Hkv, hd)
            elif ws.pair_sums and products:
                _hip.linear_multi(qkv)
                products = _hip.attn_decode_beside_product(q, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, Hq, Hkv, hd, ws.tickets,
                                                           ws.xn, w[nqkv:], ws.act, ws.pair_sums[0])
                if not products:
                    _hip.linear_multi(up_gate)
                    _hip.attn_decode(q, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, Hq, Hkv, hd)
            else:
                _hip.linear_multi(qkv, up_gate)
                _hip.attn_decode(q, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, Hq, Hkv, hd)
            if ws.resid_sums and ws.B <= self.band_rows_to and after is not None and blk.keeps_residual:
                # both sums go to the residual and the next norm's undivided rows come with parts of their sums of squares,
                # which the q/k/v launch adds for up/gate (bands only: the products above read normed rows)
                _hip.linear_resid((ws.y, att.wo), (ws.act, att.w2, after.attention_norm.weight, ws.xn, ws.sq2), ws.x, joint=True)
                xn = _hip.Normed(ws.xn, ws.sq2, cfg.norm_eps, (ws.sq2, ws.sq2_total))
                xu, pending = _hip.Normed(ws.xn, ws.sq2_total, cfg.norm_eps), None
                continue
            xn = xu = ws.xn
            if ws.B <= self.band_rows_to:
                _hip.linear_multi((ws.y, att.wo.weight, ws.a, _hip.EPI_NONE), (ws.act, att.w2.weight, ws.m, _hip.EPI_NONE))
            _hip.add(ws.m, ws.a, ws.m)                               # w2(...) + wo(...)
            if blk.keeps_residual:
                pending = ws.m                                       # y + x: with the next norm
            else:
                ws.x.copy_(ws.m)
                pending = None
        return pending, None
