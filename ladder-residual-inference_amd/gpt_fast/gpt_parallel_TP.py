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
            if N == self._fused_width():   # (its two parts)
                yield rows, nqkv, K, False
                yield rows, N - nqkv, K, True

    def _run_layers(self, ws: Workspace, pos: Tensor):
        cfg = self.config
        nqkv = (cfg.n_head_local + 2 * cfg.n_kv_local) * cfg.head_dim
        att0 = self.layers[0].attention
        if not any(hasattr(m, "scales") for m in (att0.wqkv1, att0.wo, att0.w2)):
            if ws.S == 1 and self.band_rows_from <= ws.B <= 64:
                return self._run_layers_decode(ws, pos, nqkv)
            if 4 < ws.rows <= self.parts_to or ws.rows >= self.parts_from:
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

    # Rows of a prompt up to which, and from which on, the fused input weight is two products: few rows are launches, many are passes over
    # the products' rows; in between one product leaves less of the last round of tiles empty (8B, us per prompt, one / two: 30 tokens
    # 4391 / 4288, 50 4414 / 3797, 100 4986 / 4479, 150 5381 / 5165, 190 5462 / 5592, 400 7718 / 7878, 666 10134 / 10330, 4 x 2000 92032 / 89111, of which
    # the attention's own gain is 1750; 220 to 300 and 600 to 2300 no difference but the attention's)
    parts_to, parts_from = 160, 4096

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
