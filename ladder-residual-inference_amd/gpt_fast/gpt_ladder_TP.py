"""Ladder-Residual model on the gfx950 kernels.

Public surface of the reference's gpt_fast/gpt_ladder_TP.py: `GPTLadder` (:210-288) and
`LadderTransformerBlock` (:291-361) with the same children, `ModelArgs`, `transformer_configs`,
`find_multiple`.  The ladder schedule: each module (attention, then MLP) reads the residual stream
BEFORE the output of the module just ahead of it has been added; that output -- a row-parallel
partial sum, which in the reference is in flight in an asynchronous all-reduce -- is added one
module later.  Here the partial sum simply waits in a local buffer (`Workspace.a`, `Workspace.m`)
and the deferred add is fused with the next RMSNorm (lr_add_rmsnorm)."""
import torch
import torch.nn as nn
from torch import Tensor

from . import _hip
from ._model import GPTBase, Workspace
from .config import REGISTRIES, ModelArgs, find_multiple  # noqa: F401  (re-exported like the reference)
from .utils import Attention, FeedForward, RMSNorm, all_reduce_func

transformer_configs = REGISTRIES["ladder"]


class LadderTransformerBlock(nn.Module):
    def __init__(self, config: ModelArgs) -> None:
        super().__init__()
        self.attention = Attention(config)
        self.feed_forward = FeedForward(config)
        self.ffn_norm = RMSNorm(config.dim, config.norm_eps)
        self.attention_norm = RMSNorm(config.dim, config.norm_eps)
        self.semi_compiled_model = config.semi_compiled_model  # accepted; there is nothing to compile here

    def forward(self, previous_attention_out: Tensor, previous_mlp_out: Tensor, residual: Tensor, attention_handle,
                mlp_handle, input_pos: Tensor, freqs_cis: Tensor, mask: Tensor):
        """Reference signature (gpt_ladder_TP.py:312-358).  Handles are always None: nothing is in
        flight.  Returns (attention partial sum, mlp partial sum, residual, None, None)."""
        if attention_handle is not None:
            attention_handle.wait()
        residual = residual.contiguous()
        new_residual = torch.empty_like(residual)
        normed = torch.empty_like(residual)
        eps = self.attention_norm.eps
        _hip.add_rmsnorm(residual, previous_attention_out.contiguous(), None, self.attention_norm.weight, new_residual,
                         normed, eps)
        current_attention_out = self.attention(normed, freqs_cis, mask, input_pos)
        current_attention_out, attention_handle = all_reduce_func(current_attention_out, clone=False, async_op=True)

        if mlp_handle is not None:
            mlp_handle.wait()
        residual = torch.empty_like(new_residual)
        _hip.add_rmsnorm(new_residual, previous_mlp_out.contiguous(), None, self.ffn_norm.weight, residual, normed,
                         self.ffn_norm.eps)
        current_mlp_out = self.feed_forward(normed)
        current_mlp_out, mlp_handle = all_reduce_func(current_mlp_out, clone=False, async_op=True)
        return current_attention_out, current_mlp_out, residual, attention_handle, mlp_handle

    def extra_repr(self) -> str:
        return f"semi_compiled = {self.semi_compiled_model}"


class GPTLadder(GPTBase):
    family = "ladder"
    # decode steps of batch <= 2 run as ONE persistent kernel (lr_ladder_decode_step) when the shape
    # is supported; set to False to force the per-op kernels
    use_fused_step = True

    def _prompt_pieces(self):
        return self.config.ladder_layers is None and not hasattr(self.layers[0].attention.wqkv, "scales")   # (lr_ladder_block's)

    def _pair_bytes(self, B):
        c = self.config
        if c.ladder_layers is None and hasattr(self.layers[0].attention.wqkv, "scales"):
            outputs = _hip.linear_fp8_pieces_two_bytes(B, c.dim, c.n_head_local * c.head_dim, c.ffn_local)
            if not outputs or not self._all_fp8():
                return ()
            return max(outputs, _hip.linear_fp8_product_bytes(B, 2 * c.ffn_local, c.dim, pair=True),
                       _hip.linear_fp8_product_bytes(B, self._fused_width(), c.dim),
                       _hip.linear_fp8_product_bytes(B, c.output_rows, c.dim)), outputs
        if not self._prompt_pieces():
            return ()
        outputs = _hip.linear_pieces_two_bytes(B, c.dim, c.n_head_local * c.head_dim, c.ffn_local)
        return max(outputs, _hip.beside_product_bytes(B, 2 * c.ffn_local, c.dim)), outputs

    def _all_fp8(self):
        return all(hasattr(m, "scales") for b in self.layers for m in (b.attention.wqkv, b.attention.wo, b.feed_forward.w1, b.feed_forward.w2))

    def _make_block(self, config, layer_idx):
        return LadderTransformerBlock(config)

    def setup_caches(self, max_batch_size, max_seq_length):
        before = self.max_seq_length, self.max_batch_size
        super().setup_caches(max_batch_size, max_seq_length)
        if (self.max_seq_length, self.max_batch_size) != before:
            self._fused = {}

    def _fused_step(self, B: int):
        st = getattr(self, "_fused", None)
        if st is None:
            st = self._fused = {}
        if B not in st:
            # the one-kernel step implements the all-ladder schedule only, on bf16 weights or with every projection
            # (lm_head included) in weight-only e4m3
            kinds = {p.dtype for blk in self.layers for p in blk.state_dict().values() if p.dim() == 2}
            kinds.add(self.output.weight.dtype)
            ok = B <= 2 and self.config.ladder_layers is None and \
                kinds in ({torch.bfloat16}, {torch.float8_e4m3fn})
            st[B] = _hip.FusedLadderStep(self, B) if ok else None
            if st[B] is not None and not st[B].supported:
                st[B] = None
        return st[B]

    def forward(self, idx: Tensor, input_pos=None) -> Tensor:
        B, S = idx.shape
        if S == 1 and self.use_fused_step and B <= 2 and self.freqs_cis is not None:
            fused = self._fused_step(B)
            if fused is not None:
                return self.decode_step_fused(idx, input_pos)
        return super().forward(idx, input_pos)

    def decode_step_fused(self, idx: Tensor, input_pos: Tensor, advance: bool = False, history=None, pos0: int = 0):
        """One decode step through lr_ladder_decode_step.  Returns logits [B, 1, V]; the greedy token
        is left in the workspace's next_token buffer (see greedy_next).  With advance=True the step
        also writes the token into `idx` (must be int32), `history[:, pos - pos0]`, and bumps
        `input_pos` (must be int32) on the device."""
        B = idx.shape[0]
        fused = self._fused_step(B)
        ws = self._workspace(B, 1)
        tokens = idx if idx.dtype == torch.int32 else idx.to(torch.int32)
        pos = input_pos if input_pos.dtype == torch.int32 else input_pos.to(torch.int32)
        assert not advance or (tokens is idx and pos is input_pos), "advance needs int32 token and position buffers"
        fused.step(tokens.contiguous(), pos, ws.logits.view(B, -1), ws.next_token, advance,
                   tokens if advance else None, history, pos0)
        ws.next_token_valid_for = ws.logits
        return ws.logits

    def greedy_next(self, logits: Tensor) -> Tensor:
        ws = self._ws.get((logits.shape[0], 1, self.last_logits_only))
        if ws is not None and getattr(ws, "next_token_valid_for", None) is logits:
            return ws.next_token  # already chosen inside the fused step
        return super().greedy_next(logits)

    # Decode through the per-op kernels: run the attention chain and the MLP chain of a block on two streams.
    # Off by default: as parallel branches of a captured graph the chains do overlap, but every hand-over between
    # the two hardware queues costs more than the attention chain's latency that it hides (measured on the 70B rank
    # shard, ms per step with / without: batch 8 8.6 / 8.3, batch 64 18.2 / 18.8).  Putting one step of each chain
    # into the same grid instead (wqkv beside w1, attention beside w2) was slower still: 10.3 ms at batch 8.
    overlap_modules = False
    two_chains_from = _hip.BANDS_TO + 1   # decode batches from which the MLP chain is a parallel branch (see _run_layers_decode)

    def _run_layers_decode(self, ws: Workspace, pos: Tensor):
        """Decode step (S == 1) of an all-ladder model through the per-op kernels: one launch does both residual
        updates and both norms of a block (lr_ladder_norms: the MLP's input does not contain the block's own
        attention output), then the attention chain (wqkv, RoPE + cache write, attention, wo) and the MLP chain
        (w1, SwiGLU, w2) -- one after the other, or on two streams where the reference overlaps an all-reduce with
        the next module (gpt_ladder_TP.py:339-349).  Up to 16 rows the norms launch is only the first block's: from then on
        the output projections update the residual and leave the next block its rows undivided (linear_resid).  17 to 64
        rows share a grid between the attention and the up/gate product, and leave both outputs' partial sums to the norms; e4m3
        weights that those products do not serve (inner dimensions in 128s) are passes of up to 16 rows."""
        cfg = self.config
        eps = cfg.norm_eps
        main = side = None
        if self.overlap_modules:
            main = torch.cuda.current_stream()
            side = getattr(self, "_side_stream", None)
            if side is None or side.device != main.device:
                side = self._side_stream = torch.cuda.Stream(device=main.device)
        pending_a = pending_m = None
        # decode batches of up to 32 rows on bf16 weights (from 17 on where no shared grid serves): the block's two input projections share one launch of
        # the weight-streaming kernel (q/k/v -- rotated and cached on the way out -- next to up/gate, which stores
        # silu(gate) * up directly), and so do its two output projections (wo next to w2).  Also below 5 rows,
        # where single projections go to the matrix-vector kernel: five or six launches per block instead of nine
        # weigh more than the kernel (70B rank shard, ms per step: batch 1 4.9 / 5.5, batch 4 5.0 / 8.3)
        fp8 = hasattr(self.layers[0].attention.wqkv, "scales")
        multi = side is None and ws.B <= 64 and not fp8
        beside = multi and ws.B <= 16
        # Above 32 rows the projections are products with partial sums, whose launches leave room.  Where the attention cannot share
        # a grid with the up/gate product (below), the MLP chain (up/gate, w2) runs as a second branch of the captured graph beside
        # the attention chain (q/k/v, attention, wo) -- 70B rank shard, batch 64: 7.6 ms per step, one after the other 10.0; up to 32
        # rows, in bands, nothing moves (batch 32 7.35 / 7.31)
        two_chains = multi and not beside and ws.B >= self.two_chains_from
        # from 17 rows on (q/k/v in bands up to 32) the attention shares a grid with the up/gate product, and wo one with w2, both with
        # their partial sums left to the norms -- 70B rank shard, 64 rows at 2048 tokens: 6.59 ms per step, on two branches 7.13; 32
        # rows at 1000 tokens 5.78, in bands 7.02
        pair = ws.pair_sums
        products = multi and pair and (two_chains or ws.sums is None) and ws.tickets is not None
        # the same on e4m3 weights, q/k/v a product of its own at any of these numbers of rows
        products8 = side is None and fp8 and pair and ws.tickets is not None
        if two_chains:
            cur = torch.cuda.current_stream()
            chain = getattr(self, "_chain_stream", None)
            if chain is None or chain.device != cur.device:
                chain = self._chain_stream = torch.cuda.Stream(device=cur.device)
        # weight-only e4m3 projections, up to 16 rows: the same two launches per block (lr_linear_fp8_multi)
        multi8 = side is None and fp8 and ws.B <= 16
        beside8 = multi8   # (declined by the library for a single row, where the projections are no bands)
        # and beyond, the bands' launches for up to 16 rows at a time
        n = -(-ws.B // 16)
        parts = [slice(i * ws.B // n, (i + 1) * ws.B // n) for i in range(n)] if side is None and fp8 and 1 < n <= 4 else None
        xn, xn2 = ws.xn, ws.xn2
        resid = ws.resid_sums and (multi or multi8)
        for blk, after in zip(self.layers, [*self.layers[1:], None]):
            if not isinstance(xn, _hip.Normed):
                _hip.ladder_norms(ws.x, pending_a, pending_m, blk.attention_norm.weight, blk.ffn_norm.weight, ws.x, ws.xn,
                                  ws.xn2, eps)
            if products:
                att, ff, kv = blk.attention, blk.feed_forward, blk.attention.kv_cache
                heads = cfg.n_head_local, cfg.n_kv_local, cfg.head_dim
                if ws.sums is None:
                    rope = _hip.rope_kv_epilogue(self.freqs_cis, pos, kv.k_cache, kv.v_cache, *heads)
                    _hip.linear_multi((ws.xn, att.wqkv.weight, ws.qkv, rope))
                else:
                    _hip.linear_rope_kv(ws.xn, att.wqkv.weight, ws.qkv, self.freqs_cis, pos, kv.k_cache, kv.v_cache, ws.B, 1, *heads, ws.sums)
                products = _hip.attn_decode_beside_product(ws.qkv, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, *heads, ws.tickets,
                                                           ws.xn2, ff.w1.weight, ws.act, pair[0])
                if not products:
                    self._attention(ws, blk, pos, None, ws.a, roped=True)
                    self._mlp(ws, blk, ws.m, ws.xn2)
                elif after:
                    pending_a, pending_m = _hip.linear_pieces_two(ws.y, att.wo.weight, ws.a, pair[0], ws.act, ff.w2.weight, ws.m, pair[1])
                    continue
                else:
                    _hip.linear(ws.y, att.wo.weight, ws.a, scratch=ws.sums)
                    _hip.linear(ws.act, ff.w2.weight, ws.m, scratch=ws.sums_mlp)
            elif products8 and (products8 := self._block_products8(ws, blk, pos)):
                two = _hip.linear_fp8_pieces_two(ws.y, blk.attention.wo, pair[0], ws.act, blk.feed_forward.w2, pair[1]) if after else None
                if two:
                    pending_a, pending_m = two
                    continue
                self._linear(ws, ws.y, blk.attention.wo, ws.a)
                self._linear(ws, ws.act, blk.feed_forward.w2, ws.m)
            elif two_chains:
                chain.wait_stream(cur)
                with torch.cuda.stream(chain):
                    self._mlp(ws, blk, ws.m, ws.xn2)
                self._attention(ws, blk, pos, blk.attention.wqkv, ws.a)
                cur.wait_stream(chain)
            elif multi:
                kv = blk.attention.kv_cache
                rope = _hip.rope_kv_epilogue(self.freqs_cis, pos, kv.k_cache, kv.v_cache, cfg.n_head_local,
                                             cfg.n_kv_local, cfg.head_dim)
                up_gate = (xn2, blk.feed_forward.w1.weight, ws.act, _hip.EPI_SWIGLU)
                if beside:
                    # up to 16 rows the up/gate bands leave room for a second workgroup per CU: the attention's
                    # items run in the same launch and wait for the KV cache behind the weight stream
                    _hip.linear_multi((xn, blk.attention.wqkv.weight, ws.qkv, rope))
                    beside = _hip.attn_decode_beside(ws.qkv, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B,
                                                     cfg.n_head_local, cfg.n_kv_local, cfg.head_dim, up_gate, ws.tickets)
                    if not beside:
                        _hip.linear_multi(up_gate)
                        self._attention(ws, blk, pos, None, None, roped=True)
                else:
                    _hip.linear_multi((xn, blk.attention.wqkv.weight, ws.qkv, rope), up_gate)
                    self._attention(ws, blk, pos, None, None, roped=True)
                if not (resid and after):
                    xn, xn2 = ws.xn, ws.xn2
                    _hip.linear_multi((ws.y, blk.attention.wo.weight, ws.a, _hip.EPI_NONE),
                                      (ws.act, blk.feed_forward.w2.weight, ws.m, _hip.EPI_NONE))
            elif multi8:
                att, ff, kv = blk.attention, blk.feed_forward, blk.attention.kv_cache
                rope = _hip.rope_kv_epilogue(self.freqs_cis, pos, kv.k_cache, kv.v_cache, cfg.n_head_local,
                                             cfg.n_kv_local, cfg.head_dim)
                qkv8 = (xn, att.wqkv.weight, att.wqkv.scales, ws.qkv, rope)
                up_gate8 = (xn2, ff.w1.weight, ff.w1.scales, ws.act, _hip.EPI_SWIGLU)
                if beside8:
                    _hip.linear_fp8_multi(qkv8)
                    beside8 = _hip.attn_decode_beside_fp8(ws.qkv, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B,
                                                          cfg.n_head_local, cfg.n_kv_local, cfg.head_dim, up_gate8, ws.tickets)
                    if not beside8:
                        _hip.linear_fp8_multi(up_gate8)
                        self._attention(ws, blk, pos, None, None, roped=True)
                else:
                    _hip.linear_fp8_multi(qkv8, up_gate8)
                    self._attention(ws, blk, pos, None, None, roped=True)
                if not (resid and after):
                    xn, xn2 = ws.xn, ws.xn2
                    _hip.linear_fp8_multi((ws.y, att.wo.weight, att.wo.scales, ws.a, _hip.EPI_NONE),
                                          (ws.act, ff.w2.weight, ff.w2.scales, ws.m, _hip.EPI_NONE))
            elif parts:
                att, ff, kv = blk.attention, blk.feed_forward, blk.attention.kv_cache
                for r in parts:
                    rope = _hip.rope_kv_epilogue(self.freqs_cis, pos, kv.k_cache[r], kv.v_cache[r], cfg.n_head_local, cfg.n_kv_local,
                                                 cfg.head_dim)
                    _hip.linear_fp8_multi((ws.xn[r], att.wqkv.weight, att.wqkv.scales, ws.qkv[r], rope),
                                          (ws.xn2[r], ff.w1.weight, ff.w1.scales, ws.act[r], _hip.EPI_SWIGLU))
                self._attention(ws, blk, pos, None, None, roped=True)
                for r in parts:
                    _hip.linear_fp8_multi((ws.y[r], att.wo.weight, att.wo.scales, ws.a[r], _hip.EPI_NONE),
                                          (ws.act[r], ff.w2.weight, ff.w2.scales, ws.m[r], _hip.EPI_NONE))
            elif side is not None:
                side.wait_stream(main)
                with torch.cuda.stream(side):
                    self._mlp(ws, blk, ws.m, ws.xn2)
                self._attention(ws, blk, pos, blk.attention.wqkv, ws.a)
                main.wait_stream(side)
            else:
                self._attention(ws, blk, pos, blk.attention.wqkv, ws.a)
                self._mlp(ws, blk, ws.m, ws.xn2)
            pending_a, pending_m = ws.a, ws.m
            if resid and after:
                _hip.linear_resid((ws.y, blk.attention.wo, after.attention_norm.weight, ws.xn, ws.sq),
                                  (ws.act, blk.feed_forward.w2, after.ffn_norm.weight, ws.xn2, ws.sq2), ws.x)
                if beside or beside8:   # (up/gate has its own, larger launch: q/k/v's adds the parts of its sums of squares)
                    xn, xn2 = _hip.Normed(ws.xn, ws.sq, eps, (ws.sq2, ws.sq2_total)), _hip.Normed(ws.xn2, ws.sq2_total, eps)
                else:
                    xn, xn2 = _hip.Normed(ws.xn, ws.sq, eps), _hip.Normed(ws.xn2, ws.sq2, eps)
        return pending_a, pending_m

    def _linear(self, ws: Workspace, x: Tensor, lin, out: Tensor):
        # (e4m3, 17 to 64 rows: the head 16032 x 8192 of 64 rows in one product instead of four passes)
        if not (ws.S == 1 and hasattr(lin, "scales") and ws.pair_sums and _hip.linear_fp8_product(x, lin, out, ws.pair_sums[0])):
            super()._linear(ws, x, lin, out)

    def _block_products8(self, ws: Workspace, blk, pos: Tensor) -> bool:
        """q/k/v, then the attention in one grid with up/gate, all as e4m3 products of 17 to 64 rows: ws.xn, ws.xn2 -> ws.y, ws.act.
        False, with ws.qkv and the caches rewritten at most, where the library has no such grid."""
        cfg, att, ff, kv = self.config, blk.attention, blk.feed_forward, blk.attention.kv_cache
        heads = cfg.n_head_local, cfg.n_kv_local, cfg.head_dim
        rope = _hip.rope_kv_epilogue(self.freqs_cis, pos, kv.k_cache, kv.v_cache, *heads)
        return (_hip.linear_fp8_product(ws.xn, att.wqkv, ws.qkv, ws.pair_sums[0], rope)
                and _hip.attn_decode_beside_product_fp8(ws.qkv, kv.k_cache, kv.v_cache, pos, ws.y, ws.scratch, ws.B, *heads, ws.tickets,
                                                        ws.xn2, ff.w1, ws.act, ws.pair_sums[0]))

    def _run_layers(self, ws: Workspace, pos: Tensor):
        cfg = self.config
        eps = cfg.norm_eps
        if ws.S == 1 and cfg.ladder_layers is None:
            return self._run_layers_decode(ws, pos)
        pending_a = pending_m = None  # the reference starts from zero tensors; adding zero is the identity
        if cfg.ladder_layers is None:
            # all-ladder prefill: both residual updates and both norms of a block in one pass over the rows
            # (lr_ladder_norms, as in decode: six tensor passes instead of the eight of two lr_add_rmsnorm); on bf16 weights
            # a block is one call (1B, 128 tokens: a prompt in 440 us of host time, 1250 in a call per kernel)
            if ws.S > 1 and ws.rows > 4:
                blocks = [(blk.attention_norm.weight, blk.ffn_norm.weight, att.wqkv.weight, att.wo.weight, ff.w1.weight, ff.w2.weight,
                           att.kv_cache.k_cache, att.kv_cache.v_cache)
                          for blk in self.layers for att, ff in ((blk.attention, blk.feed_forward),)]
                if all(t.dtype == torch.bfloat16 for b in blocks for t in b):
                    _hip.ladder_blocks(blocks, ws, self.freqs_cis, pos, cfg.n_head_local, cfg.n_kv_local, cfg.head_dim, eps)
                    return ws.a, ws.m
            for blk in self.layers:
                _hip.ladder_norms(ws.x, pending_a, pending_m, blk.attention_norm.weight, blk.ffn_norm.weight, ws.x,
                                  ws.xn, ws.xn2, eps)
                self._attention(ws, blk, pos, blk.attention.wqkv, ws.a)
                self._mlp(ws, blk, ws.m, ws.xn2)
                pending_a, pending_m = ws.a, ws.m
            return pending_a, pending_m
        for i, blk in enumerate(self.layers):
            if cfg.is_ladder_layer(i):
                _hip.add_rmsnorm(ws.x, pending_a, None, blk.attention_norm.weight, ws.x, ws.xn, eps)
                self._attention(ws, blk, pos, blk.attention.wqkv, ws.a)
                pending_a = ws.a
                _hip.add_rmsnorm(ws.x, pending_m, None, blk.ffn_norm.weight, ws.x, ws.xn, eps)
                self._mlp(ws, blk, ws.m)
                pending_m = ws.m
            else:
                # a dense layer of a partial-ladder model (modeling_llama_ladder.py:614-637): it sees everything
                # produced so far, adds its attention output at once, and leaves its MLP output pending -- the
                # next layer adds it first (dense) or after its attention (ladder: "prev_attn_output" is this
                # layer's state before the MLP output, :644-658)
                _hip.add_rmsnorm(ws.x, pending_a, pending_m, blk.attention_norm.weight, ws.x, ws.xn, eps)
                self._attention(ws, blk, pos, blk.attention.wqkv, ws.a)
                _hip.add_rmsnorm(ws.x, ws.a, None, blk.ffn_norm.weight, ws.x, ws.xn, eps)
                self._mlp(ws, blk, ws.m)
                pending_a, pending_m = None, ws.m
        return pending_a, pending_m
