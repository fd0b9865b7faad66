"""Lasivik: a post-norm hybrid decoder on the gfx950 kernels.

Every layer is a token mixer (gated linear attention, retention or windowed latent attention, in the order the
configuration lists) and an optional gated feed-forward; the residual is re-normalised after each sum:
    x <- norm1(alpha x + mixer(x)),   x <- norm2(alpha x + ff(x))
with gains stored around zero.  The residual stream is fp32; projections, caches and activations are bf16, or fp32 when
the model's parameters are.  Recurrent states live in fp32.  A call at position 0 starts every sequence of the batch
anew, so a cache slot is reused without being cleared; later calls continue where the previous one ended (input_pos must
be consecutive)."""
from types import SimpleNamespace

import torch
import torch.nn as nn
from torch import Tensor

from . import _hip
from ._hybrid import GPTHybrid, HybridWorkspace
from .config import REGISTRIES, LasivikArgs, LayerArgs
from .mixers import MIXERS, pad8, project
from .utils import FeedForward, RMSNorm

transformer_configs = REGISTRIES["lasivik"]


class LasivikWorkspace(HybridWorkspace):
    def __init__(self, model: "GPTLasivik", B: int, S: int, dtype, device, all_logits: bool):
        super().__init__(model, B, S, dtype, device, all_logits)
        e, rows = self._empty, self.rows
        ff = max([blk.feed_forward.w2.in_features for blk in model.layers if blk.feed_forward is not None], default=0)
        self._h, self._act = e(rows * 2 * ff), e(rows * ff)
        # zeroed once: the padding columns of a mixer's output stay zero
        self._y = {}
        for m in (blk.mixer for blk in model.layers):
            key = (m.y_cols, m.args.heads * m.args.vdim)
            if key not in self._y:
                self._y[key] = torch.zeros(rows, m.y_cols, dtype=dtype, device=device)
        # the parts of the rows' sums of squares behind a mixer and behind a feed-forward, see _run_layers_decode
        self.sq = None
        if S == 1 and model.norms_in_projections(B) and dtype == torch.bfloat16 and device.type == "cuda" and model.config.width == model.config.dim:
            n = _hip.linear_residual_rms_sums(model.config.dim)
            self.sq = tuple(e(rows, n, dt=torch.float32) for _ in range(2)) if n else None

    def y_of(self, cols: int, used: int) -> Tensor:
        return self._y[(cols, used)]

    def ffn(self, I: int):
        return self._h[:self.rows * 2 * I].view(self.rows, 2 * I), self._act[:self.rows * I].view(self.rows, I)


class HybridBlock(nn.Module):
    def __init__(self, config: LasivikArgs, layer: LayerArgs):
        super().__init__()
        self.mixer = MIXERS[layer.mixer.kind](config.dim, layer.mixer, config.norm_eps)
        self.mixer_norm = RMSNorm(config.dim, config.norm_eps)
        self.feed_forward = self.ffn_norm = None
        if layer.ffn is not None:
            self.feed_forward = FeedForward(SimpleNamespace(dim=config.dim, intermediate_size=pad8(layer.ffn),
                                                            tp_world_size=1))
            self.ffn_norm = RMSNorm(config.dim, config.norm_eps)


class GPTLasivik(GPTHybrid):
    family = "lasivik"
    workspace_class = LasivikWorkspace

    def _make_block(self, config, layer_idx):
        return HybridBlock(config, config.layers[layer_idx])

    def _embed(self, ws, idx):
        _hip.embed_residual(self.tok_embeddings.weight, idx.contiguous(), ws.x, ws.xc, self.config.embedding_scale)

    def _norm_into(self, ws, norm: RMSNorm, alpha, d):
        """x <- norm(alpha x + d), in fp32 and in the compute type."""
        _hip.residual_rmsnorm(ws.x, alpha, d, norm.weight, ws.x, ws.xc, norm.eps, self.config.width, gain_offset=1.0)

    # Decode batches from which a norm is part of the projections on either side of it.  (Two rows' wide projections, which are the
    # matrix-vector kernel's otherwise, see project, take 2 us longer in bands and the two norms of a layer 10: 4 % of an 8B step at 1000
    # tokens, 2 % of a 1B one.  One row is the matrix-vector kernel's throughout.)
    norms_in_projections_from = 2

    def norms_in_projections(self, B: int) -> bool:
        """Rows wider than 6144, two bands' worth of columns per workgroup and more: up to 8 of them (us of an output projection with its norm
        and the projection behind, norm inside / in a launch of its own: 6144 x 6144 and 12288 x 6144, 16 rows 47.6 / 49.3; 8192 x 8192 and 16384 x
        8192, 2 rows 68.2 / 71.2, 8 rows 70.4 / 70.5, 9 rows 72.3 / 71.0; 12288 x 4096 and 8192 x 12288, 8 rows 56.0 / 56.6, 16 rows 63.0 / 60.4)."""
        return self.norms_in_projections_from <= B <= (_hip.ROW_NORM_MAX_ROWS if self.config.dim <= 6144 else 8)

    def _run_layers_decode(self, ws, pos):
        """Decode step of up to 16 rows: an output projection updates the residual and leaves the rows with the norm's gain and their
        sums of squares, by which the next projection divides (linear_residual_rms)."""
        alpha, x, last = self.config.residual_scale, ws.xc, None    # last: (sums, gain, eps), what ws.x still lacks

        def add(y, lin, norm):
            sq = ws.sq[last is not None and last[0] is ws.sq[0]]    # (one pair of parts is read while the other is written)
            _hip.linear_residual_rms(y, lin.weight, ws.x, alpha, last, norm.weight, 1.0, ws.xc, sq)
            return _hip.Normed(ws.xc, sq, norm.eps), (sq, norm.weight, norm.eps)

        for blk in self.layers:
            m, ff = blk.mixer, blk.feed_forward
            y = m._y(ws)
            m.mix(ws, pos, project(x, m.in_proj, ws.proj[:, :m.proj_cols], ws.sums), y)
            x, last = add(y, m.out_proj, blk.mixer_norm)
            if ff is not None:
                act = ws.ffn(ff.w2.in_features)[1]
                _hip.linear_multi((x, ff.w1.weight, act, _hip.EPI_SWIGLU))
                x, last = add(act, ff.w2, blk.ffn_norm)
        _hip.residual_rmsnorm(ws.x, 1.0, None, last[1], ws.x, ws.xc, last[2], self.config.width, gain_offset=1.0)
        return None, None

    def _run_layers(self, ws, pos):
        if ws.sq is not None:
            return self._run_layers_decode(ws, pos)
        alpha = self.config.residual_scale
        for blk in self.layers:
            blk.mixer.run(ws, pos)
            self._norm_into(ws, blk.mixer_norm, alpha, ws.d)
            if blk.feed_forward is not None:
                self._feed_forward(ws, blk.feed_forward)
                self._norm_into(ws, blk.ffn_norm, alpha, ws.d)
        return None, None

    def _feed_forward(self, ws, ff: FeedForward):
        h, act = ws.ffn(ff.w2.in_features)
        if ws.xc.dtype == torch.float32:
            _hip.linear(ws.xc, ff.w1.weight, h)
            _hip.swiglu(h, act)
        else:
            _hip.linear_swiglu_out(ws.xc, ff.w1.weight, act, h, ws.sums)
        project(act, ff.w2, ws.d, ws.sums)

    def _head(self, ws, d1, d2):
        cfg = self.config
        x, xc = ws.x, ws.xc
        if ws.last_rows is not None:
            x, xc = self._last(ws, ws.x)
        _hip.residual_rmsnorm(x, 1.0, None, self.norm.weight, None, xc, cfg.norm_eps, cfg.width, gain_offset=1.0)
        logits = ws.logits.flatten(0, 1)
        project(xc, self.output, logits, ws.sums)
        _hip.logit_cap(logits, cfg.logit_scale, cfg.logit_softcap)
        return ws.logits
