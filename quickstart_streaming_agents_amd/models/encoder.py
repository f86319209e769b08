"""On-GPU embedding encoder (K1): bge-small-class transformer -> 1536-d.

Replaces the managed embedding models (titan-embed-v1 / ada-002, both
1536-d — terraform/core/main.tf:529,563; dims contract validate.py:56-62).
A bge-small-class bidirectional encoder (12 layers, 384 hidden, attention
block 8 heads x 64 = 512 so the head geometry matches the MFMA kernels)
with a projection head to EMBED_DIM=1536 and L2 normalization.
Random-init weights (air-gapped): embeddings are deterministic and
well-distributed; the retrieval CONTRACT (dims, cosine, top-k) is what the
pipelines rely on.

On the GPU the tokens of a batch are rows without padding: the projections are
kernels of our own with the activation inside, and attention runs on the
projection's rows as they are (ops/hip/encoder_attn.hip) — no padded bmm, no
materialized score matrix.  The CPU path keeps a padded bmm + masked-softmax
reference of the same semantics (GPU-vs-CPU parity test in
tests/test_gpu_models.py).
"""

from __future__ import annotations

from dataclasses import dataclass

import numpy as np
import torch
import torch.nn.functional as F

from ..ops import dispatch as D
from ..ops import have_ext, have_lm_ext, lm_ext
from ..vector.index import EMBED_DIM
from .layers import ints_to_device
from .tokenizer import BpeTokenizer


@dataclass
class EncoderConfig:
    name: str = "bge-small"
    vocab_size: int = 30_522
    hidden: int = 384
    n_layers: int = 12
    n_heads: int = 8          # attention block 8 x 64 (kernel geometry)
    d_head: int = 64
    ffn: int = 1536
    max_pos: int = 512
    out_dim: int = EMBED_DIM
    norm_eps: float = 1e-5

    @property
    def attn_dim(self) -> int:
        return self.n_heads * self.d_head


class EmbeddingEncoder:
    def __init__(self, cfg: EncoderConfig | None = None, device: str = "cuda",
                 dtype=torch.bfloat16, seed: int = 1):
        self.cfg = cfg or EncoderConfig()
        c = self.cfg
        self.device = device
        self.dtype = dtype
        self.tokenizer = BpeTokenizer(c.vocab_size)
        gen_dev = device if str(device).startswith("cuda") else "cpu"
        g = torch.Generator(device=gen_dev).manual_seed(seed)

        def w(*shape, std=0.02):
            # generate on-device: 8B-class random init in seconds, no 32 GB
            # host spike
            t = torch.randn(*shape, generator=g, dtype=torch.float32,
                            device=gen_dev) * std
            return t.to(device=device, dtype=dtype)

        self.tok_embed = w(c.vocab_size, c.hidden)
        self.layers = [{
            "attn_norm": torch.ones(c.hidden, device=device, dtype=dtype),
            "mlp_norm": torch.ones(c.hidden, device=device, dtype=dtype),
            "wqkv": w(3 * c.attn_dim, c.hidden),
            "wo": w(c.hidden, c.attn_dim),
            "wgu": w(2 * c.ffn, c.hidden),
            "wdown": w(c.hidden, c.ffn),
        } for _ in range(c.n_layers)]
        self.final_norm = torch.ones(c.hidden, device=device, dtype=dtype)
        self.proj = w(c.out_dim, c.hidden)
        half = c.d_head // 2
        inv = 1.0 / (10_000.0 ** (torch.arange(half, dtype=torch.float64) / half))
        ang = torch.outer(torch.arange(c.max_pos, dtype=torch.float64), inv)
        self.rope_cos = ang.cos().float().to(device)
        self.rope_sin = ang.sin().float().to(device)
        self.scale = 1.0 / (c.d_head ** 0.5)
        self._use_hip = str(device).startswith("cuda")

    def _linear(self, x: torch.Tensor, w: torch.Tensor,
                glu: bool = False, parts: bool = False) -> torch.Tensor:
        """x W^T (`parts`: for the residual's norm), with glu silu(gate) * up of
        it, w = [gate; up] (GPU).  Few tiles are short_gemm's
        (ops/hip/short_gemm.hip: 384 x 512 at 400 rows 3.6 us, 4.5 in rows_gemm,
        5.5 in the library; of long K up to 32 rows: beyond, rows_gemm's shares of K,
        which the norm adds, are sooner, 384 x 1536 with its norm at 33 / 130 / 320
        rows 6.4 / 6.7 / 7.2, 7.6 / 8.0 / 8.8 here), the others rows_gemm's or
        wide_gemm's: at 8800 rows
        1536 x 384 takes 16.5 us (short_gemm 20.7, the library 18.3), 3072 x 384
        with the activation 30 (34, 72 with a pass of its own), 384 x 512 7.4
        (10.5, 10.7), 384 x 1536 14.1 (23.4, 17.2)."""
        n, k = w.shape
        if x.dtype == w.dtype == torch.bfloat16 and \
                D.ext().short_gemm_takes(x.shape[0], n, k):
            return D.ext().short_gemm(x, w, glu)
        if not glu:
            return D.linear_parts(x, w) if parts else D.linear(x, w)
        if D.glu_linear_ok(x, w):
            return D.glu_linear(x, w, "silu", rounded=False)
        y = F.linear(x, w)
        return D.swiglu(y[:, :n // 2], y[:, n // 2:])

    @property
    def _project(self):
        return self._linear if have_lm_ext() else self._linear_alone

    def _linear_alone(self, x: torch.Tensor, w: torch.Tensor,
                      glu: bool = False, parts: bool = False) -> torch.Tensor:
        """The same with qsa_hip alone: the others are qsa_lm_hip's."""
        n, k = w.shape
        if x.dtype == w.dtype == torch.bfloat16 and k % 64 == 0 and \
                n % 32 == 0 and (k <= 512 or x.shape[0] <= 2048):
            return D.ext().short_gemm(x, w, glu)
        y = F.linear(x, w)
        return D.swiglu(y[:, :n // 2], y[:, n // 2:]) if glu else y

    # -- varlen attention plumbing (GPU path) ------------------------------
    QROWS = 64      # query tokens per attention block: one 16-row tile a wave

    def _embed_rows(self, ids: np.ndarray, lens: np.ndarray) -> torch.Tensor:
        """Mean-pooled final states [n, hidden] f32 of texts whose tokens follow
        each other in ids, all rows in one concatenation without padding."""
        dev, n = self.device, len(lens)
        off = np.cumsum(lens) - lens
        nqb = -(-lens // self.QROWS)
        qb_item = np.repeat(np.arange(n), nqb)
        qb_pos0 = (np.arange(int(nqb.sum()))
                   - (np.cumsum(nqb) - nqb)[qb_item]) * self.QROWS
        toks, qb_item, qb_pos0, off, lens_t = ints_to_device(
            dev, ids, qb_item, qb_pos0, off, lens)
        res = self.tok_embed.index_select(0, toks)
        final_h = self._native_layers(res, qb_item, qb_pos0, off, lens_t)
        if final_h is None:
            final_h = self._layers_by_call(res, qb_item, qb_pos0, off, lens_t)
        return D.ext().mean_rows(final_h, off, lens_t)

    def _native_layers(self, res, qb_item, qb_pos0, off, lens):
        """All layers as one call that launches the kernels of _layers_by_call, or
        None where it does not take them, or where a product is not _linear's."""
        if not have_lm_ext() or type(res) is not torch.Tensor or \
                torch.compiler.is_compiling() or \
                getattr(self._project, "__func__", None) is not \
                EmbeddingEncoder._linear:
            return None
        c = self.cfg
        weights = [Ly[k] for Ly in self.layers for k in
                   ("attn_norm", "mlp_norm", "wqkv", "wo", "wgu", "wdown")]
        return lm_ext().encoder_layers(
            res, weights, self.final_norm, self.rope_cos, self.rope_sin,
            qb_item, qb_pos0, off, lens, c.n_heads, self.scale, c.norm_eps)

    def _layers_by_call(self, res, qb_item, qb_pos0, off, lens):
        c, project = self.cfg, self._project
        mlp_out = None
        for Ly in self.layers:
            if mlp_out is None:
                h = D.rmsnorm(res, Ly["attn_norm"], c.norm_eps)
            else:
                h = D.rmsnorm_residual(mlp_out, res, Ly["attn_norm"],
                                       c.norm_eps)
            attn = D.ext().encoder_attn(
                project(h, Ly["wqkv"]), self.rope_cos, self.rope_sin,
                qb_item, qb_pos0, off, lens, c.n_heads, self.scale)
            o = project(attn, Ly["wo"], parts=True)
            h = D.rmsnorm_residual(o, res, Ly["mlp_norm"], c.norm_eps)
            act = project(h, Ly["wgu"], glu=True)
            mlp_out = project(act, Ly["wdown"], parts=True)
        return D.rmsnorm_residual(mlp_out, res, self.final_norm, c.norm_eps)

    def _embed_padded(self, enc: list[list[int]]) -> torch.Tensor:
        """The same by a padded batch and a materialized softmax (CPU)."""
        c = self.cfg
        n = len(enc)
        L = max(len(x) for x in enc)
        T = n * L
        toks = torch.zeros(n, L, dtype=torch.int64, device=self.device)
        for i, x in enumerate(enc):
            toks[i, :len(x)] = torch.tensor(x, dtype=torch.int64)
        lens = torch.tensor([len(x) for x in enc], dtype=torch.int32,
                            device=self.device)
        positions = torch.arange(L, dtype=torch.int32, device=self.device) \
            .repeat(n).contiguous()
        # per-row score limits: row = (seq, head, qpos) -> seq len
        row_limits = lens.repeat_interleave(c.n_heads * L).contiguous()
        res = self.tok_embed.index_select(0, toks.reshape(-1)).contiguous()
        h = None
        mlp_out = None
        for li, Ly in enumerate(self.layers):
            if li == 0:
                h = D.rmsnorm(res, Ly["attn_norm"], c.norm_eps)
            else:
                h = D.rmsnorm_residual(mlp_out, res, Ly["attn_norm"],
                                       c.norm_eps)
            qkv = F.linear(h, Ly["wqkv"])
            A = c.attn_dim
            q = qkv[:, :A].reshape(T, c.n_heads, c.d_head).contiguous()
            k = qkv[:, A:2 * A].reshape(T, c.n_heads, c.d_head).contiguous()
            v = qkv[:, 2 * A:].reshape(T, c.n_heads, c.d_head).contiguous()
            D.rope_inplace(q, k, self.rope_cos, self.rope_sin, positions)
            # [n*heads, L, D] padded bmm reference
            qh = q.reshape(n, L, c.n_heads, c.d_head).permute(0, 2, 1, 3) \
                .reshape(n * c.n_heads, L, c.d_head)
            kh = k.reshape(n, L, c.n_heads, c.d_head).permute(0, 2, 1, 3) \
                .reshape(n * c.n_heads, L, c.d_head)
            vh = v.reshape(n, L, c.n_heads, c.d_head).permute(0, 2, 1, 3) \
                .reshape(n * c.n_heads, L, c.d_head)
            scores = (torch.bmm(qh.float(), kh.float().transpose(1, 2))
                      * self.scale).reshape(n * c.n_heads * L, L) \
                .contiguous()
            D.softmax_rows_(scores, 0, False, 0, row_limits)
            attn = torch.bmm(scores.reshape(n * c.n_heads, L, L),
                             vh.float())
            attn = attn.reshape(n, c.n_heads, L, c.d_head) \
                .permute(0, 2, 1, 3).reshape(T, A).to(self.dtype) \
                .contiguous()
            o = F.linear(attn, Ly["wo"])
            h = D.rmsnorm_residual(o, res, Ly["mlp_norm"], c.norm_eps)
            gu = F.linear(h, Ly["wgu"])
            act = D.swiglu(gu[:, :c.ffn], gu[:, c.ffn:])
            mlp_out = F.linear(act, Ly["wdown"])
        final_h = D.rmsnorm_residual(mlp_out, res, self.final_norm,
                                     c.norm_eps)
        hs = final_h.reshape(n, L, c.hidden).float()
        valid = (torch.arange(L, device=self.device).unsqueeze(0)
                 < lens.unsqueeze(1)).unsqueeze(-1)
        hs = torch.where(valid, hs, torch.zeros((), device=self.device))
        return hs.sum(dim=1) / valid.float().sum(dim=1).clamp(min=1)

    @torch.no_grad()
    def embed_batch(self, texts: list[str]):
        if not texts:
            return np.zeros((0, self.cfg.out_dim), dtype=np.float32)
        c = self.cfg
        ids, lens = self.tokenizer.encode_batch(list(texts), c.max_pos)
        # mean over the tokens, project, L2-normalize
        if self._use_hip and have_ext():
            out = self._project(self._embed_rows(ids, lens).to(self.dtype),
                                self.proj)
        else:
            enc = [x.tolist() for x in np.split(ids, np.cumsum(lens)[:-1])]
            out = F.linear(self._embed_padded(enc).to(self.dtype), self.proj)
        out = out.float()
        out = out / out.norm(dim=-1, keepdim=True).clamp(min=1e-9)
        return out.cpu().numpy()

    def embed(self, text: str):
        return self.embed_batch([text])[0]
