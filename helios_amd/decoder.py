"""The reference's Qwen3 decoder forward for packed ticks, on the paged-KV path.

Mirrors Qwen3Model._forward_packed (src/helios/runtime/qwen3/model.py:92-110) and the
TransformerBlock / GroupedQueryAttention / FeedForward forwards it runs
(layers.py:13-27, :131-164, :202-232), with random-init weights (no checkpoint is
fetched). This is the caller of the hot path, kept to measure it in place: torch runs
the products on hipBLASLt, with one launch for each step between them
(``ops.add_rms_norm``, ``ops.swiglu``), or, for a few rows, products that take those steps
along (``ops.block_linear``), and the attention step goes through
``PackedBatchCache.attend_projected`` (fused q/k norm + RoPE + KV append, then paged
attention). With ``fused_rope=False`` everything but the attention is the reference's own
sequence of torch operations (norms, RoPE, SiLU, then ``attend``).

The q, k and v projections are one GEMM over concatenated weights, and gate/up another;
the arithmetic is otherwise the reference's.
"""

from __future__ import annotations

import torch

from helios_amd import ops
from helios_amd.config import Qwen3Config
from helios_amd.paged_cache import PackedBatchCache


def _rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """RMSNorm.forward (layers.py:36-40)."""
    dtype = x.dtype
    x = x.float()
    return (x * torch.rsqrt(x.pow(2).mean(dim=-1, keepdim=True) + eps) * weight).to(dtype)


def _rope_tables(config: Qwen3Config, device) -> tuple[torch.Tensor, torch.Tensor]:
    """rope_parameters (layers.py:43-51)."""
    inv = 1.0 / (config.rope_base ** (torch.arange(0, config.head_dim, 2, dtype=torch.float32) / config.head_dim))
    angles = torch.arange(config.context_length, dtype=torch.float32).unsqueeze(1) * inv.unsqueeze(0)
    angles = torch.cat((angles, angles), dim=1)
    return torch.cos(angles).to(device), torch.sin(angles).to(device)


def _apply_rope(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor) -> torch.Tensor:
    """apply_rope with position_ids (layers.py:54-72)."""
    half = x.shape[-1] // 2
    c = cos[positions].unsqueeze(1)
    s = sin[positions].unsqueeze(1)
    return (x * c + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * s).to(x.dtype)


# Ticks of at most this many rows run their products through ops.block_linear: a layer's four
# products and the steps between them take 62-71 us that way and 102 us on hipBLASLt at up to
# 16 rows (one MFMA row tile); at 17-32 rows hipBLASLt's take 77-82 us, a second row tile 88-94.
# That is hidden 2560, ffn 9728, 32/8 heads of 128. At other widths, 1 / 8 / 16 rows against
# hipBLASLt: 256 and 768 12 / 14 / 15 us against 28 / 30 / 30; 1024 and 3072 20 / 21 / 24 against
# 39 / 40 / 40; 2048 and 6144 37 / 40 / 44 against 52; 4096 and 12288 85 / 88 / 100 against 99 /
# 100 / 101; 5120 and 17408 165 / 177 / 207 against 243 / 248 / 252; 8192 and 28672 304 / 314 /
# 356 against 346 / 347 / 352.
FEW_ROWS = 16


class PagedQwen3Decoder:
    """Random-init Qwen3 weights in the reference's layout, on one device."""

    def __init__(self, config: Qwen3Config, device, *, seed: int = 0, std: float = 0.02) -> None:
        self.config = config
        self.device = torch.device(device)
        g = torch.Generator(device=self.device).manual_seed(seed)
        dt = config.dtype
        hq, hkv, d = config.n_heads * config.head_dim, config.n_kv_heads * config.head_dim, config.head_dim

        def w(*shape):
            return (torch.randn(shape, generator=g, device=self.device, dtype=torch.float32) * std).to(dt)

        self.embedding = w(config.vocab_size, config.hidden_size)  # tied with the output
        self.layers = []
        for _ in range(config.n_layers):
            self.layers.append({
                "qkv": w(hq + 2 * hkv, config.hidden_size),
                "o": w(config.hidden_size, hq),
                "gate_up": w(2 * config.hidden_dim, config.hidden_size),
                "down": w(config.hidden_size, config.hidden_dim),
                "input_norm": torch.ones(config.hidden_size, device=self.device),
                "post_norm": torch.ones(config.hidden_size, device=self.device),
                "q_norm": torch.ones(d, device=self.device),
                "k_norm": torch.ones(d, device=self.device),
            })
        self.final_norm = torch.ones(config.hidden_size, device=self.device)
        self.cos, self.sin = _rope_tables(config, self.device)

    @staticmethod
    def _few_rows(tokens: int, dtype: torch.dtype, layer: dict[str, torch.Tensor]) -> bool:
        """Whether this layer's products go to ``ops.block_linear``: few rows, and weights it
        can read."""
        return (tokens <= FEW_ROWS and dtype in (torch.bfloat16, torch.float16) and all(
            w.is_contiguous() and w.dtype == dtype and w.data_ptr() % 16 == 0 and w.shape[0] % 32 == 0
            and w.shape[1] % 64 == 0 for w in (layer["qkv"], layer["o"], layer["gate_up"], layer["down"]))
            and layer["input_norm"].data_ptr() % 16 == 0 and layer["post_norm"].data_ptr() % 16 == 0)

    def _fused_heads(self, logit_indices: torch.Tensor, dtype: torch.dtype) -> bool:
        """Whether the logits come from the fused heads kernel: one pass over the embedding
        (up to 160 rows), in a layout it can read."""
        w = self.embedding
        return (logit_indices.numel() <= 160 and dtype in (torch.bfloat16, torch.float16) and w.dtype == dtype
                and w.shape[1] % 128 == 0 and w.is_contiguous() and w.data_ptr() % 16 == 0
                and self.final_norm.dtype == torch.float32 and self.final_norm.is_contiguous())

    @torch.inference_mode()
    def forward_packed(self, input_ids: torch.Tensor, cache: PackedBatchCache, *,
                       fused_rope: bool = True, attention_events: list | None = None,
                       greedy: bool = False) -> torch.Tensor:
        """Logits of the tick's logit rows (model.py:92-110), or with ``greedy`` their
        argmax token ids (engine.py:470-473). ``attention_events`` collects (start, end)
        CUDA events around each layer's attention step.

        With ``fused_rope`` (this build's sequence) the logits or greedy ids come from the
        fused final-norm / logits / argmax kernels (no logits are written for the ids);
        otherwise the reference's logits are computed and ``argmax`` taken."""
        config = self.config
        if input_ids.shape != (1, sum(cache.counts)):
            raise ValueError(f"input_ids must be [1, {sum(cache.counts)}]: one token per packed row of the tick.")
        hq, hkv, d = config.n_heads * config.head_dim, config.n_kv_heads * config.head_dim, config.head_dim
        eps = config.rms_norm_eps
        x = self.embedding[input_ids]
        tokens = x.shape[1]
        branch = None  # the last branch's output, not yet added to the residual stream
        for index, layer in enumerate(self.layers):
            few = fused_rope and self._few_rows(tokens, x.dtype, layer)
            if few:
                if branch is not None:
                    x, branch = x + branch, None
                qkv = ops.block_linear(x, layer["qkv"], norm_weight=layer["input_norm"], eps=eps)
            elif fused_rope:
                x, h = ops.add_rms_norm(x, branch, layer["input_norm"], eps)
                qkv = h @ layer["qkv"].t()
            else:
                qkv = _rms_norm(x, layer["input_norm"], eps) @ layer["qkv"].t()
            q, k, v = qkv[..., :hq], qkv[..., hq:hq + hkv], qkv[..., hq + hkv:]
            if attention_events is not None:
                start = torch.cuda.Event(enable_timing=True)
                start.record()
            if fused_rope:
                context = cache.attend_projected(index, q, k, v, layer["q_norm"], layer["k_norm"],
                                                 self.cos, self.sin, eps)
            else:
                qh = q.reshape(1, tokens, config.n_heads, d).transpose(1, 2)
                kh = k.reshape(1, tokens, config.n_kv_heads, d).transpose(1, 2)
                vh = v.reshape(1, tokens, config.n_kv_heads, d).transpose(1, 2)
                qh = _apply_rope(_rms_norm(qh, layer["q_norm"], eps), self.cos, self.sin, cache.positions)
                kh = _apply_rope(_rms_norm(kh, layer["k_norm"], eps), self.cos, self.sin, cache.positions)
                context = cache.attend(index, qh, kh, vh)
            if attention_events is not None:
                end = torch.cuda.Event(enable_timing=True)
                end.record()
                attention_events.append((start, end))
            context = context.transpose(1, 2).reshape(1, tokens, -1)
            if few:
                x = ops.block_linear(context, layer["o"], residual=x)
                h = ops.block_linear(x, layer["gate_up"], norm_weight=layer["post_norm"], eps=eps, swiglu=True)
                x = ops.block_linear(h, layer["down"], residual=x)
                continue
            branch = context @ layer["o"].t()
            if fused_rope:
                x, h = ops.add_rms_norm(x, branch, layer["post_norm"], eps)
                branch = ops.swiglu(h @ layer["gate_up"].t()) @ layer["down"].t()
                continue
            x = x + branch
            h = _rms_norm(x, layer["post_norm"], eps)
            gate, up = (h @ layer["gate_up"].t()).chunk(2, dim=-1)
            x = x + (torch.nn.functional.silu(gate) * up) @ layer["down"].t()
        if fused_rope and branch is not None:
            x = x + branch
        cache.advance_packed()
        if greedy and fused_rope:
            return ops.final_norm_logits_argmax(x, cache.logit_indices, self.final_norm, self.embedding,
                                                eps).token_ids
        if fused_rope and self._fused_heads(cache.logit_indices, x.dtype):
            logits = ops.final_norm_logits_argmax(x, cache.logit_indices, self.final_norm, self.embedding, eps,
                                                  return_logits=True).logits
            return logits
        x = x.index_select(1, cache.logit_indices)
        logits = (_rms_norm(x, self.final_norm, eps).to(config.dtype) @ self.embedding.t())[0]
        return logits.argmax(dim=-1) if greedy else logits
