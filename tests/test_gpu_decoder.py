"""The packed decoder forward on the paged path: this build's sequence (metadata kernel,
fused norm/RoPE/append) against the reference's sequence on the same weights."""

from __future__ import annotations

import pytest
import torch

from helios_amd.config import Qwen3Config
from helios_amd.decoder import PagedQwen3Decoder
from helios_amd.paged_cache import KVPagePool, PackedBatchCache, PagedKVCache
from tests.gpu_cases import say

pytestmark = pytest.mark.gpu


def test_packed_forward_matches_reference_sequence(device):
    say("decoder packed forward")
    config = Qwen3Config(vocab_size=1000, context_length=4096, hidden_size=256, n_layers=2,
                         hidden_dim=512, dtype=torch.bfloat16)
    model = PagedQwen3Decoder(config, device, seed=1, std=0.05)
    lengths, counts = [300, 0, 511], [1, 200, 1]
    logits, pools = [], []
    for device_meta, fused in ((True, True), (False, False)):
        pool = KVPagePool(config, 16, device=device)
        g = torch.Generator(device=device).manual_seed(4)
        for t in pool.keys + pool.values:
            t.normal_(generator=g)
        caches = []
        for n in lengths:
            cache = PagedKVCache(pool, config.context_length)
            if n:
                cache.pages.extend(pool.acquire(-(-n // 256)))
                cache.length = n
            caches.append(cache)
        batch = PackedBatchCache(caches, device_metadata=device_meta)
        ids = torch.randint(0, config.vocab_size, (1, sum(counts)),
                            generator=torch.Generator(device=device).manual_seed(9), device=device)
        for tick in range(2):  # the second tick attends to keys the first one appended
            batch.prepare_packed(counts if tick == 0 else [1, 1, 1])
            out = model.forward_packed(ids if tick == 0 else ids[:, :3], batch, fused_rope=fused)
        torch.cuda.synchronize()
        logits.append(out.float().cpu())
        pools.append(pool.values[0].float().cpu())  # layer 0: same inputs on both paths
    assert logits[0].shape == (3, config.vocab_size)
    assert torch.isfinite(logits[0]).all()
    scale = logits[1].abs().max().item()
    assert (logits[0] - logits[1]).abs().max().item() <= 2e-2 * max(scale, 1.0)
    assert torch.equal(pools[0], pools[1])  # values are appended bit-exactly by both paths


def test_greedy_heads_match_logits_argmax(device, monkeypatch):
    """The fused heads' ids and logits against the library's logits (final norm, product with
    the embedding) of the same tick."""
    say("decoder greedy heads")
    config = Qwen3Config(vocab_size=1000, context_length=4096, hidden_size=256, n_layers=2,
                         hidden_dim=512, dtype=torch.bfloat16)
    model = PagedQwen3Decoder(config, device, seed=2, std=0.05)
    outs = []
    for greedy, fused in ((False, False), (True, True), (False, True)):
        monkeypatch.undo()
        if not fused:
            monkeypatch.setattr(PagedQwen3Decoder, "_fused_heads", lambda *a: False)
        pool = KVPagePool(config, 8, device=device)
        caches = [PagedKVCache(pool, config.context_length) for _ in range(3)]
        batch = PackedBatchCache(caches)
        counts = [5, 130, 1]
        ids = torch.randint(0, config.vocab_size, (1, sum(counts)),
                            generator=torch.Generator(device=device).manual_seed(3), device=device)
        batch.prepare_packed(counts)
        outs.append(model.forward_packed(ids, batch, greedy=greedy))
    torch.cuda.synchronize()
    logits, picks = outs[0].float().cpu(), outs[1].cpu()
    assert picks.shape == (3,) and picks.dtype == torch.int64
    top = logits.max(dim=-1).values
    chosen = logits.gather(1, picks.unsqueeze(1))[:, 0]
    # the kernel's pick is the argmax up to one bf16 rounding of the logits
    assert ((top - chosen) <= 2 * 2.0 ** -7 * top.abs() + 1e-4).all()
    # The same bf16 products in another order of their fp32 sums: one rounding step apart. An
    # element of the normalised row (of rms 1) may round a step (2^-7 of itself) apart as well.
    fused_logits = outs[2].float().cpu()
    moved = 2.0 ** -7 * 4 * model.embedding.abs().max().item()
    assert ((fused_logits - logits).abs() <= 2 * 2.0 ** -7 * logits.abs() + moved).all()
    assert torch.equal(picks, fused_logits.argmax(dim=-1))


@pytest.mark.parametrize("counts", [[1, 2], [1, 30]])
def test_norm_weights_of_any_layout(device, counts):
    """Norm weights that are slices of a flat buffer (4-byte aligned) and a strided final norm:
    the same values, read by the general steps where the fused ones cannot."""
    say("decoder norm layouts", counts)
    config = Qwen3Config(vocab_size=640, context_length=512, hidden_size=256, n_layers=2, hidden_dim=512,
                         dtype=torch.bfloat16)
    model = PagedQwen3Decoder(config, device, seed=6, std=0.05)
    ids = torch.randint(0, 640, (1, sum(counts)), generator=torch.Generator(device=device).manual_seed(7),
                        device=device)
    logits = []
    for moved in (False, True):
        if moved:
            for layer in model.layers:
                for name in ("input_norm", "post_norm"):
                    layer[name] = torch.cat((layer[name][:1], layer[name]))[1:]
            model.final_norm = model.final_norm.repeat_interleave(2)[::2]
        pool = KVPagePool(config, 4, device=device)
        batch = PackedBatchCache([PagedKVCache(pool, config.context_length) for _ in counts])
        batch.prepare_packed(counts)
        logits.append(model.forward_packed(ids, batch).float())
    torch.cuda.synchronize()
    # products in another order of their sums, two layers: as between the sequences above
    assert (logits[0] - logits[1]).abs().max() <= 2e-2 * max(logits[0].abs().max().item(), 1.0)
