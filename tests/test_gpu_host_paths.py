"""The short host paths of attend and attend_projected: the same launches as the general
ones where they apply, and None where they do not."""

from __future__ import annotations

import pytest
import torch

from helios_amd import ops
from helios_amd.config import Qwen3Config
from helios_amd.paged_cache import KVPagePool, PackedBatchCache, PagedKVCache

pytestmark = pytest.mark.gpu


def test_short_host_paths_give_the_bits_of_the_general_ones(device, monkeypatch):
    """attend and attend_projected hand the projections' own layouts to the library when they
    can; views of other layouts take the general path. Same outputs and pools, bit for bit."""
    config = Qwen3Config(vocab_size=64, context_length=2048, hidden_size=256, n_layers=1, hidden_dim=64,
                         dtype=torch.bfloat16)
    g = torch.Generator(device=device).manual_seed(5)
    counts, lengths = [1, 70, 1], [300, 10, 255]
    rows, hq, hkv, d = sum(counts), config.n_heads, config.n_kv_heads, config.head_dim
    qkv = torch.randn(1, rows, (hq + 2 * hkv) * d, generator=g, device=device).to(torch.bfloat16)
    parts = qkv.split((hq * d, hkv * d, hkv * d), dim=-1)
    norm = 1 + 0.1 * torch.randn(d, generator=g, device=device)
    cos = torch.randn(2048, d, generator=g, device=device)
    sin = torch.randn(2048, d, generator=g, device=device)

    def tick(projected):
        pool = KVPagePool(config, 8, device=device)
        pool.storage.normal_(generator=torch.Generator(device=device).manual_seed(6))
        caches = []
        for n in lengths:
            cache = PagedKVCache(pool, 2048)
            cache.pages.extend(pool.acquire(-(-n // 256)))
            cache.length = n
            caches.append(cache)
        batch = PackedBatchCache(caches)
        batch.prepare_packed(counts)
        if projected:
            out = batch.attend_projected(0, *parts, norm, norm, cos, sin, 1e-6)
        else:
            heads = [p.view(1, rows, -1, d).transpose(1, 2) for p in parts]
            out = batch.attend(0, *heads)
        torch.cuda.synchronize()
        return out.clone(), out.stride(), pool.storage.clone()

    for projected in (False, True):
        taken = []

        def watch(m, owner, name):
            inner = getattr(owner, name)

            def call(*a):
                out = inner(*a)
                taken.append((name, out is not None))
                return out
            m.setattr(owner, name, call)

        with monkeypatch.context() as m:
            watch(m, ops.VarlenAttnPlan, "append_attend")
            watch(m, ops.VarlenAttnPlan, "attend_rows")
            watch(m, ops, "qk_norm_rope_append_packed")
            short = tick(projected)
        assert taken == ([("qk_norm_rope_append_packed", True), ("attend_rows", True)] if projected
                         else [("append_attend", True)])
        with monkeypatch.context() as m:
            m.setattr(ops.VarlenAttnPlan, "append_attend", lambda *a: None)
            m.setattr(ops.VarlenAttnPlan, "attend_rows", lambda *a: None)
            m.setattr(ops, "qk_norm_rope_append_packed", lambda *a: None)
            general = tick(projected)
        assert torch.equal(short[0], general[0]) and short[1] == general[1]
        assert torch.equal(short[2].view(torch.int16), general[2].view(torch.int16))


def test_short_host_paths_decline_what_they_cannot_read(device):
    """Unaligned or strided new rows: None from the short path, the general path's answer
    from attend."""
    config = Qwen3Config(vocab_size=64, context_length=512, hidden_size=256, n_layers=1, hidden_dim=64,
                         dtype=torch.float16)
    pool = KVPagePool(config, 2, device=device)
    batch = PackedBatchCache([PagedKVCache(pool, 512)])
    batch.prepare_packed([5])
    g = torch.Generator(device=device).manual_seed(7)
    hq, hkv, d = config.n_heads, config.n_kv_heads, config.head_dim
    q = torch.randn(1, hq, 5, d, generator=g, device=device).half()
    flat = torch.randn(2 * hkv * 5 * d + 1, generator=g, device=device).half()
    k, v = flat[1:].view(2, 1, hkv, 5, d)  # two bytes past alignment
    plan = batch._attention_plan(5)
    pools = pool.keys[0], pool.values[0]
    assert plan.append_attend(q, k, v, *pools, batch.block_table, batch.write_slots) is None
    assert plan.append_attend(q.float(), k.contiguous(), v.contiguous(), *pools, batch.block_table,
                              batch.write_slots) is None
    out = batch.attend(0, q, k, v)
    want = batch.attend(0, q, k.clone(), v.clone())
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    with pytest.raises(ValueError):
        batch.attend(0, q, k[:, :-1], v[:, :-1])
