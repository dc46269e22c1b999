"""Timed cases of the paged-KV path: what a serving program calls, at the sizes it calls it.

Six kinds of case, all at Qwen3-4B shape (32 query / 8 KV heads, head_dim 128, pages of
256 tokens) except ``varlen``:

``attend``     one layer of a prepared tick through ``PackedBatchCache.attend``: the new K/V
               rows go into their pages, every packed row attends to its sequence.
``projected``  the same through ``PackedBatchCache.attend_projected`` (q/k norm and RoPE
               fused with the append), with requests that hold a shared prefix.
``varlen``     ``ops.varlen_attn`` on its own, as the reference calls torch's: metadata
               tensors in, no plan kept; head shapes other than Qwen3-4B's.
``heads``      ``ops.final_norm_logits_argmax`` over the tied embedding.
``restore``    ``PagedKVCache.restore_blocks(copy=True)``: cached prefix pages of all 36
               layers copied into a new request.
``tick``       a whole tick of the model: prepare, forward, commit, logits. Eight of its 36
               layers, which all cost the same: a rounding that falls the other way in one
               layer's product travels through all that follow, and after 36 of them it has
               moved the logits by 4 %.

Lengths follow from the case alone; page placement and every value from the seed.
"""

from __future__ import annotations

import math
import random

import torch

from helios_amd import ops
from helios_amd.config import Qwen3Config
from helios_amd.decoder import PagedQwen3Decoder
from helios_amd.paged_cache import KVPagePool, PackedBatchCache, PagedKVCache

PAGE = 256
HQ, HKV, D, HIDDEN, FFN, VOCAB, LAYERS = 32, 8, 128, 2560, 9728, 151936, 36
EPS, ROPE_BASE, CONTEXT = 1e-6, 1_000_000.0, 40960
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
DEVICE = "cuda"


# ------------------------------------------------------------------------- the cases
def listed():
    return [
        # The latency of one request decoding alone, short context (a chat's first tokens).
        dict(name="attend_1_decoder", kind="attend", dtype="bf16", decoders=1, lo=300, hi=300, chunks="", lens=1),
        # A decode tick of a busy server: 64 requests at 512-4096 tokens.
        dict(name="attend_64_decoders", kind="attend", dtype="bf16", decoders=64, lo=512, hi=4096, chunks="", lens=2),
        # Few requests, long documents; fp16 checkpoints are served too.
        dict(name="attend_8_long_fp16", kind="attend", dtype="fp16", decoders=8, lo=32768, hi=32768, chunks="", lens=3),
        # A mixed tick at a token budget of 2048: decoders and two prefill chunks.
        dict(name="attend_mixed", kind="attend", dtype="bf16", decoders=32, lo=1024, hi=4096,
             chunks="1024@0,992@512", lens=4),
        # A long prompt's second chunk: 4096 rows at position 4096.
        dict(name="attend_chunk_4096", kind="attend", dtype="bf16", decoders=0, lo=1, hi=1, chunks="4096@4096", lens=5),
        # Short prompts of odd lengths arriving together.
        dict(name="attend_prompts_fp16", kind="attend", dtype="fp16", decoders=0, lo=1, hi=1,
             chunks="37@0,256@0,300@0,611@0", lens=6),
        # One layer of the full tick: 128 decoders on a 4096-token system prompt, one chunk.
        dict(name="projected_prefix", kind="projected", dtype="bf16", decoders=128, lo=1024, hi=8192,
             chunks="1024@4096", prefix=16, lens=7),
        # Another model's heads (16 query / 4 KV heads, head_dim 64), metadata handed over per call.
        dict(name="varlen_head_dim_64", kind="varlen", dtype="bf16", hq=16, hkv=4, d=64, decoders=24, lo=200, hi=2048,
             chunks="512@0,333@700", lens=8),
        # The logit rows of a 129-request tick, with the logits for the sampled requests.
        dict(name="heads_129", kind="heads", dtype="bf16", rows=129, total=1152),
        # A prefix-cache hit of 16 pages copied for a request that may write into them.
        dict(name="restore_16_pages", kind="restore", dtype="bf16", pages=16),
        # The model with a handful of interactive requests: launches and weights count.
        dict(name="tick_8_decoders", kind="tick", dtype="bf16", layers=8, decoders=8, lo=256, hi=2048, chunks="", prefix=0, lens=9),
        # The model on a full continuous-batching tick.
        dict(name="tick_prefix_and_chunk", kind="tick", dtype="bf16", layers=8, decoders=128, lo=1024, hi=8192,
             chunks="1024@4096", prefix=16, lens=10),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], uniform over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["attend"] * 5 + ["projected", "varlen", "varlen", "heads", "restore", "tick"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    lens = rng.randrange(1 << 20)
    if kind == "attend":
        form = rng.choice(["decode", "mixed", "chunks"])
        decoders = 0 if form == "chunks" else _log(rng, 1, 128 if form == "decode" else 48)
        top = min(32768, 262144 // max(1, decoders))  # at most 262144 keys in all
        hi = _log(rng, 32, top)
        lo = _log(rng, max(1, hi // 8), hi)
        chunks = []
        if form != "decode":
            for _ in range(rng.randint(1, 4)):
                chunks.append("%d@%d" % (_log(rng, 2, 2048), rng.choice([0, 0, _log(rng, 1, 8192)])))
        return dict(kind=kind, dtype=dtype, decoders=decoders, lo=lo, hi=hi, chunks=",".join(chunks), lens=lens)
    if kind == "projected":
        prefix = rng.choice([0, _log(rng, 1, 16)])
        hi = _log(rng, 600, 8192)
        return dict(kind=kind, dtype=dtype, decoders=_log(rng, 1, 128), lo=_log(rng, 300, hi), hi=hi,
                    chunks=rng.choice(["", "%d@%d" % (_log(rng, 2, 1024), prefix * PAGE)]), prefix=prefix, lens=lens)
    if kind == "varlen":
        hq, hkv, d = rng.choice([(16, 4, 64), (12, 4, 96), (48, 8, 128), (16, 1, 256), (64, 2, 64), (8, 8, 128)])
        hi = _log(rng, 64, 4096)
        chunks = ["%d@%d" % (_log(rng, 2, 600), rng.choice([0, _log(rng, 1, 1024)])) for _ in range(rng.randint(0, 3))]
        return dict(kind=kind, dtype=dtype, hq=hq, hkv=hkv, d=d, decoders=_log(rng, 1, 32), lo=_log(rng, 16, hi), hi=hi,
                    chunks=",".join(chunks), lens=lens)
    if kind == "heads":
        rows = _log(rng, 1, 200)
        return dict(kind=kind, dtype=dtype, rows=rows, total=rows + _log(rng, 1, 1024))
    if kind == "restore":
        return dict(kind=kind, dtype=dtype, pages=_log(rng, 1, 24))
    hi = _log(rng, 300, 4096)
    return dict(kind="tick", dtype="bf16", layers=rng.randint(4, 8), decoders=_log(rng, 1, 48), lo=_log(rng, 100, hi),
                hi=hi, chunks=rng.choice(["", "%d@0" % _log(rng, 2, 512)]), prefix=0, lens=lens)


# ---------------------------------------------------------------- lengths and page tables
def _lengths(case):
    """(cached, new) tokens of every sequence of the tick: decoders, then chunks."""
    rng = random.Random(case["lens"])
    cached, new = [], []
    for _ in range(case["decoders"]):
        cached.append(rng.randint(case["lo"], case["hi"]) - 1)
        new.append(1)
    for part in filter(None, case["chunks"].split(",")):
        n, at = part.split("@")
        cached.append(int(at))
        new.append(int(n))
    return cached, new


def _shared(case, cached):
    return min(case.get("prefix", 0), cached // PAGE)


def _page_tables(case, seed):
    """Page ids of every sequence, covering its cached and new tokens, and the pool's size:
    a seeded permutation, the first ``prefix`` of it shared by whoever has cached them."""
    cached, new = _lengths(case)
    need = [-(-(c + n) // PAGE) - _shared(case, c) for c, n in zip(cached, new)]
    total = case.get("prefix", 0) + sum(need)
    order = list(range(total))
    random.Random(seed).shuffle(order)
    at, tables = case.get("prefix", 0), []
    for c, n in zip(cached, need):
        tables.append(order[:_shared(case, c)] + order[at:at + n])
        at += n
    return tables, total


def _unique_keys(case):
    """Cached keys that one pass has to read: every sequence's own, the shared ones once."""
    cached, _ = _lengths(case)
    shared = [_shared(case, c) for c in cached]
    return sum(c - s * PAGE for c, s in zip(cached, shared)) + max(shared, default=0) * PAGE


def _visible(case):
    """Query-key pairs that the causal mask leaves."""
    return sum(n * c + n * (n + 1) // 2 for c, n in zip(*_lengths(case)))


def _randn(shape, dtype, seed, std=1.0):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(0.0, std, generator=g)


def _seed(seed, *what):
    return random.Random("/".join(map(str, (seed, *what)))).getrandbits(62)


def _rope():
    inv = 1.0 / (ROPE_BASE ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    angles = torch.arange(CONTEXT, dtype=torch.float32).unsqueeze(1) * inv.unsqueeze(0)
    angles = torch.cat((angles, angles), dim=1)
    return torch.cos(angles).to(DEVICE), torch.sin(angles).to(DEVICE)


def _norm_weight(n, seed):
    return 1.0 + 0.1 * _randn((n,), torch.float32, seed)


# ------------------------------------------------------------------------------- inputs
def _layer_pool(seed, which, layer, total, hkv, d, dtype):
    return _randn((total, PAGE, hkv, d), dtype, _seed(seed, which, layer))


def _requests(case, seed, layers):
    """A filled pool and one request cache per sequence, its pages where the tables say."""
    dtype = DTYPES[case["dtype"]]
    cached, _ = _lengths(case)
    tables, total = _page_tables(case, seed)
    pool = KVPagePool(Qwen3Config(n_layers=layers, dtype=dtype), total, device=torch.device(DEVICE))
    for layer in range(layers):
        for which, pools in (("k", pool.keys), ("v", pool.values)):
            g = torch.Generator(device=DEVICE).manual_seed(_seed(seed, which, layer))
            pools[layer].normal_(generator=g)
    handles = pool.acquire(total)
    caches = []
    for length, table in zip(cached, tables):
        cache = PagedKVCache(pool, CONTEXT)
        cache.pages.extend(handles[i] for i in table)
        cache.length = length
        caches.append(cache)
    return pool, caches


def _qkv(case, seed, hq=HQ, hkv=HKV, d=D):
    """The tick's projections, one row per packed token, as one product's slices."""
    rows = sum(_lengths(case)[1])
    qkv = _randn((1, rows, (hq + 2 * hkv) * d), DTYPES[case["dtype"]], _seed(seed, "qkv"))
    return qkv[..., :hq * d], qkv[..., hq * d:(hq + hkv) * d], qkv[..., (hq + hkv) * d:]


def prepare(case, seed):
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    state = {"case": case}
    if kind in ("attend", "projected"):
        pool, caches = _requests(case, seed, 1)
        batch = PackedBatchCache(caches)
        batch.prepare_packed(_lengths(case)[1])
        q, k, v = _qkv(case, seed)
        rows = q.shape[1]
        if kind == "attend":
            q = q.view(1, rows, HQ, D).transpose(1, 2).contiguous()
            k = k.view(1, rows, HKV, D).transpose(1, 2)
            v = v.view(1, rows, HKV, D).transpose(1, 2)
        else:
            state["norms"] = (_norm_weight(D, _seed(seed, "qn")), _norm_weight(D, _seed(seed, "kn")))
            state["rope"] = _rope()
        state.update(pool=pool, batch=batch, qkv=(q, k, v))
    elif kind == "varlen":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        cached, new = _lengths(case)
        tables, total = _page_tables(case, seed)
        ends = [c + n for c, n in zip(cached, new)]
        width = max(map(len, tables))
        cu_q, cu_k = [0], [0]
        for n, e in zip(new, ends):
            cu_q.append(cu_q[-1] + n)
            cu_k.append(cu_k[-1] + e)
        q = _qkv(case, seed, hq, hkv, d)[0].reshape(-1, hq, d)

        def ints(values):
            return torch.tensor(values, dtype=torch.int32, device=DEVICE)

        state.update(q=q, k=_layer_pool(seed, "k", 0, total, hkv, d, dtype),
                     v=_layer_pool(seed, "v", 0, total, hkv, d, dtype), cu_q=ints(cu_q), cu_k=ints(cu_k),
                     used=ints(ends), table=ints([t + [0] * (width - len(t)) for t in tables]),
                     max_q=max(new), max_k=max(ends))
    elif kind == "heads":
        x, index, weight, embedding = _heads_inputs(case, seed)
        state.update(x=x, index=index, weight=weight, embedding=embedding)
    elif kind == "restore":
        pages = case["pages"]
        config = Qwen3Config(dtype=dtype)
        pool = KVPagePool(config, 2 * pages + 2, device=torch.device(DEVICE))
        pool.storage.normal_(generator=torch.Generator(device=DEVICE).manual_seed(_seed(seed, "pool")))
        source = PagedKVCache(pool, CONTEXT)
        source.pages.extend(pool.acquire(pages))
        source.length = pages * PAGE
        state.update(pool=pool, source=source, block=source.snapshot_block(0, source.length))
    else:
        pool, caches = _requests(case, seed, case["layers"])
        cached, new = _lengths(case)
        state.update(model=PagedQwen3Decoder(pool.config, DEVICE, seed=seed % (1 << 31)), batch=PackedBatchCache(caches),
                     caches=caches, cached=cached, new=new,
                     ids=torch.randint(0, VOCAB, (1, sum(new)), device=DEVICE,
                                       generator=torch.Generator(device=DEVICE).manual_seed(_seed(seed, "ids"))))
    return state


def _heads_inputs(case, seed):
    dtype = DTYPES[case["dtype"]]
    x = _randn((1, case["total"], HIDDEN), dtype, _seed(seed, "x"), 4.0)
    picked = sorted(random.Random(seed).sample(range(case["total"]), case["rows"]))
    embedding = _randn((VOCAB, HIDDEN), dtype, _seed(seed, "embedding"), 0.02)
    return x, torch.tensor(picked, device=DEVICE), _norm_weight(HIDDEN, _seed(seed, "fn")), embedding


# ------------------------------------------------------------------------------ one pass
def run(state):
    kind = state["case"]["kind"]
    if kind == "attend":
        pool = state["pool"]
        out = state["batch"].attend(0, *state["qkv"])
        return {"out": out, "k": pool.keys[0], "v": pool.values[0]}
    if kind == "projected":
        pool = state["pool"]
        out = state["batch"].attend_projected(0, *state["qkv"], *state["norms"], *state["rope"], EPS)
        return {"out": out, "k": pool.keys[0], "v": pool.values[0]}
    if kind == "varlen":
        return ops.varlen_attn(state["q"], state["k"], state["v"], state["cu_q"], state["cu_k"], state["max_q"],
                               state["max_k"], window_size=(-1, 0), enable_gqa=True, seqused_k=state["used"],
                               block_table=state["table"], num_splits=1)
    if kind == "heads":
        heads = ops.final_norm_logits_argmax(state["x"], state["index"], state["weight"], state["embedding"], EPS,
                                             return_logits=True)
        return {"ids": heads.token_ids, "max": heads.max_logits, "logits": heads.logits}
    if kind == "restore":
        request = PagedKVCache(state["pool"], CONTEXT)
        request.restore_blocks([state["block"]], copy=True)
        request.close()
        return state["pool"].storage
    # The tick's new tokens are taken back afterwards, as a rejected speculation is, so that
    # every pass is the same tick. The pools hold GBs: the new rows show in the logits.
    batch = state["batch"]
    batch.prepare_packed(state["new"])
    logits = state["model"].forward_packed(state["ids"], batch)
    for cache, length in zip(state["caches"], state["cached"]):
        cache.truncate(length)
    return logits


# ------------------------------------------------------------------------ what it needs
def work(case):
    kind, size = case["kind"], 2
    if kind == "heads":
        rows = case["rows"]
        return {"bytes": size * (VOCAB * HIDDEN + rows * HIDDEN + rows * VOCAB), "flops": 2 * rows * VOCAB * HIDDEN}
    if kind == "restore":
        return {"bytes": 2 * case["pages"] * 2 * LAYERS * PAGE * HKV * D * size, "flops": 0}
    hq, hkv, d = case.get("hq", HQ), case.get("hkv", HKV), case.get("d", D)
    rows = sum(_lengths(case)[1])
    keys = _unique_keys(case) + (rows if kind == "varlen" else 0)
    attend = size * (2 * keys * hkv * d + 2 * rows * hq * d)
    if kind != "varlen":
        attend += size * 4 * rows * hkv * d  # new rows read and written
    flops = 4 * hq * d * _visible(case)
    if kind != "tick":
        return {"bytes": attend, "flops": flops}
    per_layer = HIDDEN * (HQ + 2 * HKV) * D + HIDDEN * HQ * D + 3 * HIDDEN * FFN
    sequences = len(_lengths(case)[1])
    cache = size * (2 * keys + 2 * rows) * hkv * d  # K/V read, new rows written
    return {"bytes": case["layers"] * (size * per_layer + cache) + size * (VOCAB * HIDDEN + sequences * VOCAB),
            "flops": case["layers"] * (2 * rows * per_layer + flops) + 2 * sequences * VOCAB * HIDDEN}


def tolerance(case):
    kind, fine = case["kind"], case["dtype"] == "fp16"
    if kind == "restore":
        return "exact"
    if kind == "tick":
        # Products in another order of their sums, rounded to bf16 at the same places, move the
        # logits by 0.013 after six layers and by 0.020 after twelve.
        return {"rel": 0.03}
    if kind == "heads":
        # Logits rounded to the model dtype; a tie of two rounded logits may fall either way.
        return {"rel": 1e-3 if fine else 8e-3, "differ": 0.01}
    return {"rel": 2e-3 if fine else 1e-2}


# --------------------------------------------------------------------- the same in 64 bits
def _attention64(q, k_pool, v_pool, tables, cached, new):
    """q [rows, hq, d] in 64 bits over pools [pages, PAGE, hkv, d] of any type."""
    out = torch.empty_like(q)
    hq, d, hkv = q.shape[1], q.shape[2], k_pool.shape[2]
    g, at = hq // hkv, 0
    for table, c, n in zip(tables, cached, new):
        pages = torch.tensor(table, device=q.device)
        k = k_pool[pages].flatten(0, 1)[:c + n].double()
        v = v_pool[pages].flatten(0, 1)[:c + n].double()
        blocked = None
        if n > 1:
            blocked = (torch.arange(c + n, device=q.device)[None, :] > c + torch.arange(n, device=q.device)[:, None])
            blocked = blocked.repeat_interleave(g, dim=0)
        for h in range(hkv):
            rows = q[at:at + n, h * g:(h + 1) * g].reshape(n * g, d)
            s = rows @ k[:, h].t() / math.sqrt(d)
            if blocked is not None:
                s = s.masked_fill(blocked, -math.inf)
            out[at:at + n, h * g:(h + 1) * g] = (s.softmax(-1) @ v[:, h]).view(n, g, d)
        at += n
    return out


def _slots(tables, cached, new):
    """Flat pool row of every new token."""
    return torch.tensor([t[p // PAGE] * PAGE + p % PAGE for t, c, n in zip(tables, cached, new) for p in range(c, c + n)],
                        device=DEVICE)


def _norm64(x, weight, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * weight.double()


def _rope64(x, cos, sin, positions):
    half = x.shape[-1] // 2
    turned = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
    return x * cos[positions].double().unsqueeze(1) + turned * sin[positions].double().unsqueeze(1)


def exact(case, seed):
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    if kind == "restore":
        return None
    if kind == "heads":
        x, index, weight, embedding = _heads_inputs(case, seed)
        rows = _norm64(x[0][index].double(), weight, EPS)
        logits = torch.cat([rows @ part.double().t() for part in embedding.split(16384)], dim=1)
        return {"ids": None, "max": logits.max(-1).values, "logits": logits}
    cached, new = _lengths(case)
    tables, total = _page_tables(case, seed)
    if kind == "varlen":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        q = _qkv(case, seed, hq, hkv, d)[0].reshape(-1, hq, d).double()
        return _attention64(q, _layer_pool(seed, "k", 0, total, hkv, d, dtype),
                            _layer_pool(seed, "v", 0, total, hkv, d, dtype), tables, cached, new)
    slots = _slots(tables, cached, new)
    positions = torch.tensor([p for c, n in zip(cached, new) for p in range(c, c + n)], device=DEVICE)

    def layer(index, q, k, v):
        """Attention of one layer with the new rows in their places, and its pools."""
        k_pool = _layer_pool(seed, "k", index, total, HKV, D, dtype).double()
        v_pool = _layer_pool(seed, "v", index, total, HKV, D, dtype).double()
        k_pool.view(-1, HKV, D)[slots] = k
        v_pool.view(-1, HKV, D)[slots] = v
        return _attention64(q, k_pool, v_pool, tables, cached, new), k_pool, v_pool

    if kind in ("attend", "projected"):
        q, k, v = (t[0].double() for t in _qkv(case, seed))
        q, k, v = q.view(-1, HQ, D), k.view(-1, HKV, D), v.view(-1, HKV, D)
        if kind == "projected":
            cos, sin = _rope()
            q = _rope64(_norm64(q, _norm_weight(D, _seed(seed, "qn")), EPS), cos, sin, positions)
            k = _rope64(_norm64(k, _norm_weight(D, _seed(seed, "kn")), EPS), cos, sin, positions)
        out, k_pool, v_pool = layer(0, q, k, v)
        return {"out": out.transpose(0, 1).unsqueeze(0), "k": k_pool, "v": v_pool}

    # The model: weights drawn in the order and with the generator of its random init.
    g = torch.Generator(device=DEVICE).manual_seed(seed % (1 << 31))

    def weight(*shape):
        return (torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32) * 0.02).to(dtype).double()

    ids = torch.randint(0, VOCAB, (1, sum(new)), device=DEVICE,
                        generator=torch.Generator(device=DEVICE).manual_seed(_seed(seed, "ids")))[0]
    ones, (cos, sin) = torch.ones(HIDDEN, device=DEVICE), _rope()
    embedding = weight(VOCAB, HIDDEN)
    x = embedding[ids]
    for index in range(case["layers"]):
        qkv_w, o_w = weight((HQ + 2 * HKV) * D, HIDDEN), weight(HIDDEN, HQ * D)
        gate_up_w, down_w = weight(2 * FFN, HIDDEN), weight(HIDDEN, FFN)
        q, k, v = (_norm64(x, ones, EPS) @ qkv_w.t()).split((HQ * D, HKV * D, HKV * D), dim=-1)
        q = _rope64(_norm64(q.reshape(-1, HQ, D), ones[:D], EPS), cos, sin, positions)
        k = _rope64(_norm64(k.reshape(-1, HKV, D), ones[:D], EPS), cos, sin, positions)
        x = x + layer(index, q, k, v.reshape(-1, HKV, D))[0].flatten(1) @ o_w.t()
        gate, up = (_norm64(x, ones, EPS) @ gate_up_w.t()).chunk(2, dim=-1)
        x = x + (torch.nn.functional.silu(gate) * up) @ down_w.t()
    ends = torch.tensor([sum(new[:i + 1]) - 1 for i in range(len(new))], device=DEVICE)
    return _norm64(x[ends], ones, EPS) @ embedding.t()
