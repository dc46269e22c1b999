"""The any-head_dim attention kernel at the edges of its splits: units per block (64 (row,
head) pairs, 16 per decode item), 64-key tiles, 256-key decode splits, padded head dims,
and the form without work lists, against the float64 oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helios_amd import ops, synth
from tests.gpu_cases import DeviceTick, compare, say

pytestmark = pytest.mark.gpu


def _tick(q_lens, k_lens, hq, hkv, d, dtype, device, seed):
    free = [int(x) for x in synth.permutation(seed, sum(-(-k // 256) for k in k_lens) + 2)]
    tables = synth._assign_pages(k_lens, free, 256)
    w = synth.Workload(f"wide{seed}", list(q_lens), [k - n for n, k in zip(q_lens, k_lens)], tables, len(free),
                       n_q_heads=hq, n_kv_heads=hkv, head_dim=d, seed=seed)
    return DeviceTick(w, dtype, device)


# One-token rows around the tile and split edges, then chunks around the unit-block edges.
Q_LENS = [1, 1, 1, 1, 1, 1, 1, 2, 3, 16, 17, 22, 65]
K_LENS = [1, 64, 65, 256, 257, 513, 1090, 2, 70, 16, 300, 257, 641]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(3, 3, 8), (4, 2, 24), (8, 2, 64), (6, 2, 72), (17, 1, 96), (6, 1, 128),
                                      (70, 1, 32), (32, 1, 136), (4, 1, 256)])
def test_wide_edges(device, hq, hkv, d, dtype):
    say("wide edges", hq, hkv, d, dtype)
    tick = _tick(Q_LENS, K_LENS, hq, hkv, d, dtype, device, 300 + d)
    for window in ((-1, 0), (100, 5)):
        ref, ref_lse = tick.oracle(window=window)
        out, lse = tick.attend(window=window, exact_grid=True, return_lse=True)
        compare(out, ref, what=f"wide {hq}/{hkv} d={d} {window}")
        # fp32 sums of at most 1090 terms, against float64
        assert np.abs(lse.cpu().numpy() - ref_lse).max() < 1e-4


def test_wide_constant_values(device):
    """Constant V: the weights of a row sum to one, so each output rounds to that value."""
    tick = _tick([1, 40], [1500, 700], 8, 2, 64, torch.bfloat16, device, 41)
    tick.v_pool.fill_(1.0)
    tick.v_pool[..., ::2] = 0.75
    out = tick.attend()
    torch.cuda.synchronize()
    assert (out[..., 1::2] == 1.0).all() and (out[..., ::2] == 0.75).all()


@pytest.mark.parametrize("rows", [1, 20])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_keeps_p_in_fp32(device, dtype, rows):
    """A hundred keys of weight p1 with V = 1 against a hundred of p2 with V = -1 and one key
    of weight 1 with V = 0. Scores come from one dim, so they are exact; p1 - p2 is at least
    2.4e-4. In fp32 the two exps (2^-23 each) move the output by 1e-3 of itself, and so do 400
    roundings of sums up to 1 (2^-24 each, of a sum of 0.024); the rounding of the output adds
    half a step. Emulated errors with P in one, two and three operands: bf16 3.4, 5.7e-3 and
    1.8e-3; fp16 1.0, 4.4e-4 and 4.4e-4."""
    say("wide p", dtype, rows)
    hq, n, d = 16, 100, 64
    a = torch.linspace(0.5, 3.5, hq).to(dtype)
    q = torch.zeros(rows, hq, d, dtype=dtype, device=device)
    q[:, :, 0] = a.to(device)
    # masked keys fill up to a causal chunk: every row sees the first 2 n + 1
    k = torch.zeros(2 * n + 1 + rows - 1, 1, d, dtype=dtype, device=device)
    v = torch.zeros_like(k)
    k[1:2 * n + 1:2, :, 0], k[2:2 * n + 1:2, :, 0] = -0.5 - 2.0 ** -8, -0.5
    v[1:2 * n + 1:2], v[2:2 * n + 1:2] = 1.0, -1.0
    k[2 * n + 1:, :, 0] = -448.0  # of no weight
    cu_q = torch.tensor([0, rows], dtype=torch.int32, device=device)
    cu_k = torch.tensor([0, k.shape[0]], dtype=torch.int32, device=device)
    out = ops.varlen_attn(q, k, v, cu_q, cu_k, rows, k.shape[0], is_causal=True, enable_gqa=True).double().cpu()
    p1, p2 = (torch.exp(a.double() * b / 8) for b in (-0.5 - 2.0 ** -8, -0.5))
    want = (n * (p1 - p2) / (1 + n * (p1 + p2))).view(1, hq, 1)
    off = (out / want - 1).abs().max().item()
    say("relative error", off)
    assert off <= 2e-3 + (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -11)


@pytest.mark.parametrize("hq,hkv,d", [(4, 1, 256), (8, 1, 136)])
def test_wide_without_work_lists(device, hq, hkv, d, monkeypatch):
    """A workspace of the 16-bit partials' size (the least accepted) holds no fp32 partials at
    these head dims and chunks of a few rows: the same results from whole rows."""
    say("wide plain", hq, hkv, d)
    tick = _tick([min(n, 3) for n in Q_LENS], K_LENS, hq, hkv, d, torch.bfloat16, device, 500 + d)
    ref, ref_lse = tick.oracle()
    sized = ops.workspace_bytes
    least = sized(tick.w.batch, tick.w.max_q, tick.w.max_k, hq, hkv, 8)
    assert least < sized(tick.w.batch, tick.w.max_q, tick.w.max_k, hq, hkv, d)
    monkeypatch.setattr(ops, "workspace_bytes", lambda *a: least)
    out, lse = tick.attend(exact_grid=True, return_lse=True)
    compare(out, ref, what=f"wide plain {hq}/{hkv} d={d}")
    assert np.abs(lse.cpu().numpy() - ref_lse).max() < 1e-4
    # a plan with lists, run with the smaller size: whole rows again
    monkeypatch.setattr(ops, "workspace_bytes", sized)
    plan = tick.plan()
    plan.ws_bytes = least
    again = plan.run(tick.q, tick.k_pool, tick.v_pool, tick.block_table)
    assert plan.error_word() == 0 and torch.equal(again.view(torch.int16), out.view(torch.int16))
    monkeypatch.setattr(ops, "workspace_bytes", lambda *a: least - 256)
    with pytest.raises(ValueError):
        tick.plan()


def test_wide_expanded_packed_keys(device):
    """Packed keys whose row stride is 0 (one key broadcast over the sequence)."""
    say("wide stride 0")
    g = torch.Generator(device=device).manual_seed(3)
    q = torch.randn(5, 6, 64, generator=g, device=device).to(torch.bfloat16)
    k = torch.randn(1, 2, 64, generator=g, device=device).to(torch.bfloat16).expand(90, 2, 64)
    v = torch.randn(1, 2, 64, generator=g, device=device).to(torch.bfloat16).expand(90, 2, 64)
    cu_q = torch.tensor([0, 1, 5], dtype=torch.int32, device=device)
    cu_k = torch.tensor([0, 20, 90], dtype=torch.int32, device=device)
    out = ops.varlen_attn(q, k, v, cu_q, cu_k, 4, 70, is_causal=True, enable_gqa=True)
    torch.cuda.synchronize()
    want = v[0].repeat_interleave(3, dim=0).expand(5, 6, 64)
    # equal weights of one row: the row itself, up to the rounding of fp32 sums
    assert torch.equal(out, want)


def _plant(tick, seed):
    """Infinities and NaNs for V: {sequence: {(key, kv head, dim): value}}."""
    rng = np.random.default_rng(seed)
    w, planted = tick.w, {}
    hkv, d = w.n_kv_heads, w.head_dim
    for b in (2, 6, len(w.k_lens) - 1):  # decode rows of one and of five splits, the last chunk
        L, at = w.k_lens[b], {}
        for g in range(hkv):
            at[(int(rng.integers(0, L)), g, 0)] = np.inf
            at[(L - 1, g, 1)] = -np.inf
            at[(int(rng.integers(0, L)), g, 2)] = np.inf
            at[(L - 2, g, 2)] = np.inf
            at[(0, g, 3)] = np.inf
            at[(L // 2, g, 3)] = -np.inf
            at[(L // 3, g, 4)] = np.nan
            at[(L - 1, g, d - 1)] = np.inf
        planted[b] = at
    return planted


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(16, 4, 64), (3, 1, 8), (6, 2, 72), (34, 2, 96), (6, 1, 128), (4, 1, 256)])
def test_infinite_and_nan_values(device, hq, hkv, d, dtype):
    """An infinite element of V gives +-inf to the rows that see its key, NaN where both signs
    or a NaN are seen, and nothing to the others, whose results stay what they were; a NaN in K
    makes the rows that see it NaN. Key 0 is drawn to the queries, so that p is 1 there in many
    rows, exact in either type; the last keys are masked for the chunk's earlier rows."""
    say("wide inf", hq, hkv, d, dtype)
    tick = _tick(Q_LENS, K_LENS, hq, hkv, d, dtype, device, 700 + d)
    w = tick.w
    k_flat, v_flat = tick.k_pool.view(-1, hkv, d), tick.v_pool.view(-1, hkv, d)
    at = lambda b, key: w.tables[b][key // 256] * 256 + key % 256  # noqa: E731
    for b in range(w.batch):
        rows = tick.q[w.cu_seq_q[b]:w.cu_seq_q[b + 1]].float().view(-1, hkv, hq // hkv, d).mean((0, 2))
        k_flat[at(b, 0)] = (rows / rows.norm(dim=-1, keepdim=True) * 4 * d ** 0.5).to(dtype)
    for window in ((-1, 0), (100, 5)):
        before, lse0 = tick.attend(window=window, exact_grid=True, return_lse=True)
        planted = _plant(tick, d)
        keep = v_flat.clone()
        for b, elements in planted.items():
            for (key, g, dim), value in elements.items():
                v_flat[at(b, key), g, dim] = value
        k_keep, nan_keys = k_flat.clone(), {4: 0, 5: 512, 11: 256}
        for b, key in nan_keys.items():
            k_flat[at(b, key), hkv - 1, 0] = np.nan
        out, lse = tick.attend(window=window, exact_grid=True, return_lse=True)
        want = before.double().cpu().numpy()
        touched = np.zeros(want.shape, bool)
        for b, elements in planted.items():
            n, L = w.q_lens[b], w.k_lens[b]
            for i in range(n):
                pos = L - n + i
                lo = 0 if window[0] < 0 else max(0, pos - window[0])
                hi = min(L - 1, pos + window[1])
                for (key, g, dim), value in elements.items():
                    if lo <= key <= hi:
                        heads = slice(g * (hq // hkv), (g + 1) * (hq // hkv))
                        row = w.cu_seq_q[b] + i
                        with np.errstate(invalid="ignore"):
                            want[row, heads, dim] = value if not touched[row, heads.start, dim] else \
                                want[row, heads, dim] + value
                        touched[row, heads, dim] = True
        for b, key in nan_keys.items():
            for i in range(w.q_lens[b]):
                pos = w.k_lens[b] - w.q_lens[b] + i
                if (0 if window[0] < 0 else pos - window[0]) <= key <= pos + window[1]:
                    want[w.cu_seq_q[b] + i, hq - hq // hkv:] = np.nan
                    touched[w.cu_seq_q[b] + i, hq - hq // hkv:] = True
        got = out.double().cpu().numpy()
        assert touched.any() and not np.isfinite(want[touched]).any()
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        np.testing.assert_array_equal(got[touched & ~np.isnan(want)], want[touched & ~np.isnan(want)])
        # the rest: fp32 sums in another order, one rounding step apart at most
        rest, ulp = ~touched, 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
        assert (np.abs(got[rest] - want[rest]) <= ulp * np.abs(want[rest]) + 1e-6).all()
        same = ~touched.all(axis=-1).T  # the log-sum-exp of a NaN row is not specified
        assert np.abs(lse.cpu().numpy() - lse0.cpu().numpy())[same].max() < 1e-4
        v_flat.copy_(keep)
        k_flat.copy_(k_keep)


def test_workspace_without_room_for_fp32_partials(device, monkeypatch):
    """A plan whose full workspace cannot be allocated takes the smaller one and runs whole
    rows; a tuned shape, which has no smaller one, raises."""
    say("wide workspace fallback")
    tick = _tick([min(n, 3) for n in Q_LENS], K_LENS, 4, 1, 256, torch.bfloat16, device, 900)
    tuned = _tick([1, 5], [300, 40], 8, 2, 128, torch.bfloat16, device, 901)
    ref, _ = tick.oracle()
    full = {ops.workspace_bytes(t.w.batch, t.w.max_q, t.w.max_k, t.w.n_q_heads, t.w.n_kv_heads, t.w.head_dim) + 256
            for t in (tick, tuned)}
    empty = torch.empty

    def no_room(*args, **kwargs):
        if args and args[0] in full:
            raise torch.OutOfMemoryError("no room")
        return empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", no_room)
    compare(tick.attend(exact_grid=True), ref, what="wide workspace fallback")
    with pytest.raises(torch.OutOfMemoryError):
        tuned.plan()


def test_wide_items_of_more_than_64_pages(device, monkeypatch):
    """A workgroup holds 64 page ids at a time: items of 16384 keys and around it, and of 33000
    (three fetches), on shuffled pages. Whole decode rows and a chunk without work lists, and
    a chunk of so many blocks that none is split."""
    say("wide many pages, whole rows")
    tick = _tick([1, 1, 1, 1, 3], [16384, 16385, 16640, 33000, 32769], 1, 1, 136, torch.bfloat16, device, 950)
    sized = ops.workspace_bytes
    least = sized(tick.w.batch, tick.w.max_q, tick.w.max_k, 1, 1, 8)
    assert least < sized(tick.w.batch, tick.w.max_q, tick.w.max_k, 1, 1, 136)
    ref, ref_lse = tick.oracle()
    with monkeypatch.context() as m:
        m.setattr(ops, "workspace_bytes", lambda *a: least)
        out, lse = tick.attend(exact_grid=True, return_lse=True)
    compare(out, ref, what="wide many pages, whole rows")
    assert np.abs(lse.cpu().numpy() - ref_lse).max() < 1e-4

    say("wide many pages, unsplit chunk")
    # 64 heads on one: a block a row, so 520 rows are 520 items, and 512 are not split
    tick = _tick([520, 1], [17000, 16641], 64, 1, 8, torch.bfloat16, device, 951)
    rows = {0: [0, 1, 255, 518, 519], 1: [0]}
    ref, _ = tick.oracle(rows=rows)
    out = tick.attend(exact_grid=True)
    compare(out, ref, what="wide many pages, unsplit chunk", rows=np.array(rows[0] + [520]))
