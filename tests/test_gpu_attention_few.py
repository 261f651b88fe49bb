"""Few rows (attn_ring_kernel): both sides of its limit, rows with fewer chunks than the ring and
more pages than one page-table load, every tile count, causal blocks and split items, against fp64 attention
on the same bf16 inputs; and bit for bit the rows of a call large enough for attn_paged_kernel.

Bound: bf16 has 8 significant bits, so a rounding moves a value by at most 2^-8 of it.  P is rounded before
P V and the result once more: 2^-8 * sum(p |v|) + 2^-8 * |out| <= 2.1 * 2^-8 * sum(p |v|) with room for the
fp32 sums (the one-wave kernel reaches 1.65 * 2^-8 on the same inputs)."""

import numpy as np
import pytest
import torch

from yapd_amd.paged import AttnPlan

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def run(dev, rows, bl, H, lens, causal=False, **plan_kw):
    g = torch.Generator(device=dev).manual_seed(rows * 100 + bl + H)
    cols = (max(lens) + 15) // 16 + 1
    table = torch.randperm(rows * cols, generator=g, device=dev).to(torch.int32).view(rows, cols)
    pool = torch.randn(rows * cols, 2, H, 1024, generator=g, device=dev).to(BF)
    q = torch.randn(rows, bl, H, 64, generator=g, device=dev).to(BF) * 2
    out = torch.full_like(q, float("nan"))
    plan = AttnPlan(lens, bl, H, torch.device(dev), **plan_kw)
    plan.run(q, pool, table, out, 0.125, causal=causal)
    for r, n in enumerate(lens):
        pages = table[r, : (n + 15) // 16].long()
        k = pool[pages, 0].view(-1, H, 16, 64).transpose(0, 1).reshape(H, -1, 64)[:, :n].double()
        v = pool[pages, 1].view(-1, H, 64, 16).permute(1, 0, 3, 2).reshape(H, -1, 64)[:, :n].double()
        s = torch.matmul(q[r].double().transpose(0, 1), k.transpose(1, 2).contiguous()) * 0.125
        if causal:
            i = torch.arange(bl, device=dev)[:, None] + n - bl
            s = s.masked_fill(torch.arange(n, device=dev)[None] > i, float("-inf"))
        p = s.softmax(-1)
        ref, mag = torch.matmul(p, v).transpose(0, 1), torch.matmul(p, v.abs()).transpose(0, 1)
        assert ((out[r].double() - ref).abs() <= 2.1 * 2.0 ** -8 * mag + 1e-6).all(), (r, n)
    return plan


@pytest.mark.parametrize("bl", [1, 16, 17, 32, 48, 64])
@pytest.mark.parametrize("rows", [1, 3, 17, 64, 96])  # H = 16: 96 rows are the limit, 64 with bl > 32, 24 with bl > 48
@pytest.mark.parametrize("causal", [False, True])
def test_few_rows(dev, rows, bl, causal):
    lens = [max(bl, n) for n in ([1, 31, 32, 33, 64, 97, 129, 300, 541] * 11)[:rows]]
    run(dev, rows, bl, 16, lens, causal)


@pytest.mark.parametrize("rows", [24, 25, 48, 49])
@pytest.mark.parametrize("split", [False, True])
def test_four_tile_limits(dev, rows, split):
    """Blocks of 64: the ring to 24 rows, to 48 work items above that."""
    plan = run(dev, rows, 64, 16, [(70, 300, 129)[r % 3] for r in range(rows)],
               **(dict(target_items=4 * rows, min_split_keys=64) if split else {}))
    assert (plan.work.shape[0] > 48) == (split or rows > 48)


@pytest.mark.parametrize("H", [4, 8, 32])
def test_head_counts(dev, H):
    run(dev, 5, 32, H, [40, 700, 33, 64, 250])


@pytest.mark.parametrize("causal", [False, True])
def test_split_rows(dev, causal):
    """Rows split over work items, and items past 64 pages."""
    plan = run(dev, 3, 16, 16, [2000, 50, 700], causal, target_items=64, min_split_keys=64)
    assert plan.n_slots > 0
    run(dev, 2, 16, 16, [3001, 1050], causal, min_split_keys=4096)


@pytest.mark.parametrize("bl", [8, 32, 48, 64])
@pytest.mark.parametrize("causal", [False, True])
def test_rows_equal_those_of_a_large_call(dev, bl, causal):
    """97 rows run on attn_paged_kernel, their first 5 alone on the ring."""
    H, lens = 16, [max(bl, n) for n in ([70, 33, 1100, 64, 419] * 20)[:97]]
    g = torch.Generator(device=dev).manual_seed(bl)
    cols = (max(lens) + 15) // 16
    table = torch.randperm(97 * cols, generator=g, device=dev).to(torch.int32).view(97, cols)
    pool = torch.randn(97 * cols, 2, H, 1024, generator=g, device=dev).to(BF)
    q = torch.randn(97, bl, H, 64, generator=g, device=dev).to(BF)
    outs = []
    for n in (97, 5):
        out = torch.full_like(q[:n], float("nan"))
        plan = AttnPlan(lens[:n], bl, H, torch.device(dev), min_split_keys=2048)
        plan.run(q[:n], pool, table[:n], out, 0.125, causal=causal)
        outs.append(out)
    assert torch.equal(outs[0][:5], outs[1])


@pytest.mark.parametrize("rows", [2, 97])  # ring and paged kernel
def test_probabilities_are_summed_in_key_order(dev, rows):
    """A lane adds its 8 probabilities of a chunk from the first key to the last, the chunk's sum then goes onto the
    running one: with scores that are whole numbers (q = 1 in one dimension, exp2 of a whole number exact) the sums
    of every split item follow in fp32, and a sum in another order shows in their last bits."""
    H, bl = 16, 16
    lens = [(300, 211)[r % 2] for r in range(rows)]
    scale = np.float32(0.6931472)  # times log2(e) in fp32: 1
    for _ in range(4):
        if scale * np.float32(1.4426950408889634) == 1:
            break
        scale = np.nextafter(scale, np.float32(1))
    assert scale * np.float32(1.4426950408889634) == 1
    cols = 19
    rng = np.random.default_rng(rows)
    score = rng.integers(-24, 1, (rows, H, cols * 16)).astype(np.float32)
    table = torch.arange(rows * cols, dtype=torch.int32, device=dev).view(rows, cols)
    pool = torch.zeros(rows * cols, 2, H, 1024, dtype=BF, device=dev)
    pool[:, 0].view(rows, cols, H, 16, 64)[..., 0] = torch.from_numpy(score).to(dev).view(rows, H, cols, 16).transpose(1, 2).to(BF)
    q = torch.zeros(rows, bl, H, 64, dtype=BF, device=dev)
    q[..., 0] = 1
    plan = AttnPlan(lens, bl, H, torch.device(dev), target_items=4 * rows, min_split_keys=64)
    plan.run(q, pool, table, torch.empty_like(q), float(scale))
    work, ml = plan.work.cpu().numpy(), plan.part_ml.cpu().numpy()
    assert (work[:, 3] >= 0).sum() >= 2 * rows
    for r, kb, ke, slot in work[work[:, 3] >= 0]:
        m, l = np.full(H, -np.inf, np.float32), np.zeros((H, 4), np.float32)
        for k0 in range(kb, ke, 32):
            s = np.full((H, 32), -np.inf, np.float32)
            n = min(32, lens[r] - k0)
            s[:, :n] = score[r, :, k0:k0 + n]
            mn = np.maximum(m, s.max(1))
            p = np.exp2(s - mn[:, None]).astype(np.float32).reshape(H, 4, 8)
            ps = np.zeros((H, 4), np.float32)
            for i in range(8):
                ps += p[..., i]
            l = l * np.exp2(m - mn)[:, None] + ps
            m = mn
        want = (l[:, 0] + l[:, 1]) + (l[:, 2] + l[:, 3])
        assert want.dtype == np.float32
        assert (ml[slot, :, :, 0] == m).all() and (ml[slot, :, :, 1] == want).all(), (r, kb, ke)


@pytest.mark.parametrize("rows", [2, 97])  # ring and paged kernel
@pytest.mark.parametrize("empty_item", [False, True])
def test_empty_rows(dev, rows, empty_item):
    """Device kv_len 0 in the first and last row, with their planned items or with items of no keys: zeros for
    them, the other rows as without.  The table starts inside a larger buffer, whose other entries are no pages."""
    H, bl, n = 16, 32, 70
    g = torch.Generator(device=dev).manual_seed(rows)
    guard = torch.full((rows + 2, 8), 1 << 30, dtype=torch.int32, device=dev)
    table = guard[1:-1, :5]
    table.copy_(torch.randperm(rows * 5, generator=g, device=dev).view(rows, 5))
    pool = torch.randn(rows * 5, 2, H, 1024, generator=g, device=dev).to(BF)
    q = torch.randn(rows, bl, H, 64, generator=g, device=dev).to(BF)
    outs = []
    for empty in (False, True):
        plan = AttnPlan([n] * rows, bl, H, torch.device(dev))
        assert plan.work.shape[0] == rows
        if empty:
            plan.kv_len[0] = plan.kv_len[-1] = 0
            if empty_item:
                gone = (plan.work[:, 0] == 0) | (plan.work[:, 0] == rows - 1)
                plan.work[:, 2] = torch.where(gone, plan.work[:, 1], plan.work[:, 2])
        out = torch.full_like(q, float("nan"))
        plan.run(q, pool, table, out, 0.125)
        outs.append(out)
    assert not outs[1][0].any() and not outs[1][-1].any()
    assert torch.equal(outs[0][1:-1], outs[1][1:-1])


def test_long_work_list(dev):
    """A caller's own list of 300,000 items, all but one empty and bound for no slot: one row's ring launch would hold
    more threads than a grid can (300,000 x 48 heads x 320 > 2^32), the paged kernel's does not."""
    H, bl, n = 48, 64, 100
    g = torch.Generator(device=dev).manual_seed(1)
    table = torch.randperm(8, generator=g, device=dev).to(torch.int32).view(1, 8)
    pool = torch.randn(8, 2, H, 1024, generator=g, device=dev).to(BF)
    q = torch.randn(1, bl, H, 64, generator=g, device=dev).to(BF)
    outs = []
    for items in (1, 300_000):
        plan = AttnPlan([n], bl, H, torch.device(dev))
        plan.work = torch.cat([plan.work, torch.tensor([[0, 0, 0, 7]], dtype=torch.int32, device=dev).repeat(items - 1, 1)])
        out = torch.full_like(q, float("nan"))
        plan.run(q, pool, table, out, 0.125)
        outs.append(out)
    assert torch.equal(*outs)
