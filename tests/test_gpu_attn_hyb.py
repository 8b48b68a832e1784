"""Hybrid paged attention whose wavefronts work on their own, at the edges of its tiles, chunks, head groups, alignments and
block-id windows, against float64 over the decoded rows."""
import numpy as np
import pytest
import torch

import aitherkvcache_amd as akv
from tests.util import batch_of_ranges, kv_like, whole_workgroups

pytestmark = pytest.mark.gpu

# float32 outputs.  Head counts that are no multiple of four a kv head: the rounding of some float32 sums and exponentials, as
# in the vector kernel (measured up to 2e-6).  Groups of four of tq35: float16 levels of values, 2.9e-5 of a level (measured 7e-5).
EXACT, LEVELS = 6e-6, 2e-4


def limit(mode, qh, kvh):
    return LEVELS if mode == "tq35" and qh // kvh % 4 == 0 else EXACT


def make(dev, mode, kvh, blocks, bs, pitch, seed, scale=(1.0, 1.0)):
    rng = np.random.default_rng(seed)
    h = akv.HybridTurboQuant(head_dim=128, mode=mode, device=str(dev))
    h.calibrate_uniform(kvh)
    rows = []
    for i in range(2):
        r = torch.full((blocks, bs, kvh, pitch), 0x5A, dtype=torch.uint8, device=dev)
        x = torch.from_numpy((scale[i] * kv_like(rng, (blocks * bs, kvh, 128))).astype(np.float32)).to(dev)
        akv.hybrid_encode_and_store(h, x, torch.arange(blocks * bs, device=dev), r, bs)
        rows.append(r[..., :h.packed_dim])
    return rng, h, rows


def attend(q, K, V, counts=None):
    """q [heads, d], K and V [tokens, kv heads, d], each token `counts` times; float64."""
    heads, kvh = q.shape[0], K.shape[1]
    out = torch.zeros_like(q)
    for i in range(heads):
        s = K[:, i // (heads // kvh)] @ q[i] / 128 ** 0.5
        p = torch.exp(s - s.max()) * (1.0 if counts is None else counts)
        out[i] = p @ V[:, i // (heads // kvh)] / p.sum()
    return out


@pytest.mark.parametrize("mode,pitch", [("tq35", 64), ("tq35", 68), ("tq25", 44), ("tq25", 64)])
@pytest.mark.parametrize("qh,kvh,bs", [(4, 1, 16), (8, 1, 32), (8, 2, 16), (12, 3, 32), (20, 5, 16), (32, 8, 16), (3, 1, 16), (10, 2, 32), (21, 3, 16),
                                       (7, 7, 32), (18, 2, 16)])
def test_edges_vs_float64(dev, mode, pitch, qh, kvh, bs):
    ctx = np.array([1, 0, 15, 16, 17, 31, 32, 33, 64, 65, 257, 1000, 0, 3], dtype=np.int32)
    need = -(-ctx // bs)
    blocks = int(need.sum()) + 2
    rng, h, rows = make(dev, mode, kvh, blocks, bs, pitch, qh + bs)
    tables = np.full((len(ctx), int(need.max())), 10 ** 6, dtype=np.int32)
    order, at = rng.permutation(blocks), 0
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n]
        at += int(n)
    K, V = (h.decode(r.contiguous()).double().cpu() for r in rows)
    for i, n in enumerate(ctx):                        # rows that no context covers may hold anything: here float16 NaN factors
        if n % bs:
            for r in rows:
                r[int(tables[i, need[i] - 1]), int(n) % bs:] = 0xFF
    q = torch.from_numpy(rng.standard_normal((len(ctx), qh, 128)).astype(np.float32)).to(dev)
    print(f"[attn hyb] {mode} pitch={pitch} qh={qh} kvh={kvh} bs={bs}", flush=True)
    out = akv.HybridPagedAttention(h, qh).forward(q, rows[0], rows[1], torch.from_numpy(tables).to(dev), torch.from_numpy(ctx).to(dev),
                                                  block_size=bs).double().cpu()
    for i, n in enumerate(ctx):
        if n == 0:
            assert not out[i].any()
            continue
        t = torch.from_numpy(tables[i, :need[i]].astype(np.int64))
        k, v = (x[t].reshape(-1, kvh, 128)[:n] for x in (K, V))
        ref = attend(q[i].double().cpu(), k, v)
        assert (out[i] - ref).norm() <= limit(mode, qh, kvh) * ref.norm(), (i, n, float((out[i] - ref).norm() / ref.norm()))


@pytest.mark.parametrize("mode", ["tq35", "tq25"])
@pytest.mark.parametrize("qh,kvh,bs,chunks", [(16, 16, 16, 70), (48, 12, 32, 33), (4, 1, 16, 32)])
def test_more_chunks_than_a_window_of_block_ids(dev, mode, qh, kvh, bs, chunks):
    """A context so long that a wavefront goes through several windows of block ids, of 32 chunks each; its blocks repeat a few,
    which the reference counts."""
    rng, h, rows = make(dev, mode, kvh, 8, bs, h_pitch(mode), 7)
    groups = kvh * (-(-(qh // kvh) // 4))
    ranges, shares = (512, 4) if groups == 1 else (min(512, 768 // (-(-groups // 4))), 1)
    n = 32 * chunks * ranges * shares - 5
    table = rng.integers(0, 8, size=-(-n // bs)).astype(np.int32)
    q = torch.from_numpy(rng.standard_normal((1, qh, 128)).astype(np.float32)).to(dev)
    out = akv.HybridPagedAttention(h, qh).forward(q, rows[0], rows[1], torch.from_numpy(table[None]).to(dev),
                                                  torch.tensor([n], dtype=torch.int32, device=dev), block_size=bs).double().cpu()
    counts = np.zeros((8, bs))
    np.add.at(counts, table[:-1], 1.0)
    counts[table[-1], :n - (len(table) - 1) * bs] += 1.0
    K, V = (h.decode(r.contiguous()).double().cpu().reshape(-1, kvh, 128) for r in rows)
    ref = attend(q[0].double().cpu(), K, V, torch.from_numpy(counts.reshape(-1)))
    # sums of 2^17 and more float32 terms: their rounding walks to a few times that of short contexts
    assert (out[0] - ref).norm() <= max(limit(mode, qh, kvh), 4 * EXACT) * ref.norm(), float((out[0] - ref).norm() / ref.norm())


def h_pitch(mode):
    return 64 if mode == "tq35" else 44


@pytest.mark.parametrize("mode", ["tq35", "tq25"])
@pytest.mark.parametrize("qh,kvh", [(8, 2), (6, 2)])
@pytest.mark.parametrize("scale_k,scale_v,scale_q", [(1.0, 3e2, 1.0), (1.0, 1e-3, 1.0), (1e-2, 1.0, 1e2), (1e2, 1.0, 1e-30), (1e-2, 1.0, 1e4)])
def test_factors_and_queries_far_from_one(dev, mode, qh, kvh, scale_k, scale_v, scale_q):
    """Value factors near both ends of float16, queries far outside it, scores of hundreds (one token takes all)."""
    rng, h, rows = make(dev, mode, kvh, 8, 16, h_pitch(mode), 3, (scale_k, scale_v))
    n = 100
    q = torch.from_numpy((scale_q * rng.standard_normal((1, qh, 128))).astype(np.float32)).to(dev)
    out = akv.HybridPagedAttention(h, qh).forward(q, rows[0], rows[1], torch.arange(8, dtype=torch.int32, device=dev)[None],
                                                  torch.tensor([n], dtype=torch.int32, device=dev)).double().cpu()
    K, V = (h.decode(r.contiguous()).double().cpu().reshape(-1, kvh, 128)[:n] for r in rows)
    ref = attend(q[0].double().cpu(), K, V)
    # scores of some hundreds carry 2^-22 of themselves into their exponentials
    assert (out[0] - ref).norm() <= max(limit(mode, qh, kvh), 5e-4 if scale_q == 1e4 else 0.0) * ref.norm(), float((out[0] - ref).norm() / ref.norm())


def test_queries_that_are_no_numbers_stay_in_their_head(dev):
    rng, h, rows = make(dev, "tq35", 2, 8, 16, 64, 5)
    q = torch.from_numpy(rng.standard_normal((1, 8, 128)).astype(np.float32)).to(dev)
    args = (rows[0], rows[1], torch.arange(8, dtype=torch.int32, device=dev)[None], torch.tensor([90], dtype=torch.int32, device=dev))
    good = akv.HybridPagedAttention(h, 8).forward(q, *args)
    q[0, 1, 5], q[0, 6, 127] = float("nan"), float("inf")
    bad = akv.HybridPagedAttention(h, 8).forward(q, *args)
    for i in range(8):
        assert bool(torch.isnan(bad[0, i]).all()) if i in (1, 6) else torch.equal(bad[0, i], good[0, i])


@pytest.mark.parametrize("qh,kvh", [(8, 2), (3, 1)])
def test_one_bit_levels_that_are_not_symmetric(dev, qh, kvh):
    """tq25 with two levels around something other than zero: their middle weighs with the sum of all weights."""
    rng, h, rows = make(dev, "tq25", kvh, 8, 16, 44, 9)
    h.kernel_table[260:262] = torch.tensor([-0.05, 0.12], device=dev)
    q = torch.from_numpy(rng.standard_normal((1, qh, 128)).astype(np.float32)).to(dev)
    out = akv.HybridPagedAttention(h, qh).forward(q, rows[0], rows[1], torch.arange(8, dtype=torch.int32, device=dev)[None],
                                                  torch.tensor([120], dtype=torch.int32, device=dev)).double().cpu()
    K, V = (h.decode(r.contiguous()).double().cpu().reshape(-1, kvh, 128)[:120] for r in rows)
    ref = attend(q[0].double().cpu(), K, V)
    assert (out[0] - ref).norm() <= EXACT * ref.norm()


@pytest.mark.parametrize("qh,kvh", [(8, 2), (8, 1), (6, 2)])
def test_key_levels_have_more_than_sixteen_bits(dev, qh, kvh):
    """tq35 with levels that one float16 holds, so that values are exact, seven of them far below the eighth: as multiples of 2^-15
    of the largest they were off by up to 1e-4 of themselves, and outputs by 1.5e-5."""
    rng, h, rows = make(dev, "tq35", kvh, 8, 16, 64, 11)
    levels = [-0.25, -0.151, -0.0717, -0.0213, 0.0127, 0.0611, 0.1423, 4.2, -1.41, -0.4527, 0.4318, 1.623]
    h.kernel_table[256:268] = (0.1 * torch.tensor(levels, device=dev)).half().float()
    q = torch.from_numpy((2 * rng.standard_normal((1, qh, 128))).astype(np.float32)).to(dev)
    out = akv.HybridPagedAttention(h, qh).forward(q, rows[0], rows[1], torch.arange(8, dtype=torch.int32, device=dev)[None],
                                                  torch.tensor([128], dtype=torch.int32, device=dev)).double().cpu()
    K, V = (h.decode(r.contiguous()).double().cpu().reshape(-1, kvh, 128) for r in rows)
    ref = attend(q[0].double().cpu(), K, V)
    print(f"[key levels] {qh} on {kvh}: {float((out[0] - ref).norm() / ref.norm()):.2e}", flush=True)
    assert (out[0] - ref).norm() <= EXACT * ref.norm(), float((out[0] - ref).norm() / ref.norm())


def test_one_workspace_for_both_groupings(dev):
    """Groups of four query heads and other groups keep different value levels in a workspace: whichever used it last, the next
    call's are its own."""
    q = torch.from_numpy(np.random.default_rng(1).standard_normal((1, 8, 128)).astype(np.float32)).to(dev)
    tables, lens = torch.arange(8, dtype=torch.int32, device=dev)[None], torch.tensor([100], dtype=torch.int32, device=dev)
    made = {kvh: make(dev, "tq35", kvh, 8, 16, 64, 13) for kvh in (2, 8)}
    h = made[2][1]
    shared = akv.HybridPagedAttention(h, 8)
    for kvh in (2, 8, 2, 2, 8, 8):
        rows = made[kvh][2]
        assert torch.equal(shared.forward(q, *rows, tables, lens), akv.HybridPagedAttention(h, 8).forward(q, *rows, tables, lens)), kvh


@pytest.mark.parametrize("qh,kvh", [(8, 2), (6, 2)])
def test_a_new_workspace_costs_little(dev, qh, kvh):
    """The tables that a call builds in a new workspace: some 30 us and none; 650 were spent.  A later call takes 20."""
    rng, h, rows = make(dev, "tq35", kvh, 8, 16, 64, 17)
    q = torch.from_numpy(rng.standard_normal((1, qh, 128)).astype(np.float32)).to(dev)
    args = (q, *rows, torch.arange(8, dtype=torch.int32, device=dev)[None], torch.tensor([100], dtype=torch.int32, device=dev))
    att = akv.HybridPagedAttention(h, qh)
    att.forward(*args)

    def least(new):
        times = []
        for _ in range(15):
            if new:
                att._workspace.fill_(0xFF)
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            a.record()
            att.forward(*args)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return min(times)

    later, first = least(False), least(True)
    print(f"[new workspace] {qh} on {kvh}: {first:.1f} us, later {later:.1f} us", flush=True)
    assert first < later + 120


@pytest.mark.parametrize("mode,qh,kvh", [("tq35", 32, 8), ("tq25", 12, 2)])
def test_many_sequences_and_empty_ones_vs_float64(dev, mode, qh, kvh):
    """Runs of empty sequences longer than a wavefront's lanes, one sequence in most of the workgroups, many that share one."""
    rng, h, rows = make(dev, mode, kvh, 40, 16, 64 if mode == "tq35" else 44, qh)
    ctx = np.concatenate([np.zeros(100), [30000], np.zeros(130), rng.integers(1, 130, size=150), np.zeros(70), rng.integers(1, 40, size=5)]).astype(np.int32)
    tables = rng.integers(0, 40, size=(len(ctx), 30000 // 16)).astype(np.int32)
    K, V = (h.decode(r.contiguous()).double().cpu() for r in rows)
    q = torch.from_numpy(rng.standard_normal((len(ctx), qh, 128)).astype(np.float32)).to(dev)
    out = akv.HybridPagedAttention(h, qh).forward(q, rows[0], rows[1], torch.from_numpy(tables).to(dev), torch.from_numpy(ctx).to(dev)).double().cpu()
    assert not out[torch.from_numpy(ctx == 0)].any()
    for i in np.flatnonzero(ctx):
        t = torch.from_numpy(tables[i, :-(-int(ctx[i]) // 16)].astype(np.int64))
        k, v = (x[t].reshape(-1, kvh, 128)[:ctx[i]] for x in (K, V))
        ref = attend(q[i].double().cpu(), k, v)
        assert (out[i] - ref).norm() <= limit(mode, qh, kvh) * ref.norm(), (i, ctx[i])


@pytest.mark.parametrize("mode,qh,kvh,per_cu,kind", [
    # two groups of four kv head slots: three workgroups a compute unit
    ("tq35", 32, 8, 1.5, "whole, one long"), ("tq35", 32, 8, 1.5, "whole, half"), ("tq35", 32, 8, 1.5, "equal, one long"), ("tq35", 32, 8, 1.5, "equal, most"),
    ("tq35", 32, 8, 1.5, "equal, few (55)"),
    # four of them, and a kernel of which two workgroups fit a compute unit: longer ranges do not pay
    ("tq35", 40, 8, 0.75, "equal, ragged"), ("tq35", 40, 8, 0.75, "whole, short"),
    # one, in pairs of wavefronts
    ("tq25", 12, 2, 2, "whole, one long"), ("tq25", 12, 2, 2, "whole, half"), ("tq25", 12, 2, 2, "equal, most")])
def test_ranges_of_workgroups_vs_float64(dev, mode, qh, kvh, per_cu, kind):
    rng, h, rows = make(dev, mode, kvh, 40, 16, 64 if mode == "tq35" else 44, qh)
    ctx, look = batch_of_ranges(rng, kind)
    tables = rng.integers(0, 40, size=(len(ctx), int(ctx.max() + 15) // 16)).astype(np.int32)
    K, V = (h.decode(r.contiguous()).double().cpu() for r in rows)
    q = torch.from_numpy(rng.standard_normal((len(ctx), qh, 128)).astype(np.float32)).to(dev)
    attn = akv.HybridPagedAttention(h, qh)
    out = attn.forward(q, rows[0], rows[1], torch.from_numpy(tables).to(dev), torch.from_numpy(ctx).to(dev)).double().cpu()
    assert whole_workgroups(attn, int(per_cu * torch.cuda.get_device_properties(dev).multi_processor_count), ctx) == kind.startswith("whole")
    assert not out[torch.from_numpy(ctx == 0)].any()
    for i in look:
        t = torch.from_numpy(tables[i, :-(-int(ctx[i]) // 16)].astype(np.int64))
        k, v = (x[t].reshape(-1, kvh, 128)[:ctx[i]] for x in (K, V))
        ref = attend(q[i].double().cpu(), k, v)
        assert (out[i] - ref).norm() <= limit(mode, qh, kvh) * ref.norm(), (i, ctx[i])
