"""Paged attention kernel whose wavefronts work on their own (head_dim 64 and 256; head_dim 128 with one kv head, or two and few sequences),
at the edges of its tiles, chunks, head slots and block-id windows, against float64."""
import numpy as np
import pytest
import torch

import aitherkvcache_amd as akv
from oracle import tq_oracle as O
from tests.util import batch_of_ranges, kv_like, whole_workgroups

pytestmark = pytest.mark.gpu

# float32 outputs: the rounding of a few float32 sums and exponentials, 2 ** -23 each; scores of some tens carry it into
# their exponentials.  Measured up to 8e-7.
REL = 5e-6


def make(dev, d, bits, kvh, blocks, bs, seed, pad=4):
    rng = np.random.default_rng(seed)
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev), dtype=torch.float32)
    rows = [torch.full((blocks, bs, kvh, tq._packed_dim + pad), 0x5A, dtype=torch.uint8, device=dev) for _ in range(2)]
    norms = [torch.zeros(blocks, bs, kvh, device=dev) for _ in range(2)]
    slots = torch.arange(blocks * bs, device=dev)
    for r, n in zip(rows, norms):
        x = torch.from_numpy(kv_like(rng, (blocks * bs, kvh, d)).astype(np.float32)).to(dev)
        akv.fused_kv_update(x, slots, r[..., :tq._packed_dim], n, tq.rotation, tq.boundaries_inner, bits, bs)
    return rng, tq, rows, norms


def dequantised(tq, rows, norms, d, bits):
    c, _, _ = O.get_codebook(d, bits)
    codes = O._UNPACK[bits](rows[..., :tq._packed_dim].cpu().numpy(), d)
    return torch.from_numpy(np.asarray(c, dtype=np.float64)[codes] * norms.double().cpu().numpy()[..., None])


def attend(q, K, V, R, counts=None):
    """q [heads, d], K and V [tokens, kv heads, d] in the rotated frame, each token `counts` times; float64."""
    heads, kvh = q.shape[0], K.shape[1]
    out = torch.zeros_like(q)
    for h in range(heads):
        s = K[:, h // (heads // kvh)] @ (R @ q[h]) / q.shape[1] ** 0.5
        p = torch.exp(s - s.max()) * (1.0 if counts is None else counts)
        out[h] = R.T @ (p @ V[:, h // (heads // kvh)] / p.sum())
    return out


HEADS = [(8, 1, 16), (16, 2, 32), (9, 3, 16), (28, 4, 16), (24, 2, 32), (5, 5, 32), (40, 8, 16), (18, 18, 16)]


@pytest.mark.parametrize("d,bits,qh,kvh,bs", [(d, bits, *h) for d in (64, 128, 256) for bits in (4, 2) for h in HEADS if d != 128 or (h[0] <= 16 and h[1] <= 2)])
def test_edges_vs_float64(dev, d, bits, qh, kvh, bs):
    """Contexts at the edges of blocks, tiles and chunks, empty sequences; one to eight heads a kv head, groups of them beyond
    eight, head slots left over, more heads than slots."""
    ctx = np.array([1, 0, 15, 16, 17, 31, 32, 33, 64, 65, 257, 1000, 0, 3], dtype=np.int32)
    need = -(-ctx // bs)
    blocks = int(need.sum()) + 2
    rng, tq, rows, norms = make(dev, d, bits, kvh, blocks, bs, d + bits + qh)
    tables = np.full((len(ctx), int(need.max())), 10 ** 6, dtype=np.int32)
    order, at = rng.permutation(blocks), 0
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n]
        at += int(n)
    q = torch.from_numpy(rng.standard_normal((len(ctx), qh, d)).astype(np.float32)).to(dev)
    P = tq._packed_dim
    print(f"[attn wave] d={d} bits={bits} qh={qh} kvh={kvh} bs={bs}", flush=True)
    out = akv.TQPagedAttention(tq, qh).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.from_numpy(tables).to(dev),
                                               torch.from_numpy(ctx).to(dev), block_size=bs).double().cpu()
    K, V = (dequantised(tq, r, n, d, bits) for r, n in zip(rows, norms))
    R = tq.rotation.double().cpu()
    for i, n in enumerate(ctx):
        if n == 0:
            assert not out[i].any()
            continue
        t = torch.from_numpy(tables[i, :need[i]].astype(np.int64))
        k, v = (x[t].reshape(-1, kvh, d)[:n] for x in (K, V))
        ref = attend(q[i].double().cpu(), k, v, R)
        assert (out[i] - ref).norm() <= REL * ref.norm(), (i, n)


@pytest.mark.parametrize("d,qh,kvh,bs", [(d, *h) for d in (64, 128, 256) for h in HEADS if d != 128 or (h[0] <= 16 and h[1] <= 2)])
def test_edges_of_3bit_rows_vs_float64(dev, d, qh, kvh, bs):
    """The same with 3-bit rows: groups of 24 bits, at head_dim 64 half of one a lane, none on a dword of its own."""
    test_edges_vs_float64(dev, d, 3, qh, kvh, bs)


@pytest.mark.parametrize("seqs,qh,kvh", [(70, 15, 3), (64, 16, 4), (65, 16, 16), (2, 3, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_reduce_of_head_dim_256_at_its_row_counts(dev, seqs, qh, kvh, dtype):
    """Around the number of rows from which sixteen are reduced at a time (four a CU), and row counts that no tile divides."""
    rng, tq, rows, norms = make(dev, 256, 4, kvh, 12, 16, seqs)
    ctx = rng.integers(0, 100, size=seqs).astype(np.int32)
    tables = rng.integers(0, 12, size=(seqs, 7)).astype(np.int32)
    q = torch.from_numpy(rng.standard_normal((seqs, qh, 256)).astype(np.float32)).to(dev).to(dtype)
    P = tq._packed_dim
    out = akv.TQPagedAttention(tq, qh).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.from_numpy(tables).to(dev),
                                               torch.from_numpy(ctx).to(dev)).double().cpu()
    K, V = (dequantised(tq, r, n, 256, 4) for r, n in zip(rows, norms))
    R = tq.rotation.double().cpu()
    for i, n in enumerate(ctx):
        if n == 0:
            assert not out[i].any()
            continue
        k, v = (x[torch.from_numpy(tables[i].astype(np.int64))].reshape(-1, kvh, 256)[:n] for x in (K, V))
        ref = attend(q[i].double().cpu(), k, v, R)
        # (bfloat16: the rounding of the output, 2^-9 of each)
        assert (out[i] - ref).norm() <= (REL if dtype == torch.float32 else 2.0 ** -9) * ref.norm(), (i, n)


@pytest.mark.parametrize("d,qh,kvh,bs,chunks", [(256, 16, 8, 16, 70), (256, 4, 1, 32, 70), (64, 16, 16, 32, 70),
                                                (256, 8, 8, 16, 32), (256, 8, 8, 32, 64), (64, 16, 16, 16, 64), (64, 16, 16, 32, 32)])
def test_more_chunks_than_a_window_of_block_ids(dev, d, qh, kvh, bs, chunks):
    """A context so long that a wavefront goes through several windows of block ids, of 32 chunks each: `chunks` a wavefront, or
    one less; at 32 and 64 the last chunk is the last of a window.  Its blocks repeat a few, which the reference counts."""
    rng, tq, rows, norms = make(dev, d, 4, kvh, 8, bs, 7)
    shares = 8 // kvh if kvh < 8 else 1
    n = 32 * 256 * chunks * shares - (5 if chunks == 70 else 0)
    table = rng.integers(0, 8, size=-(-n // bs)).astype(np.int32)
    q = torch.from_numpy(rng.standard_normal((1, qh, d)).astype(np.float32)).to(dev)
    P = tq._packed_dim
    out = akv.TQPagedAttention(tq, qh).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.from_numpy(table[None]).to(dev),
                                               torch.tensor([n], dtype=torch.int32, device=dev), block_size=bs).double().cpu()
    counts = np.zeros((8, bs))
    np.add.at(counts, table[:-1], 1.0)
    counts[table[-1], :n - (len(table) - 1) * bs] += 1.0
    K, V = (dequantised(tq, r, x, d, 4).reshape(-1, kvh, d) for r, x in zip(rows, norms))
    ref = attend(q[0].double().cpu(), K, V, tq.rotation.double().cpu(), torch.from_numpy(counts.reshape(-1)))
    # sums of 2^19 and more float32 terms in runs of some thousand: their rounding walks to a few times that of the test above
    assert (out[0] - ref).norm() <= 4 * REL * ref.norm()


@pytest.mark.parametrize("d,bits", [(64, 4), (256, 2), (128, 4)])
@pytest.mark.parametrize("scale_v,scale_q", [(1e30, 1.0), (1e-30, 1.0), (1.0, 1e-20), (1.0, 1e20)])
def test_norms_and_queries_far_outside_float16(dev, d, bits, scale_v, scale_q):
    """Value norms and queries float16 cannot hold (keys scaled against the queries), and NaN rows past the context."""
    rng, tq, rows, norms = make(dev, d, bits, 2, 8, 16, 3)
    n = 100
    norms[0] /= scale_q
    norms[1] *= scale_v
    norms[0].view(-1, 2)[n:] = float("nan")
    norms[1].view(-1, 2)[n:] = float("nan")
    q = torch.from_numpy(rng.standard_normal((1, 8, d)).astype(np.float32)).to(dev) * scale_q
    P = tq._packed_dim
    out = akv.TQPagedAttention(tq, 8).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.arange(8, dtype=torch.int32, device=dev)[None],
                                              torch.tensor([n], dtype=torch.int32, device=dev), block_size=16).double().cpu()
    K, V = (dequantised(tq, r, x, d, bits).reshape(-1, 2, d)[:n] for r, x in zip(rows, norms))
    ref = attend(q[0].double().cpu(), K, V, tq.rotation.double().cpu())
    assert (out[0] - ref).norm() <= REL * ref.norm()


@pytest.mark.parametrize("d,bits,qh,kvh,bs", [(64, 4, 16, 2, 16), (256, 4, 8, 4, 16), (256, 2, 4, 1, 32), (128, 4, 8, 1, 16), (128, 2, 5, 1, 32)])
@pytest.mark.parametrize("seqs", [63, 64, 65, 127, 300, 4300])
def test_many_sequences(dev, d, bits, qh, kvh, bs, seqs):
    """The axis cut into equal ranges, sequences searched in the prefix by one step (up to 63), two, and more (from 4,033 on),
    runs of empty ones among them; 64-bit tables and lengths, bfloat16 queries of strided heads."""
    ctx = np.random.default_rng(seqs).integers(0, 90, size=seqs)
    ctx[seqs // 3:seqs // 3 + seqs // 6] = 0
    ctx[0], ctx[-1] = 33, 0
    need = -(-ctx // bs)
    rng, tq, rows, norms = make(dev, d, bits, kvh, 40, bs, seqs + d)
    tables = np.full((seqs, int(need.max())), -1, dtype=np.int64)
    for i, n in enumerate(need):
        tables[i, :n] = rng.integers(0, 40, size=n)
    q = torch.from_numpy(rng.standard_normal((seqs, 2 * qh, d)).astype(np.float32)).to(dev).bfloat16()[:, ::2]
    P = tq._packed_dim
    print(f"[attn wave] many sequences: d={d} bits={bits} qh={qh} kvh={kvh} bs={bs} seqs={seqs}", flush=True)
    out = akv.TQPagedAttention(tq, qh).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.from_numpy(tables).to(dev),
                                               torch.from_numpy(ctx).to(dev), block_size=bs).double().cpu()
    K, V = (dequantised(tq, r, n, d, bits) for r, n in zip(rows, norms))
    R = tq.rotation.double().cpu()
    qc = q.double().cpu()
    for i in range(0, seqs, max(1, seqs // 100)):
        n = int(ctx[i])
        if n == 0:
            assert not out[i].any(), i
            continue
        t = torch.from_numpy(tables[i, :need[i]])
        k, v = (x[t].reshape(-1, kvh, d)[:n] for x in (K, V))
        ref = attend(qc[i], k, v, R)
        assert (out[i] - ref).norm() <= 2.0 ** -8 * ref.norm(), (i, n)      # (bfloat16 outputs: half a unit in the last place each)


@pytest.mark.parametrize("qh,kvh,seqs", [(8, 1, 1), (8, 1, 16), (4, 1, 70), (16, 2, 3), (16, 1, 32), (16, 2, 40), (32, 8, 4)])
@pytest.mark.parametrize("bits", [4, 3, 2])
def test_padding_of_the_tables_changes_nothing(dev, qh, kvh, seqs, bits):
    """A serving engine's block tables are as wide as its longest context may become: the kernel, and every bit of the result,
    are those of tables cut to the contexts."""
    rng, tq, rows, norms = make(dev, 128, bits, kvh, 30, 16, seqs)
    ctx = rng.integers(1, 400, size=seqs).astype(np.int32)
    tables = rng.integers(0, 30, size=(seqs, 25)).astype(np.int32)
    padded = np.zeros((seqs, 2 * 262144 // 16 // seqs + 25), dtype=np.int32)
    padded[:, :25] = tables
    q = torch.from_numpy(rng.standard_normal((seqs, qh, 128)).astype(np.float32)).to(dev)
    P = tq._packed_dim
    out = [akv.TQPagedAttention(tq, qh).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.from_numpy(t).to(dev),
                                                torch.from_numpy(ctx).to(dev), block_size=16) for t in (tables, padded)]
    assert torch.equal(*out)


@pytest.mark.parametrize("d,qh,kvh,most", [(64, 32, 8, 3.9e-7), (128, 8, 1, 4.85e-7), (256, 16, 4, 5.85e-7)])
def test_queries_are_rotated_as_well_as_in_float32(dev, d, qh, kvh, most):
    """The mean error of a head over many queries: with float32 multiply-adds 3.8, 4.8 and 5.7e-7, which is what is asked for; with
    three products of float16 pairs 4.2, 5.0 and 6.2; measured 3.7, 4.4 and 5.4."""
    n, seqs = 300, 64
    rng, tq, rows, norms = make(dev, d, 4, kvh, 20, 16, 23)
    q = torch.from_numpy(rng.standard_normal((seqs, qh, d)).astype(np.float32)).to(dev)
    P = tq._packed_dim
    out = akv.TQPagedAttention(tq, qh).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.arange(20, dtype=torch.int32, device=dev).expand(seqs, 20),
                                               torch.full((seqs,), n, dtype=torch.int32, device=dev), block_size=16).double().cpu()
    k, v = (dequantised(tq, r, m, d, 4).reshape(-1, kvh, d)[:n] for r, m in zip(rows, norms))
    R = tq.rotation.double().cpu()
    ref = torch.stack([attend(x, k, v, R) for x in q.double().cpu()])
    error = float(((out - ref).norm(dim=-1) / ref.norm(dim=-1)).mean())
    print(f"[rotated queries] d={d}: {error:.3e}", flush=True)
    assert error <= most


def many_sequences(rng, blocks):
    """Runs of empty sequences longer than a wavefront's lanes, at the start, in between and at the end, one sequence in most of
    the workgroups, many that share one: contexts and block tables."""
    ctx = np.concatenate([np.zeros(100), [30000], np.zeros(130), rng.integers(1, 130, size=150), np.zeros(70), rng.integers(1, 40, size=5), np.zeros(66)])
    return ctx.astype(np.int32), rng.integers(0, blocks, size=(len(ctx), 30000 // 16)).astype(np.int32)


# (128, (8, 1)): on this kernel; the other cases of 128 on the one of eight head slots, whose values are float16 levels (6.7e-5)
@pytest.mark.parametrize("d,bits,qh,kvh", [(128, 4, 32, 8), (128, 3, 28, 4), (128, 2, 6, 2), (128, 4, 8, 1), (64, 4, 32, 8), (256, 2, 16, 4)])
def test_many_sequences_and_empty_ones_vs_float64(dev, d, bits, qh, kvh):
    """More (sequence, head) items than workgroups reduce at a time, in one slot, a few, and more than 64."""
    rng, tq, rows, norms = make(dev, d, bits, kvh, 40, 16, d + bits + qh)
    ctx, tables = many_sequences(rng, 40)
    q = torch.from_numpy(rng.standard_normal((len(ctx), qh, d)).astype(np.float32)).to(dev)
    P = tq._packed_dim
    out = akv.TQPagedAttention(tq, qh).forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.from_numpy(tables).to(dev),
                                               torch.from_numpy(ctx).to(dev)).double().cpu()
    K, V = (dequantised(tq, r, n, d, bits) for r, n in zip(rows, norms))
    R = tq.rotation.double().cpu()
    assert not out[torch.from_numpy(ctx == 0)].any()
    for i in np.flatnonzero(ctx):
        t = torch.from_numpy(tables[i, :-(-int(ctx[i]) // 16)].astype(np.int64))
        k, v = (x[t].reshape(-1, kvh, d)[:ctx[i]] for x in (K, V))
        ref = attend(q[i].double().cpu(), k, v, R)
        assert (out[i] - ref).norm() <= (2.7e-4 if d == 128 and kvh > 1 else REL) * ref.norm(), (i, ctx[i])


@pytest.mark.parametrize("kind", ["whole, one long", "whole, half", "equal, one long", "equal, most", "equal, few"])
# the last two on the kernel of eight head slots
@pytest.mark.parametrize("d,bits,qh,kvh", [(64, 4, 32, 8), (256, 4, 16, 4), (128, 4, 8, 1), (128, 2, 32, 8), (128, 4, 16, 4)])
def test_ranges_of_workgroups_vs_float64(dev, kind, d, bits, qh, kvh):
    """Each way the blocks of a batch are cut among the workgroups: whole ones for a sequence, also where one sequence has most of
    them and where there are just as many sequences as half the workgroups; equal ranges that cross sequences, with at most 64
    sequences, with at most 256 and with more."""
    rng, tq, rows, norms = make(dev, d, bits, kvh, 40, 16, d + bits + qh)
    ctx, look = batch_of_ranges(rng, kind)
    tables = rng.integers(0, 40, size=(len(ctx), int(ctx.max() + 15) // 16)).astype(np.int32)
    q = torch.from_numpy(rng.standard_normal((len(ctx), qh, d)).astype(np.float32)).to(dev)
    P = tq._packed_dim
    attn = akv.TQPagedAttention(tq, qh)
    out = attn.forward(q, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], torch.from_numpy(tables).to(dev), torch.from_numpy(ctx).to(dev)).double().cpu()
    # (one kv head: eight wavefronts share a range, a round of them is what whole workgroups may be longer)
    assert whole_workgroups(attn, torch.cuda.get_device_properties(dev).multi_processor_count, ctx) == (kind.startswith("whole") or (kind == "equal, few" and kvh == 1))
    assert not out[torch.from_numpy(ctx == 0)].any()
    K, V = (dequantised(tq, r, n, d, bits) for r, n in zip(rows, norms))
    R = tq.rotation.double().cpu()
    for i in look:
        t = torch.from_numpy(tables[i, :-(-int(ctx[i]) // 16)].astype(np.int64))
        k, v = (x[t].reshape(-1, kvh, d)[:ctx[i]] for x in (K, V))
        ref = attend(q[i].double().cpu(), k, v, R)
        assert (out[i] - ref).norm() <= (2.7e-4 if d == 128 and kvh > 1 else REL) * ref.norm(), (i, ctx[i])
