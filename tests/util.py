"""Shared helpers for the parity tests."""
import numpy as np

from oracle import tq_oracle as O

MAX_ULPS = 16       # a code may differ from the float32 oracle only if the float64 rotated value
                    # lies within this many float32 ulps of a decision boundary


def kv_like(rng, shape, dtype=np.float16):
    """N(0,1) entries times a lognormal(0, 0.5) scale per vector (the benchmark's distribution)."""
    g = rng.standard_normal(shape, dtype=np.float32)
    s = rng.lognormal(0.0, 0.5, size=shape[:-1]).astype(np.float32)
    return (g * s[..., None]).astype(dtype)


def code_mismatch_report(codes_a, codes_b, y64, boundaries, oracle, unit64=None, R=None):
    """The oracle's account of differing codes (count, max_ulps, histogram dict)."""
    return oracle.code_mismatch_report(codes_a, codes_b, y64, boundaries, unit64, R)


def check_codes(packed, norms, x, R, bits, ref_packed=None, ref_norms=None, d=128):
    """Bit-exact codes modulo the boundary-ulp rule; norms to 1e-6 relative."""
    _, b, _ = O.get_codebook(d, bits)
    if ref_packed is None:
        ref_packed, ref_norms = O.encode(x, R, b, bits)
    ca = O._UNPACK[bits](packed.reshape(-1, packed.shape[-1]), d)
    cb = O._UNPACK[bits](ref_packed.reshape(-1, ref_packed.shape[-1]), d)
    x64 = np.asarray(x).reshape(-1, d).astype(np.float64)
    y64 = O.rotate_unit_f64(np.asarray(x).reshape(-1, d), R)
    with np.errstate(invalid="ignore", over="ignore"):
        unit64 = x64 / (np.linalg.norm(x64, axis=-1, keepdims=True) + 1e-10)
    n, max_ulps, hist = code_mismatch_report(ca, cb, y64, b, O, unit64, R)
    total = ca.size
    print(f"[codes] bits={bits} mismatching={n}/{total} max_ulps={max_ulps:.2f} hist={hist}")
    assert max_ulps <= MAX_ULPS, hist
    assert hist.get("max_code_step", 1) == 1
    assert n <= max(3, total * 2e-5), (n, total)
    nr = np.asarray(ref_norms).reshape(-1).astype(np.float64)
    ng = np.asarray(norms).reshape(-1).astype(np.float64)
    nz = nr > 0
    assert np.max(np.abs(ng[nz] - nr[nz]) / nr[nz]) < 1e-6
    assert np.all(ng[~nz] == 0)
    return n


def whole_workgroups(attn, ranges, ctx, block_size=16):
    """How the last call of an attention object cut the blocks of its batch among `ranges` workgroups, from the records in its
    workspace (behind 4,352 bytes: range, sequence, the sequence's blocks, its tokens): whole ones for every sequence, or ranges that cross
    sequences.  The records are checked on the way."""
    records = attn._workspace[4352:4352 + 32 * ranges].cpu().numpy().view(np.int32).reshape(ranges, 8)
    ends = np.cumsum(-(-np.asarray(ctx, dtype=np.int64) // block_size))
    at, whole = 0, True
    for g0, g1, seq, sb0, sb1, tokens in records[:, :6]:
        if g0 >= g1:
            assert seq == -1
            continue
        assert g0 == at and seq == np.searchsorted(ends, g0, side="right"), (g0, g1, seq)
        assert (sb0, sb1, tokens) == (ends[seq - 1] if seq else 0, ends[seq], ctx[seq]), (g0, seq)
        whole &= bool(g1 <= sb1)
        at = g1
    assert at == ends[-1]
    return whole


def batch_of_ranges(rng, kind):
    """Contexts of a batch for each way its blocks are cut, with 65 to 256 sequences and at most 64, and the sequences to look at."""
    if kind == "whole, one long":            # runs of empty sequences longer than a wavefront, one sequence in most of the workgroups
        ctx = np.concatenate([np.zeros(70), [30000], rng.integers(1, 130, size=60), np.zeros(66), rng.integers(1, 40, size=5)])
    elif kind == "whole, half":              # as many sequences as half the workgroups
        ctx = rng.integers(290, 310, size=128)
    elif kind == "whole, short":
        ctx = rng.integers(230, 256, size=60)
    elif kind == "equal, one long":
        ctx = np.concatenate([rng.integers(1, 130, size=110), np.zeros(25), [30000], rng.integers(1, 130, size=110), np.zeros(10)])
    elif kind == "equal, most":              # more than are held by a thread each: two or three starts a thread
        ctx = np.concatenate([rng.integers(1, 130, size=300), np.zeros(100), [30000], rng.integers(1, 130, size=200), np.zeros(60)])
    elif kind == "equal, ragged":            # a decode batch of mixed lengths
        ctx = rng.integers(532, 10112, size=33)
    else:                                    # "equal, few": sequences that do not divide the workgroups
        ctx = rng.integers(7969, 8001, size=55 if kind == "equal, few (55)" else 60)
    ctx = ctx.astype(np.int32)
    some = np.flatnonzero(ctx)
    look = some if len(some) < 100 else np.concatenate([some[:3], some[30:80:5], [int(ctx.argmax())], some[100::9], some[-2:]])
    return ctx, look if "few" not in kind and "ragged" not in kind else some[[0, 1, 2, 14, 30, -2, -1]]
