"""The matrix-core decode kernel at the edges of a step and of the grid, against the oracle's codes in float64."""
import numpy as np
import pytest
import torch

import aitherkvcache_amd as akv
from aitherkvcache_amd.vllm.decompress import batch_decompress_active_blocks, decode_blocks
from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu

# Against 64 bits: the two-term operands and float32 sums stay below 2^-20 of a row's length (three products of 2^-22 and
# the float32 rounding of at most 256 terms), the cast adds half a unit of the output type (2^-11, 2^-8) of the element.
UNIT = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def check(got, packed, norms, tq, dtype):
    d = tq.head_dim
    c = tq.centroids.cpu().numpy().astype(np.float64)
    y = c[O._UNPACK[tq.bits](packed.reshape(-1, packed.shape[-1])[:, :tq._packed_dim], d).astype(np.int64)]
    ref = (y @ tq.rotation.cpu().numpy().astype(np.float64)) * norms.reshape(-1, 1).astype(np.float64)
    err = np.abs(got.reshape(-1, d).astype(np.float64) - ref)
    bound = np.abs(ref) * UNIT[dtype] * 1.01 + np.linalg.norm(ref, axis=-1, keepdims=True) * 2.0 ** -20 + (2.0 ** -25 if dtype == torch.float16 else 0)
    assert np.all(err <= bound), float(np.max(err - bound))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,bits", [(d, b) for d in (64, 128, 256) for b in (4, 3, 2)])
def test_flat_rows(dev, d, bits, dtype):
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev), dtype=dtype)
    rng = np.random.default_rng(d + bits)
    for n in (1, 15, 16, 33, 700) + ((70001,) if bits == 4 else ()):       # (the last: more steps than row groups)
        packed = rng.integers(0, 256, (n, tq._packed_dim), dtype=np.uint8)
        norms = rng.lognormal(0, 1, n).astype(np.float32)
        print(f"[decode] d={d} bits={bits} {dtype} n={n}", flush=True)
        out = tq.decode(torch.from_numpy(packed).to(dev), torch.from_numpy(norms).to(dev))
        assert out.dtype == dtype
        k = slice(None) if n < 1000 else slice(n - 500, n)
        check(out[k].float().cpu().numpy(), packed[k], norms[k], tq, dtype)


@pytest.mark.parametrize("d,bits,heads,bs,dtype", [(64, 4, 3, 16, torch.bfloat16), (64, 3, 1, 32, torch.float16), (128, 4, 8, 16, torch.float32),
                                                   (128, 2, 5, 7, torch.float16), (256, 3, 2, 16, torch.bfloat16), (256, 4, 1, 1, torch.float16)])
def test_listed_blocks(dev, d, bits, heads, bs, dtype):
    """Padding, repeated and out-of-range ids; rows behind reserved bytes; K and V in one launch, from one tensor and from
    tensors whose layouts differ; outputs that share storage; blocks that are not listed keep what they held."""
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev), dtype=dtype)
    rng = np.random.default_rng(heads)
    P, blocks = tq._packed_dim, 37
    both = torch.from_numpy(rng.integers(0, 256, (blocks, 2, bs, heads, P + 4), dtype=np.uint8)).to(dev)
    norms = [torch.from_numpy(rng.lognormal(0, 1, (blocks, bs, heads)).astype(np.float32)).to(dev) for _ in range(2)]
    table = np.array([[5, 9, 9, 9, 0, 0, 0, -1, -1], [30, 2, 36, 37, 99, 2, 5, 0, 0], [-5, -1, 17, 17, 3, 4, 17, 17, 35]], dtype=np.int64)
    listed = sorted({int(b) for b in table.ravel() if 0 <= b < 36})        # (36 lies outside the declared blocks)
    rest = [b for b in range(blocks) if b not in listed]

    def caches(form):
        k, v = both[:, 0], both[:, 1]
        return (k, v) if form != "differ" else (k, v.contiguous())

    for form in ("same", "differ", "shared"):
        for ids in (torch.from_numpy(table).to(dev), torch.from_numpy(table.astype(np.int32)).to(dev)):
            k, v = caches(form)
            if form == "shared":
                pair = torch.full((blocks, bs, heads, 2, d), 7.0, dtype=dtype, device=dev)
                outs = [pair[..., 0, :], pair[..., 1, :]]
            else:
                outs = [torch.full((blocks, bs, heads, d), 7.0, dtype=dtype, device=dev) for _ in range(2)]
            print(f"[decode blocks] d={d} bits={bits} {form} {ids.dtype}", flush=True)
            batch_decompress_active_blocks(k, v, outs[0], outs[1], tq, P, ids, 36, norms[0], norms[1])
            for o, rows, n in zip(outs, (k, v), norms):
                check(o[listed].float().cpu().numpy(), rows[listed].cpu().numpy(), n[listed].cpu().numpy(), tq, dtype)
                assert bool((o[rest] == 7.0).all())
                one = torch.full((blocks, bs, heads, d), 7.0, dtype=dtype, device=dev)
                decode_blocks(rows, n, one, tq, ids, 36)
                assert torch.equal(one, o)


@pytest.mark.parametrize("factor", [3000.0, 1e-4, 2.0 ** 100])
@pytest.mark.parametrize("d,bits", [(64, 4), (64, 3), (128, 4), (256, 4), (256, 2)])
def test_matrices_that_are_no_rotation(dev, d, bits, factor):
    """An assigned matrix may have entries far outside what two float16 terms hold: it is scaled by its largest."""
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev), dtype=torch.float32)
    tq.rotation = tq.rotation * factor
    rng = np.random.default_rng(bits)
    packed, norms = rng.integers(0, 256, (100, tq._packed_dim), dtype=np.uint8), rng.lognormal(0, 1, 100).astype(np.float32)
    out = tq.decode(torch.from_numpy(packed).to(dev), torch.from_numpy(norms).to(dev))
    check(out.cpu().numpy(), packed, norms, tq, torch.float32)


@pytest.mark.parametrize("d,bits", [(64, 4), (128, 4), (128, 3), (256, 2)])
@pytest.mark.parametrize("far", ["heads of the cache", "heads of the output", "positions of the norms"])
def test_strides_beyond_24_bits(dev, d, bits, far):
    """Heads or positions that lie further apart than 2^24 elements take the same kernel, to the same bits."""
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev), dtype=torch.float32)
    rng = np.random.default_rng(d)
    P, blocks, bs, heads = tq._packed_dim, 5, 4, 2
    rows = torch.from_numpy(rng.integers(0, 256, (blocks, bs, heads, P), dtype=np.uint8)).to(dev)
    norms = torch.from_numpy(rng.lognormal(0, 1, (blocks, bs, heads)).astype(np.float32)).to(dev)
    ids = torch.tensor([3, 0, 0, 4, 7, -1], device=dev)
    want = torch.zeros(blocks, bs, heads, d, device=dev)
    decode_blocks(rows, norms, want, tq, ids, blocks)

    def spread(t, dim):                       # the same values, `dim` 2^24 elements (and a few rows) apart
        step = (1 << 24) + 64 * t.shape[-1]
        shape = [n for i, n in enumerate(t.shape) if i != dim]
        inner = torch.zeros(shape).stride()
        strides = list(inner[:dim]) + [step] + list(inner[dim:])
        out = torch.zeros(step * t.shape[dim], dtype=t.dtype, device=dev).as_strided(t.shape, strides)
        out.copy_(t)
        return out
    got = torch.zeros_like(want)
    if far == "heads of the cache":
        rows = spread(rows, 2)
    elif far == "heads of the output":
        got = spread(got, 2)
    else:
        norms = spread(norms, 1)
    decode_blocks(rows, norms, got, tq, ids, blocks)
    assert torch.equal(got, want)


def test_more_rows_than_32_bits_count(dev):
    """A list so long that the rows of K and V pass 2^31 is decoded in pieces, by the same kernel: most of it padding."""
    tq = akv.TurboQuant(head_dim=64, bits=4, device=str(dev), dtype=torch.float32)
    rng = np.random.default_rng(0)
    blocks, bs, heads = 12, 32, 8
    rows = [torch.from_numpy(rng.integers(0, 256, (blocks, bs, heads, tq._packed_dim), dtype=np.uint8)).to(dev) for _ in range(2)]
    norms = [torch.from_numpy(rng.lognormal(0, 1, (blocks, bs, heads)).astype(np.float32)).to(dev) for _ in range(2)]
    short = torch.tensor([3, 1, 11, 5, 6, 2, 9], dtype=torch.int32, device=dev)
    ids = torch.full(((1 << 22) + 10,), -1, dtype=torch.int32, device=dev)
    piece = (1 << 29) // (bs * heads)
    for at, i in zip((0, piece - 1, piece, piece + 1, 2 * piece, len(ids) - 2, len(ids) - 1), short.tolist()):
        ids[at] = i
    outs = []
    for listed in (short, ids):
        o = [torch.zeros(blocks, bs, heads, 64, device=dev) for _ in range(2)]
        batch_decompress_active_blocks(*rows, *o, tq, tq._packed_dim, listed, blocks, *norms)
        outs.append(o)
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("d,bits,form", [(512, 4, "head_dim"), (512, 3, "head_dim")] + [(d, b, f) for d, b in ((64, 4), (128, 3), (256, 2)) for f in ("odd rows", "odd output of V")])
def test_keys_and_values_the_matrix_kernel_does_not_take_together(dev, d, bits, form):
    """Equal layouts of K and V that one launch cannot take: head_dim 512, rows of an odd pitch (the vector kernel for both), an
    output of V that lies 4 bytes off (the matrix kernel for K, the vector kernel for V)."""
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev), dtype=torch.float32)
    rng = np.random.default_rng(d + bits)
    P, blocks, bs, heads = tq._packed_dim, 9, 16, 3
    pad = 1 if form == "odd rows" else 4
    both = torch.from_numpy(rng.integers(0, 256, (2, blocks, bs, heads, P + pad), dtype=np.uint8)).to(dev)
    norms = torch.from_numpy(rng.lognormal(0, 1, (2, blocks, bs, heads)).astype(np.float32)).to(dev)
    off = 1 if form == "odd output of V" else 0
    outs = [torch.full((blocks * bs * heads * d + 4,), 7.0, device=dev)[o:o + blocks * bs * heads * d].view(blocks, bs, heads, d) for o in (0, off)]
    listed, rest = [1, 2, 7, 8], [0, 3, 4, 5, 6]
    ids = torch.tensor([[7, 1, -1], [8, 2, 30]], device=dev)
    batch_decompress_active_blocks(both[0], both[1], outs[0], outs[1], tq, P, ids, blocks, norms[0], norms[1])
    for o, rows, n in zip(outs, both, norms):
        check(o[listed].cpu().numpy(), rows[listed].cpu().numpy(), n[listed].cpu().numpy(), tq, torch.float32)
        assert bool((o[rest] == 7.0).all())
