"""The binding of the hot calls takes plain well-formed calls and leaves every other one to the long way: both give the same bytes,
and what the long way converts, allocates or refuses is converted, allocated or refused as before."""
import contextlib

import pytest
import torch

import aitherkvcache_amd as akv
from aitherkvcache_amd import _lib
from aitherkvcache_amd.hybrid_attention import hybrid_encode_and_store_pair
from aitherkvcache_amd.triattention import TriAttention, TriAttentionConfig
from aitherkvcache_amd.triattention.cache import SpectralKVCache
from aitherkvcache_amd.vllm.decompress import batch_decompress_active_blocks

pytestmark = pytest.mark.gpu
S, QH, KVH, BS, NB = 3, 8, 2, 16, 20


class Sub(torch.Tensor):
    pass


class Counting:
    """The binding with a count of the calls it took; taken=None: it takes none."""

    def __init__(self, real, take):
        self.real, self.take, self.taken = real, take, 0

    def __getattr__(self, name):
        def call(*args):
            res = getattr(self.real, name)(*args) if self.take else None
            self.taken += res is not None
            return res
        return call


@contextlib.contextmanager
def binding(monkeypatch, take):
    c = Counting(_lib.calls(), take)
    with monkeypatch.context() as m:
        m.setattr(_lib, "_calls", c)
        yield c


def uniform(dev, bits, d, dtype):
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev))
    attn = akv.TQPagedAttention(tq, QH)

    def run(x, slots, tables, lens, q):
        rows = [torch.zeros(NB, BS, KVH, tq._packed_dim, dtype=torch.uint8, device=dev) for _ in range(2)]
        norms = [torch.zeros(NB, BS, KVH, device=dev) for _ in range(2)]
        akv.fused_kv_update_pair(x[0], x[1], slots, rows[0], norms[0], rows[1], norms[1], tq.rotation, tq.boundaries_inner, bits, BS, NB,
                                 prepared=tq.prepared_rotation())
        bufs = [torch.zeros(NB, BS, KVH, d, dtype=dtype, device=dev) for _ in range(2)]
        batch_decompress_active_blocks(rows[0], rows[1], bufs[0], bufs[1], tq, tq._packed_dim, tables, NB, norms[0], norms[1])
        return rows + norms + bufs + [attn.forward(q, rows[0], norms[0], rows[1], norms[1], tables, lens, block_size=BS)]
    return run, 3


def hybrid(dev, mode, d, dtype):
    h = akv.HybridTurboQuant(head_dim=d, mode=mode, device=str(dev))
    h.calibrate_uniform(KVH)
    attn = akv.HybridPagedAttention(h, QH)

    def run(x, slots, tables, lens, q):
        rows = [torch.zeros(NB, BS, KVH, h.packed_dim, dtype=torch.uint8, device=dev) for _ in range(2)]
        hybrid_encode_and_store_pair(h, x[0], x[1], slots, rows[0], rows[1], BS)
        return rows + [attn.forward(q, rows[0], rows[1], tables, lens, block_size=BS)]
    return run, 2


def spectral(dev, _, d, dtype):
    tri = TriAttention(TriAttentionConfig(head_dim=d, num_freqs=12, coeff_bits=4, num_kv_heads=KVH, num_query_heads=QH, block_size=BS), device=str(dev))

    def run(x, slots, tables, lens, q):
        cache = SpectralKVCache(tri.config, max_blocks=NB, device=str(dev))
        cache.encode_and_store(x[0], x[1], slots)
        return list(cache._arrays()) + [tri.decode_step_paged(q, cache, tables, lens)]
    return run, 2


CASES = [(uniform, 4, 128), (uniform, 3, 64), (uniform, 2, 256), (hybrid, "tq35", 128), (hybrid, "tq25", 128), (spectral, None, 128)]


def inputs(dev, d, dtype, itype):
    gen = torch.Generator(device=dev).manual_seed(d)
    x = torch.randn(2, NB * BS, KVH, d, device=dev, generator=gen).to(dtype)
    q = torch.randn(S, QH, d, device=dev, generator=gen).to(dtype)
    tables = torch.randperm(NB, device=dev, generator=gen)[:S * 5].reshape(S, 5).to(itype)
    lens = torch.tensor([80, 33, 1], device=dev, dtype=itype)
    return x, torch.arange(NB * BS, device=dev, dtype=itype), tables, lens, q


def check(got, want):
    assert all(a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b) for a, b in zip(got, want, strict=True))


@pytest.mark.parametrize("make,fmt,d", CASES)
@pytest.mark.parametrize("dtype,itype", [(torch.float16, torch.int32), (torch.bfloat16, torch.int64), (torch.float32, torch.int64)])
def test_binding_and_long_way_give_the_same(dev, monkeypatch, make, fmt, d, dtype, itype):
    run, calls = make(dev, fmt, d, dtype)
    args = inputs(dev, d, dtype, itype)
    with binding(monkeypatch, False):
        want = run(*args)
    with binding(monkeypatch, True) as c:
        check(run(*args), want)
        assert c.taken == calls
        x, slots, tables, lens, q = args
        # every second token of a wider tensor, tables cut out of wider ones: as the strides say
        wide, wt = torch.zeros(2, NB * BS, KVH + 1, d, dtype=dtype, device=dev), torch.full((S, 9), 10 ** 6, dtype=itype, device=dev)
        wide[:, :, 1:], wt[:, 2:7] = x, tables
        c.taken = 0
        check(run(wide[:, :, 1:], slots, wt[:, 2:7], lens, q), want)
        # the long way takes: transposed queries and tokens (copied), lengths of every second entry (copied), wrapped tensors
        c.taken = 0
        turned = q.transpose(1, 2).contiguous().transpose(1, 2)
        check(run(x.transpose(2, 3).contiguous().transpose(2, 3), slots, tables, lens, turned), want)
        check(run(x, slots, tables, lens.repeat_interleave(2)[::2], q), want)
        before = c.taken
        check(run([v.as_subclass(Sub) for v in x], slots, tables, lens, q), want)
        assert c.taken > before                                     # (the calls without such a tensor)


@pytest.mark.parametrize("make,fmt,d", CASES)
def test_refusals_stay(dev, monkeypatch, make, fmt, d):
    run, _ = make(dev, fmt, d, torch.float16)
    x, slots, tables, lens, q = inputs(dev, d, torch.float16, torch.int32)
    run(x, slots, tables, lens, q)                                  # the attention's workspace is there
    refused = [(x, slots, tables, lens, q[:, :, :d // 2]), (x, slots, tables, lens, q[:, :5]), (x, slots, tables[0], lens, q), (x, slots, tables, lens, q.cpu())]
    if make is not uniform:
        refused.append((x[:, :, :, :d // 2], slots, tables, lens, q))
    if make is spectral:
        refused += [(x, slots[:5], tables, lens, q), (x, slots, tables, lens[:2], q)]
    else:
        refused.append((x, slots, tables.short(), lens, q))
    for args in refused:
        errors = []
        for take in (False, True):
            with binding(monkeypatch, take), pytest.raises(Exception) as e:
                run(*args)
            errors.append((e.type, str(e.value)))
        assert errors[0] == errors[1]


@pytest.mark.parametrize("take", [False, True])
@pytest.mark.parametrize("fmt", ["uniform", "tq35"])
def test_sizes_that_do_not_fit_are_refused(dev, monkeypatch, fmt, take):
    """Nothing is launched that would read past a table, a list of lengths or slots, or a cache; neither way.  (Larger ones are fine.)"""
    d, uni = 128, fmt == "uniform"
    x, slots, tables, lens, q = inputs(dev, d, torch.float16, torch.int32)
    t = akv.TurboQuant(head_dim=d, bits=4, device=str(dev)) if uni else akv.HybridTurboQuant(head_dim=d, mode=fmt, device=str(dev))
    if not uni:
        t.calibrate_uniform(KVH)
    attn = (akv.TQPagedAttention if uni else akv.HybridPagedAttention)(t, QH)
    prep = t.prepared_rotation() if uni else None

    def caches(positions=BS, heads=KVH, norm_blocks=NB, norm_positions=BS, norm_heads=KVH):
        rows = [torch.zeros(NB, positions, heads, t._packed_dim if uni else t.packed_dim, dtype=torch.uint8, device=dev) for _ in range(2)]
        norms = [torch.zeros(norm_blocks, norm_positions, norm_heads, device=dev) for _ in range(2)]
        return (rows[0], norms[0], rows[1], norms[1]) if uni else tuple(rows)

    def write(c, x=x, slots=slots, block=BS, blocks=NB, prep=prep):
        if uni:
            akv.fused_kv_update_pair(x[0], x[1], slots, *c, t.rotation, t.boundaries_inner, 4, block, blocks, prepared=prep)
        else:
            hybrid_encode_and_store_pair(t, x[0], x[1], slots, *c, block, blocks)
        return c

    def read(c, tables=tables, lens=lens, block=BS, kv_heads=None):
        return attn.forward(q, *c, tables, lens, block_size=block, num_kv_heads=kv_heads)

    good = write(caches())
    want = read(good)                                               # the attention's workspace is there
    with binding(monkeypatch, take) as c:
        for args in [dict(tables=tables[:2]), dict(lens=lens[:2]), dict(block=2 * BS), dict(kv_heads=2 * KVH)]:
            with pytest.raises(ValueError):
                read(good, **args)
        bad = [(caches(), dict(slots=slots[:5])), (caches(), dict(block=2 * BS)), (caches(heads=KVH - 1), {}), (caches(positions=BS // 2), {})]
        if uni:
            bad += [(caches(norm_positions=BS // 2), {}), (caches(norm_heads=KVH - 1), {}), (caches(), dict(x=x[..., :64], prep=prep))]
            for shape in (dict(norm_positions=BS // 2), dict(norm_heads=KVH - 1)):
                with pytest.raises(ValueError):
                    read(caches(**shape))
        for cache, args in bad:
            with pytest.raises(ValueError):
                write(cache, **args)
        assert c.taken == 0
        # accepted as ever: more rows and lengths than sequences, fewer heads and positions than the cache has
        assert torch.equal(read(good, tables=torch.cat([tables, tables]), lens=torch.cat([lens, lens])), want)
        assert torch.equal(read(write(caches(positions=2 * BS, heads=KVH + 1, norm_positions=2 * BS, norm_heads=KVH + 1)), kv_heads=KVH), want)
        # blocks past the end of the cache or of its norms are skipped, whatever number of blocks is named
        far = slots + (slots >= NB * BS // 2) * NB * BS
        half = write(caches(), slots=far, blocks=10 ** 6)
        for a, b in zip(half, good):
            assert torch.equal(a[:NB // 2], b[:NB // 2]) and not a[NB // 2:].any()
        if uni:
            short = write(caches(norm_blocks=NB // 2))
            assert torch.equal(short[0][:NB // 2], good[0][:NB // 2]) and torch.equal(short[3], good[3][:NB // 2]) and not short[2][NB // 2:].any()
        assert (c.taken > 0) == take


@pytest.mark.parametrize("take", [False, True])
@pytest.mark.parametrize("make,fmt,d", [(uniform, 4, 128), (hybrid, "tq35", 128), (spectral, None, 128)])
def test_out_of_memory_is_the_error_of_torch(dev, monkeypatch, make, fmt, d, take):
    """What an engine catches to shrink its batch: the output of a call does not fit the memory that is left."""
    run, _ = make(dev, fmt, d, torch.float32)
    x, slots, _, _, _ = inputs(dev, d, torch.float32, torch.int32)
    many = 20000                                                    # 82 MB of output
    torch.cuda.empty_cache()                                        # (no segment is held of which that could be a part)
    q = torch.zeros(many, QH, d, device=dev)
    tables, lens = torch.zeros(many, 1, dtype=torch.int32, device=dev), torch.zeros(many, dtype=torch.int32, device=dev)
    run(x[:, :BS], slots[:BS], tables, lens, q)                     # the attention's workspace is there
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    # a segment of torch's that is held for a part of it, as other tests may leave them: there is room in it for the output
    whole = torch.empty(600 << 20, dtype=torch.uint8, device=dev)
    del whole
    held = [torch.empty(20 << 20, dtype=torch.uint8, device=dev)]
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + (16 << 20)) / total, dev)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            while True:                                             # (what such segments have left)
                held.append(torch.empty(16 << 20, dtype=torch.uint8, device=dev))
        with binding(monkeypatch, take), pytest.raises(torch.OutOfMemoryError):
            run(x[:, :BS], slots[:BS], tables, lens, q)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
        del held
    assert not run(x[:, :BS], slots[:BS], tables, lens, q)[-1].any()
