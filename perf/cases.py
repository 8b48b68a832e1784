"""The work a serving program has this package do, as cases that can be timed.

Four kinds of pass, each through the public entry points:

  step    one decode step of one layer: the step's new keys and values go into the compressed cache
          (fused_kv_update_pair / fused_encode_and_store / hybrid_encode_and_store_pair), then every sequence attends
          over its whole context (TQPagedAttention / HybridPagedAttention)
  write   the keys and values of a prompt chunk into the compressed cache, same entry points
  read    the cache back to plain vectors, what a prompt chunk over an existing context needs before dense attention
          (batch_decompress_active_blocks; HybridTurboQuant.decode)
  tri     one TriAttention decode step over the paged spectral cache: encode_and_store, then decode_step_paged

`listed()` are the cases by name, `draw(rng)` one more of the same ranges.  A case is a flat dict:

  kind      see above
  fmt       cache format: "4bit", "3bit", "2bit" (uniform codes + float32 norms), "tq35", "tq25" (hybrid rows), "f12" (tri)
  d, heads, kv_heads, block          head size, query and kv heads of the layer, tokens per cache block
  dtype     of queries, keys, values and outputs: "bf16", "f16", "f32"
  layout    "primary": K and V rows inside one [blocks, 2, block, kv_heads, row] byte tensor, the tensor a serving engine
            allocates; "split": one tensor per kind, as the package's own cache object keeps them
  seqs, ctx_lo, ctx_hi, lens_seed    sequences and their context lengths, uniform in [ctx_lo, ctx_hi]
  tokens    of a write
"""
import math

import numpy as np
import torch

import aitherkvcache_amd as akv
from aitherkvcache_amd.triattention import TriAttention, TriAttentionConfig
from aitherkvcache_amd.triattention.cache import SpectralKVCache
from aitherkvcache_amd.vllm.decompress import batch_decompress_active_blocks
from aitherkvcache_amd.vllm.engine import primary_views
from aitherkvcache_amd.vllm.kv_cache_dtype import KV_CACHE_DTYPES, tq_dim_for_head

DEVICE = "cuda:0"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
BITS = {"4bit": 4, "3bit": 3, "2bit": 2}
FORMATS = {"4bit": "tq-t4nc", "3bit": "tq-t3nc", "2bit": "tq-t2nc", "tq35": "tq35", "tq25": "tq25"}
TRI_FREQS = 12


def listed():
    def step(name, fmt, seqs, lo, hi, **more):
        case = dict(name=name, kind="step", fmt=fmt, d=128, heads=32, kv_heads=8, block=16, dtype="bf16", layout="primary",
                    seqs=seqs, ctx_lo=lo, ctx_hi=hi, lens_seed=2)
        case.update(more)
        return case

    return [
        # a single user's chat, a few hundred tokens in: the step whose time is launches and calls
        step("step_one_user", "4bit", 1, 700, 700),
        # a full batch of short conversations
        step("step_short_batch", "4bit", 256, 64, 512),
        # the headline benchmark: 16 ragged long contexts, cache tensors of the package's own layout
        step("step_long_ragged", "4bit", 16, 1024, 40960, dtype="f16", layout="split"),
        # one of eight ranks of a 64-head model: a rank keeps one kv head and its eight query heads
        step("step_one_kv_head", "4bit", 48, 1024, 16384, heads=8, kv_heads=1),
        # the 3- and 2-bit formats at the benchmark's batch of 64 contexts around 8k
        step("step_3bit", "3bit", 64, 8192, 8192, dtype="f16", layout="split"),
        step("step_2bit", "2bit", 64, 4000, 8192),
        # the other head sizes serving engines ask for
        step("step_heads_of_64", "4bit", 48, 512, 8192, d=64),
        step("step_heads_of_256", "4bit", 24, 512, 8192, d=256, heads=16, kv_heads=4),
        # the hybrid format of the benchmark, ragged
        step("step_tq35", "tq35", 64, 4000, 8192),
        # a prompt chunk's keys and values into the cache
        dict(name="write_chunk", kind="write", fmt="4bit", d=128, heads=32, kv_heads=8, block=16, dtype="bf16", layout="primary", tokens=8192),
        # the context of four prompts back to bfloat16 blocks, for dense attention of the next chunk
        dict(name="read_context", kind="read", fmt="4bit", d=128, heads=32, kv_heads=8, block=16, dtype="bf16", layout="primary",
             seqs=4, ctx_lo=2000, ctx_hi=8000, lens_seed=2),
        # the spectral cache at its benchmark's shape
        dict(name="tri_step", kind="tri", fmt="f12", d=128, heads=32, kv_heads=8, block=16, dtype="f16", layout="split",
             seqs=8, ctx_lo=24000, ctx_hi=32768, lens_seed=2),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choices(("step", "write", "read", "tri"), (60, 18, 11, 11))[0]
    case = dict(kind=kind, fmt="f12", d=128, dtype=rng.choices(("bf16", "f16", "f32"), (55, 35, 10))[0],
                block=rng.choices((16, 32), (80, 20))[0], layout=rng.choice(("primary", "split")))
    if kind != "tri":
        case["fmt"] = rng.choices(("4bit", "3bit", "2bit", "tq35", "tq25"), (45, 14, 13, 18, 10))[0]
        if case["fmt"] in BITS:
            case["d"] = rng.choices((64, 128, 256), (17, 66, 17))[0]
    else:
        case["layout"] = "split"
    # whole layers, and the slices of them that ranks of a sharded model keep
    case["heads"], case["kv_heads"] = rng.choices(((32, 8), (64, 8), (16, 4), (8, 2), (8, 1), (28, 4), (40, 8), (16, 16)),
                                                  (34, 12, 12, 10, 10, 8, 7, 7))[0]
    if kind == "tri" and case["kv_heads"] > 8:
        case["heads"], case["kv_heads"] = 32, 8
    row = case["kv_heads"] * _row_bytes(case) * 2            # bytes of one token's keys and values
    if kind == "write":
        # serving-step batches up to whole prompt chunks
        case["tokens"] = log_int(16, max(64, min(16384, (64 << 20) // (case["kv_heads"] * case["d"] * 4))))
        return case
    # a batch that keeps between 1 and 256 sequences and at most some 200 MB of cache
    most = (200 << 20 if kind == "step" else 24 << 20 if kind == "read" else 100 << 20) // row
    case["seqs"] = log_int(1, 256) if kind == "step" else log_int(1, 32)
    mean = log_int(48, max(64, min(32768, most // case["seqs"])))
    spread = rng.choice((0.0, 0.3, 0.9))
    case["ctx_lo"], case["ctx_hi"] = max(1, int(mean * (1 - spread))), max(1, int(mean * (1 + spread)))
    case["lens_seed"] = rng.randrange(1000)
    return case


def _row_bytes(case):
    """Bytes a vector of the format takes in the cache (codes and norm)."""
    if case["fmt"] == "f12":
        return 2 * TRI_FREQS + 2
    if case["fmt"] in BITS:
        return case["d"] * BITS[case["fmt"]] // 8 + 4
    return 64 if case["fmt"] == "tq35" else 44


def _lens(case):
    rng = np.random.default_rng(case["lens_seed"])
    return rng.integers(case["ctx_lo"], case["ctx_hi"] + 1, size=case["seqs"]).astype(np.int64)


def work(case):
    vec_in = case["d"] * {"f16": 2, "bf16": 2, "f32": 4}[case["dtype"]]
    row, kvh, d = _row_bytes(case), case["kv_heads"], case["d"]
    uniform = case["fmt"] in BITS
    # operations that turn a vector into the cache's form or back: a dense rotation, or the fast transforms of the hybrid rows
    turn = 2 * d * d if uniform else 4 * d * math.log2(d) if case["fmt"] != "f12" else 4 * d
    if case["kind"] == "write":
        n = 2 * case["tokens"] * kvh
        return {"bytes": n * (vec_in + row) + 8 * case["tokens"], "flops": n * turn}
    tokens, seqs = int(_lens(case).sum()), case["seqs"]
    if case["kind"] == "read":
        out = vec_in if uniform else 4 * d
        return {"bytes": 2 * tokens * kvh * (row + out), "flops": 2 * tokens * kvh * turn}
    blocks = int((-(-_lens(case) // case["block"])).sum())
    new = 2 * seqs * kvh
    out = 4 * d if case["kind"] == "tri" else vec_in
    nbytes = 2 * tokens * kvh * row + new * (vec_in + row) + seqs * case["heads"] * (vec_in + out) + 4 * blocks + 12 * seqs
    per_token = 4 * d if case["kind"] != "tri" else 4 * 2 * TRI_FREQS
    return {"bytes": nbytes, "flops": tokens * case["heads"] * per_token + (new + 2 * seqs * case["heads"]) * turn}


def tolerance(case):
    # Codes are whole values; one that lies on a decision boundary to within float32 rounding may fall on either
    # side.  Against the path in 64 bits up to 1e-6 of the codes, 2e-6 of the bytes, differ; a hybrid row repeats such a
    # step in the signs of its residual (3e-6 of the bytes).  A cache of a few rows holds none or one of them.
    rate, once = (1e-5, 4) if case["fmt"] in BITS else (1.5e-5, 24) if case["fmt"] != "f12" else (0.0, 0)
    tokens = case["tokens"] if case["kind"] == "write" else int(_lens(case).sum())
    whole = rate + once / max(64, tokens * case["kv_heads"] * _row_bytes(case))
    if case["kind"] == "write":                    # besides codes, norms: float32 sums of squares
        return {"rel": 1e-6, "differ": whole}
    if case["kind"] == "tri":                      # float32 throughout; sums of up to 32k terms
        return {"rel": 5e-6, "differ": 0.0}
    if case["kind"] == "read" and case["fmt"] not in BITS:
        return {"rel": 1e-6}                       # float32 transforms
    if case["dtype"] != "f32":                     # the rounding of the output type: 2.1e-4 and 1.65e-3 of its own
        return {"rel": 8e-4 if case["dtype"] == "f16" else 6.6e-3, "differ": whole}
    if case["kind"] == "read":
        return {"rel": 2e-6}
    # float32 queries and outputs: at head size 128 the decoded values travel as float16 levels (6.7e-5 of 64 bits)
    return {"rel": 2.7e-4 if case["d"] == 128 and case["fmt"] != "tq25" else 5e-6, "differ": whole}


# ---- inputs -------------------------------------------------------------------------------------------------

def _vectors(gen, dtype, *shape):
    """Keys and values as a cache meets them: normal entries, the scale of a vector lognormal."""
    x = torch.randn(shape, device=DEVICE, generator=gen)
    return x.mul_(torch.exp(0.5 * torch.randn(shape[:-1], device=DEVICE, generator=gen)).unsqueeze(-1)).to(dtype)


def _spectral_keys(gen, dtype, tokens, kv_heads, d):
    """Keys whose energy falls over the RoPE pairs, what the spectral cache is made for."""
    std = (torch.arange(d // 2, device=DEVICE) + 1.0) ** -0.75
    x = torch.randn((tokens, kv_heads, d // 2, 2), device=DEVICE, generator=gen)
    return x.mul_(std[:, None]).reshape(tokens, kv_heads, d).to(dtype)


class _Cache:
    """The attributes fused_encode_and_store reads (the package's TQGPUCache without its host-side tier)."""


class _State:
    pass


def _make_cache(case, s, blocks):
    """The compressed cache of one layer, empty: s.k_rows, s.v_rows (and s.k_norms, s.v_norms) plus the quantizer."""
    kvh, bs, d = case["kv_heads"], case["block"], case["d"]
    fmt = KV_CACHE_DTYPES[FORMATS[case["fmt"]]]
    s.uniform = fmt.kind == "uniform"
    if s.uniform:
        s.tq = akv.TurboQuant(head_dim=d, bits=fmt.bits, device=DEVICE, dtype=DTYPES[case["dtype"]])
        packed = s.tq._packed_dim
        s.k_norms = torch.zeros(blocks, bs, kvh, device=DEVICE)
        s.v_norms = torch.zeros(blocks, bs, kvh, device=DEVICE)
    else:
        s.tq = akv.HybridTurboQuant(head_dim=d, mode=fmt.mode, device=DEVICE)
        s.tq.calibrate_uniform(kvh)
        packed = s.tq.packed_dim
        s.k_norms = s.v_norms = None
    s.block = bs
    s.plan = None
    if case["layout"] == "primary":
        s.kv_cache = torch.zeros(blocks, 2, bs, kvh, tq_dim_for_head(d, fmt), dtype=torch.uint8, device=DEVICE)
        s.k_rows, s.v_rows = primary_views(s.kv_cache, d, fmt)
        s.caches = [s.kv_cache]
    else:
        s.k_rows = torch.zeros(blocks, bs, kvh, packed, dtype=torch.uint8, device=DEVICE)
        s.v_rows = torch.zeros_like(s.k_rows)
        s.caches = [s.k_rows, s.v_rows]
        if s.uniform:
            s.plan = _Cache()
            s.plan.tq, s.plan.block_size, s.plan.max_blocks = s.tq, bs, blocks
            s.plan.k_packed, s.plan.v_packed = s.k_rows[None], s.v_rows[None]
            s.plan.k_norms, s.plan.v_norms = s.k_norms[None], s.v_norms[None]
    if s.uniform:
        s.caches += [s.k_norms, s.v_norms]


def _store(s, key, value, slots):
    if s.plan is not None:
        akv.fused_encode_and_store(s.plan, 0, key, value, slots)
    elif s.uniform:
        akv.fused_kv_update_pair(key, value, slots, s.k_rows, s.k_norms, s.v_rows, s.v_norms, s.tq.rotation,
                                 s.tq.boundaries_inner, s.tq.bits, block_size=s.block, prepared=s.tq.prepared_rotation())
    else:
        akv.hybrid_encode_and_store_pair(s.tq, key, value, slots, s.k_rows, s.v_rows, block_size=s.block)


def _tables(case, seed, spare):
    """Context lengths, block tables over a pool in random order, and the slot of each sequence's last token."""
    lens, bs = _lens(case), case["block"]
    need = -(-lens // bs)
    blocks = int(need.sum()) + spare
    order = np.random.default_rng(seed).permutation(blocks)
    tables = np.zeros((len(lens), int(need.max())), dtype=np.int32)
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n]
        at += int(n)
    last = tables[np.arange(len(lens)), need - 1].astype(np.int64) * bs + (lens - 1) % bs
    return (blocks, torch.from_numpy(tables).to(DEVICE), torch.from_numpy(lens.astype(np.int32)).to(DEVICE),
            torch.from_numpy(last).to(DEVICE))


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dt, kvh, d, bs = DTYPES[case["dtype"]], case["kv_heads"], case["d"], case["block"]
    s = _State()
    s.kind = case["kind"]
    if s.kind == "write":
        blocks = -(-case["tokens"] // bs) + 4
        _make_cache(case, s, blocks)
        s.key, s.value = _vectors(gen, dt, case["tokens"], kvh, d), _vectors(gen, dt, case["tokens"], kvh, d)
        # a prompt's tokens fill blocks in order; the blocks lie anywhere
        order = torch.from_numpy(np.random.default_rng(seed).permutation(blocks)).to(DEVICE)
        tok = torch.arange(case["tokens"], device=DEVICE)
        s.slots = order[tok // bs] * bs + tok % bs
        return s
    blocks, s.tables, s.lens, s.last = _tables(case, seed, spare=4)
    if s.kind == "tri":
        s.attn = TriAttention(TriAttentionConfig(head_dim=d, num_freqs=TRI_FREQS, coeff_bits=4, num_kv_heads=kvh,
                                                 num_query_heads=case["heads"], block_size=bs), device=DEVICE)
        s.cache = SpectralKVCache(s.attn.config, max_blocks=blocks, device=DEVICE)
        c = s.cache
        s.caches = [c.k_indices, c.k_packed, c.k_scales, c.v_indices, c.v_packed, c.v_scales]

        def new(n):
            return _spectral_keys(gen, dt, n, kvh, d), torch.randn((n, kvh, d), device=DEVICE, generator=gen).to(dt)
        store = s.cache.encode_and_store
    else:
        _make_cache(case, s, blocks)

        def new(n):
            return _vectors(gen, dt, n, kvh, d), _vectors(gen, dt, n, kvh, d)

        def store(key, value, slots):
            _store(s, key, value, slots)
    chunk = max(bs, (64 << 20) // (kvh * d))
    for t0 in range(0, blocks * bs, chunk):
        slots = torch.arange(t0, min(blocks * bs, t0 + chunk), device=DEVICE)
        store(*new(len(slots)), slots)
    if s.kind == "read":
        if s.uniform:
            s.k_out = torch.zeros(blocks, bs, kvh, d, dtype=dt, device=DEVICE)
            s.v_out = torch.zeros_like(s.k_out)
        else:
            s.k_flat, s.v_flat = s.k_rows[:blocks - 4].contiguous(), s.v_rows[:blocks - 4].contiguous()
        s.blocks = blocks
        return s
    s.key, s.value = new(case["seqs"])
    s.query = torch.randn((case["seqs"], case["heads"], d), device=DEVICE, generator=gen).to(dt)
    if s.kind == "step":
        s.attn = (akv.TQPagedAttention if s.uniform else akv.HybridPagedAttention)(s.tq, case["heads"])
    return s


def run(s):
    if s.kind == "write":
        _store(s, s.key, s.value, s.slots)
        return s.caches
    if s.kind == "read":
        if not s.uniform:
            return [s.tq.decode(s.k_flat), s.tq.decode(s.v_flat)]
        batch_decompress_active_blocks(s.k_rows, s.v_rows, s.k_out, s.v_out, s.tq, s.tq._packed_dim, s.tables, s.blocks,
                                       s.k_norms, s.v_norms)
        return [s.k_out, s.v_out]
    if s.kind == "tri":
        s.cache.encode_and_store(s.key, s.value, s.last)
        return [s.attn.decode_step_paged(s.query, s.cache, s.tables, s.lens)] + s.caches
    _store(s, s.key, s.value, s.last)
    if s.uniform:
        out = s.attn.forward(s.query, s.k_rows, s.k_norms, s.v_rows, s.v_norms, s.tables, s.lens, block_size=s.block)
    else:
        out = s.attn.forward(s.query, s.k_rows, s.v_rows, s.tables, s.lens, block_size=s.block)
    return [out] + s.caches
