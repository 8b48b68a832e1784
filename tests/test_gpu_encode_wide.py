"""The matrix-core encode kernel of head_dim 64 and 256 at the edges of a step and of the grid, against the oracle."""
import numpy as np
import pytest
import torch

import aitherkvcache_amd as akv
from oracle import tq_oracle as O
from tests.util import kv_like, code_mismatch_report, MAX_ULPS

pytestmark = pytest.mark.gpu


def max_ulps(d):
    """A code may differ where its float64 value lies this many float32 units from a boundary: 16 at head_dim 128 (the bar of the
    other codec tests); sums of twice as many terms, in the kernel and in the oracle alike, may drift twice as far."""
    return MAX_ULPS * max(1, d // 128)


def check_rows(packed, norms, x, R, bits, d):
    _, b, _ = O.get_codebook(d, bits)
    ref_p, ref_n = O.encode(x, R, b, bits)
    x64 = x.astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        unit = x64 / (np.linalg.norm(x64, axis=-1, keepdims=True) + 1e-10)
    n, ulps, hist = code_mismatch_report(O._UNPACK[bits](packed, d), O._UNPACK[bits](ref_p, d), O.rotate_unit_f64(x, R), b, O, unit, R)
    assert ulps <= max_ulps(d), hist
    assert n <= max(3, packed.size * 8 // bits * 2e-5), (n, hist)
    assert np.allclose(norms, ref_n, rtol=1e-6, atol=0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,bits", [(64, 4), (64, 3), (64, 2), (256, 4), (256, 3), (256, 2)])
def test_encode_steps_vs_oracle(dev, d, bits, dtype):
    """One tensor and two in a launch; fewer rows than a step, a step and its neighbours, more steps than workgroups; 1 and 3 heads; skipped, out-of-range and int32 slots; rows behind
    reserved bytes; a zero row, a NaN row and an infinite one."""
    rng = np.random.default_rng(d + bits)
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev))
    R, P, bs = tq.rotation.cpu().numpy(), tq._packed_dim, 16
    for tokens, heads in ((1, 1), (5, 3), (16, 1), (17, 1), (65, 3), (700, 3)) + (((9000, 3),) if bits == 4 else ()):
        blocks = tokens // bs + 3
        slots = rng.permutation(blocks * bs)[:tokens].astype(np.int64)
        slots[5::7] = -1
        slots[6::11] = blocks * bs + 3
        ok = (slots >= 0) & (slots < blocks * bs)
        st = torch.from_numpy(slots).to(dev).to(torch.int32 if tokens == 65 else torch.int64)
        xs = []
        for k in range(2):
            x = kv_like(rng, (tokens, heads, d)).astype(np.float32)
            if tokens > 60:
                x[2, 0] = 0.0
                x[3, 0, 7] = np.nan
                x[4, heads - 1, d - 1] = -np.inf
            xs.append(torch.from_numpy(x).to(dev).to(dtype))
        rows = [torch.full((blocks, bs, heads, P + 4), 0xA5, dtype=torch.uint8, device=dev) for _ in xs]
        norms = [torch.full((blocks, bs, heads), -5.0, device=dev) for _ in xs]
        print(f"[encode wide] d={d} bits={bits} {dtype} tokens={tokens} heads={heads}", flush=True)
        akv.fused_kv_update_pair(xs[0], xs[1], st, rows[0][..., :P], norms[0], rows[1][..., :P], norms[1], tq.rotation,
                                 tq.boundaries_inner, bits, bs)
        one = torch.full_like(rows[0], 0xA5)
        one_n = torch.full_like(norms[0], -5.0)
        akv.fused_kv_update(xs[0], st, one[..., :P], one_n, tq.rotation, tq.boundaries_inner, bits, bs)
        assert torch.equal(one, rows[0]) and torch.equal(one_n.nan_to_num(7.0, 8.0), norms[0].nan_to_num(7.0, 8.0))
        flat_p, flat_n = tq.encode(xs[1])
        where = slots[ok]
        for x, r, n in zip(xs, rows, norms):
            r, n, host = r.cpu().numpy(), n.cpu().numpy(), x.float().cpu().numpy()
            assert np.all(r[..., P:] == 0xA5) and int(np.sum(n != -5.0)) == int(ok.sum()) * heads     # nothing else was written
            got, gn = r[where // bs, where % bs][..., :P].reshape(-1, P), n[where // bs, where % bs].reshape(-1)
            src = host[ok].reshape(-1, d)
            fin = np.isfinite(src).all(-1)
            assert np.all(got[~fin] == 0xFF) and not np.isfinite(gn[~fin]).any()       # last level everywhere
            check_rows(got[fin], gn[fin], src[fin], R, bits, d)
        assert np.array_equal(flat_p.cpu().numpy()[ok].reshape(-1, P), got)


@pytest.mark.parametrize("d", [64, 256])
@pytest.mark.parametrize("dtype,scale", [(torch.float32, 1e-36), (torch.float32, 1e-22), (torch.float32, 3e18), (torch.float32, 1e30),
                                         (torch.bfloat16, 1e-36), (torch.bfloat16, 1e30), (torch.float16, 1e-3)])
def test_rows_of_any_magnitude(dev, d, dtype, scale):
    """Rows float16 cannot hold, and rows whose elements span far more than float16 does: the codes are those of float64 away
    from a boundary.  Squares that under- or overflow float32 give norm 0 or inf as they do in the oracle's arithmetic."""
    rng = np.random.default_rng(d)
    x = kv_like(rng, (64, d)).astype(np.float32)
    x[:, ::7] *= np.float32(1e-6)
    xt = (torch.from_numpy(x).double() * scale).to(dtype).to(dev)
    tq = akv.TurboQuant(head_dim=d, bits=4, device=str(dev))
    packed, norms = tq.encode(xt)
    host = xt.double().cpu().numpy()
    with np.errstate(over="ignore", under="ignore"):
        n32 = np.sqrt((host.astype(np.float32) ** 2).sum(-1, dtype=np.float32)).astype(np.float64)
    big = ~np.isfinite(n32)
    unit = host / np.where(big, 1.0, n32 + 1e-10)[:, None]
    y = np.where(big[:, None], 0.0, unit @ tq.rotation.double().cpu().numpy().T)
    b = tq.boundaries_inner.double().cpu().numpy()
    codes = O._UNPACK[4](packed.cpu().numpy(), d)
    # 16 float32 units of the row's largest value: what the sums of the rotation may drift
    clear = np.abs(y[..., None] - b).min(-1) > 16 * 2.0 ** -23 * np.maximum(np.abs(y).max(-1, keepdims=True), 1e-30)
    clear &= ~big[:, None]
    assert np.array_equal(codes[clear], np.searchsorted(b, y)[clear])
    assert np.all(codes[big] == np.searchsorted(b, 0.0))
    got = norms.double().cpu().numpy()
    assert np.array_equal(np.isinf(got), big) and np.allclose(got[~big], n32[~big], rtol=1e-6, atol=0 if scale > 1e-20 else 1e-22)


@pytest.mark.parametrize("factor", [3000.0, 1e-4, 2.0 ** 100])
@pytest.mark.parametrize("d,bits,dtype", [(64, 4, torch.float16), (64, 3, torch.float32), (256, 4, torch.bfloat16), (256, 2, torch.float32)])
def test_matrices_that_are_no_rotation(dev, d, bits, dtype, factor):
    """A matrix given with the call may have entries far outside what two float16 terms hold: it is scaled by its largest."""
    rng = np.random.default_rng(d)
    tq = akv.TurboQuant(head_dim=d, bits=bits, device=str(dev))
    R, b = tq.rotation * factor, tq.boundaries_inner * factor
    x = torch.from_numpy(kv_like(rng, (500, 2, d)).astype(np.float32)).to(dev).to(dtype)
    packed, norms = torch.zeros(32, 16, 2, tq._packed_dim, dtype=torch.uint8, device=dev), torch.zeros(32, 16, 2, device=dev)
    akv.fused_kv_update(x, torch.arange(500, device=dev), packed, norms, R, b, bits, 16)
    x64 = x.double().cpu().numpy().reshape(-1, d)
    y = x64 / np.linalg.norm(x64, axis=-1, keepdims=True) @ R.double().cpu().numpy().T
    ref = np.searchsorted(b.double().cpu().numpy(), y)
    got = O._UNPACK[bits](packed.cpu().numpy().reshape(-1, tq._packed_dim)[:1000], d)
    assert np.count_nonzero(got != ref) <= max(3, ref.size * 2e-5)      # (values that lie on a boundary to within float32)
    assert np.allclose(norms.cpu().numpy().reshape(-1)[:1000], np.linalg.norm(x64, axis=-1), rtol=1e-6)


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_shared_coordinates_and_boundaries_in_any_order(dev, bits, dtype):
    """head_dim 256: calls of few rows share a row's coordinates out over workgroups, others do not -- the same bytes and norms.
    The boundaries are counted, whatever their order; one that is NaN counts for no value."""
    tq = akv.TurboQuant(head_dim=256, bits=bits, device=str(dev))
    gen = torch.Generator(device=dev).manual_seed(bits)
    x = torch.randn(5000, 256, device=dev, generator=gen)
    x[7], x[8, 100], x[9, 3] = 0.0, float("nan"), float("inf")
    x = x.to(dtype)
    p, n = tq.encode(x)
    for rows in (1, 15, 16, 17, 1025, 3071, 3072, 3073):
        ps, ns = tq.encode(x[:rows])
        assert torch.equal(ps, p[:rows]) and torch.equal(ns.view(torch.int32), n[:rows].view(torch.int32)), rows
    slots = torch.arange(3000, device=dev)

    def paged(boundaries, m):
        packed, norms = torch.zeros(3000, 1, 1, tq._packed_dim, dtype=torch.uint8, device=dev), torch.zeros(3000, 1, 1, device=dev)
        akv.fused_kv_update(x[:m, None], slots[:m], packed, norms, tq.rotation, boundaries, bits, block_size=1)
        return packed[:m, 0, 0]
    b = tq.boundaries_inner
    for m in (20, 3000):
        assert torch.equal(paged(b.flip(0).contiguous(), m), p[:m])
        hole, top = b.clone(), b.clone()
        hole[b.numel() // 2], top[b.numel() // 2] = float("nan"), float("inf")
        finite = torch.isfinite(x[:m].float()).all(-1)              # (a NaN value lies past every boundary, infinite or not)
        assert torch.equal(paged(hole, m)[finite], paged(top.sort().values, m)[finite])
