"""Decode of the cache blocks a batch touches into a float16 / bfloat16 / float32 block buffer:
the job of TurboQuantImpl._batch_decompress_active_blocks (aither_kvcache/vllm/backend.py:
1040-1091), which the reference's prefill and non-fused decode paths run before dense attention.

The reference gathers the unique active blocks, decodes them as one flat batch and scatters the
result back.  Here the block table goes to the kernel as it is: every listed block inside the
cache is decoded from where it lies to where it belongs, K and V in one launch where their layouts
agree, with no intermediate tensors.  A block that several sequences share is decoded once per
listing, to the same values (once per run of equal neighbours, such as a table's padding).
"""
import torch

from .. import _lib


def _check(cache, norms, buf, tq, block_ids, num_blocks):
    dev = _lib.require_gpu(cache, norms, buf, block_ids)
    if cache.dtype != torch.uint8 or norms.dtype != torch.float32:
        raise TypeError("cache must be uint8 and norms float32")
    if cache.dim() != 4 or norms.dim() != 3 or buf.dim() != 4:
        raise ValueError("expected cache [B, bs, H, bytes], norms [B, bs, H], buf [B, bs, H, d]")
    if cache.stride(3) != 1 or buf.stride(3) != 1:
        raise ValueError("last dimension of cache and buf must be contiguous")
    if tuple(cache.shape[:3]) != tuple(norms.shape) or tuple(buf.shape[:3]) != tuple(norms.shape):
        raise ValueError("cache, norms and buf disagree on [blocks, block_size, kv_heads]")
    if buf.shape[3] != tq.head_dim or cache.shape[3] < tq._packed_dim:
        raise ValueError("row sizes do not match the quantizer")
    if num_blocks > cache.shape[0]:
        raise ValueError("num_blocks exceeds the cache")
    return dev


def _flat_ids(block_ids):
    ids = block_ids.reshape(-1)
    if ids.dtype not in (torch.int32, torch.int64):
        ids = ids.to(torch.int64)
    return ids if ids.is_contiguous() else ids.contiguous()


def decode_blocks(cache: torch.Tensor, norms: torch.Tensor, buf: torch.Tensor, tq,
                  block_ids: torch.Tensor, num_blocks: int) -> None:
    """cache uint8 [blocks, block_size, kv_heads, >= packed_dim], norms float32 [blocks, block_size,
    kv_heads], buf [blocks, block_size, kv_heads, head_dim]; block_ids any integer tensor (flattened
    here); ids outside [0, num_blocks) are skipped."""
    dev = _check(cache, norms, buf, tq, block_ids, num_blocks)
    ids = _flat_ids(block_ids)
    if ids.numel() == 0 or num_blocks == 0:
        return
    _lib.check(_lib.lib().akv_decode_blocks(
        cache.data_ptr(), cache.stride(0), cache.stride(1), cache.stride(2),
        norms.data_ptr(), norms.stride(0), norms.stride(1), norms.stride(2),
        ids.data_ptr(), _lib.itype_code(ids), ids.numel(), num_blocks,
        cache.shape[1], cache.shape[2], tq.head_dim,
        tq.prepared_rotation().ptr, tq.centroids.data_ptr(), tq.bits,
        buf.data_ptr(), _lib.dtype_code(buf), buf.stride(0), buf.stride(1), buf.stride(2),
        _lib.stream_ptr(dev)))


def _span(t):
    """First and last byte address a tensor reaches."""
    size = t.element_size()
    return t.data_ptr(), t.data_ptr() + (sum((n - 1) * s for n, s in zip(t.shape, t.stride())) + 1) * size


def batch_decompress_active_blocks(key_cache, value_cache, k_buf, v_buf, tq, packed_dim, block_table,
                                   num_blocks, k_norms, v_norms) -> None:
    """Argument order of the reference method (backend.py:1040-1043); the per-layer norm tensors,
    which the reference reads from class state (:1073-1075), are passed in."""
    if packed_dim != tq._packed_dim:
        raise ValueError(f"packed_dim {packed_dim} does not match the quantizer ({tq._packed_dim})")
    if block_table.is_cuda and tq.rotation.is_cuda:
        rc = _lib.calls().decode_blocks(key_cache, value_cache, k_buf, v_buf, block_table, k_norms, v_norms, tq.centroids,
                                        tq.prepared_rotation().ptr, num_blocks, tq.head_dim, tq._packed_dim, tq.bits)
        if rc is not None:
            return _lib.check(rc)
    # one launch for both where the layouts agree and V's output does not lie within reach of K's
    if (key_cache.shape == value_cache.shape and key_cache.stride() == value_cache.stride()
            and k_norms.stride() == v_norms.stride() and k_buf.shape == v_buf.shape
            and k_buf.stride() == v_buf.stride() and k_buf.dtype == v_buf.dtype and k_buf.numel() > 0
            and (_span(k_buf)[1] <= _span(v_buf)[0] or _span(v_buf)[1] <= _span(k_buf)[0])):
        dev = _check(key_cache, k_norms, k_buf, tq, block_table, num_blocks)
        if _check(value_cache, v_norms, v_buf, tq, block_table, num_blocks) != dev:
            raise ValueError("K and V lie on different devices")
        ids = _flat_ids(block_table)
        if ids.numel() == 0 or num_blocks == 0:
            return
        _lib.check(_lib.lib().akv_decode_blocks_kv(
            key_cache.data_ptr(), value_cache.data_ptr(), key_cache.stride(0), key_cache.stride(1), key_cache.stride(2),
            k_norms.data_ptr(), v_norms.data_ptr(), k_norms.stride(0), k_norms.stride(1), k_norms.stride(2),
            ids.data_ptr(), _lib.itype_code(ids), ids.numel(), num_blocks,
            key_cache.shape[1], key_cache.shape[2], tq.head_dim,
            tq.prepared_rotation().ptr, tq.centroids.data_ptr(), tq.bits,
            k_buf.data_ptr(), v_buf.data_ptr(), _lib.dtype_code(k_buf), k_buf.stride(0), k_buf.stride(1), k_buf.stride(2),
            _lib.stream_ptr(dev)))
        return
    decode_blocks(key_cache, k_norms, k_buf, tq, block_table, num_blocks)
    decode_blocks(value_cache, v_norms, v_buf, tq, block_table, num_blocks)
