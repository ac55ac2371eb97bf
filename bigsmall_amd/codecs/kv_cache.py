"""KV-cache entry codec (mirrors bigsmall/codecs/kv_cache.py:41-117).

Entry layout, as in the reference (little-endian), K then V:
    [u8 version] then per tensor: [u8 ndim][i32 x ndim shape][u32 blob_len][blob]
Versions: 1 = bf16_se_ac blobs, 2 = bf16_se_rans blobs (both constriction
bitstreams, not decodable by this engine: BigSmallVersionError), 3 = this
engine's bf16_chunked_v1 blobs, decoded on the GPU.

Element count per tensor uses max(1, dim) like the reference (kv_cache.py:109-111).
"""
from __future__ import annotations

import struct

import numpy as np

from ..exceptions import BigSmallVersionError
from . import bf16_chunked

VERSION_GPU = 3
KV_STEPS = 256          # BSCK steps for KV blobs: a 256-token block of 8x128 heads is 8 chunks


def _tensor_words(t) -> tuple[np.ndarray, list[int]]:
    import torch
    if t.dtype != torch.bfloat16:
        raise ValueError(f"compress_kv_entry expects BF16 tensors, got {t.dtype}")
    return t.detach().contiguous().cpu().view(torch.int16).numpy().view(np.uint16).reshape(-1), list(t.shape)


def encode_words(words: np.ndarray, steps: int = KV_STEPS) -> bytes:
    return bf16_chunked.encode_array(words, steps=steps) if words.size else b""


def compress_kv_entry(keys, values) -> bytes:
    """Compress one K/V pair into a version-3 entry. Device tensors are encoded
    on the GPU and only the compressed bytes come back to the host; host
    tensors use the host encoder (the reference copies to the host and encodes
    there, kv_cache.py:28-38)."""
    import torch
    from ..device import pinned_bytes
    if keys.dtype != torch.bfloat16 or values.dtype != torch.bfloat16:
        raise ValueError("compress_kv_entry requires BF16 keys and values")
    if keys.is_cuda and values.is_cuda and keys.numel() and values.numel():
        # only the blobs come back (the encoder's arena holds a worst case for
        # each), through pinned memory
        arena, spans = bf16_chunked.encode_device([keys, values], steps=KV_STEPS, compact=False)
        host = pinned_bytes(sum(n for _, n in spans))
        blobs, pos = [], 0
        for o, n in spans:
            host[pos:pos + n].copy_(arena[o:o + n], non_blocking=True)
            blobs.append(memoryview(host.numpy()[pos:pos + n]))
            pos += n
        torch.cuda.current_stream(arena.device).synchronize()
    else:
        blobs = [encode_words(_tensor_words(t)[0]) for t in (keys, values)]
    parts = [struct.pack("<B", VERSION_GPU)]
    for t, blob in zip((keys, values), blobs):
        shape = list(t.shape)
        parts += [struct.pack(f"<B{len(shape)}iI", len(shape), *(int(s) for s in shape), len(blob)), blob]
    return b"".join(parts)


def parse_kv_entry(data: bytes) -> list[tuple[list[int], int, int, int]]:
    """[(shape, n_elements, blob_offset, blob_len)] for K and V of an entry."""
    if not data:
        raise ValueError("empty KV entry")
    version = data[0]
    if version in (1, 2):
        from .. import __version__
        raise BigSmallVersionError(required="newer-than-installed", installed=__version__,
                                   detail=f"KV entry version {version} is constriction-coded; this engine "
                                          f"decodes version {VERSION_GPU}")
    if version != VERSION_GPU:
        raise ValueError(f"Unknown KV cache codec version {version}")
    pos, out = 1, []
    for _ in range(2):
        ndim = data[pos]
        pos += 1
        shape = list(struct.unpack_from(f"<{ndim}i", data, pos))
        pos += 4 * ndim
        blen, = struct.unpack_from("<I", data, pos)
        pos += 4
        if pos + blen > len(data):
            raise ValueError("KV entry truncated")
        n = 1
        for s in shape:
            n *= max(1, s)
        out.append((shape, n, pos, blen))
        pos += blen
    return out


def decompress_kv_entry(data: bytes, device: str = "cuda"):
    """Inverse of compress_kv_entry: (keys, values) as bf16 tensors on `device`."""
    import torch
    from ..device import TASK_DTYPE, chunk_tasks, decode_chunk_tasks, pinned_bytes, require_gpu
    parts = parse_kv_entry(data)
    dev = require_gpu(device if str(device) != "cpu" else None)
    # one pinned buffer and one copy: status word, task table (its own 256 bytes), K's and V's blobs
    pos = 512
    assert 256 + 2 * TASK_DTYPE.itemsize <= pos
    total = pos + sum((b + 255) & ~255 for _, _, _, b in parts)
    d = torch.empty(total, dtype=torch.uint8, device=dev)
    buf = pinned_bytes(total).numpy()
    outs, rows = [], []
    for shape, n, off, blen in parts:
        o = torch.empty(shape if all(s > 0 for s in shape) else [n], dtype=torch.bfloat16, device=dev)
        outs.append(o)
        if blen:
            inf = bf16_chunked.info(bytes(data[off:off + 32]))
            if inf.n != n:
                raise ValueError(f"KV entry: blob holds {inf.n} elements, shape needs {n}")
            buf[pos:pos + blen] = np.frombuffer(data, np.uint8, blen, off)
            rows.append((d.data_ptr() + pos, blen, o.data_ptr(), n, inf.n_chunks, inf.plane_mode))
        pos += (blen + 255) & ~255
    if rows:
        tasks, groups, max_mode = chunk_tasks(rows)
        decode_chunk_tasks(buf, d, tasks, groups, max_mode, torch.cuda.current_stream(dev), "KV entry")
    k, v = outs
    if str(device) == "cpu":
        return k.cpu(), v.cpu()
    return k, v
