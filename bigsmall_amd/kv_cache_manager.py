"""Compressed KV-cache manager (mirrors bigsmall/kv_cache_manager.py:22-91).

Whole-entry API, as in the reference: set(layer_idx, keys, values),
get(layer_idx) -> (keys, values), has, memory_usage, raw_size,
compression_ratio, clear, len, repr. Entries are version-3 (bf16_chunked_v1)
and decode on the GPU.

Block API (the reference keys one blob per layer and has no blocks; this adds
them for on-the-fly attention over a long cache):
    set_blocks(layer_idx, keys, values, block_tokens=256, token_dim=-2)
        splits K and V along the token dimension into blocks, encodes every
        block (on the GPU when K and V are device tensors, else with the host
        encoder) and keeps the compressed blocks resident in HBM, one arena
        per layer;
    get_blocks(layer_idx, block_ids) -> (K, V) with shape [len(block_ids), *block_shape]
    get_blocks_multi([(layer_idx, block_ids), ...]) -> [(K, V), ...]
        decode every requested block of every request in ONE batched kernel
        launch straight into the output tensors.
"""
from __future__ import annotations

from typing import Optional

import numpy as np

from .codecs import bf16_chunked
from .codecs import kv_cache as _kv_codec


def _block_major(blocked, td: int):
    """blocked.movedim(td, 0).contiguous(): the block index first, every block
    contiguous. Copied as 8-byte words when the innermost dimension allows it
    (the same bytes in a quarter of the elements)."""
    import torch
    if (blocked.is_contiguous() and blocked.element_size() == 2 and blocked.shape[-1] % 4 == 0
            and blocked.storage_offset() % 4 == 0 and blocked.data_ptr() % 8 == 0):
        return blocked.view(torch.int64).movedim(td, 0).contiguous().view(blocked.dtype)
    return blocked.movedim(td, 0).contiguous()


class _LayerBlocks:
    """Compressed blocks of one layer: one device arena (uint8), and per block
    of K and V {offset, nbytes, n_chunks, plane_mode} as the rows of an array."""

    def __init__(self, block_shape: list, block_elems: int, arena, k_blocks=(), v_blocks=()):
        self.block_shape, self.block_elems, self.arena = block_shape, block_elems, arena
        self.k = np.asarray(k_blocks, np.int64).reshape(-1, 4)
        self.v = np.asarray(v_blocks, np.int64).reshape(-1, 4)

    @property
    def k_blocks(self) -> list:
        return [tuple(r) for r in self.k.tolist()]

    @property
    def v_blocks(self) -> list:
        return [tuple(r) for r in self.v.tolist()]


def _block_outputs(n_blocks: int, L, dev):
    """K and V outputs [n_blocks] + block_shape. The decoder writes each block
    at a 16-byte aligned address, so when a block is not a multiple of 8
    elements the blocks sit in a buffer with a padded stride (a strided view)."""
    import torch
    stride = (L.block_elems + 7) // 8 * 8
    if stride == L.block_elems:
        k = torch.empty([n_blocks] + L.block_shape, dtype=torch.bfloat16, device=dev)
        return k, torch.empty_like(k)
    inner = [int(np.prod(L.block_shape[d + 1:])) for d in range(len(L.block_shape))]
    outs = []
    for _ in range(2):
        buf = torch.empty(max(n_blocks, 1) * stride, dtype=torch.bfloat16, device=dev)
        outs.append(buf.as_strided([n_blocks] + L.block_shape, [stride] + inner))
    return outs[0], outs[1]


# Requested blocks of a layer from which its task rows are made with array operations (a
# dozen of them, whatever the count) and not one by one. MI355X, get_blocks_multi of 32
# layers, us a call, one by one / arrays: 1 block of each 244 / 475, 4 352 / 505, 8 519 / 567,
# 12 707 / 648, 16 843 / 686.
FEW_BLOCKS = 10


def _block_rows(rows: list, L: _LayerBlocks, ids: list, k, v) -> None:
    """Append {blob, bytes, output, elements, chunks, plane mode} of each block,
    K and V in turn, to rows. Only the requested rows of the layer's tables are
    read: a list of its every block would cost more than the request."""
    base, step, outp = L.arena.data_ptr(), 2 * k.stride(0), (k.data_ptr(), v.data_ptr())
    for j, bi in enumerate(ids):
        for blocks, out in zip((L.k, L.v), outp):
            off, nbytes, n_chunks, mode = blocks[bi].tolist()
            rows.append((base + off, nbytes, out + j * step, L.block_elems, n_chunks, mode))


def _block_rows_array(L: _LayerBlocks, ids: list, k, v) -> np.ndarray:
    """The same rows as an array, K's before V's."""
    n = len(ids)
    rows, at = np.empty((2, n, 6), np.int64), np.arange(n, dtype=np.int64) * (2 * k.stride(0))
    for r, blocks, out in zip(rows, (L.k, L.v), (k, v)):
        b = blocks[ids]
        np.add(b[:, 0], L.arena.data_ptr(), out=r[:, 0])
        r[:, 1] = b[:, 1]
        np.add(at, out.data_ptr(), out=r[:, 2])
        r[:, 3] = L.block_elems
        r[:, 4:] = b[:, 2:]
    return rows.reshape(-1, 6)


class CompressedKVCache:
    """Compressed KV storage. device: where get()/get_blocks() materialise tensors."""

    def __init__(self, device: str = "cuda"):
        self.device = device
        self._compressed: dict = {}
        self._raw_size_bytes = 0
        self._blocks: dict = {}
        self._block_raw = 0

    # ---- whole-entry API (reference semantics) ------------------------------
    def set(self, layer_idx, keys, values) -> None:
        import torch
        if keys.dtype != torch.bfloat16 or values.dtype != torch.bfloat16:
            raise ValueError("CompressedKVCache.set: keys and values must be BF16")
        raw = keys.element_size() * keys.numel() + values.element_size() * values.numel()
        self._compressed[layer_idx] = _kv_codec.compress_kv_entry(keys, values)
        self._raw_size_bytes += raw

    def get(self, layer_idx):
        if layer_idx not in self._compressed:
            raise KeyError(f"layer {layer_idx} not in CompressedKVCache")
        return _kv_codec.decompress_kv_entry(self._compressed[layer_idx], device=self.device)

    def has(self, layer_idx) -> bool:
        return layer_idx in self._compressed

    def memory_usage(self) -> int:
        blocks = sum(int(L.k[:, 1].sum()) + int(L.v[:, 1].sum()) for L in self._blocks.values())
        return sum(len(b) for b in self._compressed.values()) + blocks

    def raw_size(self) -> int:
        return self._raw_size_bytes + self._block_raw

    def compression_ratio(self) -> Optional[float]:
        raw = self.raw_size()
        return None if raw == 0 else self.memory_usage() / raw

    def clear(self) -> None:
        self._compressed.clear()
        self._blocks.clear()
        self._raw_size_bytes = self._block_raw = 0

    def __len__(self) -> int:
        # a layer stored through both set() and set_blocks() counts once
        return len(set(self._compressed) | set(self._blocks))

    def __repr__(self) -> str:
        cr = self.compression_ratio()
        return (f"CompressedKVCache(layers={len(self)} compressed={self.memory_usage() / 1e6:.2f}MB "
                f"raw={self.raw_size() / 1e6:.2f}MB ratio={f'{cr * 100:.2f}%' if cr is not None else 'n/a'})")

    # ---- block API ----------------------------------------------------------
    def set_blocks(self, layer_idx, keys, values, block_tokens: int = 256, token_dim: int = -2,
                   threads: Optional[int] = None) -> int:
        """Compress K and V of a layer in blocks of `block_tokens` tokens; returns the block count."""
        import torch
        from .device import require_gpu, upload_bytes
        if keys.dtype != torch.bfloat16 or values.dtype != torch.bfloat16 or keys.shape != values.shape:
            raise ValueError("set_blocks: keys and values must be BF16 tensors of one shape")
        td = token_dim % keys.dim()
        T = keys.shape[td]
        if T % block_tokens:
            raise ValueError(f"set_blocks: {T} tokens is not a multiple of block_tokens={block_tokens}")
        nb = T // block_tokens
        if layer_idx in self._blocks:          # replacing a layer: drop its raw size from the totals
            old = self._blocks.pop(layer_idx)
            self._block_raw -= 2 * 2 * old.block_elems * len(old.k)
        block_shape = list(keys.shape)
        block_shape[td] = block_tokens
        block_elems = int(np.prod(block_shape))
        if keys.is_cuda and values.is_cuda:
            # encode on the GPU: the blocks never leave HBM
            groups = []
            for t in (keys, values):
                shape = list(t.shape)
                pre, post = int(np.prod(shape[:td])), int(np.prod(shape[td + 1:]))
                seg_len = block_tokens * post
                if t.is_contiguous() and t.data_ptr() % 4 == 0 and seg_len % 512 == 0 and (T * post) % 8 == 0:
                    # read in place: block b is `pre` segments of block_tokens * post
                    # words, T * post words apart ([blocks, segments, seg_len])
                    groups.append(t.detach().view(pre, nb, seg_len).permute(1, 0, 2))
                else:
                    blocked = t.detach().reshape(shape[:td] + [nb, block_tokens] + shape[td + 1:])
                    groups.append(_block_major(blocked, td).reshape(nb, block_elems))
            if block_elems % 2 == 0:
                arena, offs, lens = bf16_chunked.encode_device_rows(groups, steps=_kv_codec.KV_STEPS)
            else:       # odd blocks are not 4-byte aligned rows: one task per block view
                arena, spans = bf16_chunked.encode_device([g[i] for g in groups for i in range(nb)],
                                                          steps=_kv_codec.KV_STEPS)
                offs, lens = np.array([o for o, _ in spans], np.int64), np.array([n for _, n in spans], np.int64)
            per = bf16_chunked.GPU_ENCODE_LANES * _kv_codec.KV_STEPS
            nch = (block_elems + per - 1) // per
            ent = np.empty((2 * nb, 4), np.int64)
            ent[:, 0], ent[:, 1], ent[:, 2], ent[:, 3] = offs, lens, nch, bf16_chunked.MODE_DENSE
            self._blocks[layer_idx] = _LayerBlocks(block_shape, block_elems, arena, ent[:nb], ent[nb:])
            self._block_raw += 2 * keys.numel() * 2
            return nb
        blobs = {"k": [], "v": []}
        for which, t in (("k", keys), ("v", values)):
            # [..., T, ...] -> [nb, ..., block_tokens, ...] contiguous blocks
            shape = list(t.shape)
            blocked = t.detach().cpu().reshape(shape[:td] + [nb, block_tokens] + shape[td + 1:])
            blocked = blocked.movedim(td, 0).contiguous()
            words = blocked.view(torch.int16).numpy().view(np.uint16).reshape(nb, -1)
            blobs[which] = [_kv_codec.encode_words(words[i]) for i in range(nb)]
        sizes = [(len(b) + 255) & ~255 for b in blobs["k"] + blobs["v"]]
        arena_host = np.zeros(sum(sizes) + 256, np.uint8)
        entries = {"k": [], "v": []}
        pos = 0
        for which in ("k", "v"):
            for b in blobs[which]:
                arena_host[pos:pos + len(b)] = np.frombuffer(b, np.uint8)
                inf = bf16_chunked.info(b[:32])
                entries[which].append((pos, len(b), inf.n_chunks, inf.plane_mode))
                pos += (len(b) + 255) & ~255
        arena = upload_bytes(arena_host, require_gpu(self.device))
        self._blocks[layer_idx] = _LayerBlocks(block_shape, block_elems, arena, entries["k"], entries["v"])
        self._block_raw += 2 * keys.numel() * 2
        return nb

    def block_count(self, layer_idx) -> int:
        return len(self._blocks[layer_idx].k)

    def _block_ids(self, L: _LayerBlocks, layer_idx, block_ids) -> list[int]:
        """Block ids as ints, each in [0, block count): a negative id is an
        error, not a block counted from the end."""
        ids = [int(i) for i in block_ids]
        n = len(L.k)
        for bi in ids:
            if not 0 <= bi < n:
                raise IndexError(f"layer {layer_idx!r}: block {bi} out of range (layer has {n} blocks)")
        return ids

    def get_blocks(self, layer_idx, block_ids):
        return self.get_blocks_multi([(layer_idx, block_ids)])[0]

    def get_blocks_multi(self, requests, stream=None):
        """Decode the blocks of every (layer_idx, block_ids) request in one
        launch, whose task table goes up with the status word in one copy."""
        import torch
        from .device import chunk_tasks, decode_chunk_tasks, pinned_bytes, require_gpu
        dev = require_gpu(self.device)
        few, many, results = [], [], []
        for layer_idx, block_ids in requests:
            L = self._blocks[layer_idx]
            ids = self._block_ids(L, layer_idx, block_ids)
            k, v = _block_outputs(len(ids), L, dev)
            results.append((k, v))
            if len(ids) < FEW_BLOCKS:
                _block_rows(few, L, ids, k, v)
            else:
                many.append(_block_rows_array(L, ids, k, v))
        if few or many:
            if many:
                many.append(np.array(few, np.int64).reshape(-1, 6))
            tasks, groups, max_mode = chunk_tasks(np.concatenate(many) if many else few)
            s = stream if stream is not None else torch.cuda.current_stream(dev)
            if stream is not None:        # the outputs' memory and the arenas are the current stream's
                if not isinstance(s, torch.cuda.Stream):        # any object with a cuda_stream handle
                    s = torch.cuda.ExternalStream(int(s.cuda_stream), device=dev)
                s.wait_stream(torch.cuda.current_stream(dev))
            nbytes = 256 + tasks.nbytes
            decode_chunk_tasks(pinned_bytes(nbytes).numpy(), torch.empty(nbytes, dtype=torch.uint8, device=dev), tasks, groups,
                               max_mode, s, "KV blocks")
        return [(k.contiguous(), v.contiguous()) for k, v in results]

    def prepare_blocks_multi(self, requests):
        """Allocate outputs and build the batched launch for `requests` once;
        returns (launch, outputs) where launch(status, stream) decodes again.
        Outputs are strided views when a block is not a multiple of 8 elements."""
        import torch
        from .device import ChunkBatch, ChunkJob, require_gpu
        dev = require_gpu(self.device)
        rows, results = [], []
        for layer_idx, block_ids in requests:
            L = self._blocks[layer_idx]
            ids = self._block_ids(L, layer_idx, block_ids)
            k, v = _block_outputs(len(ids), L, dev)
            _block_rows(rows, L, ids, k, v)
            results.append((k, v))
        return ChunkBatch([ChunkJob(*r) for r in rows], dev), results
