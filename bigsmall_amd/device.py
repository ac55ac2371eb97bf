"""Device plumbing for the decode engine: streams, uploads, status words and
batched BSCK launches. torch provides device memory and streams; all decoding
happens in the HIP kernels of libbigsmall_hip.so.
"""
from __future__ import annotations

import contextlib

import ctypes
from dataclasses import dataclass

import numpy as np

from . import _native
from .exceptions import DecodeError

# bs_chunk_task (include/bigsmall_hip.h): 40 bytes, 8-byte aligned
TASK_DTYPE = np.dtype([("blob", "<u8"), ("blob_bytes", "<u8"), ("out", "<u8"), ("n", "<u8"),
                       ("wg_begin", "<u4"), ("n_chunks", "<u4")])
assert TASK_DTYPE.itemsize == 40


def require_gpu(device=None):
    """Return a torch.device for decoding; raise if no ROCm GPU is present."""
    import torch
    if not torch.cuda.is_available():
        raise RuntimeError("bigsmall_amd decodes on an AMD GPU (MI355X); no ROCm device is available")
    dev = torch.device(device if device is not None else "cuda")
    if dev.type != "cuda":
        raise ValueError(f"decode device must be a ROCm GPU, got {dev}")
    if dev.index is None:
        dev = torch.device("cuda", torch.cuda.current_device())
    return dev


def stream_ptr(stream=None, device=None) -> int:
    import torch
    s = stream if stream is not None else torch.cuda.current_stream(device)
    return int(s.cuda_stream)


def upload_bytes(data, device, align: int = 256):
    """Copy host bytes to a fresh device uint8 tensor (allocator blocks are
    >= 256-byte aligned)."""
    import torch
    arr = np.frombuffer(data, np.uint8) if not isinstance(data, np.ndarray) else data.view(np.uint8).reshape(-1)
    host = torch.from_numpy(arr.copy() if not arr.flags.writeable else arr)
    out = torch.empty(len(arr), dtype=torch.uint8, device=device)
    if len(arr):
        out.copy_(host)
    assert out.data_ptr() % align == 0
    return out


# Smallest pinned allocation: torch keeps a pool per power of two, and the first request of
# each pins a new block (MI355X, get_blocks_multi of 4 and 20 blocks, first call after one
# of 1 block: 690 and 480 us against 135 and 160), so all small tables share one pool.
PINNED_MIN = 1 << 16


def pinned_bytes(n: int):
    """A pinned host uint8 tensor of n bytes (on the host whatever torch's default device is)."""
    import torch
    t = torch.empty(max(n, PINNED_MIN), dtype=torch.uint8, device="cpu", pin_memory=True)
    return t if n >= PINNED_MIN else t[:n]


def upload_bytes_async(data, device, stream=None):
    """upload_bytes through pinned staging with a non-blocking copy on
    `stream` (the current stream if None): the host does not wait for the
    copy, or for the work queued before it; later work on that stream sees the
    bytes. The staging block comes from torch's pinned caching allocator,
    which keeps it from reuse until the copy has run."""
    import torch
    arr = np.frombuffer(data, np.uint8) if not isinstance(data, np.ndarray) else data.view(np.uint8).reshape(-1)
    out = torch.empty(len(arr), dtype=torch.uint8, device=device)
    if len(arr):
        host = pinned_bytes(len(arr))
        host.numpy()[:] = arr
        with torch.cuda.stream(stream) if stream is not None else contextlib.nullcontext():
            out.copy_(host, non_blocking=True)
        if stream is not None:
            out.record_stream(stream)
    return out


class StatusWord:
    """Device int32 that kernels OR their BS_DEV_* bits into."""

    def __init__(self, device=None, view=None):
        """A new zeroed word on `device`, or `view`: an int32 element of
        another device buffer that is already zero."""
        import torch
        self.t = view if view is not None else torch.zeros(1, dtype=torch.int32, device=device)

    @property
    def ptr(self) -> int:
        return self.t.data_ptr()

    def reset(self):
        self.t.zero_()

    def check(self, what: str = "decode") -> None:
        v = int(self.t.item())
        if v:
            names = [n for b, n in [(_native.BS_DEV_ERR_HEADER, "bad header"), (_native.BS_DEV_ERR_COUNT, "count mismatch"),
                                    (_native.BS_DEV_ERR_BOUNDS, "section out of bounds"),
                                    (_native.BS_DEV_ERR_STREAM, "corrupt entropy-coded stream")] if v & b]
            raise DecodeError(f"{what}: device integrity check failed ({', '.join(names)}; status=0x{v:x})")


@dataclass
class ChunkJob:
    """One BSCK blob to decode: device blob address/length, output address, counts."""
    blob_ptr: int
    blob_bytes: int
    out_ptr: int
    n: int
    n_chunks: int
    plane_mode: int = 2


def inspect_chunk_header(blob_head: bytes):
    """Parse a BSCK header. A malformed or truncated header is a data error:
    ValueError, as the reference raises for bad magic or counts
    (bigsmall/codecs/bf16_parallel.py:153-163)."""
    info = _native.BsChunkInfo()
    if len(blob_head) < 32:
        raise ValueError(f"bf16_chunked: blob too short for its header ({len(blob_head)} bytes)")
    buf = (ctypes.c_uint8 * len(blob_head)).from_buffer_copy(blob_head)
    rc = _native.lib().bs_chunk_inspect(ctypes.addressof(buf), len(blob_head), ctypes.byref(info))
    if rc == _native.BS_ERR_FORMAT:
        raise ValueError("bf16_chunked: malformed blob header")
    _native.check(rc, "bs_chunk_inspect")
    return info


def chunk_tasks(rows) -> tuple[np.ndarray, int, int]:
    """The bs_chunk_task array of one batched launch, its workgroup count and
    its highest plane mode. rows: {blob, bytes, output, elements, chunks, plane
    mode} of each task, as a list of tuples (0.5 us a row) or as the rows of an
    int64 array (15 us in all)."""
    per = _native.lib().bs_chunk_chunks_per_group()
    if isinstance(rows, list):
        tasks, groups, low = [], 0, 0
        for blob, nbytes, out, n, n_chunks, _ in rows:
            tasks.append((blob, nbytes, out, n, groups, n_chunks))
            groups += (n_chunks + per - 1) // per
            low |= blob | out
        tasks, max_mode = np.array(tasks, TASK_DTYPE), max((r[5] for r in rows), default=0)
    else:
        tasks = np.empty(len(rows), TASK_DTYPE)
        tasks.view(np.int64).reshape(-1, 5)[:, :4] = rows[:, :4]
        tasks["n_chunks"] = rows[:, 4]
        ends = (rows[:, 4] + (per - 1)) // per
        np.cumsum(ends, out=ends)
        tasks["wg_begin"][0] = 0
        tasks["wg_begin"][1:] = ends[:-1]
        groups, max_mode = int(ends[-1]), int(rows[:, 5].max())
        low = int(np.bitwise_or.reduce(rows[:, 0] | rows[:, 2]))
    if low % 16:
        raise ValueError("BSCK blobs and their outputs must be 16-byte aligned on the device")
    return tasks, groups, max_mode


def decode_chunk_tasks(buf: np.ndarray, d_buf, tasks: np.ndarray, groups: int, max_mode: int, stream, what: str) -> None:
    """Decode `tasks` (chunk_tasks) and wait for it; raises DecodeError on a bad
    status. buf is pinned host memory and d_buf a device buffer of its size:
    the status word at 0, the task table at 256, and from there on whatever the
    caller placed in it (blobs); one copy on `stream` (a torch stream) brings
    all of it over, and one copy back brings the status."""
    import torch
    buf[:256] = 0
    buf[256:256 + tasks.nbytes] = tasks.view(np.uint8)
    own = stream == torch.cuda.current_stream()       # (of the current device)
    with contextlib.nullcontext() if own else torch.cuda.stream(stream):
        d_buf.copy_(torch.from_numpy(buf), non_blocking=True)
        if not own:
            d_buf.record_stream(stream)
        st = StatusWord(view=d_buf[:4].view(torch.int32))
        rc = _native.lib().bs_chunk_decode_batch(d_buf.data_ptr() + 256, len(tasks), groups, max_mode, st.ptr,
                                                 stream_ptr(stream))
        _native.check(rc, "bs_chunk_decode_batch")
        st.check(what)                    # a copy on `stream`: waits for the decode


class ChunkBatch:
    """A prepared batched launch: a device array of bs_chunk_task and its grid
    size. Reusable: launch() may be called repeatedly (e.g. for timing)."""

    def __init__(self, jobs: list[ChunkJob], device):
        import torch
        L = _native.lib()
        per = L.bs_chunk_chunks_per_group()
        tasks = np.zeros(len(jobs), TASK_DTYPE)
        wg = 0
        for i, j in enumerate(jobs):
            if j.blob_ptr % 16 or j.out_ptr % 16:
                raise ValueError("BSCK blobs and their outputs must be 16-byte aligned on the device")
            tasks[i] = (j.blob_ptr, j.blob_bytes, j.out_ptr, j.n, wg, j.n_chunks)
            wg += (j.n_chunks + per - 1) // per
        self.n_tasks = len(jobs)
        self.max_mode = max((j.plane_mode for j in jobs), default=0)
        self.total_groups = wg
        self.jobs = jobs
        self.tasks_dev = torch.from_numpy(tasks.view(np.uint8).copy()).to(device)

    def launch(self, status: StatusWord, stream=None) -> None:
        if self.n_tasks == 0:
            return
        rc = _native.lib().bs_chunk_decode_batch(self.tasks_dev.data_ptr(), self.n_tasks, self.total_groups,
                                                 self.max_mode, status.ptr, stream_ptr(stream))
        _native.check(rc, "bs_chunk_decode_batch")
