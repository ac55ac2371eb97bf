"""Performance cases of the decode engine: the calls a program makes when it
loads, streams or caches tensors through this package.

A case is a dict of plain values. `prepare` makes what a program has in hand
before the call (compressed blobs in HBM, a launch plan, a filled cache, a
container file), `run` is one pass through the public entry points.
"""
import math
import tempfile
from pathlib import Path

import numpy as np
import torch

import bigsmall_amd
from bigsmall_amd.codecs import _refstreams, bf16_chunked, zstd_host
from bigsmall_amd.codecs.kv_cache import compress_kv_entry, decompress_kv_entry
from bigsmall_amd.codecs.zstd_gpu import ZstdLaunch
from bigsmall_amd.device import ChunkBatch, ChunkJob, StatusWord, upload_bytes
from bigsmall_amd.kv_cache_manager import CompressedKVCache

# compressed bytes per raw byte of each kind of values, as the engine's codecs reach it
RATIO = {"normal": 0.663, "student": 0.69, "half_zeros": 0.40, "fp8": 0.84, "kv": 0.67}


def listed():
    return [
        # one transformer layer of a Llama-3-8B-shaped model, decoded in one batched launch: what
        # streaming inference and the model load do for every layer
        {"name": "layer_8b", "kind": "layer", "hidden": 4096, "kv": 1024, "ff": 14336},
        # one key projection alone: a single small matrix fetched on demand (a tensor-by-tensor reader)
        {"name": "tensor_k_proj", "kind": "tensor", "rows": 1024, "cols": 4096, "values": "normal", "coder": "rans"},
        # a half-pruned MLP matrix under the table coder, which is what the encoder picks for it
        {"name": "tensor_pruned", "kind": "tensor", "rows": 4096, "cols": 14336, "values": "half_zeros",
         "coder": "tans"},
        # an fp8 MLP matrix (exponent pairs)
        {"name": "tensor_fp8", "kind": "tensor", "rows": 4096, "cols": 14336, "values": "fp8", "coder": "rans"},
        # attention over a compressed cache that needs a few blocks of one layer: latency
        {"name": "kv_get_few", "kind": "kv_get", "layers": 1, "heads": 8, "dim": 128, "tokens": 8192,
         "block_tokens": 256, "blocks": 4},
        # block-sparse attention over a long cache: 64 blocks in each of 8 layers, one launch
        {"name": "kv_get_many", "kind": "kv_get", "layers": 8, "heads": 8, "dim": 128, "tokens": 32768,
         "block_tokens": 256, "blocks": 64},
        # a prefilled layer's K and V going into the cache as blocks
        {"name": "kv_set_blocks", "kind": "kv_set", "heads": 8, "dim": 128, "tokens": 32768, "block_tokens": 256},
        # a short sequence's whole K/V entry compressed to host bytes and back (the reference's set / get)
        {"name": "kv_entry", "kind": "kv_entry", "heads": 8, "dim": 128, "tokens": 1024},
        # a layer of a container that the reference wrote with its stream-parallel codec
        {"name": "ref_parallel_layer", "kind": "ref", "codec": "bf16_parallel_v1", "hidden": 2048, "kv": 512,
         "ff": 5632},
        # a small layer in the reference's one-chain codec
        {"name": "ref_tans_layer", "kind": "ref", "codec": "bf16_se_tans", "hidden": 512, "kv": 512, "ff": 1408},
        # the norm vectors of an 8B-shaped model as the reference's encoder stores them (lowcard, zstd indices)
        {"name": "zstd_norms", "kind": "norms", "count": 65, "width": 4096, "distinct": 16},
        # a whole container file into HBM: read, host-to-device copy and decode
        {"name": "load_model", "kind": "load", "layers": 4, "hidden": 1024, "ff": 2816, "vocab": 8192},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges."""
    kind = rng.choice(["layer", "tensor", "tensor", "kv_get", "kv_set", "kv_entry", "ref", "ref", "norms", "load"])
    if kind == "layer":
        h = 8 * _log(rng, 64, 512)
        return {"kind": kind, "hidden": h, "kv": max(8, h // rng.choice([1, 2, 4, 8])), "ff": 8 * _log(rng, h // 4, h * 7 // 16)}
    if kind == "tensor":
        n, cols = _log(rng, 1 << 13, 1 << 26), _log(rng, 65, 16384)
        values = rng.choice(["normal", "student", "half_zeros", "fp8"])
        coder = "tans" if values == "half_zeros" else rng.choice(["rans", "rans", "tans"])
        return {"kind": kind, "rows": max(1, n // cols), "cols": cols, "values": values, "coder": coder}
    if kind in ("kv_get", "kv_set", "kv_entry"):
        c = {"kind": kind, "heads": rng.choice([1, 2, 4, 8, 32]), "dim": rng.choice([64, 80, 96, 128])}
        if kind == "kv_entry":
            return dict(c, tokens=_log(rng, 9, 4096))
        bt = rng.choice([64, 128, 256])
        c.update(block_tokens=bt, tokens=bt * _log(rng, 4, max(4, (1 << 25) // (bt * c["heads"] * c["dim"]))))
        if kind == "kv_get":
            c.update(layers=rng.choice([1, 2, 4, 8]), blocks=_log(rng, 1, min(64, c["tokens"] // bt)))
        return c
    if kind == "ref":
        codec = rng.choice(["bf16_parallel_v1", "bf16_parallel_v1", "bf16_se_tans", "bf16_se_single_kernel"])
        h = 8 * (_log(rng, 32, 256) if codec == "bf16_parallel_v1" else _log(rng, 24, 80))
        return {"kind": kind, "codec": codec, "hidden": h, "kv": max(8, h // rng.choice([1, 2, 4])),
                "ff": 8 * _log(rng, h // 4, h * 7 // 16)}
    if kind == "norms":
        return {"kind": kind, "count": _log(rng, 2, 160), "width": _log(rng, 500, 8192), "distinct": rng.randint(3, 16)}
    h = 8 * _log(rng, 32, 128)
    return {"kind": "load", "layers": rng.randint(1, 6), "hidden": h, "ff": 8 * _log(rng, h // 4, h * 3 // 8),
            "vocab": _log(rng, 1000, 16000)}


# ---- inputs (made on the GPU from the seed)

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _values(shape, kind, g):
    """Weights std 0.02 (or fp8 bytes of N(0, 1)) as a device tensor."""
    x = torch.randn(shape, generator=g, device="cuda")
    if kind == "fp8":
        return x.to(torch.float8_e4m3fn).view(torch.uint8)
    if kind == "student":                                  # t with 3 degrees of freedom, scaled to std 0.02
        chi = sum(torch.randn(shape, generator=g, device="cuda").square_() for _ in range(3))
        x = x * torch.rsqrt(chi / 3) / math.sqrt(3)
    elif kind == "half_zeros":
        x = x * (torch.rand(shape, generator=g, device="cuda") >= 0.5)
    return (x * 0.02).to(torch.bfloat16)


def _norm(n, g):
    return (1 + 0.01 * torch.randn(n, generator=g, device="cuda")).to(torch.bfloat16)


def _kv(shape, g):
    """K or V: N(0, 1), each head scaled by a factor of its own."""
    s = 0.5 + 1.5 * torch.rand(shape[0], 1, 1, generator=g, device="cuda")
    return (torch.randn(shape, generator=g, device="cuda") * s).to(torch.bfloat16)


def _matrices(c):
    h, kv, ff = c["hidden"], c["kv"], c["ff"]
    return [(h, h), (kv, h), (kv, h), (h, h), (ff, h), (ff, h), (h, ff)]


def _sources(c, seed):
    """The tensors behind a decode case, in output order."""
    g = _gen(seed)
    kind = c["kind"]
    if kind == "layer":
        return [_values(s, "normal", g) for s in _matrices(c)] + [_norm(c["hidden"], g) for _ in range(2)]
    if kind == "tensor":
        return [_values((c["rows"], c["cols"]), c["values"], g)]
    if kind == "ref":
        return [_values(s, "normal", g) for s in _matrices(c)]
    if kind == "norms":
        out = []
        for _ in range(c["count"]):
            table = torch.randn(c["distinct"], generator=g, device="cuda") * 0.05 + 1
            out.append(table[torch.randint(c["distinct"], (c["width"],), generator=g, device="cuda")].to(torch.bfloat16))
        return out
    if kind == "load":
        h, ff, t = c["hidden"], c["ff"], {}
        t["model.embed_tokens.weight"] = _values((c["vocab"], h), "normal", g)
        for i in range(c["layers"]):
            p = f"model.layers.{i}."
            t[p + "input_layernorm.weight"] = _norm(h, g)
            t[p + "post_attention_layernorm.weight"] = _norm(h, g)
            for n in ("q", "k", "v", "o"):
                t[p + f"self_attn.{n}_proj.weight"] = _values((h, h), "normal", g)
            for n, s in (("gate", (ff, h)), ("up", (ff, h)), ("down", (h, ff))):
                t[p + f"mlp.{n}_proj.weight"] = _values(s, "normal", g)
        t["model.norm.weight"] = _norm(h, g)
        return t
    shape = (c["heads"], c["tokens"], c["dim"])
    return [(_kv(shape, g), _kv(shape, g)) for _ in range(c.get("layers", 1))]


def _requests(c, seed):
    g = _gen(seed + 1)
    n = c["tokens"] // c["block_tokens"]
    return [(i, torch.randperm(n, generator=g, device="cuda")[:c["blocks"]].tolist()) for i in range(c["layers"])]


def _row(width):
    """Elements from one norm vector's output to the next (each starts on a 256-byte boundary)."""
    return (width + 127) // 128 * 128


def _host_words(t):
    t = t.contiguous().cpu()
    return t.view(-1).numpy() if t.dtype == torch.uint8 else t.view(torch.int16).numpy().view(np.uint16).reshape(-1)


def prepare(case, seed):
    c, kind = case, case["kind"]
    src = _sources(c, seed)
    if kind in ("layer", "tensor"):
        jobs, outs, keep = [], [], []
        for t in src:
            w = _host_words(t)
            if c.get("coder") == "tans":
                blob = bf16_chunked.encode_array(w, steps=bf16_chunked.tans_steps(bf16_chunked.DEFAULT_STEPS),
                                                 lanes=bf16_chunked.TANS_LANES, coder=bf16_chunked.CODER_TANS)
            else:
                blob = bf16_chunked.encode_array(w)
            d, o, inf = upload_bytes(blob, t.device), torch.empty_like(t), bf16_chunked.info(blob)
            jobs.append(ChunkJob(d.data_ptr(), len(blob), o.data_ptr(), w.size, inf.n_chunks, inf.plane_mode))
            outs.append(o)
            keep.append(d)
        dev = src[0].device
        return {"kind": kind, "launch": ChunkBatch(jobs, dev), "status": StatusWord(dev), "outs": outs, "keep": keep}
    if kind == "ref":
        dev, items, outs, keep = src[0].device, [], [], []
        for t in src:
            w = _host_words(t)
            blob = _refstreams.encode_host(c["codec"], w)
            d, o = upload_bytes(blob, dev), torch.empty_like(t)
            items.append((_refstreams.PARSERS[c["codec"]](blob, w.size), d.data_ptr(), o.data_ptr()))
            outs.append(o)
            keep.append(d)
        # a tensor of fewer elements than the batched path takes gets a launch of its own, as in a group decode
        big = [i for i in items if _refstreams.serial_ok(i[0])]
        small = [(_refstreams.RefLaunch(p, b, dev), o) for p, b, o in items if not _refstreams.serial_ok(p)]
        return {"kind": kind, "batch": _refstreams.RefBatch(big, dev) if big else None, "small": small,
                "status": StatusWord(dev), "outs": outs, "keep": keep}
    if kind == "norms":
        dev = src[0].device
        z, keep = ZstdLaunch(dev), []
        out = torch.zeros(len(src), _row(c["width"]), dtype=torch.bfloat16, device=dev)
        for t, o in zip(src, out):
            blob, _ = zstd_host.encode_lowcard(_host_words(t).tobytes(), 2)
            d = upload_bytes(blob, dev)
            z.add_lowcard(d.data_ptr(), blob, o.data_ptr(), t.numel(), 2)
            keep.append(d)
        z.prepare()
        return {"kind": kind, "launch": z, "status": StatusWord(dev), "outs": [out], "keep": keep}
    if kind == "load":
        tmp = tempfile.TemporaryDirectory()
        path = Path(tmp.name) / "model.bs"
        bigsmall_amd.compress({k: v.cpu() for k, v in src.items()}, path)
        return {"kind": kind, "path": path, "tmp": tmp}
    if kind == "kv_entry":
        return {"kind": kind, "k": src[0][0], "v": src[0][1]}
    cache = CompressedKVCache(device="cuda")
    if kind == "kv_set":
        k, v = src[0]
        pool = torch.zeros(4 * k.numel() + 2048 * (c["tokens"] // c["block_tokens"]), dtype=torch.uint8, device=k.device)
        return {"kind": kind, "cache": cache, "k": k, "v": v, "block_tokens": c["block_tokens"], "pool": pool}
    for i, (k, v) in enumerate(src):
        cache.set_blocks(i, k, v, block_tokens=c["block_tokens"])
    return {"kind": kind, "cache": cache, "requests": _requests(c, seed)}


def run(state):
    kind = state["kind"]
    if kind in ("layer", "tensor", "norms"):
        state["launch"].launch(state["status"])
        return state["outs"] + [state["status"].t]
    if kind == "ref":
        stream = torch.cuda.current_stream().cuda_stream
        if state["batch"] is not None:
            state["batch"].launch(state["status"].ptr, stream)
        for launch, out_ptr in state["small"]:
            launch.launch(out_ptr, state["status"].ptr, stream)
        return state["outs"] + [state["status"].t]
    if kind == "load":
        return bigsmall_amd.load(state["path"], device="cuda", progress=False)
    if kind == "kv_entry":
        entry = compress_kv_entry(state["k"], state["v"])
        k, v = decompress_kv_entry(entry, device="cuda")
        return [len(entry), k, v]
    if kind == "kv_set":
        cache = state["cache"]
        blocks = cache.set_blocks(0, state["k"], state["v"], block_tokens=state["block_tokens"])
        arena = cache._blocks[0].arena                     # every blob, back to back: into the program's own pool
        state["pool"][:arena.numel()].copy_(arena)
        return [blocks, cache.memory_usage(), state["pool"]]
    return [t for kv in state["cache"].get_blocks_multi(state["requests"]) for t in kv]


# ---- what a pass cannot do without: compressed bytes and decoded bytes, each once (no matrix products)

def work(case):
    c, kind = case, case["kind"]
    if kind == "layer":
        n = 2 * (sum(a * b for a, b in _matrices(c)) + 2 * c["hidden"])
        return {"bytes": n * (1 + RATIO["normal"]), "flops": 0}
    if kind == "tensor":
        n = c["rows"] * c["cols"] * (1 if c["values"] == "fp8" else 2)
        return {"bytes": n * (1 + RATIO[c["values"]]), "flops": 0}
    if kind == "ref":
        return {"bytes": 2 * sum(a * b for a, b in _matrices(c)) * (1 + RATIO["normal"]), "flops": 0}
    if kind == "norms":                                    # about half a byte of indices, two of output per element
        return {"bytes": c["count"] * c["width"] * 2.5, "flops": 0}
    if kind == "load":                                     # file bytes read, copied to the GPU and decoded
        h, ff = c["hidden"], c["ff"]
        n = 2 * (c["vocab"] * h + c["layers"] * (4 * h * h + 3 * h * ff + 2 * h) + h)
        return {"bytes": n * (1 + RATIO["normal"]), "flops": 0}
    per_token = 2 * 2 * c["heads"] * c["dim"]              # K and V
    if kind == "kv_get":
        return {"bytes": c["layers"] * c["blocks"] * c["block_tokens"] * per_token * (1 + RATIO["kv"]), "flops": 0}
    both = 2 if kind == "kv_entry" else 1                  # compressed and decompressed again
    return {"bytes": both * c["tokens"] * per_token * (1 + RATIO["kv"]), "flops": 0}


def tolerance(case):
    """Lossless codecs: every output is the same bits."""
    return "exact"


def exact(case, seed):
    """The tensors that the blobs were made of; None for compressed bytes."""
    c, kind = case, case["kind"]
    if kind == "kv_set":
        return None
    src = _sources(c, seed)
    if kind == "norms":
        src = [torch.nn.functional.pad(torch.stack(src), (0, _row(c["width"]) - c["width"]))]
    if kind in ("layer", "tensor", "ref", "norms"):
        return src + [torch.zeros(1, dtype=torch.int32)]   # and a clean status word
    if kind == "load":
        return src
    if kind == "kv_entry":
        return [None, src[0][0], src[0][1]]
    out, bt = [], c["block_tokens"]
    for (i, ids), (k, v) in zip(_requests(c, seed), src):
        for t in (k, v):
            out.append(t.view(c["heads"], -1, bt, c["dim"]).transpose(0, 1)[ids].contiguous())
    return out
