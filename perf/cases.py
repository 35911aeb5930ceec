"""Performance cases of the paged KV write and gather.

Each case is one pass of work that a serving program gives this library,
through its public entry points: the PyTorch op
(``_C_cache_ops.reshape_and_cache_flash_kvx``, case["entry"] == "op"), the
torch helpers (``paged.write_kv`` / ``paged.gather_kv``, "paged"), or the C
entry points with descriptors that an engine builds once per layer and keeps
("abi", as ``bench.py`` and ``kvx_bench`` call them).

The cases cover the real range of the path: decode writes of a few to a few
hundred tokens, chunked prefill writes that start inside blocks, gathers of
short, ordinary, skewed and long batches; the NHD, HND, x-packed and vLLM
cache layouts; blocks of 8 to 256 tokens; PACKED, RAGGED and KV_OFFSETS
tables; F16, BF16 and F32 payloads, FP8 E4M3 / E5M2 caches with per-tensor
and per-head scales; int32 and int64 indices; the row shapes that the tests
and the benchmark use.
"""
from __future__ import annotations

import ctypes as C
import random

import torch

from kvx_amd import abi, paged, torch_ops
from kvx_amd.abi import Layout, ScaleGranularity, Status

_DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32,
          "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2}
_BYTES = {"f16": 2, "bf16": 2, "f32": 4, "e4m3": 1, "e5m2": 1}
_FP8_MAX = {"e4m3": 448.0, "e5m2": 57344.0}
_INDEX = {"s32": torch.int32, "s64": torch.int64}
_DEVICE = "cuda:0"


def _write(name, entry, layout, block, heads, dim, io, cache, seqs, lo, hi, **more):
    """A write of `seqs` sequences, lo..hi new tokens each (1: decode)."""
    case = {"name": name, "op": "write", "entry": entry, "layout": layout, "block": block,
            "heads": heads, "dim": dim, "io": io, "cache": cache, "seqs": seqs, "lo": lo,
            "hi": hi, "spread": "uniform", "lens_seed": 1, "inside": True, "padded": 0,
            "pool_blocks_per_seq": 1, "layers": 1, "scales": "tensor", "index": "s64"}
    case.update(more)
    return case


def _gather(name, entry, layout, table, block, heads, dim, io, cache, seqs, lo, hi, **more):
    """A gather of `seqs` sequences of lo..hi tokens into [seqs, width, H, D]."""
    case = {"name": name, "op": "gather", "entry": entry, "layout": layout, "table": table,
            "block": block, "heads": heads, "dim": dim, "io": io, "cache": cache, "seqs": seqs,
            "lo": lo, "hi": hi, "spread": "uniform", "lens_seed": 1, "width": 0,
            "scales": "tensor", "index": "s32"}
    case.update(more)
    return case


def listed():
    return [
        # The smallest call: the decode write of a batch of four in one
        # layer, from a vLLM-style engine.  Launch latency is all of it.
        _write("decode_write_4", "op", "nhd", 16, 8, 128, "bf16", "bf16", 4, 1, 1,
               pool_blocks_per_seq=64),
        # One decode step of Llama-3-8B shape over eight layers, 256
        # sequences with 5% padding, from an engine that keeps a descriptor
        # per layer.
        _write("decode_write_256_8_layers", "abi", "nhd", 16, 8, 128, "bf16", "bf16", 256, 1, 1,
               padded=13, pool_blocks_per_seq=8, layers=8),
        # A decode write into vLLM's paged-attention pair (x-packed K, V with
        # the token axis innermost), an odd batch.
        _write("decode_write_vllm_201", "paged", "vllm", 16, 8, 128, "f16", "f16", 201, 1, 1,
               pool_blocks_per_seq=16),
        # The benchmark's chunked prefill: 16 chunks of 2048 tokens, x-packed
        # K, row-major V.
        _write("prefill_write_packed_k", "abi", "packed_k", 16, 8, 128, "bf16", "bf16", 16, 2048,
               2048, inside=False, pool_blocks_per_seq=512),
        # Ragged prefill chunks that continue inside blocks, quantized to an
        # E4M3 cache with per-tensor scales.
        _write("prefill_write_fp8", "paged", "nhd", 16, 8, 128, "bf16", "e4m3", 8, 700, 2300,
               lens_seed=2),
        # The same into x-packed K and V in blocks of 128 tokens.
        _write("prefill_write_packed_b128", "paged", "packed", 128, 8, 128, "bf16", "bf16", 6,
               500, 1800, lens_seed=3),
        # The smallest gather: TinyLlama rows, eight short sequences.
        _gather("gather_short", "paged", "nhd", "packed", 16, 4, 64, "f16", "f16", 8, 100, 128,
                width=128),
        # Full-context decode gather, Llama-3-8B rows, U[512, 8192] tokens.
        _gather("gather_decode_64", "abi", "nhd", "packed", 16, 8, 128, "bf16", "bf16", 64, 512,
                8192, width=8192),
        # The same from an E4M3 cache, dequantized to bf16.
        _gather("gather_fp8_32", "abi", "nhd", "packed", 16, 8, 128, "bf16", "e4m3", 32, 512,
                8192, width=8192, lens_seed=2),
        # MLA rows (one latent of 576 elements) through a RAGGED table: many
        # short and a few long sequences.
        _gather("gather_ragged_mla", "paged", "nhd", "ragged", 64, 1, 576, "bf16", "bf16", 96,
                64, 16384, spread="skewed", lens_seed=3),
        # Long contexts in TensorRT-LLM's pools: KV_OFFSETS, HND blocks.
        _gather("gather_offsets_long", "abi", "hnd", "offsets", 32, 8, 128, "f16", "f16", 4,
                12000, 32768, lens_seed=4),
        # vLLM's pair with an FP8 cache in 32-token blocks, skewed lengths.
        _gather("gather_vllm_fp8", "paged", "vllm", "packed", 32, 8, 128, "bf16", "e4m3", 48, 100,
                8192, spread="skewed", lens_seed=5),
    ]


_ROWS = [(8, 128), (8, 128), (8, 128), (4, 64), (1, 128), (2, 128), (16, 64), (6, 128), (3, 128),
         (8, 96), (8, 80), (1, 576), (8, 256)]
_BLOCKS = [16, 16, 16, 32, 32, 64, 128, 256, 8]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case of the ranges above."""
    heads, dim = rng.choice(_ROWS)
    block = rng.choice(_BLOCKS)
    io = rng.choice(["bf16", "bf16", "f16", "f32"])
    cache = rng.choice([io, io, "e4m3", "e5m2"])
    scales = rng.choice(["tensor", "tensor", "head"])
    index = rng.choice(["s32", "s64"])
    common = {"scales": scales, "index": index, "lens_seed": rng.randrange(1 << 30)}
    row = heads * dim * (_BYTES[io] + _BYTES[cache]) * 2  # bytes of one token
    if rng.random() < 0.5:
        layout = rng.choice(["nhd", "nhd", "hnd", "packed", "packed_k", "vllm"])
        entries = ["paged", "abi"] + (["op"] if layout == "nhd" and scales == "tensor" else [])
        if rng.random() < 0.4:  # decode
            seqs = _log_uniform(rng, 1, 512)
            case = _write("", rng.choice(entries), layout, block, heads, dim, io, cache, seqs, 1,
                          1, padded=seqs // 20, pool_blocks_per_seq=4, **common)
        else:  # prefill chunks
            tokens = min(_log_uniform(rng, 64, 32768), (256 << 20) // row)
            seqs = max(1, min(_log_uniform(rng, 1, 32), tokens // 16))
            hi = max(2, 2 * tokens // seqs * 2 // 3)
            case = _write("", rng.choice(entries), layout, block, heads, dim, io, cache, seqs,
                          max(1, hi // 2), hi, inside=rng.random() < 0.7, **common)
    else:
        table = rng.choice(["packed", "packed", "ragged", "offsets"])
        layout = rng.choice(["nhd", "nhd", "hnd", "packed"]
                            + (["vllm"] if table != "offsets" else []))
        spread = rng.choice(["uniform", "skewed"])
        tokens = min(_log_uniform(rng, 128, 131072), (512 << 20) // row)
        seqs = max(1, min(_log_uniform(rng, 1, 128), tokens // 32))
        hi = min(32768, max(16, 2 * tokens // seqs))
        lo = max(1, hi // 16 if spread == "uniform" else hi // 64)
        case = _gather("", rng.choice(["paged", "abi"]), layout, table, block, heads, dim, io,
                       cache, seqs, lo, hi, spread=spread, **common)
    del case["name"]
    return case


# ---------------------------------------------------------------------------
# Sequences of a case: they depend on the case alone, the data on the seed.

def _lens(case):
    rng = random.Random(case["lens_seed"])
    lo, hi = case["lo"], case["hi"]
    if case["spread"] == "skewed":
        return [min(hi, _log_uniform(rng, lo, hi)) for _ in range(case["seqs"])]
    return [rng.randint(lo, hi) for _ in range(case["seqs"])]


def _starts(case, lens):
    """First position of each written sequence's new tokens."""
    rng = random.Random(case["lens_seed"] + 1)
    if not case["inside"]:
        return [0] * len(lens)
    return [rng.randrange(4 * case["block"]) for _ in lens]


def _width(case, lens):
    return case["width"] or max(lens)


def work(case):
    row = 2 * case["heads"] * case["dim"] * (_BYTES[case["io"]] + _BYTES[case["cache"]])
    index = 4 if case["index"] == "s32" else 8
    lens = _lens(case)
    if case["op"] == "write":
        total = (sum(lens) - case["padded"]) * row + sum(lens) * index
        return {"bytes": case["layers"] * total, "flops": 0}
    blocks = sum((n + case["block"] - 1) // case["block"] for n in lens)
    entries = {"packed": blocks * index, "ragged": sum(lens) * index + (len(lens) + 1) * 4,
               "offsets": blocks * 8}[case["table"]]
    return {"bytes": sum(lens) * row + entries + len(lens) * index, "flops": 0}


def tolerance(case):
    # Copies, and casts whose rounding is defined bit for bit.
    return "exact"


# ---------------------------------------------------------------------------
# Data.

def _generator(seed):
    return torch.Generator(device=_DEVICE).manual_seed(seed)


def _pack(case):
    return 16 // _BYTES[case["cache"]]


def _alloc(case, blocks):
    dt, bs, h, d = _DTYPE[case["cache"]], case["block"], case["heads"], case["dim"]
    x = _pack(case)
    layout = case["layout"]
    if layout == "vllm":  # [nb, H, D / x, bs, x] and [nb, H, D, bs]
        return paged.alloc_custom_cache(blocks, bs, h, d, dt, _DEVICE, "bhpox", "bhdo", x)
    k, v = {"nhd": (Layout.BLOCK_NHD, Layout.BLOCK_NHD),
            "hnd": (Layout.BLOCK_HND, Layout.BLOCK_HND),
            "packed": (Layout.BLOCK_HND_PACKED, Layout.BLOCK_HND_PACKED),
            "packed_k": (Layout.BLOCK_HND_PACKED, Layout.BLOCK_NHD)}[layout]
    return paged.alloc_cache(blocks, bs, h, d, dt, _DEVICE, k, v, x)


def _storage(t):
    """The dense storage of a cache tensor, whose axes a view may permute."""
    order = sorted(range(t.dim()), key=lambda i: -t.stride(i))
    return t.permute(order)


def _tables(case, lens, rng_seed, per_seq=None):
    """Random block ids: [S, width in blocks] int64 on the CPU (-1 unused),
    and the pool's blocks."""
    need = [(n + case["block"] - 1) // case["block"] for n in lens]
    used = sum(need)
    pool = max(used + used // 4 + 8, (per_seq or 0) * len(lens))
    ids = torch.randperm(pool, generator=torch.Generator().manual_seed(rng_seed))[:used]
    table = torch.full((len(lens), max(need)), -1, dtype=torch.int64)
    mask = torch.arange(max(need))[None] < torch.tensor(need)[:, None]
    table[mask] = ids
    return table, pool


def _scales(case, gen):
    """K and V scales as a calibration gives them (amax of N(0, 2) / largest
    code), and the torch values that multiply [..., H, D]."""
    if case["cache"] == case["io"]:
        return None, None, None, None
    top = _FP8_MAX[case["cache"]]
    cal = torch.randn((2, 128, case["heads"], case["dim"]), generator=gen, device=_DEVICE) * 2
    if case["scales"] == "head":
        v = (cal.abs().amax(dim=(1, 3)) / top).float()
        ks, vs = v[0].contiguous(), v[1].contiguous()
        return (paged.Scales(ks, ScaleGranularity.PER_HEAD),
                paged.Scales(vs, ScaleGranularity.PER_HEAD), ks[:, None], vs[:, None])
    v = (cal.abs().amax(dim=(1, 2, 3)) / top).float()
    ks, vs = v[0].reshape(1), v[1].reshape(1)
    return ks, vs, ks, vs


def _check(status):
    if status != Status.OK:
        raise RuntimeError(f"kvx status {status}")


def _write_data(case, seed):
    gen = _generator(seed)
    dev = torch.device(_DEVICE)
    lens = _lens(case)
    starts = _starts(case, lens)
    table, pool = _tables(case, [s + n for s, n in zip(starts, lens)], seed,
                          case["pool_blocks_per_seq"])
    lens_t = torch.tensor(lens)
    total = int(lens_t.sum())
    seq = torch.repeat_interleave(torch.arange(len(lens)), lens_t)
    first = torch.cumsum(lens_t, 0) - lens_t
    pos = torch.arange(total) - first[seq] + torch.tensor(starts)[seq]
    bs = case["block"]
    slots = table[seq, pos // bs] * bs + pos % bs
    if case["padded"]:
        pad = torch.randperm(total, generator=torch.Generator().manual_seed(case["lens_seed"]))
        slots[pad[: case["padded"]]] = -1
    slots = slots.to(dev, _INDEX[case["index"]])
    ks, vs, ksv, vsv = _scales(case, gen)
    sigma = 2.0 if case["cache"] != case["io"] else 1.0
    layers = []
    for _ in range(case["layers"]):
        cache = _alloc(case, pool)
        cache.key_cache.zero_()
        cache.value_cache.zero_()
        shape = (total, case["heads"], case["dim"])
        key = torch.randn(shape, generator=gen, device=dev) * sigma
        value = torch.randn(shape, generator=gen, device=dev) * sigma
        layers.append((cache, key.to(_DTYPE[case["io"]]), value.to(_DTYPE[case["io"]])))
    return layers, slots, (ks, vs), (ksv, vsv)


def _fill(t, case, gen):
    """Cached rows ~ N(0, 1), or FP8 codes of N(0, 2) rows at their scale."""
    flat = _storage(t).reshape(-1)
    top = _FP8_MAX.get(case["cache"])
    for part in flat.split(1 << 26):
        x = torch.empty(part.shape, device=t.device, dtype=torch.float32)
        x.normal_(generator=gen)
        if top is not None:
            x.mul_(top / 4.5).clamp_(-top, top)
        part.copy_(x)


def _gather_data(case, seed):
    gen = _generator(seed)
    dev = torch.device(_DEVICE)
    lens = _lens(case)
    table, blocks = _tables(case, lens, seed)
    idx = _INDEX[case["index"]]
    if case["table"] == "offsets":
        layout = {"nhd": Layout.BLOCK_NHD, "hnd": Layout.BLOCK_HND,
                  "packed": Layout.BLOCK_HND_PACKED}[case["layout"]]
        cache, kv = paged.alloc_block_pool(blocks, case["block"], case["heads"], case["dim"],
                                           _DTYPE[case["cache"]], _DEVICE, layout, _pack(case))
        _fill(cache.key_cache, case, gen)
        pair = torch.stack([2 * table, 2 * table + 1], dim=1)[:, None]
        pair[(table < 0)[:, None, None].expand_as(pair)] = 0x7FFFFFFF
        tb = paged.pool_table(cache, pair.to(dev, torch.int32))
    else:
        cache = kv = _alloc(case, blocks)
        _fill(cache.key_cache, case, gen)
        _fill(cache.value_cache, case, gen)
        if case["table"] == "ragged":
            lens_t = torch.tensor(lens)
            seq = torch.repeat_interleave(torch.arange(len(lens)), lens_t)
            first = torch.cumsum(lens_t, 0) - lens_t
            pos = torch.arange(int(lens_t.sum())) - first[seq]
            indptr = torch.cat([torch.zeros(1, dtype=torch.int64), torch.cumsum(lens_t, 0)])
            tb = paged.RaggedTable(table[seq, pos // case["block"]].to(dev, idx),
                                   indptr.to(dev, torch.int32))
        else:
            tb = table.to(dev, idx)
    ks, vs, ksv, vsv = _scales(case, gen)
    width = _width(case, lens)
    out = [torch.zeros((len(lens), width, case["heads"], case["dim"]), dtype=_DTYPE[case["io"]],
                       device=dev) for _ in range(2)]
    lens_d = torch.tensor(lens, dtype=idx, device=dev)
    return cache, kv, tb, table, lens_d, width, out, (ks, vs), (ksv, vsv)


def prepare(case, seed):
    if case["op"] == "write":
        layers, slots, scales, _ = _write_data(case, seed)
        state = {"case": case, "layers": layers, "slots": slots, "scales": scales}
        if case["entry"] == "op":
            torch_ops.load()
            one = torch.ones(1, dtype=torch.float32, device=_DEVICE)
            state["op_scales"] = tuple(one if s is None else s for s in scales)
            state["op_dtype"] = ("auto" if case["cache"] == case["io"]
                                 else {"e4m3": "fp8", "e5m2": "fp8_e5m2"}[case["cache"]])
        elif case["entry"] == "abi":
            state["lib"] = abi.load()
            state["calls"] = [(cache.desc(), paged.build_write(cache, key, value, slots, *scales))
                              for cache, key, value in layers]
        return state
    cache, _, tb, _, lens, width, out, scales, _ = _gather_data(case, seed)
    state = {"case": case, "cache": cache, "table": tb, "lens": lens, "width": width, "out": out,
             "scales": scales}
    if case["entry"] == "abi":
        state["lib"] = abi.load()
        state["call"] = (paged.gather_cache_desc(cache, tb),
                         paged.build_gather(out[0], out[1], tb, lens, width))
        if scales[0] is not None:
            state["scale_descs"] = tuple(paged.scale_desc_of(s) for s in scales)
    return state


def run(state):
    case = state["case"]
    if case["op"] == "write":
        return _run_write(state, case["entry"])
    return _run_gather(state, case["entry"])


def _run_write(state, entry):
    ks, vs = state["scales"]
    out = []
    if entry == "abi":
        stream = torch.cuda.current_stream().cuda_stream
        write = state["lib"].kvx_launch_write_kv
        for cd, wd in state["calls"]:
            _check(write(C.byref(cd), C.byref(wd), stream))
    for cache, key, value in state["layers"]:
        if entry == "op":
            torch_ops.reshape_and_cache_flash_kvx(key, value, cache.key_cache, cache.value_cache,
                                                  state["slots"], state["op_dtype"],
                                                  *state["op_scales"])
        elif entry == "paged":
            _check(paged.write_kv(cache, key, value, state["slots"], k_scale=ks, v_scale=vs))
        out += [cache.key_cache, cache.value_cache]
    return out


def _run_gather(state, entry):
    ks, vs = state["scales"]
    ko, vo = state["out"]
    if entry == "abi":
        stream = torch.cuda.current_stream().cuda_stream
        lib = state["lib"]
        cd, gd = state["call"]
        if ks is not None:
            ksd, vsd = state["scale_descs"]
            _check(lib.kvx_launch_gather_kv_dequant(C.byref(cd), C.byref(gd), C.byref(ksd),
                                                    C.byref(vsd), stream))
        else:
            _check(lib.kvx_launch_gather_kv(C.byref(cd), C.byref(gd), stream))
    else:
        _check(paged.gather_kv(state["cache"], ko, vo, state["table"], state["lens"],
                               state["width"], k_scale=ks, v_scale=vs))
    return [ko, vo]


# ---------------------------------------------------------------------------
# The casts in 64 bits.  Copies have no computed numbers.

def _logical(t, layout_is_hnd, packed):
    """A cache tensor as [blocks, block_size, H, D]."""
    if packed:  # [b, h, p, o, x]
        b, h, p, o, x = t.shape
        return t.permute(0, 3, 1, 2, 4).reshape(b, o, h, p * x)
    return t.permute(0, 2, 1, 3) if layout_is_hnd else t


def exact(case, seed):
    if case["cache"] == case["io"] or work(case)["bytes"] > (1 << 31):
        return None
    if case["op"] == "write":
        layers, slots, _, (ksv, vsv) = _write_data(case, seed)
        top = _FP8_MAX[case["cache"]]
        bs = case["block"]
        slots = slots.long()
        ok = slots >= 0
        out = []
        for cache, key, value in layers:
            for t, rows, s in ((cache.key_cache, key, ksv), (cache.value_cache, value, vsv)):
                r = torch.zeros((cache.num_blocks, bs, case["heads"], case["dim"]),
                                dtype=torch.float64, device=t.device)
                q = (rows.double() / s.double()).clamp_(-top, top)
                r[slots[ok] // bs, slots[ok] % bs] = q[ok]
                out.append(_as_cache(case, r, t))
        return out
    cache, kv, _, table, lens, width, out, _, (ksv, vsv) = _gather_data(case, seed)
    lens = lens.long()
    bs = case["block"]
    pos = torch.arange(width, device=lens.device)
    valid = pos[None] < lens[:, None]
    ids = table.to(lens.device)[:, (pos // bs).clamp(max=table.shape[1] - 1)]
    res = []
    for t, s, lay in ((kv.key_cache, ksv, kv.k_layout), (kv.value_cache, vsv, kv.v_layout)):
        if lay == Layout.BLOCK_CUSTOM:
            rows = t.reshape(t.shape[0], t.shape[1], case["heads"], case["dim"])
        else:
            rows = _logical(t, lay == Layout.BLOCK_HND, lay == Layout.BLOCK_HND_PACKED)
        r = torch.zeros(out[0].shape, dtype=torch.float64, device=t.device)
        at = ids[valid], (pos % bs).expand_as(ids)[valid]
        r[valid] = rows.view(torch.uint8)[at].view(t.dtype).double() * s.double()
        res.append(r)
    return res


def _as_cache(case, r, like):
    """Logical [b, o, H, D] values in the shape of a cache tensor."""
    b, o, h, d = r.shape
    if tuple(like.shape) == (b, o, h, d):
        return r
    if like.dim() == 5 and case["layout"] == "vllm":  # logical (b, o, h, p, x)
        return r.reshape(like.shape)
    if like.dim() == 5:  # [b, h, p, o, x]
        x = like.shape[4]
        return r.reshape(b, o, h, d // x, x).permute(0, 2, 3, 1, 4)
    return r.permute(0, 2, 1, 3)
