"""GPU parity of the tiled write (write_tiles_kernel) at its edges,
bit-identical to the CPU oracle over whole caches: blocks of 2 to 256 tokens
and of sizes that are not a power of two, prefill chunks of random lengths
that start anywhere in a block, decode batches, -1 and out-of-range slots,
batches of one token up to several workgroups' rows, direct, staged and
narrow tensors, copies and FP8 quantization with every scale granularity."""
import numpy as np
import pytest
import torch

from kvx_amd.abi import DType, Layout, ScaleGranularity as SG

from gpu_helpers import TORCH_DT, ScaleArg, check_write, custom_cache, make_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"
NHD, HND, PK = Layout.BLOCK_NHD, Layout.BLOCK_HND, Layout.BLOCK_HND_PACKED


def cache_of(layout, dtype, nb, bs, H, D, gen):
    x = 16 // {DType.F32: 4, DType.F8_E4M3: 1, DType.F8_E5M2: 1}.get(dtype, 2)
    if layout == "vllm":
        return custom_cache(dtype, nb, bs, H, D, "bhpox", "bhdo", kx=x, gen=gen)
    if layout == "x8":  # packs of 8 bytes beside runs of two of them
        e = max(1, x // 2)
        return custom_cache(dtype, nb, bs, H, D, "bhpox", "bhpox", kx=e, vx=2 * x, gen=gen)
    k, v = {"hnd": (HND, HND), "packed": (PK, PK), "packed_k": (PK, NHD)}[layout]
    return make_cache(k, v, dtype, nb, bs, H, D, pack=x, gen=gen)


def slots_of(kind, T, bs, nb, rng):
    if kind == "decode":
        s = rng.permutation(nb * bs)[:T].astype(np.int64)
        s[rng.random(T) < 0.2] = -1
        s[rng.random(T) < 0.1] = nb * bs + 5
        return s
    # chunks of consecutive positions over random blocks, each starting
    # anywhere in its first block; some tokens spoiled
    out, free = [], list(rng.permutation(nb))
    while sum(map(len, out)) < T:
        n = int(rng.integers(1, min(T, 150) + 1))
        start = int(rng.integers(0, bs))
        need = (start + n + bs - 1) // bs
        if need > len(free):
            break
        ids = np.array([free.pop() for _ in range(need)], np.int64)
        pos = start + np.arange(n)
        out.append(ids[pos // bs] * bs + pos % bs)
    s = np.concatenate(out)[:T]
    if kind == "spoiled":
        at = rng.integers(0, s.size, size=max(1, s.size // 20))
        s[at] = -1
        at = rng.integers(0, s.size, size=max(1, s.size // 40))
        s[at] = nb * bs + rng.integers(0, 3, size=at.size)
    return s


CASES = [(lay, bs, kind) for lay in ("hnd", "packed", "packed_k", "vllm", "x8")
         for bs, kind in ((2, "chunks"), (8, "chunks"), (16, "spoiled"), (24, "chunks"),
                          (32, "chunks"), (48, "spoiled"), (64, "chunks"), (256, "spoiled"),
                          (128, "chunks"), (16, "decode"), (64, "decode"))]


@pytest.mark.parametrize("tokens", [1, 33, 700])
@pytest.mark.parametrize("layout,bs,kind", CASES)
def test_copy(layout, bs, kind, tokens):
    seed = CASES.index((layout, bs, kind)) * 3 + tokens
    rng = np.random.default_rng(seed)
    gen = torch.Generator().manual_seed(seed)
    dtype = [DType.BF16, DType.F32, DType.F16][seed % 3]
    H, D = [(8, 128), (3, 128), (2, 96), (4, 64)][seed % 4]
    nb = (2 * tokens + 40 * bs) // bs + 8
    pc, kb, vb = cache_of(layout, dtype, nb, bs, H, D, gen)
    s = slots_of(kind, tokens, bs, nb, rng)
    key, val = (torch.randn((s.size, H, D), generator=gen).to(TORCH_DT[dtype]).to(DEV)
                for _ in range(2))
    slots = torch.from_numpy(s).to(DEV, torch.int32 if seed % 2 else torch.int64)
    check_write(pc, kb, vb, key, val, slots, io_dtype=dtype, cache_dtype=dtype)


@pytest.mark.parametrize("kind", ["tensor", "block_head"])
@pytest.mark.parametrize("layout,bs,slots_kind", [c for c in CASES if c[1] != 2])
def test_quantize(layout, bs, slots_kind, kind):
    seed = 1000 + CASES.index((layout, bs, slots_kind)) * 2 + (kind == "tensor")
    rng = np.random.default_rng(seed)
    gen = torch.Generator().manual_seed(seed)
    fp8 = [DType.F8_E4M3, DType.F8_E5M2][seed % 2]
    io = [DType.BF16, DType.F32, DType.F16][seed % 3]
    H, D, T = 4, [128, 96][seed % 2], 400
    nb = (2 * T + 40 * bs) // bs + 8
    pc, kb, vb = cache_of(layout, fp8, nb, bs, H, D, gen)
    s = slots_of(slots_kind, T, bs, nb, rng)
    key, val = ((torch.randn((s.size, H, D), generator=gen) * 2).to(TORCH_DT[io]).to(DEV)
                for _ in range(2))
    if kind == "tensor":
        ks, vs = 0.013, 0.0071
    else:
        ks, vs = (ScaleArg(SG.PER_BLOCK_HEAD,
                           torch.empty((nb, H)).uniform_(0.002, 0.05, generator=gen).numpy())
                  for _ in range(2))
    check_write(pc, kb, vb, key, val, torch.from_numpy(s).to(DEV), io_dtype=io, cache_dtype=fp8,
                k_scale=ks, v_scale=vs)


@pytest.mark.parametrize("start", range(0, 64, 7))
@pytest.mark.parametrize("layout", ["packed", "vllm"])
def test_one_chunk_from_every_phase(layout, start):
    """One long chunk: every workgroup's rows go on from its neighbour's."""
    gen = torch.Generator().manual_seed(start)
    H, D, bs, T, nb = 8, 128, 64, 517, 16
    pc, kb, vb = cache_of(layout, DType.BF16, nb, bs, H, D, gen)
    ids = torch.randperm(nb, generator=gen)[: (start + T + bs - 1) // bs]
    pos = start + torch.arange(T)
    slots = ids[pos // bs] * bs + pos % bs
    key, val = (torch.randn((T, H, D), generator=gen).bfloat16().to(DEV) for _ in range(2))
    check_write(pc, kb, vb, key, val, slots.to(DEV), io_dtype=DType.BF16, cache_dtype=DType.BF16)


@pytest.mark.parametrize("fp8,tokens", [(None, 3200), (None, 1500), (DType.F8_E4M3, 5600),
                                        (DType.F8_E4M3, 2800)])
@pytest.mark.parametrize("bs", [16, 20])
def test_row_major_pairs_by_size(fp8, tokens, bs):
    """NHD pairs on both sides of the size rule that picks the kernel."""
    rng = np.random.default_rng(tokens + bs)
    gen = torch.Generator().manual_seed(tokens + bs)
    H, D, nb = 8, 128, tokens // bs + 300
    dtype = fp8 or DType.BF16
    pc, kb, vb = make_cache(NHD, NHD, dtype, nb, bs, H, D, gen=gen)
    s = slots_of("spoiled", tokens, bs, nb, rng)
    key, val = (torch.randn((s.size, H, D), generator=gen).bfloat16().to(DEV) for _ in range(2))
    check_write(pc, kb, vb, key, val, torch.from_numpy(s).to(DEV), io_dtype=DType.BF16,
                cache_dtype=dtype, k_scale=0.01 if fp8 else None, v_scale=0.02 if fp8 else None)


# (cache, io, tokens) of 8 x 128 rows whose narrow tiles have 32 rows and align
# on 32 slots, so that all 64 lanes hold slots (test_dispatch_plan.py pins those
# shapes).  4200 bf16 tokens take 16 KiB tiles.
WHOLE = [(DType.BF16, DType.BF16, 1100), (DType.BF16, DType.BF16, 4200),
         (DType.F8_E4M3, DType.BF16, 2100), (DType.F8_E5M2, DType.F32, 4200)]


@pytest.mark.parametrize("kind", ["chunks", "spoiled"])
@pytest.mark.parametrize("bs", [32, 64, 128])
@pytest.mark.parametrize("cache,io,tokens", WHOLE)
def test_narrow_tiles_of_32_rows(cache, io, tokens, bs, kind):
    """vLLM's pair, chunks that start anywhere in a block: units of 16 bytes,
    runs that a workgroup takes over from its rows, and (spoiled) single runs."""
    seed = tokens + bs + len(kind)
    rng = np.random.default_rng(seed)
    gen = torch.Generator().manual_seed(seed)
    H, D = 8, 128
    nb = (2 * tokens + 40 * bs) // bs + 8
    pc, kb, vb = cache_of("vllm", cache, nb, bs, H, D, gen)
    s = slots_of(kind, tokens, bs, nb, rng)
    key, val = ((torch.randn((s.size, H, D), generator=gen) * 2).to(TORCH_DT[io]).to(DEV)
                for _ in range(2))
    sc = {}
    if cache != io and kind == "chunks":
        sc = dict(k_scale=0.013, v_scale=0.0071)
    elif cache != io:
        sc = {f"{t}_scale": ScaleArg(
            SG.PER_BLOCK_HEAD, torch.empty((nb, H)).uniform_(0.002, 0.05, generator=gen).numpy())
            for t in "kv"}
    check_write(pc, kb, vb, key, val, torch.from_numpy(s).to(DEV), io_dtype=io, cache_dtype=cache,
                **sc)


@pytest.mark.parametrize("tokens", [1, 15, 16, 17, 31, 33, 64, 129])
@pytest.mark.parametrize("start", [0, 1, 15, 40])
@pytest.mark.parametrize("heads", [1, 3])
def test_narrow_tiles_of_small_batches(heads, start, tokens):
    """One chunk into an E4M3 vLLM pair in 64-token blocks: tiles 32 bytes wide
    whose units start and end inside the rows of one or two workgroups."""
    gen = torch.Generator().manual_seed(start + tokens)
    D, bs, nb = 128, 64, 8
    pc, kb, vb = cache_of("vllm", DType.F8_E4M3, nb, bs, heads, D, gen)
    ids = torch.randperm(nb, generator=gen)
    pos = start + torch.arange(tokens)
    slots = ids[pos // bs] * bs + pos % bs
    key, val = (torch.randn((tokens, heads, D), generator=gen).bfloat16().to(DEV)
                for _ in range(2))
    check_write(pc, kb, vb, key, val, slots.to(DEV), io_dtype=DType.BF16,
                cache_dtype=DType.F8_E4M3, k_scale=0.01, v_scale=0.02)
