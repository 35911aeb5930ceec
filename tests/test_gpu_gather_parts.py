"""GPU parity of gathers of blocks of 64 to 512 tokens, which the transposing
gather takes in parts of 64, bit-identical to the CPU oracle: every layout and
table format, copies and FP8 dequantization, lengths that end in each part,
skipped ids, RAGGED rows of one part in different blocks, head runs that are
not a power of two."""
import numpy as np
import pytest
import torch

from kvx_amd import paged
from kvx_amd.abi import DType, Layout, ScaleGranularity as SG

from gpu_helpers import (TORCH_DT, OffsetsPool, ScaleArg, check_gather, check_gather_offsets,
                         check_gather_ragged, custom_cache, make_cache, random_fill)

pytestmark = pytest.mark.gpu
DEV = "cuda"
NHD, HND, PK = Layout.BLOCK_NHD, Layout.BLOCK_HND, Layout.BLOCK_HND_PACKED


@pytest.mark.parametrize("kind", ["bf16", "f32", "e4m3", "e5m2 to f32"])
@pytest.mark.parametrize("bs", [64, 128, 256, 512])
@pytest.mark.parametrize("layout,shape,table", [
    (layout, shape, table)
    for layout, shape in (("hnd", (3, 128)), ("hnd", (4, 96)), ("packed", (2, 64)),
                          ("packed_k", (8, 128)), ("vllm", (4, 32)))
    for table in ("packed", "ragged", "offsets")
    if not (layout == "vllm" and table == "offsets")])  # pools hold canonical blocks
def test_gather(layout, shape, table, bs, kind):
    H, D = shape
    seed = bs + D + len(kind) + len(table)
    rng = np.random.default_rng(seed)
    gen = torch.Generator().manual_seed(seed)
    dtype, io = {"bf16": (DType.BF16, DType.BF16), "f32": (DType.F32, DType.F32),
                 "e4m3": (DType.F8_E4M3, DType.BF16),
                 "e5m2 to f32": (DType.F8_E5M2, DType.F32)}[kind]
    fp8 = dtype != io
    x = {DType.BF16: 8, DType.F32: 4}.get(dtype, 16)
    nb, L = 9, 2 * bs + 75
    lens = [L, 1, 63, 64, 65, bs - 1, bs, bs + 70, 0, L + 5]
    S, mbps = len(lens), -(-L // bs)
    ld = torch.tensor(lens, dtype=torch.int32, device=DEV)
    ko = random_fill(torch.empty((S, L, H, D), dtype=TORCH_DT[io], device=DEV), gen)
    vo = random_fill(torch.empty_like(ko), gen)
    kw = dict(cache_dtype=dtype, io_dtype=io)
    if fp8:
        if table != "offsets":
            kw.update({f"{t}_scale": ScaleArg(SG.PER_BLOCK_HEAD, rng.uniform(0.01, 0.05, (nb, H)))
                       for t in "kv"})
        else:
            kw.update(k_scale=0.02, v_scale=0.03)
    lays = {"hnd": (HND, HND), "packed": (PK, PK), "packed_k": (PK, NHD)}.get(layout)
    ids = rng.integers(-1, nb + 1, size=(S, mbps)).astype(np.int32)
    ids[0] = rng.permutation(nb)[:mbps]
    if table == "offsets":
        pool = OffsetsPool(*lays, dtype, nb, bs, H, D, pack=x, pitch_pad=64, gen=gen)
        raw = rng.integers(0, nb + 2, size=(S, 1, 2, mbps)).astype(np.uint32)
        raw |= (rng.random(raw.shape) < 0.3).astype(np.uint32) << 31
        check_gather_offsets(pool, ko, vo, torch.from_numpy(raw.view(np.int32)).to(DEV), ld, L,
                             **kw)
        return
    if lays is None:
        pc, kb, vb = custom_cache(dtype, nb, bs, H, D, "bhpox", "bhdo", kx=x, gen=gen)
    else:
        pc, kb, vb = make_cache(*lays, dtype, nb, bs, H, D, pack=x, gen=gen)
    if table == "packed":
        check_gather(pc, kb, vb, ko, vo, torch.from_numpy(ids).to(DEV), ld, L, **kw)
        return
    rows = np.repeat(ids, bs, axis=1)[:, :L].copy()
    rows[4, 3::5] = nb - 1
    rows[7, 66::9] = -1
    indptr = (np.arange(S + 1) * L).astype(np.int64)
    check_gather_ragged(pc, kb, vb, ko, vo,
                        paged.RaggedTable(torch.from_numpy(rows.reshape(-1)).to(DEV),
                                          torch.from_numpy(indptr).to(DEV)), ld, L, **kw)


@pytest.mark.parametrize("bs", [128, 256])
@pytest.mark.parametrize("table", ["packed", "ragged", "offsets"])
def test_parts_of_odd_rows(table, bs):
    """576-byte rows: 64-byte tiles of 64 rows."""
    test_gather("packed", (1, 576), table, bs, "e4m3")


@pytest.mark.parametrize("kind", ["e4m3", "e5m2 to f32"])
@pytest.mark.parametrize("shape", [(1, 576), (8, 128)])
def test_parts_of_one_byte_runs(shape, kind):
    """vLLM's FP8 pair, PACKED, in parts of 128 rows and (8 x 128) of 64."""
    test_gather("vllm", shape, "packed", 256, kind)
