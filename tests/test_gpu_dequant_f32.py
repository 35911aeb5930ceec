"""GPU parity of the FP8 gathers into f32 (chunks of four codes), bit-identical
to the CPU oracle: head sizes that are and are not whole chunks of 4, 8 and 16
codes, every layout and table format, per-tensor and per-head scales, partial
blocks, -1 and out-of-range ids."""
import numpy as np
import pytest
import torch

from kvx_amd import paged
from kvx_amd.abi import DType, Layout, ScaleGranularity as SG

from gpu_helpers import (OffsetsPool, ScaleArg, check_gather, check_gather_offsets,
                         check_gather_ragged, make_cache, random_fill)

pytestmark = pytest.mark.gpu
DEV = "cuda"
NHD, HND, PK = Layout.BLOCK_NHD, Layout.BLOCK_HND, Layout.BLOCK_HND_PACKED


@pytest.mark.parametrize("table", ["packed", "ragged", "offsets"])
@pytest.mark.parametrize("shape,layout", [
    (shape, layout)
    for shape in ((8, 128), (4, 12), (4, 36), (1, 576), (3, 7), (2, 16))
    for layout in (NHD, HND, PK)
    if not (layout == PK and shape[1] % 4)])  # packs of 4
def test_gather_into_f32(shape, layout, table):
    H, D = shape
    seed = H * 1000 + D + 7 * int(layout)
    rng = np.random.default_rng(seed)
    gen = torch.Generator().manual_seed(seed)
    fp8 = [DType.F8_E4M3, DType.F8_E5M2][seed % 2]
    bs, nb, S, L = [16, 64][D % 3 == 0], 40, 5, 150
    pack = 16 if D % 16 == 0 else 4
    if seed % 3 == 0:
        ks, vs = (ScaleArg(SG.PER_HEAD, rng.uniform(0.01, 0.05, H)) for _ in range(2))
    else:
        ks, vs = 0.013, 0.0071
    lens = torch.tensor([L, L - 20, L - 9, bs + 1, L + 7], dtype=torch.int32, device=DEV)
    ko = random_fill(torch.empty((S, L, H, D), dtype=torch.float32, device=DEV), gen)
    vo = random_fill(torch.empty_like(ko), gen)
    mbps = (L + bs - 1) // bs
    kw = dict(cache_dtype=fp8, io_dtype=DType.F32, k_scale=ks, v_scale=vs)
    if table == "offsets":
        pool = OffsetsPool(layout, layout, fp8, nb, bs, H, D, pack=pack, pitch_pad=16, gen=gen)
        raw = rng.integers(0, nb + 2, size=(S, 1, 2, mbps)).astype(np.uint32)
        raw |= (rng.random(raw.shape) < 0.3).astype(np.uint32) << 31
        check_gather_offsets(pool, ko, vo, torch.from_numpy(raw.view(np.int32)).to(DEV), lens, L,
                             **kw)
        return
    pc, kb, vb = make_cache(layout, layout, fp8, nb, bs, H, D, pack=pack, gen=gen)
    ids = rng.integers(-1, nb + 1, size=(S, mbps)).astype(np.int32)
    if table == "packed":
        check_gather(pc, kb, vb, ko, vo, torch.from_numpy(ids).to(DEV), lens, L, **kw)
        return
    rows = np.repeat(ids, bs, axis=1)[:, :L].copy()
    rows[1, ::5] = nb - 1  # a sequence whose tiles name several blocks
    indptr = np.arange(S + 1, dtype=np.int32) * L
    check_gather_ragged(pc, kb, vb, ko, vo,
                        paged.RaggedTable(torch.from_numpy(rows.reshape(-1)).to(DEV),
                                          torch.from_numpy(indptr).to(DEV)), lens, L, **kw)


@pytest.mark.parametrize("table", ["ragged", "offsets"])
@pytest.mark.parametrize("heads", [40, 63])
def test_wide_rows(heads, table):
    """Rows of 1280 and 2016 four-code chunks, in the flat indexed gathers."""
    D, bs, nb, S, L = 128, 16, 12, 3, 45
    rng = np.random.default_rng(heads)
    gen = torch.Generator().manual_seed(heads)
    scales = [ScaleArg(SG.PER_HEAD, rng.uniform(0.01, 0.05, heads)) for _ in range(2)]
    lens = torch.tensor([L, bs + 1, L + 7], dtype=torch.int32, device=DEV)
    ko = random_fill(torch.empty((S, L, heads, D), dtype=torch.float32, device=DEV), gen)
    vo = random_fill(torch.empty_like(ko), gen)
    kw = dict(cache_dtype=DType.F8_E4M3, io_dtype=DType.F32, k_scale=scales[0], v_scale=scales[1])
    if table == "offsets":
        pool = OffsetsPool(NHD, NHD, DType.F8_E4M3, nb, bs, heads, D, pitch_pad=16, gen=gen)
        raw = rng.integers(0, nb + 1, size=(S, 1, 2, 3)).astype(np.uint32)
        raw |= (rng.random(raw.shape) < 0.3).astype(np.uint32) << 31
        check_gather_offsets(pool, ko, vo, torch.from_numpy(raw.view(np.int32)).to(DEV), lens, L,
                             **kw)
        return
    pc, kb, vb = make_cache(NHD, NHD, DType.F8_E4M3, nb, bs, heads, D, gen=gen)
    rows = np.repeat(rng.integers(-1, nb + 1, size=(S, 3)).astype(np.int32), bs, axis=1)[:, :L]
    rows = rows.copy()
    rows[1, ::5] = nb - 1
    indptr = np.arange(S + 1, dtype=np.int32) * L
    check_gather_ragged(pc, kb, vb, ko, vo,
                        paged.RaggedTable(torch.from_numpy(rows.reshape(-1)).to(DEV),
                                          torch.from_numpy(indptr).to(DEV)), lens, L, **kw)
