"""GPU parity of gathers whose grid mostly lies past the sequences: RAGGED
batches on both sides of the rule that doubles a tile's rows, and every table
format with lengths of 0, negative, cut inside a tile and past max_seq_len."""
import numpy as np
import pytest
import torch

from kvx_amd import paged
from kvx_amd.abi import DType, Layout, ScaleGranularity as SG

from gpu_helpers import (TORCH_DT, OffsetsPool, ScaleArg, check_gather, check_gather_offsets,
                         check_gather_ragged, make_cache, random_fill)

pytestmark = pytest.mark.gpu
DEV = "cuda"
NHD, HND, PK = Layout.BLOCK_NHD, Layout.BLOCK_HND, Layout.BLOCK_HND_PACKED


@pytest.mark.parametrize("extra", [-1, 0])
def test_ragged_sparse_tiles(extra):
    """49152 filled tiles of one 1552-byte row (the rule's least), or one
    token fewer: whole blocks, blocks that change inside a doubled tile, and
    skipped ids."""
    rng = np.random.default_rng(5)
    gen = torch.Generator().manual_seed(5)
    H, D, bs, S = 1, 776, 16, 24
    lens = np.full(S, 300)
    lens[3] = 12000
    lens[11] = 49152 + extra - lens[:11].sum() - lens[12:].sum()
    L = int(lens.max())
    assert lens.sum() == 49152 + extra and lens.sum() * 3 < S * L
    nb = 3300
    pc, kb, vb = make_cache(NHD, NHD, DType.BF16, nb, bs, H, D, gen=gen)
    rows = [np.repeat(rng.integers(0, nb, size=-(-n // bs)), bs)[:n] for n in lens]
    rows[3][::7] = nb - 2  # rows of a tile in different blocks
    rows[5][::3] = -1
    rows[6][:] = nb
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    table = paged.RaggedTable(torch.from_numpy(np.concatenate(rows).astype(np.int32)).to(DEV),
                              torch.from_numpy(indptr).to(DEV))
    ko = torch.zeros((S, L, H, D), dtype=torch.bfloat16, device=DEV)
    vo = torch.zeros_like(ko)
    dl = lens.copy()
    dl[0], dl[1], dl[2], dl[4] = 0, -3, 77, L + 9
    check_gather_ragged(pc, kb, vb, ko, vo, table, torch.from_numpy(dl.astype(np.int32)).to(DEV),
                        L, cache_dtype=DType.BF16, io_dtype=DType.BF16)


@pytest.mark.parametrize("cache,io,H,D,base", [(DType.BF16, DType.BF16, 1, 392, 2),
                                               (DType.F8_E4M3, DType.BF16, 2, 776, 1),
                                               (DType.F8_E5M2, DType.F32, 1, 1552, 1)])
def test_ragged_sparse_tiles_of_other_rows(cache, io, H, D, base):
    """The rule in effect on tiles of two rows (four), and on FP8 rows with
    per-block-head scales: whole blocks and rows of a tile in several blocks."""
    rng = np.random.default_rng(D)
    gen = torch.Generator().manual_seed(D)
    bs, S, total = 16, 24, base * 49152
    L = 3 * total // S + 33
    lens = np.full(S, L)
    lens[7:] = (total - 7 * L) // (S - 7)
    lens[-1] += total - lens.sum()
    assert lens.sum() == total and lens.max() == L and total * 3 < S * L
    nb = 500
    pc, kb, vb = make_cache(NHD, NHD, cache, nb, bs, H, D, gen=gen)
    rows = [np.repeat(rng.integers(0, nb, size=-(-n // bs)), bs)[:n] for n in lens]
    rows[3][::7] = nb - 2
    rows[9][::3] = -1
    indptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    table = paged.RaggedTable(torch.from_numpy(np.concatenate(rows).astype(np.int32)).to(DEV),
                              torch.from_numpy(indptr).to(DEV))
    sc = {}
    if cache != io:
        sc = {f"{t}_scale": ScaleArg(SG.PER_BLOCK_HEAD, rng.uniform(0.01, 0.05, (nb, H)))
              for t in "kv"}
    ko = torch.zeros((S, L, H, D), dtype=TORCH_DT[io], device=DEV)
    vo = torch.zeros_like(ko)
    dl = lens.copy()
    dl[0], dl[1], dl[8] = 77, L + 9, 0
    check_gather_ragged(pc, kb, vb, ko, vo, table, torch.from_numpy(dl.astype(np.int32)).to(DEV),
                        L, cache_dtype=cache, io_dtype=io, **sc)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("layout,bs,table", [
    (layout, bs, table)
    for layout, bs in ((NHD, 16), (HND, 16), (HND, 64), (PK, 32), (NHD, 24))
    for table in ("packed", "ragged", "offsets")
    if not (bs == 24 and table == "offsets")])  # KV_OFFSETS blocks are a power of two
def test_lengths_at_every_edge(layout, bs, table, fp8):
    rng = np.random.default_rng(bs + fp8)
    gen = torch.Generator().manual_seed(bs)
    dtype, io = (DType.F8_E4M3, DType.BF16) if fp8 else (DType.BF16, DType.BF16)
    H, D, L, nb = 8, 128, 700, 90
    edges = [0, -1, 1, bs - 1, bs, bs + 1, 2 * bs, L - 1, L, L + 1, 8 * bs + 3]
    S, mbps = len(edges), -(-L // bs)
    lens = torch.tensor(edges, dtype=torch.int32, device=DEV)
    ko = random_fill(torch.empty((S, L, H, D), dtype=TORCH_DT[io], device=DEV), gen)
    vo = random_fill(torch.empty_like(ko), gen)
    sc = dict(k_scale=0.02, v_scale=0.03) if fp8 else {}
    kw = dict(cache_dtype=dtype, io_dtype=io, **sc)
    ids = rng.integers(-1, nb + 1, size=(S, mbps)).astype(np.int32)
    pack = 16 if fp8 else 8
    if table == "offsets":
        pool = OffsetsPool(layout, layout, dtype, nb, bs, H, D, pack=pack, gen=gen)
        raw = rng.integers(0, nb + 2, size=(S, 1, 2, mbps)).astype(np.uint32)
        raw |= (rng.random(raw.shape) < 0.3).astype(np.uint32) << 31
        check_gather_offsets(pool, ko, vo, torch.from_numpy(raw.view(np.int32)).to(DEV), lens, L,
                             **kw)
        return
    pc, kb, vb = make_cache(layout, layout, dtype, nb, bs, H, D, pack=pack, gen=gen)
    if table == "packed":
        check_gather(pc, kb, vb, ko, vo, torch.from_numpy(ids).to(DEV), lens, L, **kw)
        return
    rows = np.repeat(ids, bs, axis=1)[:, :L]
    indptr = (np.arange(S + 1) * L).astype(np.int32)
    check_gather_ragged(pc, kb, vb, ko, vo,
                        paged.RaggedTable(torch.from_numpy(rows.reshape(-1).copy()).to(DEV),
                                          torch.from_numpy(indptr).to(DEV)), lens, L, **kw)
