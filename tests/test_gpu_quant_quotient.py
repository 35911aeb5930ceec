"""GPU parity of the FP8 quantizing write at the edges of its quotient: rows
of values at and next to every boundary between codes times the scale, for
scales that take the two-operation quotient and scales that divide
(fp_convert.h's quant_scale), bit-identical to the CPU oracle."""
import numpy as np
import pytest
import torch

from kvx_amd.abi import DType, Layout

from gpu_helpers import TORCH_DT, check_write, make_cache

pytestmark = pytest.mark.gpu
DEV = "cuda"

SCALES = [1.0, 0.0223, -0.37, 3.0,
          float(np.uint32(0x3F800040).view(np.float32)),   # 64 above a multiple of 2^20
          float(np.uint32(0x3F80003F).view(np.float32)),   # 63: divides
          float(np.uint32(0x3C9FFFC1).view(np.float32)),   # -63: divides
          2.0 ** -60, 2.0 ** 60, 2.0 ** -61, 1e-40, 0.0, float("inf"), float("nan")]


def boundary_values(fp8, scale):
    codes = torch.arange(0, 0x7F if fp8 == DType.F8_E4M3 else 0x7C, dtype=torch.uint8)
    v = codes.view(TORCH_DT[fp8]).float().numpy()
    mids = np.concatenate([(v[1:] + v[:-1]) / 2, v, v[-1:] * 4]).astype(np.float32)
    with np.errstate(all="ignore"):
        x = np.abs(mids * np.float32(scale if np.isfinite(scale) and scale else 1.0))
    u = x.view(np.uint32).astype(np.int64)
    u = np.clip(u[:, None] + np.arange(-2, 3)[None], 0, 0x7FFFFFFF).reshape(-1)
    u = np.concatenate([u, [0, 1, 0x7FFFFF, 0x7F7FFFFF, 0x7F800000, 0x7FC00000, 0x7F800001]])
    x = np.concatenate([u, u | 0x80000000]).astype(np.uint32).view(np.float32)
    return torch.from_numpy(np.resize(x, (-(-x.size // 64)) * 64).copy())


@pytest.mark.parametrize("io", [DType.F32, DType.BF16, DType.F16])
@pytest.mark.parametrize("fp8", [DType.F8_E4M3, DType.F8_E5M2])
@pytest.mark.parametrize("scale", SCALES)
def test_quantizing_write_at_code_boundaries(scale, fp8, io):
    gen = torch.Generator().manual_seed(7)
    key = boundary_values(fp8, scale).reshape(-1, 1, 64)
    val = boundary_values(fp8, 0.0071).reshape(-1, 1, 64)
    T = min(key.shape[0], val.shape[0])
    key, val = (t[:T].to(TORCH_DT[io]).contiguous().to(DEV) for t in (key, val))
    bs = 16
    nb = T // bs + 2
    pc, kb, vb = make_cache(Layout.BLOCK_NHD, Layout.BLOCK_HND_PACKED, fp8, nb, bs, 1, 64, pack=16,
                            gen=gen)
    slots = torch.randperm(nb * bs, generator=gen)[:T].to(DEV)
    check_write(pc, kb, vb, key, val, slots, io_dtype=io, cache_dtype=fp8, k_scale=scale,
                v_scale=0.0071)
