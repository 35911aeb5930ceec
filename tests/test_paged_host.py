"""The native descriptor builder of write_kv / gather_kv (csrc/paged_host.cpp)
against the ctypes helpers, on the CPU: over layouts, dtypes, strides, tables
and scales it hands an entry point the same bytes, and what it does not take
goes on to the helpers and raises what they raise."""
import ctypes as C
import warnings

import pytest
import torch

from kvx_amd import abi, build, paged
from kvx_amd.abi import Layout, ScaleGranularity as SG

SEEN = {}
STREAM = 0x1234


def _capture(n, second):
    def fn(cd, d, *rest):
        SEEN["cd"] = C.string_at(cd, C.sizeof(abi.CacheDesc))
        SEEN["d"] = C.string_at(d, C.sizeof(second))
        SEEN["rest"] = [C.string_at(r, C.sizeof(abi.ScaleDesc)) if i < n - 3 and n == 5 else r
                        for i, r in enumerate(rest)]
        return 2

    return fn


P = C.c_void_p
WRITE = C.CFUNCTYPE(C.c_int, P, P, P)(_capture(3, abi.WriteDesc))
PREFILL = C.CFUNCTYPE(C.c_int, P, P, C.c_int32, P)(_capture(4, abi.WriteDesc))
GATHER = C.CFUNCTYPE(C.c_int, P, P, P)(_capture(3, abi.GatherDesc))
DEQUANT = C.CFUNCTYPE(C.c_int, P, P, P, P, P)(_capture(5, abi.GatherDesc))


@pytest.fixture
def entry_points(monkeypatch):
    fns = {"kvx_launch_write_kv": WRITE, "kvx_write_kv": WRITE,
           "kvx_launch_write_kv_prefill": PREFILL, "kvx_launch_gather_kv": GATHER,
           "kvx_gather_kv": GATHER, "kvx_launch_gather_kv_dequant": DEQUANT}
    monkeypatch.setattr(paged, "_address", lambda lib, name: C.cast(fns[name], P).value)
    SEEN.clear()


def caches():
    for dt in (torch.bfloat16, torch.float32, torch.float8_e4m3fn, torch.float8_e5m2):
        for lay in (Layout.BLOCK_NHD, Layout.BLOCK_HND, Layout.BLOCK_HND_PACKED):
            yield paged.alloc_cache(5, 4, 2, 16, dt, "cpu", lay)
        yield paged.alloc_custom_cache(5, 4, 2, 16, dt, "cpu", "bhpox", "bhdo")
    kc = torch.zeros(5, 4, 3, 16, dtype=torch.float16)[:, :, :2]
    yield paged.PagedCache(kc, kc.clone(), Layout.BLOCK_NHD, Layout.BLOCK_NHD, 5, 4, 2, 16)


SCALES = [None, torch.ones(1), torch.ones(()), paged.Scales(torch.ones(2), SG.PER_HEAD),
          paged.Scales(torch.ones(5, 4)[:, ::2], SG.PER_BLOCK_HEAD),
          paged.Scales(torch.ones(()), SG.PER_TENSOR), paged.Scales(torch.ones(1), SG.NONE)]


@pytest.mark.parametrize("scale", SCALES)
@pytest.mark.parametrize("per_seq", [None, 3, -7])
@pytest.mark.parametrize("slot_dtype", [torch.int32, torch.int64])
def test_write_descriptors(entry_points, scale, per_seq, slot_dtype):
    for pc in caches():
        for io in (torch.bfloat16, torch.float32):
            key = torch.zeros(6, 2, 16, dtype=io)
            val = torch.zeros(6, 4, 16, dtype=io)[:, ::2]  # strided: the library decides
            slots = torch.zeros(6, dtype=slot_dtype)
            st = paged.write_kv(pc, key, val, slots, tokens_per_seq=per_seq, k_scale=scale,
                                v_scale=scale, stream=STREAM)
            assert st == abi.Status.UNSUPPORTED
            assert SEEN["cd"] == bytes(pc.desc())
            assert SEEN["d"] == bytes(paged.build_write(pc, key, val, slots, scale, scale))
            assert SEEN["rest"] == ([STREAM] if per_seq is None else [per_seq, STREAM])


def tables():
    yield torch.zeros(3, 4, dtype=torch.int32)
    yield torch.zeros(3, 4, dtype=torch.int64)
    yield paged.RaggedTable(torch.zeros(9, dtype=torch.int64), torch.zeros(4, dtype=torch.int32))
    pool = torch.zeros(4096, dtype=torch.uint8).view(torch.bfloat16)
    for sec in (None, pool.clone()):
        yield paged.OffsetsTable(torch.zeros(3, 1, 2, 4, dtype=torch.int32), pool, sec, 256)


@pytest.mark.parametrize("scale,entry", [(s, "launch") for s in SCALES] + [(None, "abi")])
def test_gather_descriptors(entry_points, scale, entry):
    for pc in caches():
        for tb in tables():
            ko = torch.zeros(3, 16, 2, 16, dtype=torch.float16)
            vo = torch.zeros_like(ko)
            lens = torch.zeros(3, dtype=torch.int32)
            st = paged.gather_kv(pc, ko, vo, tb, lens, 16, k_scale=scale, v_scale=scale,
                                 stream=STREAM, entry=entry)
            assert st == abi.Status.UNSUPPORTED
            assert SEEN["cd"] == bytes(paged.gather_cache_desc(pc, tb))
            assert SEEN["d"] == bytes(paged.build_gather(ko, vo, tb, lens, 16))
            if scale is None:
                assert SEEN["rest"] == [STREAM]
            else:
                sd = bytes(paged.scale_desc_of(scale))
                assert SEEN["rest"] == [sd, sd, STREAM]


def test_what_the_helpers_refuse_still_raises(entry_points):
    pc = next(caches())
    key = torch.zeros(6, 2, 16, dtype=torch.bfloat16)
    slots = torch.zeros(6, dtype=torch.int64)
    lens = torch.zeros(3, dtype=torch.int32)
    out = torch.zeros(3, 16, 2, 16, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="unsupported dtype"):
        paged.write_kv(pc, key, key, slots.to(torch.uint8), stream=STREAM)
    with pytest.raises(ValueError, match="unsupported dtype"):
        paged.write_kv(pc, key.double(), key, slots, stream=STREAM)
    with pytest.raises(AttributeError):
        paged.write_kv(pc, None, key, slots, stream=STREAM)
    with pytest.raises(ValueError):
        paged.gather_kv(pc, out, out, torch.zeros(3, dtype=torch.int32), lens, 16, stream=STREAM)
    bad = paged.OffsetsTable(torch.zeros(3, 1, 3, 4, dtype=torch.int32), key, None, 256)
    with pytest.raises(ValueError, match="KV_OFFSETS"):
        paged.gather_kv(pc, out, out, bad, lens, 16, stream=STREAM)
    with pytest.raises(Exception):
        torch.func.vmap(lambda k: paged.write_kv(pc, k, k, slots, stream=STREAM) and k)(
            key[None])
    assert not SEEN


@pytest.mark.parametrize("file", ["missing", "of another build"])
def test_without_the_module_the_helpers_serve(monkeypatch, tmp_path, file):
    """As before there was one: the library sees the same descriptors."""
    path = tmp_path / "_paged_host.so"
    if file != "missing":
        path.write_bytes(b"not for this Python")
    monkeypatch.setattr(paged, "_HOST_PATH", path)
    monkeypatch.setattr(paged, "_HOST", None)
    lib = abi.bind_like(C.CDLL(str(abi.LIB_PATH)))
    lib.kvx_launch_write_kv = WRITE
    lib.kvx_launch_gather_kv = GATHER
    monkeypatch.setattr(abi, "_LIB", lib)
    SEEN.clear()
    pc = next(caches())
    key = torch.zeros(6, 2, 16, dtype=torch.bfloat16)
    slots = torch.zeros(6, dtype=torch.int64)
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        assert paged.write_kv(pc, key, key, slots, stream=STREAM) == abi.Status.UNSUPPORTED
        assert SEEN["d"] == bytes(paged.build_write(pc, key, key, slots))
        out = torch.zeros(3, 16, 2, 16, dtype=torch.bfloat16)
        table, lens = torch.zeros(3, 4, dtype=torch.int32), torch.zeros(3, dtype=torch.int32)
        assert paged.gather_kv(pc, out, out, table, lens, 16,
                               stream=STREAM) == abi.Status.UNSUPPORTED
        assert SEEN["d"] == bytes(paged.build_gather(out, out, table, lens, 16))
    assert len(seen) == (file != "missing")


def test_build_without_rocm_says_so(monkeypatch):
    monkeypatch.setattr(torch.version, "hip", None)
    with pytest.raises(RuntimeError, match="ROCm build of PyTorch"):
        build.build_paged_host()
