"""The launch planning without a GPU: builds the library's host layer over
stand-in kernel families (dispatch_plan_stubs.cpp) and returns, for a write
or gather, the kernel that the planning picks and its shape.  Addresses are
made up: nothing is launched."""
from __future__ import annotations

import ctypes as C
import functools
import json
import subprocess
import tempfile
from pathlib import Path

from kvx_amd import abi, build
from kvx_amd.abi import DType, Layout, Memory, Status, TableFormat, contiguous_strides

TESTS = Path(__file__).resolve().parent
DEVICE = Memory.DEVICE
ADDR = 0x10000  # 64 KiB aligned, never read
BYTES = {DType.F32: 4, DType.F16: 2, DType.BF16: 2, DType.F8_E4M3: 1, DType.F8_E5M2: 1}
VLLM = "vllm"      # x-packed K, token-innermost V
PACKED_K = "packed_k"  # x-packed K, row-major V


@functools.cache
def lib() -> C.CDLL:
    flags = [build.hipcc(), "--cuda-host-only", "-O1", "-std=c++17", "-fPIC", "-x", "hip",
             f"-I{build.INCLUDE}", f"-I{build.CSRC}"]
    sources = [build.CSRC / "abi.cpp", build.CSRC / "launch.cpp", build.CSRC / "dispatch.hip",
               TESTS / "dispatch_plan_stubs.cpp"]
    with tempfile.TemporaryDirectory(prefix="kvx_plan_") as tmp:
        objs = [f"{tmp}/{s.name}.o" for s in sources]
        jobs = [subprocess.Popen([*flags, "-c", str(s), "-o", o], stderr=subprocess.PIPE, text=True)
                for s, o in zip(sources, objs)]
        for j in jobs:
            err = j.communicate()[1]
            assert j.returncode == 0, err
        subprocess.run([build.hipcc(), "-shared", "-o", f"{tmp}/libkvx_plan.so", *objs], check=True)
        loaded = abi.bind_like(C.CDLL(f"{tmp}/libkvx_plan.so"))
    loaded.kvx_plan.restype = C.c_char_p
    return loaded


def _plan(status: int) -> dict:
    # without a device hipGetLastError reports one missing after the planning
    assert Status(status) in (Status.OK, Status.INTERNAL_ERROR), Status(status)
    return json.loads(lib().kvx_plan())


def _tensor(layout, nb, bs, H, D, es, pad):
    """Shape, strides and layout code of one cache tensor; pad: elements
    between a row's heads (NHD) or after each head's run (HND)."""
    if layout == "bhdo":
        order = (nb, H, D, bs)
        st = contiguous_strides(order)
        return (nb, bs, H, D), (st[0], st[3], st[1], st[2]), Layout.BLOCK_CUSTOM
    if layout == Layout.BLOCK_HND_PACKED:
        x = 16 // es
        shape = (nb, H, D // x, bs, x)
        return shape, contiguous_strides(shape), layout
    shape = (nb, bs, H, D) if layout == Layout.BLOCK_NHD else (nb, H, bs, D)
    return shape, contiguous_strides(shape[:3] + (D + pad,)), layout


def _cache(layout, dtype, nb, bs, H, D, pad):
    es = BYTES[dtype]
    if layout == VLLM:
        kv = (Layout.BLOCK_HND_PACKED, "bhdo")
    elif layout == PACKED_K:
        kv = (Layout.BLOCK_HND_PACKED, Layout.BLOCK_NHD)
    else:
        kv = (layout, layout)
    t = []
    for one in kv:
        shape, stride, code = _tensor(one, nb, bs, H, D, es, pad)
        t.append(abi._tensor(dtype, code, DEVICE, shape, stride, ADDR))
    return abi.cache_desc(nb, bs, H, D, *t)


def _scales(w):
    w.k_scale_desc = abi.scale_desc(ADDR)
    w.v_scale_desc = abi.scale_desc(ADDR)


def write(layout, cache, io, bs, H, D, T, *, nb=4096, pad=0) -> dict:
    c = _cache(layout, cache, nb, bs, H, D, pad)
    w = abi.make_write(T, H, D, io, DEVICE, ADDR, ADDR, DType.S64, ADDR)
    if cache != io:
        _scales(w)
    return _plan(lib().kvx_launch_write_kv(C.byref(c), C.byref(w), None))


def gather(layout, table, cache, io, bs, H, D, *, S=48, L=1200, entries=None, nb=8192,
           pad=0) -> dict:
    """table: "packed", "ragged" (`entries` of them, default S * L) or
    "offsets"."""
    c = _cache(layout, cache, nb, bs, H, D, pad)
    mbps = -(-L // bs)
    t = abi.make_block_table_packed(S, mbps, DType.S32, ADDR)
    if table == "ragged":
        t.format = int(TableFormat.RAGGED)
        t.indptr_dtype = int(DType.S32)
        t.max_blocks_per_seq = 1
        t.indptr = ADDR
        t.indices_count = S * L if entries is None else entries
        t.indptr_count = S + 1
    elif table == "offsets":
        t.format = int(TableFormat.KV_OFFSETS)
        t.indices_count = S * 2 * mbps
        t.flags = abi.TABLE_FLAG_KVCACHEINDEX
        c.pool.size = C.sizeof(abi.PoolDesc)
        c.pool.memory = int(DEVICE)
        c.pool.bytes_per_block = bs * H * (D + pad) * BYTES[cache]
        c.pool.primary = ADDR
    g = abi.make_gather(S, L, H, D, io, DEVICE, ADDR, ADDR, t,
                        abi.make_seq_lens(S, DType.S32, ADDR))
    if cache == io:
        return _plan(lib().kvx_launch_gather_kv(C.byref(c), C.byref(g), None))
    k, v = abi.scale_desc(ADDR), abi.scale_desc(ADDR)
    return _plan(lib().kvx_launch_gather_kv_dequant(C.byref(c), C.byref(g), C.byref(k),
                                                    C.byref(v), None))
