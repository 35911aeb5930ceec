// Stand-ins for the kernel families (kernels_*.hip) that launch nothing and
// write down what the launch planning chose: tests/dispatch_plan.py links
// them with the library's own abi.cpp, launch.cpp and dispatch.hip, compiled
// for the host only, so that the rules that pick a kernel can be tested
// without a GPU.  kvx_plan() returns the last plan as JSON.
#include <stdio.h>

#include <string>

#include "kernels.h"

namespace {
std::string g_plan = "{}";

void note(const char *kernel, const std::string &rest) {
  g_plan = std::string("{\"kernel\": \"") + kernel + "\"" + rest + "}";
}
std::string field(const char *name, int64_t v) {
  return std::string(", \"") + name + "\": " + std::to_string(v);
}
}  // namespace

extern "C" const char *kvx_plan() { return g_plan.c_str(); }

// Chunks in flight of the flat dequantizing gathers of `codes` codes.
extern "C" int kvx_flat_unroll(int codes, int f32) {
  using namespace kvx::dev;
  if (f32) return flat_unroll<DequantOp<4, KVX_DTYPE_F32, KVX_DTYPE_F8_E4M3>>();
  return codes == 4 ? flat_unroll<DequantOp<4, KVX_DTYPE_BF16, KVX_DTYPE_F8_E4M3>>()
                    : flat_unroll<DequantOp<8, KVX_DTYPE_BF16, KVX_DTYPE_F8_E4M3>>();
}

namespace kvx {
namespace dev {
namespace {

void plan_write(int chunk, const WriteArgs &a, const WriteLaunch &w) {
  if (!w.tiles) {
    note(w.flat_grid > 0 ? "write_flat" : "write", field("chunk", chunk));
    return;
  }
  std::string s = field("threads", w.tile_threads) + field("lds", w.tile_lds) + ", \"t\": [";
  for (int i = 0; i < 2; ++i) {
    const WriteTileTensor &t = w.wt.t[i];
    s += std::string(i ? ", " : "") + "{\"kind\": " + std::to_string(t.kind) +
         field("rows", t.rows) + field("tw", t.tw) + field("run", t.run) + field("seg", t.seg) +
         field("align", t.align) + field("workgroups", t.workgroups) + "}";
  }
  note("write_tiles", s + "]");
}

void plan_gather(int chunk, const GatherArgs &a) {
  const char *k = "gather_rows";
  if (a.format == KVX_BLOCK_TABLE_PACKED) {
    if (a.flat) k = "gather_flat";
  } else if (a.ragged_tile) {
    k = "gather_ragged_tile";
  } else {
    k = a.flat ? "gather_indexed_flat" : "gather_indexed";
  }
  note(k, field("chunk", chunk) + field("nchunks", a.nchunks) + field("rows", a.rows_per_wg));
}

void plan_tiles(const TileArgs &t) {
  note("gather_tiles", field("rows", 1 << t.bs_log2) + field("parts", 1 << t.parts_log2) +
                           field("tw", t.tw) + field("threads", t.threads));
}

}  // namespace

void run_write_copy(int chunk, const WriteArgs &a, const WriteLaunch &w, hipStream_t) {
  plan_write(chunk, a, w);
}
#define KVX_PLAN_WRITE(name) \
  void name(int ge, const WriteArgs &a, const WriteLaunch &w, hipStream_t) { plan_write(ge, a, w); }
KVX_PLAN_WRITE(run_write_quant_e4m3_f32)
KVX_PLAN_WRITE(run_write_quant_e4m3_f16)
KVX_PLAN_WRITE(run_write_quant_e4m3_bf16)
KVX_PLAN_WRITE(run_write_quant_e5m2_f32)
KVX_PLAN_WRITE(run_write_quant_e5m2_f16)
KVX_PLAN_WRITE(run_write_quant_e5m2_bf16)

void run_gather_copy(int chunk, const GatherArgs &a, int64_t, hipStream_t) {
  plan_gather(chunk, a);
}
#define KVX_PLAN_GATHER(name) \
  void name(int ge, const GatherArgs &a, int64_t, hipStream_t) { plan_gather(ge, a); }
KVX_PLAN_GATHER(run_gather_dequant_e4m3_f32)
KVX_PLAN_GATHER(run_gather_dequant_e4m3_f16)
KVX_PLAN_GATHER(run_gather_dequant_e4m3_bf16)
KVX_PLAN_GATHER(run_gather_dequant_e5m2_f32)
KVX_PLAN_GATHER(run_gather_dequant_e5m2_f16)
KVX_PLAN_GATHER(run_gather_dequant_e5m2_bf16)

void run_tiles_copy(const TileArgs &t, int, bool, bool, int64_t, uint32_t, hipStream_t) {
  plan_tiles(t);
}
void run_tiles_dequant_e4m3(int, const TileArgs &t, int, bool, bool, int64_t, uint32_t,
                            hipStream_t) {
  plan_tiles(t);
}
void run_tiles_dequant_e5m2(int, const TileArgs &t, int, bool, bool, int64_t, uint32_t,
                            hipStream_t) {
  plan_tiles(t);
}

}  // namespace dev
}  // namespace kvx
