// Host side of the int8 weight-only GEMMs (csrc/mo_gemm.hip): argument checks, module loading
// from the embedded gfx950 code object, the launch plans. C ABI: mo_int8_linear_forward/backward
// (the plan below) and mo_int8_strip_forward/backward (strip_plan, for calls with few rows).
//
// Launch plan: the large tile (256 x 256) carries the work; when its grid would leave the GPU's
// last round of workgroups less than half full, the rows of that partial round go to a second
// launch, and a grid smaller than one round of large tiles is such a launch alone. That launch
// uses the small tile (128 x 128, two workgroups a CU), or, with the weight-in-registers kernel
// and a workspace, the large tile with its reduction split: `splits` workgroups per tile, each
// over a contiguous part of the reduction, write fp32 planes to the workspace, and
// mo_int8_split_reduce adds them in split order and rounds. The large and small tiles add the
// same products in the same order, so moving rows between them does not change results; a
// split reduction rounds its sum differently, and the rows it computes are the same for any
// call with the same row count in that launch, features and device.
#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include <atomic>
#include <map>
#include <mutex>
#include <string>

#include "../../include/moss_offload.h"

extern "C" const unsigned char mo_gemm_code[];

namespace mo {
int set_error(int code, const std::string& msg);
int set_hip_error(int e, const char* what);
}  // namespace mo

namespace {

constexpr uint32_t kLarge = 256, kSmall = 128;  // output tile edges (mo_gemm.hip Cfg)

struct Kernel {
  hipFunction_t fn = nullptr;
  uint32_t threads = 0, tile = 0;
};

struct GemmModule {
  hipModule_t module = nullptr;
  int cus = 0;
  // [backward][small][tail]
  Kernel k[2][2][2];
  hipFunction_t decode = nullptr;     // mo_int8_decode_kernel
  hipFunction_t decode_transposed = nullptr;
  hipFunction_t ws_fwd = nullptr;     // mo_int8_ws_fwd: weight in registers, column scales
  hipFunction_t ws_kscale = nullptr;  // mo_int8_ws_kscale: the same on a transposed weight, per-k scales
  hipFunction_t transpose = nullptr;  // mo_int8_transpose_kernel
  hipFunction_t ws_fwd_split = nullptr, ws_kscale_split = nullptr, split_reduce = nullptr;
  hipFunction_t strip[2][5] = {};  // [backward][kStrips index]
};

// The strip kernels (mo_gemm.hip): output tile, K groups of a workgroup, and what the cost model
// knows of them on an MI355X, in us: a call's fixed part, and a step of 64 of every K group with
// one workgroup on a CU and with `resident` (all that fit). Fitted to 5 300 timed calls (64 to
// 5 500 rows of ten weight shapes, both directions, one to 32 splits): the model's choice takes
// 1.4 % longer than the fastest one on average, 18 % at worst.
struct Strip {
  const char* name;
  uint32_t bm, bn, k_groups;
  int resident;
  double fixed, alone, together;
};
constexpr int kStripCount = 5;
constexpr Strip kStrips[kStripCount] = {
    {"128x256", 128, 256, 1, 2, 6.0, 0.73, 1.38},    // wide grids
    {"128x256k2", 128, 256, 2, 1, 6.6, 1.40, 1.40},  // long reductions over few tiles
    {"128x128", 128, 128, 1, 3, 4.6, 0.55, 1.22},    // grids between one and two rounds
    {"64x64k4", 64, 64, 4, 1, 6.3, 0.67, 0.67},      // a 3 072-wide output of a few hundred rows
    {"32x64k4", 32, 64, 4, 2, 4.0, 0.49, 1.31},      // fewer rows than that
};
// Below 28 steps (reductions under 1792) a split gains nothing on the GPU (112 calls replayed from
// graphs: 0.87 to 1.20 of the unsplit time, 1.00 on average), and its second launch takes the host
// 5 us (24 rows of 192 from 1280: 18.6 us split, where the large-tile path takes 14.5).
constexpr uint32_t kMinStripSplit = 28;
constexpr double kStripReduce = 1.5, kStripReducePerMb = 0.28;  // the plane sum: fixed, per MB of planes

// Which kernel takes the large-tile rows of a launch plan (mo_int8_set_kernel).
std::atomic<uint32_t> g_kernel{MO_INT8_KERNEL_REGISTERS};

std::mutex g_mu;
std::map<int, GemmModule> g_modules;

int gemm_module(GemmModule* out) {
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return mo::set_hip_error((int)e, "hipGetDevice");
  std::lock_guard<std::mutex> lock(g_mu);
  auto it = g_modules.find(device);
  if (it == g_modules.end()) {
    GemmModule m;
    if ((e = hipModuleLoadData(&m.module, mo_gemm_code)) != hipSuccess)
      return mo::set_hip_error((int)e, "hipModuleLoadData (int8 GEMM code object)");
    if ((e = hipDeviceGetAttribute(&m.cus, hipDeviceAttributeMultiprocessorCount, device)) != hipSuccess)
      return mo::set_hip_error((int)e, "hipDeviceGetAttribute (CU count)");
    for (int bwd = 0; bwd < 2; ++bwd)
      for (int small = 0; small < 2; ++small)
        for (int tail = 0; tail < 2; ++tail) {
          const std::string name = std::string("mo_int8_linear_") + (bwd ? "bwd" : "fwd") + (small ? "_small" : "_large") +
                                   (tail ? "_tail" : "");
          Kernel& k = m.k[bwd][small][tail];
          if ((e = hipModuleGetFunction(&k.fn, m.module, name.c_str())) != hipSuccess)
            return mo::set_hip_error((int)e, "hipModuleGetFunction (int8 GEMM)");
          k.tile = small ? kSmall : kLarge;
          k.threads = small ? 256 : (bwd ? 256 : 512);  // waves of each configuration x 64
        }
    if ((e = hipModuleGetFunction(&m.decode, m.module, "mo_int8_decode_kernel")) != hipSuccess)
      return mo::set_hip_error((int)e, "hipModuleGetFunction (int8 decode)");
    if ((e = hipModuleGetFunction(&m.decode_transposed, m.module, "mo_int8_decode_transposed_kernel")) != hipSuccess)
      return mo::set_hip_error((int)e, "hipModuleGetFunction (int8 transposed decode)");
    if ((e = hipModuleGetFunction(&m.ws_fwd, m.module, "mo_int8_ws_fwd")) != hipSuccess ||
        (e = hipModuleGetFunction(&m.ws_kscale, m.module, "mo_int8_ws_kscale")) != hipSuccess ||
        (e = hipModuleGetFunction(&m.transpose, m.module, "mo_int8_transpose_kernel")) != hipSuccess ||
        (e = hipModuleGetFunction(&m.ws_fwd_split, m.module, "mo_int8_ws_fwd_split")) != hipSuccess ||
        (e = hipModuleGetFunction(&m.ws_kscale_split, m.module, "mo_int8_ws_kscale_split")) != hipSuccess ||
        (e = hipModuleGetFunction(&m.split_reduce, m.module, "mo_int8_split_reduce")) != hipSuccess)
      return mo::set_hip_error((int)e, "hipModuleGetFunction (int8 weight-in-registers kernels)");
    for (int bwd = 0; bwd < 2; ++bwd)
      for (int i = 0; i < kStripCount; ++i) {
        const std::string name = std::string("mo_int8_strip_") + (bwd ? "bwd_" : "fwd_") + kStrips[i].name;
        if ((e = hipModuleGetFunction(&m.strip[bwd][i], m.module, name.c_str())) != hipSuccess)
          return mo::set_hip_error((int)e, "hipModuleGetFunction (int8 strip)");
      }
    it = g_modules.emplace(device, m).first;
  }
  *out = it->second;
  return 0;
}

int check(uint64_t a, uint64_t w, uint64_t scale, uint64_t c, uint32_t rows, uint32_t in_f, uint32_t out_f) {
  if (!a || !w || !scale || !c) return mo::set_error(MO_E_INVALID, "null matrix pointer");
  if (rows == 0 || in_f == 0 || out_f == 0) return mo::set_error(MO_E_INVALID, "empty matrix");
  if (in_f % 16 || out_f % 16)
    return mo::set_error(MO_E_INVALID, "in_features and out_features must be multiples of 16 (got " +
                                           std::to_string(in_f) + ", " + std::to_string(out_f) + ")");
  if ((a | w | c) % 16) return mo::set_error(MO_E_INVALID, "matrix pointers must be 16-byte aligned");
  if (scale % 4) return mo::set_error(MO_E_INVALID, "scale pointer must be 4-byte aligned");
  // 32-bit buffer offsets: one tile's rows of either activation, and the whole weight
  if (in_f > (1u << 20) || out_f > (1u << 20) || (uint64_t)in_f * out_f >= (1ull << 31))
    return mo::set_error(MO_E_INVALID, "weight too large (in_features, out_features <= 2^20 and in * out < 2^31)");
  if ((uint64_t)rows * (out_f > in_f ? out_f : in_f) >= (1ull << 40)) return mo::set_error(MO_E_INVALID, "matrix too large");
  return 0;
}

enum class Tile { Large, Small, Split };

struct Part {
  Tile tile;
  uint32_t row0, rows;
  uint32_t splits, split_steps;  // Split: workgroups per tile, reduction steps (of 64) each
};

constexpr uint32_t kMinSplitSteps = 12;  // a split covers at least 12 x 64 of the reduction
constexpr uint32_t kLoopSteps = 6;       // the register kernel's loop runs steps in sixes

// The launch for rows [row0, row0 + n) that do not fill a round of large tiles: a split
// reduction on the large tile when `steps` (the reduction in steps of 64; 0 = no split) allows
// at least two splits of kMinSplitSteps, the tiles times the splits fit one round, and the
// rows fill at least three quarters of their large tiles; the small tile otherwise, and for an
// empty output (the workspace functions plan calls that the launches refuse). A split's
// length is rounded up to whole loop iterations (the last split takes what remains), which
// keeps the time of the longest split and launches fewer workgroups.
Part short_part(uint32_t row0, uint32_t n, uint32_t cols, uint32_t steps, int cus) {
  const uint64_t tm = (n + kLarge - 1) / kLarge, tiles = tm * ((cols + kLarge - 1) / kLarge);
  if (steps && tiles && 4ull * n >= 3ull * tm * kLarge && tiles <= (uint64_t)cus / 2) {
    uint64_t s = (uint64_t)cus / tiles;
    if (s > steps / kMinSplitSteps) s = steps / kMinSplitSteps;
    if (s >= 2) {
      uint32_t per = (uint32_t)((steps + s - 1) / s);
      per = (per + kLoopSteps - 1) / kLoopSteps * kLoopSteps;
      const uint32_t splits = (steps + per - 1) / per;
      if (splits >= 2) return {Tile::Split, row0, n, splits, per};
    }
  }
  return {Tile::Small, row0, n, 1, 0};
}

// Split [0, rows) between the large tile and a short launch (see the file comment).
int plan(uint32_t rows, uint32_t cols, uint32_t steps, int cus, Part parts[2]) {
  const uint64_t tm = (rows + kLarge - 1) / kLarge, tc = (cols + kLarge - 1) / kLarge, total = tm * tc;
  const uint64_t rounds = total / (uint64_t)cus, rem = total % (uint64_t)cus;
  if (rounds == 0) {
    parts[0] = short_part(0, rows, cols, steps, cus);
    return 1;
  }
  if (rem == 0 || 2 * rem >= (uint64_t)cus) {
    parts[0] = {Tile::Large, 0, rows, 1, 0};
    return 1;
  }
  const uint64_t main_rows = (rounds * (uint64_t)cus / tc) * kLarge;
  if (main_rows == 0) {
    parts[0] = {Tile::Small, 0, rows, 1, 0};
    return 1;
  }
  if (main_rows >= rows) {
    parts[0] = {Tile::Large, 0, rows, 1, 0};
    return 1;
  }
  parts[0] = {Tile::Large, 0, (uint32_t)main_rows, 1, 0};
  parts[1] = short_part((uint32_t)main_rows, rows - (uint32_t)main_rows, cols, steps, cus);
  return 2;
}

// fp32 planes of a plan's split launch (0 if it has none), rounded up to 256 bytes.
uint64_t split_bytes(const Part* parts, int n, uint32_t cols) {
  uint64_t b = 0;
  for (int p = 0; p < n; ++p)
    if (parts[p].tile == Tile::Split) b = (uint64_t)parts[p].splits * parts[p].rows * cols * 4;
  return (b + 255) & ~uint64_t(255);
}

// Reduction steps a split may use: the weight-in-registers kernel takes reductions of whole
// steps of 64 only.
uint32_t split_steps_of(uint32_t reduction) { return reduction % 64 ? 0 : reduction / 64; }

int cu_count(int* cus) {
  GemmModule m;
  if (int rc = gemm_module(&m)) return rc;
  *cus = m.cus;
  return 0;
}

int launch(const Kernel& k, void** params, uint32_t rows, uint32_t cols, uint64_t stream) {
  const uint64_t tiles_m = (rows + k.tile - 1) / k.tile, tiles_c = (cols + k.tile - 1) / k.tile;
  const uint64_t grid = tiles_m * tiles_c;
  if (grid >= (1ull << 31)) return mo::set_error(MO_E_INVALID, "grid too large");
  const hipError_t e =
      hipModuleLaunchKernel(k.fn, (uint32_t)grid, 1, 1, k.threads, 1, 1, 0, (hipStream_t)stream, params, nullptr);
  if (e != hipSuccess) return mo::set_hip_error((int)e, "int8 GEMM launch");
  return 0;
}

// The weight-in-registers kernels: 256 x 256 tiles, four waves.
Kernel registers_kernel(hipFunction_t fn) { return Kernel{fn, 256, kLarge}; }

// Sums a split launch's fp32 planes into C (rows x cols bf16; bias may be 0).
int launch_split_reduce(const GemmModule& m, uint64_t planes, uint64_t bias, uint64_t c, uint32_t rows, uint32_t cols,
                        uint32_t splits, uint64_t stream) {
  const void* P = (const void*)planes;
  const void* Bi = (const void*)bias;
  void* C = (void*)c;
  void* params[] = {&P, &Bi, &C, &rows, &cols, &splits};
  const uint64_t lanes = (uint64_t)rows * (cols / 8);
  const hipError_t e = hipModuleLaunchKernel(m.split_reduce, (uint32_t)((lanes + 255) / 256), 1, 1, 256, 1, 1, 0,
                                             (hipStream_t)stream, params, nullptr);
  if (e != hipSuccess) return mo::set_hip_error((int)e, "int8 split reduction launch");
  return 0;
}

// A split part: `splits` x tiles workgroups of the split kernel writing fp32 planes to `planes`,
// then the reduction into C (rows of the part, `cols` wide; bias may be 0).
int launch_split(const GemmModule& m, hipFunction_t fn, const Part& part, uint64_t a, uint64_t b, uint64_t scale,
                 uint64_t bias, uint64_t c, uint64_t planes, uint32_t cols, uint32_t reduction, uint64_t stream) {
  const uint64_t tiles_m = (part.rows + kLarge - 1) / kLarge, tiles_c = (cols + kLarge - 1) / kLarge;
  const void* A = (const void*)a;
  const void* B = (const void*)b;
  const void* S = (const void*)scale;
  void* P = (void*)planes;
  int M = (int)part.rows, N = (int)cols, K = (int)reduction, tm = (int)tiles_m, splits = (int)part.splits,
      per = (int)part.split_steps;
  void* params[] = {&A, &B, &S, &P, &M, &N, &K, &tm, &splits, &per};
  hipError_t e = hipModuleLaunchKernel(fn, (uint32_t)(tiles_m * tiles_c * part.splits), 1, 1, 256, 1, 1, 0,
                                       (hipStream_t)stream, params, nullptr);
  if (e != hipSuccess) return mo::set_hip_error((int)e, "int8 GEMM split launch");
  return launch_split_reduce(m, planes, bias, c, part.rows, cols, part.splits, stream);
}

// A strip call: shape, workgroups per tile and the reduction steps of 64 each covers.
struct StripPlan {
  int shape;
  uint32_t splits, split_steps;
};

uint64_t div_up(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// Modelled time (us) of a strip call with `splits` workgroups per tile, of `per` steps each.
double strip_cost(const Strip& s, uint32_t rows, uint32_t cols, uint32_t splits, uint32_t per, int cus) {
  const uint64_t each = div_up(div_up(rows, s.bm) * div_up(cols, s.bn) * splits, (uint64_t)cus);  // workgroups a CU
  const uint64_t rounds = each / s.resident, left = each % s.resident;
  const uint64_t steps = (div_up(per, s.k_groups) + 1) & ~1ull;  // the loop runs steps in pairs
  double step = (double)rounds * s.together;
  if (left) step += s.alone + (s.together - s.alone) * (double)(left - 1) / (s.resident > 1 ? s.resident - 1 : 1);
  double cost = s.fixed + (double)steps * step;
  if (splits > 1) cost += kStripReduce + kStripReducePerMb * (double)splits * rows * cols * 4e-6;
  return cost;
}

// The cheapest strip call. Splits: at most 32, of at least 6 steps, from reductions of kMinStripSplit
// steps on, while the workgroups stay within four and a half rounds of the CUs (more only pay for
// planes). The 64 x 64 tile, one workgroup a CU, only while its grid fits one round: past it the
// 32-row tile, two a CU, or the 128-row ones were faster at every size measured.
StripPlan strip_plan(uint32_t rows, uint32_t cols, uint32_t steps, int cus, bool may_split) {
  StripPlan best{0, 1, steps};
  double best_cost = 0;
  for (int i = 0; i < kStripCount; ++i) {
    const Strip& s = kStrips[i];
    const uint64_t tiles = div_up(rows, s.bm) * div_up(cols, s.bn);
    uint32_t tried = 0;
    for (uint32_t want = 1; want <= 32; ++want) {
      if (want > 1 && (!may_split || steps < kMinStripSplit || steps / want < 6 || 2 * tiles * want > 9ull * cus))
        break;
      const uint32_t per = (steps + want - 1) / want, splits = (steps + per - 1) / per;
      if (splits == tried) continue;
      tried = splits;
      if (s.bm == 64 && tiles * splits > (uint64_t)cus) break;
      const double cost = strip_cost(s, rows, cols, splits, per, cus);
      if (best_cost == 0 || cost < best_cost) {
        best = StripPlan{i, splits, per};
        best_cost = cost;
      }
    }
  }
  return best;
}

uint64_t strip_bytes(const StripPlan& p, uint32_t rows, uint32_t cols) {
  return p.splits > 1 ? ((uint64_t)p.splits * rows * cols * 4 + 255) & ~uint64_t(255) : 0;
}

int strip_check(uint64_t reduction) {
  if (reduction % 64) return mo::set_error(MO_E_INVALID, "strip kernels take reductions that are multiples of 64");
  return 0;
}

// One strip call: C[rows][cols] from a reduction of A's columns.
int strip_call(bool backward, uint64_t a, uint64_t w, uint64_t scale, uint64_t bias, uint64_t c, uint32_t rows,
               uint32_t cols, uint32_t reduction, uint64_t workspace, uint64_t workspace_bytes, uint64_t stream) {
  if (int rc = strip_check(reduction)) return rc;
  if (workspace % 16) return mo::set_error(MO_E_INVALID, "workspace pointer must be 16-byte aligned");
  GemmModule m;
  if (int rc = gemm_module(&m)) return rc;
  const StripPlan p = strip_plan(rows, cols, reduction / 64, m.cus, workspace != 0);
  if (workspace && workspace_bytes < strip_bytes(p, rows, cols))
    return mo::set_error(MO_E_INVALID, "workspace smaller than mo_int8_strip_workspace_bytes");
  const Strip& s = kStrips[p.shape];
  const uint64_t grid = div_up(rows, s.bm) * div_up(cols, s.bn) * p.splits;
  if (grid >= (1ull << 31)) return mo::set_error(MO_E_INVALID, "grid too large");
  const void* A = (const void*)a;
  const void* W = (const void*)w;
  const void* S = (const void*)scale;
  const void* Bi = (const void*)bias;
  void* C = (void*)c;
  void* P = (void*)workspace;
  int M = (int)rows, N = (int)cols, K = (int)reduction, splits = (int)p.splits, per = (int)p.split_steps;
  void* params[] = {&A, &W, &S, &Bi, &C, &P, &M, &N, &K, &splits, &per};
  const uint32_t threads = 64 * 4 * (s.bm == 128 ? s.k_groups : 1);  // 64-column tiles: one wave a K group
  const hipError_t e = hipModuleLaunchKernel(m.strip[backward][p.shape], (uint32_t)grid, 1, 1, threads, 1, 1, 0,
                                             (hipStream_t)stream, params, nullptr);
  if (e != hipSuccess) return mo::set_hip_error((int)e, "int8 strip launch");
  if (p.splits > 1) return launch_split_reduce(m, workspace, bias, c, rows, cols, p.splits, stream);
  return 0;
}

}  // namespace

extern "C" {

int mo_int8_decode_transposed(uint64_t w, uint64_t scale, uint64_t out, uint32_t out_features, uint32_t in_features,
                              uint64_t stream) {
  if (int rc = check(w, w, scale, out, 1, in_features, out_features)) return rc;
  GemmModule m;
  if (int rc = gemm_module(&m)) return rc;
  const void* q = (const void*)w;
  const void* sc = (const void*)scale;
  void* o = (void*)out;
  uint32_t rows = out_features, cols = in_features;
  void* params[] = {&q, &sc, &o, &rows, &cols};
  const uint32_t blocks = ((rows + 127) / 128) * ((cols + 127) / 128);
  const hipError_t e = hipModuleLaunchKernel(m.decode_transposed, blocks, 1, 1, 256, 1, 1, 0, (hipStream_t)stream,
                                             params, nullptr);
  if (e != hipSuccess) return mo::set_hip_error((int)e, "int8 transposed decode launch");
  return 0;
}

int mo_int8_decode(uint64_t w, uint64_t scale, uint64_t out, uint32_t out_features, uint32_t in_features,
                   uint64_t stream) {
  if (!w || !scale || !out) return mo::set_error(MO_E_INVALID, "null pointer");
  if (out_features == 0 || in_features == 0) return mo::set_error(MO_E_INVALID, "empty weight");
  if (in_features % 16) return mo::set_error(MO_E_INVALID, "in_features must be a multiple of 16");
  if ((w | out) % 16 || scale % 4) return mo::set_error(MO_E_INVALID, "misaligned pointer");
  if ((uint64_t)in_features * out_features >= (1ull << 31)) return mo::set_error(MO_E_INVALID, "weight too large");
  GemmModule m;
  if (int rc = gemm_module(&m)) return rc;
  const uint64_t chunks = (uint64_t)out_features * (in_features / 16);
  const void* q = (const void*)w;
  const void* sc = (const void*)scale;
  void* o = (void*)out;
  uint32_t rows = out_features, cols = in_features;
  void* params[] = {&q, &sc, &o, &rows, &cols};
  const hipError_t e = hipModuleLaunchKernel(m.decode, (uint32_t)((chunks + 255) / 256), 1, 1, 256, 1, 1, 0,
                                             (hipStream_t)stream, params, nullptr);
  if (e != hipSuccess) return mo::set_hip_error((int)e, "int8 decode launch");
  return 0;
}

uint64_t mo_int8_forward_workspace_bytes(uint32_t rows, uint32_t in_features, uint32_t out_features) {
  int cus = 0;
  if (cu_count(&cus)) return 0;
  Part parts[2];
  const int n = plan(rows, out_features, split_steps_of(in_features), cus, parts);
  return split_bytes(parts, n, out_features);
}

int mo_int8_linear_forward(uint64_t x, uint64_t w, uint64_t scale, uint64_t bias, uint64_t y, uint32_t rows,
                           uint32_t in_features, uint32_t out_features, uint64_t workspace, uint64_t workspace_bytes,
                           uint64_t stream) {
  if (int rc = check(x, w, scale, y, rows, in_features, out_features)) return rc;
  if (bias % 2) return mo::set_error(MO_E_INVALID, "bias pointer must be 2-byte aligned");
  if (workspace % 16) return mo::set_error(MO_E_INVALID, "workspace pointer must be 16-byte aligned");
  GemmModule m;
  if (int rc = gemm_module(&m)) return rc;
  const int tail = in_features % 64 != 0;
  const bool registers = !tail && g_kernel.load() == MO_INT8_KERNEL_REGISTERS;
  Part parts[2];
  const int n = plan(rows, out_features, registers && workspace ? split_steps_of(in_features) : 0, m.cus, parts);
  if (workspace && workspace_bytes < split_bytes(parts, n, out_features))
    return mo::set_error(MO_E_INVALID, "workspace smaller than mo_int8_forward_workspace_bytes");
  for (int p = 0; p < n; ++p) {
    const uint64_t a = x + (uint64_t)parts[p].row0 * in_features * 2;
    const uint64_t c = y + (uint64_t)parts[p].row0 * out_features * 2;
    if (parts[p].tile == Tile::Split) {
      if (int rc = launch_split(m, m.ws_fwd_split, parts[p], a, w, scale, bias, c, workspace, out_features,
                                in_features, stream))
        return rc;
      continue;
    }
    const bool small = parts[p].tile == Tile::Small;
    const Kernel k = !small && registers ? registers_kernel(m.ws_fwd) : m.k[0][small][tail];
    const void* A = (const void*)a;
    const void* B = (const void*)w;
    const void* S = (const void*)scale;
    const void* Bi = (const void*)bias;
    void* C = (void*)c;
    int M = (int)parts[p].rows, NC = (int)out_features, R = (int)in_features;
    int tiles_m = (int)((parts[p].rows + k.tile - 1) / k.tile);
    void* params[] = {&A, &B, &S, &Bi, &C, &M, &NC, &R, &tiles_m};
    if (int rc = launch(k, params, parts[p].rows, out_features, stream)) return rc;
  }
  return 0;
}

// The transposed int8 weight, then (when the plan splits a reduction) the fp32 planes.
uint64_t mo_int8_backward_workspace_bytes(uint32_t rows, uint32_t in_features, uint32_t out_features) {
  const uint64_t transposed = ((uint64_t)in_features * out_features + 255) & ~uint64_t(255);
  int cus = 0;
  if (cu_count(&cus)) return transposed;
  Part parts[2];
  const int n = plan(rows, in_features, split_steps_of(out_features), cus, parts);
  return transposed + split_bytes(parts, n, in_features);
}

int mo_int8_linear_backward(uint64_t dy, uint64_t w, uint64_t scale, uint64_t dx, uint32_t rows, uint32_t in_features,
                            uint32_t out_features, uint64_t workspace, uint64_t workspace_bytes, uint64_t stream) {
  if (int rc = check(dy, w, scale, dx, rows, in_features, out_features)) return rc;
  if (workspace % 16) return mo::set_error(MO_E_INVALID, "workspace pointer must be 16-byte aligned");
  GemmModule m;
  if (int rc = gemm_module(&m)) return rc;
  const int tail = out_features % 64 != 0;
  const bool registers = !tail && g_kernel.load() == MO_INT8_KERNEL_REGISTERS && workspace;
  const uint64_t transposed_bytes = ((uint64_t)in_features * out_features + 255) & ~uint64_t(255);
  Part parts[2];
  const int n = plan(rows, in_features, registers ? split_steps_of(out_features) : 0, m.cus, parts);
  if (workspace && workspace_bytes < transposed_bytes + split_bytes(parts, n, in_features))
    return mo::set_error(MO_E_INVALID, "workspace smaller than mo_int8_backward_workspace_bytes");
  bool transposed = false;
  for (int p = 0; p < n; ++p) {
    const bool small = parts[p].tile == Tile::Small;
    const bool ws = !small && registers;
    if (ws && !transposed) {
      // the weight with the reduction (out) contiguous, for the weight-in-registers kernels
      const void* src = (const void*)w;
      void* dst = (void*)workspace;
      uint32_t r = out_features, c = in_features;
      void* tparams[] = {&src, &dst, &r, &c};
      const uint64_t blocks = (uint64_t)((out_features + 127) / 128) * ((in_features + 127) / 128);
      const hipError_t e = hipModuleLaunchKernel(m.transpose, (uint32_t)blocks, 1, 1, 256, 1, 1, 0,
                                                 (hipStream_t)stream, tparams, nullptr);
      if (e != hipSuccess) return mo::set_hip_error((int)e, "int8 transpose launch");
      transposed = true;
    }
    const uint64_t a = dy + (uint64_t)parts[p].row0 * out_features * 2;
    const uint64_t c = dx + (uint64_t)parts[p].row0 * in_features * 2;
    if (parts[p].tile == Tile::Split) {
      if (int rc = launch_split(m, m.ws_kscale_split, parts[p], a, workspace, scale, 0, c,
                                workspace + transposed_bytes, in_features, out_features, stream))
        return rc;
      continue;
    }
    const Kernel k = ws ? registers_kernel(m.ws_kscale) : m.k[1][small][tail];
    const void* A = (const void*)a;
    const void* B = ws ? (const void*)workspace : (const void*)w;
    const void* S = (const void*)scale;
    void* C = (void*)c;
    int M = (int)parts[p].rows, NC = (int)in_features, R = (int)out_features;
    int tiles_m = (int)((parts[p].rows + k.tile - 1) / k.tile);
    void* params[] = {&A, &B, &S, &C, &M, &NC, &R, &tiles_m};
    if (int rc = launch(k, params, parts[p].rows, in_features, stream)) return rc;
  }
  return 0;
}

int mo_int8_launch_plan(uint32_t rows, uint32_t cols, uint32_t reduction, uint32_t cus, uint32_t kernel,
                        uint32_t* n_parts, uint32_t* parts) {
  if (!n_parts || !parts) return mo::set_error(MO_E_INVALID, "null output pointer");
  if (rows == 0 || cols == 0 || reduction == 0 || cus == 0) return mo::set_error(MO_E_INVALID, "empty shape");
  if (kernel != MO_INT8_KERNEL_REGISTERS && kernel != MO_INT8_KERNEL_LDS)
    return mo::set_error(MO_E_INVALID, "unknown int8 kernel selection");
  Part p[2];
  const uint32_t steps = kernel == MO_INT8_KERNEL_REGISTERS ? split_steps_of(reduction) : 0;
  const int n = plan(rows, cols, steps, (int)cus, p);
  for (int i = 0; i < n; ++i) {
    parts[5 * i + 0] = p[i].tile == Tile::Large ? 0u : p[i].tile == Tile::Small ? 1u : 2u;
    parts[5 * i + 1] = p[i].row0;
    parts[5 * i + 2] = p[i].rows;
    parts[5 * i + 3] = p[i].splits;
    parts[5 * i + 4] = p[i].split_steps;
  }
  *n_parts = (uint32_t)n;
  return 0;
}

uint64_t mo_int8_strip_workspace_bytes(uint32_t rows, uint32_t cols, uint32_t reduction) {
  int cus = 0;
  if (rows == 0 || cols == 0 || reduction == 0 || reduction % 64 || cu_count(&cus)) return 0;
  return strip_bytes(strip_plan(rows, cols, reduction / 64, cus, true), rows, cols);
}

int mo_int8_strip_forward(uint64_t x, uint64_t w, uint64_t scale, uint64_t bias, uint64_t y, uint32_t rows,
                          uint32_t in_features, uint32_t out_features, uint64_t workspace, uint64_t workspace_bytes,
                          uint64_t stream) {
  if (int rc = check(x, w, scale, y, rows, in_features, out_features)) return rc;
  if (bias % 2) return mo::set_error(MO_E_INVALID, "bias pointer must be 2-byte aligned");
  return strip_call(false, x, w, scale, bias, y, rows, out_features, in_features, workspace, workspace_bytes, stream);
}

int mo_int8_strip_backward(uint64_t dy, uint64_t w, uint64_t scale, uint64_t dx, uint32_t rows, uint32_t in_features,
                           uint32_t out_features, uint64_t workspace, uint64_t workspace_bytes, uint64_t stream) {
  if (int rc = check(dy, w, scale, dx, rows, in_features, out_features)) return rc;
  return strip_call(true, dy, w, scale, 0, dx, rows, in_features, out_features, workspace, workspace_bytes, stream);
}

int mo_int8_strip_plan(uint32_t rows, uint32_t cols, uint32_t reduction, uint32_t cus, uint32_t may_split,
                       uint32_t* plan) {
  if (!plan) return mo::set_error(MO_E_INVALID, "null output pointer");
  if (rows == 0 || cols == 0 || reduction == 0 || cus == 0) return mo::set_error(MO_E_INVALID, "empty shape");
  if (int rc = strip_check(reduction)) return rc;
  const StripPlan p = strip_plan(rows, cols, reduction / 64, (int)cus, may_split != 0);
  const Strip& s = kStrips[p.shape];
  plan[0] = s.bm, plan[1] = s.bn, plan[2] = s.k_groups, plan[3] = p.splits, plan[4] = p.split_steps;
  return 0;
}

int mo_int8_set_kernel(uint32_t kernel) {
  if (kernel != MO_INT8_KERNEL_REGISTERS && kernel != MO_INT8_KERNEL_LDS)
    return mo::set_error(MO_E_INVALID, "unknown int8 kernel selection");
  g_kernel.store(kernel);
  return 0;
}

}  // extern "C"
