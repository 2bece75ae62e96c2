// Host side of kernel (b), the skinny GEMM (the kernel itself is in qgemm_skinny_kernel.h,
// instantiated per quant type by qgemm_skinny_<type>.hip): tiles per wavefront, the grid, and the
// estimates that choose between it and the tiled kernel.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "qgemm_internal.h"
#include "qgemm_skinny_kernel.h"

namespace mlxr {

std::atomic<int> g_skinny_tiles{0}, g_skinny_waves{0}, g_skinny_splits{0};

namespace {

using namespace skinny;

const SkinnyKern& kern_for(int qtype, bool f16, int xr, int rt, int kg, bool sw, bool split) {
  switch (qtype) {
    case QT_Q4_K: return kern_q4k(f16, xr, rt, kg, sw, split);
    case QT_Q6_K: return kern_q6k(f16, xr, rt, kg, sw, split);
    case QT_Q5_K: return kern_q5k(f16, xr, rt, kg, sw, split);
    case QT_Q4_0: return kern_q40(f16, xr, rt, kg, sw, split);
    case QT_Q4_1: return kern_q41(f16, xr, rt, kg, sw, split);
    default: return kern_q80(f16, xr, rt, kg, sw, split);
  }
}

int rows_of_block(int M) { return M <= 8 ? 8 : M <= 16 ? 16 : 32; }

int current_device() {
  int dev = 0;
  return hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64 ? 0 : dev;
}
// Workgroups of k a CU of the current device holds, asked once per device (with the LDS limit
// raised); 0: an error, in *e.
int residents(const SkinnyKern& k, int dev, hipError_t* e) {
  int occ = k.residents[dev].load(std::memory_order_acquire);
  if (occ == 0) {
    if (k.lds > 65536) {
      *e = hipFuncSetAttribute(k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, k.lds);
      if (*e != hipSuccess) return 0;
    }
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k.fn, k.threads, (size_t)k.lds) != hipSuccess || occ <= 0)
      occ = 1;
    k.residents[dev].store(occ, std::memory_order_release);
  }
  return occ;
}

// How a launch is laid out: weight tiles of a wavefront, wavefronts of a workgroup (8, or 1 for short
// K), splits of K over workgroups, and its estimated time.
struct Plan {
  int rt, kg, ks;
  double us;
};

// Fitted to 17000 launches measured on MI355X (36 shapes of [512 .. 65536] x [512 .. 28672], fused SwiGLU of
// 12, M = 6 .. 2048, all types, weights from memory), to the times and to what the choices by them
// lose: 5% off on average; the variant chosen, tiled kernel included, is 0.15% slower than the best
// on average and more than 5% slower for 1% of the shapes.  us of a turn (one super-block for each
// of eight wavefronts) of a workgroup, by rows of X (8, 16, 32) and tiles (1, 2, 4), Q4_K; the
// workgroups of a CU take as many.  A lone wavefront's super-block takes kLoneLat + n * kLoneCu on a
// CU of n.  The other types by their dequantization.
constexpr double kTurn[3][3] = {{1.063, 2.184, 3.945}, {1.370, 2.437, 4.345}, {1.987, 2.910, 5.014}};
constexpr double kLoneLat[3][3] = {{0.421, 0.830, 2.321}, {0.534, 1.080, 2.314}, {0.698, 1.308, 2.071}};
constexpr double kLoneCu[3][3] = {{0.064, 0.220, 0.132}, {0.034, 0.133, 0.172}, {0.108, 0.170, 0.488}};
struct TypeCost {
  double turn[3], lone;
};
TypeCost type_cost(int qtype) {
  switch (qtype) {
    case QT_Q5_K: return {{1.115, 1.202, 1.212}, 1.200};
    case QT_Q6_K: return {{1.202, 1.295, 1.293}, 1.265};
    case QT_Q8_0: return {{1.092, 1.108, 1.120}, 1.045};
    case QT_Q4_0: return {{0.946, 0.937, 0.964}, 0.909};
    case QT_Q4_1: return {{0.945, 0.946, 0.975}, 0.892};
    default: return {{1.0, 1.0, 1.0}, 1.0};
  }
}
// What the weights' bytes take, MB/us (TB/s), by tiles (Q8_0, whose rows are read in 32-byte pieces,
// 1.31 times that), and the activations, read by every item: eight wavefronts, a lone one.
constexpr double kBytes[2][3] = {{4.113, 4.547, 4.693}, {4.521, 4.541, 11.461}};
constexpr double kXBytes[2] = {32.2, 15.5};

// us of a launch of `items` items of `turns` turns (kg = 1: super-blocks), `occ` workgroups on a CU.
// Whole rounds of the device's workgroups, then the rest: the first workgroups, neighbours on an
// XCD, take one item more.  A part of the weights' bytes is read from memory again by each further
// block of M.
double plan_us(int qtype, int xr, int rt, int kg, long items, long turns, int occ, long cus, int mblocks, double bytes,
               double xbytes) {
  const int x = xr == 8 ? 0 : xr == 16 ? 1 : 2, t = rt == 1 ? 0 : rt == 2 ? 1 : 2;
  const long slots = occ * cus;
  const long full = items / slots, rest = items % slots;
  const long n = full > 0 ? std::min<long>(occ, (rest + cus / 8 - 1) / (cus / 8)) : (rest + cus - 1) / cus;
  const TypeCost tc = type_cost(qtype);
  double a, m;
  if (kg == 1) {
    auto dur = [&](long n) { return n ? turns * (kLoneLat[x][t] + kLoneCu[x][t] * n) * tc.lone + 3.7 : 0.0; };
    // items after the first of their workgroup start with their operands loaded
    a = full > 0 ? dur(occ) + 0.73 * ((full - 1) * dur(occ) + dur(n)) : dur(n);
    m = (bytes * (0.81 + 0.19 * mblocks) / kBytes[1][t] + xbytes / kXBytes[1]) * 1e-6;
  } else {
    auto dur = [&](long n) { return n ? turns * kTurn[x][t] * tc.turn[t] * n + 0.74 : 0.0; };
    a = 2.67 + full * dur(occ) + dur(n);
    m = 2.67 + (bytes * (0.68 + 0.32 * mblocks) / (kBytes[0][t] * (qtype == QT_Q8_0 ? 1.31 : 1.0)) + xbytes / kXBytes[0]) * 1e-6;
  }
  return std::sqrt(std::sqrt(a * a * a * a + m * m * m * m));
}

// The plan of a launch: the fastest by plan_us.  (One rule on the items for three quarters of the CUs
// took two tiles for 5120 rows in two blocks of M, two rounds where four need one: Q4_K 5120 x
// 13824 at M = 33 47.4 us, at four tiles 36.9.)
// Eight wavefronts share a K of more than 1024, where the split of K and so the sums depend on K
// alone.  Up to 1024 each has at most one super-block, a lone wavefront takes them in the same
// order, and the sums are the same bits: a wide weight then need not meet in LDS once per item
// (Q4_K 65536 x 1024 at M = 8 20.4 -> 14.0 us, 16384 x 256 7.5 -> 4.2; 1536 x 1024 4.1 with eight
// wavefronts, 5.7 with one).
// With a workspace, a long K of a weight of few rows is split over workgroups too, which a second
// launch adds (Q4_K 1024 x 14336 at M = 16 12.4 -> 8.7 us; Q8_0 2048 x 14336 18.0 -> 15.3; 4096 x
// 14336 20.9, split 25.2).  Fewer than four turns pay for it at M = 17 .. 32 and in SwiGLU (Q8_0 896 x
// 4864 at M = 32 11.1 -> 8.8 us); elsewhere they gain 8% at most and stay whole.
Plan plan_for(const RunArgs* const* items, int n, bool swiglu) {
  const RunArgs& a = *items[0];
  const int M = a.M, K = a.L.K, xr = rows_of_block(M);
  const bool f16 = a.x_dtype == DT_F16;
  const int tiles = g_skinny_tiles.load(std::memory_order_relaxed), waves = g_skinny_waves.load(std::memory_order_relaxed),
            splits = g_skinny_splits.load(std::memory_order_relaxed);
  const int nsb = (K + 255) / 256, turns = (nsb + 7) / 8, dev = current_device();
  const long cus = device_cu_count();
  double bytes = 0;
  for (int i = 0; i < n; ++i) bytes += (double)items[i]->L.total;
  Plan best{0, 0, 0, 1e30};
  auto consider = [&](int rt, int kg, int ks) {
    const int rows = (swiglu ? 8 : 16) * rt;
    long slabs = 0;
    for (int i = 0; i < (swiglu ? 1 : n); ++i) slabs += (items[i]->L.N + rows - 1) / rows;
    hipError_t e;
    const int occ = std::max(1, residents(kern_for(a.L.qtype, f16, xr, rt, kg, swiglu, ks > 1), dev, &e));
    const long parts = (long)((M + xr - 1) / xr) * ks, nitems = slabs * parts;
    if (ks > 1 && (uint64_t)(nitems * parts) >= (1ull << 32)) return;
    const int mblocks = (M + xr - 1) / xr;
    double us = plan_us(a.L.qtype, xr, rt, kg, nitems, kg == 1 ? nsb : (turns + ks - 1) / ks, occ, cus, mblocks, bytes,
                        2.0 * slabs * mblocks * xr * K);
    if (ks > 1) us += 3.1 + (double)ks * M * a.L.N * (swiglu ? 16 : 8) / 6.3e6;  // the second launch
    if (us < best.us) best = Plan{rt, kg, ks, us};
  };
  for (int rt : {1, 2, 4}) {
    if (swiglu && rt == 1) continue;
    if (tiles && rt != (swiglu ? std::max(tiles, 2) : tiles)) continue;
    if (waves != 1 || K > 1024) consider(rt, 8, 1);
    if (waves != 8 && K <= 1024) consider(rt, 1, 1);
  }
  if ((n == 1 || swiglu) && a.ws && tiles == 0 && waves == 0 && (turns >= 4 || (M <= 32 && (M > 16 || swiglu)) || splits > 1)) {
    const size_t plane = (size_t)M * (size_t)a.L.N * (swiglu ? 8u : 4u);
    if (splits > 1) best.us = 1e30;
    for (int s = 2; s <= std::min(turns, 16); ++s) {
      const int tps = (turns + s - 1) / s, ks = (turns + tps - 1) / tps;
      if (ks == s && (splits == 0 || splits == s) && ks * plane <= a.ws_bytes) consider(swiglu ? 2 : 1, 8, ks);
    }
    if (best.us == 1e30) consider(swiglu ? 2 : 1, 8, 1);
  }
  return best;
}

hipError_t launch_any(const RunArgs* const* items, int n, bool swiglu, hipStream_t s) {
  SkinnyParams sp;
  const RunArgs& a = *items[0];
  const Plan pl = plan_for(items, n, swiglu);
  const int xr = rows_of_block(a.M), rows = (swiglu ? 8 : 16) * pl.rt, turns = (a.L.K + 256 * pl.kg - 1) / (256 * pl.kg);
  int slabs = 0;
  for (int i = 0; i < MAX_SG; ++i) {
    const RunArgs& b = *items[i < n ? i : 0];
    SkinnyGroup& g = sp.g[i];
    g.packed = b.packed;
    g.y = b.y;
    g.bias = b.bias;
    g.N = b.L.N;
    g.slab0 = slabs;
    g.y_dtype = b.y_dtype;
    g.bias_dtype = b.bias_dtype;
    const bool f32 = pl.ks > 1 || b.y_dtype == DT_F32;
    g.wide = (b.L.N & 3) == 0 && ((uintptr_t)(pl.ks > 1 ? a.ws : b.y) & (f32 ? 15u : 7u)) == 0;
    if (i < (swiglu ? 1 : n)) slabs += (b.L.N + rows - 1) / rows;
    if (swiglu) g.slab0 = 0;
  }
  sp.x = a.x;
  sp.M = a.M;
  sp.K = a.L.K;
  sp.ngroups = n;
  sp.parts = (a.M + xr - 1) / xr * pl.ks;
  sp.ks = pl.ks;
  sp.kdiv = pl.ks > 1 ? (uint32_t)(((1ull << 32) + pl.ks - 1) / pl.ks) : 0u;
  sp.mdiv = sp.parts > 1 ? (uint32_t)(((1ull << 32) + sp.parts - 1) / sp.parts) : 0u;
  sp.tps = (turns + pl.ks - 1) / pl.ks;
  sp.ws = pl.ks > 1 ? (float*)a.ws : nullptr;
  sp.ws_ld = (swiglu ? 2 : 1) * a.L.N;
  sp.ws_split = (size_t)a.M * (size_t)sp.ws_ld;
  const SkinnyKern& k = kern_for(a.L.qtype, a.x_dtype == DT_F16, xr, pl.rt, pl.kg, swiglu, pl.ks > 1);
  hipError_t e = hipSuccess;
  const int occ = residents(k, current_device(), &e);
  if (occ == 0) return e;
  const int nitems = slabs * sp.parts, grid = std::min(nitems, occ * device_cu_count());
  sp.per = nitems / grid;
  sp.rem = nitems % grid;
  void* args[1] = {&sp};
  e = hipLaunchKernel(k.fn, dim3((unsigned)grid), dim3((unsigned)k.threads), args, (size_t)k.lds, s);
  if (e != hipSuccess || pl.ks == 1) return e;
  const RunArgs& u = *items[n - 1];
  return swiglu ? launch_splitk_reduce_swiglu(sp.ws, sp.ws_split, pl.ks, a.bias, u.bias, a.bias_dtype, a.y, a.y_dtype,
                                              a.M, a.L.N, s)
                : launch_splitk_reduce(sp.ws, sp.ws_split, pl.ks, a.bias, a.bias_dtype, a.y, a.y_dtype, a.M, a.L.N, s);
}

// Splits of K that the workspace sizes reported for these calls hold (skinny_workspace_bytes).  The
// sizes stay what callers have been told, as they decide which calls mlxr_qgemm_run_noalloc
// takes; a launch uses as many of the splits as pay, or none.
int splits_of(int groups, int nkt, int steps) {  // at most `groups`, of whole `steps` of the nkt
  const int ks = std::max(1, std::min(groups, nkt / steps));
  const int per = ((nkt + ks - 1) / ks + steps - 1) / steps * steps;
  return (nkt + per - 1) / per;
}
// 64 rows of X, steps of 64: a workgroup of 32 weight rows per CU.
int sized_splits_wide(int M, int N, int K, int qtype) {
  const int slabs = (N + 31) / 32 * ((M + 63) / 64), cus = device_cu_count();
  return splits_of(slabs < cus ? cus / slabs : 1, (K + 63) / 64, qtype == QT_Q8_0 ? 4 : 8);
}
// Up to 32 rows, steps of 128: a workgroup of eight wavefronts per slab and CU where the slabs
// alone are fewer than half of that.
int sized_splits_narrow(int slabs, int K) {
  const int cus = device_cu_count();
  return splits_of(2L * slabs <= cus ? (cus + slabs - 1) / slabs : 1, (K + 127) / 128, 4);
}

}  // namespace

hipError_t launch_skinny(const RunArgs& a, hipStream_t s) {
  const RunArgs* items[1] = {&a};
  return launch_any(items, 1, false, s);
}
hipError_t launch_skinny_grouped(const RunArgs* const* items, int n, hipStream_t s) {
  return launch_any(items, n, false, s);
}
hipError_t launch_skinny_swiglu(const RunArgs& gate, const RunArgs& up, hipStream_t s) {
  RunArgs u = up;
  u.y = gate.y;
  const RunArgs* items[2] = {&gate, &u};
  return launch_any(items, 2, true, s);
}

double skinny_us(const RunArgs* const* items, int n, bool swiglu) { return plan_for(items, n, swiglu).us; }
void skinny_layout(const RunArgs* const* items, int n, bool swiglu, int* layout) {
  const Plan pl = plan_for(items, n, swiglu);
  layout[0] = pl.rt;
  layout[1] = pl.kg;
  layout[2] = pl.ks;
}

size_t skinny_swiglu_workspace_bytes(int M, int N, int K) {
  const int ks = sized_splits_narrow((N + 15) / 16, K);
  return ks > 1 ? (size_t)ks * (size_t)M * (size_t)N * 8u : 0;
}

namespace {
// The kernel divides an item by the blocks of M with a multiplication (mdiv), which is exact while
// items x blocks is below 2^32; one tile per wavefront has the most items.
bool items_fit(int64_t slabs, int M) {
  const uint64_t mb = ((uint64_t)M + 31) / 32;
  return (uint64_t)slabs * mb * mb < (1ull << 32);
}
}  // namespace

bool skinny_fits(const RunArgs& a) {
  const size_t lim = operand_limit();
  if ((size_t)a.M * (size_t)a.L.K * 2u >= lim) return false;
  for (int i = 0; i < a.L.nplanes; ++i)
    if (a.L.size[i] >= lim) return false;
  return items_fit((a.L.N + 15) / 16, a.M);
}

bool skinny_group_fits(const RunArgs* const* items, int n) {
  int64_t slabs = 0;
  for (int i = 0; i < n; ++i) {
    if (!skinny_fits(*items[i])) return false;
    slabs += (items[i]->L.N + 15) / 16;
  }
  return items_fit(slabs, items[0]->M);
}

double skinny_sizing_us(int M, int N, int K) {
  // each 32-row slab reads its 64-row blocks of X from L2 (~7.5 TB/s device-wide), plus
  // ~8 us of launch, prologue and epilogue (measured on MI355X, Llama-3-8B shapes)
  return 8.0 + (double)((N + 31) / 32) * M * K * 2.0 / 7.5e6;
}

size_t skinny_workspace_bytes(int M, int N, int K, int qtype) {
  const int ks = M <= 32 ? sized_splits_narrow((N + 31) / 32, K) : sized_splits_wide(M, N, K, qtype);
  return ks > 1 ? (size_t)ks * (size_t)M * (size_t)N * 4u : 0;
}

}  // namespace mlxr
