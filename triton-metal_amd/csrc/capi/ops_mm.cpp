// Selection and launch of the pipelined MFMA matrix products (gemm_pipe.h),
// shared by tm_matmul / tm_linear and tm_dot.
#include <algorithm>
#include <cstdio>
#include <cstring>

#include "runtime.h"

using namespace tmhip;

namespace {

// Kernel arguments; must match struct MmParams in gemm_pipe.h.
struct MmParams {
  const void* A;
  const void* B;
  void* C;
  const void* Z;
  long long sa_b, sb_b, sc_b, sz_b;
  long long sc_m, sc_n, sz_m, sz_n;
  int M, N, K;
  int lda, ldb;
  int tiles_m, tiles_n;
  int epi;
  int out_dt, z_dt;
  int vec_z;
  int fix;
};

// Tile shapes 64 RT x 64 CT (the "d" form with a deeper ring of stages, for
// tiles that have a CU to themselves) and what they cost, fitted to times on
// one box (bf16 and e4m3, 64 to 4096 rows, K = 4096): one 128-byte k step takes
// t1 ns while few of the chip's CUs have a tile (the latency of a step) and
// tn * n once each has n of them (what the CU's LDS copies and the clock under
// full MFMA load allow); `res` tiles share a CU; fixed ns per round for the
// pipeline's fill and the epilogue.  The larger tile moves fewer bytes into LDS
// per MFMA, the smaller ones leave less of the last round idle and wait less
// where there are few tiles (256 CUs, the whole chip): us for 44 / 42 / 22 / 22d / 21 / 11, weights and
// activations coming from HBM
//   4096 x 4096 x 4096    117 / 137 / 144 / 159 / 179 / 234
//   2000 x 11008 x 4096   231 / 222 / 241 / 264 / 292 / 360
//   3000 x 2700 x 8000    184 / 207 / 217 / 199 / 214 / 232
//   1000 x 4096 x 4096     89 /  54 /  51 /  42 /  47 /  59
//   1136 x 1968 x 1024     28 /  17 /  14 /  11 /  12 /  13
//     64 x 8192 x 4096     76 /  48 /  47 /  33 /  30 /  22
struct TileCost {
  const char* name;
  int rt, ct, res;
  double t1, tn;    // 16-bit operands, ns
  double t1b, tnb;  // 8-bit
  double fixed;
};
const TileCost kTiles[] = {
    {"44", 4, 4, 1, 1000, 1560, 2200, 3000, 13500},
    {"42", 4, 2, 1, 600, 950, 1200, 1750, 5500},
    {"22", 2, 2, 2, 450, 590, 900, 920, 4000},
    {"22d", 2, 2, 1, 350, 600, 650, 950, 3300},
    {"21", 2, 1, 2, 300, 340, 550, 560, 2500},
    {"11", 1, 1, 2, 235, 215, 450, 360, 2000},
};

double tile_cost(const TileCost& t, long long tiles, int steps, bool fp8) {
  const double per_cu = tiles / 256.0;
  const long long up = (tiles + 255) / 256;  // tiles of the fullest CU
  const double t1 = fp8 ? t.t1b : t.t1, tn = fp8 ? t.tnb : t.tn;
  double step, rounds;
  if (up == 1) {
    step = std::max(t1, t1 + (tn - t1) * per_cu);
    rounds = 1;
  } else if (t.res == 1 || up <= 2 * t.res) {
    // rounds of res tiles, the last one perhaps of fewer
    const long long rest = up % t.res;
    step = tn * (up - rest) + (rest ? std::max(t1, tn * rest) : 0.0);
    rounds = (double)((up + t.res - 1) / t.res);
  } else {
    // many rounds: the CUs take tiles as they finish
    step = tn * per_cu * 1.03;
    rounds = per_cu / t.res;
  }
  return steps * step + t.fixed * rounds;
}

}  // namespace

namespace tmhip {

bool mm_plan(const MmCall& c, MmPlan* pl) {
  const bool fp8 = c.in_dt == TM_DT_FP8_E4M3 || c.in_dt == TM_DT_FP8_E5M2;
  if (!(is_half(c.in_dt) || fp8) || !is_float(c.out_dt) || c.K <= 0 || c.batch <= 0 ||
      c.batch > 65535 || c.M <= 0 || c.N <= 0)
    return false;
  if (c.Z && !is_float(c.z_dt)) return false;
  if (c.sc_n != 1) return false;
  const int es = fp8 ? 1 : 2, al = 16 / es, bk = 128 / es;
  // operands contiguous along k or along the rows.  The copies' 32-bit offsets
  // reach over one tile's rows or one step's k rows.  Pieces that no copy may
  // take whole are filled by elements (gemm_pipe.h): the one across K's end
  // of k-contiguous rows, and of row-contiguous operands that do not start on
  // 16 bytes the one across the end of the last k row.
  pl->fix = 0;
  const auto mode = [&](const void* p, long long sb, long long sr, long long sk, int kbit,
                        bool* rc) {
    const bool al16 = aligned16(p) && (c.batch == 1 || sb % al == 0);
    const long long lim = 0x7f000000LL / es;
    if ((uintptr_t)p % es) return false;
    if (sk == 1 && sr > 0 && sr < lim / 256 && c.K < lim / 2) {
      *rc = false;
      if (c.K % al) pl->fix |= kbit;
      return true;
    }
    if (sr == 1 && sk >= al && sk < lim / (bk + 1)) {  // a piece reaches into one more row at most
      *rc = true;
      if (!al16 || sk % al) pl->fix |= kbit << 2;
      return true;
    }
    return false;
  };
  if (!mode(c.A, c.sa_b, c.sa_m, c.sa_k, 1, &pl->arc) ||
      !mode(c.B, c.sb_b, c.sb_n, c.sb_k, 2, &pl->brc))
    return false;
  const int steps = (c.K + bk - 1) / bk;
  double best = 0;
  pl->tile = nullptr;
  for (const TileCost& t : kTiles) {
    const long long tm = (c.M + 64 * t.rt - 1) / (64 * t.rt), tn = (c.N + 64 * t.ct - 1) / (64 * t.ct);
    if (tm * tn > 0x7fffffffLL) continue;
    const double cost = tile_cost(t, tm * tn * c.batch, steps, fp8);
    if (pl->tile && cost >= best) continue;
    best = cost;
    pl->tile = t.name;
    pl->tiles_m = (int)tm;
    pl->tiles_n = (int)tn;
  }
  if (!pl->tile) return false;
  const char* dt = c.in_dt == TM_DT_F16    ? "f16"
                   : c.in_dt == TM_DT_BF16 ? "bf16"
                   : c.in_dt == TM_DT_FP8_E4M3 ? "e4m3" : "e5m2";
  snprintf(pl->name, sizeof pl->name, "mm_%s_%c%c_%s", dt, pl->arc ? 'r' : 'k',
           pl->brc ? 'r' : 'k', pl->tile);
  return true;
}

int mm_launch(const MmCall& c, const MmPlan& pl, void* stream) {
  MmParams p;
  memset(&p, 0, sizeof p);
  p.A = c.A; p.B = c.B; p.C = c.C; p.Z = c.Z;
  p.sa_b = c.sa_b; p.sb_b = c.sb_b; p.sc_b = c.sc_b; p.sz_b = c.sz_b;
  p.sc_m = c.sc_m; p.sc_n = c.sc_n; p.sz_m = c.sz_m; p.sz_n = c.sz_n;
  p.M = c.M; p.N = c.N; p.K = c.K;
  p.lda = (int)(pl.arc ? c.sa_k : c.sa_m);
  p.ldb = (int)(pl.brc ? c.sb_k : c.sb_n);
  p.tiles_m = pl.tiles_m; p.tiles_n = pl.tiles_n;
  p.epi = c.Z ? 1 : 0;
  p.out_dt = c.out_dt; p.z_dt = c.z_dt;
  p.vec_z = c.Z && c.sz_n == 1;
  p.fix = pl.fix;
  return launch(kernel_named(pl.name), dim3((unsigned)(pl.tiles_m * (long long)pl.tiles_n),
                                            (unsigned)c.batch),
                dim3(256), 0, stream, p);
}

}  // namespace tmhip
