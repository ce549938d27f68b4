// gqk_gemm_plan.hip - host side of the GEMM: the choice of tile geometry and schedule, its workspace.
#include "gqk_gemm.h"
#include <algorithm>
#include "gqk_common.h"

namespace gqk {

// CUs of the current device, cached per device
static int gb_cus() {
  static int cache[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cache[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 0;
    cache[dev] = n;
  }
  return cache[dev];
}

// Stream-K workgroups for R remainder tiles: at most G, at least four super-blocks per workgroup and
// at most 6 workgroups per tile.
static int64_t stream_k_workgroups(int G, int64_t R, int nb) {
  return std::max<int64_t>(1, std::min<int64_t>({(int64_t)G, R * nb / 4, 6 * R}));
}

static int64_t slot_bytes(int mb, int nr, int wk) { return (int64_t)((4 * mb + wk - 1) / wk) * 64 * nr * wk * 16; }

// The launch of a layer of n_desc descriptor rows at M rows: every geometry's time is estimated from its
// schedule and the cheapest taken.  A round of workgroups costs a start (descriptor, first weights and
// x, k-group combine, store) and its k-steps; split tiles add the exchange of partials.  The step times
// (us, one workgroup per CU) are fits to Q4_K and Q6_K launches over nine shapes (1000 x 4096 to
// 34816 x 5120, 5120 x 17408) at 40-1024 rows, each geometry forced in turn: the pick is within 5% of
// the best geometry in nine cases of ten and 1.2 times it at worst (so for eleven types and mixed layers,
// profiles/gemm_geometry_sweep.md).  Why more than one geometry (us,
// Q4_K): at 64 rows 34816 x 5120 takes 41.5 with 5 row blocks (218 workgroups, one round), 60.7 with 4
// (272: two rounds) and 52.0 with 8; 5120 x 17408 28.4 with 2 row blocks split 3 ways, 31.2 with 4
// split 6 ways, whose last contributor sums twice the partials; at 128 rows 38.6 (4 row blocks, 128
// tokens) against 54 (2 x 64 tokens, every weight decoded twice).
static GemmPick pick(int bm, int n_desc, int M, int nb, int cus) {
  GemmPick best{};
  double best_us = 1e30;
  const int per = bm == 256 ? 8 : 4;
  const int64_t blocks = (int64_t)n_desc * per;
  auto consider = [&](int mb, int nr, int wk, double step_us, double exch_us) {
    GemmPick p{};
    p.mb = mb, p.nr = nr, p.wk = wk, p.per = per, p.G = cus, p.S = 1;
    p.slot_bytes = slot_bytes(mb, nr, wk);
    const int64_t W = (blocks + nr - 1) / nr * ((M + 32 * mb - 1) / (32 * mb));
    double us;
    if (mb == 8) {   // persistent; its tiles are whole descriptor rows
      if (bm != 256) return;
      const int64_t R = W % cus;
      p.gsk = (int)stream_k_workgroups(cus, R, nb);
      p.grid = (int)(W >= cus ? cus : p.gsk);
      p.slots = R ? R + p.gsk - 1 : 0;
      // The whole rounds, then the remainder tiles on gsk workgroups: few of them where R or nb is small,
      // so that such a tail lasts as long as a round.  Spread over every workgroup in the estimate (as it
      // was) it hid: us, the form taken then -> now, at R = 2-56: Q4_K 33024 x 5120 at 384 rows 186 -> 176,
      // Q5_K 24778 x 1280 at 563 90 -> 70, IQ4_XS 18043 x 512 at 1094 76 -> 53, Q8_0 24140 x 256 at 564 77
      // -> 32.  After whole rounds the exchange waits for less (12 of 16 us: 16 took others 5-8% slower).
      us = 10. + (double)(W / cus) * 4 * nb * step_us +
           (R ? (double)R * nb / p.gsk * 4 * step_us + (W >= cus ? 0.75 : 1.) * exch_us : 0.);
    } else {
      int64_t S = 1;
      if (W < cus) S = std::max<int64_t>(1, std::min<int64_t>({cus / W, nb / wk, 8}));
      p.S = (int)S;
      p.slots = S > 1 ? W * S : 0;
      if (W * S > 0x7FFFFFFF) return;
      p.grid = (int)(W * S);
      const int64_t steps = 4 * (((nb + S - 1) / S + wk - 1) / wk);
      us = (double)((W * S + cus - 1) / cus) * (8. + steps * step_us) + (S > 1 ? exch_us * (1 + S * 0.25) : 0.);
    }
    if (us < best_us) best_us = us, best = p;
  };
  consider(2, 2, 4, 0.60, 3.);
  consider(2, 4, 4, 1.05, 3.);
  consider(2, 5, 3, 1.27, 3.);
  consider(4, 4, 2, 0.83, 4.);
  consider(4, 5, 2, 1.30, 4.);
  consider(8, 8, 1, 1.65, 16.);
  return best;
}

// Workspace of a launch: ctr_bytes of counters (the plan's counter region: at least G ints), then the
// partial slots.
static int64_t pick_bytes(const GemmPick& p, int64_t ctr_bytes) {
  return p.slots > 0 ? ctr_bytes + p.slots * p.slot_bytes : 0;
}

int64_t gemm_workspace(int bm, int n_desc, int M, int nb, int64_t ctr_bytes) {
  const int cus = gb_cus();
  if (cus <= 0) return -1;
  return pick_bytes(pick(bm, n_desc, M, nb, cus), ctr_bytes);
}

// Any M: the 256 x 256 tiles' remainder R <= G - 1 and their stream-K workgroups gsk <= G, so
// R + gsk - 1 <= 2 G - 2 slots; the split forms use at most one slot per CU, each smaller.
int64_t gemm_workspace_max() {
  const int cus = gb_cus();
  if (cus <= 0) return -1;
  return GQK_CTR_BYTES + (int64_t)(2 * cus - 2) * slot_bytes(8, 8, 1);
}

int gemm_pick(int bm, int n_desc, int M, int nb, int cus, int32_t* out) {
  if (bm != 64 && bm != 128 && bm != 256) return GQK_ERR_FORM;
  if (cus == 0) cus = gb_cus();
  if (cus <= 0) return GQK_ERR_HIP;
  const GemmPick p = pick(bm, n_desc, M, nb, cus);
  const int32_t v[7] = {p.mb, p.nr, p.wk, p.S, p.mb == 8 ? p.gsk : 0, p.grid, (int32_t)p.slots};
  for (int i = 0; i < 7; ++i) out[i] = v[i];
  return GQK_OK;
}

int launch_gemm(const uint8_t* packed, const int32_t* desc, int n_desc, int types_mask, const void* x, int64_t ldx,
                int M, int64_t K, void* y, int64_t ldy, const void* bias, int bm, int64_t ctr_bytes, void* ws,
                int64_t ws_bytes, hipStream_t st) {
  if (bm != 64 && bm != 128 && bm != 256) return GQK_ERR_FORM;
  const int nb = (int)(K / 256), cus = gb_cus();
  if (cus <= 0) return GQK_ERR_HIP;
  if ((int64_t)cus * 4 > ctr_bytes || (ctr_bytes & 255)) return GQK_ERR_FORM;
  const GemmPick p = pick(bm, n_desc, M, nb, cus);
  const int64_t need = pick_bytes(p, ctr_bytes);
  if (need > 0 && (ws == nullptr || ws_bytes < need || ((uintptr_t)ws & 255))) return GQK_ERR_SHAPE;
  int* ctr = need > 0 ? (int*)ws : nullptr;
  float* part = need > 0 ? (float*)((char*)ws + ctr_bytes) : nullptr;
  auto go = p.mb == 2 ? launch_gemm_mb2 : p.mb == 4 ? launch_gemm_mb4 : launch_gemm_mb8;
  return go(p, types_mask, n_desc, M, st, packed, desc, (const uint16_t*)x, ldx, (uint16_t*)y, ldy,
            (const uint16_t*)bias, part, ctr);
}

}  // namespace gqk
