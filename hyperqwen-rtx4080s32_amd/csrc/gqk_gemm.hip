// gqk_gemm.hip - the grouped dequant-GEMM (batch rows M > 32, the prefill regime).
//
// Replaces the reference's prefill paths: the wide int8 forms of the grouped kernel and, for
// Q4_K / Q5_K, dequantize_tiles + cuBLAS bf16 (gguf-plugin/gluon/interface.py:159-188,
// gguf-plugin/gluon/tiles.py:141-149).
//
// A tile is 32 MB tokens x 32 NR weight rows.  NR waves own one 32-row block each and all of the tile's
// tokens; WK groups of such waves split the tile's k-range.  Each lane decodes its row's weights of a
// 64-weight step to bf16 (round-to-nearest-even of the exact fp32 gguf-py value) straight into the B
// operand of v_mfma_f32_32x32x16_bf16, so a weight is decoded once per tile, never stored to LDS, and
// no wave waits for another's decode.  The activations are the shared operand: each k-group's stage of
// x (32 MB tokens x 64 k) goes to LDS by direct-to-LDS buffer loads, four stages deep, one barrier a
// step.  The groups' sums meet in LDS at the end of the tile.
//
// What bounds it (Q4_K 34816 x 5120 and 5120 x 17408, copies of the kernel with one part taken out):
// at 64 rows, 43 us, start, combine and store take 9, the MFMAs alone 15 more, the weights' latency 11,
// the decode 10; at 2048 rows, 629 us, MFMAs alone take 490 (the chip holds ~1.8 GHz there), x through
// LDS 90, the decode 30-90, the remainder tiles' exchange 30-40.  The form this replaced staged the
// decoded weights in LDS behind a barrier per step, 128 rows per workgroup with up to six workgroups
// per tile: us before -> now, Q4_K at 64 / 128 / 200 / 512 / 2048 rows: 34816 x 5120 57 -> 42, 76 -> 61,
// 122 -> 109, 215 -> 197, 701 -> 650; 5120 x 17408 44 -> 28, 54 -> 40, 81 -> 60, 129 -> 108, 360 -> 328;
// 5120 x 5120 23 -> 15, 29 -> 19, 40 -> 28, 49 -> 44, 131 -> 125 (eleven types at 64 / 128 rows:
// 1.1-1.7 times as fast).
//
// This file is compiled once per token-block count GQK_GEMM_MB (MB).
#include "gqk_gemm.h"
#include "gqk_tile.h"

namespace gqk {

// Where a tile's accumulators go: straight to y (part == nullptr), or - for a tile whose k-steps
// are shared by several workgroups (stream-K) - to this workgroup's fp32 partial slot, the last
// contributor to arrive summing every slot in k order (deterministic) and writing y.
struct GOut {
  float* part;   // partial slots, BM x BN fp32 each
  int* ctr;      // the tile's arrival counter (zero at rest, reset by the last contributor)
  int slot0;     // slot of the tile's first contributor
  int nc;        // contributors
  int self;      // this workgroup's index among them
};

// The geometries (gqk_gemm.h lists them).  One workgroup per CU: its k-groups' stages fill the LDS (MB
// of 2 and 4) or its accumulators the registers (MB = 8: 128 of 256 a lane at two waves per SIMD).
// Four stages: a step multiplies one, the next is complete at its barrier (so its first fragments load
// before the barrier after), two are in flight.
template <int MB_, int NR_, int WK_>
struct Geo {
  static constexpr int MB = MB_, NR = NR_, WK = WK_, NW = NR * WK, BM = 32 * MB, BN = 32 * NR, NT = 64 * NW;
  static constexpr int D = 4;                       // x stages in LDS
  static constexpr int STG = BM * GB_K;             // bf16 per stage
  static constexpr int XN = BM * GB_K * 2 / 1024;   // 1 KiB x loads per stage,
  static constexpr int XI = (XN + NR - 1) / NR;     // per wave (the last ones may double up)
  static constexpr int LDS = WK * D * STG * 2;
  static constexpr int CH = (MB * 4 + WK - 1) / WK;   // 16-byte accumulator chunks per thread after the combine
  static constexpr int SLOT = CH * NT * 4;          // floats of a partial slot
  static constexpr int WPE = (NW + 3) / 4;          // waves per SIMD: one workgroup per CU
  static constexpr int PS = MB == 4 && WK > 1 ? 2 : 1;           // passes of the k groups' sums through LDS
  static constexpr int RED = WK > 1 ? WK * NR * MB * 4096 / PS : 0;
  static constexpr int LDSX = LDS > RED ? LDS : RED;
  static_assert(LDSX + 6160 <= 163840, "LDS");
};

// One wave's share of a tile: block rb (32 rows) of descriptor row dsc, tokens m0 .. m0 + 32 MB - 1,
// super-blocks [b0, b1) split over the k-groups.  x comes by buffer loads, not global ones: the
// compiler counts a global direct-to-LDS load as a flat access and drains every load before the next
// LDS read (measured: 684 -> 655 us at 2048 rows); the weights too (scalar base + one lane offset: no
// address registers).  FAR: rows of x further apart than 32-bit byte offsets from the tile's first one
// reach (GQK_MAX_LDX) come by global loads from a 64-bit address each (Q4_K 5120 x 5120 at 64 / 128 rows
// 20 MiB apart 15.3 / 23.1 us; near rows 14.6 / 19.6, a launch per row 1054 / 2105).
template <class GE, int T, bool FAR>
__device__ __forceinline__ void gemm_tile(const uint8_t* __restrict__ packed, const int32_t* __restrict__ dsc,
                                        int rb, const uint16_t* __restrict__ x, int64_t ldx, int M, int m0, int b0, int b1,
                                        const GOut& go, uint16_t* __restrict__ y, int64_t ldy,
                                        const uint16_t* __restrict__ bias, uint16_t* xlds, int* flag, const GTabs& tb) {
  constexpr int REC = gqk_layout<T>::REC, MB = GE::MB, NT = GE::NT, XI = GE::XI, NR = GE::NR, WK = GE::WK, CH = GE::CH;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave % NR, wg = wave / NR;   // row block, k group
  const int r = lane & 31, h = lane >> 5;
  const int nb = dsc[D_NB], ntiles = dsc[D_NTILES];
  const int64_t off = (int64_t)(uint32_t)dsc[D_OFF_LO] | ((int64_t)dsc[D_OFF_HI] << 32);
  const int64_t tile0 = dsc[D_TILE0];
  const int btile = rb >> 1, brow = 32 * (rb & 1) + r;   // the wave's 32-row block of the descriptor row
  const uint8_t* wb = packed + g_uniform(off + (tile0 + (btile < ntiles ? btile : 0)) * nb * (int64_t)(64 * REC));
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc((void*)(x + (int64_t)m0 * ldx), 0, 0xFFFFFFFFu, GQK_GB_WORD3);
  std::conditional_t<FAR, int64_t, uint32_t> xoff[XI];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int row = 8 * min(wr + NR * i, GE::XN - 1) + (lane >> 3);
    xoff[i] = min(row, M - 1 - m0) * (decltype(+xoff[i]))(2 * ldx) + 16u * ((lane & 7) ^ ((row >> 1) & 7));
  }
  uint16_t* xs = xlds + wg * (GE::D * GE::STG);
  const int koff[4] = {B2<T>::off0(h), B2<T>::off0(h) + 8, B2<T>::off1(h), B2<T>::off1(h) + 8};
  const int swz = (r >> 1) & 7;
  typedef const __attribute__((address_space(3))) uint8_t* lptr;
  lptr xq[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) xq[q] = (lptr)(const void*)xs + r * (2 * GB_K) + ((koff[q] >> 3) ^ swz) * 16;

  v16f acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
  // the group's super-blocks
  const int n = b1 - b0, g0 = b0 + wg * n / WK, g1 = b0 + (wg + 1) * n / WK, nmax = (n + WK - 1) / WK;
  const int last = 4 * g1 - 1;
  B2<T> w0, w1, w2, w3;
  v8bf A[MB];
  auto dma = [&](int buf, int s) __attribute__((always_inline)) {
#ifdef __HIP_DEVICE_COMPILE__   // the host pass rejects 16-byte direct-to-LDS loads
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const auto to = (__attribute__((address_space(3))) void*)(xs + buf * GE::STG + 512 * min(wr + NR * i, GE::XN - 1));
      if constexpr (FAR)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)((const uint8_t*)(x + (int64_t)m0 * ldx) + xoff[i] + (int64_t)s * (2 * GB_K)),
            to, 16, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, to, 16, xoff[i], s * (2 * GB_K), 0, 0);
    }
#endif
  };
  auto aread = [&](lptr b, int i) __attribute__((always_inline)) {
    return *(const __attribute__((address_space(3))) v8bf*)(b + 64 * GB_K * i);
  };
  // the chunk-q base of a stage (one add, where the compiler would re-derive it per read)
  auto abase = [&](int buf, int q) __attribute__((always_inline)) {
    lptr b = xq[q] + buf * (2 * GE::STG);
    if (buf * 2 * GE::STG + 64 * GB_K * (MB - 1) > 65535) asm("" : "+v"(b));
    return b;
  };
  // Half P of a step's decode: quarters 2P, 2P + 1 of out(), the B operands of MFMA slices 2P and
  // 2P + 1 in the order qs[] (a decoder that fills o in order gives slices 2P, 2P + 1; the others
  // P and P + 2).
  constexpr bool SEQ = b2_seq<B2<T>>::value;
  constexpr int qs[4] = {0, SEQ ? 1 : 2, SEQ ? 2 : 1, 3};
  struct Half { uint32_t o[8]; };
  auto half = [&](auto P, const B2<T>& w, const GS& st, int kq, Half& d, int part) __attribute__((always_inline)) {
    constexpr int p = decltype(P)::value;
    uint32_t o[16];
    w.out(st, kq, h, o, tb, 2 * p + part);
    if constexpr (SEQ) {
#pragma unroll
      for (int k = 0; k < 4; ++k) d.o[4 * part + k] = o[4 * (2 * p + part) + k];
    } else {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        d.o[2 * part + k] = o[2 * (2 * p + part) + k];
        d.o[4 + 2 * part + k] = o[8 + 2 * (2 * p + part) + k];
      }
    }
  };
  Half ba, bb;
  GS st;
  // Step j of super-block sb: w holds its raw weights, wn those of the next step; ba holds half 0
  // decoded.  wl takes the weights three steps ahead.
  auto step = [&](auto J, int sb, const B2<T>& w, const B2<T>& wn, B2<T>& wl) __attribute__((always_inline)) {
    constexpr int j = decltype(J)::value;
    const int s = 4 * sb + j;
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(XI + 2) : "memory");
    dma((j + 3) & 3, min(s + 3, last));
    __builtin_amdgcn_sched_barrier(0);
    uint32_t z = 0;   // opaque: every step issues its own loads (the barrier's count relies on it)
    asm volatile("" : "+s"(z));
    wl.load(g_src(wb + (int64_t)(j < 1 ? sb : min(sb + 1, g1 - 1)) * (64 * REC)) + z, brow, (j + 3) & 3, h);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const lptr nb_ = t < 3 ? abase(j, qs[t + 1]) : abase((j + 1) & 3, 0);
      const Half& d = t < 2 ? ba : bb;
      const v8bf B = __builtin_bit_cast(v8bf, v4u{d.o[4 * (t & 1)], d.o[4 * (t & 1) + 1], d.o[4 * (t & 1) + 2], d.o[4 * (t & 1) + 3]});
      if (t == 2) st = wn.prep((j + 1) & 3, h);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[i], B, acc[i], 0, 0, 0);
        A[i] = aread(nb_, i);
        if constexpr (MB > 2) __builtin_amdgcn_sched_barrier(0);
      }
      if (t < 2) half(std::integral_constant<int, 1>{}, w, st, j, bb, t);
      else half(std::integral_constant<int, 0>{}, wn, st, (j + 1) & 3, ba, t - 2);
    }
  };
  if (g0 < g1) {
    const GSrc c0 = g_src(wb + (int64_t)g0 * (64 * REC));
    w0.load(c0, brow, 0, h);
    w1.load(c0, brow, 1, h);
    w2.load(c0, brow, 2, h);
    __builtin_amdgcn_sched_barrier(0);
    dma(0, 4 * g0);
    dma(1, 4 * g0 + 1);
    dma(2, 4 * g0 + 2);
    __builtin_amdgcn_sched_barrier(0);
    st = w0.prep(0, h);
    half(std::integral_constant<int, 0>{}, w0, st, 0, ba, 0);
    half(std::integral_constant<int, 0>{}, w0, st, 0, ba, 1);
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(XI) : "memory");   // x of the first two steps
#pragma unroll
  for (int i = 0; i < MB; ++i) A[i] = aread(xq[0], i);
  int it = 0;
  // Before step s' barrier a wave's part of x(s + 1) is in LDS: after its loads (two steps ago) the
  // wave issued x(s + 2) and two steps' weights, so x(s + 1) is complete when at most XI + 2 loads are
  // outstanding (memory operations complete in order).  At the second step only the first one's weights
  // follow x(s + 1): the count needs two weight loads a step, which every decoder issues.
  for (int sb = g0; sb < g1; ++sb, ++it) {
    step(std::integral_constant<int, 0>{}, sb, w0, w1, w3);
    step(std::integral_constant<int, 1>{}, sb, w1, w2, w0);
    step(std::integral_constant<int, 2>{}, sb, w2, w3, w1);
    step(std::integral_constant<int, 3>{}, sb, w3, w0, w2);
  }
  if constexpr (WK > 1)
    for (; it < nmax; ++it)   // a group with one super-block less meets the others' barriers
#pragma unroll
      for (int j = 0; j < 4; ++j) asm volatile("s_barrier" ::: "memory");
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // C block i: lane -> row 32 rb + r, tokens 32 i + 8 (v / 4) + 4 h + v % 4: 16-byte chunk e = 4 i + v / 4.
  // The k groups' sums meet in LDS (over the x stages), PS passes of EP chunks; group wg keeps CP of
  // each pass.
  constexpr int PS = GE::PS, EP = 4 * MB / PS, CP = CH / PS;
  v4f out[CH];
  auto chunk = [&](int e) __attribute__((always_inline)) {
    return v4f{acc[e >> 2][4 * (e & 3)], acc[e >> 2][4 * (e & 3) + 1], acc[e >> 2][4 * (e & 3) + 2], acc[e >> 2][4 * (e & 3) + 3]};
  };
  if constexpr (WK > 1) {
    v4f* red = (v4f*)xlds;   // [group][chunk][row wave][lane]
#pragma unroll
    for (int p = 0; p < PS; ++p) {
#pragma unroll
      for (int e = 0; e < EP; ++e) red[((wg * EP + e) * NR + wr) * 64 + lane] = chunk(p * EP + e);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int c = 0; c < CP; ++c) {
        const int e = EP % WK == 0 ? wg * CP + c : min(wg * CP + c, EP - 1);
        v4f a = red[(e * NR + wr) * 64 + lane];
#pragma unroll
        for (int g = 1; g < WK; ++g) a += red[((g * EP + e) * NR + wr) * 64 + lane];
        out[p * CP + c] = a;
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the next pass or tile refills the region
    }
  } else {
#pragma unroll
    for (int c = 0; c < CH; ++c) out[c] = chunk(c);
  }
  const int nvalid = dsc[D_NVALID];
  const int64_t col0 = dsc[D_COL0];
  const int row = 32 * rb + r;
  // first token of chunk c (chunks past the tile's: none)
  auto tok = [&](int c) {
    const int e = wg * CP + c % CP;
    return EP % WK == 0 || e < EP ? m0 + 8 * (c / CP * EP + e) + 4 * h : M;
  };
  auto store_y = [&](int c, const v4f& a, float bv) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int t = tok(c) + v;
      if (t < M) y[(int64_t)t * ldy + col0 + row] = __builtin_bit_cast(uint16_t, (__bf16)(a[v] + bv));
    }
  };
  // the layer bias (bf16 per output column) joins before the one rounding to bf16
  const float bv = bias != nullptr && row < nvalid ? __builtin_bit_cast(float, (uint32_t)bias[col0 + row] << 16) : 0.f;
  if (go.part == nullptr) {
    if (row < nvalid)
#pragma unroll
      for (int c = 0; c < CH; ++c) store_y(c, out[c], bv);
    return;
  }
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      go.part + (int64_t)go.slot0 * GE::SLOT, 0, go.nc * GE::SLOT * 4, GQK_GB_WORD3);
  auto slot_off = [&](int q, int c) { return ((q * CH + c) * NT + tid) * 16; };
  if (tid == 0) *flag = __hip_atomic_load(go.ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const bool last_now = *flag == go.nc - 1;
  __syncthreads();
  if (!last_now) {
#pragma unroll
    for (int c = 0; c < CH; ++c)
      if (tok(c) < M && row < nvalid) __builtin_amdgcn_raw_buffer_store_b128(out[c], rs, slot_off(go.self, c), 0, GQK_GB_SC1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) *flag = __hip_atomic_fetch_add(go.ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*flag != go.nc - 1) return;
  }
  asm volatile("" ::: "memory");
  // the last contributor: slot 0 + slot 1 + ... in k order (its own from registers), the loads of CB
  // chunks of QB slots in flight together, unconditional (slot clamped to the last): chunks never
  // written only reach sums that are never stored
  constexpr int QB = CH >= 4 ? 2 : 4, CB = CH < 8 ? CH : 8;
#pragma unroll
  for (int c0 = 0; c0 < CH; c0 += CB) {
    v4f sum[CB];
    for (int q0 = 0; q0 < go.nc; q0 += QB) {
      v4f t[QB][CB];
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int c = 0; c < CB; ++c)
          t[b][c] = __builtin_amdgcn_raw_buffer_load_b128(rs, slot_off(min(q0 + b, go.nc - 1), c0 + c), 0, GQK_GB_SC1);
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        const int q = q0 + b;
        if (q < go.nc) {
#pragma unroll
          for (int c = 0; c < CB; ++c) {
            const v4f v = q == go.self ? out[c0 + c] : t[b][c];
            sum[c] = q == 0 ? v : sum[c] + v;
          }
        }
      }
    }
    if (row < nvalid)
#pragma unroll
      for (int c = 0; c < CB; ++c) store_y(c0 + c, sum[c], bv);
  }
  if (tid == 0) __hip_atomic_store(go.ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Tile t -> (descriptor row, token block).  Groups of up to eight token blocks take consecutive
// tile ids, so with tiles dealt round robin to the workgroups and the dispatcher's round robin
// over the eight XCDs, each XCD keeps one token block of x hot in its L2 while the weight blocks
// stream by.
__device__ __forceinline__ void gb_map(int i, int n_desc, int nmb, int& d, int& mb) {
  const int full = (nmb / 8) * 8 * n_desc;
  if (i < full) {
    const int grp = i / (8 * n_desc), r = i % (8 * n_desc);
    mb = grp * 8 + (r & 7);
    d = r >> 3;
  } else {
    const int rem = nmb % 8, r = i - full;
    mb = (nmb / 8) * 8 + r % rem;
    d = r / rem;
  }
}

// MB < 8: workgroup (tile, token block, k-split of S), partials of the S splits summed by the last to
// arrive.  MB = 8: persistent over G workgroups (no workgroup ever waits for another): the first
// floor(T / G) * G tiles whole, dealt round robin; the remaining R tiles' super-blocks split evenly over
// gsk workgroups (stream-K), shared tiles combined the same way.  The waves of a workgroup may hold
// blocks of different shards and types: every type's code meets the same barriers.
// FAR: the mixed-type build (ONLY = 0) serves every layer.
template <class GE, int ONLY, bool FAR = false>
__global__ __launch_bounds__(GE::NT) __attribute__((amdgpu_waves_per_eu(GE::WPE))) void gemm_kernel(
    const uint8_t* __restrict__ packed, const int32_t* __restrict__ desc, int n_desc, const uint16_t* __restrict__ x,
    int64_t ldx, int M, uint16_t* __restrict__ y, int64_t ldy, const uint16_t* __restrict__ bias, float* part, int* ctr,
    int per, int G, int gsk, int S) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[GE::LDSX + GB_TAB_BYTES + 16];
  uint16_t* xs = (uint16_t*)lds;
  int* flag = (int*)(lds + GE::LDSX + GB_TAB_BYTES);
  const bool fill = ONLY == 0 || ONLY == GQK_IQ3_S;
  const GTabs tb = g_tables(lds + GE::LDSX, fill, GE::NT);
  if (fill) __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nmb = (M + GE::BM - 1) / GE::BM;
  const int nb = __builtin_amdgcn_readfirstlane(desc[D_NB]);
  // Inlined by force: in the mixed-type 256 x 256 build the compiler left it out of line, where its code
  // is longer than a branch reaches and the long branches overwrote the return address (the kernel never
  // ended), and its uniform operands came back from the stack as vector values.  us, the form before the
  // register decode (out of line too) -> this: Q4_K + Q6_K 7168 x 5120 at 768 / 2048 rows 164 -> 89, 298 ->
  // 165; Q5_K + IQ4_XS 34816 x 5120 at 512 / 2048 409 -> 208, 1347 -> 685.
  auto run = [&](int tile, int mb, int b0, int b1, const GOut& go) __attribute__((always_inline)) {
    tile = __builtin_amdgcn_readfirstlane(tile);
    mb = __builtin_amdgcn_readfirstlane(mb);
    b0 = __builtin_amdgcn_readfirstlane(b0);
    b1 = __builtin_amdgcn_readfirstlane(b1);
    // the wave's 32-row block: a descriptor row holds `per` of them; past the last row a copy without outputs
    const int rbi = tile * GE::NR + wave % GE::NR, d = rbi / per;
    const int rb = d < n_desc ? rbi % per : per;
    const int32_t* dsc = desc + (int64_t)min(d, n_desc - 1) * GQK_DESC_WORDS;
    const int type = __builtin_amdgcn_readfirstlane(dsc[D_TYPE]);
#define RUN(TY)                                                                                          \
    if ((ONLY == 0 || ONLY == TY) && type == TY)                                                         \
      gemm_tile<GE, TY, FAR>(packed, dsc, rb, x, ldx, M, mb * GE::BM, b0, b1, go, y, ldy, bias, xs, flag, tb);
    RUN(GQK_Q4_0) RUN(GQK_Q5_0) RUN(GQK_Q8_0) RUN(GQK_Q2_K) RUN(GQK_Q3_K) RUN(GQK_Q4_K) RUN(GQK_Q5_K) RUN(GQK_Q6_K)
    RUN(GQK_IQ4_NL) RUN(GQK_IQ3_S) RUN(GQK_IQ4_XS)
#undef RUN
  };
  if constexpr (GE::MB < 8) {
    // workgroup = (tile, token block, split): split s of S takes super-blocks [s nb / S, (s + 1) nb / S)
    // Unsplit, the token blocks of a tile go to one XCD (workgroup b runs on XCD b % 8), whose L2 then
    // reads the tile's weights once; the tiles past the last whole eight stay in order.  us, plain order ->
    // this (the others even): Q4_K + Q6_K 7168 x 5120 at 136 / 256 rows 30.0 -> 28.7, 32.8 -> 31.3; IQ4_XS
    // 5120 x 5120 at 333 34.0 -> 32.8; Q4_K 34816 x 5120 at 384 173 -> 169.  A contiguous range of tiles
    // per XCD is as fast, but 1% slower than plain order for that mixed layer at 384 rows.
    const int sp = blockIdx.x % S, u = blockIdx.x / S;
    int tile = u / nmb, mb = u % nmb;
    if (S == 1 && u < ((int)gridDim.x / nmb & ~7) * nmb) {
      tile = (u >> 3) / nmb * 8 + (u & 7);
      mb = (u >> 3) % nmb;
    }
    GOut go{nullptr, nullptr, 0, 1, 0};
    if (S > 1) go = GOut{part, ctr + u, u * S, S, sp};
    run(tile, mb, (int)((int64_t)sp * nb / S), (int)((int64_t)(sp + 1) * nb / S), go);
    return;
  }
  const int T = n_desc * nmb;
  const int tfull = (T / G) * G;
  const int R = T - tfull;
  const int64_t I = (int64_t)R * nb;
  const int w = blockIdx.x;
  auto owner = [&](int64_t i) { return (int)(((i + 1) * gsk + I - 1) / I - 1); };
  int64_t it = 0, end = 0;
  if (R > 0 && w < gsk) {
    it = (int64_t)w * I / gsk;
    end = (int64_t)(w + 1) * I / gsk;
  }
  for (int t_dp = w;;) {
    int t, b0, b1;
    GOut go{nullptr, nullptr, 0, 1, 0};
    if (t_dp < tfull) {
      t = t_dp;
      b0 = 0;
      b1 = nb;
      t_dp += G;
    } else if (it < end) {
      const int r = (int)(it / nb);
      b0 = (int)(it % nb);
      b1 = (int)min<int64_t>(nb, b0 + (end - it));
      t = tfull + r;
      if (b0 != 0 || b1 != nb) {
        const int wf = owner((int64_t)r * nb), wl = owner((int64_t)r * nb + nb - 1);
        go = GOut{part, ctr + r, r + wf, wl - wf + 1, w - wf};
      }
      it += b1 - b0;
    } else {
      break;
    }
    int d, mb;
    gb_map(t, n_desc, nmb, d, mb);
    run(d, mb, b0, b1, go);
  }
}

#define GQK_GEMM_CAT2(a, b) a##b
#define GQK_GEMM_CAT(a, b) GQK_GEMM_CAT2(a, b)

template <class GE>
static int launch_geo(const GemmPick& p, int only, int n_desc, int M, hipStream_t st, const uint8_t* packed,
                      const int32_t* desc, const uint16_t* x, int64_t ldx, uint16_t* y, int64_t ldy,
                      const uint16_t* bias, float* part, int* ctr) {
  const dim3 grid(p.grid), block(GE::NT);
  if (ldx > GQK_MAX_LDX) {
    hipLaunchKernelGGL((gemm_kernel<GE, 0, true>), grid, block, 0, st, packed, desc, n_desc, x, ldx, M, y, ldy, bias, part, ctr, p.per, p.G, p.gsk, p.S);
    return GQK_OK;
  }
  switch (only) {
#define C(T) case T: hipLaunchKernelGGL((gemm_kernel<GE, T>), grid, block, 0, st, packed, desc, n_desc, x, ldx, M, y, ldy, bias, part, ctr, p.per, p.G, p.gsk, p.S); return GQK_OK;
    C(GQK_Q4_0) C(GQK_Q5_0) C(GQK_Q8_0) C(GQK_Q2_K) C(GQK_Q3_K) C(GQK_Q4_K) C(GQK_Q5_K) C(GQK_Q6_K)
    C(GQK_IQ4_NL) C(GQK_IQ3_S) C(GQK_IQ4_XS)
#undef C
    default:
      hipLaunchKernelGGL((gemm_kernel<GE, 0>), grid, block, 0, st, packed, desc, n_desc, x, ldx, M, y, ldy, bias, part, ctr, p.per, p.G, p.gsk, p.S);
  }
  return GQK_OK;
}

// this object's geometries
int GQK_GEMM_CAT(launch_gemm_mb, GQK_GEMM_MB)(const GemmPick& p, int only, int n_desc, int M, hipStream_t st,
                                              const uint8_t* packed, const int32_t* desc, const uint16_t* x,
                                              int64_t ldx, uint16_t* y, int64_t ldy, const uint16_t* bias, float* part,
                                              int* ctr) {
#define GQK_GEMM_LAUNCH(MB, NR, WK)                                                                         \
  if constexpr (MB == GQK_GEMM_MB)                                                                          \
    if (p.mb == MB && p.nr == NR)                                                                           \
      return launch_geo<Geo<MB, NR, WK>>(p, only, n_desc, M, st, packed, desc, x, ldx, y, ldy, bias, part, ctr);
  GQK_GEMM_GEOS(GQK_GEMM_LAUNCH)
#undef GQK_GEMM_LAUNCH
  return GQK_ERR_FORM;
}

}  // namespace gqk
