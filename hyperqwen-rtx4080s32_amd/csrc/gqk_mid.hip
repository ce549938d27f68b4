// gqk_mid.hip - the mid form of the grouped linear (9..32 batch rows): the GEMV's work split with the
// GEMM's arithmetic.
#include "gqk_tile.h"

namespace gqk {

// ---- the mid form: 17..32 batch rows -----------------------------------------------------------
// The GEMV's work split (one workgroup per descriptor row: a 64-row tile and a k-range of
// super-blocks that its waves divide; tiles shared by several rows combine fp32 partials in
// split order, the last to arrive writing y) with the GEMM's arithmetic: each weight decoded
// once to bf16 (round-to-nearest-even of the exact fp32 value, the same B2 decoders) straight
// into registers, and v_mfma_f32_32x32x16_bf16 over all 32 tokens.  No LDS staging of weights and
// no barrier in the main loop: lane l acts as decoder thread (row l % 32 and 32 + l % 32, part
// l / 32) of each 64-weight step, which is exactly the MFMA's B-operand layout (column l % 32,
// k-chunk l / 32); its A operand is x of token l % 32 at the same eight k.  One step of weights
// and x is in flight while the previous one is decoded.  x goes through a 4 KiB LDS region of
// the wave: read straight in the A layout, every load touched 32 token rows (32 bytes of each
// 128-byte line), and loaded coalesced (8 whole rows per load) then re-read from LDS the launch
// is 14-20% faster on gate_up (Q4_K, Q6_K, Q8_0, IQ4_XS at M = 32), 20% on Q6_K down, 3-6% on
// qkv and the low-bit down shards, even on Q4_K down / o_proj.  Measured against the 32 x 128
// GEMM tile form it replaced (before the x staging; Q4_K gate_up / qkv / o_proj / down at
// M = 32: 0.87 / 0.86 / 0.84 / 0.76 of its time; Q2_K, Q8_0, Q6_K down 0.80 / 0.77 / 0.86,
// IQ4_XS gate_up 0.94; Q6_K and Q8_0 gate_up 1.04).  Tried: weights two steps ahead (more
// registers, fewer waves: 0-8% slower) and 64 tokens per wave (226-260 VGPRs: 23-45% slower than
// a GEMM form with 64-token tiles).  x and the weights come by buffer loads (a scalar base and one lane
// offset each, no address arithmetic) and the k-loop is unrolled over a super-block; us at 32 rows
// before -> now, gate_up / down / qkv / o_proj: Q4_K 38.8 -> 37.8, 25.6 -> 25.3, 12.1 -> 11.2, 11.2 ->
// 10.4; Q5_K 45.7 -> 42.1, 29.1 -> 27.9, 15.4 -> 14.4, 12.4 -> 11.1; IQ4_XS 40.7 -> 38.0, 29.1 -> 25.6,
// 13.7 -> 11.9, 13.2 -> 11.4; Q3_K 40.2 -> 34.9, 28.2 -> 24.6, 13.3 -> 11.0, 12.9 -> 10.8; a Q5_K +
// IQ4_XS layer 49.4 -> 40.5, 33.2 -> 26.9.
// FAR: rows of x further apart than 32-bit byte offsets reach (GQK_MAX_LDX), by 64-bit addresses.
template <int T, int NRB = 2, bool FAR = false>
__device__ __forceinline__ void mid_wave(const uint8_t* __restrict__ tbase, const uint16_t* __restrict__ x, int64_t ldx,
                                         int M, uint16_t* xl, int kw0, int kw1, int c, int r, const GTabs& tb,
                                         v16f (&acc)[NRB], int r0 = 0) {
  constexpr int REC = gqk_layout<T>::REC;
  if (kw0 >= kw1) return;
  // k offsets (within a 64-weight step) of the lane's four 8-weight chunks, in MFMA order
  const int koff[4] = {B2<T>::off0(c), B2<T>::off0(c) + 8, B2<T>::off1(c), B2<T>::off1(c) + 8};
  // x of a step (32 tokens x 64 k = 32 rows of 128 bytes) comes in with coalesced loads: load i
  // of lane j takes row 8 i + j / 8, 16-byte chunk (j % 8) ^ swz(row), and the wave writes the four
  // loads to its LDS region in lane order; the A operand (token l % 32, chunk koff / 8) is then read
  // at slot chunk ^ swz(token).  swz(t) = (t >> 1) & 7 puts the 16 rows a quarter-wave reads in 16
  // distinct 16-byte bank groups.
  const int lane = threadIdx.x & 63;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, 0xFFFFFFFFu, GQK_GB_WORD3);
  std::conditional_t<FAR, int64_t, uint32_t> xoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = 8 * i + (lane >> 3);
    xoff[i] = min(t, M - 1) * (decltype(+xoff[i]))(2 * ldx) + 16u * ((lane & 7) ^ ((t >> 1) & 7));
  }
  const int rs = (r >> 1) & 7;
  // The two widest types in the slab keep plain weight loads (us at 32 rows, buffer -> plain: Q8_0 qkv /
  // o_proj 17.4 / 16.0 -> 16.4 / 14.9, Q6_K 16.2 / 14.8 -> 15.6 / 13.8; the others gain by the buffer's),
  // and Q8_0 in the 64-row form for both (gate_up / down at 20 rows 46.6 / 30.2 -> 45.4 / 29.9).
  constexpr bool WPTR = T == GQK_Q8_0 || NRB == 1 && T == GQK_Q6_K, XPTR = FAR || T == GQK_Q8_0 && NRB == 2;
  struct Step { B2<T> w[NRB]; v4u xg[4]; };
  Step p0, p1;
  auto load = [&](Step& p, int kb, int kq) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if constexpr (XPTR) p.xg[i] = *(const v4u*)((const uint8_t*)x + xoff[i] + (int64_t)(4 * kb + kq) * (2 * GB_K));
      else p.xg[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, xoff[i], (4 * kb + kq) * (2 * GB_K), 0);
    const uint8_t* rp = tbase + (int64_t)kb * (64 * REC);
#pragma unroll
    for (int b = 0; b < NRB; ++b)
      if constexpr (WPTR) p.w[b].load(rp, r0 + 32 * b + r, kq, c);
      else p.w[b].load(g_src(rp), r0 + 32 * b + r, kq, c);
  };
  auto compute = [&](const Step& p, int kq) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) ((v4u*)xl)[64 * i + lane] = p.xg[i];
    v8bf a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = *(const v8bf*)(xl + (r * 8 + ((koff[q] >> 3) ^ rs)) * 8);
#pragma unroll
    for (int b = 0; b < NRB; ++b) {
      const GS st = p.w[b].prep(kq, c);
      uint32_t o[16];
#pragma unroll
      for (int i = 0; i < 4; ++i) p.w[b].out(st, kq, c, o, tb, i);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            a[q], __builtin_bit_cast(v8bf, v4u{o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]}), acc[b], 0, 0, 0);
    }
  };
  // Loads are unconditional (clamped to the wave's end, re-read from L2 at the tail).  A super-block's
  // four steps per trip, so the decoders' shifts and branches on the step fold away, with the next
  // loads held where they are written (without that the compiler hoists them and takes two waves per
  // SIMD); Q8_0's decode does not depend on the step and two steps a trip measured 3% faster.
  if constexpr (T == GQK_Q8_0) {
    const int last = 4 * kw1 - 1;
    load(p0, kw0, 0);
    load(p1, kw0, 1);
    for (int s = 4 * kw0;; s += 2) {
      const int s2 = min(s + 2, last), s3 = min(s + 3, last);
      compute(p0, s & 3);
      load(p0, s2 >> 2, s2 & 3);
      if (s + 1 > last) break;
      compute(p1, (s + 1) & 3);
      load(p1, s3 >> 2, s3 & 3);
      if (s + 2 > last) break;
    }
    return;
  }
  load(p0, kw0, 0);
  load(p1, kw0, 1);
  for (int kb = kw0; kb < kw1; ++kb) {
    const int kn = min(kb + 1, kw1 - 1);
    compute(p0, 0);
    load(p0, kb, 2);
    __builtin_amdgcn_sched_barrier(0);
    compute(p1, 1);
    load(p1, kb, 3);
    __builtin_amdgcn_sched_barrier(0);
    compute(p0, 2);
    load(p0, kn, 0);
    __builtin_amdgcn_sched_barrier(0);
    compute(p1, 3);
    load(p1, kn, 1);
    __builtin_amdgcn_sched_barrier(0);
  }
}

#define MID_RED_BYTES (3 * 2 * 16 * 64 * 4 + 16)   // the waves' sums combined in LDS (nw <= 4), a flag

// Three waves per SIMD: every type fits 168 VGPRs without scratch (151-168); Q8_0 has its loads placed
// as well as two waves' registers allow instead (above).
template <int ONLY, bool FAR = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ONLY == GQK_Q8_0 || FAR ? 1 : 3))) void gemv_mid_kernel(const uint8_t* __restrict__ packed, const int32_t* __restrict__ desc,
                                                       const uint16_t* __restrict__ x, int64_t ldx, int M,
                                                       uint16_t* __restrict__ y, int64_t ldy,
                                                       const uint16_t* __restrict__ bias, float* __restrict__ part,
                                                       int* __restrict__ ctr) {
  constexpr int MP = 32;   // tokens of the plan (partial slots [slot][64 rows][MP])
  __shared__ __attribute__((aligned(16))) uint8_t lds[MID_RED_BYTES + GB_TAB_BYTES];
  __shared__ __attribute__((aligned(16))) uint16_t xlds[4 * 2048];   // a 4 KiB x step per wave
  const int32_t* dsc = desc + (int64_t)blockIdx.x * GQK_DESC_WORDS;
  const int type = dsc[D_TYPE];
  // the wave index is uniform: as an SGPR its k-range, addresses and branches stay scalar (Q6_K,
  // Q2_K 4-9% faster at M = 32)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int c = lane >> 5, r = lane & 31;
  GTabs tb;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    tb.kv[i] = (uint32_t)(c_kvalues[4 * i] + 128) | ((uint32_t)(c_kvalues[4 * i + 1] + 128) << 8) |
               ((uint32_t)(c_kvalues[4 * i + 2] + 128) << 16) | ((uint32_t)(c_kvalues[4 * i + 3] + 128) << 24);
  tb.grid = (uint32_t*)(lds + MID_RED_BYTES);
  tb.sign = (uint4*)(lds + MID_RED_BYTES + 512 * 4);
  if ((ONLY == 0 || ONLY == GQK_IQ3_S) && type == GQK_IQ3_S) {   // uniform over the workgroup
    uint32_t* grid = (uint32_t*)(lds + MID_RED_BYTES);
    uint4* sign = (uint4*)(lds + MID_RED_BYTES + 512 * 4);
    for (int t = threadIdx.x; t < 512; t += blockDim.x) grid[t] = c_iq3s_grid[t];
    for (int t = threadIdx.x; t < 256; t += blockDim.x) {
      uint32_t m[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) m[q] = (((t >> (2 * q)) & 1) << 15) | (((t >> (2 * q + 1)) & 1) << 31);
      sign[t] = make_uint4(m[0], m[1], m[2], m[3]);
    }
    __syncthreads();
  }
  const int64_t off = (int64_t)(uint32_t)dsc[D_OFF_LO] | ((int64_t)dsc[D_OFF_HI] << 32);
  const int64_t tile = dsc[D_TILE0];
  const int nb = dsc[D_NB], kb0 = dsc[D_KB0], nk = dsc[D_KB1] - kb0;
  const int kw0 = kb0 + (wave * nk) / nw, kw1 = kb0 + ((wave + 1) * nk) / nw;
  uint16_t* xl = xlds + wave * 2048;
  v16f acc[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[b][v] = 0.f;
#define RUN(T)                                                                                                 \
  if ((ONLY == 0 || ONLY == T) && type == T)                                                                   \
    mid_wave<T, 2, FAR>(packed + g_uniform(off + tile * nb * (int64_t)(64 * gqk_layout<T>::REC)), x, ldx, M, xl, kw0, kw1, c, r, tb, acc);
  RUN(GQK_Q4_0) RUN(GQK_Q5_0) RUN(GQK_Q8_0) RUN(GQK_Q2_K) RUN(GQK_Q3_K) RUN(GQK_Q4_K) RUN(GQK_Q5_K) RUN(GQK_Q6_K)
  RUN(GQK_IQ4_NL) RUN(GQK_IQ3_S) RUN(GQK_IQ4_XS)
#undef RUN

  // combine the waves (fixed order) in wave 0
  float* red = (float*)lds;   // [wave - 1][b][v][lane]
  int* flag = (int*)(lds + 3 * 2 * 16 * 64 * 4);
  if (wave > 0)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) red[(((wave - 1) * 2 + b) * 16 + v) * 64 + lane] = acc[b][v];
  __syncthreads();
  if (wave == 0)
    for (int w = 1; w < nw; ++w)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[b][v] += red[(((w - 1) * 2 + b) * 16 + v) * 64 + lane];

  // C block b: lane -> weight row 32 b + r, tokens 8 (v / 4) + 4 c + v % 4
  const int nvalid = dsc[D_NVALID];
  const int64_t col0 = dsc[D_COL0];
  const int nc = dsc[D_NC];   // workgroups sharing this tile
  // quarter qd of the outputs: block qd / 2, values 8 (qd % 2) .. + 7 of each lane
  auto store_q = [&](int qd, const float (&a)[8]) {
    const int b = qd >> 1, v0 = 8 * (qd & 1), row = 32 * b + r;
    if (row >= nvalid) return;
    // the layer bias (bf16 per output column) joins before the one rounding to bf16
    const float bv = bias != nullptr ? __builtin_bit_cast(float, (uint32_t)bias[col0 + row] << 16) : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int v = v0 + e, t = 8 * (v >> 2) + 4 * c + (v & 3);
      if (t < M) y[(int64_t)t * ldy + col0 + row] = __builtin_bit_cast(uint16_t, (__bf16)(a[e] + bv));
    }
  };
  if (nc == 1) {
    if (wave > 0) return;
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
      float a[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] = acc[qd >> 1][8 * (qd & 1) + e];
      store_q(qd, a);
    }
    return;
  }
  // Split-K exchange, as in the GEMV: the nc partials of a tile in slots D_SLOT0 .. + nc - 1 as
  // [slot][64 rows][32 tokens], moved by device-coherent (sc1) 16-byte buffer accesses only.  Wave
  // 0's sums go through LDS so that every wave stores quarters wave, wave + nw, .. of the partial;
  // all stores complete before the arrival count (one barrier), and in the last workgroup to
  // arrive every wave sums its quarters of the slots in split order and writes y; the counter is
  // reset for the next launch.
  __syncthreads();   // wave 0 has read the other waves' sums
  if (wave == 0)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) red[(b * 16 + v) * 64 + lane] = acc[b][v];
  __syncthreads();
  const int sp = dsc[D_SPLIT], ctr_i = dsc[D_CTR];
  float* tp = part + (int64_t)dsc[D_SLOT0] * 64 * MP;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(tp, 0, nc * 64 * MP * 4, GQK_GB_WORD3);
  auto soff = [&](int q, int b, int g) { return ((q * 64 + 32 * b + r) * MP + 8 * g + 4 * c) * 4; };
  for (int qd = wave; qd < 4; qd += nw) {
    const int b = qd >> 1, g0 = 2 * (qd & 1);
    float a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = red[(b * 16 + 8 * (qd & 1) + e) * 64 + lane];
    __builtin_amdgcn_raw_buffer_store_b128(v4f{a[0], a[1], a[2], a[3]}, rs, soff(sp, b, g0), 0, GQK_GB_SC1);
    __builtin_amdgcn_raw_buffer_store_b128(v4f{a[4], a[5], a[6], a[7]}, rs, soff(sp, b, g0 + 1), 0, GQK_GB_SC1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's partial stores are complete
  __syncthreads();
  if (threadIdx.x == 0) *flag = __hip_atomic_fetch_add(&ctr[ctr_i], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*flag != nc - 1) return;
  asm volatile("" ::: "memory");
  // split slots per round trip (loads clamped to the last slot): two measured 0.4-1.2 us faster
  // than four on `down` at M = 20 / 32 and eight 0.5-1.1 us slower; one is even with two
  constexpr int QB = 2;
  for (int qd = wave; qd < 4; qd += nw) {
    const int b = qd >> 1, g0 = 2 * (qd & 1);
    float a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = 0.f;
    for (int q0 = 0; q0 < nc; q0 += QB) {
      v4f t[QB][2];
#pragma unroll
      for (int j = 0; j < QB; ++j)
#pragma unroll
        for (int h2 = 0; h2 < 2; ++h2)
          t[j][h2] = __builtin_amdgcn_raw_buffer_load_b128(rs, soff(min(q0 + j, nc - 1), b, g0 + h2), 0, GQK_GB_SC1);
#pragma unroll
      for (int j = 0; j < QB; ++j)
        if (q0 + j < nc)
#pragma unroll
          for (int e = 0; e < 8; ++e) a[e] += t[j][e >> 2][e & 3];
    }
    store_q(qd, a);
  }
  if (threadIdx.x == 0) __hip_atomic_store(&ctr[ctr_i], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // next launch
}

// The mid form's slab variant (9..32 rows, x padded to 32 tokens; shards of at most one 32-row
// slab per CU): one
// workgroup per 32-row half (D_SPLIT) of a 64-row tile over the whole k-range, its waves splitting
// the k-range as in the mid form (two super-blocks each at K = 5120) with one 32 x 32 block of
// rows each; no split-K partials (whose 8 KiB per workgroup at 32 tokens made the exchange ~30% of
// the mid form's qkv / o_proj launches).  Each wave's sums go to its own 4 KiB x region once its
// products are done, and after one barrier every thread sums one output over the waves in order.
template <int ONLY, bool FAR = false>
__global__ __launch_bounds__(64 * GQK_SLAB_MAX_WAVES) void gemv_mid_slab_kernel(
    const uint8_t* __restrict__ packed, const int32_t* __restrict__ desc, const uint16_t* __restrict__ x,
    int64_t ldx, int M, uint16_t* __restrict__ y, int64_t ldy, const uint16_t* __restrict__ bias) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[GB_TAB_BYTES];
  __shared__ __attribute__((aligned(16))) uint16_t xlds[GQK_SLAB_MAX_WAVES * 2048];   // a 4 KiB x step per wave
  const int32_t* dsc = desc + (int64_t)blockIdx.x * GQK_DESC_WORDS;
  const int type = dsc[D_TYPE];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int c = lane >> 5, r = lane & 31;
  GTabs tb;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    tb.kv[i] = (uint32_t)(c_kvalues[4 * i] + 128) | ((uint32_t)(c_kvalues[4 * i + 1] + 128) << 8) |
               ((uint32_t)(c_kvalues[4 * i + 2] + 128) << 16) | ((uint32_t)(c_kvalues[4 * i + 3] + 128) << 24);
  tb.grid = (uint32_t*)lds;
  tb.sign = (uint4*)(lds + 512 * 4);
  if ((ONLY == 0 || ONLY == GQK_IQ3_S) && type == GQK_IQ3_S) {   // uniform over the workgroup
    uint32_t* grid = (uint32_t*)lds;
    uint4* sign = (uint4*)(lds + 512 * 4);
    for (int t = threadIdx.x; t < 512; t += blockDim.x) grid[t] = c_iq3s_grid[t];
    for (int t = threadIdx.x; t < 256; t += blockDim.x) {
      uint32_t m[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) m[q] = (((t >> (2 * q)) & 1) << 15) | (((t >> (2 * q + 1)) & 1) << 31);
      sign[t] = make_uint4(m[0], m[1], m[2], m[3]);
    }
    __syncthreads();
  }
  const int64_t off = (int64_t)(uint32_t)dsc[D_OFF_LO] | ((int64_t)dsc[D_OFF_HI] << 32);
  const int64_t tile = dsc[D_TILE0];
  const int h = dsc[D_SPLIT];                        // the slab: rows 32 h .. 32 h + 31 of the tile
  const int nb = dsc[D_NB], kb0 = dsc[D_KB0], nk = dsc[D_KB1] - kb0;
  const int kw0 = kb0 + (wave * nk) / nw, kw1 = kb0 + ((wave + 1) * nk) / nw;
  uint16_t* xl = xlds + wave * 2048;
  v16f acc[1];
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[0][v] = 0.f;
#define RUN(T)                                                                                                 \
  if ((ONLY == 0 || ONLY == T) && type == T)                                                                   \
    mid_wave<T, 1, FAR>(packed + g_uniform(off + tile * nb * (int64_t)(64 * gqk_layout<T>::REC)), x, ldx, M, xl, kw0, kw1, c, r, tb, \
                   acc, 32 * h);
  RUN(GQK_Q4_0) RUN(GQK_Q5_0) RUN(GQK_Q8_0) RUN(GQK_Q2_K) RUN(GQK_Q3_K) RUN(GQK_Q4_K) RUN(GQK_Q5_K) RUN(GQK_Q6_K)
  RUN(GQK_IQ4_NL) RUN(GQK_IQ3_S) RUN(GQK_IQ4_XS)
#undef RUN

  // combine: C block lane -> row 32 h + r, tokens 8 (v / 4) + 4 c + v % 4; [v][lane] per wave
  float* red = (float*)xl;
#pragma unroll
  for (int v = 0; v < 16; ++v) red[v * 64 + lane] = acc[0][v];
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const int nvalid = dsc[D_NVALID];
  const int64_t col0 = dsc[D_COL0];
  for (int o = threadIdx.x; o < 32 * 32; o += blockDim.x) {
    const int t = o >> 5, rho = o & 31;
    const int v = 4 * (t >> 3) + (t & 3), l = 32 * ((t >> 2) & 1) + rho;
    float sum = 0.f;
    for (int w = 0; w < nw; ++w) sum += ((const float*)(xlds + w * 2048))[v * 64 + l];
    const int row = 32 * h + rho;
    if (t < M && row < nvalid) {
      const float bv = bias != nullptr ? __builtin_bit_cast(float, (uint32_t)bias[col0 + row] << 16) : 0.f;
      y[(int64_t)t * ldy + col0 + row] = __builtin_bit_cast(uint16_t, (__bf16)(sum + bv));
    }
  }
}

int launch_gemv_mid(const uint8_t* packed, const int32_t* desc, int n_desc, int types_mask, const void* x, int64_t ldx,
                    int M, int nw, bool slab, void* y, int64_t ldy, const void* bias, float* part, int* ctr,
                    hipStream_t st) {
  const uint16_t* xx = (const uint16_t*)x;
  uint16_t* yy = (uint16_t*)y;
  const uint16_t* bb = (const uint16_t*)bias;
  const bool far = ldx > GQK_MAX_LDX;   // the mixed-type builds serve every layer there
  if (slab) {
    if (nw < 1 || nw > GQK_SLAB_MAX_WAVES) return GQK_ERR_FORM;
    const dim3 grid(n_desc), block(64 * nw);
    if (far) {
      hipLaunchKernelGGL((gemv_mid_slab_kernel<0, true>), grid, block, 0, st, packed, desc, xx, ldx, M, yy, ldy, bb);
      return GQK_OK;
    }
    switch (types_mask) {
#define C(T) case T: hipLaunchKernelGGL((gemv_mid_slab_kernel<T>), grid, block, 0, st, packed, desc, xx, ldx, M, yy, ldy, bb); return GQK_OK;
      C(GQK_Q4_0) C(GQK_Q5_0) C(GQK_Q8_0) C(GQK_Q2_K) C(GQK_Q3_K) C(GQK_Q4_K) C(GQK_Q5_K) C(GQK_Q6_K)
      C(GQK_IQ4_NL) C(GQK_IQ3_S) C(GQK_IQ4_XS)
#undef C
      default:
        hipLaunchKernelGGL((gemv_mid_slab_kernel<0>), grid, block, 0, st, packed, desc, xx, ldx, M, yy, ldy, bb);
    }
    return GQK_OK;
  }
  if (nw < 1 || nw > 4) return GQK_ERR_FORM;
  const dim3 grid(n_desc), block(64 * nw);
  if (far) {
    hipLaunchKernelGGL((gemv_mid_kernel<0, true>), grid, block, 0, st, packed, desc, xx, ldx, M, yy, ldy, bb, part, ctr);
    return GQK_OK;
  }
  switch (types_mask) {
#define C(T) case T: hipLaunchKernelGGL((gemv_mid_kernel<T>), grid, block, 0, st, packed, desc, xx, ldx, M, yy, ldy, bb, part, ctr); return GQK_OK;
    C(GQK_Q4_0) C(GQK_Q5_0) C(GQK_Q8_0) C(GQK_Q2_K) C(GQK_Q3_K) C(GQK_Q4_K) C(GQK_Q5_K) C(GQK_Q6_K)
    C(GQK_IQ4_NL) C(GQK_IQ3_S) C(GQK_IQ4_XS)
#undef C
    default:
      hipLaunchKernelGGL((gemv_mid_kernel<0>), grid, block, 0, st, packed, desc, xx, ldx, M, yy, ldy, bb, part, ctr);
  }
  return GQK_OK;
}

}  // namespace gqk
