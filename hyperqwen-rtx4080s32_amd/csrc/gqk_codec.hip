// gqk_codec.hip - GGML block decode to fp32 (the dequantize API) and the tile repack.
//
// dequantize: every weight is computed as gguf-py computes it (gguf.quants.dequantize, the
// reference dequantizer of this path: gguf-plugin/patches/gguf-prefill-dispatch.patch:42-45,
// gguf-plugin/gluon/tiles.py:141-149): (d * sc) * q - dmin * m in fp32.  d * sc * q is exact in
// fp32 for every type (<= 24 significant bits), so only the K-quant min subtraction rounds,
// once; bf16 / fp16 outputs are the round-to-nearest-even of that fp32 value.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include "gqk_common.h"
#include "gqk_internal.h"

namespace gqk {

// Where a 256-weight record's bytes lie: RawSrc reads GGUF rows (any alignment), TileSrc a tile chunk in
// LDS.  ld<P, V>(j): the V at bytes j .. of plane P (j a multiple of its width; it never crosses a segment
// of the plane); RawSrc::raw<V>(b): the V at byte b of the raw record.
template <int T, int P>
__device__ __forceinline__ int raw_of(int j) {   // raw byte of byte j of plane P (equal segments concatenated)
  constexpr gqk_plane pl = gqk_planes<T>::v.planes[P];
  return pl.seg_off + (j / pl.seg_len) * pl.seg_stride + j % pl.seg_len;
}
template <int T, int P>
__device__ __forceinline__ constexpr int plane_off() {
  int o = 0;
  for (int p = 0; p < P; ++p) o += gqk_planes<T>::v.planes[p].size;
  return o;
}
template <typename V> __device__ __forceinline__ V load_any(const uint8_t* p) {
  V v;
  __builtin_memcpy(&v, p, sizeof v);
  return v;
}
template <int T>
struct RawSrc {
  const uint8_t* rec;
  static constexpr bool PACKED6 = false;
  template <int P, typename V> __device__ __forceinline__ V ld(int j) const { return load_any<V>(rec + raw_of<T, P>(j)); }
  template <typename V> __device__ __forceinline__ V raw(int b) const { return load_any<V>(rec + b); }
};
template <int T>
struct TileSrc {
  const uint8_t* chunk;   // plane-major chunk in LDS
  int r;                  // row of the tile
  static constexpr bool PACKED6 = true;
  template <int P, typename V> __device__ __forceinline__ V ld(int j) const {
    constexpr int W = gqk_col_width(gqk_planes<T>::v.planes[P].size), o = 64 * plane_off<T, P>();
    return *(const V*)(chunk + o + ((j / W) * 64 + r) * W + j % W);
  }
};

__device__ __forceinline__ float f16_of(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
template <int N>
__device__ __forceinline__ float ub(const uint32_t (&v)[N / 4], int i) { return (float)((v[i >> 2] >> (8 * (i & 3))) & 0xFF); }
__device__ __forceinline__ uint2 msk(const uint2& v, int sh, uint32_t m) { return make_uint2((v.x >> sh) & m, (v.y >> sh) & m); }
__device__ __forceinline__ uint2 orr(const uint2& a, const uint2& b) { return make_uint2(a.x | b.x, a.y | b.y); }
// bit i of byte b -> bit 4 of byte i (four at a time)
__device__ __forceinline__ uint2 spread4(uint32_t b) {
  return make_uint2((((b & 0xF) * 0x00204081u) & 0x01010101u) << 4, (((b >> 4) * 0x00204081u) & 0x01010101u) << 4);
}
// four nibbles (a byte each) through a 16-entry byte table in four registers
__device__ __forceinline__ uint32_t table16(uint32_t n, const uint32_t (&t)[4]) {
  const uint32_t s = n & 0x07070707u, lo = __builtin_amdgcn_perm(t[1], t[0], s), hi = __builtin_amdgcn_perm(t[3], t[2], s);
  const uint32_t m = ((n >> 3) & 0x01010101u) * 0xFFu;
  return (hi & m) | (lo & ~m);
}
__device__ __forceinline__ uint2 kvalues8(const uint2& n) {   // the IQ4 values + 128
  uint32_t t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    t[i] = (uint32_t)(c_kvalues[4 * i] + 128) | ((uint32_t)(c_kvalues[4 * i + 1] + 128) << 8) |
           ((uint32_t)(c_kvalues[4 * i + 2] + 128) << 16) | ((uint32_t)(c_kvalues[4 * i + 3] + 128) << 24);
  return make_uint2(table16(n.x, t), table16(n.y, t));
}

// N fp32 weights of a record, from weight N i (N = 8 or 4).  q: eight integers in bytes, minus off;
// w = dl * q, or dl * q - ml (K-quants with a min).  grid: the IQ3_S words in LDS.
template <int T, int N, class S>
__device__ __forceinline__ void decode(const S& s, int i, const uint32_t* grid, float (&w)[N]) {
  const int e = N == 8 ? i : i >> 1;   // the eight weights 8 e .. that hold them
  const int g = e >> 2, sub = e & 3;   // 32-weight group, eight of it
  float dl, ml = 0.f, off = 0.f;
  constexpr bool MIN = T == GQK_Q2_K || T == GQK_Q4_K || T == GQK_Q5_K;
  uint2 q;
  uint32_t qn[N / 4];   // the N integers
  // N == 4: the half by arithmetic.  i & 1 ? q.y : q.x became an indexed load of q kept in memory (LDS),
  // whose address takes the workgroup size from the dispatch packet, a read of host memory: Q4_K to
  // fp32 from rows, us with that -> so: 4096 x 512 19.2 -> 5.4, 4096 x 4096 29.2 -> 16.3, 17408 x 5120
  // 137 -> 105 (with 32 weights a thread 6.6, 27.9, 145).
  auto narrow = [&] {
    const uint32_t lo = q.x, hi = q.y;
    if constexpr (N == 8) qn[0] = lo, qn[1] = hi;
    else qn[0] = lo ^ ((lo ^ hi) & -(uint32_t)(i & 1));
  };
  if constexpr (T == GQK_Q4_0 || T == GQK_IQ4_NL || T == GQK_Q5_0) {   // low nibbles: weights 0..15, high: 16..31
    constexpr int PD = T == GQK_Q5_0 ? 2 : 1;
    dl = f16_of(s.template ld<PD, uint16_t>(2 * g));
    q = msk(s.template ld<0, uint2>(16 * g + 8 * (sub & 1)), 4 * (sub >> 1), 0x0F0F0F0Fu);
    off = 8.f;
    if constexpr (T == GQK_Q5_0) {
      q = orr(q, spread4(s.template ld<1, uint8_t>(4 * g + sub)));
      off = 16.f;
    } else if constexpr (T == GQK_IQ4_NL) {
      q = kvalues8(q);
      off = 128.f;
    }
  } else if constexpr (T == GQK_Q8_0) {
    dl = f16_of(s.template ld<1, uint16_t>(2 * g));
    q = s.template ld<0, uint2>(32 * g + 8 * sub);
    q.x ^= 0x80808080u, q.y ^= 0x80808080u;
    off = 128.f;
  } else if constexpr (T == GQK_Q2_K) {   // scales[16] | qs[64] | d | dmin; weight 128 h + 32 t + l = bits 2t of byte 32 h + l
    const int h = g >> 2, t = g & 3;
    const uint32_t dd = s.template ld<2, uint32_t>(0), sc = s.template ld<1, uint8_t>(8 * h + 2 * t + (sub >> 1));
    dl = f16_of((uint16_t)dd) * (float)(sc & 0xF);
    ml = f16_of((uint16_t)(dd >> 16)) * (float)(sc >> 4);
    q = msk(s.template ld<0, uint2>(32 * h + 8 * sub), 2 * t, 0x03030303u);
  } else if constexpr (T == GQK_Q3_K) {   // hmask[32] | qs[64] | scales[12] | d   (kq_ref.py:40-56)
    const int h = g >> 2, jj = g & 3, k = 2 * g + (sub >> 1);
    const int lo = (s.template ld<2, uint8_t>(k % 8) >> (4 * (k / 8))) & 0xF;
    const int hi = (s.template ld<2, uint8_t>(8 + k % 4) >> (2 * (k / 4))) & 3;
    dl = f16_of(s.template ld<3, uint16_t>(0)) * (float)((lo | (hi << 4)) - 32);
    const uint2 hm = msk(s.template ld<1, uint2>(8 * sub), g, 0x01010101u);
    q = orr(msk(s.template ld<0, uint2>(32 * h + 8 * sub), 2 * jj, 0x03030303u), make_uint2(hm.x << 2, hm.y << 2));
    off = 4.f;
  } else if constexpr (T == GQK_Q4_K || T == GQK_Q5_K) {   // d | dmin | scales[12] | (qh[32]) | qs[128]   (q4k.py:5-20, kq_ref.py:57-68)
    constexpr int PH = T == GQK_Q4_K ? 1 : 2;
    const uint32_t dd = s.template ld<PH, uint32_t>(0);
    const uint32_t sa = s.template ld<PH, uint32_t>(4), sb = s.template ld<PH, uint32_t>(8), sv = s.template ld<PH, uint32_t>(12);
    const int j = 8 * (g & 3);   // 6-bit scale and min of sub-block g (kq_ref.py:17-27)
    const uint32_t a = (sa >> j) & 0xFF, b = (sb >> j) & 0xFF, c = (sv >> j) & 0xFF;
    const int sc = g < 4 ? a & 63 : (c & 0xF) | ((a >> 6) << 4), m = g < 4 ? b & 63 : (c >> 4) | ((b >> 6) << 4);
    dl = f16_of((uint16_t)dd) * (float)sc;
    ml = f16_of((uint16_t)(dd >> 16)) * (float)m;
    q = msk(s.template ld<0, uint2>(32 * (g >> 1) + 8 * sub), 4 * (g & 1), 0x0F0F0F0Fu);
    if constexpr (T == GQK_Q5_K) {
      const uint2 hb = msk(s.template ld<1, uint2>(8 * sub), g, 0x01010101u);
      q = orr(q, make_uint2(hb.x << 4, hb.y << 4));
    }
  } else if constexpr (T == GQK_Q6_K) {   // ql[128] | qh[64] | int8 scales[16] | d   (kq_ref.py:69-79)
    const int g16 = e >> 1;
    dl = f16_of(s.template ld<2, uint16_t>(0)) * (float)(int8_t)s.template ld<1, uint8_t>(g16);
    if constexpr (S::PACKED6) {   // the six-bit values re-packed per scale group (gqk_q6_pos)
      uint32_t P[3];
#pragma unroll
      for (int m = 0; m < 3; ++m) P[m] = s.template ld<0, uint32_t>(gqk_q6_pos(g16, m, 0));
      const uint32_t top = ((P[0] >> 6) & 0x03030303u) | ((P[1] >> 4) & 0x0C0C0C0Cu) | ((P[2] >> 2) & 0x30303030u);
      q = e & 1 ? make_uint2(P[2] & 0x3F3F3F3Fu, top) : make_uint2(P[0] & 0x3F3F3F3Fu, P[1] & 0x3F3F3F3Fu);
    } else {
      const int h = g >> 2, t = g & 3;
      const uint2 hi = msk(s.template raw<uint2>(128 + 32 * h + 8 * sub), 2 * t, 0x03030303u);
      q = orr(msk(s.template raw<uint2>(64 * h + 32 * (t & 1) + 8 * sub), 4 * (t >> 1), 0x0F0F0F0Fu), make_uint2(hi.x << 4, hi.y << 4));
    }
    off = 32.f;
  } else if constexpr (T == GQK_IQ4_XS) {   // d | scales_h u16 | scales_l[4] | qs[128]   (iq4xs.py:5-11)
    const uint32_t dd = s.template ld<1, uint32_t>(0);
    const int ls = ((s.template ld<1, uint8_t>(4 + g / 2) >> (4 * (g % 2))) & 0xF) | (((dd >> (16 + 2 * g)) & 3) << 4);
    dl = f16_of((uint16_t)dd) * (float)(ls - 32);
    q = kvalues8(msk(s.template ld<0, uint2>(16 * g + 8 * (sub & 1)), 4 * (sub >> 1), 0x0F0F0F0Fu));
    off = 128.f;
  } else {   // IQ3_S: d | qs[64] | qh[8] | signs[32] | scales[4]   (iq3s_tile_dequant.py:30-53)
    static_assert(T == GQK_IQ3_S, "type");
    const int sc = (s.template ld<3, uint8_t>(g / 2) >> (4 * (g % 2))) & 0xF;
    dl = f16_of(s.template ld<4, uint16_t>(0)) * (float)(1 + 2 * sc);
    const uint32_t qs = s.template ld<0, uint16_t>(8 * g + 2 * sub), qh = s.template ld<2, uint8_t>(g), sg = s.template ld<1, uint8_t>(4 * g + sub);
    q = make_uint2(grid[(qs & 0xFF) | ((qh << (8 - 2 * sub)) & 256)], grid[(qs >> 8) | ((qh << (7 - 2 * sub)) & 256)]);
    narrow();
    const uint32_t sn = N == 8 ? sg : sg >> (4 * (i & 1));
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float v = dl * ub<N>(qn, j);
      w[j] = (sn >> j) & 1 ? -v : v;
    }
    return;
  }
  narrow();
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float v = ub<N>(qn, j) - off;   // an exact integer
    w[j] = MIN ? dl * v - ml : dl * v;
  }
}

template <typename O> __device__ __forceinline__ O cvt_out(float v);
template <> __device__ __forceinline__ float cvt_out<float>(float v) { return v; }
// The fp32 value is made opaque before the narrowing conversion: otherwise the compiler may fuse
// the last multiply into the conversion (v_fma_mixlo_f16(a, b, +0)), which turns a -0.0 product
// (negative scale x zero quant, kept by gguf-py) into +0.0.
template <> __device__ __forceinline__ __bf16 cvt_out<__bf16>(float v) {
  asm volatile("" : "+v"(v));
  return (__bf16)v;
}
template <> __device__ __forceinline__ _Float16 cvt_out<_Float16>(float v) {
  asm volatile("" : "+v"(v));
  return (_Float16)v;
}

// N values to their place: one 16-byte store where the rows allow it (VEC)
template <typename O, bool VEC, int N>
__device__ __forceinline__ void store_n(O* o, const float (&w)[N]) {
  static_assert(N * sizeof(O) == 16, "16 bytes a thread");
  O c[N];
#pragma unroll
  for (int j = 0; j < N; ++j) c[j] = cvt_out<O>(w[j]);
  if constexpr (VEC) {
    *(uint4*)o = __builtin_bit_cast(uint4, c);
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) o[j] = c[j];
  }
}

#define DQ_ITEMS 4                    // items per thread
#define DQ_SPAN (256 * DQ_ITEMS)      // items per workgroup
template <int T> __device__ __forceinline__ const uint32_t* iq3s_grid(uint32_t* lds) {
  if constexpr (T == GQK_IQ3_S) {
    for (int t = threadIdx.x; t < 512; t += 256) lds[t] = c_iq3s_grid[t];
    __syncthreads();
  }
  return lds;
}

// One item = 16 output bytes (eight 16-bit weights, four fp32 ones) of a row, consecutive threads
// consecutive items, so that a wave writes 1 KiB of whole lines and its reads of a record fall in a few
// lines.  Bound by the writes (bf16: 3.5 bytes out per byte of Q4_K in); 34816 x 5120 from 32 weights a
// thread (byte reads, stores 64 bytes apart) -> this, us: bf16 Q4_K 169 -> 108, Q6_K 146 -> 100, Q8_0
// 145 -> 95, Q4_0 137 -> 84, IQ4_XS 165 -> 83, IQ3_S 150 -> 101.  magic = ceil(2^32 / items per row).
template <int T, typename O, bool VEC>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ W, int64_t stride, int64_t n,
                                                      int64_t K, O* __restrict__ out, int64_t ldo, uint32_t magic) {
  __shared__ uint32_t lds[T == GQK_IQ3_S ? 512 : 1];
  const uint32_t* grid = iq3s_grid<T>(lds);
  constexpr int N = 16 / sizeof(O), IR = 256 / N;   // weights per item, items per record
  const int64_t ipr = K / N, base = (int64_t)blockIdx.x * DQ_SPAN;
  const int64_t row0 = base / ipr, rem0 = base - row0 * ipr;
#pragma unroll
  for (int k = 0; k < DQ_ITEMS; ++k) {
    const uint32_t d = k * 256 + threadIdx.x;
    int64_t row = row0, it = rem0 + d;
    if (ipr >= DQ_SPAN) {
      if (it >= ipr) it -= ipr, ++row;
    } else {   // it < 2 DQ_SPAN: the product with magic is exact
      const uint32_t r = __umulhi((uint32_t)it, magic);
      row += r;
      it -= (int64_t)(r * (uint32_t)ipr);
    }
    if (row >= n) return;
    const RawSrc<T> s{W + row * stride + it / IR * gqk_layout<T>::REC};
    float w[N];
    decode<T, N>(s, (int)(it % IR), grid, w);
    store_n<O, VEC, N>(out + row * ldo + it * N, w);
  }
}

template <int T>
static int launch_dequant_t(const void* W, int64_t stride, int64_t n, int64_t K, void* out, int64_t ldo, int dtype,
                            hipStream_t st) {
  const int64_t ipr = K / (dtype == 0 ? 4 : 8), wgs = (n * ipr + DQ_SPAN - 1) / DQ_SPAN;
  if (wgs >= ((int64_t)1 << 31)) return GQK_ERR_SHAPE;
  const dim3 grid((unsigned)wgs), block(256);
  const uint32_t magic = (uint32_t)(((1ull << 32) + ipr - 1) / ipr);
  const int esz = dtype == 0 ? 4 : 2;
  const bool vec = ((uintptr_t)out % 16 == 0) && ((ldo * esz) % 16 == 0);
#define L(O, V) hipLaunchKernelGGL((dequant_kernel<T, O, V>), grid, block, 0, st, (const uint8_t*)W, stride, n, K, (O*)out, ldo, magic)
  if (dtype == 0) {
    if (vec) L(float, true); else L(float, false);
  } else if (dtype == 1) {
    if (vec) L(__bf16, true); else L(__bf16, false);
  } else {
    if (vec) L(_Float16, true); else L(_Float16, false);
  }
#undef L
  return GQK_OK;
}

int launch_dequant(int type, const void* W, int64_t stride, int64_t n, int64_t K, void* out, int64_t ldo, int dtype,
                   hipStream_t st) {
  switch (type) {
#define C(T) case T: return launch_dequant_t<T>(W, stride, n, K, out, ldo, dtype, st);
    C(GQK_Q4_0) C(GQK_Q5_0) C(GQK_Q8_0) C(GQK_Q2_K) C(GQK_Q3_K) C(GQK_Q4_K) C(GQK_Q5_K) C(GQK_Q6_K)
    C(GQK_IQ4_NL) C(GQK_IQ3_S) C(GQK_IQ4_XS)
#undef C
  }
  return GQK_ERR_TYPE;
}

// ---------------------------------------------------------------------------------------------
// Repack raw rows <-> tiles.  One workgroup per chunk (tile t, super-block kb): 64 rows x REC bytes,
// through the 64 raw records in LDS.  Rows past n are zeros in the tiles (repack) and are not written
// (unrepack).  Each byte crosses HBM once in each direction.  The plane table is a compile-time constant
// per type, so the index arithmetic folds to shifts and multiplies by constants.

// visits the 16-byte words of plane P of a chunk: f(word index in the chunk, row of byte i, raw
// byte of byte i) for i = 0..15 through g(i) -> (r, b)
template <int T, int P, class F>
__device__ __forceinline__ void plane_words(int tid, F&& f) {
  constexpr gqk_plane pl = gqk_planes<T>::v.planes[P];
  constexpr int W = gqk_col_width(pl.size), poff = plane_off<T, P>();
  for (int w = tid; w < 4 * pl.size; w += 256) {     // 64 rows * size bytes / 16
    const int x = 16 * w, col = x / (64 * W), rem = x % (64 * W);
    f(4 * poff + w, [&](int i, int& r, int& b) {
      r = (rem + i) / W;
      b = raw_of<T, P>(col * W + (rem + i) % W);
    });
  }
}

template <int T, int P = 0, class F>
__device__ __forceinline__ void every_plane_word(int tid, F&& f) {
  if constexpr (P < gqk_planes<T>::v.nplanes) {
    plane_words<T, P>(tid, f);
    every_plane_word<T, P + 1>(tid, f);
  }
}

// ---- Q6_K: the six-bit values re-packed per scale group (gqk_q6_pos) <-> GGUF's ql / qh ----------
// q of weight k of a re-packed record
__device__ __forceinline__ uint32_t q6_packed(const uint8_t* rec, int k) {
  const int g = k >> 4, j = k & 15;
  if (j < 12) return rec[gqk_q6_pos(g, j >> 2, j & 3)] & 63;
  uint32_t v = 0;
#pragma unroll
  for (int m = 0; m < 3; ++m) v |= (uint32_t)(rec[gqk_q6_pos(g, m, j - 12)] >> 6) << (2 * m);
  return v;
}
// In place on the chunk's 64 records in LDS (raw[row][REC]): restores GGUF's ql / qh.  Every thread computes its share into registers
// before any is written (barriers between), so the pass reads only the old layout.
__device__ __forceinline__ void q6_convert(uint8_t* raw, int tid) {
  constexpr int REC = 210, PER = 64 * 48 / 256;   // 48 dwords of 192 bytes per row, 12 per thread
  uint32_t v[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int it = tid + 256 * k, r = it / 48, w = it % 48;
    const uint8_t* rec = raw + r * REC;
    uint32_t d = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int b = 4 * w + i;   // output byte
      uint32_t byte;
      if (b < 128) {               // ql byte b: low nibbles of weights 128 hh + p and 128 hh + 64 + p
        const int hh = b >> 6, p = b & 63;
        byte = (q6_packed(rec, 128 * hh + p) & 15) | ((q6_packed(rec, 128 * hh + 64 + p) & 15) << 4);
      } else {                     // qh byte: the high pairs of weights 128 hh + p + 32 t
        const int hh = (b - 128) >> 5, p = (b - 128) & 31;
        byte = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) byte |= (q6_packed(rec, 128 * hh + p + 32 * t) >> 4) << (2 * t);
      }
      d |= byte << (8 * i);
    }
    v[k] = d;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int it = tid + 256 * k, r = it / 48, w = it % 48;
    uint8_t* rec = raw + r * REC;
#pragma unroll
    for (int i = 0; i < 4; ++i) rec[4 * w + i] = (uint8_t)(v[k] >> (8 * i));
  }
  __syncthreads();
}

// The 64 raw records of a chunk from its plane-major words (16-byte loads), into raw[row][REC] in
// LDS (Q6_K's six-bit values converted back to ql / qh before the function returns).
template <int T>
__device__ __forceinline__ void chunk_to_raw(const uint4* __restrict__ in, uint8_t* raw, int tid) {
  constexpr int REC = gqk_planes<T>::v.rec;
  auto scatter = [&](int wi, auto&& at) {
    const uint4 q = in[wi];
    const uint32_t v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      int r, b;
      at(i, r, b);
      raw[r * REC + b] = (uint8_t)(v[i >> 2] >> (8 * (i & 3)));
    }
  };
  every_plane_word<T>(tid, scatter);
  if constexpr (T == GQK_Q6_K) {
    __syncthreads();
    q6_convert(raw, tid);
  }
}

// Bytes o .. o + U - 1 (o even) of an LDS row whose base is 16-byte aligned: whole dwords and a byte shift.
template <int U>
__device__ __forceinline__ void lds_bytes(const uint8_t* row, int o, uint32_t* d) {
  if constexpr (U == 2) {
    d[0] = *(const uint16_t*)(row + o);
  } else {
    const uint32_t* p = (const uint32_t*)(row + (o & ~3));
    uint32_t v[U / 4 + 1];
#pragma unroll
    for (int i = 0; i <= U / 4; ++i) v[i] = p[i];
#pragma unroll
    for (int i = 0; i < U / 4; ++i) d[i] = __builtin_amdgcn_alignbyte(v[i + 1], v[i], o & 3);
  }
}
// Writes plane P of a chunk from the 64 raw records in LDS (row stride RS): every 16-byte word is made of
// units that are contiguous in the record.
template <int T, int P, int RS>
__device__ __forceinline__ void write_plane(const uint8_t* raw, uint4* out, int tid) {
  constexpr gqk_plane pl = gqk_planes<T>::v.planes[P];
  constexpr int W = gqk_col_width(pl.size), U = W < pl.seg_len ? W : pl.seg_len < 16 ? pl.seg_len : 16;
  static_assert(U == 2 || U == 4 || U == 8 || U == 16, "unit");
  for (int w = tid; w < 4 * pl.size; w += 256) {     // 64 rows * size bytes / 16
    const int x = 16 * w, col = x / (64 * W), rem = x % (64 * W);
    uint32_t d[4];
    if constexpr (U == 2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint32_t u[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int b = rem + 4 * i + 2 * k;
          lds_bytes<2>(raw + b / W * RS, raw_of<T, P>(col * W + b % W), u + k);
        }
        d[i] = u[0] | (u[1] << 16);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16 / U; ++i) {
        const int b = rem + U * i;
        lds_bytes<U>(raw + b / W * RS, raw_of<T, P>(col * W + b % W), d + U / 4 * i);
      }
    }
    out[4 * plane_off<T, P>() + w] = make_uint4(d[0], d[1], d[2], d[3]);
  }
}
// Q6_K's first plane: the six-bit values re-packed per scale group (gqk_q6_pos), four at a time.  q of
// weights k .. k + 3 (k % 4 = 0) of a raw record: four low bits from ql, two from qh.
__device__ __forceinline__ uint32_t q6_raw4(const uint8_t* rec, int k) {
  const int hh = k >> 7, t = (k >> 5) & 3, p = k & 31;
  const uint32_t lo = *(const uint32_t*)(rec + 64 * hh + 32 * (t & 1) + p) >> (4 * (t >> 1));
  const uint32_t hi = *(const uint32_t*)(rec + 128 + 32 * hh + p) >> (2 * t);
  return (lo & 0x0F0F0F0Fu) | ((hi & 0x03030303u) << 4);
}
template <int RS>
__device__ __forceinline__ void write_plane_q6(const uint8_t* raw, uint4* out, int tid) {
  for (int w = tid; w < 4 * 192; w += 256) {
    const int col = w >> 6, a = col / 3, m = col % 3;
    const uint8_t* rec = raw + (w & 63) * RS;
    uint32_t d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = 16 * (4 * a + i);
      d[i] = q6_raw4(rec, k + 4 * m) | (((q6_raw4(rec, k + 12) >> (2 * m)) & 0x03030303u) << 6);
    }
    out[w] = make_uint4(d[0], d[1], d[2], d[3]);
  }
}
template <int T, int P, int RS>
__device__ __forceinline__ void write_planes(const uint8_t* raw, uint4* out, int tid) {
  if constexpr (P < gqk_planes<T>::v.nplanes) {
    if constexpr (T == GQK_Q6_K && P == 0) write_plane_q6<RS>(raw, out, tid);
    else write_plane<T, P, RS>(raw, out, tid);
    write_planes<T, P + 1, RS>(raw, out, tid);
  }
}

// Raw rows -> tiles, bound by HBM.  The chunk's 64 records go to LDS by 16-byte loads of any alignment
// (the last one of a record overlaps the one before and is shifted into place), all in flight before
// the first is stored, and the planes come back by dwords.  Workgroup b runs on XCD b % 8, which takes
// a contiguous range of chunks: consecutive super-blocks of a row share 128-byte lines, and each XCD's
// L2 then fetches them once.
// 34816 x 5120 from 2-byte row loads and byte gathers -> this, us: Q4_K 76 -> 37, Q6_K 198 -> 57 (its
// six-bit values went byte by byte through a second pass), Q8_0 148 -> 73, Q5_K 93 -> 44, IQ4_XS 72 -> 35,
// Q2_K 36 -> 18 (5.1-6.4 TB/s read + written).
template <int T>
__global__ __launch_bounds__(256) void repack_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                     int64_t stride, int64_t n, int64_t nb, int64_t chunks) {
  constexpr int REC = gqk_planes<T>::v.rec, NV = REC / 16, TAIL = REC % 16, NT = NV + (TAIL != 0);
  constexpr int RS = 16 * NT, IT = (64 * NT + 255) / 256;
  __shared__ __attribute__((aligned(16))) uint8_t raw[64 * RS + 16];
  const int tid = threadIdx.x;
  const int64_t per = (chunks + 7) / 8, chunk = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || chunk >= chunks) return;
  const int64_t kb = chunk % nb, row0 = chunk / nb * 64;
  const uint8_t* rows = src + row0 * stride + kb * REC;
  uint4 v[IT];
#pragma unroll
  for (int k = 0; k < IT; ++k) {
    const int i = k * 256 + tid, r = i / NT, c = i % NT;
    v[k] = make_uint4(0, 0, 0, 0);
    if (i < 64 * NT && row0 + r < n) v[k] = load_any<uint4>(rows + r * stride + (c < NV ? 16 * c : REC - 16));
  }
#pragma unroll
  for (int k = 0; k < IT; ++k) {
    const int i = k * 256 + tid, r = i / NT, c = i % NT;
    uint4 q = v[k];
    if (TAIL != 0 && c == NV) {   // bytes 16 - TAIL .. 15 of the load belong at byte 16 NV
      constexpr int sh = 16 - TAIL, sd = sh / 4, sb = sh % 4;
      const uint32_t s[9] = {q.x, q.y, q.z, q.w, 0, 0, 0, 0, 0};
      q = make_uint4(__builtin_amdgcn_alignbyte(s[sd + 1], s[sd], sb), __builtin_amdgcn_alignbyte(s[sd + 2], s[sd + 1], sb),
                     __builtin_amdgcn_alignbyte(s[sd + 3], s[sd + 2], sb), __builtin_amdgcn_alignbyte(s[sd + 4], s[sd + 3], sb));
    }
    if (i < 64 * NT) *(uint4*)(raw + r * RS + 16 * c) = q;
  }
  __syncthreads();
  write_planes<T, 0, RS>(raw, (uint4*)(dst + chunk * (64 * REC)), tid);
}

// Tiles -> raw rows
template <int T, bool WIDE>
__global__ __launch_bounds__(256) void unrepack_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                       int64_t stride, int64_t n, int64_t nb) {
  constexpr int REC = gqk_planes<T>::v.rec, CB = 64 * REC;          // chunk bytes (a multiple of 64)
  __shared__ __attribute__((aligned(16))) uint8_t raw[CB + 16];   // the 64 raw records, [row][REC]
  const int tid = threadIdx.x;
  const int64_t chunk = blockIdx.x, kb = chunk % nb, tile = chunk / nb;
  const int64_t row0 = tile * 64;
  chunk_to_raw<T>((const uint4*)(src + chunk * CB), raw, tid);
  __syncthreads();
  uint8_t* rows = dst + row0 * stride + kb * REC;
  if (WIDE) {
    for (int i = tid; i < CB / 2; i += 256) {
      const int r = i / (REC / 2), h = i % (REC / 2);
      if (row0 + r < n) *(uint16_t*)(rows + r * stride + 2 * h) = *(const uint16_t*)(raw + r * REC + 2 * h);
    }
  } else {
    for (int i = tid; i < CB; i += 256) {
      const int r = i / REC, b = i % REC;
      if (row0 + r < n) rows[r * stride + b] = raw[i];
    }
  }
}

template <int T>
static void launch_repack_t(bool to_tiles, bool wide, int64_t chunks, hipStream_t st, const uint8_t* s, uint8_t* d,
                            int64_t stride, int64_t n, int64_t nb) {
  const dim3 block(256);
  if (to_tiles)
    hipLaunchKernelGGL((repack_kernel<T>), dim3((unsigned)((chunks + 7) / 8 * 8)), block, 0, st, s, d, stride, n, nb, chunks);
  else if (wide)
    hipLaunchKernelGGL((unrepack_kernel<T, true>), dim3((unsigned)chunks), block, 0, st, s, d, stride, n, nb);
  else
    hipLaunchKernelGGL((unrepack_kernel<T, false>), dim3((unsigned)chunks), block, 0, st, s, d, stride, n, nb);
}

int launch_repack(int type, const void* W, int64_t stride, int64_t n, int64_t K, void* tiles, bool to_tiles,
                  hipStream_t st) {
  const gqk_type* t = gqk_type_get(type);
  if (!t) return GQK_ERR_TYPE;
  const int64_t nb = K / 256, ntiles = (n + 63) / 64;
  const int64_t chunks = ntiles * nb;
  if (chunks == 0) return GQK_OK;
  if (chunks >= ((int64_t)1 << 31)) return GQK_ERR_SHAPE;
  // unrepack: 2-byte accesses along the raw rows when every row starts 2-byte aligned (every REC is even)
  const bool wide = (t->rec % 2 == 0) && (stride % 2 == 0) && ((uintptr_t)W % 2 == 0);
  const uint8_t* s = (const uint8_t*)(to_tiles ? W : tiles);
  uint8_t* d = (uint8_t*)(to_tiles ? tiles : W);
  switch (type) {
#define C(T) case T: launch_repack_t<T>(to_tiles, wide, chunks, st, s, d, stride, n, nb); return GQK_OK;
    C(GQK_Q4_0) C(GQK_Q5_0) C(GQK_Q8_0) C(GQK_Q2_K) C(GQK_Q3_K) C(GQK_Q4_K) C(GQK_Q5_K) C(GQK_Q6_K)
    C(GQK_IQ4_NL) C(GQK_IQ3_S) C(GQK_IQ4_XS)
#undef C
  }
  return GQK_ERR_TYPE;
}

// ---------------------------------------------------------------------------------------------
// Dequantize straight from the tiles: one workgroup per chunk (tile t, super-block kb) copies the chunk
// to LDS as it lies, then decodes items of 16 output bytes from its planes.  A wave takes eight rows x
// eight items: 128 bytes per row, whole lines.  Each tile byte is read once.  34816 x 5120 to bf16 from
// the chunk scattered back to raw records byte by byte -> this, us: Q4_K 129 -> 83, Q6_K 148 -> 94, Q8_0
// 151 -> 106, IQ4_XS 171 -> 85, IQ3_S 153 -> 82 (5.2-5.5 TB/s read + written).
template <int T, typename O, bool VEC>
__global__ __launch_bounds__(256) void tile_dequant_kernel(const uint8_t* __restrict__ tiles, int64_t n, int64_t nb,
                                                           O* __restrict__ out, int64_t ldo) {
  constexpr int REC = gqk_planes<T>::v.rec, CB = 64 * REC;
  constexpr int N = 16 / sizeof(O), IP = 32 / N;   // weights per item, passes of eight items per row
  __shared__ __attribute__((aligned(16))) uint8_t raw[CB];
  __shared__ uint32_t lds[T == GQK_IQ3_S ? 512 : 1];
  const int tid = threadIdx.x;
  const int64_t chunk = blockIdx.x, kb = chunk % nb, tile = chunk / nb;
  const uint4* in = (const uint4*)(tiles + chunk * CB);
#pragma unroll
  for (int k = 0; k < (CB / 16 + 255) / 256; ++k) {
    const int i = k * 256 + tid;
    if (i < CB / 16) ((uint4*)raw)[i] = in[i];
  }
  const uint32_t* grid = iq3s_grid<T>(lds);
  __syncthreads();
  const int64_t rows = n - tile * 64;
#pragma unroll
  for (int k = 0; k < 2 * IP; ++k) {   // pass k: rows 32 (k / IP) + 8 wave + lane / 8, items 8 (k % IP) + lane % 8
    const int r = 32 * (k / IP) + 8 * (tid >> 6) + ((tid & 63) >> 3), e = 8 * (k % IP) + (tid & 7);
    if (r >= rows) continue;
    float w[N];
    decode<T, N>(TileSrc<T>{raw, r}, e, grid, w);
    store_n<O, VEC, N>(out + (tile * 64 + r) * ldo + kb * 256 + e * N, w);
  }
}

template <int T>
static int launch_tile_dequant_t(const void* tiles, int64_t n, int64_t K, void* out, int64_t ldo, int dtype,
                                 hipStream_t st) {
  const int64_t nb = K / 256, chunks = (n + 63) / 64 * nb;
  if (chunks == 0) return GQK_OK;
  if (chunks >= ((int64_t)1 << 31)) return GQK_ERR_SHAPE;
  const dim3 grid((unsigned)chunks), block(256);
  const int esz = dtype == 0 ? 4 : 2;
  const bool vec = ((uintptr_t)out % 16 == 0) && ((ldo * esz) % 16 == 0);
  const uint8_t* t = (const uint8_t*)tiles;
#define L(O, V) hipLaunchKernelGGL((tile_dequant_kernel<T, O, V>), grid, block, 0, st, t, n, nb, (O*)out, ldo)
  if (dtype == 0) {
    if (vec) L(float, true); else L(float, false);
  } else if (dtype == 1) {
    if (vec) L(__bf16, true); else L(__bf16, false);
  } else {
    if (vec) L(_Float16, true); else L(_Float16, false);
  }
#undef L
  return GQK_OK;
}

int launch_tile_dequant(int type, const void* tiles, int64_t n, int64_t K, void* out, int64_t ldo, int dtype,
                        hipStream_t st) {
  switch (type) {
#define C(T) case T: return launch_tile_dequant_t<T>(tiles, n, K, out, ldo, dtype, st);
    C(GQK_Q4_0) C(GQK_Q5_0) C(GQK_Q8_0) C(GQK_Q2_K) C(GQK_Q3_K) C(GQK_Q4_K) C(GQK_Q5_K) C(GQK_Q6_K)
    C(GQK_IQ4_NL) C(GQK_IQ3_S) C(GQK_IQ4_XS)
#undef C
  }
  return GQK_ERR_TYPE;
}

}  // namespace gqk
