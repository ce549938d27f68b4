// gqk_tile.h - device code shared by the GEMM and the mid form: the tile-plane loads and the per-step
// decoders B2<T>, which turn 32 weights of one row of a 64-weight step into bf16 (round-to-nearest-even
// of the exact fp32 gguf-py value).
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include "gqk_common.h"
#include "gqk_internal.h"

namespace gqk {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

#define GQK_GB_WORD3 0x00020000   // buffer resource word 3: raw untyped dword access
#define GQK_GB_SC1 16             // device-scope cache policy (write through / bypass the XCD L2)

__device__ __forceinline__ float g_h2f(uint32_t bits16) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(bits16 & 0xFFFF));
}
__device__ __forceinline__ uint32_t g_bf16x2(float lo, float hi) {
  typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
  v2bf p;
  p[0] = (__bf16)lo;
  p[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, p);
}

template <int N>
__device__ __forceinline__ void gld(uint32_t* dst, const uint8_t* p) {
  if constexpr (N % 16 == 0) {
#pragma unroll
    for (int i = 0; i < N / 16; ++i) {
      uint4 v = *(const uint4*)(p + 16 * i);
      dst[4 * i] = v.x; dst[4 * i + 1] = v.y; dst[4 * i + 2] = v.z; dst[4 * i + 3] = v.w;
    }
  } else if constexpr (N == 8) {
    uint2 v = *(const uint2*)p;
    dst[0] = v.x; dst[1] = v.y;
  } else if constexpr (N == 4) {
    dst[0] = *(const uint32_t*)p;
  } else if constexpr (N == 12) {
    const uint32_t* q = (const uint32_t*)p;
    dst[0] = q[0]; dst[1] = q[1]; dst[2] = q[2];
  } else {
    static_assert(N == 2, "plane slice size");
    dst[0] = *(const uint16_t*)p;
  }
}

// a value the whole wave shares, in scalar registers
__device__ __forceinline__ int64_t g_uniform(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// A byte address with a part the whole wave shares (scalar base, scalar offset) and a lane's 32-bit
// offset: one buffer load, no address arithmetic in vector registers.  c + n moves the shared part,
// c[n] adds a lane offset.
struct GSrc {
  __amdgpu_buffer_rsrc_t rs;
  uint32_t so, vo;
  __device__ __forceinline__ GSrc operator+(uint32_t n) const { return GSrc{rs, so + n, vo}; }
  __device__ __forceinline__ GSrc operator[](uint32_t n) const { return GSrc{rs, so, vo + n}; }
};
__device__ __forceinline__ GSrc g_src(const uint8_t* base) {
  return GSrc{__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0xFFFFFFFFu, GQK_GB_WORD3), 0, 0};
}
template <int N>
__device__ __forceinline__ void gld(uint32_t* dst, const GSrc& p) {
  if constexpr (N % 16 == 0) {
#pragma unroll
    for (int i = 0; i < N / 16; ++i) {
      const v4u v = __builtin_amdgcn_raw_buffer_load_b128(p.rs, p.vo, p.so + 16 * i, 0);
      dst[4 * i] = v.x; dst[4 * i + 1] = v.y; dst[4 * i + 2] = v.z; dst[4 * i + 3] = v.w;
    }
  } else if constexpr (N == 8) {
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    const v2u v = __builtin_amdgcn_raw_buffer_load_b64(p.rs, p.vo, p.so, 0);
    dst[0] = v.x; dst[1] = v.y;
  } else if constexpr (N == 4) {
    dst[0] = __builtin_amdgcn_raw_buffer_load_b32(p.rs, p.vo, p.so, 0);
  } else {
    static_assert(N == 2, "plane slice size");
    dst[0] = __builtin_amdgcn_raw_buffer_load_b16(p.rs, p.vo, p.so, 0);
  }
}
// a lane's offset from a plain address
__device__ __forceinline__ const uint8_t* g_at(const uint8_t* c, uint32_t n) { return c + n; }
__device__ __forceinline__ GSrc g_at(const GSrc& c, uint32_t n) { return c[n]; }

// 16-byte column `col` of row r in a plane with 16-byte columns (column-major: (col * 64 + r) * 16)
template <class C>
__device__ __forceinline__ C col16(const C& plane, uint32_t r, uint32_t col, uint32_t byte = 0) {
  return g_at(plane, (col * 64 + r) * 16 + byte);
}

#define GB_K 64                  // weights per step
#define GB_2P24 16777216.f

struct GTabs {
  uint32_t kv[4];          // IQ4 kvalues + 128, four per dword
  const uint32_t* grid;    // IQ3_S grid magnitudes (LDS, 512 words)
  const uint4* sign;       // IQ3_S sign masks of a sign byte: bits 15 / 31 of four bf16 pairs (LDS)
};

// Per-step constants of a decoder (scales and biases of the step's two scale groups, or one),
// computed once per step by prep() and used by each quarter of out().
struct GS {
  float dl0, b0, dl1, b1;   // the scales times 2^24 (cvt4)
  uint32_t aux;
};

// fma(dl, u_i, bias) for the four unsigned bytes u_i of u -> two bf16 pairs (RNE).  dl24 is dl * 2^24:
// a byte widened to 16 bits is the fp16 (subnormal) value u_i * 2^-24, which v_fma_mix_f32 multiplies
// by dl24 in the same instruction that converts it, exactly; a v_perm_b32 widens two bytes at once.
__device__ __forceinline__ void cvt4(uint32_t u, float dl24, float bias, uint32_t* o) {
  typedef _Float16 v2h __attribute__((ext_vector_type(2)));
  const v2h a = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0u, u, 0x0C010C00u));
  const v2h b = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0u, u, 0x0C030C02u));
  o[0] = g_bf16x2(__builtin_fmaf((float)a[0], dl24, bias), __builtin_fmaf((float)a[1], dl24, bias));
  o[1] = g_bf16x2(__builtin_fmaf((float)b[0], dl24, bias), __builtin_fmaf((float)b[1], dl24, bias));
}
// IQ4 lookup of four nibbles (bytes 0..15 of n): kvalues + 128 as four unsigned bytes
__device__ __forceinline__ uint32_t kv4(uint32_t n, const GTabs& tb) {
  const uint32_t s = n & 0x07070707u;
  const uint32_t lo = __builtin_amdgcn_perm(tb.kv[1], tb.kv[0], s);
  const uint32_t hi = __builtin_amdgcn_perm(tb.kv[3], tb.kv[2], s);
  const uint32_t m = ((n >> 3) & 0x01010101u) * 0xFFu;
  return (hi & m) | (lo & ~m);
}
// Q4_K / Q5_K 6-bit scale and min of sub-block j (get_scale_min_k4) from the 12 scale bytes
__device__ __forceinline__ void k4_scale(const uint32_t* hdr, int j, int& sc, int& m) {
  const uint64_t s01 = (uint64_t)hdr[1] | ((uint64_t)hdr[2] << 32);
  if (j < 4) {
    sc = (int)((s01 >> (8 * j)) & 63);
    m = (int)((s01 >> (8 * j + 32)) & 63);
  } else {
    const uint32_t b = (hdr[3] >> (8 * (j - 4))) & 0xFF;   // byte j + 4
    sc = (int)((b & 0xF) | (((s01 >> (8 * (j - 4))) & 0xC0) >> 2));
    m = (int)((b >> 4) | (((s01 >> (8 * j)) & 0xC0) >> 2));
  }
}
// Q4_K / Q5_K constants of step kq: sub-blocks 2 kq (dl0, b0) and 2 kq + 1 (dl1, b1)
__device__ __forceinline__ GS k4_prep(const uint32_t* hdr, int kq) {
  int sc0, m0, sc1, m1;
  k4_scale(hdr, 2 * kq, sc0, m0);
  k4_scale(hdr, 2 * kq + 1, sc1, m1);
  const float d = g_h2f(hdr[0]) * GB_2P24, dm = g_h2f(hdr[0] >> 16);
  return GS{d * (float)sc0, -(dm * (float)m0), d * (float)sc1, -(dm * (float)m1), 0};
}
// Q3_K signed 6-bit scale i (0..15) from the 12 packed bytes
__device__ __forceinline__ int q3_scale(const uint32_t* sb, int i) {
  const uint64_t s01 = (uint64_t)sb[0] | ((uint64_t)sb[1] << 32);
  const int lo = (int)(((s01 >> (8 * (i & 7))) >> (4 * (i >> 3))) & 0xF);
  const int hi = (int)((sb[2] >> (8 * (i & 3) + 2 * (i >> 2))) & 3);
  return (lo | (hi << 4)) - 32;
}

template <int T> struct B2;
// out(i) of a decoder fills o[2 i], o[2 i + 1], o[8 + 2 i], o[9 + 2 i] unless its B2 sets SEQ
template <class B, class = void> struct b2_seq : std::false_type {};
template <class B> struct b2_seq<B, std::void_t<decltype(B::SEQ)>> : std::integral_constant<bool, B::SEQ> {};

template <> struct B2<GQK_Q4_0> {   // block b = 2 kq + h: low nibbles -> 16 weights, high -> next 16
  uint32_t q[4], d;
  static __device__ int off0(int h) { return 32 * h; }
  static __device__ int off1(int h) { return 32 * h + 16; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    gld<16>(q, col16(c, r, 2 * kq + h)); gld<2>(&d, g_at(c + 64 * 128, r * 16 + 2 * (2 * kq + h)));
  }
  __device__ GS prep(int, int) const {
    const float dd = g_h2f(d);
    return GS{dd * GB_2P24, -8.f * dd, 0.f, 0.f, 0};
  }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs&, int i) const {
    cvt4(q[i] & 0x0F0F0F0Fu, st.dl0, st.b0, o + 2 * i);
    cvt4((q[i] >> 4) & 0x0F0F0F0Fu, st.dl0, st.b0, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_IQ4_NL> {
  uint32_t q[4], d;
  static __device__ int off0(int h) { return 32 * h; }
  static __device__ int off1(int h) { return 32 * h + 16; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    gld<16>(q, col16(c, r, 2 * kq + h)); gld<2>(&d, g_at(c + 64 * 128, r * 16 + 2 * (2 * kq + h)));
  }
  __device__ GS prep(int, int) const {
    const float dd = g_h2f(d);
    return GS{dd * GB_2P24, -128.f * dd, 0.f, 0.f, 0};
  }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs& tb, int i) const {
    cvt4(kv4(q[i] & 0x0F0F0F0Fu, tb), st.dl0, st.b0, o + 2 * i);
    cvt4(kv4((q[i] >> 4) & 0x0F0F0F0Fu, tb), st.dl0, st.b0, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_Q5_0> {
  uint32_t q[4], qh, d;
  static __device__ int off0(int h) { return 32 * h; }
  static __device__ int off1(int h) { return 32 * h + 16; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    const uint32_t b = 2 * kq + h;
    gld<16>(q, col16(c, r, b)); gld<4>(&qh, col16(c + 64 * 128, r, b >> 2, 4 * (b & 3)));
    gld<2>(&d, g_at(c + 64 * 160, r * 16 + 2 * b));
  }
  __device__ GS prep(int, int) const {
    const float dd = g_h2f(d);
    return GS{dd * GB_2P24, -16.f * dd, 0.f, 0.f, 0};
  }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs&, int i) const {
    const uint32_t hl = ((((qh >> (4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
    const uint32_t hh = ((((qh >> (16 + 4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
    cvt4((q[i] & 0x0F0F0F0Fu) | hl, st.dl0, st.b0, o + 2 * i);
    cvt4(((q[i] >> 4) & 0x0F0F0F0Fu) | hh, st.dl0, st.b0, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_Q8_0> {   // block b = 2 kq + h, 32 int8 in two 16-byte columns
  static constexpr bool SEQ = true;   // out(i) fills o[4 i .. 4 i + 3]
  uint32_t q[8], d;
  static __device__ int off0(int h) { return 32 * h; }
  static __device__ int off1(int h) { return 32 * h + 16; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    const uint32_t b = 2 * kq + h;
    gld<16>(q, col16(c, r, 2 * b)); gld<16>(q + 4, col16(c, r, 2 * b + 1)); gld<2>(&d, g_at(c + 64 * 256, r * 16 + 2 * b));
  }
  __device__ GS prep(int, int) const {
    const float dd = g_h2f(d);
    return GS{dd * GB_2P24, -128.f * dd, 0.f, 0.f, 0};
  }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs&, int i) const {
    cvt4(q[2 * i] ^ 0x80808080u, st.dl0, st.b0, o + 4 * i);
    cvt4(q[2 * i + 1] ^ 0x80808080u, st.dl0, st.b0, o + 4 * i + 2);
  }
};

template <> struct B2<GQK_Q2_K> {   // groups 2 kq, 2 kq + 1 share the 16 bytes of the row's part h
  uint32_t q[4], scw, dd;
  static __device__ int off0(int h) { return 16 * h; }
  static __device__ int off1(int h) { return 32 + 16 * h; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    gld<16>(q, col16(c, r, 2 * (kq >> 1) + h)); gld<4>(&scw, g_at(c + 64 * 64, r * 16 + 4 * kq)); gld<4>(&dd, g_at(c + 64 * 80, r * 4));
  }
  __device__ GS prep(int, int h) const {
    const float d = g_h2f(dd) * GB_2P24, dmin = g_h2f(dd >> 16);
    const uint32_t s0 = (scw >> (8 * h)) & 0xFF, s1 = (scw >> (8 * (2 + h))) & 0xFF;
    return GS{d * (float)(s0 & 0xF), -(dmin * (float)(s0 >> 4)), d * (float)(s1 & 0xF), -(dmin * (float)(s1 >> 4)), 0};
  }
  __device__ void out(const GS& st, int kq, int, uint32_t (&o)[16], const GTabs&, int i) const {
    const int j0 = 2 * (kq & 1);
    cvt4((q[i] >> (2 * j0)) & 0x03030303u, st.dl0, st.b0, o + 2 * i);
    cvt4((q[i] >> (2 * j0 + 2)) & 0x03030303u, st.dl1, st.b1, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_Q3_K> {
  uint32_t q[4], hm[4], sb[3], d;
  static __device__ int off0(int h) { return 16 * h; }
  static __device__ int off1(int h) { return 32 + 16 * h; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    gld<16>(q, col16(c, r, 2 * (kq >> 1) + h));
    gld<16>(hm, col16(c + 64 * 64, r, h));
#pragma unroll
    for (int i = 0; i < 3; ++i) gld<4>(sb + i, g_at(c + 64 * 96, 256 * i + r * 4));   // three 4-byte columns
    gld<2>(&d, g_at(c + 64 * 108, r * 2));
  }
  __device__ GS prep(int kq, int h) const {
    const float dd = g_h2f(d);
    const float dl0 = dd * (float)q3_scale(sb, 4 * kq + h), dl1 = dd * (float)q3_scale(sb, 4 * kq + 2 + h);
    return GS{dl0 * GB_2P24, -4.f * dl0, dl1 * GB_2P24, -4.f * dl1, 0};
  }
  __device__ void out(const GS& st, int kq, int, uint32_t (&o)[16], const GTabs&, int i) const {
    const int j0 = 2 * (kq & 1), g0 = 2 * kq;
    const uint32_t u0 = ((q[i] >> (2 * j0)) & 0x03030303u) | (((hm[i] >> g0) & 0x01010101u) << 2);
    const uint32_t u1 = ((q[i] >> (2 * j0 + 2)) & 0x03030303u) | (((hm[i] >> (g0 + 1)) & 0x01010101u) << 2);
    cvt4(u0, st.dl0, st.b0, o + 2 * i);
    cvt4(u1, st.dl1, st.b1, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_Q4_K> {   // low nibbles: sub-block 2 kq, high: 2 kq + 1; part h = bytes 16h .. 16h + 15
  uint32_t q[4], hdr[4];
  static __device__ int off0(int h) { return 16 * h; }
  static __device__ int off1(int h) { return 32 + 16 * h; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    gld<16>(q, col16(c, r, 2 * kq + h)); gld<16>(hdr, g_at(c + 64 * 128, r * 16));
  }
  __device__ GS prep(int kq, int) const { return k4_prep(hdr, kq); }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs&, int i) const {
    cvt4(q[i] & 0x0F0F0F0Fu, st.dl0, st.b0, o + 2 * i);
    cvt4((q[i] >> 4) & 0x0F0F0F0Fu, st.dl1, st.b1, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_Q5_K> {
  uint32_t q[4], qh[4], hdr[4];
  static __device__ int off0(int h) { return 16 * h; }
  static __device__ int off1(int h) { return 32 + 16 * h; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    gld<16>(q, col16(c, r, 2 * kq + h)); gld<16>(qh, col16(c + 64 * 128, r, h)); gld<16>(hdr, g_at(c + 64 * 160, r * 16));
  }
  __device__ GS prep(int kq, int) const { return k4_prep(hdr, kq); }
  __device__ void out(const GS& st, int kq, int, uint32_t (&o)[16], const GTabs&, int i) const {
    cvt4((q[i] & 0x0F0F0F0Fu) | (((qh[i] >> (2 * kq)) & 0x01010101u) << 4), st.dl0, st.b0, o + 2 * i);
    cvt4(((q[i] >> 4) & 0x0F0F0F0Fu) | (((qh[i] >> (2 * kq + 1)) & 0x01010101u) << 4), st.dl1, st.b1, o + 8 + 2 * i);
  }
};

// Q6_K from the re-packed six-bit plane: step kq's 16-weight groups 4 kq .. 4 kq + 3 sit in columns
// 3 kq .. 3 kq + 2 (dword d of column 3 kq + m = P_m of group 4 kq + d); part h takes groups
// 4 kq + 2 h and 4 kq + 2 h + 1, dwords 2 h, 2 h + 1: 8 contiguous bytes of each column
template <> struct B2<GQK_Q6_K> {
  uint32_t P[3][2], scw, d;
  static __device__ int off0(int h) { return 32 * h; }
  static __device__ int off1(int h) { return 32 * h + 16; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
#pragma unroll
    for (int m = 0; m < 3; ++m) gld<8>(P[m], col16(c, r, 3 * kq + m, 8 * h));
    gld<4>(&scw, g_at(c + 64 * 192, r * 16 + 4 * kq)); gld<2>(&d, g_at(c + 64 * 208, r * 2));
  }
  __device__ GS prep(int, int h) const {
    const float dd = g_h2f(d);
    const float dl0 = dd * (float)(int8_t)((scw >> (16 * h)) & 0xFF), dl1 = dd * (float)(int8_t)((scw >> (16 * h + 8)) & 0xFF);
    return GS{dl0 * GB_2P24, -32.f * dl0, dl1 * GB_2P24, -32.f * dl1, 0};
  }
  // weights 4 i .. 4 i + 3 of the part's group j (0, 1) as four bytes
  __device__ uint32_t q4(int j, int i) const {
    if (i < 3) return P[i][j] & 0x3F3F3F3Fu;
    return ((P[0][j] >> 6) & 0x03030303u) | ((P[1][j] >> 4) & 0x0C0C0C0Cu) | ((P[2][j] >> 2) & 0x30303030u);
  }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs&, int i) const {
    cvt4(q4(0, i), st.dl0, st.b0, o + 2 * i);
    cvt4(q4(1, i), st.dl1, st.b1, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_IQ4_XS> {
  uint32_t q[4], hdr[2];
  static __device__ int off0(int h) { return 32 * h; }
  static __device__ int off1(int h) { return 32 * h + 16; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    gld<16>(q, col16(c, r, 2 * kq + h)); gld<8>(hdr, g_at(c + 64 * 128, r * 8));
  }
  __device__ GS prep(int kq, int h) const {
    const int g = 2 * kq + h;
    const int ls = (int)(((hdr[1] >> (4 * g)) & 0xF) | (((hdr[0] >> (16 + 2 * g)) & 3) << 4));
    const float dl = g_h2f(hdr[0]) * (float)(ls - 32);
    return GS{dl * GB_2P24, -128.f * dl, 0.f, 0.f, 0};
  }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs& tb, int i) const {
    cvt4(kv4(q[i] & 0x0F0F0F0Fu, tb), st.dl0, st.b0, o + 2 * i);
    cvt4(kv4((q[i] >> 4) & 0x0F0F0F0Fu, tb), st.dl0, st.b0, o + 8 + 2 * i);
  }
};

template <> struct B2<GQK_IQ3_S> {   // group g = 2 kq + h: 32 weights, magnitudes from the grid, signs as bf16 masks
  static constexpr bool SEQ = true;   // out(i) fills o[4 i .. 4 i + 3]
  uint32_t qs[2], sg, qh[2], scb, d;
  static __device__ int off0(int h) { return 32 * h; }
  static __device__ int off1(int h) { return 32 * h + 16; }
  template <class C>
  __device__ __forceinline__ void load(const C& c, uint32_t r, uint32_t kq, uint32_t h) {
    const uint32_t g = 2 * kq + h;
    gld<8>(qs, col16(c, r, g >> 1, 8 * (g & 1)));
    gld<4>(&sg, col16(c + 64 * 64, r, g >> 2, 4 * (g & 3)));
    gld<8>(qh, g_at(c + 64 * 96, r * 8));
    gld<4>(&scb, g_at(c + 64 * 104, r * 4));
    gld<2>(&d, g_at(c + 64 * 108, r * 2));
  }
  __device__ GS prep(int kq, int h) const {
    const int g = 2 * kq + h;
    const float dl = g_h2f(d) * (float)(1 + 2 * (int)((scb >> (4 * g)) & 0xF));
    const uint32_t qhb = (uint32_t)(((uint64_t)qh[0] | ((uint64_t)qh[1] << 32)) >> (8 * g)) & 0xFF;
    return GS{dl * GB_2P24, 0.f, 0.f, 0.f, qhb};
  }
  __device__ void out(const GS& st, int, int, uint32_t (&o)[16], const GTabs& tb, int i) const {
    const float dl = st.dl0;
    const uint32_t qhb = st.aux;
    {
      const int l = i;
      const uint32_t qsw = qs[l >> 1] >> (16 * (l & 1));
      const uint32_t i1 = (qsw & 0xFF) | ((qhb << (8 - 2 * l)) & 256);
      const uint32_t i2 = ((qsw >> 8) & 0xFF) | ((qhb << (7 - 2 * l)) & 256);
      const uint4 sm = tb.sign[(sg >> (8 * l)) & 0xFF];
      uint32_t p[4];
      cvt4(tb.grid[i1], dl, 0.f, p);
      cvt4(tb.grid[i2], dl, 0.f, p + 2);
      o[4 * l] = p[0] ^ sm.x; o[4 * l + 1] = p[1] ^ sm.y; o[4 * l + 2] = p[2] ^ sm.z; o[4 * l + 3] = p[3] ^ sm.w;
    }
  }
};

// LDS bytes of the IQ3_S tables
#define GB_TAB_BYTES (512 * 4 + 256 * 16)

// The IQ lookup tables: the IQ4 values in registers, the IQ3_S grid and sign masks at `lds`, filled by
// the nt threads of the workgroup when FILL (the caller synchronises before the first use).
__device__ __forceinline__ GTabs g_tables(uint8_t* lds, bool fill, int nt) {
  GTabs tb;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    tb.kv[i] = (uint32_t)(c_kvalues[4 * i] + 128) | ((uint32_t)(c_kvalues[4 * i + 1] + 128) << 8) |
               ((uint32_t)(c_kvalues[4 * i + 2] + 128) << 16) | ((uint32_t)(c_kvalues[4 * i + 3] + 128) << 24);
  uint32_t* grid = (uint32_t*)lds;
  uint4* sign = (uint4*)(lds + 512 * 4);
  tb.grid = grid;
  tb.sign = sign;
  if (fill) {
    for (int t = threadIdx.x; t < 512; t += nt) grid[t] = c_iq3s_grid[t];
    for (int t = threadIdx.x; t < 256; t += nt) {
      uint32_t m[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) m[p] = (((t >> (2 * p)) & 1) << 15) | (((t >> (2 * p + 1)) & 1) << 31);
      sign[t] = make_uint4(m[0], m[1], m[2], m[3]);
    }
  }
  return tb;
}

}  // namespace gqk
