// qgemv_dot.hip -- decode GEMV of the block types through int8 dot products (gemv_q,
// tier.cpp:299-306): every q4_0, q4_1, q5_0, q5_1, iq4_nl, iq4_xs, q2_K and q3_K weight, and
// the q8_0, q6_K, q4_K and q5_K shapes where it beats the MFMA kernels (qgemv_dispatch).
//
// The roof is HBM: N*rb bytes of weights, each read once, straight into registers (nothing
// of the weight goes through LDS).  What such a kernel loses to is VALU work per weight,
// so a weight costs one byte of a word and a quarter of v_dot4_i32_i8 per digit:
//   * x is prepared once per workgroup: per 32 elements a power of two 2^e that puts
//     max |x| into [2^28, 2^29), x_int = trunc(x * 2^e) in four balanced int8 digits, and
//     the two 16-element sums of x.  A block of 32 takes 36 dwords of LDS: digit plane l
//     (8 dwords, element order) at 8 l, then 2^-e, S_lo, S_hi and a word that marks or lists
//     the wide blocks, and puts consecutive blocks on distinct bank groups (36 mod 64).
//   * each format unpacks its codes to signed int8 words: codes are moved to the top bits of
//     their byte where an offset is subtracted (one xor instead of a subtraction), and
//     formats with a minimum are centred, d q + m = d (q - c) + (c d + m), so the large
//     terms cancel in the scale and not in the sum (q4_K 1024x5120: 8.6e-8 off 64 bits,
//     3.2e-7 where the two terms are summed apart).
//   * the digit dots of 32 (or 16) elements are exact in int32, combined to fp32 and scaled
//     once per block (d * sc * 2^-e, and the minimum times S): gemv_q's sum regrouped by block.
// One workgroup of 16 waves per CU, so x is prepared once per CU.  A lane takes one unit of a
// row at a time; L consecutive lanes and P parts share a row, chosen by the host so that
// the slots (1024 / L per workgroup) come out even.  The next unit's bytes are loaded
// before the current one is computed, and the first before x is prepared.
//
// Measured (MI355X, us a call, graph replays over rotated copies of the weight; before: the generic
// kernel for iq4 and the K types, one that staged rows in LDS for q4 and q5, MFMA for the others):
//   iq4_xs 14336x5120 54.4 -> 14.5, 5120x14336 113 -> 17.0, 1024x5120 14.9 -> 4.9;  iq4_nl 53.4 -> 13.7
//   q3_K   14336x5120 39.1 -> 17.2, 4096x14336 67 -> 16.4, 1024x5120 15.6 -> 4.9
//   q2_K   14336x5120 27.1 -> 15.9, 5120x14336 85 -> 17.3
//   q4_0   14336x5120 22.3 -> 11.4, 5120x14336 36.0 -> 13.6, 4096x14336 29.2 -> 11.4
//   q4_1, q5_0, q5_1 14336x5120 21.4 -> 11.7, 27.2 -> 13.2, 27.6 -> 13.7
//   q8_0   9000x8192 24.5 -> 17.6, 20000x5120 29.2 -> 22.3, 1024x5120 5.3 -> 4.8
//   q6_K   1024x5120 7.7 -> 5.4, 2500x8192 14.0 -> 10.5, 9001x11264 69 -> 29.2
// What bounds it at 14336x5120 (counters): 2.6 (q4_0) to 4.8 (q3_K) VALU instructions a weight,
// x included, whose issue takes 4.8 to 9.0 us a SIMD; LDS reads of x that take 4.5 us a CU (units of
// 128: 9, two thirds of it bank conflicts of lanes four blocks apart); the weight's bytes at a large
// copy's rate 8.5 us (q4_0), in part overlapped, after some 3 us of launch, x and first loads.
// Two rows a lane, 512-thread workgroups (one or two per CU) and deeper prefetch were within
// 10 % of this on large shapes and slower on small ones.
//
// x_int keeps all 24 bits of an element within 2^5 of its block's largest, 23 within 2^6.  A block
// is wide where a run of eight elements is not zero but has none within 2^6 to 2^7 (an outlier among
// ordinary values, which counts for nothing in a row whose weight is zero there), or where max |x|
// < 2^-97 (e is at most 126).  It counts as zero in the digits and sums, and its products are added
// to each row's sum in fp32, one by one as gemv_q adds them (rows_wide).  Of blocks of a normal
// variable none is wide, of silu(g) u one in 80000.  Measured, us: the marks 0.1 a call; x with an
// outlier in each 1024 elements, 1024x5120 4.6 -> 6.8, iq4_xs 14336x5120 14.1 -> 18.4.
//
// NaN or Inf in x (the digits carry finite x only), and any row whose sum is not finite
// (an infinite or NaN block scale, an overflow), is computed again element by element as
// the generic kernel does, so those rows have gemv_q's result classes.
#include <algorithm>
#include <cmath>

#include "tm_device.h"

namespace tiermm {

int device_cus(int* cus);

namespace {

constexpr int XB = 36;  // dwords of a prepared 32-element block of x

// Register loads start at dword boundaries (the vector cache splits those that do not into more
// accesses); bytes that start two past a dword are shifted into place with v_alignbit.
typedef uint32_t u32x4d __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2d __attribute__((ext_vector_type(2), aligned(4)));
#define TM_GLOBAL __attribute__((address_space(1)))
template <int N>
__device__ __forceinline__ void ldw(const uint8_t* p, uint32_t* w) {  // N dwords
  int i = 0;
#pragma unroll
  for (; i + 4 <= N; i += 4) {
    const u32x4 v = *(const TM_GLOBAL u32x4d*)(size_t)(p + 4 * i);
    w[i] = v[0]; w[i + 1] = v[1]; w[i + 2] = v[2]; w[i + 3] = v[3];
  }
  if (i + 2 <= N) {
    const u32x2 v = *(const TM_GLOBAL u32x2d*)(size_t)(p + 4 * i);
    w[i] = v[0]; w[i + 1] = v[1];
    i += 2;
  }
  if (i < N) w[i] = *(const TM_GLOBAL uint32_t*)(size_t)(p + 4 * i);
}
__device__ __forceinline__ uint32_t abit(uint32_t hi, uint32_t lo, uint32_t sh) { return __builtin_amdgcn_alignbit(hi, lo, sh); }

// int8 dots of the four digits of 16 elements (words w0 .. w0 + 3 of a block)
struct XBlk {
  u32x4 d[4][2];  // digit l, words 4h .. 4h + 3
  float f, s0, s1;
  __device__ __forceinline__ void load(const float* xs, int blk) {
    const float* p = xs + blk * XB;
#pragma unroll
    for (int l = 0; l < 4; ++l)
#pragma unroll
      for (int h = 0; h < 2; ++h) d[l][h] = *(const u32x4*)(p + 8 * l + 4 * h);
    const float4 m = *(const float4*)(p + 32);
    f = m.x; s0 = m.y; s1 = m.z;
  }
  template <int H>
  __device__ __forceinline__ void dot16(const uint32_t (&w)[8], int (&c)[4]) const {
#pragma unroll
    for (int l = 0; l < 4; ++l)
#pragma unroll
      for (int k = 0; k < 4; ++k) c[l] = __builtin_amdgcn_sdot4((int)w[4 * H + k], (int)d[l][H][k], c[l], false);
  }
};
// the digit dots as fp32 (both int32 halves exact, their conversions round once)
__device__ __forceinline__ float digits(const int (&c)[4]) {
  return fmaf((float)(c[3] * 256 + c[2]), 65536.f, (float)(c[1] * 256 + c[0]));
}
__device__ __forceinline__ float dot32(const XBlk& x, const uint32_t (&w)[8]) {
  int c[4] = {0, 0, 0, 0};
  x.dot16<0>(w, c);
  x.dot16<1>(w, c);
  return digits(c) * x.f;
}
template <int H>
__device__ __forceinline__ float dot16(const XBlk& x, const uint32_t (&w)[8]) {
  int c[4] = {0, 0, 0, 0};
  x.dot16<H>(w, c);
  return digits(c) * x.f;
}

// Formats: a unit is UE elements (64: two blocks of 32; 128: half a super-block), Raw = one
// lane's dwords of it, acc<T>() adds the unit's 32-element block T of one row.
// No load reaches past the unit's own bytes: where a block starts on a dword, the dword
// that would is a repeat of the one before it (its bytes are not used then).
template <int QT>
struct Fm;

__device__ __forceinline__ uint32_t lo4s(uint32_t q) { return ((q << 4) & 0xf0f0f0f0u) ^ 0x80808080u; }  // 16 (q - 8)
__device__ __forceinline__ uint32_t hi4s(uint32_t q) { return (q & 0xf0f0f0f0u) ^ 0x80808080u; }
// bits 0..3 of h to bit 7 of the bytes
__device__ __forceinline__ uint32_t fifth(uint32_t h) { return (__umul24(h & 15u, 0x00204081u) << 7) & 0x80808080u; }

// Words of the nibbles at byte 4 i + O (O = 0 or 2) of w: w[k] low, w[4 + k] high
template <int O>
__device__ __forceinline__ uint32_t at(const uint32_t* w, int i) { return O ? abit(w[i + 1], w[i], 16) : w[i]; }

template <>
struct Fm<QT_Q4_0> {  // d, 16 nibble bytes, twice: 36 bytes
  static constexpr int UE = 64;
  struct Raw {
    uint32_t w[9];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) { ldw<9>(row + (uint32_t)u * 36, r.w); }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t q = T ? r.w[5 + k] : at<2>(r.w, k);
      w[k] = lo4s(q);
      w[4 + k] = hi4s(q);
    }
    return fmaf(h2f(T ? r.w[4] >> 16 : r.w[0] & 0xffffu) * 0.0625f, dot32(x, w), s);
  }
};

template <>
struct Fm<QT_Q4_1> {  // d q + m = d (q - 8) + (8 d + m); d, m, 16 nibble bytes, twice
  static constexpr int UE = 64;
  struct Raw {
    uint32_t w[10];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) { ldw<10>(row + (uint32_t)u * 40, r.w); }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[k] = lo4s(r.w[5 * T + 1 + k]);
      w[4 + k] = hi4s(r.w[5 * T + 1 + k]);
    }
    const float d = h2f(r.w[5 * T] & 0xffffu);
    s = fmaf(0.0625f * d, dot32(x, w), s);
    return fmaf(fmaf(8.f, d, h2f(r.w[5 * T] >> 16)), x.s0 + x.s1, s);
  }
};

template <>
struct Fm<QT_Q5_0> {  // 8 (q - 16): the five bits at the top of their byte, top bit flipped
  static constexpr int UE = 64;
  struct Raw {
    uint32_t w[11];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) { ldw<11>(row + (uint32_t)u * 44, r.w); }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    const uint32_t qh = T ? r.w[6] : at<2>(r.w, 0);
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t q = T ? r.w[7 + k] : at<2>(r.w, 1 + k);
      w[k] = (((q << 3) & 0x78787878u) | fifth(qh >> (4 * k))) ^ 0x80808080u;
      w[4 + k] = (((q >> 1) & 0x78787878u) | fifth(qh >> (16 + 4 * k))) ^ 0x80808080u;
    }
    return fmaf(h2f(T ? r.w[5] >> 16 : r.w[0] & 0xffffu) * 0.125f, dot32(x, w), s);
  }
};

template <>
struct Fm<QT_Q5_1> {  // d q + m = d (q - 16) + (16 d + m)
  static constexpr int UE = 64;
  struct Raw {
    uint32_t w[12];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) { ldw<12>(row + (uint32_t)u * 48, r.w); }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    const uint32_t qh = r.w[6 * T + 1];
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t q = r.w[6 * T + 2 + k];
      w[k] = (((q << 3) & 0x78787878u) | fifth(qh >> (4 * k))) ^ 0x80808080u;
      w[4 + k] = (((q >> 1) & 0x78787878u) | fifth(qh >> (16 + 4 * k))) ^ 0x80808080u;
    }
    const float d = h2f(r.w[6 * T] & 0xffffu);
    s = fmaf(0.125f * d, dot32(x, w), s);
    return fmaf(fmaf(16.f, d, h2f(r.w[6 * T] >> 16)), x.s0 + x.s1, s);
  }
};

template <>
struct Fm<QT_Q8_0> {
  static constexpr int UE = 64;
  struct Raw {
    uint32_t w[17];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) { ldw<17>(row + (uint32_t)u * 68, r.w); }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = T ? r.w[9 + k] : at<2>(r.w, k);
    return fmaf(h2f(T ? r.w[8] >> 16 : r.w[0] & 0xffffu), dot32(x, w), s);
  }
};

// The IQ4 level of each byte's low nibble (kIq4Levels): two 8-entry byte permutes, and a
// third that picks between them by bit 3.
constexpr uint32_t iq4_word(int i) {
  return (uint32_t)(uint8_t)kIq4Levels[i] | (uint32_t)(uint8_t)kIq4Levels[i + 1] << 8 |
         (uint32_t)(uint8_t)kIq4Levels[i + 2] << 16 | (uint32_t)(uint8_t)kIq4Levels[i + 3] << 24;
}
__device__ __forceinline__ uint32_t iq4_levels(uint32_t v) {
  const uint32_t sel = v & 0x07070707u;
  const uint32_t lo = __builtin_amdgcn_perm(iq4_word(4), iq4_word(0), sel);
  const uint32_t hi = __builtin_amdgcn_perm(iq4_word(12), iq4_word(8), sel);
  return __builtin_amdgcn_perm(hi, lo, ((v >> 1) & 0x04040404u) | 0x03020100u);
}

template <>
struct Fm<QT_IQ4_NL> {
  static constexpr int UE = 64;
  using Raw = Fm<QT_Q4_0>::Raw;
  __device__ static void load(const uint8_t* row, int u, Raw& r) { Fm<QT_Q4_0>::load(row, u, r); }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t q = T ? r.w[5 + k] : at<2>(r.w, k);
      w[k] = iq4_levels(q);
      w[4 + k] = iq4_levels(q >> 4);
    }
    return fmaf(h2f(T ? r.w[4] >> 16 : r.w[0] & 0xffffu), dot32(x, w), s);
  }
};

template <>
struct Fm<QT_IQ4_XS> {  // unit = two sub-blocks: the super-block's 8 header bytes and 32 nibble bytes
  static constexpr int UE = 64;
  struct Raw {
    uint32_t h[2], q[8];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) {
    const uint8_t* p = row + (uint32_t)(u >> 2) * 136;
    ldw<2>(p, r.h);
    ldw<8>(p + 8 + 32 * (u & 3), r.q);
  }
  template <int T>
  __device__ static float acc(const Raw& r, int u, const XBlk& x, float s) {
    const int j = 2 * (u & 3) + T;
    const int sc = (int)(((r.h[1] >> (4 * j)) & 15u) | (((r.h[0] >> (16 + 2 * j)) & 3u) << 4)) - 32;
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[k] = iq4_levels(r.q[4 * T + k]);
      w[4 + k] = iq4_levels(r.q[4 * T + k] >> 4);
    }
    return fmaf(h2f(r.h[0] & 0xffffu) * (float)sc, dot32(x, w), s);
  }
};

template <>
struct Fm<QT_Q4_K> {  // two sub-blocks: the header, 32 nibble bytes; d sc q - dmin m = d sc (q - 8) + (8 d sc - dmin m)
  static constexpr int UE = 64;
  struct Raw {
    uint32_t h[4], q[8];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) {
    const uint8_t* p = row + (uint32_t)(u >> 2) * 144;
    ldw<4>(p, r.h);
    ldw<8>(p + 16 + 32 * (u & 3), r.q);
  }
  template <int T>
  __device__ static float acc(const Raw& r, int u, const XBlk& x, float s) {
    int sc, mn;
    kq_scale_min(2 * (u & 3) + T, r.h[1], r.h[2], r.h[3], sc, mn);
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = T ? hi4s(r.q[k]) : lo4s(r.q[k]);
    const float e = h2f(r.h[0] & 0xffffu) * (float)sc;
    s = fmaf(0.0625f * e, dot32(x, w), s);
    return fmaf(fmaf(8.f, e, -h2f(r.h[0] >> 16) * (float)mn), x.s0 + x.s1, s);
  }
};

template <>
struct Fm<QT_Q5_K> {  // as q4_K with the fifth bits: d sc (q - 16) + (16 d sc - dmin m)
  static constexpr int UE = 64;
  struct Raw {
    uint32_t h[4], qh[8], q[8];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) {
    const uint8_t* p = row + (uint32_t)(u >> 2) * 176;
    ldw<4>(p, r.h);
    ldw<8>(p + 16, r.qh);
    ldw<8>(p + 48 + 32 * (u & 3), r.q);
  }
  template <int T>
  __device__ static float acc(const Raw& r, int u, const XBlk& x, float s) {
    const int j = 2 * (u & 3) + T;
    int sc, mn;
    kq_scale_min(j, r.h[1], r.h[2], r.h[3], sc, mn);
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      w[k] = (((T ? r.q[k] >> 1 : r.q[k] << 3) & 0x78787878u) | (((r.qh[k] >> j) << 7) & 0x80808080u)) ^ 0x80808080u;
    const float e = h2f(r.h[0] & 0xffffu) * (float)sc;
    s = fmaf(0.125f * e, dot32(x, w), s);
    return fmaf(fmaf(16.f, e, -h2f(r.h[0] >> 16) * (float)mn), x.s0 + x.s1, s);
  }
};

template <>
struct Fm<QT_Q2_K> {  // half a: 8 scale bytes, 32 code bytes at four shifts; d, dmin
  // d sc q - dmin m = (d sc / 2) (2q - 3) + (3 d sc / 2 - dmin m): the codes are centred, so
  // what the minimum takes off again is taken off in the scale, with one rounding
  static constexpr int UE = 128;
  struct Raw {
    uint32_t sc[2], q[8], dm[1];
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) {
    const uint8_t* p = row + (uint32_t)(u >> 1) * 84;
    const int a = u & 1;
    ldw<2>(p + 8 * a, r.sc);
    ldw<8>(p + 16 + 32 * a, r.q);
    ldw<1>(p + 80, r.dm);
  }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = __builtin_amdgcn_perm(0u, 0x0301fffdu, (r.q[k] >> (2 * T)) & 0x03030303u);
    const uint32_t sw = r.sc[T >> 1] >> (16 * (T & 1));
    const float d = 0.5f * h2f(r.dm[0] & 0xffffu), dmin = h2f(r.dm[0] >> 16);
    const float e0 = d * (float)(sw & 15u), e1 = d * (float)((sw >> 8) & 15u);
    s = fmaf(e0, dot16<0>(x, w), s);
    s = fmaf(e1, dot16<1>(x, w), s);
    s = fmaf(fmaf(3.f, e0, -dmin * (float)((sw >> 4) & 15u)), x.s0, s);
    return fmaf(fmaf(3.f, e1, -dmin * (float)((sw >> 12) & 15u)), x.s1, s);
  }
};

template <>
struct Fm<QT_Q3_K> {  // half a; 32 (q - 4): three bits at the top of their byte, top bit flipped
  static constexpr int UE = 128;
  struct Raw {
    uint32_t hm[9], q[9], t[4], sh;
    uint16_t d;
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) {
    const uint8_t* b = row + (uint32_t)(u >> 1) * 110;
    const uint8_t* p = (const uint8_t*)((uintptr_t)b & ~(uintptr_t)3);  // every part starts 0 or 2 past a dword with b
    r.sh = 8 * ((uint32_t)(uintptr_t)b & 3u);
    ldw<9>(p, r.hm);
    ldw<9>(p + 32 + 32 * (u & 1), r.q);
    ldw<3>(p + 96, r.t);
    ldw<1>(p + (r.sh ? 108 : 104), r.t + 3);
    r.d = *(const TM_GLOBAL uint16_t*)(size_t)(b + 108);
  }
  template <int T>
  __device__ static float acc(const Raw& r, int u, const XBlk& x, float s) {
    const int a4 = 4 * (u & 1);
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t q = abit(r.q[k + 1], r.q[k], r.sh), hb = abit(r.hm[k + 1], r.hm[k], r.sh) >> a4;
      const uint32_t lo = (T < 3 ? q << (5 - 2 * T) : q >> 1) & 0x60606060u;
      w[k] = (lo | ((hb << (7 - T)) & 0x80808080u)) ^ 0x80808080u;
    }
    // scale bytes 0..11
    const uint32_t t0 = abit(r.t[1], r.t[0], r.sh), t1 = abit(r.t[2], r.t[1], r.sh), t2 = abit(r.t[3], r.t[2], r.sh);
    const uint32_t lw = (T < 2 ? t0 : t1) >> a4, hw = t2 >> (a4 + 2 * (T >> 1));
    constexpr int B = 16 * (T & 1);
    const int c0 = (int)(((lw >> B) & 15u) | (((hw >> B) & 3u) << 4)) - 32;
    const int c1 = (int)(((lw >> (B + 8)) & 15u) | (((hw >> (B + 8)) & 3u) << 4)) - 32;
    const float p = fmaf((float)c0, dot16<0>(x, w), (float)c1 * dot16<1>(x, w));
    return fmaf(h2f(r.d) * 0.03125f, p, s);
  }
};

template <>
struct Fm<QT_Q6_K> {  // half a; 4 (q - 32): six bits at the top of their byte, top bit flipped
  static constexpr int UE = 128;
  struct Raw {
    uint32_t l[17], h[9], sc[3], sh;
    uint16_t d;
  };
  __device__ static void load(const uint8_t* row, int u, Raw& r) {
    const uint8_t* b = row + (uint32_t)(u >> 1) * 210;
    const uint8_t* p = (const uint8_t*)((uintptr_t)b & ~(uintptr_t)3);
    const int a = u & 1;
    r.sh = 8 * ((uint32_t)(uintptr_t)b & 3u);
    ldw<17>(p + 64 * a, r.l);
    ldw<9>(p + 128 + 32 * a, r.h);
    ldw<2>(p + 192 + 8 * a, r.sc);
    ldw<1>(p + 8 * a + (r.sh ? 200 : 196), r.sc + 2);
    r.d = *(const TM_GLOBAL uint16_t*)(size_t)(b + 208);
  }
  template <int T>
  __device__ static float acc(const Raw& r, int, const XBlk& x, float s) {
    uint32_t w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t l = abit(r.l[8 * (T & 1) + k + 1], r.l[8 * (T & 1) + k], r.sh), h = abit(r.h[k + 1], r.h[k], r.sh);
      const uint32_t n = (T < 2 ? l << 2 : l >> 2) & 0x3c3c3c3cu;
      w[k] = (n | ((h << (6 - 2 * T)) & 0xc0c0c0c0u)) ^ 0x80808080u;
    }
    const uint32_t sw = abit(r.sc[(T >> 1) + 1], r.sc[T >> 1], r.sh) >> (16 * (T & 1));
    const float p = fmaf((float)(int8_t)(sw & 255u), dot16<0>(x, w), (float)(int8_t)((sw >> 8) & 255u) * dot16<1>(x, w));
    return fmaf(h2f(r.d) * 0.25f, p, s);
  }
};

// ------------------------------------------------------------------ reductions
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int DPP_X1 = 0xb1, DPP_X2 = 0x4e, DPP_HMIRROR = 0x141, DPP_MIRROR = 0x140;
// sum over the L (16, 32 or 64) consecutive lanes that hold this one, in every lane
__device__ __forceinline__ float lanes_sum(float v, int L) {
  v += dpp<DPP_X1>(v);
  v += dpp<DPP_X2>(v);
  v += dpp<DPP_HMIRROR>(v);
  v += dpp<DPP_MIRROR>(v);
  if (L > 16) {
    const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(t[0]) + __uint_as_float(t[1]);
  }
  if (L > 32) {
    const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(t[0]) + __uint_as_float(t[1]);
  }
  return v;
}

// gemv_q's element-by-element fp32 sum of one row, by L lanes (l = this one's index)
template <int QT>
__device__ __noinline__ float row_exact(const uint8_t* row, const float* x, int K, int l, int L) {
  float s = 0.f;
  for (int c = 8 * l; c < K; c += 8 * L) {
    float v[8];
    Dec<QT>::run(row, c, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) s = fmaf(v[k], x[c + k], s);
  }
  for (int o = 1; o < L; o <<= 1) s += __shfl_xor(s, o, 64);
  return s;
}

// The word of block i of the prepared x that marks it as wide (1 or 0); then block i of the list
__device__ __forceinline__ int& wide_word(float* xs, int i) { return *(int*)(xs + i * XB + 35); }
// Lists the wide blocks of nb, in order, in place of their marks, and gives their count: one
// wave, which reads 64 marks, then writes to words that it has read
__device__ __forceinline__ int list_wide(float* xs, int nb, int lane) {
  int n = 0;
  for (int i = 0; i < nb; i += 64) {
    const bool w = i + lane < nb && wide_word(xs, min(i + lane, nb - 1));
    const uint64_t m = __ballot(w);
    if (w) wide_word(xs, n + __builtin_popcountll(m & ((1ull << lane) - 1))) = i + lane;
    n += __builtin_popcountll(m);
  }
  return n;
}

// The rows g, g + gstep, ... below ng of W again, each by L lanes (l = this one's index), after their
// digits' sums were stored in y: their products with the n listed blocks, 8 elements a lane, are added.
// Rows whose sum then is not finite, and all with n = -1 (one of them had no finite digits' sum), take
// row_exact.  y is read past the vector cache, which may hold a line of it from before other waves
// stored to it.
template <int QT>
__device__ __noinline__ void rows_wide(const uint8_t* W, size_t rb, const float* x, float* y, float* xs, int n, int K,
                                       int l, int L, int g, int ng, int gstep) {
  for (; g < ng; g += gstep) {
    const uint8_t* row = W + (size_t)(uint32_t)g * rb;
    float s = 0.f;
    for (int j = l; j < 4 * n; j += L) {
      const int c = 32 * wide_word(xs, j >> 2) + 8 * (j & 3);
      float v[8];
      Dec<QT>::run(row, c, v);
#pragma unroll
      for (int k = 0; k < 8; ++k) s = fmaf(v[k], x[c + k], s);
    }
    for (int o = 1; o < L; o <<= 1) s += __shfl_xor(s, o, 64);
    s += __hip_atomic_load(y + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (n < 0 || !__builtin_isfinite(s)) s = row_exact<QT>(row, x, K, l, L);
    if (l == 0) y[g] = s;
  }
}

// ---------------------------------------------------------------------- kernel
constexpr int NT = 1024;
constexpr int X_WIDE = 1, X_BAD = 2;  // x has wide blocks; x has NaN or Inf
// gq, gr: rows per workgroup (gq, one more for the first gr); ls = log2 L, ps = log2 P.
struct DotArgs {
  const uint8_t* W;
  size_t rb;
  const float* x;
  float* y;
  int N, K, gq, gr, ls, ps;
};

template <int QT>
__global__ __launch_bounds__(NT) void qgemv_dot(const DotArgs p) {
  using F = Fm<QT>;
  extern __shared__ __attribute__((aligned(16))) float xs[];  // K / 32 blocks of XB dwords, NT / 64 + 1 flags, parts
  const uint8_t* W = p.W;
  const size_t rb = p.rb;
  const float* x = p.x;
  const int K = p.K, ls = p.ls, ps = p.ps;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int L = 1 << ls, l = tid & (L - 1), slot = tid >> ls, NS = NT >> ls, P = 1 << ps;
  const int U = K / F::UE, b = (int)blockIdx.x;
  int* flags = (int*)(xs + (K >> 5) * XB);
  float* part = (float*)(flags + NT / 64 + 1);
  // this workgroup's rows [g0, g0 + ng); a slot takes part pt of the rows
  // slot / P, + gstep, ..., I units of each: u0, u0 + step, ... (the same count for all)
  const int ng = p.gq + (b < p.gr ? 1 : 0), g0 = b * p.gq + min(b, p.gr);
  const int pt = slot & (P - 1), gstep = NS >> ps, step = P << ls, u0 = (pt << ls) + l;
  const int I = (U + step - 1) >> (ls + ps);
  // items of this wave: those of its first slot (its other slots have as many or one row fewer)
  const int gw = (wave << (6 - ls)) >> ps;
  int total = 0;
  for (int q = gw; q < ng; q += gstep) total += I;

  // load cursor: the row, its address, the unit, units done of the row
  int lg = slot >> ps, lu = u0, li = 0;
  const uint8_t* lp;
  auto point = [&]() __attribute__((always_inline)) {
    lp = W + (size_t)(uint32_t)(g0 + min(lg, ng - 1)) * rb;
  };
  auto load = [&](typename F::Raw& d) __attribute__((always_inline)) {
    F::load(lp, min(lu, U - 1), d);
    lu += step;
    if (++li == I) {
      li = 0;
      lu = u0;
      lg += gstep;
      point();
    }
  };
  typename F::Raw ra, rc;
  point();
  if (total > 0) load(ra);

  // ---- x digits: four elements a thread, eight lanes to a block
  bool bad = false, wide = false;
  for (int i = tid; i < (K >> 2); i += NT) {
    const float4 v = *(const float4*)(x + 4 * i);
    float s = (v.x + v.y) + (v.z + v.w);
    bad |= !__builtin_isfinite(s);  // NaN, Inf, or a sum that overflows
    float m = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    m = fmaxf(m, dpp<DPP_X1>(m));
    float lo = m > 0.f ? m : INFINITY;  // the least of the eights' maxima
    s += dpp<DPP_X1>(s);
    m = fmaxf(m, dpp<DPP_X2>(m));
    lo = fminf(lo, dpp<DPP_X2>(lo));
    s += dpp<DPP_X2>(s);
    m = fmaxf(m, dpp<DPP_HMIRROR>(m));
    lo = fminf(lo, dpp<DPP_HMIRROR>(lo));
    const float so = dpp<DPP_HMIRROR>(s);  // the other half's sum
    int e = 0;
    bool wd = false;
    if (m > 0.f) {
      int ex;
      (void)frexpf(m, &ex);
      e = min(126, max(-126, 29 - ex));
      wd = ldexpf(lo, e) < 0x1p22f || ex < -97;
      wide |= wd;
    }
    uint32_t yv[4];
    yv[0] = (uint32_t)(int)ldexpf(v.x, e) + 0x00808080u;
    yv[1] = (uint32_t)(int)ldexpf(v.y, e) + 0x00808080u;
    yv[2] = (uint32_t)(int)ldexpf(v.z, e) + 0x00808080u;
    yv[3] = (uint32_t)(int)ldexpf(v.w, e) + 0x00808080u;
    const uint32_t p01l = __builtin_amdgcn_perm(yv[1], yv[0], 0x05010400u), p01h = __builtin_amdgcn_perm(yv[1], yv[0], 0x07030602u);
    const uint32_t p23l = __builtin_amdgcn_perm(yv[3], yv[2], 0x05010400u), p23h = __builtin_amdgcn_perm(yv[3], yv[2], 0x07030602u);
    uint32_t* b = (uint32_t*)xs + (i >> 3) * XB + (i & 7);
    b[0] = __builtin_amdgcn_perm(p23l, p01l, 0x05040100u) ^ 0x80808080u;
    b[8] = __builtin_amdgcn_perm(p23l, p01l, 0x07060302u) ^ 0x80808080u;
    b[16] = __builtin_amdgcn_perm(p23h, p01h, 0x05040100u) ^ 0x80808080u;
    b[24] = __builtin_amdgcn_perm(p23h, p01h, 0x07060302u);
    if ((i & 7) == 0)
      *(float4*)(xs + (i >> 3) * XB + 32) = wd ? make_float4(0.f, 0.f, 0.f, __int_as_float(1)) : make_float4(ldexpf(1.f, -e), s, so, 0.f);
  }
  {
    const bool wbad = __ballot(bad) != 0, wwide = __ballot(wide) != 0;
    if (lane == 0) flags[wave] = (wbad ? X_BAD : 0) | (wwide ? X_WIDE : 0);
  }
  __syncthreads();

  int xf = 0;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) xf |= flags[i];
  const bool xbad = xf >= X_BAD, xwide = xf == X_WIDE;  // the same for every wave
  bool odd = false;  // a sum is not finite
  float acc = 0.f;
  int g = slot >> ps, u = u0, ci = 0;
  auto compute = [&](const typename F::Raw& raw) __attribute__((always_inline)) {
    if (u < U) {
      auto block = [&](auto T) __attribute__((always_inline)) {
        XBlk xb;
        xb.load(xs, u * (F::UE / 32) + decltype(T)::value);
        acc = F::template acc<decltype(T)::value>(raw, u, xb, acc);
      };
      using std::integral_constant;
      block(integral_constant<int, 0>{});
      block(integral_constant<int, 1>{});
      if constexpr (F::UE == 128) {
        block(integral_constant<int, 2>{});
        block(integral_constant<int, 3>{});
      }
    }
    u += step;
    if (++ci == I) {  // the row is complete
      ci = 0;
      u = u0;
      float s = lanes_sum(acc, L);
      acc = 0.f;
      if (g < ng) {
        if (ps) {
          if (l == 0) part[(g << ps) + pt] = s;
        } else {
          if (__builtin_expect(xbad || !__builtin_isfinite(s), 0)) {
            s = row_exact<QT>(W + (size_t)(uint32_t)(g0 + g) * rb, x, K, l, L);
            odd = true;
          }
          if (l == 0) p.y[g0 + g] = s;
        }
      }
      g += gstep;
    }
  };
  int it = 0;
  for (; it + 2 < total; it += 2) {
    load(rc);
    compute(ra);
    load(ra);
    compute(rc);
  }
  if (total - it == 2) {
    load(rc);
    compute(ra);
    compute(rc);
  } else if (total - it == 1) {
    compute(ra);
  }
  if (ps) {
    __syncthreads();
    for (int i = slot; i < ng; i += NS) {
      float s = 0.f;
      for (int q = 0; q < P; ++q) s += part[(i << ps) + q];
      if (__builtin_expect(xbad || !__builtin_isfinite(s), 0)) {
        s = row_exact<QT>(W + (size_t)(uint32_t)(g0 + i) * rb, x, K, l, L);
        odd = true;
      }
      if (l == 0) p.y[g0 + i] = s;
    }
  }
  if (__builtin_expect(__ballot(xwide) != 0, 0)) {
    if (wave == 0) {
      const int c = list_wide(xs, K >> 5, lane);
      if (lane == 0) flags[NT / 64] = c;
    }
    __syncthreads();
    rows_wide<QT>(W + (size_t)(uint32_t)g0 * rb, rb, x, p.y + g0, xs, odd ? -1 : flags[NT / 64], K, l, L, slot, ng, NS);
  }
}

constexpr int kDotMaxLds = 160 * 1024;
size_t dot_lds(int K, int rows, int ps) {
  return (size_t)(K / 32) * XB * 4 + (NT / 64 + 1) * 4 + (ps ? ((size_t)rows << ps) * 4 : 0);
}

template <int QT>
int launch_dot(const void* W, size_t rb, const float* x, float* y, int N, int K, int cus, hipStream_t s) {
  DotArgs a{};
  a.W = (const uint8_t*)W; a.rb = rb; a.x = x; a.y = y; a.N = N; a.K = K;
  const int U = K / Fm<QT>::UE, nb = std::min(N, cus), ng = (N + nb - 1) / nb;
  // lanes and parts per row: the fewest unit steps per slot; on a tie the fewest parts
  // (a row in one part is stored without the barrier and the sum over parts), then the
  // widest rows
  long best = -1;
  for (int ps = 0; ps <= 4; ++ps)
    for (int ls = 6; ls >= 4; --ls) {
      const int gstep = (NT >> ls) >> ps;
      if (!gstep || (ps && dot_lds(K, ng, ps) > (size_t)kDotMaxLds)) continue;
      const long it = (long)((ng + gstep - 1) / gstep) * ((U + (1 << (ps + ls)) - 1) >> (ps + ls));
      if (best < 0 || it < best) {
        best = it;
        a.ls = ls;
        a.ps = ps;
      }
    }
  a.gq = N / nb; a.gr = N % nb;
  static std::atomic<uint64_t> attr{0};
  int st = lds_attr_once(attr, (const void*)qgemv_dot<QT>, kDotMaxLds, "tiermm_qgemv");
  if (st) return st;
  qgemv_dot<QT><<<nb, NT, dot_lds(K, ng, a.ps), s>>>(a);
  TM_LAUNCH_CHECK("tiermm_qgemv: launch");
  return TIERMM_OK;
}

}  // namespace

// Types the dot kernel decodes, in whole units of 64, W on a dword (rows of q3_K and q6_K
// then start on any even address); K up to the LDS that the prepared x takes.
bool qgemv_dot_takes(const void* W, int qtype, int K) {
  if (K <= 0 || K % 64 || ((uintptr_t)W & 3) || dot_lds(K, 0, 0) > (size_t)kDotMaxLds) return false;
  switch (qtype) {
    case QT_Q4_0: case QT_Q4_1: case QT_Q5_0: case QT_Q5_1: case QT_Q8_0: case QT_IQ4_NL:
    case QT_Q2_K: case QT_Q3_K: case QT_Q4_K: case QT_Q5_K: case QT_Q6_K: case QT_IQ4_XS: return true;
    default: return false;
  }
}

int qgemv_dot(const void* W, int qtype, size_t rb, const float* x, float* y, int N, int K, hipStream_t s) {
  int cus = 0;
  int st = device_cus(&cus);
  if (st) return st;
  switch (qtype) {
    case QT_Q4_0: return launch_dot<QT_Q4_0>(W, rb, x, y, N, K, cus, s);
    case QT_Q4_1: return launch_dot<QT_Q4_1>(W, rb, x, y, N, K, cus, s);
    case QT_Q5_0: return launch_dot<QT_Q5_0>(W, rb, x, y, N, K, cus, s);
    case QT_Q5_1: return launch_dot<QT_Q5_1>(W, rb, x, y, N, K, cus, s);
    case QT_Q8_0: return launch_dot<QT_Q8_0>(W, rb, x, y, N, K, cus, s);
    case QT_IQ4_NL: return launch_dot<QT_IQ4_NL>(W, rb, x, y, N, K, cus, s);
    case QT_Q2_K: return launch_dot<QT_Q2_K>(W, rb, x, y, N, K, cus, s);
    case QT_Q3_K: return launch_dot<QT_Q3_K>(W, rb, x, y, N, K, cus, s);
    case QT_Q6_K: return launch_dot<QT_Q6_K>(W, rb, x, y, N, K, cus, s);
    case QT_Q4_K: return launch_dot<QT_Q4_K>(W, rb, x, y, N, K, cus, s);
    case QT_Q5_K: return launch_dot<QT_Q5_K>(W, rb, x, y, N, K, cus, s);
    case QT_IQ4_XS: return launch_dot<QT_IQ4_XS>(W, rb, x, y, N, K, cus, s);
    default: return set_error(TIERMM_UNSUPPORTED, "tiermm_qgemv: type %d", qtype);
  }
}

}  // namespace tiermm
