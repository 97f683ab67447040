// qgemm_skinny.hip -- quantized GEMM for few rows of x (1 .. 48): short prompts of a running
// chat, routed experts of a small batch.  q4_K, q5_K, q6_K, q8_0, q5_0, in both modes.
//
// What bounds it: at these row counts the weight bytes are read once for a few MFMAs, so the
// floor is their read.  The fused kernel (qgemm_fused.hip) spends the time elsewhere: it decodes
// each weight to fp16 in LDS through fp32 arithmetic (F32: two parts, after a pass over all
// block scales for the row exponents) and multiplies 128- or 256-row tiles that are mostly
// padding.  Here a lane decodes the 16 weights that it holds as an MFMA operand, in registers:
//   - the bytes of a unit (256 elements of 16 * WR * RW rows) come by LDS DMA, whose consecutive
//     lanes read consecutive 16-byte chunks of a row (loaded straight into the lanes that need
//     them, every lane of a load is in another row);
//   - codes are read as fp16 subnormals (no conversions), and for F32 the block scale is applied
//     to the sums where the code times its sub-block scale is a whole number that fp16 holds
//     (q4_K, q5_K: two products, x hi and lo, where the fused kernel has three, and no pass over
//     the scales).  The codes are centred, d sc q - dmin m = d sc (q - c) + (c d sc - dmin m), c = 8
//     or 16, and the second term, one fp32 factor a sub-block, is one product with the sub-block
//     sums of the split x.  With the codes as they are the two terms are each several times their
//     difference, and what rounds in either stays: q4_K 300x5120, M = 37, rows of x that are
//     constant 1.1e-5 off 64 bits -> 2.8e-7, 3 + n 1.2e-6 -> 2.1e-7 (fused kernel 4.0e-7);
//   - x is split and laid out as operand fragments once, by a launch before.
// Measured, all launches of a call, in us, graph replays over rotated weights (fused kernel -> this one):
//   F32, N = 14336, K = 5120:  q4_K M = 2  58.7 -> 25.9, M = 37  61.3 -> 39.2;  q5_K M = 2  63.5 -> 28.7,
//     M = 37  66.0 -> 41.9;  q6_K M = 2  61.6 -> 34.6, M = 37  64.2 -> 47.3;  q8_0 M = 2  69.9 -> 32.6
//   F32, N = 1024, K = 4096:  q4_K M = 2  23.8 -> 14.3, M = 37  25.3 -> 21.0
//   x-ref, N = 14336, K = 5120:  q4_K M = 2  45.8 -> 24.3, M = 16  47.9 -> 27.3, M = 32  44.3 -> 31.7;
//     q6_K M = 16  56.9 -> 34.9;  q8_0 M = 16  63.6 -> 38.5;  q5_0 M = 4  49.6 -> 29.0
// with errors against fp64 no larger (F32 q4_K, N(0, 1): 4.0e-7 -> 1.4e-7).  What is left over the
// weights' read (8 us at q4_K) is the split and reduce launches (4 to 5 us each) and, at M = 37 in the
// kernel's 34 us, 15 us of VALU issue (mostly decode), 7 of MFMAs, 6 of LDS reads and 13 of the
// vector memory's return path, which overlap in part: four waves a SIMD meet at a barrier every unit.
#include <algorithm>

#include "tm_device.h"

namespace tiermm {

int device_cus(int* cus);

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));

constexpr int SK_G = 64;          // groups per launch
constexpr int SK_MT = 3;          // 16-row tiles of x, at most
constexpr int SK_WR = 2;          // 16-row W tiles of a wave
// Up to sk_pack rows, the parts of x share one MFMA tile: row m of part p at tile row m + p sk_pack
// (x-ref three parts of 4 rows, F32 two of 8).  One product then does the work of three (two), x takes
// a third (half) of the loads and LDS, and that room holds a third unit of weights in flight and the
// meeting apart from the ring, so the loads no longer stop between two items.
// Measured before and after on one card, us a call: 8 tokens, top 8 of 64 experts, hidden 2048, ffn
// 1408 (both products and the combine) 127 -> 108, 1 token 44.7 -> 41.9; F32 q4_K 14336x5120 M = 8
// 27.1 -> 26.2.  (The fused kernel took 243 for the 8 tokens.)
constexpr int sk_pack(bool f32) { return f32 ? 8 : 4; }
// Row waves of a workgroup, each for four K quarters, by the row tiles of x
constexpr int sk_rw(int mt) { return mt == 1 ? 2 : 4; }
constexpr int sk_bn(int mt) { return 16 * SK_WR * sk_rw(mt); }
constexpr int SK_UNIT = 256;      // K per step of the K loop (8 MFMA steps of 32)

struct SkArgs {
  const uint16_t* X;  // fragments [unit][step 8][part][tile][64 lanes][8 halfs]
  const uint16_t* S;  // F32, formats with minima: sub-block sums [unit][tile][t 2][64 lanes][4 halfs], or with
                      // one row tile a group (flat) [unit][tile][sub-block 8][16 rows] floats
  float* Y;
  float* P;           // KS > 1: partial sums of split z at P + z * ps, rows of N floats
  const int32_t* xexp;
  size_t rb, ps;
  int ldy, N, K, KS, mtot, ngroups, flat;
  float beta;
  int tile0[SK_G + 1];  // workgroup tiles of group g: [tile0[g], tile0[g + 1])
  int row0[SK_G], rows[SK_G], mt0[SK_G];  // rows of x and Y; its first x tile
  int first[SK_G];                         // rows of the groups before it
  const uint8_t* W[SK_G];
};

// ------------------------------------------------------------ x fragments
// Element (row m, k) of x is half e of lane 16 kg + m of fragment step s of unit k / 256:
// within the unit's half kh = 128 elements, k = 64 (kg / 2) + 32 t + 16 (kg % 2) + 8 u + e,
// s = 4 kh + 2 t + u.  (A lane's weights are then 16 consecutive elements of two
// neighbouring 32-element blocks.)  PERM: the 8 halfs in the order 0 2 1 3 4 6 5 7, in
// which the F32 decoders pair nibbles.
template <int NP, bool PERM, bool PACK>
__device__ __forceinline__ void put_frag(uint16_t* X, size_t mtot, size_t tile, int m, int k,
                                         const uint16_t (&h)[NP][8]) {
  const int r = k & 127, kg = 2 * (r >> 6) + ((r >> 4) & 1);
  const int s = 4 * ((k >> 7) & 1) + 2 * ((r >> 5) & 1) + ((r >> 3) & 1);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const size_t f = ((size_t)((k >> 8) * 8 + s) * (PACK ? 1 : NP) + (PACK ? 0 : p)) * mtot + tile;
    const int row = PACK ? m + p * sk_pack(NP == 2) : m;
    const uint16_t(&v)[8] = h[p];
    const u32x4 o = PERM ? u32x4{v[0] | (uint32_t)v[2] << 16, v[1] | (uint32_t)v[3] << 16, v[4] | (uint32_t)v[6] << 16,
                                 v[5] | (uint32_t)v[7] << 16}
                         : u32x4{v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16, v[4] | (uint32_t)v[5] << 16,
                                 v[6] | (uint32_t)v[7] << 16};
    *(u32x4*)(X + f * 512 + (16 * kg + row) * 8) = o;
  }
}
__device__ __forceinline__ void load8(const float* x, bool al, float (&v)[8]) {
  if (al) {
    const float4 a = *(const float4*)x, b = *(const float4*)(x + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = x[e];
  }
}
// The last of the n <= 64 ascending starts that is <= i: one load a lane, instead of a scalar
// walk whose every step waits for its load
__device__ __forceinline__ int group_of(const int* start, int n, int i) {
  const int lane = threadIdx.x & 63;
  return __builtin_popcountll(__ballot(lane < n && start[lane < n ? lane : 0] <= i)) - 1;
}
// Row, tile and row in the tile of the i-th row of the groups
__device__ __forceinline__ int row_place(const SkArgs& p, int i, size_t& tile, int& m) {
  const int g = p.ngroups == 1 ? 0 : __builtin_amdgcn_readfirstlane(group_of(p.first, p.ngroups, i));
  const int q = i - p.first[g];
  tile = p.mt0[g] + (q >> 4);
  m = q & 15;
  return p.row0[g] + q;
}

// x-ref: the three fp16 parts (split3_fp_k, tier.cpp:869-870); one row per block.  K past the
// row is zero up to a whole unit.
template <bool PACK>
__global__ __launch_bounds__(1024) void sk_split3(const float* __restrict__ x, const SkArgs p,
                                                 uint16_t* __restrict__ X) {
  const int K = p.K, kp = (K + SK_UNIT - 1) / SK_UNIT * SK_UNIT;
  size_t tile;
  int m;
  const int row = row_place(p, (int)blockIdx.x, tile, m);
  const float* xr = x + (size_t)row * K;
  const bool al = ((uintptr_t)xr & 15) == 0;
  for (int k = 8 * threadIdx.x; k < kp; k += 8 * blockDim.x) {
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (k < K) load8(xr + k, al, v);
    uint16_t h[3][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[0][e] = f2h(v[e]);
      const float r1 = v[e] - h2f(h[0][e]);
      h[1][e] = f2h(r1);
      h[2][e] = f2h(r1 - h2f(h[1][e]));
    }
    put_frag<3, false, PACK>(X, p.mtot, tile, m, k, h);
  }
}
// The same fragments from parts that are split already (planes part_stride apart; kt > 0:
// K-tiled over kt rows).
template <bool PACK>
__global__ __launch_bounds__(1024) void sk_relayout3(const uint16_t* __restrict__ parts, size_t stride, size_t kt,
                                                    const SkArgs p, uint16_t* __restrict__ X) {
  const int K = p.K, kp = (K + SK_UNIT - 1) / SK_UNIT * SK_UNIT;
  size_t tile;
  int m;
  const int row = row_place(p, (int)blockIdx.x, tile, m);
  for (int k = 8 * threadIdx.x; k < kp; k += 8 * blockDim.x) {
    uint16_t h[3][8];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const size_t at = q * stride + (kt ? ktile_index((size_t)row, k, kt) : (size_t)row * K + k);
      const u32x4 w = k < K ? *(const u32x4*)(parts + at) : u32x4{0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 8; ++e) h[q][e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
    put_frag<3, false, PACK>(X, p.mtot, tile, m, k, h);
  }
}

// F32: the two-part split with a power of two per row (x3s_split's), and with S the
// sub-block sums S_b = sum of hi + lo (what the products see of x) over the 32 elements of
// sub-block b: fp32 values (flat), or over 32 in two fp16 parts: lane (m, kg) of the unit's sum
// fragment t holds hi, hi, lo, lo of sub-block b = 4 (kg % 2) + 2 (kg / 2) + t.
template <bool PACK>
__global__ __launch_bounds__(1024) void sk_split2(const float* __restrict__ x, const SkArgs p, uint16_t* __restrict__ X,
                                                 uint16_t* __restrict__ S, int32_t* __restrict__ xexp) {
  __shared__ float red[16];
  const int K = p.K, kp = (K + SK_UNIT - 1) / SK_UNIT * SK_UNIT;
  size_t tile;
  int m;
  const int row = row_place(p, (int)blockIdx.x, tile, m);
  const float* xr = x + (size_t)row * K;
  const bool al = ((uintptr_t)xr & 15) == 0;
  float amax = 0.f;
  for (int k = 8 * threadIdx.x; k < K; k += 8 * blockDim.x) {
    float v[8];
    load8(xr + k, al, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[e]));
  }
#pragma unroll
  for (int d = 32; d; d >>= 1) amax = fmaxf(amax, __shfl_xor(amax, d, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  for (unsigned i = 0; i < blockDim.x >> 6; ++i) amax = fmaxf(amax, red[i]);
  const int ex = x3s_exp(amax);
  const float sc = ldexpf(1.f, ex);
  if (threadIdx.x == 0) xexp[row] = ex;
  for (int k = 8 * threadIdx.x; k < kp; k += 8 * blockDim.x) {
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (k < K) load8(xr + k, al, v);
    uint16_t h[2][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = v[e] * sc;
      h[0][e] = f2h(f);
      h[1][e] = f2h(f - h2f(h[0][e]));
      v[e] = h2f(h[0][e]) + h2f(h[1][e]);  // exact
    }
    put_frag<2, true, PACK>(X, p.mtot, tile, m, k, h);
    if (S) {  // four neighbouring lanes hold a sub-block; in pairs, so that equal values add without rounding
      float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
      sum += __shfl_xor(sum, 1, 64);
      sum += __shfl_xor(sum, 2, 64);
      const float s32 = sum * 0.03125f;
      const uint32_t s0 = f2h(s32), s1 = f2h(s32 - h2f((uint16_t)s0));
      const int b = (k >> 5) & 7, kg = 2 * ((b >> 1) & 1) + (b >> 2);
      uint16_t* f = S + ((size_t)(k >> 8) * p.mtot + tile) * 512;
      if ((k & 31) == 0 && p.flat) {
        float* o = (float*)f + 16 * b + m;
        *o = sum;
        if (PACK) o[sk_pack(true)] = 0.f;
      } else if ((k & 31) == 0) {
        u32x2* o = (u32x2*)(f + 256 * (b & 1) + (16 * kg + m) * 4);
        *o = u32x2{s0 * 0x10001u, s1 * 0x10001u};
        if (PACK) o[sk_pack(true)] = u32x2{0, 0};  // the sums count once, with the hi parts
      }
    }
  }
}

// ------------------------------------------------------------ weight decoders
// A unit of a row is its bytes of 256 elements.  In LDS it starts at the dword that holds its
// first byte (ph = 0 or 2 bytes before it) and is CH chunks of 16 bytes long; with TAIL the dword
// after those lies in a region of its own (tail).  A lane of quarter (kh, t) reads the 16 elements
// of block 4 kh + 2 (kg / 2) + t that start at 16 (kg % 2).  dec<F32> gives fp16(q_val) for
// x-ref; for F32 integers times 2^PW or (PLANES == 2) block values in two fp16 parts, and post()
// is what their sums are multiplied by.
template <int QT>
struct Sk;

__device__ __forceinline__ uint32_t abit(uint32_t hi, uint32_t lo, uint32_t sh) {
  return __builtin_amdgcn_alignbit(hi, lo, sh);
}
__device__ __forceinline__ uint32_t rotr(uint32_t v, int n) { return abit(v, v, (uint32_t)n & 31u); }
__device__ __forceinline__ h2v as_h2(uint32_t v) { return __builtin_bit_cast(h2v, v); }
__device__ __forceinline__ uint32_t as_u(h2v v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2v dup(float f) { return h2v{(_Float16)f, (_Float16)f}; }
// Codes are read as fp16 subnormals: the 8-bit code c in a 16-bit lane is c * 2^-24, with no
// conversion.  A pair of x-ref weights fp16(fma(s, code, m)) from such a pair and s * 2^24: one
// v_fma_mixlo / _mixhi each (fp32 fma, then rounded to fp16).
__device__ __forceinline__ uint32_t mix2(uint32_t codes, float s24, float m) {
  const h2v c = as_h2(codes);
  return as_u(h2v{(_Float16)fmaf((float)c[0], s24, m), (_Float16)fmaf((float)c[1], s24, m)});
}
// The same for the four codes of v's bytes in element order
__device__ __forceinline__ void mix4(uint32_t v, float s24, float m, uint32_t& o0, uint32_t& o1) {
  o0 = mix2(__builtin_amdgcn_perm(0u, v, 0x0c010c00u), s24, m);
  o1 = mix2(__builtin_amdgcn_perm(0u, v, 0x0c030c02u), s24, m);
}
// v is NaN where it is not finite: a block with such a scale makes its row NaN
__device__ __forceinline__ float or_nan(float v) { return __builtin_isfinite(v) ? v : __builtin_nanf(""); }
// Two fp16 parts of s * (integers in q): hi rounded, lo the remainder
__device__ __forceinline__ void two_parts(h2v q, h2v s, uint32_t& hi, uint32_t& lo) {
  const h2v p = q * s;
  hi = as_u(p);
  lo = as_u(__builtin_elementwise_fma(q, s, -p));
}
// 16 bytes at byte offset off (even) of a unit, off counted from its LDS start; `end`: the offset
// of the tail dword
__device__ __forceinline__ void win16(const uint8_t* w, const uint8_t* tail, int end, int off, uint32_t (&o)[4]) {
  const int al = off & ~3;
  const uint32_t sh = (uint32_t)(off & 2) * 8u;
  uint32_t p[5];
#pragma unroll
  for (int k = 0; k < 4; ++k) p[k] = *(const uint32_t*)(w + al + 4 * k);
  p[4] = *(const uint32_t*)(al + 16 >= end ? tail : w + al + 16);
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = abit(p[k + 1], p[k], sh);
}
__device__ __forceinline__ float half_at(const uint8_t* p) { return h2f(*(const uint16_t*)p); }
// The largest of v over the four lanes (n, kg) of a row n
__device__ __forceinline__ float kg_max(float v) {
  const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
  const auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(u[0]), __uint_as_float(u[1]));
}
// 2^e that brings the largest |d| of a row's blocks in the quarter into [2^6, 2^7), so that
// d 2^e times a code (at most 128) stays below 2^14
__device__ __forceinline__ float block_norm(float d) {
  const float m = kg_max(fabsf(d));
  int ex;
  (void)frexpf(m, &ex);
  return m > 0.f && m < INFINITY ? ldexpf(1.f, 7 - ex) : 1.f;
}

// q4_K / q5_K: scale (MIN: minimum) bytes of a half unit's four sub-blocks
template <bool MIN>
__device__ __forceinline__ uint32_t kq_bytes(u32x4 h, int kh) {
  const uint32_t lo = MIN ? h[2] : h[1];
  return kh ? ((h[3] >> (MIN ? 4 : 0)) & 0x0f0f0f0fu) | ((lo >> 2) & 0x30303030u) : lo & 0x3f3f3f3fu;
}
// q4_K / q5_K, codes centred by C: the factor C d sc - dmin m of this lane's sub-block
template <int C>
__device__ __forceinline__ float kq_factor(u32x4 h, int kh, int t, int kg) {
  const int sh = 16 * (kg >> 1) + 8 * t;
  const float m = h2f(h[0] >> 16) * (float)((kq_bytes<true>(h, kh) >> sh) & 0xffu);  // exact
  return fmaf((float)C * h2f(h[0] & 0xffffu), (float)((kq_bytes<false>(h, kh) >> sh) & 0xffu), -m);
}
// The same in two fp16 parts, times a power of two that keeps it below 2^15 (126 max(C |d|, |dmin|)
// bounds it), against the hi and lo sums, in the lanes kg % 2 == kh and zero in the others; inv = 32
// over that power, which takes the product to the factor's own scale
template <int C>
__device__ __forceinline__ u32x2 kq_offset(u32x4 h, int kh, int t, int kg, float& inv) {
  const float b = kq_factor<C>(h, kh, t, kg);
  // the exponent is 0 for 0, Inf and NaN; non-finite factors stay so
  const int e = 8 - __builtin_amdgcn_frexp_expf(fmaxf((float)C * fabsf(h2f(h[0] & 0xffffu)), fabsf(h2f(h[0] >> 16))));
  inv = ldexpf(32.f, -e);
  const float v = ldexpf(b, e);
  const uint32_t hi = f2h(v), lo = f2h(v - h2f((uint16_t)hi));
  const uint32_t w = (kg & 1) == kh ? hi | lo << 16 : 0u;
  return u32x2{w, w};
}

template <>
struct Sk<QT_Q4_K> {
  static constexpr int UB = 144, CH = 9, PLANES = 1;
  static constexpr bool TAIL = false, MINS = true;
  u32x4 h, q;
  __device__ __forceinline__ void read(const uint8_t* w, const uint8_t*, int, int kh, int, int kg, bool) {
    h = *(const u32x4*)w;
    q = *(const u32x4*)(w + 16 + 64 * kh + 16 * kg);
  }
  template <bool F32>
  __device__ __forceinline__ void dec(int kh, int t, int kg, uint32_t (&o)[8], uint32_t (&)[8], float) const {
    const int sh = 16 * (kg >> 1) + 8 * t;
    const uint32_t sc = (kq_bytes<false>(h, kh) >> sh) & 0xffu;
    if constexpr (!F32) {
      const uint32_t mn = (kq_bytes<true>(h, kh) >> sh) & 0xffu;
      const float dsc = h2f(h[0] & 0xffffu) * (float)sc, dm = h2f(h[0] >> 16) * (float)mn;
#pragma unroll
      for (int k = 0; k < 4; ++k) mix4((q[k] >> (4 * t)) & 0x0f0f0f0fu, dsc * 0x1p24f, -dm, o[2 * k], o[2 * k + 1]);
    } else {
      // sc (q - 8) 2^-14, sc |q - 8| at most 504: exact.  q as a subnormal times sc 2^10, less 8 sc 2^-14
      const h2v a = dup((float)(sc << 10)), z = dup((float)sc * -0x1p-11f);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        o[2 * k] = as_u(__builtin_elementwise_fma(as_h2((q[k] >> (4 * t)) & 0x000f000fu), a, z));
        o[2 * k + 1] = as_u(__builtin_elementwise_fma(as_h2((q[k] >> (8 + 4 * t)) & 0x000f000fu), a, z));
      }
    }
  }
  __device__ __forceinline__ float norm() const { return 1.f; }
  // (a d that is not finite makes the factor or its parts, and the row, NaN)
  __device__ __forceinline__ float post(float) const { return h2f(h[0] & 0xffffu) * 0x1p14f; }
  __device__ __forceinline__ u32x2 offset(int kh, int t, int kg, float& inv) const {
    return kq_offset<8>(h, kh, t, kg, inv);
  }
  __device__ __forceinline__ float factor(int kh, int t, int kg) const { return kq_factor<8>(h, kh, t, kg); }
};

template <>
struct Sk<QT_Q5_K> {
  static constexpr int UB = 176, CH = 11, PLANES = 1;
  static constexpr bool TAIL = false, MINS = true;
  u32x4 h, qh, q;
  __device__ __forceinline__ void read(const uint8_t* w, const uint8_t*, int, int kh, int, int kg, bool) {
    h = *(const u32x4*)w;
    qh = *(const u32x4*)(w + 16 + 16 * (kg & 1));
    q = *(const u32x4*)(w + 48 + 64 * kh + 16 * kg);
  }
  template <bool F32>
  __device__ __forceinline__ void dec(int kh, int t, int kg, uint32_t (&o)[8], uint32_t (&)[8], float) const {
    const int sb = 4 * kh + 2 * (kg >> 1) + t, sh = 16 * (kg >> 1) + 8 * t;
    const uint32_t sc = (kq_bytes<false>(h, kh) >> sh) & 0xffu;
    uint32_t v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = ((q[k] >> (4 * t)) & 0x0f0f0f0fu) | (rotr(qh[k], sb - 4) & 0x10101010u);
    if constexpr (!F32) {
      const uint32_t mn = (kq_bytes<true>(h, kh) >> sh) & 0xffu;
      const float dsc = h2f(h[0] & 0xffffu) * (float)sc, dm = h2f(h[0] >> 16) * (float)mn;
#pragma unroll
      for (int k = 0; k < 4; ++k) mix4(v[k], dsc * 0x1p24f, -dm, o[2 * k], o[2 * k + 1]);
    } else {  // sc (q - 16) 2^-14, sc |q - 16| at most 1008: exact
      const h2v a = dup((float)(sc << 10)), z = dup((float)sc * -0x1p-10f);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        o[2 * k] = as_u(__builtin_elementwise_fma(as_h2(v[k] & 0x00ff00ffu), a, z));
        o[2 * k + 1] = as_u(__builtin_elementwise_fma(as_h2((v[k] >> 8) & 0x00ff00ffu), a, z));
      }
    }
  }
  __device__ __forceinline__ float norm() const { return 1.f; }
  // (a d that is not finite makes the factor or its parts, and the row, NaN)
  __device__ __forceinline__ float post(float) const { return h2f(h[0] & 0xffffu) * 0x1p14f; }
  __device__ __forceinline__ u32x2 offset(int kh, int t, int kg, float& inv) const {
    return kq_offset<16>(h, kh, t, kg, inv);
  }
  __device__ __forceinline__ float factor(int kh, int t, int kg) const { return kq_factor<16>(h, kh, t, kg); }
};

template <>
struct Sk<QT_Q6_K> {
  static constexpr int UB = 210, CH = 13, PLANES = 2;
  static constexpr bool TAIL = true, MINS = false;
  uint32_t wl[4], wh[4];
  float d;
  int sc;
  __device__ __forceinline__ void read(const uint8_t* w, const uint8_t* tail, int ph, int kh, int t, int kg, bool) {
    const int hf = kg & 1;
    win16(w, tail, 16 * CH, ph + 64 * kh + 32 * t + 16 * hf, wl);
    win16(w, tail, 16 * CH, ph + 128 + 32 * kh + 16 * hf, wh);
    const int so = ph + 192 + 8 * kh + 4 * (kg >> 1) + 2 * t + hf;
    sc = (int)*(const int8_t*)(so >= 16 * CH ? tail + (so - 16 * CH) : w + so);
    d = half_at(tail + ph);
  }
  template <bool F32>
  __device__ __forceinline__ void dec(int, int t, int kg, uint32_t (&o)[8], uint32_t (&ol)[8], float) const {
    // block r = 2 (kg / 2) + t of the half: nibble kg / 2, qh bits 2 r
    const int n4 = 4 * (kg >> 1), h2 = 4 * (kg >> 1) + 2 * t;
    uint32_t v[4];  // 4 q as bytes
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = (rotr(wl[k], n4 - 2) & 0x3c3c3c3cu) | (rotr(wh[k], h2 - 6) & 0xc0c0c0c0u);
    if constexpr (!F32) {
      const float ds = d * (float)sc;
#pragma unroll
      for (int k = 0; k < 4; ++k) mix4(v[k], ds * 0x1p22f, -32.f * ds, o[2 * k], o[2 * k + 1]);
    } else {
      // sc * (q - 32), at most 4096, in two fp16 parts
      const h2v u = dup(0x1p15f), off = dup(-0.25f), s = dup((float)(sc * 128));
#pragma unroll
      for (int k = 0; k < 4; ++k) {  // (q - 32) / 128 first
        two_parts(__builtin_elementwise_fma(as_h2(v[k] & 0x00ff00ffu), u, off), s, o[2 * k], ol[2 * k]);
        two_parts(__builtin_elementwise_fma(as_h2((v[k] >> 8) & 0x00ff00ffu), u, off), s, o[2 * k + 1], ol[2 * k + 1]);
      }
    }
  }
  __device__ __forceinline__ float norm() const { return 1.f; }
  __device__ __forceinline__ float post(float) const { return or_nan(d); }
};

// q8_0 / q5_0 for F32: d 2^e * (code - ZERO) in two fp16 parts, code bytes in v
template <int ZERO>
__device__ __forceinline__ void block_parts(const uint32_t (&v)[4], float d, uint32_t (&o)[8], uint32_t (&ol)[8]) {
  const h2v s = dup(d), off = dup(-1024.f - ZERO);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    two_parts(as_h2((v[k] & 0x00ff00ffu) | 0x64006400u) + off, s, o[2 * k], ol[2 * k]);
    two_parts(as_h2(((v[k] >> 8) & 0x00ff00ffu) | 0x64006400u) + off, s, o[2 * k + 1], ol[2 * k + 1]);
  }
}

template <>
struct Sk<QT_Q8_0> {
  static constexpr int UB = 272, CH = 17, PLANES = 2;
  static constexpr bool TAIL = true, MINS = false;
  uint32_t v[4];  // code + 128 as bytes
  float d;
  __device__ __forceinline__ void read(const uint8_t* w, const uint8_t* tail, int ph, int kh, int t, int kg, bool in) {
    const int off = ph + 34 * (4 * kh + 2 * (kg >> 1) + t);
    d = in ? half_at(w + off) : 0.f;
    win16(w, tail, 16 * CH, off + 2 + 16 * (kg & 1), v);
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] ^= 0x80808080u;
  }
  template <bool F32>
  __device__ __forceinline__ void dec(int, int, int, uint32_t (&o)[8], uint32_t (&ol)[8], float nm) const {
    if constexpr (!F32) {
#pragma unroll
      for (int k = 0; k < 4; ++k) mix4(v[k], d * 0x1p24f, -128.f * d, o[2 * k], o[2 * k + 1]);
    } else {
      block_parts<128>(v, d * nm, o, ol);
    }
  }
  __device__ __forceinline__ float norm() const { return block_norm(or_nan(d)); }
  __device__ __forceinline__ float post(float nm) const { return 1.f / nm; }
};

template <>
struct Sk<QT_Q5_0> {
  static constexpr int UB = 176, CH = 11, PLANES = 2;
  static constexpr bool TAIL = true, MINS = false;
  uint32_t v[4];  // codes 0 .. 31 as bytes
  float d;
  __device__ __forceinline__ void read(const uint8_t* w, const uint8_t* tail, int ph, int kh, int t, int kg, bool in) {
    const int hf = kg & 1, off = ph + 22 * (4 * kh + 2 * (kg >> 1) + t);
    d = in ? half_at(w + off) : 0.f;
    const uint32_t q = *(const uint16_t*)(w + off + 2 + 2 * hf);  // the 16 fifth bits
    win16(w, tail, 16 * CH, off + 6, v);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      v[k] = ((v[k] >> (4 * hf)) & 0x0f0f0f0fu) | (((__umul24((q >> (4 * k)) & 15u, 0x00204081u)) & 0x01010101u) << 4);
  }
  template <bool F32>
  __device__ __forceinline__ void dec(int, int, int, uint32_t (&o)[8], uint32_t (&ol)[8], float nm) const {
    if constexpr (!F32) {
#pragma unroll
      for (int k = 0; k < 4; ++k) mix4(v[k], d * 0x1p24f, -16.f * d, o[2 * k], o[2 * k + 1]);
    } else {
      block_parts<16>(v, d * nm, o, ol);
    }
  }
  __device__ __forceinline__ float norm() const { return block_norm(or_nan(d)); }
  __device__ __forceinline__ float post(float nm) const { return 1.f / nm; }
};

// ---------------------------------------------------------------------- kernel
constexpr int SK_LDS = 160 * 1024;
template <int QT, bool F32, int MT, bool PACK = false>
struct SkLayout {
  using D = Sk<QT>;
  static constexpr int NP = PACK ? 1 : F32 ? 2 : 3;  // x fragments of a step and tile
  static constexpr int RW = sk_rw(MT), WV = 4 * RW, BN = sk_bn(MT);
  static constexpr bool MINS = F32 && D::MINS;
  static constexpr int FR = (8 * NP + (MINS ? 1 : 0)) * MT;        // x fragments (KiB) of a unit
  static constexpr int WG = BN * D::CH / 64;                    // weight loads (KiB) of a unit
  static constexpr int WB = WG * 1024 + (D::TAIL ? BN * 4 : 0);  // bytes
  static constexpr int XB = FR * 1024;
  static constexpr int RED = WV * SK_WR * MT * 1024;         // the K quarters' meeting
  // Units in LDS (ST), and whether the meeting has room beside them (else it takes their place)
  static constexpr int S3 = 3 * (XB + WB), S2 = 2 * (XB + WB);
  static constexpr bool APART = S2 + RED <= SK_LDS / (4 / RW);
  static constexpr int ST = (APART ? S3 + RED : S3) <= SK_LDS / (4 / RW) ? 3 : 2;
  static constexpr int RING = ST == 3 ? S3 : S2;
  static constexpr int LDS = APART ? RING + RED : RING > RED ? RING : RED;
  static constexpr bool FITS = LDS <= SK_LDS;
};

__device__ __forceinline__ void dma4(const void* p, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(p),
               "s"(__builtin_amdgcn_readfirstlane(lds_addr))
               : "memory");
}
// Waits until at most n (0 .. 6) of the wave's loads are in flight
__device__ __forceinline__ void vm_wait_n(int n) {
  switch (n) {
    case 0: vm_wait<0>(); break;
    case 1: vm_wait<1>(); break;
    case 2: vm_wait<2>(); break;
    case 3: vm_wait<3>(); break;
    case 4: vm_wait<4>(); break;
    case 5: vm_wait<5>(); break;
    default: vm_wait<6>();
  }
}

template <int QT, bool F32, int MT, bool PACK>
__global__ __launch_bounds__(256 * sk_rw(MT))
    __attribute__((amdgpu_waves_per_eu(4, 8))) void qgemm_skinny(const SkArgs p) {
  using L = SkLayout<QT, F32, MT, PACK>;
  using D = Sk<QT>;
  constexpr int NP = L::NP, WR = SK_WR, PL = F32 ? D::PLANES : 1, CH = D::CH, ST = L::ST;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rw = wave % L::RW, t = wave / L::RW & 1, kh = wave / (2 * L::RW);
  const int n = lane & 15, kg = lane >> 4;
  const int nu = (p.K + SK_UNIT - 1) / SK_UNIT, nfull = p.K / SK_UNIT;
  // Items: the workgroup tiles times the K splits, taken in turn by the workgroups
  const int nt_all = p.tile0[p.ngroups], items = nt_all * p.KS;
  struct Item {
    int grp, n0, kz, u0, u1;
  };
  auto item = [&](int i) __attribute__((always_inline)) {
    const int b = i % nt_all, kz = i / nt_all;
    const int g = p.ngroups == 1 ? 0 : __builtin_amdgcn_readfirstlane(group_of(p.tile0, p.ngroups, b));
    return Item{g, (b - p.tile0[g]) * L::BN, kz, nu * kz / p.KS, nu * (kz + 1) / p.KS};
  };
  const int rbytes = (int)((long)p.K * D::UB / SK_UNIT);  // of a row

  // The weight bytes of a unit in LDS: BN rows of CH 16-byte chunks, in 1 KiB loads g (chunks
  // 64 g + lane) that the waves take in turn; then, with TAIL, a dword a row (the last waves)
  constexpr int TW = L::WV - L::BN / 64;  // the first wave that loads tail dwords
  constexpr int NG = (L::WG + L::WV - 1) / L::WV, NX = (L::FR + L::WV - 1) / L::WV;
  // produce() loads the next unit of the workgroup's items in order; its addresses advance by units.
  Item pi = item((int)blockIdx.x);
  int pb = (int)blockIdx.x, pu = pi.u0, ahead = 0;
  uintptr_t src[NG], xsrc[NX], tsrc;
  auto start = [&]() __attribute__((always_inline)) {
    const uintptr_t W = (uintptr_t)p.W[pi.grp] + (size_t)pi.u0 * D::UB;
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int row = (64 * (wave + L::WV * i) + lane) / CH;
      src[i] = W + (size_t)(uint32_t)min(pi.n0 + row, p.N - 1) * p.rb;
    }
    tsrc = W + (size_t)(uint32_t)min(pi.n0 + max(wave - TW, 0) * 64 + lane, p.N - 1) * p.rb;
#pragma unroll
    for (int i = 0; i < NX; ++i) {  // fragment j of step/part set f, the sums after the steps
      const int fj = wave + L::WV * i, f = fj / MT;
      const size_t tile = (size_t)p.mt0[pi.grp] + fj % MT;
      xsrc[i] = (uintptr_t)(f < 8 * NP ? p.X + ((size_t)(pi.u0 * 8 * NP + f) * p.mtot + tile) * 512
                                       : p.S + ((size_t)pi.u0 * p.mtot + tile) * 512) + lane * 16;
    }
  };
  start();
  const int per_unit = (L::WG - wave + L::WV - 1) / L::WV + (D::TAIL && wave >= TW ? 1 : 0) +
                       (L::FR - wave + L::WV - 1) / L::WV;  // the wave's loads
  auto produce = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int fj = wave + L::WV * i;
      if (fj < L::FR) {
        dma16((const void*)xsrc[i], lds_addr(lds) + (uint32_t)(slot * L::FR + fj) * 1024);
        xsrc[i] += (fj < 8 * NP * MT ? 8 * NP : 1) * (size_t)p.mtot * 1024;
      }
    }
    const uint32_t base = lds_addr(lds) + ST * L::XB + (uint32_t)slot * L::WB;
    if (pu < nfull) {
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const int g = wave + L::WV * i;
        if (g < L::WG) {
          const uintptr_t f = D::TAIL ? src[i] & ~(uintptr_t)3 : src[i];
          dma16((const void*)(f + 16 * ((64 * g + lane) % CH)), base + (uint32_t)g * 1024);
          src[i] += D::UB;
        }
      }
      if (D::TAIL && wave >= TW) {
        // the dword after the chunks, where a byte of the unit lies in it (where W's last row ends in the
        // middle of a dword, the rest of that dword is read too)
        const int off = D::UB % 16 || (tsrc & 2) ? 16 * CH : 16 * CH - 4;
        dma4((const void*)((tsrc & ~(uintptr_t)3) + off), base + L::WG * 1024 + (uint32_t)(wave - TW) * 256);
        tsrc += D::UB;
      }
      ahead = per_unit;
    } else {  // the last unit of a row whose K is not a multiple of 256: by dwords, none past the row
      const uintptr_t W = (uintptr_t)p.W[pi.grp];
      for (int g = wave; g < 4 * L::WG; g += L::WV) {
        const int row = (64 * g + lane) / (4 * CH), dw = (64 * g + lane) % (4 * CH);
        const uintptr_t r = W + (size_t)(uint32_t)min(pi.n0 + row, p.N - 1) * p.rb;
        const uintptr_t a = ((r + (size_t)pu * D::UB) & ~(uintptr_t)3) + 4 * dw;
        const uintptr_t last = (r + rbytes - 1) & ~(uintptr_t)3;
        dma4((const void*)(a < last ? a : last), base + (uint32_t)g * 256);
      }
      ahead = 0;
    }
    if (++pu == pi.u1) {
      pb += (int)gridDim.x;
      if (pb < items) {
        pi = item(pb);
        pu = pi.u0;
        start();
      }
    }
  };

  // One unit after the other through the ring, on over the items where the meeting lies apart
  auto more = [&](int i) __attribute__((always_inline)) { return L::APART ? pb < items : pb == i; };
  int slot = 0;
  bool stored = false;  // stores of an item count among the loads in flight
  for (int i0 = (int)blockIdx.x; i0 < items; i0 += (int)gridDim.x) {
    const Item it = item(i0);
    const uintptr_t W = (uintptr_t)p.W[it.grp];
    const int M = p.rows[it.grp], row0 = p.row0[it.grp];
    float4v acc[WR][MT];
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
    int ph[WR];  // 2 where a row starts in the middle of a dword
#pragma unroll
    for (int i = 0; i < WR; ++i)
      ph[i] = (int)(W + (size_t)(uint32_t)min(it.n0 + (rw * WR + i) * 16 + n, p.N - 1) * p.rb) & 2;
    if (!L::APART || i0 == (int)blockIdx.x) {
      produce(0);
      if (ST == 3) {
        ahead = 0;
        if (more(i0)) produce(1);
      }
      slot = 0;
    }
    for (int u = it.u0; u < it.u1; ++u) {
      // unit u is in LDS; with three slots the last unit loaded, the next one, may still be in flight
      // (a unit by dwords is waited for at once)
      vm_wait_n(ST == 3 && !stored ? ahead : 0);
      stored = false;
      __syncthreads();  // for every wave; and the slot of the unit before is free
      const uint8_t* xs = lds + slot * L::XB + lane * 16;
      const uint8_t* ws = lds + ST * L::XB + slot * L::WB;
      const int next = slot == 0 ? ST - 1 : slot - 1;
      slot = slot + 1 == ST ? 0 : slot + 1;
      D cur[WR];
      uint32_t o[WR][8], ol[WR][8];
      float nm[WR];
#pragma unroll
      for (int i = 0; i < WR; ++i) {
        const int row = (rw * WR + i) * 16 + n;
        cur[i].read(ws + row * (16 * CH), ws + L::WG * 1024 + row * 4, (ph[i] + D::UB * u) & 2, kh, t, kg,
                    SK_UNIT * u + 128 * kh + 64 * (kg >> 1) + 32 * t < p.K);
        if constexpr (F32) nm[i] = cur[i].norm();
        cur[i].template dec<F32>(kh, t, kg, o[i], ol[i], F32 ? nm[i] : 1.f);
        if (i == 0) {
          ahead = 0;
          if (more(i0)) produce(next);
        }
      }
      float4v c[F32 ? WR : 1][MT];
      if constexpr (F32)
#pragma unroll
        for (int i = 0; i < WR; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j) c[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint8_t* xf = xs + ((4 * kh + 2 * t + s) * NP * MT) * 1024;
        half8 w[WR], wl[WR];
#pragma unroll
        for (int i = 0; i < WR; ++i) {
          w[i] = __builtin_bit_cast(half8, u32x4{o[i][4 * s], o[i][4 * s + 1], o[i][4 * s + 2], o[i][4 * s + 3]});
          if constexpr (PL == 2)
            wl[i] = __builtin_bit_cast(half8, u32x4{ol[i][4 * s], ol[i][4 * s + 1], ol[i][4 * s + 2], ol[i][4 * s + 3]});
        }
        // x-ref: lo, mid, hi (tier.cpp:940); F32: lo w, hi w_lo, hi w.  Tiles inside, so that
        // neighbouring products add to different accumulators
#pragma unroll
        for (int q = NP - 1; q >= 0; --q) {
          half8 a[MT];
#pragma unroll
          for (int j = 0; j < MT; ++j) a[j] = *(const half8*)(xf + (q * MT + j) * 1024);
          if constexpr (PL == 2)
            if (q == 0)
#pragma unroll
              for (int j = 0; j < MT; ++j)
#pragma unroll
                for (int i = 0; i < WR; ++i) c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], wl[i], c[i][j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int i = 0; i < WR; ++i) {
              float4v& d = F32 ? c[F32 ? i : 0][j] : acc[i][j];
              d = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j], w[i], d, 0, 0, 0);
            }
        }
      }
      if constexpr (F32) {
#pragma unroll
        for (int i = 0; i < WR; ++i) {
          float s = cur[i].post(nm[i]);
          if constexpr (!L::MINS) asm volatile("" : "+v"(s));  // (else the NaN select moves behind each product)
          if constexpr (L::MINS && MT == 1) {
            // one row tile: 8 fp32 products take fewer instructions than the factor's two parts, which
            // cost as much for one tile as for three (q4_K 14336x5120, us: M = 2 27.0 -> 25.9, M = 16
            // 29.6 -> 27.3)
            const uint32_t b = __float_as_uint(cur[i].factor(kh, t, kg));
            const auto bb = __builtin_amdgcn_permlane32_swap(b, b, false, false);  // sub-blocks 4 kh + t, 4 kh + 2 + t
            const float* sp = (const float*)(xs - lane * 16 + 8 * NP * 1024) + 16 * (4 * kh + t) + 4 * kg;
            const float4v s0 = *(const float4v*)sp, s1 = *(const float4v*)(sp + 32);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              acc[i][0][r] = fmaf(s0[r], __uint_as_float(bb[0]), acc[i][0][r]);
              acc[i][0][r] = fmaf(s1[r], __uint_as_float(bb[1]), acc[i][0][r]);
              acc[i][0][r] = fmaf(c[i][0][r], s, acc[i][0][r]);
            }
          } else if constexpr (L::MINS) {
            float inv;
            const half4 off = __builtin_bit_cast(half4, cur[i].offset(kh, t, kg, inv));
#pragma unroll
            for (int j = 0; j < MT; ++j) {
              const half4 a = *(const half4*)(xs - lane * 8 + (8 * NP * MT + j) * 1024 + t * 512);
              const float4v m = __builtin_amdgcn_mfma_f32_16x16x16f16(a, off, float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(c[i][j][r], s, fmaf(m[r], inv, acc[i][j][r]));
            }
          } else {
#pragma unroll
            for (int j = 0; j < MT; ++j)
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(c[i][j][r], s, acc[i][j][r]);
          }
        }
      }
    }

    // the K quarters of a row meet in LDS, in order; each quarter stores a share of the tiles
    if (!L::APART) __syncthreads();
    const int quarter = 2 * kh + t;
    float4v* red = (float4v*)(lds + (L::APART ? L::RING : 0)) + lane;
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) red[((quarter * L::RW + rw) * WR * MT + i * MT + j) * 64] = acc[i][j];
    __syncthreads();
    for (int ij = quarter; ij < WR * MT; ij += 4) {
      const int i = ij / MT, j = ij % MT, col = it.n0 + (rw * WR + i) * 16 + n;
      if (PACK && 4 * kg >= M) continue;
      auto quarters = [&](int at) __attribute__((always_inline)) {
        float4v v = red[(rw * WR * MT + ij) * 64 + at];
#pragma unroll
        for (int q = 1; q < 4; ++q) v += red[((q * L::RW + rw) * WR * MT + ij) * 64 + at];
        return v;
      };
      float4v v;
      if constexpr (!PACK) v = quarters(0);
      else if constexpr (F32) v = quarters(32) + quarters(0);  // tile row m + 8 is 32 lanes on, m + 4 16
      else v = quarters(32) + quarters(16) + quarters(0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = j * 16 + 4 * kg + r;
        if (m >= M || col >= p.N) continue;
        float y = v[r];
        if constexpr (F32) y = ldexpf(y, -p.xexp[row0 + m]);
        if (p.KS > 1) {
          p.P[(size_t)it.kz * p.ps + (size_t)m * p.N + col] = y;
        } else {
          float* o = p.Y + (size_t)(row0 + m) * p.ldy + col;
          *o = p.beta != 0.f ? fmaf(p.beta, *o, y) : y;
        }
      }
    }
    stored = true;
    if (!L::APART) __syncthreads();
  }
}

template <int QT, bool F32, int MT, bool PACK = false>
int launch_sk(const SkArgs& a, int cus, hipStream_t s, const char* who) {
  using L = SkLayout<QT, F32, MT, PACK>;
  if constexpr (L::FITS) {
    static std::atomic<uint64_t> attr{0};
    int st = lds_attr_once(attr, (const void*)qgemm_skinny<QT, F32, MT, PACK>, L::LDS, who);
    if (st) return st;
    const int grid = std::min(a.tile0[a.ngroups] * a.KS, cus * (4 / L::RW));
    qgemm_skinny<QT, F32, MT, PACK><<<(unsigned)grid, 64 * L::WV, L::LDS, s>>>(a);
    TM_LAUNCH_CHECK(who);
    return TIERMM_OK;
  }
  return set_error(TIERMM_UNSUPPORTED, "%s: %d row tiles", who, MT);
}
template <int QT, bool F32>
int launch_sk_mt(int mt, const SkArgs& a, int cus, hipStream_t s, const char* who) {
  switch (mt) {
    case 0: return launch_sk<QT, F32, 1, true>(a, cus, s, who);
    case 1: return launch_sk<QT, F32, 1>(a, cus, s, who);
    case 2: return launch_sk<QT, F32, 2>(a, cus, s, who);
    default: return launch_sk<QT, F32, 3>(a, cus, s, who);
  }
}
template <bool F32>
int launch_sk_qt(int qt, int mt, const SkArgs& a, int cus, hipStream_t s, const char* who) {
  switch (qt) {
    case QT_Q4_K: return launch_sk_mt<QT_Q4_K, F32>(mt, a, cus, s, who);
    case QT_Q5_K: return launch_sk_mt<QT_Q5_K, F32>(mt, a, cus, s, who);
    case QT_Q6_K: return launch_sk_mt<QT_Q6_K, F32>(mt, a, cus, s, who);
    case QT_Q8_0: return launch_sk_mt<QT_Q8_0, F32>(mt, a, cus, s, who);
    default: return launch_sk_mt<QT_Q5_0, F32>(mt, a, cus, s, who);
  }
}
template <int QT, bool F32>
constexpr int sk_tiles() {
  return SkLayout<QT, F32, 3>::FITS ? 3 : SkLayout<QT, F32, 2>::FITS ? 2 : 1;
}
// The row tiles that fit in LDS beside the weights
template <bool F32>
int sk_max_tiles(int qt) {
  switch (qt) {
    case QT_Q4_K: return sk_tiles<QT_Q4_K, F32>();
    case QT_Q5_K: return sk_tiles<QT_Q5_K, F32>();
    case QT_Q6_K: return sk_tiles<QT_Q6_K, F32>();
    case QT_Q8_0: return sk_tiles<QT_Q8_0, F32>();
    case QT_Q5_0: return sk_tiles<QT_Q5_0, F32>();
    default: return 0;
  }
}

bool sk_mins(int qt) { return qt == QT_Q4_K || qt == QT_Q5_K; }
size_t al256b(size_t b) { return (b + 255) & ~(size_t)255; }

// K splits of one GEMM: a workgroup for each CU, at least one unit a split
int sk_splits(int mt, int N, int K, int cus) {
  const int tiles = (N + sk_bn(mt) - 1) / sk_bn(mt), nu = (K + SK_UNIT - 1) / SK_UNIT;
  int ks = std::max(1, std::min(nu, cus * (4 / sk_rw(mt)) / tiles));
  while (K / (4 * ks) > kAccChunkFrom) ++ks;  // K per accumulator (x-ref; four K quarters each)
  ks = (nu + (nu + ks - 1) / ks - 1) / ((nu + ks - 1) / ks);  // the fewest splits with that many units each
  return ks;
}

}  // namespace

// Whether the few-row kernel takes an M-row product (or an expert of M rows) of this type: up to
// the row tiles whose fragments fit in LDS beside the weights (F32: 48 rows, q8_0 32; x-ref: 32,
// q8_0 16).  It is the faster one up to there at every shape measured, least at its largest M of
// a small weight (N = 1024, K = 4096: q4_K F32 M = 48 25.5 -> 21.9 us, x-ref M = 32 19.5 -> 18.3);
// a variant with a fourth row tile (one wave set a CU, spills) lost at M = 64, 61.6 -> 70.7 us.
bool qgemm_skinny_takes(int qt, int M, int N, int K, bool f32) {
  return M >= 1 && N >= 1 && K >= 1 && M <= 16 * (f32 ? sk_max_tiles<true>(qt) : sk_max_tiles<false>(qt));
}

// Workspace: the x fragments (and sums) of mtot 16-row tiles, the rows' exponents, the partials.
struct SkWs {
  size_t x, s, e, p, total;
};
static SkWs sk_ws(int qt, size_t mtot, size_t rows, int N, int K, bool f32, int ks) {
  const size_t nu = (K + SK_UNIT - 1) / SK_UNIT;
  SkWs w{};
  w.x = 0;
  w.s = w.x + al256b(nu * 8 * (f32 ? 2 : 3) * mtot * 1024);
  w.e = w.s + (f32 && sk_mins(qt) ? al256b(nu * mtot * 1024) : 0);
  w.p = w.e + (f32 ? al256b(rows * 4) : 0);
  w.total = w.p + (ks > 1 ? (size_t)ks * rows * N * 4 : 0);
  return w;
}

size_t qgemm_skinny_ws_bytes(int qt, int M, int N, int K, bool f32, int cus) {
  return sk_ws(qt, (size_t)(M + 15) / 16, (size_t)M, N, K, f32, sk_splits((M + 15) / 16, N, K, cus)).total;
}
// The same for n groups of rows[g] rows in one call (no K split).
size_t qgemm_skinny_group_ws_bytes(int qt, const int* rows, int n, int N, int K) {
  size_t mtot = 0, r = 0;
  for (int g = 0; g < n; ++g) {
    mtot += (size_t)(rows[g] + 15) / 16;
    r += (size_t)rows[g];
  }
  return sk_ws(qt, mtot, r, N, K, false, 1).total;
}

// An upper bound of the same over every routing of P rows to n experts.
size_t qgemm_skinny_routed_ws_bytes(size_t P, int n, int K) {
  return sk_ws(QT_Q4_K, std::min(P, (size_t)n + P / 16), P, 0, K, false, 1).total;
}

int qgemm_splitk_sum(const float* P, size_t ps, int ks, float* Y, int ldy, int rows, int N, float beta, hipStream_t s,
                     const char* who);

// n groups (rows[g] > 0 rows of x and Y from row0[g], weight W[g] of type qt).  xparts given:
// x comes split in three parts (x3-ref, one group), parts pstride apart, K-tiled over kt
// rows when kt > 0; otherwise X is split here.  split (one group): K may be split, and ws holds
// qgemm_skinny_ws_bytes; else qgemm_skinny_group_ws_bytes, which has no room for partial sums -- a
// routed batch in which one expert of a type has rows is a group of one, and must not split either
// (its rows would be summed in another order than beside other experts, too).
int qgemm_skinny(const void* const* W, int qt, const int* row0, const int* rows, int n, size_t rb, const float* X,
                 const uint16_t* xparts, size_t pstride, size_t kt, float* Y, int ldy, int N, int K, float beta,
                 bool f32, bool split, void* ws, size_t ws_bytes, int cus, hipStream_t s, const char* who) {
  const int ks = split && n == 1 ? sk_splits((rows[0] + 15) / 16, N, K, cus) : 1;
  // Parts are packed where that takes no further launch: where it leaves some groups of up to 16 rows
  // for a launch of their own, that costs more (64 experts, hidden 2048, ffn 1408, us: 16 tokens
  // 149 -> 157, 32 tokens 166 -> 176) than the packed ones gain.
  bool packed = true;
  for (int g = 0; g < n; ++g) packed = packed && (rows[g] <= sk_pack(f32) || rows[g] > 16);
  // launches of up to SK_G groups with the same number of row tiles (0: one of packed parts)
  for (int kind = 0, g0 = 0; kind <= SK_MT; g0 < n ? kind : (g0 = 0, ++kind)) {
    const bool pack = kind == 0;
    const int mt = std::max(kind, 1);
    SkArgs a{};
    a.Y = Y; a.rb = rb; a.ldy = ldy; a.N = N; a.K = K; a.KS = ks; a.beta = beta; a.flat = mt == 1;
    int total = 0, last = 0;
    for (; g0 < n && a.ngroups < SK_G; ++g0) {
      if ((packed && rows[g0] <= 16 ? 0 : (rows[g0] + 15) / 16) != kind) continue;
      const int j = a.ngroups++;
      a.row0[j] = row0[g0];
      a.rows[j] = rows[g0];
      a.W[j] = (const uint8_t*)W[g0];
      a.mt0[j] = a.mtot;
      a.mtot += mt;
      a.first[j] = total;
      total += rows[g0];
      last = row0[g0] + rows[g0];
      a.tile0[j + 1] = a.tile0[j] + (N + sk_bn(mt) - 1) / sk_bn(mt);
    }
    if (!a.ngroups) continue;
    const SkWs w = sk_ws(qt, (size_t)a.mtot, (size_t)last, N, K, f32, ks);
    if (w.total > ws_bytes)
      return set_error(TIERMM_EINVAL, "%s: few-row workspace of %zu bytes, %zu needed", who, ws_bytes, w.total);
    uint8_t* b = (uint8_t*)ws;
    uint16_t* x = (uint16_t*)(b + w.x);
    uint16_t* sums = f32 && sk_mins(qt) ? (uint16_t*)(b + w.s) : nullptr;
    int32_t* xe = (int32_t*)(b + w.e);
    a.X = x; a.S = sums; a.xexp = xe; a.P = (float*)(b + w.p); a.ps = (size_t)rows[0] * N;
    // a whole row at once, 8 elements a thread: its time is the latency of its loads (with the group
    // search skipped for one group, 256 threads -> this, a call in us: F32 q4_K 1024x4096 M = 2
    // 16.0 -> 14.0, M = 37 21.7 -> 19.8; 14336x5120 M = 2 25.7 -> 24.5, M = 37 40.4 -> 39.5)
    const int nu = (K + SK_UNIT - 1) / SK_UNIT;
    const unsigned thr = (unsigned)std::min(1024, (nu * SK_UNIT + 511) / 512 * 64);
    if (xparts) (pack ? sk_relayout3<true> : sk_relayout3<false>)<<<total, thr, 0, s>>>(xparts, pstride, kt, a, x);
    else if (f32) (pack ? sk_split2<true> : sk_split2<false>)<<<total, thr, 0, s>>>(X, a, x, sums, xe);
    else (pack ? sk_split3<true> : sk_split3<false>)<<<total, thr, 0, s>>>(X, a, x);
    TM_LAUNCH_CHECK(who);
    int st = f32 ? launch_sk_qt<true>(qt, kind, a, cus, s, who) : launch_sk_qt<false>(qt, kind, a, cus, s, who);
    if (st) return st;
    if (ks > 1) {
      st = qgemm_splitk_sum(a.P, a.ps, ks, Y + (size_t)row0[0] * ldy, ldy, rows[0], N, beta, s, who);
      if (st) return st;
    }
  }
  return TIERMM_OK;
}

}  // namespace tiermm
