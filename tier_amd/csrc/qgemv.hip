// qgemv.hip -- tiermm_qgemv: decode-time (M=1) dequant-GEMV, gemv_q (tier.cpp:299-306).
//
// Kernel per type: Q4_K, Q5_K, Q6_K and Q8_0 run on int8 MFMA (qgemv_q4k.hip,
// qgemv_q4k_ws.hip, qgemv_q6k.hip) where that measured faster; the rest of their shapes and
// the other integer-coded types on the dot kernel (qgemv_dot.hip); the other types, and
// rows that no kernel above takes, on the generic kernel.
//
// Generic kernel (every type): the block stages x in LDS once; each wave
// owns R consecutive rows and its lanes walk the row in 8-element chunks
// (lane-strided, like gemv_q's k += warpSize loop but 8 wide), decoding each
// chunk exactly as q_val and accumulating in fp32; the R row partials are then
// reduced across the wave with xor shuffles.  x is read from LDS once per chunk
// and reused for the R rows.
#include "tm_device.h"

namespace tiermm {

int check_qweight(const char* who, const void* W, int qtype, size_t rb, int cols, int dense_unit);

namespace {

constexpr int kMaxLdsK = 16384;  // x staged whole in LDS (64 KiB) up to this K; read from global above

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// XL: x staged in LDS (K <= kMaxLdsK); else read from global memory, where the
// workgroups' repeated reads of the same K floats stay in L2.
template <int QT, int R, bool XL>
__global__ __launch_bounds__(256) void qgemv_generic(const uint8_t* __restrict__ W, size_t rb,
                                                     const float* __restrict__ x, float* __restrict__ y, int N,
                                                     int K) {
  extern __shared__ float xsh[];
  const float* xs = XL ? xsh : x;
  if (XL) {
    for (int i = threadIdx.x * 4; i < K; i += 256 * 4) *(float4*)&xsh[i] = *(const float4*)&x[i];
    __syncthreads();
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row0 = (blockIdx.x * 4 + wave) * R;
  if (row0 >= N) return;
  const uint8_t* rp[R];
#pragma unroll
  for (int r = 0; r < R; ++r) rp[r] = W + (size_t)min(row0 + r, N - 1) * rb;
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.f;
  for (int c = lane * 8; c < K; c += 512) {
    const float4 xa = *(const float4*)&xs[c], xb = *(const float4*)&xs[c + 4];
    const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float v[8];
      Dec<QT>::run(rp[r], c, v);
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[r] = fmaf(v[k], xv[k], acc[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float s = wave_sum(acc[r]);
    if (lane == 0 && row0 + r < N) y[row0 + r] = s;
  }
}

template <int QT>
int launch_generic(const void* W, size_t rb, const float* x, float* y, int N, int K, hipStream_t s) {
  constexpr int R = 2;
  const unsigned grid = (unsigned)((N + 4 * R - 1) / (4 * R));
  if (K <= kMaxLdsK)
    qgemv_generic<QT, R, true><<<grid, 256, (size_t)K * 4, s>>>((const uint8_t*)W, rb, x, y, N, K);
  else
    qgemv_generic<QT, R, false><<<grid, 256, 0, s>>>((const uint8_t*)W, rb, x, y, N, K);
  TM_LAUNCH_CHECK("tiermm_qgemv: launch");
  return TIERMM_OK;
}

// ------------------------------------------------------- dense-row GEMV
// gemv<T> (tier.cpp:2261-2268) for fp32 / fp16 (tier_fp16) / bf16 rows: y[r] =
// sum_k float(W[r][k]) * x[k], fp32 accumulation.  x is staged in LDS; a wave
// owns R rows and its lanes read 16 bytes of each row per step (VEC elements),
// so every load instruction covers 1 KiB of a row; rows whose length is not a
// whole number of 16-byte chunks take the element-wise path.
template <int T>
struct Dense;
template <>
struct Dense<TIERMM_F32> {
  static constexpr int VEC = 4, BYTES = 4;
  __device__ static void load(const uint8_t* p, float (&v)[8]) {
    const float4 a = *(const float4*)p;
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  }
  __device__ static float at(const uint8_t* row, int k) { return ((const float*)row)[k]; }
};
template <>
struct Dense<TIERMM_F16> {
  static constexpr int VEC = 8, BYTES = 2;
  __device__ static void load(const uint8_t* p, float (&v)[8]) {
    const uint4 a = *(const uint4*)p;
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = h2f(w[i] & 0xffffu);
      v[2 * i + 1] = h2f(w[i] >> 16);
    }
  }
  __device__ static float at(const uint8_t* row, int k) { return h2f(((const uint16_t*)row)[k]); }
};
template <>
struct Dense<TIERMM_BF16> {
  static constexpr int VEC = 8, BYTES = 2;
  __device__ static void load(const uint8_t* p, float (&v)[8]) {
    const uint4 a = *(const uint4*)p;
    const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
  __device__ static float at(const uint8_t* row, int k) {
    return __uint_as_float((uint32_t)((const uint16_t*)row)[k] << 16);
  }
};

template <int T, int R, bool XL>
__global__ __launch_bounds__(256) void gemv_dense(const uint8_t* __restrict__ W, const float* __restrict__ x,
                                                  float* __restrict__ y, int N, int K) {
  using D = Dense<T>;
  extern __shared__ float xsh[];  // x staged in LDS when XL (K <= kMaxLdsK), else read from global
  const float* xs = XL ? xsh : x;
  if (XL) {
    for (int i = threadIdx.x; i < K; i += 256) xsh[i] = x[i];
    __syncthreads();
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row0 = (blockIdx.x * 4 + wave) * R;
  if (row0 >= N) return;
  const size_t rbytes = (size_t)K * D::BYTES;
  const uint8_t* rp[R];
#pragma unroll
  for (int r = 0; r < R; ++r) rp[r] = W + (size_t)min(row0 + r, N - 1) * rbytes;
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.f;
  if ((rbytes & 15) == 0) {
    for (int k = lane * D::VEC; k < K; k += 64 * D::VEC) {
      float v[R][8];
#pragma unroll
      for (int r = 0; r < R; ++r) D::load(rp[r] + (size_t)k * D::BYTES, v[r]);
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < D::VEC; ++e) acc[r] = fmaf(v[r][e], xs[k + e], acc[r]);
    }
  } else {
    for (int k = lane; k < K; k += 64)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] = fmaf(D::at(rp[r], k), xs[k], acc[r]);
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float t = wave_sum(acc[r]);
    if (lane == 0 && row0 + r < N) y[row0 + r] = t;
  }
}

template <int T>
int launch_dense(const void* W, const float* x, float* y, int N, int K, hipStream_t s) {
  constexpr int R = 4;
  const unsigned grid = (unsigned)((N + 4 * R - 1) / (4 * R));
  if (K <= kMaxLdsK)
    gemv_dense<T, R, true><<<grid, 256, (size_t)K * 4, s>>>((const uint8_t*)W, x, y, N, K);
  else
    gemv_dense<T, R, false><<<grid, 256, 0, s>>>((const uint8_t*)W, x, y, N, K);
  TM_LAUNCH_CHECK("tiermm_gemv: launch");
  return TIERMM_OK;
}

}  // namespace

int qgemv_q4k(const void* W, size_t rb, const float* x, float* y, int N, int K, hipStream_t s);
int qgemv_q4k_ws(const void* W, size_t rb, const float* x, float* y, int N, int K, hipStream_t s);
int qgemv_q5k_ws(const void* W, size_t rb, const float* x, float* y, int N, int K, hipStream_t s);
bool qgemv_ws_takes(int qtype, int N, int K);
bool qgemv_ws_batch_takes(int qtype, const int* N, int count, int K);
int qgemv_ws_batch(const void* const* W, int qtype, size_t rb, const float* x, float* const* y, const int* N,
                   int count, int K, hipStream_t s);
bool qgemv_mfma_fits(const void* W, int qtype, size_t rb, int K);
bool qgemv_q6k_fits(const void* W, size_t rb, int N, int K);
int qgemv_q6k(const void* W, size_t rb, const float* x, float* y, int N, int K, hipStream_t s);
int qgemv_mfma(const void* W, int qtype, size_t rb, const float* x, float* y, int N, int K, hipStream_t s);
bool qgemv_dot_takes(const void* W, int qtype, int K);
int qgemv_dot(const void* W, int qtype, size_t rb, const float* x, float* y, int N, int K, hipStream_t s);
constexpr int kQ4kMaxK = 28672;  // equals the limit in qgemv_q4k.hip

int qgemv_dispatch(const void* W, int qtype, size_t rb, const float* x, float* y, int N, int K, hipStream_t s) {
  const int tiles = (N + 15) / 16;
  switch (qtype) {
    // dense rows (gemv_q over q_val's F32/F16/BF16 cases): the dense-row kernel
    case QT_F32: return launch_dense<TIERMM_F32>(W, x, y, N, K, s);
    case QT_F16: return launch_dense<TIERMM_F16>(W, x, y, N, K, s);
    case QT_BF16: return launch_dense<TIERMM_BF16>(W, x, y, N, K, s);
    case QT_Q4_K:  // below 64 row tiles the dot kernel: 301x8192 8.6 -> 4.6 us, 640x5120 5.25 -> 4.6
      if (qgemv_ws_takes(QT_Q4_K, N, K)) return qgemv_q4k_ws(W, rb, x, y, N, K, s);
      if (tiles >= 64 && K <= kQ4kMaxK) return qgemv_q4k(W, rb, x, y, N, K, s);
      break;
    case QT_Q5_K:  // the same above K = 5120 (301x8192 9.6 -> 6.6 us; 640x5120 5.7 against 6.5)
      if (qgemv_mfma_fits(W, qtype, rb, K) && (tiles >= 64 || K <= 5120))
        return qgemv_ws_takes(QT_Q5_K, N, K) ? qgemv_q5k_ws(W, rb, x, y, N, K, s) : qgemv_mfma(W, qtype, rb, x, y, N, K, s);
      break;
    case QT_Q8_0:
      // MFMA where it measured faster: 129-512 row tiles up to K = 5120 (4096x5120 6.7 against
      // 8.3 us, 8192x5120 11.0 against 11.4; 1024x5120 5.3 against 4.8, 20000x5120 29.2 against
      // 22.3), 129-256 above 8192 (4096x14336 14.2 against 15.1; 5120x14336 20.4 against 18.2); not
      // between (2500x8192 11.8 against 7.9)
      if (qgemv_mfma_fits(W, qtype, rb, K) && tiles > 128 && (K <= 5120 ? tiles <= 512 : K > 8192 && tiles <= 256))
        return qgemv_mfma(W, qtype, rb, x, y, N, K, s);
      break;
    case QT_Q6_K:  // MFMA above 160 row tiles (4096x5120 7.9 against 9.8 us; 2500x4096 7.1 against 6.7)
      if (tiles > 160 && qgemv_q6k_fits(W, rb, N, K)) return qgemv_q6k(W, rb, x, y, N, K, s);
      break;
    default: break;
  }
  if (qgemv_dot_takes(W, qtype, K)) return qgemv_dot(W, qtype, rb, x, y, N, K, s);
  return with_qtype(qtype, [&](auto qt) { return launch_generic<decltype(qt)::value>(W, rb, x, y, N, K, s); });
}

}  // namespace tiermm

using namespace tiermm;

extern "C" int tiermm_qgemv(const void* W, int qtype, size_t rb, const float* x, float* y, int N, int K,
                            tiermm_stream_t stream) {
  int st = check_qweight("tiermm_qgemv", W, qtype, rb, K, 1);
  if (st) return st;
  if (N < 0) return set_error(TIERMM_EINVAL, "tiermm_qgemv: N < 0");
  if (N == 0) return TIERMM_OK;
  if (!x || !y || ((uintptr_t)x % 16)) return set_error(TIERMM_EINVAL, "tiermm_qgemv: x must be 16-byte aligned");
  if ((qtype == QT_F32 || qtype == QT_F16 || qtype == QT_BF16) && ((uintptr_t)W % 16))
    return set_error(TIERMM_EINVAL, "tiermm_qgemv: dense rows must start 16-byte aligned");
  return qgemv_dispatch(W, qtype, rb, x, y, N, K, (hipStream_t)stream);
}

// gemv_q of up to TIERMM_QGEMV_BATCH matrices that share x, K and the block type.  Where
// the whole-tile kernel takes their concatenated rows (q4_K / q5_K, K <= 5120, its tile
// rule on the total) they run as one launch; otherwise one tiermm_qgemv each.  Either
// way every y[i] is the same, bit for bit, as tiermm_qgemv on W[i].
extern "C" int tiermm_qgemv_batch(const void* const* W, int qtype, size_t rb, const float* x, float* const* y,
                                  const int* N, int count, int K, tiermm_stream_t stream) {
  if (!W || !y || !N || count < 1 || count > TIERMM_QGEMV_BATCH)
    return set_error(TIERMM_EINVAL, "tiermm_qgemv_batch: 1..%d matrices with weight, output and row arrays",
                     TIERMM_QGEMV_BATCH);
  const void* w[TIERMM_QGEMV_BATCH];
  float* yy[TIERMM_QGEMV_BATCH];
  int n[TIERMM_QGEMV_BATCH], live = 0;
  for (int i = 0; i < count; ++i) {
    if (N[i] < 0) return set_error(TIERMM_EINVAL, "tiermm_qgemv_batch: N[%d] < 0", i);
    if (N[i] > 0) {  // matrices without rows take no part (their pointers are not read)
      int st = check_qweight("tiermm_qgemv_batch", W[i], qtype, rb, K, 1);
      if (st) return st;
      if (!y[i]) return set_error(TIERMM_EINVAL, "tiermm_qgemv_batch: y[%d] is null", i);
      w[live] = W[i];
      yy[live] = y[i];
      n[live++] = N[i];
    }
  }
  if (!live) return TIERMM_OK;
  if (!x || ((uintptr_t)x % 16)) return set_error(TIERMM_EINVAL, "tiermm_qgemv_batch: x must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  bool fits = qgemv_ws_batch_takes(qtype, n, live, K);
  for (int i = 0; fits && i < live && qtype == QT_Q5_K; ++i) fits = qgemv_mfma_fits(w[i], qtype, rb, K);
  if (fits) return qgemv_ws_batch(w, qtype, rb, x, yy, n, live, K, s);
  for (int i = 0; i < live; ++i) {
    if ((qtype == QT_F32 || qtype == QT_F16 || qtype == QT_BF16) && ((uintptr_t)w[i] % 16))
      return set_error(TIERMM_EINVAL, "tiermm_qgemv_batch: dense rows must start 16-byte aligned");
    int st = qgemv_dispatch(w[i], qtype, rb, x, yy[i], n[i], K, s);
    if (st) return st;
  }
  return TIERMM_OK;
}

extern "C" int tiermm_gemv(const void* W, int wtype, const float* x, float* y, int N, int K, tiermm_stream_t stream) {
  if (wtype != TIERMM_F32 && wtype != TIERMM_F16 && wtype != TIERMM_BF16)
    return set_error(TIERMM_UNSUPPORTED, "tiermm_gemv: weight type %d", wtype);
  if (N < 0 || K < 0) return set_error(TIERMM_EINVAL, "tiermm_gemv: negative size");
  if (N == 0) return TIERMM_OK;
  if (!W || !x || !y || ((uintptr_t)W % 16))
    return set_error(TIERMM_EINVAL, "tiermm_gemv: W must be non-null and 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  if (wtype == TIERMM_F32) return launch_dense<TIERMM_F32>(W, x, y, N, K, s);
  if (wtype == TIERMM_F16) return launch_dense<TIERMM_F16>(W, x, y, N, K, s);
  return launch_dense<TIERMM_BF16>(W, x, y, N, K, s);
}
