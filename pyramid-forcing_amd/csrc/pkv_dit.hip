// Row operations of the causal DiT block that drives the pyramid cache in the
// end-to-end rollout (wan/modules/causal_model.py:395-420 of the reference):
// LayerNorm with modulation or affine weights, RMSNorm of q and k
// (wan/modules/model.py:70-99), the gated residual updates of the fp32
// residual stream, and the tanh GELU of the feed-forward.  Each is one
// launch instead of the chain of elementwise and reduction kernels that
// eager PyTorch runs for it.
//
// The row kernels give one wave to a row: lane i holds the 16-byte vectors
// i, i + 64, ... of the row in registers (up to kMaxVec of them), the sums
// are wave reductions, and the row is read from memory once.  LayerNorm
// takes the mean first and then the sum of squared deviations (two-pass in
// registers), so a large mean does not cancel the variance.

#include "pkv_common.h"

namespace pkv {

constexpr int kDitRowsPerBlock = 4;  // one wave per row
constexpr int kMaxVec = 16;          // 16-byte vectors per lane: rows up to 4096 fp32 / 8192 bf16

__device__ inline float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

__device__ inline float4 ld_f4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

// 16 bytes at any 4-byte boundary (gfx950 loads need no more)
__device__ inline float4 ld_f4u(const float *p) {
  typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
  const f4u v = *reinterpret_cast<const f4u *>(p);
  return make_float4(v[0], v[1], v[2], v[3]);
}

// a + float(b) * gate[4j..4j+3] with one rounding per element (fma), or
// a + float(b) without a gate: the residual update of 4 columns, shared by
// the residual kernel and the fused residual + LayerNorm so both round alike
__device__ inline float4 residual4(float4 a, uint2 b, const float *gate, int j) {
  const float y0 = bf16_to_f32(static_cast<uint16_t>(b.x & 0xffff)), y1 = bf16_to_f32(static_cast<uint16_t>(b.x >> 16));
  const float y2 = bf16_to_f32(static_cast<uint16_t>(b.y & 0xffff)), y3 = bf16_to_f32(static_cast<uint16_t>(b.y >> 16));
  if (gate) {
    const float4 g = ld_f4(gate + 4 * j);
    return make_float4(__fmaf_rn(y0, g.x, a.x), __fmaf_rn(y1, g.y, a.y), __fmaf_rn(y2, g.z, a.z),
                       __fmaf_rn(y3, g.w, a.w));
  }
  return make_float4(__fadd_rn(a.x, y0), __fadd_rn(a.y, y1), __fadd_rn(a.z, y2), __fadd_rn(a.w, y3));
}

// out[r, :] = bf16(LN(x[r, :]) * m + a), LN without affine weights; m =
// (one_plus ? 1 + mul : mul) and a = add, each optional (1 and 0).  kRes
// first applies the residual update x[r, :] += float(y[r, :]) * gate in
// registers and writes the updated row back, so the row is read once.  K
// vectors of 4 values per lane, the first kSure of them in the row on every
// lane, the others guarded (ln_instance).  Bound by memory, and, since a launch
// of a few thousand rows has all of its waves resident at once, by the chain of
// reads and sums of one row: K fits the row (6 vectors at 1,536 columns), the
// row's y is read with it, and the weights are read between the two sums.
// 4,680 rows of 1,536: 15.0 us with the residual update (86 MB, 5.7 TB/s) and
// 8.8 us without, against 17.5 and 10.0 with 8 guarded vectors and the weights
// read last; of 1,280: 12.2 and 7.4, against 16.5 and 9.2 with 6 guarded ones.
template <int K, bool kRes, int kSure>
__global__ void __launch_bounds__(64 * kDitRowsPerBlock) ln_mod_kernel(float *x, int64_t rows, int C,
                                                                       const float *mul, const float *add,
                                                                       int one_plus, float eps, uint16_t *out,
                                                                       const uint16_t *y, int64_t y_stride,
                                                                       const float *gate) {
  const int lane = threadIdx.x & 63;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kDitRowsPerBlock + (threadIdx.x >> 6);
  if (r >= rows) return;
  float *xr = x + r * C;
  const int nv = C / 4;
  float4 v[K];
  uint2 yv[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int j = lane + 64 * k;
    const bool in = k < kSure || j < nv;
    v[k] = in ? ld_f4(xr + 4 * j) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (kRes && in) yv[k] = *reinterpret_cast<const uint2 *>(y + r * y_stride + 4 * j);
  }
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int j = lane + 64 * k;
    if (kRes && (k < kSure || j < nv)) {
      v[k] = residual4(v[k], yv[k], gate, j);
      *reinterpret_cast<float4 *>(xr + 4 * j) = v[k];
    }
    s += (v[k].x + v[k].y) + (v[k].z + v[k].w);
  }
  const float mean = wave_sum(s) / static_cast<float>(C);
  // the weights are on their way while the second sum is taken (rows of more
  // vectors have no registers left for them)
  constexpr bool kEarly = K <= 6;
  float4 mv[kEarly ? K : 1], av[kEarly ? K : 1];
  if constexpr (kEarly) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int j = k < kSure ? lane + 64 * k : min(lane + 64 * k, nv - 1);
      if (mul) mv[k] = ld_f4(mul + 4 * j);
      if (add) av[k] = ld_f4(add + 4 * j);
    }
  }
  float q = 0.0f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int j = lane + 64 * k;
    if (k < kSure || j < nv) {
      const float a = v[k].x - mean, b = v[k].y - mean, c = v[k].z - mean, d = v[k].w - mean;
      q += (a * a + b * b) + (c * c + d * d);
    }
  }
  const float rstd = rsqrtf(wave_sum(q) / static_cast<float>(C) + eps);
  uint16_t *orow = out + r * C;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int j = lane + 64 * k;
    if (k >= kSure && j >= nv) continue;
    float y[4] = {(v[k].x - mean) * rstd, (v[k].y - mean) * rstd, (v[k].z - mean) * rstd, (v[k].w - mean) * rstd};
    if (mul) {
      const float4 m = kEarly ? mv[kEarly ? k : 0] : ld_f4(mul + 4 * j);
      const float mm[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] *= one_plus ? 1.0f + mm[e] : mm[e];
    }
    if (add) {
      const float4 a = kEarly ? av[kEarly ? k : 0] : ld_f4(add + 4 * j);
      y[0] += a.x;
      y[1] += a.y;
      y[2] += a.z;
      y[3] += a.w;
    }
    *reinterpret_cast<uint2 *>(orow + 4 * j) = make_uint2(cvt_bf16x2(y[0], y[1]), cvt_bf16x2(y[2], y[3]));
  }
}

// out[r, :] = bf16(x * rsqrt(mean(x^2) + eps) * w) in fp32, x bf16.  K
// vectors of 8 values per lane, the last one guarded unless kFull (the row is
// exactly K * 64 vectors long).  Bound by latency more than by memory: at
// 4,680 rows of 1,536 every wave of the launch is resident at once, so its time
// is one chain of read, wave sum, store.  The weights are therefore read with
// the row, not after its sum, and K fits the row: 6.9 us (4.2 TB/s) for 4,680
// rows of 1,536 out of rows of 4,608, 8.4 us with 4 guarded vectors and the
// weights read last.
template <int K, bool kFull>
__global__ void __launch_bounds__(64 * kDitRowsPerBlock) rms_kernel(const uint16_t *x, int64_t x_stride, int64_t rows,
                                                                    int C, const float *w, float eps,
                                                                    uint16_t *out, int64_t out_stride) {
  const int lane = threadIdx.x & 63;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kDitRowsPerBlock + (threadIdx.x >> 6);
  if (r >= rows) return;
  const uint16_t *xr = x + r * x_stride;
  const int nv = C / 8;
  uint4 v[K];
  constexpr bool kEarly = K <= 4;  // (longer rows have no registers left for the weights)
  float4 g[kEarly ? K : 1][2];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int j = lane + 64 * k;
    v[k] = kFull || j < nv ? *reinterpret_cast<const uint4 *>(xr + 8 * j) : make_uint4(0, 0, 0, 0);
  }
  auto weights = [&](int j, float4 (&to)[2]) {
    to[0] = to[1] = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    if (w && (kFull || j < nv)) {
      to[0] = ld_f4u(w + 8 * j);
      to[1] = ld_f4u(w + 8 * j + 4);
    }
  };
  if constexpr (kEarly) {
#pragma unroll
    for (int k = 0; k < K; ++k) weights(lane + 64 * k, g[k]);
  }
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t wd[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = bf16_to_f32(static_cast<uint16_t>(wd[e] & 0xffff));
      const float b = bf16_to_f32(static_cast<uint16_t>(wd[e] >> 16));
      s += a * a + b * b;
    }
  }
  const float rn = rsqrtf(wave_sum(s) / static_cast<float>(C) + eps);
  uint16_t *orow = out + r * out_stride;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int j = lane + 64 * k;
    if (!kFull && j >= nv) continue;
    const uint32_t wd[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
    float4 (&gk)[2] = g[kEarly ? k : 0];
    if constexpr (!kEarly) weights(j, gk);
    const float gg[8] = {gk[0].x, gk[0].y, gk[0].z, gk[0].w, gk[1].x, gk[1].y, gk[1].z, gk[1].w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float a = bf16_to_f32(static_cast<uint16_t>(wd[e] & 0xffff)) * rn;
      float b = bf16_to_f32(static_cast<uint16_t>(wd[e] >> 16)) * rn;
      if (w) {
        a *= gg[2 * e];
        b *= gg[2 * e + 1];
      }
      o[e] = cvt_bf16x2(a, b);
    }
    *reinterpret_cast<uint4 *>(orow + 8 * j) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// x[r, c] += float(y[r, c]) * gate[c] (gate optional: 1), 4 columns per thread
__global__ void __launch_bounds__(256) residual_kernel(float *x, int64_t rows, int C, const uint16_t *y,
                                                       int64_t y_stride, const float *gate) {
  const int nv = C / 4;
  const int64_t total = rows * nv;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t r = i / nv;
    const int j = static_cast<int>(i % nv);
    const float4 a = ld_f4(x + r * C + 4 * j);
    const uint2 b = *reinterpret_cast<const uint2 *>(y + r * y_stride + 4 * j);
    *reinterpret_cast<float4 *>(x + r * C + 4 * j) = residual4(a, b, gate, j);
  }
}

// out = bf16(0.5 x (1 + tanh(u))), u = sqrt(2 / pi) (x + 0.044715 x^3), in fp32, 8 values per thread.
// 0.5 (1 + tanh(u)) = 1 / (1 + e^(-2u)), so the value is x / (1 + 2^(t)) with
// t = -2 log2(e) u: one v_exp_f32 and one v_rcp_f32 (each within about 1 ulp
// of fp32, far below the bf16 rounding of the result) instead of a library
// tanh.  Large |u| give x (t -> -inf) or a signed zero (t -> +inf).
__device__ inline float gelu_tanh_f32(float x) {
  constexpr float kC1 = -2.0f * 1.4426950408889634f * 0.7978845608028654f;  // -2 log2(e) sqrt(2/pi)
  constexpr float kC3 = kC1 * 0.044715f;
  const float t = x * fmaf(kC3, x * x, kC1);
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
}

__global__ void __launch_bounds__(256) gelu_tanh_kernel(const uint16_t *x, int64_t n8, uint16_t *out) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n8;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const uint4 v = *reinterpret_cast<const uint4 *>(x + 8 * i);
    const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float f[2] = {bf16_to_f32(static_cast<uint16_t>(wd[e] & 0xffff)), bf16_to_f32(static_cast<uint16_t>(wd[e] >> 16))};
      o[e] = cvt_bf16x2(gelu_tanh_f32(f[0]), gelu_tanh_f32(f[1]));
    }
    *reinterpret_cast<uint4 *>(out + 8 * i) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

static int row_grid(int64_t rows);

// LayerNorm rows (kRes: after the residual update from y and gate)
// the instance for rows of `vec` vectors per lane (ln_mod_kernel), full: the
// last one too.  Up to 8 it is exact; beyond, registers decide more than guards
// do, and with the residual 12 vectors all guarded are the fastest (3,072
// columns 30.5 us, 37.3 with the first 8 unguarded; without it 19.8 and 19.7).
template <bool kRes>
static auto *ln_instance(int vec, bool full) {
  switch (vec) {
    case 1: return full ? ln_mod_kernel<1, kRes, 1> : ln_mod_kernel<1, kRes, 0>;
    case 2: return full ? ln_mod_kernel<2, kRes, 2> : ln_mod_kernel<2, kRes, 1>;
    case 3: return full ? ln_mod_kernel<3, kRes, 3> : ln_mod_kernel<3, kRes, 2>;
    case 4: return full ? ln_mod_kernel<4, kRes, 4> : ln_mod_kernel<4, kRes, 3>;
    case 5: return full ? ln_mod_kernel<5, kRes, 5> : ln_mod_kernel<5, kRes, 4>;
    case 6: return full ? ln_mod_kernel<6, kRes, 6> : ln_mod_kernel<6, kRes, 5>;
    case 7: return full ? ln_mod_kernel<7, kRes, 7> : ln_mod_kernel<7, kRes, 6>;
    case 8: return full ? ln_mod_kernel<8, kRes, 8> : ln_mod_kernel<8, kRes, 7>;
    default: return vec <= 12 ? ln_mod_kernel<12, kRes, kRes ? 0 : 8> : ln_mod_kernel<kMaxVec, kRes, 12>;
  }
}

template <bool kRes>
static int launch_ln_k(float *x, int64_t rows, int cols, const float *mul, const float *add, int mul_plus_one,
                       float eps, uint16_t *out, const uint16_t *y, int64_t y_stride, const float *gate, hipStream_t st,
                       const char *who) {
  const int vec = (cols / 4 + 63) / 64;
  if (vec > kMaxVec) return fail(PKV_ERR_UNSUPPORTED, "%s: cols (%d) above %d", who, cols, 64 * 4 * kMaxVec);
  auto *k = ln_instance<kRes>(vec, cols % 256 == 0);
  hipLaunchKernelGGL(k, dim3(row_grid(rows)), dim3(64 * kDitRowsPerBlock), 0, st, x, rows, cols, mul, add, mul_plus_one,
                     eps, out, y, y_stride, gate);
  return check_launch("ln_mod_kernel");
}

static int launch_ln(float *x, int64_t rows, int cols, const float *mul, const float *add, int mul_plus_one, float eps,
                     uint16_t *out, const uint16_t *y, int64_t y_stride, const float *gate, hipStream_t st,
                     const char *who) {
  return y ? launch_ln_k<true>(x, rows, cols, mul, add, mul_plus_one, eps, out, y, y_stride, gate, st, who)
           : launch_ln_k<false>(x, rows, cols, mul, add, mul_plus_one, eps, out, y, y_stride, gate, st, who);
}

static int row_grid(int64_t rows) {
  const int64_t g = (rows + kDitRowsPerBlock - 1) / kDitRowsPerBlock;
  return static_cast<int>(g);
}

static int flat_grid(int64_t items) {
  int64_t g = (items + 255) / 256;
  if (g > 65536) g = 65536;
  return static_cast<int>(g < 1 ? 1 : g);
}

}  // namespace pkv

using namespace pkv;

extern "C" int pkv_dit_layer_norm(const float *x, int64_t rows, int32_t cols, const float *mul, const float *add,
                                  int32_t mul_plus_one, float eps, uint16_t *out, pkv_stream_t stream) {
  if (rows == 0) return PKV_OK;
  if (!x || !out || rows < 0 || cols <= 0) return fail(PKV_ERR_INVALID, "dit_layer_norm: bad arguments");
  if (cols % 4) return fail(PKV_ERR_INVALID, "dit_layer_norm: cols (%d) must be a multiple of 4", cols);
  if (rows > 0x7fffffffLL * kDitRowsPerBlock) return fail(PKV_ERR_UNSUPPORTED, "dit_layer_norm: too many rows");
  return launch_ln(const_cast<float *>(x), rows, cols, mul, add, mul_plus_one, eps, out, nullptr, 0, nullptr,
                   as_stream(stream), "dit_layer_norm");
}

extern "C" int pkv_dit_residual_layer_norm(float *x, int64_t rows, int32_t cols, const uint16_t *y,
                                           int64_t y_row_stride, const float *gate, const float *mul,
                                           const float *add, int32_t mul_plus_one, float eps, uint16_t *out,
                                           pkv_stream_t stream) {
  if (rows == 0) return PKV_OK;
  if (!x || !y || !out || rows < 0 || cols <= 0) return fail(PKV_ERR_INVALID, "dit_residual_layer_norm: bad arguments");
  if (cols % 4 || y_row_stride % 4 || y_row_stride < cols)
    return fail(PKV_ERR_INVALID, "dit_residual_layer_norm: cols and the row stride must be multiples of 4 (cols %d)",
                cols);
  if (rows > 0x7fffffffLL * kDitRowsPerBlock)
    return fail(PKV_ERR_UNSUPPORTED, "dit_residual_layer_norm: too many rows");
  return launch_ln(x, rows, cols, mul, add, mul_plus_one, eps, out, y, y_row_stride, gate, as_stream(stream),
                   "dit_residual_layer_norm");
}

extern "C" int pkv_dit_rms_norm(const uint16_t *x, int64_t x_row_stride, int64_t rows, int32_t cols, const float *weight,
                                float eps, uint16_t *out, int64_t out_row_stride, pkv_stream_t stream) {
  if (rows == 0) return PKV_OK;
  if (!x || !out || rows < 0 || cols <= 0) return fail(PKV_ERR_INVALID, "dit_rms_norm: bad arguments");
  if (cols % 8 || x_row_stride % 8 || out_row_stride % 8 || x_row_stride < cols || out_row_stride < cols)
    return fail(PKV_ERR_INVALID, "dit_rms_norm: cols and row strides must be multiples of 8 (cols %d)", cols);
  if (rows > 0x7fffffffLL * kDitRowsPerBlock) return fail(PKV_ERR_UNSUPPORTED, "dit_rms_norm: too many rows");
  const int vec = (cols / 8 + 63) / 64;
  if (vec > kMaxVec) return fail(PKV_ERR_UNSUPPORTED, "dit_rms_norm: cols (%d) above %d", cols, 64 * 8 * kMaxVec);
  const bool full = cols % 512 == 0;
  auto *k = vec == 1   ? (full ? rms_kernel<1, true> : rms_kernel<1, false>)
            : vec == 2 ? (full ? rms_kernel<2, true> : rms_kernel<2, false>)
            : vec == 3 ? (full ? rms_kernel<3, true> : rms_kernel<3, false>)
            : vec == 4 ? (full ? rms_kernel<4, true> : rms_kernel<4, false>)
            : vec <= 8 ? rms_kernel<8, false>
                       : rms_kernel<kMaxVec, false>;
  hipLaunchKernelGGL(k, dim3(row_grid(rows)), dim3(64 * kDitRowsPerBlock), 0, as_stream(stream), x, x_row_stride, rows,
                     cols, weight, eps, out, out_row_stride);
  return check_launch("rms_kernel");
}

extern "C" int pkv_dit_residual(float *x, int64_t rows, int32_t cols, const uint16_t *y, int64_t y_row_stride,
                                const float *gate, pkv_stream_t stream) {
  if (rows == 0) return PKV_OK;
  if (!x || !y || rows < 0 || cols <= 0) return fail(PKV_ERR_INVALID, "dit_residual: bad arguments");
  if (cols % 4 || y_row_stride % 4 || y_row_stride < cols)
    return fail(PKV_ERR_INVALID, "dit_residual: cols and the row stride must be multiples of 4 (cols %d)", cols);
  hipLaunchKernelGGL(residual_kernel, dim3(flat_grid(rows * (cols / 4))), dim3(256), 0, as_stream(stream), x, rows,
                     cols, y, y_row_stride, gate);
  return check_launch("residual_kernel");
}

extern "C" int pkv_dit_gelu_tanh(const uint16_t *x, int64_t n, uint16_t *out, pkv_stream_t stream) {
  if (n == 0) return PKV_OK;
  if (!x || !out || n < 0) return fail(PKV_ERR_INVALID, "dit_gelu_tanh: bad arguments");
  if (n % 8) return fail(PKV_ERR_INVALID, "dit_gelu_tanh: n (%lld) must be a multiple of 8", static_cast<long long>(n));
  hipLaunchKernelGGL(gelu_tanh_kernel, dim3(flat_grid(n / 8)), dim3(256), 0, as_stream(stream), x, n / 8, out);
  return check_launch("gelu_tanh_kernel");
}
