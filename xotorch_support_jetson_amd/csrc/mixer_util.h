// Small device and host helpers shared by the mixed-layer kernel files (mixers.hip, hybrid.hip).
#pragma once
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include "common.h"

namespace xot {
namespace mix {

constexpr int PAGE_TOK = 64;

__device__ __forceinline__ float ldf(const float* p) { return *p; }
__device__ __forceinline__ float ldf(const uint16_t* p) { return bf2f(*p); }
__device__ __forceinline__ void stf(float* p, float v) { *p = v; }
__device__ __forceinline__ void stf(uint16_t* p, float v) { *p = f2bf(v); }

__device__ __forceinline__ float sigmoidf_(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float siluf_(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float gelu_tanhf_(float x) { return 0.5f * x * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * x * x * x))); }
__device__ __forceinline__ float softplusf_(float x) { return log1pf(expf(-fabsf(x))) + fmaxf(x, 0.0f); }
__device__ __forceinline__ float logsigmoidf_(float x) { return fminf(x, 0.0f) - log1pf(expf(-fabsf(x))); }

// a score s scaled by log2 e -> cap tanh(s / cap) scaled likewise (inv_cap2 = 2 / cap, cap_l2 = cap log2 e), with the base-2
// exponential and the reciprocal of the hardware: tanh(x) = 1 - 2 / (e^2x + 1)
__device__ __forceinline__ float capped_l2(float s_l2, float inv_cap2, float cap_l2) {
  return cap_l2 - 2.0f * cap_l2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(s_l2 * inv_cap2) + 1.0f);
}

// sum over the workgroup; red: at least (threads / 64) floats of LDS
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float t = 0.0f;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}

// sequence of token t: the b with cu[b] <= t < cu[b + 1]
__device__ __forceinline__ int seq_of(const int* cu, int B, int t) {
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ void ld8(const float* p, float* o) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
  o[0] = a[0]; o[1] = a[1]; o[2] = a[2]; o[3] = a[3]; o[4] = b[0]; o[5] = b[1]; o[6] = b[2]; o[7] = b[3];
}
__device__ __forceinline__ void ld8(const uint16_t* p, float* o) {
  const s16x8 a = ld16(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = bf2f(a[i]);
}

__device__ __forceinline__ void st2(float* p, float a, float b) {
  typedef float f32x2_s __attribute__((ext_vector_type(2)));
  *reinterpret_cast<f32x2_s*>(p) = f32x2_s{a, b};
}
__device__ __forceinline__ void st2(uint16_t* p, float a, float b) {
  *reinterpret_cast<uint32_t*>(p) = (uint32_t)f2bf(a) | (uint32_t)f2bf(b) << 16;
}
__device__ __forceinline__ void st4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void st4(uint16_t* p, f32x4 v) {
  *reinterpret_cast<s16x4*>(p) = s16x4{(short)f2bf(v[0]), (short)f2bf(v[1]), (short)f2bf(v[2]), (short)f2bf(v[3])};
}

// element / four elements of a GEMM result that may still be S split-K slabs, ss floats apart (S = 1: a plain result)
__device__ __forceinline__ float slab1(const float* p, int S, int64_t ss) {
  float v = p[0];
  for (int s0 = 1; s0 < S; s0 += 4) {  // (four loads in flight, without branches: slabs past the last repeat it, unused)
    float a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = p[min(s0 + i, S - 1) * ss];
#pragma unroll
    for (int i = 0; i < 4; ++i) v += s0 + i < S ? a[i] : 0.0f;
  }
  return v;
}
__device__ __forceinline__ f32x4 slab4(const float* p, int S, int64_t ss) {
  f32x4 v = *reinterpret_cast<const f32x4*>(p);
  for (int s0 = 1; s0 < S; s0 += 4) {
    f32x4 a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = *reinterpret_cast<const f32x4*>(p + min(s0 + i, S - 1) * ss);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s0 + i < S) v += a[i];
  }
  return v;
}

// The same in two halves, so that the loads of up to F slabs are in flight together with whatever else a row needs: a pass over a
// few rows is a chain of load latencies (most of its data was written by other XCDs a moment ago), not of bytes.  The order of
// the sum is slab4's.
template <int F>
struct Slab4 {
  f32x4 a[F];
  __device__ __forceinline__ void ask(const float* p, int S, int64_t ss) {
    a[0] = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
    for (int i = 1; i < F; ++i)
      if (i < S) a[i] = *reinterpret_cast<const f32x4*>(p + i * ss);
  }
  __device__ __forceinline__ f32x4 sum(const float* p, int S, int64_t ss) const {
    f32x4 v = a[0];
#pragma unroll
    for (int i = 1; i < F; ++i)
      if (i < S) v += a[i];
    for (int s0 = F; s0 < S; s0 += 4) {  // (the rest as slab4 takes them)
      f32x4 b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = *reinterpret_cast<const f32x4*>(p + min(s0 + i, S - 1) * ss);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s0 + i < S) v += b[i];
    }
    return v;
  }
};
constexpr int SLABS_ASKED = 12;  // of a row pass that sums split-K slabs (48 registers a vector of four)
// A row pass of few rows is its chain of latencies: 512 threads a row, every slab asked for at once.  At 200 rows the bytes of the
// slabs count already (a step of 200 tokens lost 0.7 % with that form), so the line lies where the decode steps end
inline bool few_rows(int64_t T) { return T <= 64; }

// Per-head norm and gate of prompts: out = o / rms(o) * w * gate * scale for heads of at most 128 values in whole vectors of four.
// What bounds it is the bytes: o and the gate once in fp32.  Half a wave has a head of TOK tokens and asks for o and the gate of all of
// them before the first is used, 16 bytes a lane (a wave per head with 4 or 8 bytes a lane kept too little in flight).  Cold, before and
// now, heads of 128: 4593 tokens x 32 heads logistic gate 89 us, 67 and silu gate 75, 67; 12807 x 16 117, 87 and 88, 87; heads of 68,
// 4593 x 16 36, 22 and 29, 22; behind the kernels that write its inputs 12807 x 16 silu 69, 47 and 4593 x 16 logistic 37, 18.  w: head h's weights from h wh on.
template <typename AT, bool SIG, int TOK>
__global__ __launch_bounds__(256) void gated_norm_half_k(const float* __restrict__ o, const float* __restrict__ w, int wh,
                                                         const float* __restrict__ P, int ldp, int g_off, float eps, float scale,
                                                         AT* __restrict__ out, int ldo, int T, int H, int dv) {
  const int t0 = blockIdx.x * TOK, h = blockIdx.y * 8 + (threadIdx.x >> 5), i = 4 * (threadIdx.x & 31);
  const bool in = h < H && i < dv;
  const int hc = min(h, H - 1), ic = in ? i : 0;  // (idle lanes read a valid place and write nothing)
  auto ld = [](const float* p) { return *reinterpret_cast<const f32x4*>(p); };
  f32x4 v[TOK], g[TOK];
#pragma unroll
  for (int r = 0; r < TOK; ++r) {
    const int64_t t = min(t0 + r, T - 1);
    v[r] = ld(o + (t * H + hc) * dv + ic);
    g[r] = ld(P + t * ldp + g_off + hc * dv + ic);
  }
  const f32x4 wv = ld(w + hc * wh + ic);
#pragma unroll
  for (int r = 0; r < TOK; ++r) {
    float ss = in ? (v[r][0] * v[r][0] + v[r][1] * v[r][1]) + (v[r][2] * v[r][2] + v[r][3] * v[r][3]) : 0.0f;
    ss = group16_sum(xor_sum<16>(ss));
    const float k = scale / sqrtf(ss / (float)dv + eps);
    if (!in || t0 + r >= T) continue;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = v[r][e] * k * wv[e] * (SIG ? sigmoidf_(g[r][e]) : siluf_(g[r][e]));
    st4(out + (int64_t)(t0 + r) * ldo + h * dv + i, y);
  }
}
// the forms it takes; each caller adds the size from which it is the faster one
inline bool gated_norm_half_ok(int64_t dv, int64_t strides, uintptr_t pointers) {
  return dv >= 68 && dv <= 128 && dv % 4 == 0 && strides % 4 == 0 && pointers % 16 == 0;
}

// ------------------------------------------------------------------ host side
#define MCHECK(cond, ...) TORCH_CHECK(cond, "xot mixers: ", __VA_ARGS__)

inline hipStream_t stream() { return at::hip::getCurrentHIPStream().stream(); }
inline bool is_act(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat; }
inline void f32c(const at::Tensor& t, const char* name) {
  MCHECK(t.is_cuda() && t.scalar_type() == at::kFloat && t.is_contiguous(), name, " must be a contiguous fp32 GPU tensor");
}
inline void i32c(const at::Tensor& t, const char* name) {
  MCHECK(t.is_cuda() && t.scalar_type() == at::kInt && t.is_contiguous(), name, " must be a contiguous int32 GPU tensor");
}
// fused projection output: fp32 rows of unit inner stride
inline int ld_of(const at::Tensor& P, const char* name) {
  MCHECK(P.is_cuda() && P.scalar_type() == at::kFloat && P.dim() == 2 && P.stride(1) == 1, name, " must be fp32 [T, n] rows");
  return (int)P.stride(0);
}
// fused projection output, plain [T, n] rows or unreduced split-K slabs [S, T, n]
struct Slabs {
  const float* p;
  int64_t T, n;
  int ld, S;
  int64_t ss;
  bool vec;  // rows and slabs start on 16-byte boundaries
};
inline Slabs slabs_of(const at::Tensor& P, const char* name) {
  MCHECK(P.is_cuda() && P.scalar_type() == at::kFloat && (P.dim() == 2 || P.dim() == 3) && P.stride(-1) == 1, name,
         " must be fp32 [T, n] rows or [slabs, T, n]");
  Slabs r;
  r.p = P.data_ptr<float>();
  r.T = P.size(-2);
  r.n = P.size(-1);
  r.ld = (int)P.stride(-2);
  r.S = P.dim() == 3 ? (int)P.size(0) : 1;
  r.ss = P.dim() == 3 ? P.stride(0) : 0;
  r.vec = r.ld % 4 == 0 && r.ss % 4 == 0 && (reinterpret_cast<uintptr_t>(r.p) & 15) == 0;
  return r;
}
inline void cols_ok(const Slabs& P, int64_t off, int64_t n, const char* what) {
  MCHECK(off >= 0 && n >= 0 && off + n <= P.n, what, ": columns [", off, ", ", off + n, ") outside the projection");
}
inline void cols_ok(const at::Tensor& P, int64_t off, int64_t n, const char* what) {
  MCHECK(off >= 0 && n >= 0 && off + n <= P.size(1), what, ": columns [", off, ", ", off + n, ") outside the projection");
}
// activation output rows (bf16 / fp32), maybe a column slice of a wider buffer
inline int act_ld(const at::Tensor& t, int64_t T, int64_t n, const char* name) {
  MCHECK(t.is_cuda() && is_act(t) && t.dim() == 2 && t.size(0) == T && t.size(1) == n && t.stride(1) == 1, name,
         " must be [T, ", n, "] bf16 / fp32 rows");
  return (int)t.stride(0);
}
// activation rows whose first n columns are written (K padding beyond stays untouched)
inline int act_ld_min(const at::Tensor& t, int64_t T, int64_t n, const char* name) {
  MCHECK(t.is_cuda() && is_act(t) && t.dim() == 2 && t.size(0) == T && t.size(1) >= n && t.stride(1) == 1, name,
         " must be [T, >= ", n, "] bf16 / fp32 rows");
  return (int)t.stride(0);
}

}  // namespace mix
}  // namespace xot
