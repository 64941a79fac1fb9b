// Linear recurrences of a step of single tokens, with the per-head gated RMS norm that follows them in the layers whose norm
// groups are the heads:  S <- recurrence(S), o = S^T q,  out = o / rms(o) * w * gate * scale.
//
// Workgroup = (sequence, value head); 512 threads = 32 value channels x 16 groups of key rows, NC rounds of channels.  What bounds
// it is the state, read and written once (48 sequences x 16 heads x 128 x 128 fp32: 101 MB): every load of it is asked for at once,
// in whole 256-byte runs, next to k, q and the decays, which come straight from memory (one token: nothing to stage).  The general
// kernel (mixers.hip linear_recurrence_k) has 8 KB of state a workgroup behind a pass through LDS, and the norm and the decays of
// gated linear attention were launches of their own; here a head's outputs meet in LDS, and a parallel block's gated activation, 4.9 us
// on its own, fills in behind the heads.  us, before / here: delta rule as above
// 26.2 + 4.7 (norm) / 17.5 (5.8 TB/s), gated linear attention 64 x 128 4.7 (decays) + 15.4 + 4.7 / 11.3; 6 sequences, channel decays
// 5.7 + 3.9 / 6.1.
// MODE 0: gated linear attention, S = diag(a) S + k v^T with a = exp(logsigmoid(a2 . P[a1 ...] + b) / tau) made here.  MODE 1:
// delta rule, S *= g; u = beta (v - S^T k); S += k u^T.  MODE 4: the delta rule with a decay per key channel.
#include "mixer_util.h"

namespace xot {
namespace {

using namespace mix;

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// sum over the 16 lanes of a DPP row
__device__ __forceinline__ float row_sum(float v) {
  v = dpp_add<0xB1>(v);
  v = dpp_add<0x4E>(v);
  v = dpp_add<0x141>(v);
  return dpp_add<0x140>(v);
}

struct StepArgs {
  const float *q, *k, *v, *decay, *beta;
  int ldq, ldk, ldv;
  float q_scale;
  float* state;
  const int *slots, *cu;
  int H, G;
  // MODE 0: decays' low-rank row, weights [H d, rank], bias
  const float *a1, *a2, *a2_b;
  int ld1, rank;
  float inv_tau;
  // norm weight of channel i of head h: w[h wh + i]; gate: silu, or the logistic function
  const float *w, *gate;
  int wh, ldg;
  bool sig, bf;
  float eps, scale;
  void* out;
  int ldo;
};

// A parallel block's gated activation gelu(gate) * up, which only needs the projections as well (workgroups behind the heads')
struct GeluArgs {
  const float* P;
  int ld, gate, up, F;  // up < 0: gate and up columns alternate in tiles of 16
  void* out;
  int ldo;
  bool bf;
  int total;  // groups of four columns
};

__device__ __forceinline__ void gelu_part(const GeluArgs& a, int idx) {
  if (idx >= a.total) return;
  const int nw = a.F / 4, t = idx / nw, i = (idx - t * nw) * 4;
  const float* gp = a.P + (int64_t)t * a.ld + a.gate + (a.up < 0 ? 32 * (i >> 4) + (i & 15) : i);
  const float* up = a.up < 0 ? gp + 16 : a.P + (int64_t)t * a.ld + a.up + i;
  const f32x4 z = *reinterpret_cast<const f32x4*>(gp), u = *reinterpret_cast<const f32x4*>(up);
  f32x4 y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = gelu_tanhf_(z[e]) * u[e];
  if (a.bf) st4(static_cast<uint16_t*>(a.out) + (int64_t)t * a.ldo + i, y);
  else st4(static_cast<float*>(a.out) + (int64_t)t * a.ldo + i, y);
}

constexpr int CW = 32;

template <int D, int MODE, int NC>
__global__ __launch_bounds__(512) void recurrence_step_k(StepArgs a, int heads, GeluArgs ge) {
  constexpr int KJ = D / 64, dv = CW * NC;  // float4s of key rows a thread has
  __shared__ float so[dv];
  __shared__ __attribute__((aligned(16))) float sd[MODE == 0 ? D : 4];
  const int tid = threadIdx.x, rg = tid & 15, cl = tid >> 4;
  if ((int)blockIdx.x >= heads) {  // (heads: sequences x value heads)
    gelu_part(ge, ((int)blockIdx.x - heads) * 512 + tid);
    return;
  }
  const int b = blockIdx.x / a.H, h = blockIdx.x - b * a.H;
  const int slot = a.slots[b], t = a.cu[b];
  if (slot < 0 || a.cu[b + 1] <= t) return;  // (the same for all threads)
  const int hk = h / (a.H / a.G);
  auto ld = [](const float* p) { return *reinterpret_cast<const f32x4*>(p); };
  float* S = a.state + (((int64_t)slot * a.H + h) * dv + cl) * D + rg * 4;
  f32x4 s[NC][KJ], k[KJ], q[KJ], dec[KJ];
  float v[NC], g = 0.0f, be = 0.0f;
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int j = 0; j < KJ; ++j) s[c][j] = ld(S + c * CW * D + 64 * j);
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    const int i = hk * D + 64 * j + rg * 4;
    k[j] = ld(a.k + (int64_t)t * a.ldk + i);
    q[j] = ld(a.q + (int64_t)t * a.ldq + i);
    if (MODE == 4) dec[j] = ld(a.decay + ((int64_t)t * a.H + h) * D + 64 * j + rg * 4);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) v[c] = a.v[(int64_t)t * a.ldv + h * dv + c * CW + cl];
  if (MODE == 1) g = a.decay[(int64_t)t * a.H + h];
  if (MODE != 0) be = a.beta[(int64_t)t * a.H + h];
  float gv = 0.0f, wv = 0.0f;  // gate and norm weight of output channel tid
  if (tid < dv) {
    gv = a.gate[(int64_t)t * a.ldg + h * dv + tid];
    wv = a.w[h * a.wh + tid];
  }
  if constexpr (MODE == 0) {
    if (tid < D) {
      const float *wr = a.a2 + (int64_t)(h * D + tid) * a.rank, *p = a.a1 + (int64_t)t * a.ld1;
      float z = 0.0f;
#pragma unroll 4
      for (int r = 0; r < a.rank; ++r) z += wr[r] * p[r];
      sd[tid] = expf(logsigmoidf_(z + a.a2_b[h * D + tid]) * a.inv_tau);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < KJ; ++j) dec[j] = *reinterpret_cast<const f32x4*>(sd + 64 * j + rg * 4);
  }
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    q[j] *= a.q_scale;
    if (MODE == 1) dec[j] = f32x4{g, g, g, g};
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    float u = v[c];
    if (MODE != 0) {
      f32x4 p = {};
#pragma unroll
      for (int j = 0; j < KJ; ++j) {
        s[c][j] *= dec[j];
        p += s[c][j] * k[j];
      }
      u = be * (u - row_sum((p[0] + p[1]) + (p[2] + p[3])));
    }
    f32x4 o = {};
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
      s[c][j] = MODE != 0 ? s[c][j] + k[j] * u : dec[j] * s[c][j] + k[j] * u;
      o += s[c][j] * q[j];
      *reinterpret_cast<f32x4*>(S + c * CW * D + 64 * j) = s[c][j];
    }
    const float r = row_sum((o[0] + o[1]) + (o[2] + o[3]));
    if (rg == 0) so[c * CW + cl] = r;
  }
  __syncthreads();
  if (tid >= (dv + 63) / 64 * 64) return;  // whole waves
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < dv; i += 64) {
    const float x = i + (tid & 63) < dv ? so[i + (tid & 63)] : 0.0f;
    ss += x * x;
  }
  const float n = a.scale / sqrtf(wave_sum(ss) / (float)dv + a.eps);
  if (tid >= dv) return;
  const float y = so[tid] * n * wv * (a.sig ? sigmoidf_(gv) : siluf_(gv));
  if (a.bf) static_cast<uint16_t*>(a.out)[(int64_t)t * a.ldo + h * dv + tid] = f2bf(y);
  else static_cast<float*>(a.out)[(int64_t)t * a.ldo + h * dv + tid] = y;
}

// The whole of it for T = B single tokens where it is covered: key dims of 64 and 128, value dims of 32, 64 and 128, rows on 16 bytes.
// Arguments as in linear_recurrence (delta rules alone; gla: (a1 [T, rank] rows, a2, a2_b, tau), a decay per key channel),
// then the norm's weight ([dv], or one per head [H dv]), the gate's rows, whether its function is the logistic one, eps, out's scale;
// with gelu_P the arguments of gelu_mul, whose work joins the launch.
bool recurrence_step(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const c10::optional<at::Tensor>& decay,
                     const c10::optional<at::Tensor>& beta, double q_scale, at::Tensor& state, const at::Tensor& state_slots,
                     const at::Tensor& cu_q, const c10::optional<at::Tensor>& a1, const c10::optional<at::Tensor>& a2,
                     const c10::optional<at::Tensor>& a2_b, double tau, const at::Tensor& w, const at::Tensor& gate, bool sig, double eps,
                     double scale, at::Tensor& out, const c10::optional<at::Tensor>& gelu_P, int64_t gate_off, int64_t up_off, int64_t F,
                     const c10::optional<at::Tensor>& act) {
  StepArgs a{};
  a.ldq = ld_of(q, "q"), a.ldk = ld_of(k, "k"), a.ldv = ld_of(v, "v");
  f32c(state, "state");
  i32c(state_slots, "state_slots");
  i32c(cu_q, "cu_q");
  f32c(w, "w");
  MCHECK(state.dim() == 4, "state must be [slots, H, dv, d]");
  const int64_t T = q.size(0), H = state.size(1), dv = state.size(2), d = state.size(3), B = state_slots.numel();
  if (T != B || T == 0 || (d != 64 && d != 128) || (dv != 32 && dv != 64 && dv != 128) || a2.has_value() == beta.has_value()) return false;
  MCHECK(q.size(1) % d == 0 && q.size(1) == k.size(1) && k.size(0) == T && v.size(0) == T && v.size(1) == H * dv, "recurrence_step: shape mismatch");
  const int64_t G = q.size(1) / d;
  MCHECK(G > 0 && H % G == 0 && cu_q.numel() == B + 1, "recurrence_step: heads or offsets");
  auto on16 = [](const at::Tensor& t, int ld) { return ld % 4 == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; };
  if (!on16(q, a.ldq) || !on16(k, a.ldk) || !on16(state, 0)) return false;
  int mode = 0;
  if (beta.has_value()) {
    MCHECK(decay.has_value(), "the delta rule needs its decays");
    f32c(*beta, "beta");
    f32c(*decay, "decay");
    MCHECK(beta->numel() == T * H && (decay->numel() == T * H || decay->numel() == T * H * d), "beta must be [T, H], the decay [T, H] or [T, H d]");
    mode = decay->numel() == T * H ? 1 : 4;
    if (!on16(*decay, 0)) return false;
    a.beta = beta->data_ptr<float>();
    a.decay = decay->data_ptr<float>();
  } else {
    MCHECK(a1.has_value() && a2_b.has_value() && tau > 0 && G == H, "gated linear attention: decay projections, one q / k head per value head");
    f32c(*a2, "a2");
    f32c(*a2_b, "a2_b");
    a.ld1 = ld_of(*a1, "a1");
    MCHECK(a1->size(0) == T && a2->dim() == 2 && a2->size(0) == H * d && a2->size(1) == a1->size(1) && a2_b->numel() == H * d,
           "gated linear attention: shape mismatch");
    a.a1 = a1->data_ptr<float>();
    a.a2 = a2->data_ptr<float>();
    a.a2_b = a2_b->data_ptr<float>();
    a.rank = (int)a1->size(1);
    a.inv_tau = (float)(1.0 / tau);
  }
  a.q = q.data_ptr<float>(), a.k = k.data_ptr<float>(), a.v = v.data_ptr<float>();
  a.q_scale = (float)q_scale;
  a.state = state.data_ptr<float>();
  a.slots = state_slots.data_ptr<int>(), a.cu = cu_q.data_ptr<int>();
  a.H = (int)H, a.G = (int)G;
  MCHECK(w.numel() == dv || w.numel() == H * dv, "the norm's weight must hold dv or H dv numbers");
  a.w = w.data_ptr<float>();
  a.wh = w.numel() == dv ? 0 : (int)dv;
  a.ldg = ld_of(gate, "gate");
  MCHECK(gate.size(0) == T && gate.size(1) >= H * dv, "the gate must be [T, >= H dv]");
  a.gate = gate.data_ptr<float>();
  a.ldo = act_ld_min(out, T, H * dv, "out");
  a.out = out.data_ptr();
  a.sig = sig, a.bf = out.scalar_type() == at::kBFloat16;
  a.eps = (float)eps, a.scale = (float)scale;
  GeluArgs ge{};
  if (gelu_P.has_value()) {
    ge.ld = ld_of(*gelu_P, "P");
    MCHECK(act.has_value() && gelu_P->size(0) == T, "the activation's rows");
    ge.ldo = act_ld_min(*act, T, F, "activation");
    cols_ok(*gelu_P, gate_off, up_off == -1 ? (F + 15) / 16 * 32 : F, "gate");
    if (up_off != -1) cols_ok(*gelu_P, up_off, F, "up");
    if ((ge.ld | gate_off | F | ge.ldo | (up_off == -1 ? 0 : up_off)) % 4 != 0 || T * F >= (int64_t(1) << 31) ||
        ((reinterpret_cast<uintptr_t>(gelu_P->data_ptr()) | reinterpret_cast<uintptr_t>(act->data_ptr())) & 15) != 0)
      return false;
    ge.P = gelu_P->data_ptr<float>();
    ge.gate = (int)gate_off, ge.up = (int)up_off, ge.F = (int)F;
    ge.out = act->data_ptr();
    ge.bf = act->scalar_type() == at::kBFloat16;
    ge.total = (int)(T * F / 4);
  }
  MCHECK(B * H < (int64_t(1) << 30), "recurrence_step: too many heads");
  const int heads = (int)(B * H), grid = heads + (ge.total + 511) / 512;
  auto go = [&](auto D, auto MODE) {
    constexpr int D_ = decltype(D)::value, M_ = decltype(MODE)::value;
    if (dv == 32) recurrence_step_k<D_, M_, 1><<<grid, 512, 0, stream()>>>(a, heads, ge);
    else if (dv == 64) recurrence_step_k<D_, M_, 2><<<grid, 512, 0, stream()>>>(a, heads, ge);
    else recurrence_step_k<D_, M_, 4><<<grid, 512, 0, stream()>>>(a, heads, ge);
  };
  auto by_mode = [&](auto D) {
    if (mode == 0) go(D, std::integral_constant<int, 0>());
    else if (mode == 1) go(D, std::integral_constant<int, 1>());
    else go(D, std::integral_constant<int, 4>());
  };
  if (d == 64) by_mode(std::integral_constant<int, 64>());
  else by_mode(std::integral_constant<int, 128>());
  return true;
}

}  // namespace

void bind_recurrence_step(pybind11::module& m) { m.def("recurrence_step", &recurrence_step); }

}  // namespace xot
