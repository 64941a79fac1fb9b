// linear_recurrence for prompts: 16 tokens of a sequence at a time on the fp32 matrix units (gfx950).
//
// The token-by-token kernel (mixers.hip) is bound by its chain: about 970 cycles a token whatever the batch, two dot products
// with their cross-lane sums between one token and the next.  Over a chunk of 16 tokens the same recurrence is a handful
// of small products, with everything that does not need the state taken out of the chain.  P_i: the decays' product over
// the chunk's tokens up to i (one number per head, or one per key channel), G_ij = P_i / P_j, S the state before the chunk:
//   delta rule   U = M (V - (P K) S),  M = (I + tril(b_i G_ij k_i.k_j, -1))^-1 diag(b)      plain write   U = b V
//   O = (P Q) S + N U,  N = tril(G_ij q_i.k_j)            S <- P_16 S + (G_16,j K)^T U
//   * chunk_prep_k, a wave per (chunk, head), all of them in parallel: q.k and k.k products, the decays, the triangular
//     inverse by forward substitution -> M, N (16 x 16) and the scalar decays into a workspace, 2.1 KB per chunk and head.
//   * chunk_scan_k, the chain: a workgroup per (sequence, head, 32 value channels), a wave per 16 of them and half of the key
//     dims: the partial products are exchanged through LDS, and from 512 workgroups on a SIMD has two waves, one's products
//     under the other's waits (a wave with all key dims and 64 channels a workgroup: 294 us instead of 191 for one prompt of 2000,
//     427 / 419 for eight then).  The state stays in MFMA accumulators: tile t, register r, lane group g holds key row
//     16 t + 4 g + r of value channel lane % 16, and as a B operand the same register is rows 4 g + r of the tile for g = 0 .. 3
//     -- the A operands only have to name their k dims in that order, four consecutive floats a lane.  So the state never
//     moves, U and M, N meet the same way, and a chunk is 3 D / 8 + 8 MFMAs a wave (plain write: D / 4 + 4); q, k and the decays
//     pass LDS once per workgroup, two chunks ahead in registers.
// Bound by that chain: about 1.4 us a chunk at D 128 where 56 MFMAs of 32 cycles are 0.75 (the rest: two barriers, LDS
// reads and the four-step products with M and N between them).  Tarepel-design prompts (8 of 961 .. 2431 tokens, 16 heads
// of 128 x 128): 1018 -> 316 us, delta rule with channel decays 1124 -> 477.
// v_mfma_f32_16x16x4_f32 multiplies and accumulates in fp32 as the vector units do; no operand is rounded.
//
// Decays per key channel: where a prefix product P leaves 2^-100 .. 2^100 (a decay of 0, or a value that is no number, among
// others) the chunk takes exact pairwise products instead, so no ratio of vanishing products is formed.
#include "mixer_util.h"
#include "recurrence_chunk.h"

namespace xot {
namespace {
using namespace mix;

constexpr int CT = 16;                          // tokens a chunk
constexpr int MN = 2 * CT * CT + 2 * CT;        // workspace floats per (chunk, head): M, N, P_i, G_16,j
constexpr float FAR = 1.2676506e30f;            // 2^100
constexpr int RING = 2;                         // chunks in flight from memory (even: the LDS buffer alternates)

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// inclusive product over the 16 lanes of a DPP row, in lane order (lanes without a source keep their value: x * 1)
template <int CTRL>
__device__ __forceinline__ float row_mul(float v) {
  const float m = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(1.0f), __float_as_int(v), CTRL, 0xf, 0xf, false));
  return v * m;
}
__device__ __forceinline__ float row_scan(float v) {
  v = row_mul<0x111>(v);  // row_shr 1, 2, 4, 8
  v = row_mul<0x112>(v);
  v = row_mul<0x114>(v);
  return row_mul<0x118>(v);
}

// chunk slots of a step: sequence b's chunks start at cu[b] / 16 + b (at least ceil(n / 16) slots before the next one's)
__device__ __forceinline__ int slot_base(const int* cu, int b) { return cu[b] / CT + b; }

template <int D, bool CHAN, bool DELTA>
__global__ __launch_bounds__(64) void chunk_prep_k(const float* __restrict__ q, int ldq, const float* __restrict__ k, int ldk,
                                                   const float* __restrict__ decay, int dstride,
                                                   const float* __restrict__ beta, float q_scale,
                                                   const int* __restrict__ state_slots, const int* __restrict__ cu_q, int B,
                                                   int H, int G, float* __restrict__ ws) {
  __shared__ float sA[CT][CT + 1];
  const int s = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, i = lane & 15, g = lane >> 4;
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (slot_base(cu_q, mid) <= s) lo = mid; else hi = mid - 1;
  }
  const int t0 = cu_q[lo], n = cu_q[lo + 1] - t0, c = s - slot_base(cu_q, lo);
  if (state_slots[lo] < 0 || c * CT >= n) return;
  const int tok = c * CT + i;
  const bool valid = tok < n;
  const int64_t t = t0 + min(tok, n - 1);
  const int hk = h / (H / G);
  f32x4 qf[D / 16], kf[D / 16], af[CHAN ? D / 16 : 1];
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    qf[j] = *reinterpret_cast<const f32x4*>(q + t * ldq + hk * D + 16 * j + 4 * g);
    kf[j] = *reinterpret_cast<const f32x4*>(k + t * ldk + hk * D + 16 * j + 4 * g);
    if (CHAN) af[CHAN ? j : 0] = *reinterpret_cast<const f32x4*>(decay + (t * H + h) * D + 16 * j + 4 * g);
  }
  const float gi = CHAN || !valid ? 1.0f : decay[t * dstride + h];
  const float bi = DELTA && valid ? beta[t * H + h] : 0.0f;
  if (!valid) {
#pragma unroll
    for (int j = 0; j < D / 16; ++j) {
      qf[j] = kf[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (CHAN) af[CHAN ? j : 0] = f32x4{1.f, 1.f, 1.f, 1.f};
    }
  }
  float* M = ws + ((int64_t)s * H + h) * MN;
  // accumulators: row 4 g + r (token i), column lane % 16 (token j)
  f32x4 qs[8], ks[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) qs[r] = ks[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 gam = {1.f, 1.f, 1.f, 1.f};
  if (CHAN) {
    bool near = true;
    f32x4 P[D / 16];
#pragma unroll
    for (int j = 0; j < D / 16; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        P[j][r] = row_scan(af[CHAN ? j : 0][r]);
        near = near && P[j][r] >= 1.0f / FAR && P[j][r] <= FAR;
      }
    if (__all(near)) {
#pragma unroll
      for (int j = 0; j < D / 16; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float ki = kf[j][r] / P[j][r];
          qs[r + 4 * (j & 1)] = mfma4(qf[j][r] * P[j][r], ki, qs[r + 4 * (j & 1)]);
          if (DELTA) ks[r + 4 * (j & 1)] = mfma4(kf[j][r] * P[j][r], ki, ks[r + 4 * (j & 1)]);
        }
    } else {
      // row by row: kh_j = k_j times the decays after j, multiplied on token by token
      f32x4 kh[D / 16];
#pragma unroll
      for (int j = 0; j < D / 16; ++j) kh[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int row = 0; row < CT; ++row) {
        const int src = (lane & 48) + row;
        float dq = 0.0f, dk = 0.0f;
#pragma unroll
        for (int j = 0; j < D / 16; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float ar = __shfl(af[CHAN ? j : 0][r], src), qr = __shfl(qf[j][r], src), kr = __shfl(kf[j][r], src);
            kh[j][r] = i == row ? kf[j][r] : i < row ? kh[j][r] * ar : 0.0f;
            dq += qr * kh[j][r];
            if (DELTA) dk += kr * kh[j][r];
          }
        dq = xor_sum<16>(dq);
        dq = xor_sum<32>(dq);
        dk = xor_sum<16>(dk);
        dk = xor_sum<32>(dk);
        if ((row >> 2) == g) {
          qs[0][0] = (row & 3) == 0 ? dq : qs[0][0], ks[0][0] = (row & 3) == 0 ? dk : ks[0][0];
          qs[0][1] = (row & 3) == 1 ? dq : qs[0][1], ks[0][1] = (row & 3) == 1 ? dk : ks[0][1];
          qs[0][2] = (row & 3) == 2 ? dq : qs[0][2], ks[0][2] = (row & 3) == 2 ? dk : ks[0][2];
          qs[0][3] = (row & 3) == 3 ? dq : qs[0][3], ks[0][3] = (row & 3) == 3 ? dk : ks[0][3];
        }
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < D / 16; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        qs[r + 4 * (j & 1)] = mfma4(qf[j][r], kf[j][r], qs[r + 4 * (j & 1)]);
        if (DELTA) ks[r + 4 * (j & 1)] = mfma4(kf[j][r], kf[j][r], ks[r + 4 * (j & 1)]);
      }
    // G_ij: the decays after j up to i, multiplied on token by token (no quotient)
    float p = 1.0f, all = 1.0f, after = 1.0f;
#pragma unroll
    for (int row = 0; row < CT; ++row) {
      const float d = __shfl(gi, row);
      p = row > i ? p * d : 1.0f;
      all *= d;
      if (row > i) after *= d;
      if ((row >> 2) == g) {
        if ((row & 3) == 0) gam[0] = p; else if ((row & 3) == 1) gam[1] = p; else if ((row & 3) == 2) gam[2] = p; else gam[3] = p;
      }
      if (row == lane) M[2 * CT * CT + lane] = all;
    }
    if (lane < CT) M[2 * CT * CT + CT + lane] = after;
  }
  const f32x4 qk = ((qs[0] + qs[1]) + (qs[2] + qs[3])) + ((qs[4] + qs[5]) + (qs[6] + qs[7]));
  const f32x4 kk = ((ks[0] + ks[1]) + (ks[2] + ks[3])) + ((ks[4] + ks[5]) + (ks[6] + ks[7]));
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 4 * g + r;
    const float br = __shfl(bi, row);
    M[CT * CT + row * CT + i] = row >= i ? qk[r] * gam[r] * q_scale : 0.0f;
    if (DELTA) sA[row][i] = row > i ? kk[r] * gam[r] * br : 0.0f;
  }
  if (!DELTA) return;
  __syncthreads();
  // column i of (I + A)^-1 by forward substitution, 16 lanes (the other groups repeat it)
  float x[CT];
#pragma unroll
  for (int row = 0; row < CT; ++row) {
    float a0 = row == i ? 1.0f : 0.0f, a1 = 0.0f;
#pragma unroll
    for (int m = 0; m < row; ++m) {
      if (m & 1) a1 -= sA[row][m] * x[m];
      else a0 -= sA[row][m] * x[m];
    }
    x[row] = a0 + a1;
  }
#pragma unroll
  for (int row = 0; row < CT; ++row)
    if ((row >> 2) == g) M[row * CT + i] = row >= i ? x[row] * bi : 0.0f;  // (selected: bi may be no number)
}

// buffer over `bytes` from p on: loads past the end give 0, stores past it are dropped
__device__ __forceinline__ __amdgpu_buffer_rsrc_t window(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ f32x4 load4(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, int off) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// The scan's sequences in the order of their workgroups (0: the longest), `per` workgroups a sequence.  Two workgroups share a
// CU at about twice the time a chunk, so the long sequences are spread over the XCDs (heads fastest) and start first: with
// the sequences fastest an XCD had one of eight to itself.  Delta rule, 16 heads of 128 x 128, us before and so: 8 of 961 ..
// 2433 tokens 385 and 333, 16 of 110 .. 1820 536 and 244, 64 of 51 .. 1460 1433 and 708.  Where the launch is between one and
// two workgroups a CU, the second ones, which take the CUs in the order of the first, are the shortest, beside the shortest
// of the first that have a neighbour at all: 8 of 961 .. 2433 333 -> 316, 5 of 364 .. 1728 197 -> 183.
__device__ __forceinline__ int scan_order(int turn, int B, int per) {
  const int first = 256 / per, second = B - first;
  if (second <= 0 || second > first) return turn;
  return turn >= first ? B - 1 - (turn - first) : turn < second ? first - second + turn : turn - second;
}

template <int D, bool CHAN, bool DELTA>
__global__ __launch_bounds__(256, 2) void chunk_scan_k(
    const float* __restrict__ q, int ldq, const float* __restrict__ k, int ldk, const float* __restrict__ v, int ldv,
    const float* __restrict__ decay, const float* __restrict__ inscale, float q_scale, float* __restrict__ state,
    const int* __restrict__ state_slots, const int* __restrict__ cu_q, int B, int H, int G, int dv, int dvin,
    const float* __restrict__ ws, float* __restrict__ out) {
  constexpr int LD = D + 4;                       // LDS row: consecutive tokens four banks apart
  constexpr int NF = CT * D / 1024;               // float4s of k (and of q) a thread
  constexpr int HALVES = 128 / D, TH = CT / HALVES;  // channel decays: threads per (channel, operand), tokens of each
  constexpr bool KD = DELTA || !CHAN;             // k (channel decays: k P) rows, and the decayed k of the state update
  __shared__ __attribute__((aligned(16))) float sq[2][CT][LD], sk[KD ? 2 : 1][KD ? CT : 1][LD], sb[CHAN ? 2 : 1][CHAN ? CT : 1][LD];
  __shared__ __attribute__((aligned(16))) float sp[2][CHAN ? D : 4];
  __shared__ f32x4 sx[4][DELTA ? 2 : 1][64];      // the waves' partial products, for the wave with the other key dims
  constexpr int TILES = D / 32;                   // 16-row state tiles of a wave: half of the key dims
  const int h = blockIdx.x;
  const int b = nth_longest(B, scan_order((int)blockIdx.z, B, H * (int)gridDim.y), [&](int j) { return cu_q[j + 1] - cu_q[j]; });
  const int slot = state_slots[b];
  const int t0 = cu_q[b], n = cu_q[b + 1] - t0;
  if (slot < 0 || n <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 1;
  const int col = (int)blockIdx.y * 32 + (wave & 1) * 16 + i;
  const bool live = col < dv;
  const int hk = h / (H / G);
  const int d0 = half * (D / 2);                  // the wave's first key dim
  float* St = state + (((int64_t)slot * H + h) * dv + (live ? col : 0)) * D + d0 + 4 * g;
  f32x4 S[TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j) S[j] = *reinterpret_cast<const f32x4*>(St + 16 * j);
  const float* W = ws + ((int64_t)slot_base(cu_q, b) * H + h) * MN;
  const int64_t wstep = (int64_t)H * MN;

  // Every load of a chunk goes through a buffer that ends with the sequence: its base moves in scalar registers and a
  // lane's offset never changes, so a chunk's loads cost the vector unit nothing (64-bit addresses and clamped rows were
  // 2700 of 6500 cycles a chunk, 4600 with channel decays).  RING chunks ahead, in registers: the thread's share of q, k and
  // the decays; the wave's value rows; M, N, decays.  Nothing is computed from what is loaded until it is used.
  struct Share {
    f32x4 q[CHAN ? 1 : NF], k[CHAN ? 1 : NF];
    float a[CHAN ? CT : 1], x[CHAN ? TH : 1];
  };
  struct Wave {
    f32x4 v, m, nn, p, e;
    float all;
  };
  const int chunks = (n + CT - 1) / CT;
  const int ch = tid % D, part = tid / D, first = CHAN ? (part % HALVES) * TH : 0;
  const bool is_q = __builtin_amdgcn_readfirstlane(part >= HALVES);  // (whole waves)
  const float *q0 = q + (int64_t)t0 * ldq + hk * D, *k0 = k + (int64_t)t0 * ldk + hk * D, *v0 = v + (int64_t)t0 * ldv + h * dvin;
  const float *a0 = decay + ((int64_t)t0 * H + h) * D, *b0 = inscale + (int64_t)t0 * H + h;
  const float* x0 = is_q ? q0 : k0;
  const int ldx = is_q ? ldq : ldk;
  const int vcol = min(col, dvin - 1);
  auto fetch = [&](int cc, Share& s) {  // (past the end: the last chunk again, not used)
    const int c = min(cc, chunks - 1), left = n - c * CT;  // rows from here to the end
    if (CHAN) {
      const __amdgpu_buffer_rsrc_t ra = window(a0 + (int64_t)c * CT * H * D, ((int64_t)(left - 1) * H + 1) * D * 4);
      const __amdgpu_buffer_rsrc_t rx = window(x0 + (int64_t)c * CT * ldx, ((int64_t)(left - 1) * ldx + D) * 4);
#pragma unroll
      for (int j = 0; j < CT; ++j) s.a[CHAN ? j : 0] = load1(ra, (j * H * D + ch) * 4);
#pragma unroll
      for (int j = 0; j < TH; ++j) s.x[CHAN ? j : 0] = load1(rx, ((first + j) * ldx + ch) * 4);
    } else {
      const __amdgpu_buffer_rsrc_t rq = window(q0 + (int64_t)c * CT * ldq, ((int64_t)(left - 1) * ldq + D) * 4);
      const __amdgpu_buffer_rsrc_t rk = window(k0 + (int64_t)c * CT * ldk, ((int64_t)(left - 1) * ldk + D) * 4);
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        const int e = tid + 256 * j, tt = e / (D / 4), f = e % (D / 4);
        s.q[CHAN ? 0 : j] = load4(rq, (tt * ldq + 4 * f) * 4);
        s.k[CHAN ? 0 : j] = load4(rk, (tt * ldk + 4 * f) * 4);
      }
    }
  };
  auto fetch_wave = [&](int cc, Wave& w) {
    const int c = min(cc, chunks - 1), left = n - c * CT;
    const __amdgpu_buffer_rsrc_t rm = window(W + c * wstep, MN * 4);
    w.nn = load4(rm, (CT * CT + i * CT + 4 * g) * 4);
    if (DELTA) w.m = load4(rm, (i * CT + 4 * g) * 4);
    if (!CHAN) {
      w.p = load4(rm, (2 * CT * CT + 4 * g) * 4);
      w.e = load4(rm, (2 * CT * CT + CT + 4 * g) * 4);
      w.all = load1(rm, (2 * CT * CT + CT - 1) * 4);
    }
    const __amdgpu_buffer_rsrc_t rv = window(v0 + (int64_t)c * CT * ldv, ((int64_t)(left - 1) * ldv + dvin) * 4);
#pragma unroll
    for (int r = 0; r < 4; ++r) w.v[r] = load1(rv, ((4 * g + r) * ldv + vcol) * 4);
    if (!DELTA && inscale) {
      const __amdgpu_buffer_rsrc_t rb = window(b0 + (int64_t)c * CT * H, ((int64_t)(left - 1) * H + 1) * 4);
#pragma unroll
      for (int r = 0; r < 4; ++r) w.m[r] = load1(rb, (4 * g + r) * H * 4);
    }
  };
  auto stage = [&](int c, int buf, const Share& s) {  // tokens past the end: k = q = 0 and a decay of 1 leave the state as it is
    if (CHAN) {
      float a[CT], pre[CT], suf[CT];
      float x = 1.0f;
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        a[j] = c * CT + j < n ? s.a[CHAN ? j : 0] : 1.0f;
        x *= a[j];
        pre[j] = x;
      }
      if (part == 0) sp[buf][CHAN ? ch : 0] = x;
      x = 1.0f;
#pragma unroll
      for (int j = CT - 1; j >= 0; --j) {
        suf[j] = x;
        x *= a[j];
      }
      // (compile-time register indices: each of the halves' tokens selected, not addressed)
#pragma unroll
      for (int j = 0; j < TH; ++j) {
        const bool up = HALVES > 1 && first != 0;
        const float p = up ? pre[j + CT - TH] : pre[j], e = up ? suf[j + CT - TH] : suf[j];
        // (q and k threads write different rows by address, without a branch)
        float* row = is_q ? &sq[buf][0][0] : &sb[CHAN ? buf : 0][0][0];
        row[(first + j) * LD + ch] = s.x[CHAN ? j : 0] * (is_q ? p * q_scale : e);
        if (KD && !is_q) sk[KD ? buf : 0][KD ? first + j : 0][ch] = s.x[CHAN ? j : 0] * p;
      }
    } else {
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        const int e = tid + 256 * j, tt = e / (D / 4), f = e % (D / 4);
        *reinterpret_cast<f32x4*>(&sq[buf][tt][4 * f]) = s.q[CHAN ? 0 : j] * q_scale;
        *reinterpret_cast<f32x4*>(&sk[KD ? buf : 0][KD ? tt : 0][4 * f]) = s.k[CHAN ? 0 : j];
      }
    }
  };
  const int64_t ldo = (int64_t)H * dv;
  float* o0 = out + (int64_t)t0 * ldo + h * dv;
  // barrier that leaves loads and stores to memory in flight (LDS writes done): the prefetch lives across it
  auto bar = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // c + L b, L lower triangular (lane: row i of L, tokens 4 g + r; row r of b and c: token 4 g + r).  The products with the zeros
  // above its diagonal would carry an infinity or a NaN of b back to earlier tokens: such a chunk sums what is below alone
  // (all lanes of the wave; no memory operation, so that the loads in flight are waited for as without it).
  auto lower = [&](f32x4 l, f32x4 b, f32x4 c) {
    uint32_t top = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) top = max(top, __float_as_uint(b[r]) & 0x7fffffffu);
    if (__builtin_expect(__any(top >= 0x7f800000u), 0)) {
#pragma unroll
      for (int m = 0; m < CT; ++m) {
        const float bm = __shfl(b[m & 3], (m >> 2) * 16 + i);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float lm = __shfl(l[m & 3], (m >> 2) * 16 + 4 * g + r);
          c[r] = m <= 4 * g + r ? c[r] + lm * bm : c[r];
        }
      }
      return c;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) c = mfma4(l[r], b[r], c);
    return c;
  };
  Share sh[RING];
  Wave wv[RING];
#pragma unroll
  for (int u = 0; u < RING; ++u) {
    fetch(u, sh[u]);
    fetch_wave(u, wv[u]);
  }
  stage(0, 0, sh[0]);
  bar();
  auto chunk = [&](int c, int buf, Share& mine, Share& ahead, Wave& cur) {
    fetch(c + RING, mine);
    // (four partial sums each: shorter chains, and sums of D / 4 terms instead of D)
    f32x4 xs[4], ys[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) xs[r] = ys[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const f32x4 qa = *reinterpret_cast<const f32x4*>(&sq[buf][i][d0 + 16 * j + 4 * g]);
      f32x4 ka;
      if (DELTA) ka = *reinterpret_cast<const f32x4*>(&sk[KD ? buf : 0][KD ? i : 0][d0 + 16 * j + 4 * g]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (DELTA) xs[r] = mfma4(ka[r], S[j][r], xs[r]);
        ys[r] = mfma4(qa[r], S[j][r], ys[r]);
      }
    }
    // the decayed state meets the chunk's write after the products that read it
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const f32x4 p = CHAN ? *reinterpret_cast<const f32x4*>(&sp[buf][CHAN ? d0 + 16 * j + 4 * g : 0]) : f32x4{cur.all, cur.all, cur.all, cur.all};
#pragma unroll
      for (int r = 0; r < 4; ++r) S[j][r] *= p[r];
    }
    f32x4 X = (xs[0] + xs[1]) + (xs[2] + xs[3]);
    f32x4 Y = (ys[0] + ys[1]) + (ys[2] + ys[3]);
    if (DELTA) sx[wave][DELTA ? 1 : 0][lane] = X;
    if (half == 1) sx[wave][0][lane] = Y;
    bar();
    if (DELTA) X += sx[wave ^ 2][DELTA ? 1 : 0][lane];
    Y += sx[wave | 2][0][lane];  // (used by the waves of the first half)
    f32x4 U;  // the value rows (0 past the end); the normaliser's channel is fed with ones
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      U[r] = col < dvin ? cur.v[r] : col < dv && c * CT + 4 * g + r < n ? 1.0f : 0.0f;
      if (!DELTA && inscale) U[r] *= cur.m[r];
    }
    if (DELTA) {
      f32x4 R;
#pragma unroll
      for (int r = 0; r < 4; ++r) R[r] = U[r] - (CHAN ? X[r] : cur.p[r] * X[r]);
      U = lower(cur.m, R, f32x4{0.f, 0.f, 0.f, 0.f});
    }
    if (!CHAN) {
#pragma unroll
      for (int r = 0; r < 4; ++r) Y[r] *= cur.p[r];
    }
    Y = lower(cur.nn, U, Y);
    f32x4 E = U;
    if (!CHAN) {
#pragma unroll
      for (int r = 0; r < 4; ++r) E[r] *= cur.e[r];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < TILES; ++j) {
        const int e = d0 + 16 * j + i;
        const float ka = CHAN ? sb[CHAN ? buf : 0][CHAN ? 4 * g + r : 0][e] : sk[KD ? buf : 0][KD ? 4 * g + r : 0][e];
        S[j] = mfma4(ka, E[r], S[j]);
      }
    const __amdgpu_buffer_rsrc_t ro = window(o0 + (int64_t)c * CT * ldo, ((int64_t)(n - c * CT - 1) * ldo + dv) * 4);
#pragma unroll
    for (int r = 0; r < 4; ++r)  // (channels past the end and the second half's waves: an offset no window reaches)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(Y[r]), ro, live && half == 0 ? (int)(((4 * g + r) * ldo + col) * 4) : -16, 0, 0);
    fetch_wave(c + RING, cur);
    stage(c + 1, buf ^ 1, ahead);  // (its last readers passed the barrier that ended the previous chunk)
    bar();
  };
  // whole rings without a branch between the chunks (at a join the compiler waits for every load that one of the paths may
  // have issued last), then the rest
  int c = 0;
  for (; c + RING <= chunks; c += RING) {
#pragma unroll
    for (int u = 0; u < RING; ++u) chunk(c + u, u & 1, sh[u], sh[(u + 1) % RING], wv[u]);
  }
#pragma unroll
  for (int u = 0; u < RING - 1; ++u)
    if (c + u < chunks) chunk(c + u, u & 1, sh[u], sh[u + 1], wv[u]);
  if (live) {
#pragma unroll
    for (int j = 0; j < TILES; ++j) *reinterpret_cast<f32x4*>(St + 16 * j) = S[j];
  }
}

template <int D, bool CHAN, bool DELTA>
void go(const ChunkRecurrence& a) {
  const int slots = a.T / CT + a.B;
  const dim3 pg((unsigned)slots, (unsigned)a.H), sg((unsigned)a.H, (unsigned)((a.dv + 31) / 32), (unsigned)a.B);
  chunk_prep_k<D, CHAN, DELTA><<<pg, 64, 0, stream()>>>(a.q, a.ldq, a.k, a.ldk, a.decay, a.dstride, a.beta, a.q_scale,
                                                        a.state_slots, a.cu_q, a.B, a.H, a.G, a.ws);
  chunk_scan_k<D, CHAN, DELTA><<<sg, 256, 0, stream()>>>(a.q, a.ldq, a.k, a.ldk, a.v, a.ldv, a.decay, DELTA ? nullptr : a.beta,
                                                         a.q_scale, a.state, a.state_slots, a.cu_q, a.B, a.H, a.G, a.dv, a.dvin,
                                                         a.ws, a.out);
}

}  // namespace

int64_t chunk_recurrence_ws(int64_t T, int64_t B, int64_t H) { return (T / CT + B) * H * MN; }

void chunk_recurrence(const ChunkRecurrence& a) {
#define XOT_CHUNK(D)                                              \
  do {                                                            \
    if (a.chan && a.delta) go<D, true, true>(a);                  \
    else if (a.chan) go<D, true, false>(a);                       \
    else if (a.delta) go<D, false, true>(a);                      \
    else go<D, false, false>(a);                                  \
  } while (0)
  if (a.d == 64) XOT_CHUNK(64);
  else XOT_CHUNK(128);
#undef XOT_CHUNK
}

}  // namespace xot
