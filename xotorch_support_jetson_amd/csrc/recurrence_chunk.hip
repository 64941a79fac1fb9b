// linear_recurrence for prompts: 16 tokens of a sequence at a time on the fp32 matrix units (gfx950).
//
// The token-by-token kernel (mixers.hip) is bound by its chain: about 970 cycles a token whatever the batch, two dot products
// with their cross-lane sums between one token and the next.  Over a chunk of 16 tokens the same recurrence is a handful
// of small products, with everything that does not need the state taken out of the chain.  P_i: the decays' product over
// the chunk's tokens up to i (one number per head, or one per key channel), G_ij = P_i / P_j, S the state before the chunk:
//   delta rule   U = M (V - (P K) S),  M = (I + tril(b_i G_ij k_i.k_j, -1))^-1 diag(b)      plain write   U = b V
//   O = (P Q) S + N U,  N = tril(G_ij q_i.k_j)            S <- P_16 S + (G_16,j K)^T U
//   * chunk_prep_k, a wave per (chunk, head), all of them in parallel: q.k and k.k products, the decays, the triangular
//     inverse by forward substitution -> M, N (16 x 16) and the scalar decays into a workspace, 2.1 KB per chunk and head.  With channel
//     decays the scan's operands P Q, P K and (G K)^T follow them, up to 24 KB: what it costs to write them (16 heads of 128 x 128,
//     4593 tokens: 45 us without, 64 with) every workgroup of the scan was paying again, 16 products a thread and chunk on the chain.
//   * chunk_scan_k, the chain: a workgroup per (sequence, head, 16 or 32 value channels), a wave per 16 of them and a quarter or half
//     of the key dims.  The state stays in MFMA accumulators: tile t, register r, lane group g holds key row
//     16 t + 4 g + r of value channel lane % 16, and as a B operand the same register is rows 4 g + r of the tile for g = 0 .. 3
//     -- the A operands only have to name their k dims in that order, four consecutive floats a lane.  So the state never
//     moves, U and M, N meet the same way, and q and k come from memory as the operands they are, one to three chunks ahead in
//     registers: nothing is staged for a workgroup, and a chunk has one barrier, behind which the partial products k S of the
//     other key dims are read (those of q S a chunk later, they are not on the chain).
// What bounds it: with few sequences the chain, k S -> exchange -> M -> write, 1.0 us a chunk at D 128 (1.5 with q, k and decays through
// LDS, all waves' products of half of the key dims and two barriers; a wave issues one instruction at a time, and loads,
// addresses and selections between the MFMAs were as many as them).  With many the matrix unit: 54 MFMAs of 32 cycles a wave of
// half of the key dims, at 55 % of its rate.  One prompt of 2000 tokens, both kernels, us before and now: delta rule 16 heads of 128 x 128
// 197 and 129, with channel decays 306 and 136, per-channel decays 16 heads of 64 x 128 153 and 81, plain write 32 heads of 128 x 64 156 and
// 103; 5 of 364 .. 1728: 185, 293, 141, 150 and 143, 181, 87, 104; 8 of 961 .. 2433: 307, 488, 219, 253 and 292, 402, 197, 223; 32 of
// 50 .. 1515: 314, 476, 211, 283 and 317, 439, 202, 243.
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
// workspace floats of a (chunk, head): with channel decays the scan's operands follow, the decay over the chunk (D), then P Q, (G K)^T
// and (delta rule) P K by state tile and lane
constexpr int rec_floats(int D, bool chan, bool delta) { return MN + (chan ? D + (delta ? 3 : 2) * CT * D : 0); }
constexpr int64_t WS_MOST = 128 << 20;          // workspace floats (Portions)

// A record is 2.2 KB a chunk and head, with channel decays up to 27 KB (key dims of 128 under the delta rule: 3.3 times the decays that
// it replaces).  Steps whose records fit 512 MB (19.7 thousand tokens of 16 such heads) go at once, longer ones in portions, each with as
// many chunks of every sequence, so that the sequences go on side by side.  Where the lengths are unlike enough to double the portions,
// a portion would be fewer than 64 chunks of each or the longest is not known, portions are slots as they come.  The same heads, us at once
// / in portions / as slots come: three of 9000 tokens 980 / 1024 / 1415, of 20000 2147 / 2254 / 3475, six of 8000 1556 / 1640 / 2054;
// 64 of 512, which go as slots come, 907 / - / 952.  (16 to 32 us of the portions are the launches for what the longest, if it was
// understated, would leave.)
struct Portions {
  int count, slots, each;  // slots of the workspace; each: chunks of a sequence in a portion, or 0
};
Portions portions(int64_t T, int64_t B, int64_t H, int rec, int64_t longest) {
  const int64_t slots = T / CT + B, most = std::max<int64_t>(WS_MOST / (H * rec), 1), parts = (slots + most - 1) / most;
  const int64_t each = most / B, chunks = (longest + CT - 1) / CT;
  if (parts > 1 && longest > 0 && each >= 64 && chunks <= 2 * parts * each) {
    const int64_t turns = (chunks + each - 1) / each, even = (chunks + turns - 1) / turns;
    return {(int)turns, (int)(B * even), (int)even};
  }
  return {(int)parts, (int)((slots + parts - 1) / parts), 0};
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// a b, rounded before anything is added to it
__device__ __forceinline__ f32x4 times(f32x4 a, f32x4 b) {
#pragma clang fp contract(off)
  return a * b;
}

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

// exclusive product of the lanes behind, in the same row
__device__ __forceinline__ float row_after(float v) {
  v = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(1.0f), __float_as_int(v), 0x101, 0xf, 0xf, false));  // row_shl 1
  v = row_mul<0x101>(v);
  v = row_mul<0x102>(v);
  v = row_mul<0x104>(v);
  return row_mul<0x108>(v);
}

// chunk slots of a step: sequence b's chunks start at cu[b] / 16 + b (at least ceil(n / 16) slots before the next one's)
__device__ __forceinline__ int slot_base(const int* cu, int b) { return cu[b] / CT + b; }

// Bound by the bytes, what it reads and the operands it writes, and by registers, of which three waves a SIMD leave 168: tile by tile in a
// chunk with channel decays, and once more from memory where a prefix product left the range (all tiles held: one wave a SIMD, 69 us).
// What the tiles are made of is loaded ahead of them all, 96 registers at key dims of 128, and under the delta rule with channel decays 17 of
// them (22 where the decays are made) are in scratch memory meanwhile, 68 (92) bytes a lane.
// MADE: the decays (and the delta rule's write strengths) come from src, in the vector unit's time.  A pass of its own that wrote them cost,
// behind the kernels that write its inputs, 48 us for 12807 tokens of 16 heads of 64 (rank 16) and 40 for 4593 of 16 of 128, of
// which the exponentials here take 29 (58 -> 87) and 25 (64 -> 89).
template <int D, bool CHAN, bool DELTA, bool MADE>
__global__ __launch_bounds__(64, CHAN ? 3 : 2) void chunk_prep_k(const float* __restrict__ q, int ldq, const float* __restrict__ k, int ldk,
                                                   const float* __restrict__ decay, int dstride,
                                                   const float* __restrict__ beta, float q_scale,
                                                   const int* __restrict__ state_slots, const int* __restrict__ cu_q, int B,
                                                   int H, int G, int heads, DecaySource src, int from, int each, int done,
                                                   float* __restrict__ ws) {
  __shared__ float sA[CT][CT + 1];
  __shared__ __attribute__((aligned(16))) float sT[CHAN ? 2 : 1][CHAN ? CT : 1][CT + 4];  // a tile's way from dims to tokens
  constexpr bool SHARE = !CHAN && !DELTA;
  const int per = SHARE ? H / heads : H;  // workgroups a chunk, neighbours: they read and write whole rows together (channel
                                         // decays made, 4593 tokens x 16 heads of 128 100 -> 91 us; delta rule, 12807 48 -> 44)
  const int s = (int)(blockIdx.x / per), h = blockIdx.x % per * (SHARE ? heads : 1), lane = threadIdx.x, i = lane & 15, g = lane >> 4;
  int lo = 0, hi = B - 1, c;
  if (each) {
    lo = s / each;
    c = from + s % each;
  } else {
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (slot_base(cu_q, mid) <= from + s) lo = mid; else hi = mid - 1;
    }
    c = from + s - slot_base(cu_q, lo);
  }
  const int t0 = cu_q[lo], n = cu_q[lo + 1] - t0;
  if (state_slots[lo] < 0 || c < done || c * CT >= n) return;
  const int tok = c * CT + i;
  const bool valid = tok < n;
  const int64_t t = t0 + min(tok, n - 1);
  const int hk = h / (H / G);
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  // tile j of the tokens' q, k (past the end: 0) and what their decays come from
  auto load_q = [&](int j) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(q + t * ldq + hk * D + 16 * j + 4 * g);
    return valid ? x : zero4;
  };
  auto load_k = [&](int j) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(k + t * ldk + hk * D + 16 * j + 4 * g);
    return valid ? x : zero4;
  };
  auto load_a = [&](int j) {
    if constexpr (!CHAN || (MADE && !DELTA)) return zero4;
    else if constexpr (MADE) return *reinterpret_cast<const f32x4*>(src.w + t * src.ldw + h * D + 16 * j + 4 * g);
    else return *reinterpret_cast<const f32x4*>(decay + (t * H + h) * D + 16 * j + 4 * g);
  };
  f32x4 qf[D / 16], kf[D / 16], af[D / 16];
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    qf[j] = load_q(j);
    kf[j] = load_k(j);
    af[j] = load_a(j);
  }
  const float rate = MADE && DELTA ? -expf(src.A_log[h]) : 0.0f;
  auto decays = [&](int j, f32x4 a) {  // tile j of the decays (past the end: 1)
    if constexpr (MADE) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(src.b + h * D + 16 * j + 4 * g);
      if constexpr (!DELTA) {
        // (the product, dims by tokens, has them where the loads have theirs: row 4 g + r is dim 16 j + 4 g + r, column i the token; of
        // each 16 of the rank a lane brings 4 g .. 4 g + 3)
        for (int k0 = 0; k0 < src.ldw; k0 += 16) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(src.P + t * src.ldp + src.p_off + k0 + 4 * g);
          const f32x4 w = *reinterpret_cast<const f32x4*>(src.w + (int64_t)(h * D + 16 * j + i) * src.ldw + k0 + 4 * g);
#pragma unroll
          for (int r = 0; r < 4; ++r) a = mfma4(w[r], x[r], a);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        a[r] = DELTA ? expf(rate * softplusf_(a[r] + b[r])) : expf(logsigmoidf_(a[r] + b[r]) * src.inv_tau);
    }
    return valid ? a : f32x4{1.f, 1.f, 1.f, 1.f};
  };
  float gi = CHAN || !valid ? 1.0f : decay[t * dstride + h];
  const float bi = !DELTA || !valid ? 0.0f : MADE ? sigmoidf_(src.P[t * src.ldp + src.p_off + h]) : beta[t * H + h];
  float* M = ws + ((int64_t)s * H + h) * rec_floats(D, CHAN, DELTA);
  // accumulators: row 4 g + r (token i), column lane % 16 (token j)
  f32x4 qs[8], ks[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) qs[r] = ks[r] = zero4;
  f32x4 gam = {1.f, 1.f, 1.f, 1.f};
  if (CHAN) {
    // Tile by tile, so that what is loaded is what takes registers: the scan's operands P Q and P K as they are here and (decays after a
    // token) K with tokens and dims exchanged, and the products for chunks whose prefix products all stay near one
    bool near = true;
    float* op = M + MN;
#pragma unroll
    for (int j = 0; j < D / 16; ++j) {
      const f32x4 a = decays(j, af[j]);
      f32x4 P, ki;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        P[r] = row_scan(a[r]);
        near = near && P[r] >= 1.0f / FAR && P[r] <= FAR;
        ki[r] = kf[j][r] / P[r];
      }
      if (i == CT - 1) *reinterpret_cast<f32x4*>(op + 16 * j + 4 * g) = P;
      const f32x4 pq = qf[j] * P, pk = kf[j] * P;
      *reinterpret_cast<f32x4*>(op + D + j * 256 + lane * 4) = pq * q_scale;
      if (DELTA) *reinterpret_cast<f32x4*>(op + D + 2 * CT * D + j * 256 + lane * 4) = pk;
      f32x4 gk;
#pragma unroll
      for (int r = 0; r < 4; ++r) gk[r] = kf[j][r] * row_after(a[r]);
      *reinterpret_cast<f32x4*>(&sT[CHAN ? j & 1 : 0][CHAN ? i : 0][4 * g]) = gk;  // (one wave: its LDS accesses keep their order)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        qs[r + 4 * (j & 1)] = mfma4(pq[r], ki[r], qs[r + 4 * (j & 1)]);
        if (DELTA) ks[r + 4 * (j & 1)] = mfma4(pk[r], ki[r], ks[r + 4 * (j & 1)]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) gk[r] = sT[CHAN ? j & 1 : 0][CHAN ? 4 * g + r : 0][i];
      *reinterpret_cast<f32x4*>(op + D + CT * D + j * 256 + lane * 4) = gk;
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!__all(near)) {
      // row by row: kh_j = k_j times the decays after j, multiplied on token by token (from memory again)
#pragma unroll
      for (int r = 0; r < 8; ++r) qs[r] = ks[r] = zero4;
      for (int j = 0; j < D / 16; ++j) {
        const f32x4 qj = load_q(j), kj = load_k(j), a = decays(j, load_a(j));
        f32x4 kh = zero4;
        for (int row = 0; row < CT; ++row) {
          const int from = (lane & 48) + row;
          float dq = 0.0f, dk = 0.0f;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float ar = __shfl(a[r], from), qr = __shfl(qj[r], from), kr = __shfl(kj[r], from);
            kh[r] = i == row ? kj[r] : i < row ? kh[r] * ar : 0.0f;
            dq += qr * kh[r];
            if (DELTA) dk += kr * kh[r];
          }
          dq = xor_sum<16>(dq);
          dq = xor_sum<32>(dq);
          dk = xor_sum<16>(dk);
          dk = xor_sum<32>(dk);
          if ((row >> 2) == g) {
            qs[0][0] += (row & 3) == 0 ? dq : 0.0f, ks[0][0] += (row & 3) == 0 ? dk : 0.0f;
            qs[0][1] += (row & 3) == 1 ? dq : 0.0f, ks[0][1] += (row & 3) == 1 ? dk : 0.0f;
            qs[0][2] += (row & 3) == 2 ? dq : 0.0f, ks[0][2] += (row & 3) == 2 ? dk : 0.0f;
            qs[0][3] += (row & 3) == 3 ? dq : 0.0f, ks[0][3] += (row & 3) == 3 ? dk : 0.0f;
          }
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
  }
  const f32x4 qk = ((qs[0] + qs[1]) + (qs[2] + qs[3])) + ((qs[4] + qs[5]) + (qs[6] + qs[7]));
  const f32x4 kk = ((ks[0] + ks[1]) + (ks[2] + ks[3])) + ((ks[4] + ks[5]) + (ks[6] + ks[7]));
  for (int e = 0;; ++e) {
    float gn = 1.0f;  // (the next head's, in flight under this one's)
    if (SHARE && e + 1 < heads) gn = valid ? decay[t * dstride + h + e + 1] : 1.0f;
    if (!CHAN) {
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
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 4 * g + r;
      const float br = __shfl(bi, row);
      M[CT * CT + row * CT + i] = row >= i ? qk[r] * gam[r] * q_scale : 0.0f;
      if (DELTA) sA[row][i] = row > i ? kk[r] * gam[r] * br : 0.0f;
    }
    if (DELTA) {
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
    if (!SHARE || e + 1 >= heads) return;
    M += rec_floats(D, CHAN, DELTA);
    gi = gn;
  }
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

// CG groups of 16 value channels a workgroup, KP waves each: wave (kp, cg) has key dims kp D / KP .. of group cg.  Of every sequence
// the chunks whose records the workspace holds (Portions): `each` from its chunk `from` on, or those in `slots` slots from slot `from` of
// the step, but the first `done` of each; between portions the state is in its place in memory.
template <int D, bool CHAN, bool DELTA, int KP, int CG, int WPE, int RING>
__global__ __launch_bounds__(64 * KP * CG, WPE) void chunk_scan_k(
    const float* __restrict__ q, int ldq, const float* __restrict__ k, int ldk, const float* __restrict__ v, int ldv,
    const float* __restrict__ inscale, float q_scale, float* __restrict__ state, const int* __restrict__ state_slots,
    const int* __restrict__ cu_q, int B, int H, int G, int dv, int dvin, int from, int slots, int each, int done,
    const float* __restrict__ ws, float* __restrict__ out) {
  static_assert(KP == 2 || KP == 4, "the order of the sums is that of quarters of the key dims");
  constexpr int TILES = D / 16 / KP;              // 16-row state tiles of a wave
  constexpr int QW = 4 / KP, QT = TILES / QW;     // quarters of the key dims in a wave, tiles of each
  constexpr int REC = rec_floats(D, CHAN, DELTA);
  // the write's operand, k with tokens and dims exchanged: from the workspace (channel decays), from the rows of k that the delta
  // rule's product has through LDS, or element by element (16 heads of 128 x 128, 8 of 961 .. 2433 tokens: delta rule 312 us
  // element by element and 298 through LDS; plain write 247 and 304, where those rows are no operand otherwise)
  constexpr bool TURN = DELTA && !CHAN, SINGLE = !DELTA && !CHAN;
  constexpr int LT = D / KP + 4;                  // LDS row of a wave's k: consecutive tokens four banks apart
  __shared__ __attribute__((aligned(16))) float sk[TURN ? KP * CG : 1][TURN ? CT * LT : 1];
  __shared__ f32x4 sx[DELTA ? 2 : 1][CG][DELTA ? KP : 1][64];  // partial products of the waves of a group
  __shared__ f32x4 sy[2][CG][KP][64];
  const int h = blockIdx.x;
  const int b = nth_longest(B, scan_order((int)blockIdx.z, B, H * (int)gridDim.y), [&](int j) { return cu_q[j + 1] - cu_q[j]; });
  const int slot = state_slots[b];
  const int base = slot_base(cu_q, b) - from;  // the sequence's first slot in the portion, or (negative) before it
  const int c0 = each ? from : max(-base, done), first = each ? b * each : base + c0;
  const int t0 = cu_q[b] + CT * c0, n = min(cu_q[b + 1] - t0, CT * (each ? each : slots - first));
  if (slot < 0 || n <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cg = wave % CG, kp = wave / CG;
  const int col = ((int)blockIdx.y * CG + cg) * 16 + i;
  const bool live = col < dv;
  const int hk = h / (H / G);
  const int d0 = kp * (D / KP);                   // the wave's first key dim
  float* St = state + (((int64_t)slot * H + h) * dv + (live ? col : 0)) * D + d0 + 4 * g;
  f32x4 S[TILES];
#pragma unroll
  for (int j = 0; j < TILES; ++j) S[j] = *reinterpret_cast<const f32x4*>(St + 16 * j);
  const float* W = ws + ((int64_t)first * H + h) * REC;
  const int64_t wstep = (int64_t)H * REC;

  // What a chunk is made of, two chunks ahead in registers: q, k (channel decays: P Q, P K from the workspace) as A operands of the
  // products with the state, (channel decays) (G K)^T for the write, and value rows, M, N and decays.
  // Every load goes through a buffer that ends with the sequence: its base moves in scalar registers and a lane's offset never
  // changes, so a chunk's loads cost the vector unit nothing; rows past the end give zeros, which leave the state as it is.
  struct Ops {
    f32x4 q[TILES], k[DELTA ? TILES : 1], t[TURN ? 1 : TILES], d[CHAN ? TILES : 1];
    f32x4 v, m, nn, p, e;
    float all;
  };
  const int chunks = (n + CT - 1) / CT;
  // A lane's place in the rows moves on by a chunk with every load; the windows end with the sequence, its state records with its chunks
  const __amdgpu_buffer_rsrc_t rq = window(q + (int64_t)t0 * ldq + hk * D, ((int64_t)(n - 1) * ldq + D) * 4),
                               rk = window(k + (int64_t)t0 * ldk + hk * D, ((int64_t)(n - 1) * ldk + D) * 4),
                               rv = window(v + (int64_t)t0 * ldv + h * dvin, ((int64_t)(n - 1) * ldv + dvin) * 4),
                               rb = window(inscale + (int64_t)t0 * H + h, inscale ? ((int64_t)(n - 1) * H + 1) * 4 : 0),
                               ro = window(out + ((int64_t)t0 * H + h) * dv, ((int64_t)(n - 1) * H * dv + dv) * 4);
  const int vcol = min(col, dvin - 1);
  uint32_t oq = (i * ldq + d0 + 4 * g) * 4, ok = (i * ldk + d0 + 4 * g) * 4, ot[4], ov[4], ob[4], oo[4];
  uint32_t om = (i * CT + 4 * g) * 4, od = (CHAN ? MN + d0 + 4 * g : 2 * CT * CT + 4 * g) * 4;
  uint32_t oc = (MN + D + kp * TILES * 256 + lane * 4) * 4;  // channel decays: P Q; (G K)^T and P K follow
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    ot[r] = ((4 * g + r) * ldk + d0 + i) * 4;
    ov[r] = ((4 * g + r) * ldv + vcol) * 4;
    ob[r] = (4 * g + r) * H * 4;
    // (a chunk's rows are stored in the next one's turn.  What is before the first chunk, channels past the end and the waves that do
    // not have the sum: past every window)
    oo[r] = live && kp == 0 ? (uint32_t)(((4 * g + r - CT) * H * dv + col) * 4) : 0x80000000u;
    asm volatile("" : "+v"(ot[r]), "+v"(ov[r]), "+v"(oo[r]));
  }
  asm volatile("" : "+v"(oq), "+v"(ok), "+v"(om), "+v"(od), "+v"(oc));  // (constants added to them are then the loads' own)
  const uint32_t ostep = live && kp == 0 ? CT * H * dv * 4 : 0;  // (the places past every window stay there)
  const float *Wq = W, *Wr = W;  // the records of the next loads
  int cq = 0, cr = 0;            // their chunks
  auto record = [&](const float* w, int c) { return window(w, c < chunks ? REC * 4 : 0); };
  // load s of a chunk's operands of the products with the state, then a step to the next chunk
  auto load_q = [&](__amdgpu_buffer_rsrc_t w, Ops& o, int j) {
    if (j < TILES) o.q[j] = CHAN ? load4(w, oc + 1024 * j) : load4(rq, oq + 64 * j);
  };
  auto load_k = [&](__amdgpu_buffer_rsrc_t w, Ops& o, int j) {
    if (DELTA && j < TILES) o.k[DELTA ? j : 0] = CHAN ? load4(w, oc + (8 * CT * D + 1024 * j)) : load4(rk, ok + 64 * j);
  };
  auto next_state = [&]() {
    ++cq;
    if (CHAN) {
      Wq += wstep;
    } else {
      oq += CT * ldq * 4;
      ok += CT * ldk * 4;
    }
  };
  // the rest of a chunk, NR loads
  constexpr int NF = CHAN ? 2 * TILES : SINGLE ? 3 + 4 * TILES : 3, NR = NF + 1 + 4 + (DELTA ? 1 : 4);
  auto load_rest = [&](__amdgpu_buffer_rsrc_t w, Ops& o, int s) {
    if (s < 4) {
      o.v[s & 3] = load1(rv, ov[s & 3]);
    } else if (s == 4) {
      o.nn = load4(w, om + CT * CT * 4);
    } else if (DELTA && s == 5) {
      o.m = load4(w, om);
    } else if (!DELTA && s < 9) {
      o.m[(s - 5) & 3] = load1(rb, ob[(s - 5) & 3]);
    } else if (s < NR) {
      const int f = s - (NR - NF);
      if constexpr (CHAN) {
        if (f < TILES) o.d[CHAN ? f : 0] = load4(w, od + 64 * f);
        else o.t[f % TILES] = load4(w, oc + (4 * CT * D + 1024 * (f % TILES)));
      } else {
        if (f == 0) o.all = load1(w, (2 * CT * CT + CT - 1) * 4);
        else if (f == 1) o.p = load4(w, od);
        else if (f == 2) o.e = load4(w, od + CT * 4);
        else if constexpr (SINGLE) o.t[(f - 3) % TILES][(f - 3) / TILES] = load1(rk, ot[(f - 3) / TILES] + 64 * ((f - 3) % TILES));
      }
    }
  };
  auto next_rest = [&]() {
    ++cr;
    Wr += wstep;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ov[r] += CT * ldv * 4;
      if (SINGLE) ot[r] += CT * ldk * 4;
      if (!DELTA) ob[r] += CT * H * 4;
    }
  };
  auto store = [&](f32x4 Y) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(Y[r]), ro, oo[r], 0, 0);
      oo[r] += ostep;
    }
  };
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
    float odd = 0.0f * b[0];
#pragma unroll
    for (int r = 1; r < 4; ++r) odd = __builtin_fmaf(0.0f, b[r], odd);
    if (__builtin_expect(__any(odd != odd), 0)) {
      int at = lane;
      asm volatile("" : "+v"(at));  // (or its addresses are kept in registers through the whole scan)
      const int ai = at & 15, ag = 4 * (at >> 4);
      for (int mm = 0; mm < CT; mm += 4)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const float bm = __shfl(b[m], mm * 4 + ai);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float lm = __shfl(l[m], mm * 4 + ag + r);
            c[r] = mm + m <= ag + r ? c[r] + lm * bm : c[r];
          }
        }
      return c;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) c = mfma4(l[r], b[r], c);
    return c;
  };
  Ops ops[RING];
#pragma unroll
  for (int u = 0; u < RING; ++u) {
    const __amdgpu_buffer_rsrc_t wq = record(Wq, cq), wr = record(Wr, cr);
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      load_k(wq, ops[u], j);
      load_q(wq, ops[u], j);
    }
    next_state();
    if (u == RING - 1) break;
#pragma unroll
    for (int j = 0; j < NR; ++j) load_rest(wr, ops[u], j);
    next_rest();
  }
  // Products with the state are summed by quarters of the key dims, these in pairs, whichever waves hold them: a sequence's numbers do
  // not depend on the form of the scan, which the step's other sequences have a part in, and are the same in all waves of a group.
  auto pairs = [&](f32x4 mine, const f32x4 (&other)[KP - 1]) {
    if constexpr (KP == 2) return mine + other[0];
    else return (mine + other[0]) + (other[1] + other[2]);
  };
  f32x4 last = {0.f, 0.f, 0.f, 0.f};  // the chunk before: N U (kp 0); the waves' parts of P Q S are in LDS
  auto parts = [&](int buf) {
    f32x4 other[KP - 1];
#pragma unroll
    for (int w = 1; w < KP; ++w) other[w - 1] = sy[buf][cg][kp ^ w][lane];
    return last + pairs(sy[buf][cg][kp][lane], other);
  };
  // Loads and stores between the MFMAs, which hold the matrix unit 32 cycles each: behind them they were on the chain
  auto pin = [&]() { __builtin_amdgcn_sched_barrier(0x86); };  // (vector, scalar and LDS operations may pass)
  auto chunk = [&](int c, int buf, Ops& o, Ops& before) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 xs[2], ys[2], X, mine;  // (partial sums: shorter chains, and sums of fewer terms)
    const __amdgpu_buffer_rsrc_t wq = record(Wq, cq), wr = record(Wr, cr);
    int s = 0;
    float* kt = &sk[TURN ? wave : 0][0];
    if constexpr (TURN) {  // (the wave's own: no barrier)
#pragma unroll
      for (int j = 0; j < TILES; ++j) *reinterpret_cast<f32x4*>(kt + i * LT + 16 * j + 4 * g) = o.k[DELTA ? j : 0];
    }
    if constexpr (DELTA) {
#pragma unroll
      for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          xs[r & 1] = mfma4(o.k[DELTA ? j : 0][r], S[j][r], r < 2 && j % QT == 0 ? zero : xs[r & 1]);
          load_rest(wr, before, s++);
          load_rest(wr, before, s++);
          pin();
          if (r == 3 && j % QT == QT - 1) X = j < QT ? xs[0] + xs[1] : X + (xs[0] + xs[1]);
        }
      sx[DELTA ? buf : 0][cg][DELTA ? kp : 0][lane] = X;
    }
    bar();
    f32x4 xo[KP - 1];
    if constexpr (DELTA) {
#pragma unroll
      for (int w = 1; w < KP; ++w) xo[w - 1] = sx[DELTA ? buf : 0][cg][DELTA ? kp ^ w : 0][lane];
    }
    const f32x4 y = parts(buf ^ 1);
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ys[r & 1] = mfma4(o.q[j][r], S[j][r], r < 2 && j % QT == 0 ? zero : ys[r & 1]);
        if (r == 0) load_k(wq, o, j);
        if constexpr (DELTA) {
          load_rest(wr, before, s++);
        } else {
          load_rest(wr, before, s++);
          load_rest(wr, before, s++);
        }
        pin();
        if (r == 3 && j % QT == QT - 1) {
          f32x4 part = ys[0] + ys[1];
          if (!CHAN) part = times(part, o.p * q_scale);
          mine = j < QT ? part : mine + part;
        }
      }
#pragma unroll
    for (; s < NR; ++s) load_rest(wr, before, s);
    next_rest();
    store(y);
    // the decayed state meets the chunk's write after the products that read it
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const f32x4 p = CHAN ? o.d[CHAN ? j : 0] : f32x4{o.all, o.all, o.all, o.all};
#pragma unroll
      for (int r = 0; r < 4; ++r) S[j][r] *= p[r];
    }
    f32x4 U;  // the value rows; the normaliser's channel is fed with ones (past the end k is 0: no such row reaches anything)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      U[r] = DELTA || col < dvin ? o.v[r] : 1.0f;
      if (!DELTA) U[r] *= inscale ? o.m[r] : 1.0f;
    }
    if constexpr (DELTA) {
      X = pairs(X, xo);
      f32x4 R;
#pragma unroll
      for (int r = 0; r < 4; ++r) R[r] = U[r] - (CHAN ? X[r] : o.p[r] * X[r]);
      U = lower(o.m, R, zero);
    }
    f32x4 E = U;
    if (!CHAN) {
#pragma unroll
      for (int r = 0; r < 4; ++r) E[r] *= o.e[r];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < TILES; ++j) {
        S[j] = mfma4(TURN ? kt[(4 * g + r) * LT + 16 * j + i] : o.t[TURN ? 0 : j][r], E[r], S[j]);
        if (r == 0) load_q(wq, o, j);
        pin();
      }
    next_state();
    sy[buf][cg][kp][lane] = mine;
    if (kp == 0) last = lower(o.nn, U, zero);
  };
  // (ends left where the chunks end, none joined again: at a join the compiler waits for every load that one of the paths may have
  // issued last, and a copy of the loop's body for the rest keeps a second set of operands in registers)
  for (int c = 0;; c += RING) {
    bool end = false;
#pragma unroll
    for (int u = 0; u < RING; ++u) {
      chunk(c + u, (c + u) & 1, ops[u], ops[(u + RING - 1) % RING]);
      end = c + u + 1 >= chunks;
      if (end) break;
    }
    if (end) break;
  }
  bar();
  store(parts((chunks - 1) & 1));
  if (live) {
#pragma unroll
    for (int j = 0; j < TILES; ++j) *reinterpret_cast<f32x4*>(St + 16 * j) = S[j];
  }
}

template <int D, bool CHAN, bool DELTA, int KP, int CG, int WPE, int RING>
void scan(const ChunkRecurrence& a, int from, int slots, int each, int done) {
  const dim3 grid((unsigned)a.H, (unsigned)((a.dv + 16 * CG - 1) / (16 * CG)), (unsigned)a.B);
  chunk_scan_k<D, CHAN, DELTA, KP, CG, WPE, RING><<<grid, 64 * KP * CG, 0, stream()>>>(
      a.q, a.ldq, a.k, a.ldk, a.v, a.ldv, DELTA ? nullptr : a.beta, a.q_scale, a.state, a.state_slots, a.cu_q, a.B, a.H, a.G, a.dv,
      a.dvin, from, slots, each, done, a.ws, a.out);
}

// a portion
template <int D, bool CHAN, bool DELTA>
void go(const ChunkRecurrence& a, int from, int slots, int each, int done) {
  // plain write, a decay per head: the heads of a q / k head share its products where that leaves enough waves (32 heads on 8, with the
  // scan: 5 of 364 .. 1728 tokens 110 -> 100 us, 8 of 961 .. 2433 247 -> 223; three of 1000 not; two heads under the delta rule gave nothing)
  const int heads = !CHAN && !DELTA && (int64_t)slots * a.G >= 2048 ? a.H / a.G : 1;
  const unsigned pg = (unsigned)slots * (unsigned)(a.H / heads);
  auto prep = [&](auto kern) {
    kern<<<pg, 64, 0, stream()>>>(a.q, a.ldq, a.k, a.ldk, a.decay, a.dstride, a.beta, a.q_scale, a.state_slots, a.cu_q, a.B, a.H, a.G,
                                  heads, a.src, from, each, done, a.ws);
  };
  if constexpr (CHAN) {
    if (a.src.P != nullptr) prep(chunk_prep_k<D, CHAN, DELTA, true>);
    else prep(chunk_prep_k<D, CHAN, DELTA, false>);
  } else {
    prep(chunk_prep_k<D, CHAN, DELTA, false>);
  }
  // Steps whose longest sequence takes longer than the CUs' share of all chunks are bound by its chain: four waves of a quarter of the
  // key dims each, 16 channels a workgroup, three chunks ahead.  Others by the matrix unit: two halves and 32 channels, which
  // repeat the products with M and N less.  The line by tokens x workgroups of 32 channels a sequence / (256 x the longest), us
  // quarters / halves, delta rule 16 heads of 128 x 128: 0.25 (one of 2000) 130 / 167, 0.5 77 / 93, 0.66 (5 of 364 .. 1728) 149 / 164,
  // 0.75 (three of 1000) 111 / 98, 1.3 (8 of 961 .. 2433) 332 / 298.  A sequence's state, first loads and end cost its workgroups
  // what 40 tokens do: one of 570 behind 64 single tokens 102 / 84 (0.4 by its tokens alone), behind 8 49 / 60, 16 heads of 64 x 128 with one
  // decay each behind 233 190 / 99.
  const int64_t per = (int64_t)a.H * ((a.dv + 31) / 32);
  const int64_t tokens = std::min<int64_t>(a.T, (int64_t)CT * slots) + 40 * (int64_t)a.B;
  const int64_t longest = std::min<int64_t>(a.longest, (int64_t)CT * (each ? each : slots));
  if (tokens * per < 180 * longest) scan<D, CHAN, DELTA, 4, 1, 2, 3>(a, from, slots, each, done);
  else if (a.B * per <= 512 || !DELTA) scan<D, CHAN, DELTA, 2, 2, 2, 2>(a, from, slots, each, done);
  // (four waves a SIMD: 12 of 130 tokens 51.7 -> 49.1 us; with channel decays at key dims of 128 four registers are in scratch memory)
  else if constexpr (DELTA) scan<D, CHAN, DELTA, 2, 2, 4, 1>(a, from, slots, each, done);
}

template <int D, bool CHAN, bool DELTA>
void go(const ChunkRecurrence& a) {
  const Portions p = portions(a.T, a.B, a.H, rec_floats(D, CHAN, DELTA), a.known ? a.longest : 0);
  for (int turn = 0; turn < p.count; ++turn) go<D, CHAN, DELTA>(a, turn * (p.each ? p.each : p.slots), p.slots, p.each, 0);
  const int done = p.count * p.each;  // chunks of every sequence
  if (done == 0 || (int64_t)CT * done >= a.T) return;
  // what is left of sequences longer than the longest was said to be, as slots come (nothing: workgroups that end at once)
  const Portions rest = portions(a.T, a.B, a.H, rec_floats(D, CHAN, DELTA), 0);
  for (int turn = 0; turn < rest.count; ++turn) go<D, CHAN, DELTA>(a, turn * rest.slots, rest.slots, 0, done);
}

}  // namespace

int64_t chunk_recurrence_ws(int64_t T, int64_t B, int64_t H, int64_t d, bool chan, bool delta, int64_t max_qlen) {
  const int rec = rec_floats((int)d, chan, delta);
  const Portions p = portions(T, B, H, rec, max_qlen), rest = p.each ? portions(T, B, H, rec, 0) : p;
  return std::max(p.slots, rest.slots) * H * rec;
}

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
