// Decode GEMM whose workgroups own their output columns for the whole of K:  Y[M, N] = X[M, K] . W[N, K]^T, M <= 16, on the
// pre-shuffled layout ([N/16][K/32] blocks of 16 rows x 32 k, 1 KB).
//
// gemm_stream puts 64 or more columns on a workgroup's four waves, so a projection of a few thousand columns needs K split
// over workgroups to cover the 256 CUs: fp32 slabs and a second launch of 4.5 to 6 us to add them, whatever their size.  Here
// eight waves split K among themselves over 16, 32 or 64 columns: every wave streams its own 1-KB weight blocks (two stages of
// eight in flight) and the matching k columns of X, and the eight partial tiles meet in LDS.  So the epilogue has the whole
// sum -- bias, residual, gated pairs, or RoPE and the paged KV write (ROPE: a workgroup's two column tiles are the rotation
// partners i and i + Dh/2 of one head) -- and the second launch is gone.
// Cold-cache us, best split of gemm_stream with its reduce -> here, 1 / 6 rows: 3072 x 2048 10.4 -> 7.8 / 10.3 -> 8.4,
// 16384 x 2048 SiLU 20.5 -> 17.3 / 21.0 -> 18.3, 2048 x 5632 15.5 -> 10.3 / 15.6 -> 12.0; bound by the ramp of one wave's
// loads and the LDS exchange at these sizes (2 - 4 TB/s), by the loads of X beyond: every workgroup reads all of it, and from 24
// rows on the split wins again (4096 x 14336 at 24 rows 28.0 -> 38.7), which is why one row tile is all there is.  Shapes
// with columns enough for one pass of gemm_stream stay there, too (28672 x 4096 42 against 48): ops.linear times both.
// NORM (batch-1 decode): the input row is rmsnorm(residual + the previous projection's slabs), computed by the first
// four waves in splitk_resid_rmsnorm's order while all eight have their first weight blocks in flight.
#include "common.h"
#include "gemm_common.h"
#include "kernels.h"

namespace xot {
namespace {

constexpr int KW = 8, NTH = 64 * KW;  // waves of a workgroup, splitting K

__device__ __forceinline__ s16x8 buf16(__amdgpu_buffer_rsrc_t r, int voff, int soff, bool nt) {
  return __builtin_bit_cast(s16x8, nt ? __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 2)
                                      : __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

template <int NT, int EPI, bool F32, int NORM, int SM, bool ROPE>
__global__ __launch_bounds__(NTH) void gemm_wave_kernel(const uint16_t* __restrict__ X, int ldx,
                                                        const uint16_t* __restrict__ W, const uint16_t* __restrict__ bias,
                                                        const uint16_t* __restrict__ R, int ldr, void* __restrict__ Yv, int ldy,
                                                        int M, int K, float epi_arg, NormPro np, RopeOut ro) {
  static_assert(!ROPE || NT == 2, "a rotation pair of column tiles");
  static_assert(!epi_is_glu(EPI) || NT % 2 == 0, "gate / up tile pairs");
  constexpr int U = 8 / NT;  // k blocks a stage
  extern __shared__ __attribute__((aligned(16))) char smem[];
  f32x4(*red)[NT][64] = reinterpret_cast<f32x4(*)[NT][64]>(smem);                      // [KW]
  uint16_t* x1 = reinterpret_cast<uint16_t*>(smem + sizeof(f32x4) * KW * NT * 64);     // NORM: the row [K]
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = K >> 5, b0 = wave * nb / KW, b1 = (wave + 1) * nb / KW;

  int tile[NT];  // 16-row groups of W
  int head = 0, ra = 0;
  if constexpr (ROPE) {
    const int per = ro.Dh >> 5;
    head = blockIdx.x / per;
    ra = (blockIdx.x - head * per) * 16;
    tile[0] = (head * ro.Dh + ra) >> 4;
    tile[1] = tile[0] + (ro.Dh >> 5);
  } else {
#pragma unroll
    for (int j = 0; j < NT; ++j) tile[j] = blockIdx.x * NT + j;
  }
  __amdgpu_buffer_rsrc_t wr[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wr[j] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(W + (size_t)tile[j] * nb * 512), (short)0, nb * 1024, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X), (short)0, -1, 0x00020000);
  const int xo = (min(c, M - 1) * ldx + 8 * g) * 2;  // the lane's row (past M the last again; not written)

  struct Stage {
    s16x8 w[U][NT], x[NORM ? 1 : U];
  };
  auto load = [&](Stage& s, int it) {  // k blocks b0 + it U .. (past the wave's range: its last block again, not used)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int b = max(min(b0 + it * U + u, b1 - 1), 0);
#pragma unroll
      for (int j = 0; j < NT; ++j) s.w[u][j] = buf16(wr[j], lane * 16, b * 1024, true);
      if constexpr (!NORM) s.x[u] = buf16(xr, xo, b * 64, false);
    }
  };
  f32x4 acc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto one = [&](const Stage& s, int it, int u) {
    s16x8 a;
    if constexpr (NORM) a = ld16(x1 + (b0 + it * U + u) * 32 + 8 * g);  // (every MFMA row the same: row 0 is written)
    else a = s.x[u];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = mfma16(a, s.w[u][j], acc[j]);
  };
  auto whole = [&](const Stage& s, int it) {
#pragma unroll
    for (int u = 0; u < U; ++u) one(s, it, u);
  };
  auto part = [&](const Stage& s, int it) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (b0 + it * U + u < b1) one(s, it, u);
  };
  Stage sa, sb;
  s16x8 ha[NORM ? NORM : 1], la[NORM ? NORM : 1];
  f32x4 p[NORM ? NORM : 1][NORM ? SM : 1][2];
  const int nchunk = np.D >> 3;
  // SM slabs from s0 on of the thread's chunks (past the last: the last again, not added)
  auto slabs = [&](int s0) {
#pragma unroll
    for (int i = 0; i < (NORM ? NORM : 0); ++i)
#pragma unroll
      for (int sl = 0; sl < SM; ++sl) {
        const float* sp = np.ws + min(s0 + sl, np.S - 1) * np.sstride + min((tid & 255) + 256 * i, nchunk - 1) * 8;
        p[i][sl][0] = *reinterpret_cast<const f32x4*>(sp);
        p[i][sl][1] = *reinterpret_cast<const f32x4*>(sp + 4);
      }
  };
  if constexpr (NORM > 0) {  // (asked for before the weights: loads return in order, and the row's chain is the longer one)
#pragma unroll
    for (int i = 0; i < NORM; ++i) {
      const int cc = min((tid & 255) + 256 * i, nchunk - 1);
      ha[i] = ld16(np.h + cc * 8);
      la[i] = ld16(np.lnw + cc * 8);
    }
    if (np.S > 0) slabs(0);
    __builtin_amdgcn_sched_barrier(0);
  }
  load(sa, 0);
  load(sb, 1);
  if constexpr (NORM > 0) {
    __builtin_amdgcn_sched_barrier(0);
    // one row: residual + bias + slabs -> bf16 residual (stored by workgroup 0), its RMS norm times the weight -> x1.  256
    // threads, 8 consecutive elements each per round, in the order of splitk_resid_rmsnorm_kernel<*, *, 256>
    __shared__ float nred[4];
    if (wave < 4) {
      float v[NORM][8], ss = 0.f;
#pragma unroll
      for (int i = 0; i < NORM; ++i) {
        const int cc = tid + 256 * i;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = bf2f(ha[i][e]);
        if (np.bias != nullptr && cc < nchunk) {
          const s16x8 ba = ld16(np.bias + cc * 8);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[i][e] += bf2f(ba[e]);
        }
      }
      for (int s0 = 0; s0 < np.S; s0 += SM) {
        if (s0 > 0) slabs(s0);
#pragma unroll
        for (int i = 0; i < NORM; ++i)
#pragma unroll
          for (int sl = 0; sl < SM; ++sl)
            if (s0 + sl < np.S) {
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                v[i][e] += p[i][sl][0][e];
                v[i][4 + e] += p[i][sl][1][e];
              }
            }
      }
#pragma unroll
      for (int i = 0; i < NORM; ++i) {
        const int cc = tid + 256 * i;
        if (cc >= nchunk) continue;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          ha[i][e] = (short)f2bf(v[i][e]);
          const float r = bf2f(ha[i][e]);
          ss += r * r;
        }
        if (blockIdx.x == 0) st16(np.hout + cc * 8, ha[i]);
      }
      ss = wave_sum(ss);
      if (lane == 0) nred[wave] = ss;
    }
    __syncthreads();
    if (wave < 4) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) ss += nred[k];
      const float inv = rsqrtf(ss / (float)np.D + np.eps);
#pragma unroll
      for (int i = 0; i < NORM; ++i) {
        const int cc = tid + 256 * i;
        if (cc >= nchunk) continue;
        s16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (short)f2bf(bf2f(ha[i][e]) * inv * bf2f(la[i][e]));
        st16(x1 + cc * 8, o);
      }
    }
    __syncthreads();
  }
  {
    const int nfull = (b1 - b0) / U, nit = (b1 - b0 + U - 1) / U;
    int it = 0;
    for (; it + 2 <= nfull; it += 2) {
      whole(sa, it);
      load(sa, it + 2);
      whole(sb, it + 1);
      load(sb, it + 3);
    }
    if (it < nit) part(sa, it);
    if (it + 1 < nit) part(sb, it + 1);
  }
#pragma unroll
  for (int j = 0; j < NT; ++j) red[wave][j][lane] = acc[j];
  __syncthreads();

  // the waves' partial tiles in wave order; lane (g, c) of tile j: tokens 4 g + r, column c of the tile
  auto total = [&](int t, int l) {
    f32x4 v = red[0][t][l];
#pragma unroll
    for (int w = 1; w < KW; ++w) v += red[w][t][l];
    return v;
  };
  auto put = [&](int m, int col, float v) {
    if constexpr (F32) reinterpret_cast<float*>(Yv)[(size_t)m * ldy + col] = v;
    else reinterpret_cast<uint16_t*>(Yv)[(size_t)m * ldy + col] = f2bf(v);
  };
  if constexpr (ROPE) {
    const int half = ro.Dh >> 1;
    if (tid < 64) {
      const int l = tid, d = ra + (l & 15);
      f32x4 lo = total(0, l), hi = total(1, l);
      if (bias != nullptr) {
        lo += bf2f(bias[head * ro.Dh + d]);
        hi += bf2f(bias[head * ro.Dh + half + d]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 4 * (l >> 4) + r;
        if (m >= M) continue;
        const int64_t slot = ro.slots[m] < ro.nslots ? ro.slots[m] : -1;
        const int64_t page = slot >= 0 ? slot / ro.BS : 0;
        const int off = slot >= 0 ? (int)(slot % ro.BS) : 0;
        if (head >= ro.H + ro.Hkv) {
          if (slot < 0) continue;
          uint16_t* dst = ro.vc + ((size_t)page * ro.Hkv + (head - ro.H - ro.Hkv)) * ro.Dh * ro.BS;
          dst[v_page_off(off, d, ro.Dh)] = f2bf(lo[r]);
          dst[v_page_off(off, half + d, ro.Dh)] = f2bf(hi[r]);
          continue;
        }
        uint16_t* dst;
        if (head < ro.H) {
          dst = ro.q + ((size_t)m * ro.H + head) * ro.Dh;
        } else {
          if (slot < 0) continue;
          dst = ro.kc + (((size_t)page * ro.Hkv + (head - ro.H)) * ro.BS + off) * ro.Dh;
        }
        const float* cs = ro.cos_sin + (size_t)min(max(ro.pos[m], 0), ro.max_pos - 1) * ro.Dh;
        dst[d] = f2bf(lo[r] * cs[d] - hi[r] * cs[half + d]);
        dst[half + d] = f2bf(hi[r] * cs[d] + lo[r] * cs[half + d]);
      }
    }
  } else if constexpr (epi_is_glu(EPI)) {
    if (tid < 32 * NT) {
      const int p = tid >> 6, l = tid & 63;
      f32x4 gv = total(2 * p, l), uv = total(2 * p + 1, l);
      const int n = tile[0] * 16 + 32 * p + (l & 15);  // gate row of W; its up row is 16 further
      if (bias != nullptr) {
        gv += bf2f(bias[n]);
        uv += bf2f(bias[n + 16]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 4 * (l >> 4) + r;
        if (m < M) put(m, tile[0] * 8 + 16 * p + (l & 15), glu_pair<EPI>(gv[r], uv[r], epi_arg));
      }
    }
  } else {
    if (tid < 64 * NT) {
      const int t = tid >> 6, l = tid & 63, n = tile[0] * 16 + 16 * t + (l & 15);
      f32x4 v = total(t, l);
      if (bias != nullptr) v += bf2f(bias[n]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 4 * (l >> 4) + r;
        if (m >= M) continue;
        if constexpr (EPI == EPI_RESID) v[r] += bf2f(R[(size_t)m * ldr + n]);
        put(m, n, epi_elem<EPI>(v[r]));
      }
    }
  }
}

template <int NT, int EPI, bool F32, int NORM, int SM, bool ROPE>
void go(const WaveGemm& a, hipStream_t st) {
  const size_t smem = sizeof(f32x4) * KW * NT * 64 + (NORM ? a.K * 2 : 0);  // at most 32 + 16 KB
  gemm_wave_kernel<NT, EPI, F32, NORM, SM, ROPE><<<a.N / (16 * NT), NTH, smem, st>>>(a.X, a.ldx, a.W, a.bias, a.R, a.ldr, a.Y, a.ldy,
                                                                                 a.M, a.K, a.epi_arg, a.np, a.ro);
}

template <int EPI, bool F32, int NORM, int SM>
int columns(const WaveGemm& a, int nt, hipStream_t st) {
  if (nt == 1) {
    if constexpr (epi_is_glu(EPI)) return -1;
    else go<1, EPI, F32, NORM, SM, false>(a, st);
  } else if (nt == 2) {
    go<2, EPI, F32, NORM, SM, false>(a, st);
  } else {
    go<4, EPI, F32, NORM, SM, false>(a, st);
  }
  return 0;
}

template <int NORM, int SM>
int normed(const WaveGemm& a, int epi, int nt, hipStream_t st) {
  if (a.ro.q == nullptr) return epi == EPI_SILU ? columns<EPI_SILU, false, NORM, SM>(a, nt, st) : columns<EPI_NONE, false, NORM, SM>(a, nt, st);
  go<2, EPI_NONE, false, NORM, SM, true>(a, st);
  return 0;
}

}  // namespace

int launch_gemm_wave(const WaveGemm& a, bool out_f32, int epi, int nt, hipStream_t st) {
  if (a.M <= 0) return 0;
  const bool rope = a.ro.q != nullptr, norm = a.np.h != nullptr;
  if (a.M > 16 || a.K % 128 != 0 || a.K <= 0 || (nt != 1 && nt != 2 && nt != 4) || a.N % (16 * nt) != 0) return -1;
  if (!norm && (a.ldx % 8 != 0 || (int64_t)a.M * a.ldx * 2 >= (int64_t(1) << 31))) return -1;
  if (epi_is_glu(epi) && nt == 1) return -1;
  if (rope && (nt != 2 || epi != EPI_NONE || out_f32 || a.ro.Dh % 32 != 0 || a.N != (a.ro.H + 2 * a.ro.Hkv) * a.ro.Dh || a.ro.max_pos < 1)) return -1;
  if (norm) {
    if (a.M != 1 || out_f32 || (epi != EPI_NONE && epi != EPI_SILU) || a.np.D != a.K || a.K > 8192 || a.np.S < 0 ||
        a.np.lnw == nullptr || a.np.hout == nullptr || (a.np.S > 0 && (a.np.ws == nullptr || a.np.sstride < a.K)))
      return -1;
    // (slabs of the first round trip: 8 where the row is short, or they would keep a second workgroup off the CU)
    if (a.K <= 2048) return a.np.S > 4 ? normed<1, 8>(a, epi, nt, st) : normed<1, 4>(a, epi, nt, st);
    return a.K <= 4096 ? normed<2, 4>(a, epi, nt, st) : normed<4, 2>(a, epi, nt, st);
  }
  if (rope) {
    go<2, EPI_NONE, false, 0, 1, true>(a, st);
    return 0;
  }
  switch (epi) {
    case EPI_NONE: return out_f32 ? columns<EPI_NONE, true, 0, 1>(a, nt, st) : columns<EPI_NONE, false, 0, 1>(a, nt, st);
    case EPI_RESID: return out_f32 ? -1 : columns<EPI_RESID, false, 0, 1>(a, nt, st);
    case EPI_SILU: return out_f32 ? -1 : columns<EPI_SILU, false, 0, 1>(a, nt, st);
    case EPI_CLAMP_GLU: return out_f32 ? -1 : columns<EPI_CLAMP_GLU, false, 0, 1>(a, nt, st);
    case EPI_RELU2: return out_f32 ? -1 : columns<EPI_RELU2, false, 0, 1>(a, nt, st);
  }
  return -1;
}

}  // namespace xot
