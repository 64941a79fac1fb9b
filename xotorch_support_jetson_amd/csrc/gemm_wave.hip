// Decode GEMM whose waves own whole column tiles:  Y[M, N] = X[M, K] . W[N, K]^T, M <= 64, on the pre-shuffled layout
// ([N/16][K/32] blocks of 16 rows x 32 k, 1 KB).
//
// A workgroup has nt column tiles, KW waves each: a wave streams its own part of ONE tile's K, eight consecutive blocks (8 KB) a
// stage, two stages in flight.  What bounds a decode product is the weight stream, and the stream is fastest when every CU has
// the same share of it and each wave reads long runs: 28672 x 4096 in pieces of 2 x 4 KB from two tiles 47 us, in 8 KB runs of
// one 41, which is what a plain read of the same bytes takes.  So the rows of X, which all waves need, must not cost loads of
// their own between the weights' (gathered per block as MFMA operands they were a third of the time at 16 rows): the workgroup
// copies them chunk by chunk (a chunk: the KW parts' next eight blocks) through a swizzled LDS double buffer.
// The KW partial tiles meet in LDS, so the epilogue has the whole sum -- bias, residual, gated pairs, or RoPE and the paged KV
// write (ROPE: neighbouring tiles hold the rotation partners i and i + Dh/2 of one head) -- and no slabs, no reduce launch.
// Cold weights in a graph, us, the eight-way K split of 16 / 32 columns with gathered rows that stood here before / here: 1 row
// 16384 x 2048 SiLU 15.8 / 12.3 (a plain read: 12.6), 6 rows 11264 x 2048 clamped 13.9 / 10.9, 6144 x 2048 8.4 / 7.0, 12 rows
// 128256 x 2048 94 (gemm_stream) / 86.  Beyond 16 rows, gemm_stream / here: 48 x 20224 x 2048 23.3 / 19.6, 37 x 21888 x 2048 SiLU
// 25.9 / 20.6, 24 x 28672 x 4096 SiLU 47.2 / 45.2, 24 x 6144 x 4096 with RoPE 16.3 / 15.2.
// NORM (batch-1 decode): the input row is rmsnorm(residual), computed by the first four waves in splitk_resid_rmsnorm's order while all
// have their first weight blocks in flight.
#include <algorithm>

#include "common.h"
#include "gemm_common.h"
#include "kernels.h"

namespace xot {
namespace {

constexpr int U = 8;  // k blocks a stage

// 16 bytes a lane, zeros past the end of r: all of the offset is in the lane's register, for the scalar offset of a buffer load is no
// part of its bounds check
__device__ __forceinline__ s16x8 buf16(__amdgpu_buffer_rsrc_t r, unsigned off, bool nt) {
  return __builtin_bit_cast(s16x8, nt ? __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 2)
                                      : __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}

// MT: 16-row tiles of X.  XL: X pieces (1 KB) a wave copies per chunk.  rw: rows of X kept in LDS (a power of two >= M up to 16,
// whole tiles beyond; MFMA rows past it repeat them)
template <int MT, int KW, int XL, int EPI, bool F32, int NORM, bool ROPE>
__global__ __launch_bounds__(512, MT == 1 && XL <= 4 && !ROPE ? 4 : 2) void gemm_wave_kernel(const uint16_t* __restrict__ X, int ldx, const uint16_t* __restrict__ W,
                                                        const uint16_t* __restrict__ bias, const uint16_t* __restrict__ R,
                                                        int ldr, void* __restrict__ Yv, int ldy, int M, int N, int K, int rw,
                                                        float epi_arg, NormPro np, RopeOut ro) {
  static_assert(NORM == 0 || MT == 1, "the norm prologue has one row");
  constexpr int CB = U * KW, SL = CB * 4;  // k blocks of a chunk, 16-byte slots of a row's chunk
  constexpr bool PAIR = ROPE || epi_is_glu(EPI);
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6, nt = nw / KW;
  const int t = wave / KW, p = wave - t * KW;
  const int ntiles = N >> 4, nb = K >> 5, nch = (nb + CB - 1) / CB;

  // 16-row group of W that tile t of this workgroup is (ROPE: tiles 2 i and 2 i + 1 hold dims ra .. and Dh/2 + ra .. of a head)
  auto tile_of = [&](int t) {
    const int n = blockIdx.x * nt + t;
    if constexpr (!ROPE) return n;
    const int per = ro.Dh >> 5, pr = n >> 1, head = pr / per;
    return (head * ro.Dh >> 4) + pr - head * per + (n & 1) * per;
  };
  // (a last workgroup's waves without a tile read the last one and write nothing)
  const int tile = tile_of(min(t, ntiles - 1 - (int)blockIdx.x * nt));
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(W + (size_t)tile * nb * 512), (short)0, nb * 1024, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X), (short)0, NORM ? 0 : ((M - 1) * ldx + K) * 2, 0x00020000);

  struct Stage {
    s16x8 w[U];
  };
  auto load = [&](Stage& s, int ch) {  // the wave's blocks of chunk ch (past K: zeros, not used)
#pragma unroll
    for (int u = 0; u < U; ++u) s.w[u] = buf16(wr, lane * 16u + (ch * CB + p * U + u) * 1024u, true);
  };
  // piece l of a chunk's rows of X: 64 consecutive slots of one row (or of 64 / SL rows)
  constexpr int LR = SL >= 64 ? SL / 64 : 1, RL = SL >= 64 ? 1 : 64 / SL;
  const int npc = (M * LR + RL - 1) / RL;
  s16x8 xv[XL];
  auto xload = [&](int ch) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int l = min(wave + i * nw, npc - 1);
      // (a chunk past K: the next row's numbers or, behind the last row, zeros; not used)
      if constexpr (RL > 1) xv[i] = buf16(xr, min(l * RL + lane / SL, M - 1) * ldx * 2u + (lane % SL) * 16u + ch * CB * 64u, false);
      else xv[i] = buf16(xr, lane * 16u + (l / LR) * ldx * 2u + (l % LR) * 1024u + ch * CB * 64u, false);
    }
  };
  const int half = rw * SL * 16;  // bytes of one of the two buffers
  auto xstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int l = wave + i * nw;
      if (l < npc) {
        const int row = RL > 1 ? l * RL + lane / SL : l / LR, slot = RL > 1 ? lane % SL : (l % LR) * 64 + lane;
        if (RL == 1 || row < M) *reinterpret_cast<s16x8*>(smem + buf * half + (row * SL + (slot ^ (row & 15))) * 16) = xv[i];
      }
    }
  };
  // LDS offsets of the A fragments: slot 4 u + g of the wave's part; the swizzle reaches the slot's low four bits only
  int fo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = MT > 1 ? c : c & (rw - 1);
    fo[j] = (row * SL + p * U * 4 + ((4 * j + g) ^ row)) * 16;
  }
  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto frag = [&](int q, int base) {  // q = u MT + i
    const int u = q / MT, i = q % MT;
    return *reinterpret_cast<const s16x8*>(smem + base + fo[u & 3] + (u >> 2) * 256 + i * 16 * SL * 16);
  };
  auto compute = [&](const Stage& s, int ch) {
    const int base = NORM ? ch * SL * 16 : (ch & 1) * half;
    if (ch * CB + p * U + U <= nb) {
      constexpr int PF = MT == 1 ? 2 : 4;  // fragments read ahead of their MFMA
      s16x8 a[PF];
#pragma unroll
      for (int q = 0; q < PF; ++q) a[q] = frag(q, base);
#pragma unroll
      for (int q = 0; q < U * MT; ++q) {
        const s16x8 cur = a[q % PF];
        if (q + PF < U * MT) a[q % PF] = frag(q + PF, base);
        acc[q % MT] = mfma16(cur, s.w[q / MT], acc[q % MT]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (ch * CB + p * U + u < nb) {
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[i] = mfma16(frag(u * MT + i, base), s.w[u], acc[i]);
        }
    }
  };

  // ROPE: unit q (a pair of tiles and a row tile) of the epilogue, its rows' slots and table entries.  The wave's first unit asks for
  // them here, or two dependent loads would stand between the sums and the stores
  const int have = min(nt, ntiles - (int)blockIdx.x * nt);  // tiles of this workgroup
  struct Rot {
    int pos[4];
    int64_t slot[4];
    float c[4], s[4];
  } rot;
  auto rope_rows = [&](int q) {
    const int i = q % MT;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = min(16 * i + 4 * g + r, M - 1);
      rot.pos[r] = ro.pos[m];
      rot.slot[r] = ro.slots[m];
    }
  };
  auto rope_table = [&](int q) {
    const int per = ro.Dh >> 5, n = (blockIdx.x * nt >> 1) + q / MT, d = n % per * 16 + c;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* cs = ro.cos_sin + (size_t)min(max(rot.pos[r], 0), ro.max_pos - 1) * ro.Dh + d;
      rot.c[r] = cs[0];
      rot.s[r] = cs[ro.Dh >> 1];
    }
  };
  const int units = (have >> 1) * MT;
  const bool rope_here = ROPE && wave < units;
  if (rope_here) rope_rows(wave);

  Stage sa, sb;
  if constexpr (NORM > 0) {
    s16x8 ha[NORM], la[NORM];
    const int nchunk = np.D >> 3;
    // (asked for before the weights: loads return in order, and the row's chain is the longer one)
#pragma unroll
    for (int i = 0; i < NORM; ++i) {
      const int cc = min((tid & 255) + 256 * i, nchunk - 1);
      ha[i] = ld16(np.h + cc * 8);
      la[i] = ld16(np.lnw + cc * 8);
    }
    __builtin_amdgcn_sched_barrier(0);
    load(sa, 0);
    load(sb, 1);
    __builtin_amdgcn_sched_barrier(0);
    if (rope_here) rope_table(wave);
    __builtin_amdgcn_sched_barrier(0);
    // one row: the residual (stored again by workgroup 0), its RMS norm times the weight -> LDS.  256 threads, 8 consecutive elements
    // each per round, in the order of splitk_resid_rmsnorm_kernel<*, *, 256>
    __shared__ float nred[4];
    if (wave < 4) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NORM; ++i) {
        const int cc = tid + 256 * i;
        if (cc >= nchunk) continue;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
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
        *reinterpret_cast<s16x8*>(smem + cc * 16) = o;
      }
    }
    __syncthreads();
    int ch = 0;
    for (; ch + 2 < nch; ch += 2) {
      compute(sa, ch);
      load(sa, ch + 2);
      compute(sb, ch + 1);
      load(sb, ch + 3);
    }
    compute(sa, ch);
    if (ch + 1 < nch) compute(sb, ch + 1);
  } else {
    // (X first: loads return in order, and its way through LDS is the longer one)
    xload(0);
    load(sa, 0);
    __builtin_amdgcn_sched_barrier(0);
    load(sb, 1);
    __builtin_amdgcn_sched_barrier(0);
    if (rope_here) rope_table(wave);
    __builtin_amdgcn_sched_barrier(0);
    xstore(0);
    __builtin_amdgcn_sched_barrier(0);
    xload(1);
    __syncthreads();
    int ch = 0;
    for (; ch + 2 < nch; ch += 2) {  // (a chunk's rows go where the chunk before last was read: one barrier a chunk)
      compute(sa, ch);
      xstore(1);
      __syncthreads();
      xload(ch + 2);
      load(sa, ch + 2);
      __builtin_amdgcn_sched_barrier(0);
      compute(sb, ch + 1);
      xstore(0);
      __syncthreads();
      xload(ch + 3);
      load(sb, ch + 3);
      __builtin_amdgcn_sched_barrier(0);
    }
    compute(sa, ch);
    if (ch + 1 < nch) {
      xstore(1);
      __syncthreads();
      compute(sb, ch + 1);
    }
  }

  // partial tiles of a tile's waves in K order; lane (g, c): tokens 16 i + 4 g + r, column c of the tile
  f32x4* red = reinterpret_cast<f32x4*>(smem);  // [nw][MT][64]
  if constexpr (KW > 1 || PAIR) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i) red[(wave * MT + i) * 64 + lane] = acc[i];
    __syncthreads();
  }
  auto total = [&](int t, int i) {
    f32x4 v = red[(t * KW * MT + i) * 64 + lane];
#pragma unroll
    for (int q = 1; q < KW; ++q) v += red[((t * KW + q) * MT + i) * 64 + lane];
    return v;
  };
  auto put = [&](int m, int col, float v) {
    if constexpr (F32) reinterpret_cast<float*>(Yv)[(size_t)m * ldy + col] = v;
    else reinterpret_cast<uint16_t*>(Yv)[(size_t)m * ldy + col] = f2bf(v);
  };
  if constexpr (ROPE) {
    const int hd = ro.Dh >> 1, per = ro.Dh >> 5;
    for (int q = wave; q < units; q += nw) {
      if (q != wave) {
        rope_rows(q);
        rope_table(q);
      }
      const int pr = q / MT, i = q - pr * MT, n = (blockIdx.x * nt >> 1) + pr, head = n / per, d = (n - head * per) * 16 + c;
      f32x4 lo = total(2 * pr, i), hi = total(2 * pr + 1, i);
      if (bias != nullptr) {
        lo += bf2f(bias[head * ro.Dh + d]);
        hi += bf2f(bias[head * ro.Dh + hd + d]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * g + r;
        if (m >= M) continue;
        const int64_t slot = rot.slot[r] < ro.nslots ? rot.slot[r] : -1;
        const int64_t page = slot >= 0 ? slot / ro.BS : 0;
        const int off = slot >= 0 ? (int)(slot % ro.BS) : 0;
        if (head >= ro.H + ro.Hkv) {
          if (slot < 0) continue;
          uint16_t* dst = ro.vc + ((size_t)page * ro.Hkv + (head - ro.H - ro.Hkv)) * ro.Dh * ro.BS;
          dst[v_page_off(off, d, ro.Dh)] = f2bf(lo[r]);
          dst[v_page_off(off, hd + d, ro.Dh)] = f2bf(hi[r]);
          continue;
        }
        uint16_t* dst;
        if (head < ro.H) {
          dst = ro.q + ((size_t)m * ro.H + head) * ro.Dh;
        } else {
          if (slot < 0) continue;
          dst = ro.kc + (((size_t)page * ro.Hkv + (head - ro.H)) * ro.BS + off) * ro.Dh;
        }
        dst[d] = f2bf(lo[r] * rot.c[r] - hi[r] * rot.s[r]);
        dst[hd + d] = f2bf(hi[r] * rot.c[r] + lo[r] * rot.s[r]);
      }
    }
  } else if constexpr (epi_is_glu(EPI)) {
    for (int q = wave; q < units; q += nw) {
      const int pr = q / MT, i = q - pr * MT, n0 = (blockIdx.x * nt + 2 * pr) * 16;  // gate rows of W; the up rows follow
      f32x4 gv = total(2 * pr, i), uv = total(2 * pr + 1, i);
      if (bias != nullptr) {
        gv += bf2f(bias[n0 + c]);
        uv += bf2f(bias[n0 + 16 + c]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * g + r;
        if (m < M) put(m, n0 / 2 + c, glu_pair<EPI>(gv[r], uv[r], epi_arg));
      }
    }
  } else {
    auto out = [&](int t, int i, f32x4 v) {
      const int n = (blockIdx.x * nt + t) * 16 + c;
      if (bias != nullptr) v += bf2f(bias[n]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * g + r;
        if (m >= M) continue;
        if constexpr (EPI == EPI_RESID) v[r] += bf2f(R[(size_t)m * ldr + n]);
        put(m, n, epi_elem<EPI>(v[r]));
      }
    };
    if constexpr (KW == 1) {
      if (t < have) {
#pragma unroll
        for (int i = 0; i < MT; ++i) out(t, i, acc[i]);
      }
    } else {
      for (int q = wave; q < have * MT; q += nw) out(q / MT, q % MT, total(q / MT, q % MT));
    }
  }
}

template <int MT, int KW, int XL, int EPI, bool F32, int NORM, bool ROPE>
int go(const WaveGemm& a, int nt, hipStream_t st) {
  constexpr int CB = U * KW;
  int rw = 16 * MT;
  if (MT == 1)
    while (rw / 2 >= a.M) rw /= 2;
  const int nw = nt * KW, nb = a.K / 32;
  const size_t xbytes = NORM ? (size_t)(nb + CB - 1) / CB * CB * 64 : (size_t)2 * rw * CB * 64;
  const size_t smem = std::max(xbytes, KW > 1 || ROPE || epi_is_glu(EPI) ? (size_t)nw * MT * 1024 : 0);
  auto kern = gemm_wave_kernel<MT, KW, XL, EPI, F32, NORM, ROPE>;
  static_assert(2 * 16 * MT * CB * 64 <= 65536 && 8 * MT * 1024 <= 65536, "LDS a launch takes without asking");
  kern<<<(a.N / 16 + nt - 1) / nt, 64 * nw, smem, st>>>(a.X, a.ldx, a.W, a.bias, a.R, a.ldr, a.Y, a.ldy, a.M, a.N, a.K, rw, a.epi_arg,
                                                        a.np, a.ro);
  return 0;
}

// Waves per tile (cold weights in a graph, us).  One row tile: eight waves in all, but never more than four a tile: 3072 x 2048 at
// 1 row by single tiles, 4 / 8 waves 5.0 / 5.2, 6144 x 2048 at 6 rows 8.0 / 10.2; 11264 x 2048 by fours, 1 / 2 waves 12.2 / 10.9.
// More rows: the chunk's X takes the LDS that more parts would need, and the waves' stages are enough in flight: 20224 x 2048 at
// 48 rows by threes, 1 / 2 waves 20.8 / 24.1; two only beside a lone pair (6144 x 4096 at 24 rows 16.4 / 14.7).
template <int EPI, bool F32, int NORM, bool ROPE>
int one_row_tile(const WaveGemm& a, int nt, hipStream_t st) {
  constexpr bool LONE = !ROPE && !epi_is_glu(EPI);
  if (nt == 1) {
    if constexpr (LONE) return go<1, 4, NORM ? 4 : 8, EPI, F32, NORM, ROPE>(a, nt, st);  // (half the waves copy X)
    else return -1;
  }
  if (nt == 2) return go<1, 4, 4, EPI, F32, NORM, ROPE>(a, nt, st);
  return nt <= 4 ? go<1, 2, 4, EPI, F32, NORM, ROPE>(a, nt, st) : -1;
}

template <int EPI, bool F32, bool ROPE>
int by_rows(const WaveGemm& a, int nt, hipStream_t st) {
  const int mt = (a.M + 15) / 16;
  if (mt == 1) return one_row_tile<EPI, F32, 0, ROPE>(a, nt, st);
  if (nt < mt) return -1;  // (a wave copies at most eight pieces of a chunk)
  if (mt == 2) return nt == 2 ? go<2, 2, 8, EPI, F32, 0, ROPE>(a, nt, st) : go<2, 1, 8, EPI, F32, 0, ROPE>(a, nt, st);
  return mt == 3 ? go<3, 1, 8, EPI, F32, 0, ROPE>(a, nt, st) : go<4, 1, 8, EPI, F32, 0, ROPE>(a, nt, st);
}

template <int NORM>
int normed(const WaveGemm& a, int epi, int nt, hipStream_t st) {
  if (a.ro.q != nullptr) return one_row_tile<EPI_NONE, false, NORM, true>(a, nt, st);
  return epi == EPI_SILU ? one_row_tile<EPI_SILU, false, NORM, false>(a, nt, st)
                         : one_row_tile<EPI_NONE, false, NORM, false>(a, nt, st);
}

// Up to 8 rows, one column tile a workgroup (HALF: half of one, its eight columns), the eight waves a part of K each: a wave copies
// the rows of X that its own blocks need through LDS of its own, so no wave waits for another before the partial tiles meet.
// HALF: a load takes the tile half's 128-byte runs of two k blocks, the first in columns 0 .. 7 of the MFMA operand, the second in
// 8 .. 15; each block's rows of X multiply it all and the sums of the other block's columns are not used.
// Bound by the weight stream: 2048 columns by whole tiles keep half of the CUs, which take 50 GB/s each at most (2048 x 8192 at one
// row 9.4 us by tiles, 7.9 by halves; x 5632 7.4 and 6.2, 8.7 with four waves a tile that meet at barriers); from 9 rows on slabs are the
// faster, for every workgroup copies all of X (2048 x 5632 at 16 rows 9.1 / 6.9).
// NP (one row): X is the merge of a lone sequence's attention parts, NP at most, in attn_decode_split_kernel's arithmetic: a wave merges
// what its own blocks multiply, while its weights are on their way.
template <bool HALF, int XL, int EPI, bool F32, int NP = 0>
__global__ __launch_bounds__(512, 2) void gemm_solo_kernel(const uint16_t* __restrict__ X, int ldx, const uint16_t* __restrict__ W,
                                                           const uint16_t* __restrict__ bias, const uint16_t* __restrict__ R, int ldr,
                                                           void* __restrict__ Yv, int ldy, int M, int N, int K, LoneMerge mg) {
  static_assert(NP == 0 || XL == 1, "merged parts are one row");
  constexpr int KW = 8, CB = U * KW, SL = U * 4;   // waves, k blocks of a chunk, 16-byte slots of a row's part of it
  constexpr int RL = 64 / SL, ROWS = XL * RL;      // rows of a 1 KB piece of X; rows in LDS (MFMA rows past them repeat them)
  constexpr int NI = HALF ? U / 2 : U;             // weight loads of a stage
  __shared__ __attribute__((aligned(16))) char smem[KW * XL * 1024 > KW * 1024 ? KW * XL * 1024 : KW * 1024];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = HALF ? blockIdx.x >> 1 : blockIdx.x, col0 = HALF ? (blockIdx.x & 1) * 8 : 0;
  const int nb = K >> 5, nch = (nb + CB - 1) / CB;
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(W + (size_t)tile * nb * 512), (short)0, nb * 1024, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X), (short)0, NP ? 0 : ((M - 1) * ldx + K) * 2, 0x00020000);
  char* xs = smem + p * (XL * 1024);
  struct Stage {
    s16x8 w[NI];
  };
  const unsigned woff = HALF ? (c >> 3) * 1024u + (g * 16 + col0 + (c & 7)) * 16u : lane * 16u;
  auto load = [&](Stage& s, int ch) {  // the wave's blocks of chunk ch (past K: zeros, not used)
#pragma unroll
    for (int u = 0; u < NI; ++u) s.w[u] = buf16(wr, woff + (ch * CB + p * U + u * (U / NI)) * 1024u, true);
  };
  const int prow = lane / SL, pslot = lane % SL;
  auto xload = [&](s16x8 (&x)[XL], int ch) {  // (past K: the next row's numbers or zeros, not used)
#pragma unroll
    for (int i = 0; i < XL; ++i)
      x[i] = buf16(xr, min(i * RL + prow, M - 1) * ldx * 2u + pslot * 16u + (ch * CB + p * U) * 64u, false);
  };
  auto xstore = [&](const s16x8 (&x)[XL]) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int row = i * RL + prow;
      *reinterpret_cast<s16x8*>(xs + (row * SL + (pslot ^ (row & 15))) * 16) = x[i];
    }
  };
  const int row0 = c & (ROWS - 1);
  int fo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) fo[j] = (row0 * SL + ((4 * j + g) ^ row0)) * 16;
  f32x4 acc[HALF ? 2 : 1];
#pragma unroll
  for (int i = 0; i < (HALF ? 2 : 1); ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const Stage& s, int ch) {
    const int left = nb - ch * CB - p * U;  // blocks of K from the wave's part on (a multiple of four)
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < left) {
        const s16x8 a = *reinterpret_cast<const s16x8*>(xs + fo[u & 3] + (u >> 2) * 256);
        f32x4& t = acc[HALF ? u & 1 : 0];
        t = mfma16(a, s.w[HALF ? u >> 1 : u], t);
      }
  };
  Stage sa, sb;
  s16x8 xa[XL], xb[XL];
  if constexpr (NP > 0) {  // (at most two chunks: xa and xb are all of X)
    const int pages = (min(max(mg.ctx[0], 0), mg.max_blocks * 64) + 63) / 64, ppp = decode_lone_pages(pages, mg.Hkv);
    const int np = min(max(1, (pages + ppp - 1) / ppp), NP);
    struct Part {
      f32x2_t ml;
      f32x4 o[2];
    };
    auto parts = [&](Part (&t)[NP], int ch) {
      const int k = min((ch * CB + p * U) * 32 + pslot * 8, K - 8);
#pragma unroll
      for (int q = 0; q < NP; ++q) {  // (past the last: the last again, not used)
        const int at = min(q, np - 1) * K + k, sh = mg.Dh == 128 ? 7 : 6;
        t[q].ml = *reinterpret_cast<const f32x2_t*>(mg.ml + (at >> sh) * 2);
        t[q].o[0] = *reinterpret_cast<const f32x4*>(mg.o + at);
        t[q].o[1] = *reinterpret_cast<const f32x4*>(mg.o + at + 4);
      }
    };
    auto merge = [&](const Part (&t)[NP]) {
      float M = -1e30f, L = 0.f;
#pragma unroll
      for (int q = 0; q < NP; ++q) M = fmaxf(M, t[q].ml[0]);
      f32x4 o[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int q = 0; q < NP; ++q)
        if (q < np) {
          const float f = exp2f(t[q].ml[0] - M);
          L += t[q].ml[1] * f;
#pragma unroll
          for (int i = 0; i < 2; ++i) o[i] += t[q].o[i] * f;
        }
      s16x8 x;
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = (short)f2bf(L > 0.f ? o[e >> 2][e & 3] / L : 0.f);
      return x;
    };
    Part ta[NP], tb[NP];
    parts(ta, 0);
    if (nch > 1) parts(tb, 1);
    __builtin_amdgcn_sched_barrier(0);
    load(sa, 0);
    load(sb, 1);
    __builtin_amdgcn_sched_barrier(0);
    xa[0] = merge(ta);
    if (nch > 1) xb[0] = merge(tb);
  } else {
    xload(xa, 0);
    load(sa, 0);
    __builtin_amdgcn_sched_barrier(0);
    xload(xb, 1);
    load(sb, 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  for (int ch = 0; ch < nch; ch += 2) {  // (a wave's LDS accesses keep their order: no wait between a chunk's reads and the next writes)
    xstore(xa);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NP == 0) xload(xa, ch + 2);
    compute(sa, ch);
    __builtin_amdgcn_sched_barrier(0);
    load(sa, ch + 2);
    __builtin_amdgcn_sched_barrier(0);
    if (ch + 1 >= nch) break;
    xstore(xb);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NP == 0) xload(xb, ch + 3);
    compute(sb, ch + 1);
    __builtin_amdgcn_sched_barrier(0);
    load(sb, ch + 3);
    __builtin_amdgcn_sched_barrier(0);
  }
  f32x4 v = acc[0];
  if constexpr (HALF) {  // columns c and c ^ 8 are one, over the even and the odd blocks
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float t = c < 8 ? acc[0][r] : acc[1][r];
      v[r] = t + __uint_as_float(row_turn<8>(__float_as_uint(t)));
    }
  }
  __syncthreads();
  f32x4* red = reinterpret_cast<f32x4*>(smem);  // [KW][64]
  red[p * 64 + lane] = v;
  __syncthreads();
  if (p != 0 || (HALF && c >= 8)) return;
#pragma unroll
  for (int q = 1; q < KW; ++q) v += red[q * 64 + lane];
  const int n = tile * 16 + col0 + c;
  if (bias != nullptr) v += bf2f(bias[n]);
#pragma unroll
  for (int r = 0; r < 4; ++r) {  // lane (g, c): token 4 g + r
    const int m = 4 * g + r;
    if (m >= M) continue;
    float y = v[r];
    if constexpr (EPI == EPI_RESID) y += bf2f(R[(size_t)m * ldr + n]);
    if constexpr (F32) reinterpret_cast<float*>(Yv)[(size_t)m * ldy + n] = y;
    else reinterpret_cast<uint16_t*>(Yv)[(size_t)m * ldy + n] = f2bf(y);
  }
}

template <bool HALF, int EPI, bool F32>
int solo_rows(const WaveGemm& a, hipStream_t st) {
  const int grid = HALF ? a.N / 8 : a.N / 16;
#define XOT_SOLO(XLV) \
  gemm_solo_kernel<HALF, XLV, EPI, F32><<<grid, 512, 0, st>>>(a.X, a.ldx, a.W, a.bias, a.R, a.ldr, a.Y, a.ldy, a.M, a.N, a.K, a.mg)
  if (a.M <= 2) XOT_SOLO(1);
  else if (a.M <= 4) XOT_SOLO(2);
  else XOT_SOLO(4);
#undef XOT_SOLO
  return 0;
}

constexpr int MERGE_PARTS = 4;
template <bool HALF>
int solo_merge(const WaveGemm& a, hipStream_t st) {
  gemm_solo_kernel<HALF, 1, EPI_RESID, false, MERGE_PARTS><<<HALF ? a.N / 8 : a.N / 16, 512, 0, st>>>(
      nullptr, 0, a.W, a.bias, a.R, a.ldr, a.Y, a.ldy, 1, a.N, a.K, a.mg);
  return 0;
}

template <int EPI, bool F32>
int solo(const WaveGemm& a, hipStream_t st) {
  return a.N <= 2048 ? solo_rows<true, EPI, F32>(a, st) : solo_rows<false, EPI, F32>(a, st);
}

}  // namespace

int launch_gemm_wave(const WaveGemm& a, bool out_f32, int epi, int nt, hipStream_t st) {
  if (a.M <= 0) return 0;
  const bool rope = a.ro.q != nullptr, norm = a.np.h != nullptr;
  if (a.M > 64 || a.K % 128 != 0 || a.K <= 0 || nt < 0 || nt > 8 || a.N % 16 != 0) return -1;
  if ((int64_t)a.K * 32 >= (int64_t(1) << 31)) return -1;  // (32-bit byte offsets into a tile)
  if (!norm && (a.ldx % 8 != 0 || (int64_t)a.M * a.ldx * 2 >= (int64_t(1) << 31))) return -1;
  if ((rope || epi_is_glu(epi)) && (nt % 2 != 0 || a.N % 32 != 0)) return -1;
  if (rope && (epi != EPI_NONE || out_f32 || a.ro.Dh % 32 != 0 || a.N != (a.ro.H + 2 * a.ro.Hkv) * a.ro.Dh || a.ro.max_pos < 1)) return -1;
  if (norm) {
    if (nt == 0 || a.M != 1 || out_f32 || (epi != EPI_NONE && epi != EPI_SILU) || a.np.D != a.K || a.K > 8192 || a.np.lnw == nullptr ||
        a.np.hout == nullptr)
      return -1;
    return a.K <= 2048 ? normed<1>(a, epi, nt, st) : a.K <= 4096 ? normed<2>(a, epi, nt, st) : normed<4>(a, epi, nt, st);
  }
  if (a.mg.o != nullptr) {  // (two chunks of K)
    if (nt != 0 || a.M != 1 || out_f32 || epi != EPI_RESID || rope || norm || a.K > 2 * 2048 || a.mg.max_parts > MERGE_PARTS || a.K % a.mg.Dh != 0) return -1;
    return a.N <= 2048 ? solo_merge<true>(a, st) : solo_merge<false>(a, st);
  }
  if (nt == 0) {
    if (rope || norm || a.M > 8) return -1;
    if (epi == EPI_RESID) return out_f32 ? -1 : solo<EPI_RESID, false>(a, st);
    if (epi != EPI_NONE) return -1;
    return out_f32 ? solo<EPI_NONE, true>(a, st) : solo<EPI_NONE, false>(a, st);
  }
  if (rope) return by_rows<EPI_NONE, false, true>(a, nt, st);
  switch (epi) {
    case EPI_NONE: return out_f32 ? by_rows<EPI_NONE, true, false>(a, nt, st) : by_rows<EPI_NONE, false, false>(a, nt, st);
    case EPI_RESID: return out_f32 ? -1 : by_rows<EPI_RESID, false, false>(a, nt, st);
    case EPI_SILU: return out_f32 ? -1 : by_rows<EPI_SILU, false, false>(a, nt, st);
    case EPI_CLAMP_GLU: return out_f32 ? -1 : by_rows<EPI_CLAMP_GLU, false, false>(a, nt, st);
    case EPI_RELU2: return out_f32 ? -1 : by_rows<EPI_RELU2, false, false>(a, nt, st);
  }
  return -1;
}

}  // namespace xot
