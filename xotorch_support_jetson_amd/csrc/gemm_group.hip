// Grouped decode GEMM of routed experts on the pre-shuffled layout ([N/16][K/32] blocks of 16 rows x 32 k, 1 KB per expert):
// Y[slot] = X[gather ? gather[slot] : slot] . W[e]^T for the slots off[e] .. off[e + 1] of expert e.
//
// A workgroup has eight column tiles of one expert, a wave each: the wave streams its tile's K (or its K slice) from end to end in
// 8 KB runs, two stages in flight, while the workgroup copies the expert's rows of X chunk by chunk through a swizzled LDS double
// buffer.  What bounds it is the weight stream; the rows of an expert are few and not known to the host, so the number of 16-row
// tiles is taken from the offsets: an expert with three rows copies, reads and multiplies one tile, where a launch sized for
// the step's tokens would work through four or eight.  Weights are asked for before the gathered rows (their indices are the only
// thing a workgroup waits for first).  A tile's sum runs through K in one order whatever the number of rows.
// Experts that every token passes (shared ones) are a few tiles more of the same launches instead of two products of their own.
#include "common.h"
#include "gemm_common.h"
#include "kernels.h"

namespace xot {
namespace {

constexpr int U = 8, TW = 8, SL = 4 * U;  // k blocks a stage; waves = column tiles of a workgroup; 16-byte slots of a row's chunk
constexpr int ROWS = 64, HALF = ROWS * SL * 16;

// 16 bytes a lane, zeros past the end of r: all of the offset is in the lane's register, for the scalar offset of a buffer load is no
// part of its bounds check
__device__ __forceinline__ s16x8 buf16(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(s16x8, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
// (inside: a scalar offset behind which all lanes' bytes lie within r)
__device__ __forceinline__ s16x8 buf16nt(__amdgpu_buffer_rsrc_t r, int off, int inside) {
  return __builtin_bit_cast(s16x8, __builtin_amdgcn_raw_buffer_load_b128(r, off, inside, 2));
}

struct Stage {
  s16x8 w[U];
};

// One block of M <= 16 MT rows.  (Of the 128 registers that four waves a SIMD leave, one and two row tiles take 104 to 125; three
// spill 8 to 16, four 73 to 112, up to 116 bytes a lane.)  wr: the wave's tile and K slice; xr: X from the slice's first column on, to
// the end of its last row; rows: gather entries of the block's slots, or null with the slots' rows from row0 on.
template <int MT, int EPI, bool F32>
__device__ __forceinline__ void group_rows(char* smem, __amdgpu_buffer_rsrc_t wr, __amdgpu_buffer_rsrc_t xr, const int* rows, int row0,
                                           int ldx, int nb, int M, void* Yv, int ldy, int n0, float epi_arg) {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (or addresses of all row counts' paths are computed ahead and held in registers)
  const int lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nch = (nb + U - 1) / U;
  auto load = [&](Stage& s, int ch) {  // (past the slice: its last block again, not used)
#pragma unroll
    for (int u = 0; u < U; ++u) s.w[u] = buf16nt(wr, lane * 16, min(ch * U + u, nb - 1) * 1024);
  };
  // a wave copies MT pieces (1 KB: two rows) of a chunk; rows past M repeat the last one (they reach no stored output)
  const int row = 2 * wave + (lane >> 5), so = (row * SL + ((lane & 31) ^ row)) * 16;
  int xo[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = min(row + 16 * i, M - 1);
    xo[i] = (rows != nullptr ? rows[m] : row0 + m) * ldx * 2 + (lane & 31) * 16;
  }
  s16x8 xv[MT];
  auto xload = [&](int ch) {
#pragma unroll
    for (int i = 0; i < MT; ++i) xv[i] = buf16(xr, xo[i] + min(ch, nch - 1) * SL * 16);  // (a last chunk may pass X's end)
  };
  auto xstore = [&](int buf) {
#pragma unroll
    for (int i = 0; i < MT; ++i) *reinterpret_cast<s16x8*>(smem + buf * HALF + so + i * 16 * SL * 16) = xv[i];
  };
  // A fragments: slot 4 u + g of row 16 i + c
  int fo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) fo[j] = (c * SL + ((4 * j + g) ^ c)) * 16;
  auto frag = [&](int q, int base) {  // q = u MT + i
    const int u = q / MT, i = q % MT;
    return *reinterpret_cast<const s16x8*>(smem + base + fo[u & 3] + (u >> 2) * 256 + i * 16 * SL * 16);
  };
  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto blocks = [&](const Stage& s, int base, auto un) {  // the stage's first un blocks
    constexpr int PF = 2, Q = decltype(un)::value * MT;  // fragments read ahead of their MFMA
    s16x8 a[PF];
#pragma unroll
    for (int q = 0; q < PF; ++q) a[q] = frag(q, base);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const s16x8 cur = a[q % PF];
      if (q + PF < Q) a[q % PF] = frag(q + PF, base);
      acc[q % MT] = mfma16(cur, s.w[q / MT], acc[q % MT]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto whole = [&](const Stage& s, int buf) { blocks(s, buf * HALF, std::integral_constant<int, U>{}); };
  auto final = [&](const Stage& s, int buf) {  // (K slices are multiples of 128)
    if (nb % U == 0) whole(s, buf);
    else blocks(s, buf * HALF, std::integral_constant<int, U / 2>{});
  };

  Stage sa, sb;
  load(sa, 0);
  __builtin_amdgcn_sched_barrier(0);
  xload(0);
  __builtin_amdgcn_sched_barrier(0);
  load(sb, 1);
  __builtin_amdgcn_sched_barrier(0);
  xstore(0);
  __builtin_amdgcn_sched_barrier(0);
  xload(1);
  __syncthreads();
  int ch = 0;
  for (; ch + 2 < nch; ch += 2) {  // (a chunk's rows go where the chunk before last was read: one barrier a chunk)
    whole(sa, 0);
    xstore(1);
    __syncthreads();
    xload(ch + 2);
    load(sa, ch + 2);
    __builtin_amdgcn_sched_barrier(0);
    whole(sb, 1);
    xstore(0);
    __syncthreads();
    xload(ch + 3);
    load(sb, ch + 3);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (ch + 1 < nch) {
    whole(sa, 0);
    xstore(1);
    __syncthreads();
    final(sb, 1);
  } else {
    final(sa, 0);
  }

  auto put = [&](int m, int col, float v) {  // (Yv: this block's first row; at most 64 rows)
    if constexpr (F32) reinterpret_cast<float*>(Yv)[m * ldy + col] = v;
    else reinterpret_cast<uint16_t*>(Yv)[m * ldy + col] = f2bf(v);
  };
  asm volatile("" : "+v"(tid));
  if constexpr (epi_is_glu(EPI)) {  // tiles 2 p and 2 p + 1: gate and up rows of 16 output columns
    f32x4* red = reinterpret_cast<f32x4*>(smem);  // [TW][MT][64]
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i) red[(wave * MT + i) * 64 + lane] = acc[i];
    __syncthreads();
    for (int q = wave; q < TW / 2 * MT; q += TW) {
      const int p = q / MT, i = q - p * MT;
      const f32x4 gv = red[(2 * p * MT + i) * 64 + lane], uv = red[((2 * p + 1) * MT + i) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * g + r;
        if (m < M) put(m, n0 / 2 + 16 * p + c, glu_pair<EPI>(gv[r], uv[r], epi_arg));
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * g + r;
        if (m < M) put(m, n0 + 16 * wave + c, acc[i][r]);
      }
  }
}

// Shared experts of every token, behind the routed ones: n matrices like theirs (a column tile's blocks
// `stride` apart), whose slots follow the routed ones, T tokens each.  A block of 64 tokens has workgroups of its own.
struct Shared {
  const uint16_t* W;
  int n, T, blocks, slot0;  // blocks of 64 tokens
  long expert, stride;      // 1 KB blocks between shared experts, and between column tiles
};

// Rows 64 .. of an expert with more, as blocks of their own: the q-th such block of all experts (one wave's search through the
// offsets; the result is uniform), or -1
__device__ __forceinline__ int more_rows(const int* __restrict__ off, int E, int q, int* r0) {
  const int lane = threadIdx.x & 63;
  for (int b = 0; b < E; b += 64) {
    const int i = min(b + lane, E - 1), n = b + lane < E ? max(off[i + 1] - off[i] - 1, 0) / ROWS : 0;
    int sum = n;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int v = __shfl_up(sum, m, 64);
      if (lane >= m) sum += v;
    }
    const unsigned long long behind = __ballot(sum > q);
    if (behind != 0) {
      const int l = __builtin_ctzll(behind);
      *r0 = (q - __builtin_amdgcn_readlane(sum - n, l) + 1) * ROWS;
      return b + l;
    }
    q -= __builtin_amdgcn_readlane(sum, 63);
  }
  return -1;
}

// blockIdx: (column group, K slice, shared expert and block of tokens | expert | further blocks of experts with more than 64 rows).
// Those last ones are as many as the slots can make and mostly leave at once, all at the launch's end; one workgroup through all of an
// expert's blocks streamed its weights once a block, one after the other (64 experts of 1408 x 2048, 340 tokens that all
// want the same six: gate/up + down 184 + 139 us, here 82 + 42; evenly spread 138 + 72, here 131 + 69).
template <int EPI, bool F32>
__global__ __launch_bounds__(64 * TW, 4) void gemm_group_kernel(const uint16_t* __restrict__ X, int ldx, int xrows,
                                                                const uint16_t* __restrict__ W, void* __restrict__ Yv, int ldy,
                                                                const int* __restrict__ off, const int* __restrict__ gather, int E, int N,
                                                                int K, long ysplit, float epi_arg, Shared sh) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nb = (K >> 5) / gridDim.y, kb = blockIdx.y * nb, tile = blockIdx.x * TW + wave;
  int e = (int)blockIdx.z - sh.n * sh.blocks, first, M, x0;  // slots, and without gather their rows of X
  const uint16_t* wt;
  if (e >= 0) {
    int r0 = 0;
    if (e >= E) e = more_rows(off, E, e - E, &r0);
    if (e < 0) return;
    x0 = first = off[e] + r0, M = min(ROWS, off[e + 1] - first);
    wt = W + (((size_t)e * (N >> 4) + tile) * (K >> 5) + kb) * 512;
  } else {  // (first: their work does not hang on the routing, and a block is a full one)
    const int j = blockIdx.z / sh.blocks, t0 = (blockIdx.z - j * sh.blocks) * ROWS;
    first = sh.slot0 + j * sh.T + t0, M = min(ROWS, sh.T - t0), x0 = gather != nullptr ? t0 : first;
    wt = sh.W + (j * sh.expert + tile * sh.stride + kb) * 512;
  }
  if (M <= 0) return;
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(wt), (short)0, nb * 1024, 0x00020000);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(X + kb * 32), (short)0,
                                                                      ((xrows - 1) * ldx + K - kb * 32) * 2, 0x00020000);
  if constexpr (F32) Yv = reinterpret_cast<float*>(Yv) + blockIdx.y * ysplit;
  const size_t yo = (size_t)first * ldy;
  void* y = F32 ? (void*)(reinterpret_cast<float*>(Yv) + yo) : (void*)(reinterpret_cast<uint16_t*>(Yv) + yo);
  const int* rows = gather != nullptr && e >= 0 ? gather + first : nullptr;
  const int n0 = blockIdx.x * TW * 16;
  if (M <= 16) group_rows<1, EPI, F32>(smem, wr, xr, rows, x0, ldx, nb, M, y, ldy, n0, epi_arg);
  else if (M <= 32) group_rows<2, EPI, F32>(smem, wr, xr, rows, x0, ldx, nb, M, y, ldy, n0, epi_arg);
  else if (M <= 48) group_rows<3, EPI, F32>(smem, wr, xr, rows, x0, ldx, nb, M, y, ldy, n0, epi_arg);
  else group_rows<4, EPI, F32>(smem, wr, xr, rows, x0, ldx, nb, M, y, ldy, n0, epi_arg);
}

}  // namespace

int launch_gemm_group(const uint16_t* X, int ldx, int xrows, const uint16_t* W, void* Y, int ldy, bool out_f32, int epi, const int* off,
                      const int* gather, int E, int max_rows, int N, int K, int S, long ysplit, float epi_arg, const uint16_t* Wsh,
                      int nsh, bool sh_cols, int slot0, hipStream_t st) {
  if (max_rows <= 0) return 0;
  if (N % 128 != 0 || S < 1 || K % (128 * S) != 0 || ldx % 8 != 0 || xrows < 1) return -1;
  if (((int64_t)xrows * ldx + K) * 2 >= (int64_t(1) << 31) || (int64_t)K * 32 >= (int64_t(1) << 31)) return -1;  // 32-bit byte offsets
  if (S > 1 && (epi != EPI_NONE || !out_f32)) return -1;
  if (epi != EPI_NONE && (out_f32 || (epi != EPI_SILU && epi != EPI_CLAMP_GLU))) return -1;
  const long kbl = K / 32;
  const Shared sh{Wsh, nsh, max_rows, (max_rows + ROWS - 1) / ROWS, slot0, sh_cols ? kbl : N / 16 * kbl, sh_cols ? nsh * kbl : kbl};
  const int more = max_rows > ROWS ? slot0 / ROWS : 0;  // (each has 64 rows of its expert before it)
  if (E + (int64_t)nsh * sh.blocks + more > 65535) return -1;
  const dim3 grid(N / 128, S, E + nsh * sh.blocks + more);
  auto go = [&](auto kern) {
    kern<<<grid, 64 * TW, 2 * HALF, st>>>(X, ldx, xrows, W, Y, ldy, off, gather, E, N, K, S > 1 ? ysplit : 0L, epi_arg, sh);
  };
  if (epi == EPI_SILU) go(gemm_group_kernel<EPI_SILU, false>);
  else if (epi == EPI_CLAMP_GLU) go(gemm_group_kernel<EPI_CLAMP_GLU, false>);
  else if (out_f32) go(gemm_group_kernel<EPI_NONE, true>);
  else go(gemm_group_kernel<EPI_NONE, false>);
  return 0;
}

}  // namespace xot
