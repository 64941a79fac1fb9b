// Shared device helpers for the CDNA4 (gfx950) kernel library.
//
// Everything here is written for wave64 + MFMA on MI355X: bf16 is carried as raw
// 16-bit storage and widened to fp32 for arithmetic, memory traffic is 16 B per
// lane (8 bf16) wherever the layout allows, and the matrix work goes through
// __builtin_amdgcn_mfma_f32_16x16x32_bf16 (16x16 output tile, K=32 per issue).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

namespace xot {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVE = 64;

__device__ __forceinline__ float bf2f(uint16_t u) { return __uint_as_float(((uint32_t)u) << 16); }
__device__ __forceinline__ float bf2f(short s) { return bf2f((uint16_t)s); }
__device__ __forceinline__ uint16_t f2bf(float f) {
  __hip_bfloat16 h = __float2bfloat16(f);
  return __builtin_bit_cast(uint16_t, h);
}

// 16x16x32 bf16 MFMA.  Operand maps (lane l, j = 0..7):
//   A[row = l&15][k = 8*(l>>4) + j],  B[k = 8*(l>>4) + j][col = l&15]
//   C/D: col = l&15, row = 4*(l>>4) + reg
// Any permutation of k applied identically to A and B leaves the product unchanged;
// the kernels use that to make each lane's operand bytes contiguous in memory.
__device__ __forceinline__ f32x4 mfma16(const s16x8& a, const s16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Exchanges between lanes that stay in the vector ALU: a step through LDS (__shfl_xor, ds_bpermute) costs its round trip of about 100
// cycles, these a few.  What a lane adds or compares is the same, so are the results, bit for bit.  Small launches, whose reductions
// stand in a chain of dependent steps, gain: Zepalorn generations of 6 requests 9.70 -> 9.46 ms, of 9 of Tarepel 5.85 -> 5.76.
// f(v of this lane, v of lane ^ M), f symmetric: M 32 and 16 swap halves and rows of 16
template <int M, class F>
__device__ __forceinline__ auto lane_xor(uint32_t v, F f) {
  static_assert(M == 32 || M == 16, "halves, or rows of 16");
  const auto r = M == 32 ? __builtin_amdgcn_permlane32_swap(v, v, false, false) : __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return f(r[0], r[1]);
}
// v of the lane N places on in this row of 16 (cyclic): the partner lane ^ N of a reduction that has done the larger steps, for its
// values then repeat every 2 N lanes
template <int N>
__device__ __forceinline__ uint32_t row_turn(uint32_t v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x120 + N, 0xf, 0xf, false);
}
template <int M>
__device__ __forceinline__ float xor_sum(float v) {
  return lane_xor<M>(__float_as_uint(v), [](uint32_t a, uint32_t b) { return __uint_as_float(a) + __uint_as_float(b); });
}
template <int M>
__device__ __forceinline__ float xor_max(float v) {
  return lane_xor<M>(__float_as_uint(v), [](uint32_t a, uint32_t b) { return fmaxf(__uint_as_float(a), __uint_as_float(b)); });
}
// reductions across the 16 lanes that share (l>>4)
__device__ __forceinline__ float group16_sum(float v) {
  v += __uint_as_float(row_turn<8>(__float_as_uint(v)));
  v += __uint_as_float(row_turn<4>(__float_as_uint(v)));
  v += __uint_as_float(row_turn<2>(__float_as_uint(v)));
  v += __uint_as_float(row_turn<1>(__float_as_uint(v)));
  return v;
}
__device__ __forceinline__ float group16_max(float v) {
  v = fmaxf(v, __uint_as_float(row_turn<8>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(row_turn<4>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(row_turn<2>(__float_as_uint(v))));
  v = fmaxf(v, __uint_as_float(row_turn<1>(__float_as_uint(v))));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) { return group16_sum(xor_sum<16>(xor_sum<32>(v))); }
// The wave's sums of eight values at once, 18 operations instead of eight times eight: each of the first three steps adds two
// values' halves, so that lane wave_sum8_lane(i), and the seven behind it, end with the sum of v[i].
__device__ __forceinline__ float wave_sum8(const float (&v)[8]) {
  float u[4], w[2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[2 * j]), __float_as_uint(v[2 * j + 1]), false, false);
    u[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(u[2 * j]), __float_as_uint(u[2 * j + 1]), false, false);
    w[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) w[j] += __uint_as_float(row_turn<8>(__float_as_uint(w[j])));
  float s = threadIdx.x & 8 ? w[1] : w[0];
  s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x141, 0xf, 0xf, false));  // the eight lanes mirrored
  s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x4e, 0xf, 0xf, false));   // lane ^ 2
  return s + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0xb1, 0xf, 0xf, false));  // lane ^ 1
}
__device__ __forceinline__ constexpr int wave_sum8_lane(int i) { return 32 * (i & 1) + 16 * ((i >> 1) & 1) + 8 * (i >> 2); }
__device__ __forceinline__ float wave_max(float v) { return group16_max(xor_max<16>(xor_max<32>(v))); }
// the largest v of the wave with its id, the lowest id among equals
__device__ __forceinline__ void wave_argmax(float& v, int& id) {
  auto take = [&](uint32_t ov, uint32_t oi) {
    const float o = __uint_as_float(ov);
    if (o > v || (o == v && (int)oi < id)) {
      v = o;
      id = (int)oi;
    }
  };
  auto swap = [&](auto rv, auto ri) {  // {lower, upper} halves or rows: one is this lane's own
    v = __uint_as_float(rv[0]);
    id = (int)ri[0];
    take(rv[1], ri[1]);
  };
  swap(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false),
       __builtin_amdgcn_permlane32_swap((uint32_t)id, (uint32_t)id, false, false));
  swap(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false),
       __builtin_amdgcn_permlane16_swap((uint32_t)id, (uint32_t)id, false, false));
  take(row_turn<8>(__float_as_uint(v)), row_turn<8>((uint32_t)id));
  take(row_turn<4>(__float_as_uint(v)), row_turn<4>((uint32_t)id));
  take(row_turn<2>(__float_as_uint(v)), row_turn<2>((uint32_t)id));
  take(row_turn<1>(__float_as_uint(v)), row_turn<1>((uint32_t)id));
}

__device__ __forceinline__ uint32_t wave_sum_u(uint32_t v) {
  auto add = [](uint32_t a, uint32_t b) { return a + b; };
  v = lane_xor<16>(lane_xor<32>(v, add), add);
  v += row_turn<8>(v);
  v += row_turn<4>(v);
  v += row_turn<2>(v);
  return v + row_turn<1>(v);
}
__device__ __forceinline__ uint32_t wave_max_u(uint32_t v) {
  auto most = [](uint32_t a, uint32_t b) { return max(a, b); };
  v = lane_xor<16>(lane_xor<32>(v, most), most);
  v = max(v, row_turn<8>(v));
  v = max(v, row_turn<4>(v));
  v = max(v, row_turn<2>(v));
  return max(v, row_turn<1>(v));
}

// The sequence at place p of B when the longest come first (len(b); equal ones as they are given).  Each wave finds it for
// itself: a sequence a lane, one compare a sequence, none where all are as long (32 prompts of 200 tokens, 24 heads on 3: 30.1 us in
// the given order, 34.6 with two compares a sequence, 30.3 now).  Above 32 sequences the given order stays: there are then
// several rounds of workgroups.  What a long sequence met late costs them, us with 4000 tokens first / last among 39 prompts of 60
// to 360: prompt attention of 32 heads 260 / 262, chunk-local attention 79 / 91, delta-rule scans of 16 heads 464 / 635; among 99
// 417 / 420, 139 / 151, 605 / 981.
template <typename F>
__device__ __forceinline__ int nth_longest(int B, int p, F len) {
  if (B <= 1 || B > 32) return p;
  const int lane = threadIdx.x & 63, n = lane < B ? len(lane) : 0;
  if (__ballot(lane < B && n != __builtin_amdgcn_readfirstlane(n)) == 0) return p;
  const uint32_t key = lane < B ? (uint32_t)n * 64u + 63u - lane : 0;  // larger: longer, or as long and given earlier; no two alike
  int rank = 0;
  for (int j0 = 0; j0 < B; j0 += 8)
#pragma unroll
    for (int j = 0; j < 8; ++j) rank += (uint32_t)__builtin_amdgcn_readlane((int)key, j0 + j) > key ? 1 : 0;
  return __builtin_ctzll(__ballot(lane < B && rank == p));
}

// Work of a prompt attention workgroup, of a grid (tiles, kv heads, sequences).  Consecutive workgroups go to the 8 XCDs in
// turn.  Where the (sequence, kv head) pairs are a multiple of 8 they are dealt to the XCDs in turn, longest context first,
// and an XCD takes a pair's tiles one after the other, the last rows (most keys) first: the pair's pages come from one L2,
// and every XCD has its share of the long sequences.  Otherwise the pairs run fastest: all pairs' heaviest tiles first, a
// pair over several XCDs.
struct PromptWork {
  int tile, head, seq;
};
__device__ __forceinline__ PromptWork prompt_work(const int* ctx_lens) {
  const uint32_t tiles = gridDim.x, heads = gridDim.y, pairs = heads * gridDim.z;
  const uint32_t lin = blockIdx.x + tiles * (blockIdx.y + heads * blockIdx.z);
  uint32_t pair, turn;
  if ((pairs & 7) == 0) {
    const uint32_t j = lin >> 3, r = j / tiles;
    pair = r * 8 + (lin & 7);
    turn = j - r * tiles;
  } else {
    turn = lin / pairs;
    pair = lin - turn * pairs;
  }
  const uint32_t p = pair / heads;
  const int seq = nth_longest((int)gridDim.z, (int)p, [&](int b) { return ctx_lens[b]; });
  return {(int)(tiles - 1 - turn), (int)(pair - p * heads), seq};
}

__device__ __forceinline__ s16x8 ld16(const void* p) { return *reinterpret_cast<const s16x8*>(p); }
// non-temporal 16-B load (global_load_dwordx4 ... nt): bytes read once per kernel (KV pages in decode)
__device__ __forceinline__ s16x8 ld16nt(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const s16x8*>(p));
}
__device__ __forceinline__ void st16(void* p, const s16x8& v) { *reinterpret_cast<s16x8*>(p) = v; }

__device__ __forceinline__ float silu(float x) { return x / (1.0f + __expf(-x)); }

// Paged V cache: a 64-key page of one KV head is stored chunk-major, 8 chunks of 8 keys, each chunk [Dh][8]:
// element offset of (key, d) inside the page.  Readers (the attention kernels) load 8 consecutive keys of one dim
// as one 16-B run; a writer's token fills 2 B in each of Dh 16-B runs packed 8 to a 128-B line.
__host__ __device__ __forceinline__ int v_page_off(int key, int d, int Dh) { return ((key >> 3) * Dh + d) * 8 + (key & 7); }

}  // namespace xot
