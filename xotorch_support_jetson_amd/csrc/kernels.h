// Host-side launchers of the gfx950 kernel library (raw pointers + stream; no torch types so the
// kernel translation units compile without the torch headers).  Launchers that can reject a shape
// return -1 and launch nothing; the Python layer turns that into a loud error.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xot {

void launch_rmsnorm(const uint16_t* x, const uint16_t* res, const uint16_t* w, uint16_t* out, uint16_t* res_out,
                    int rows, int D, float eps, hipStream_t s);
void launch_rmsnorm_bwd(const uint16_t* x, const uint16_t* w, const uint16_t* dy, uint16_t* dx, float* dw,
                        float* dw_part, int rows, int D, float eps, hipStream_t s, const uint16_t* res = nullptr);
int rmsnorm_bwd_part_rows();
void launch_embedding(const int32_t* ids, const uint16_t* table, uint16_t* out, int T, int D, int vocab,
                      hipStream_t s);
void launch_silu_mul(const uint16_t* gu, uint16_t* out, int T, int F, hipStream_t s);
void launch_silu_mul_il(const uint16_t* gu, uint16_t* out, int T, int F, hipStream_t s);
void launch_silu_mul_bwd(const uint16_t* gu, const uint16_t* dout, uint16_t* dgu, int T, int F, hipStream_t s);
void launch_splitk_rope_kv_write(const float* ws, int S, const uint16_t* bias, const int32_t* pos,
                                 const float* cos_sin, const int64_t* slots, uint16_t* q_out, uint16_t* kc,
                                 uint16_t* vc, int T, int H, int Hkv, int Dh, int BS, int max_pos, long nslots,
                                 hipStream_t s);
void launch_rope_kv_write(const uint16_t* qkv, const int32_t* pos, const float* cos_sin, const int64_t* slots,
                          uint16_t* q_out, uint16_t* kc, uint16_t* vc, int T, int H, int Hkv, int Dh, int BS,
                          int max_pos, long nslots, hipStream_t s);
void launch_rope_apply(const uint16_t* x, uint16_t* y, const int32_t* pos, const float* cos_sin, int T, int nh,
                       int Dh, long ldx, long ldy, int max_pos, bool inverse, hipStream_t s);

int launch_gemm_skinny(const uint16_t* X, int ldx, const uint16_t* W, int ldw, const uint16_t* bias,
                       const uint16_t* R, int ldr, void* Y, int ldy, bool out_f32, int epi, int M, int N, int K,
                       int nt, hipStream_t s);
int launch_gemm_stream(const uint16_t* X, int ldx, const uint16_t* W, int ldw, const uint16_t* bias,
                       const uint16_t* R, int ldr, void* Y, int ldy, bool out_f32, int epi, float* ws, long ws_elems,
                       int M, int N, int K, int ntw, int S, bool wshuf, bool reduce, float epi_arg, hipStream_t s);
// Batch-1 decode GEMM whose input row is the residual row's RMSNorm, x = rmsnorm(h) * lnw, recomputed by every workgroup
// (no norm launch); workgroup (0, 0) stores the row to hout too (never h itself: the other workgroups are still reading
// h).  Pre-shuffled bf16 weights, epi none / silu, split-K into ws.
struct NormPro {
  const uint16_t* h;
  const uint16_t* lnw;
  uint16_t* hout;
  float eps;
  int D;
};
int launch_gemm_stream_norm(const uint16_t* W, const uint16_t* bias, void* Y, int ldy, int epi, float* ws,
                            long ws_elems, int N, int K, int ntw, int S, bool reduce, const NormPro& np,
                            hipStream_t s);
// decode GEMM whose workgroups hold whole K sums (gemm_wave.hip): M <= 64, N % 16 == 0, K % 128 == 0, pre-shuffled W; nt column tiles a
// workgroup (1 .. 4 up to 16 rows; ceil(M / 16) .. 8 beyond; even for gated pairs and rope).  np.h: one row, its norm prologue; ro.q:
// the QKV projection, rotated and written to q and the paged caches
struct RopeOut {
  uint16_t *q, *kc, *vc;
  const int32_t* pos;
  const float* cos_sin;
  const int64_t* slots;
  int H, Hkv, Dh, BS, max_pos;
  int64_t nslots;
};
// a lone sequence's attention left in parts (attn_decode_split_kernel, defer): o [parts][K], ml [parts][K / Dh][2], at most max_parts,
// cut by decode_lone_pages of ctx[0] tokens (max_blocks pages at most) over Hkv heads; o_proj's GEMM merges them (X none)
struct LoneMerge {
  const float *o, *ml;
  const int32_t* ctx;
  int max_blocks, Hkv, Dh, max_parts;
};
struct WaveGemm {
  const uint16_t* X;
  int ldx;
  const uint16_t *W, *bias, *R;
  int ldr;
  void* Y;
  int ldy, M, N, K;
  float epi_arg;
  NormPro np;
  RopeOut ro;
  LoneMerge mg;
};
int launch_gemm_wave(const WaveGemm& a, bool out_f32, int epi, int nt, hipStream_t st);
// decode GEMM with weight-only FP8 (e4m3 pre-shuffled tiles + per-row fp32 scale), bf16 activations
int launch_gemm_stream8(const uint16_t* X, int ldx, const uint8_t* W, const float* wscale, const uint16_t* bias,
                        const uint16_t* R, int ldr, void* Y, int ldy, bool out_f32, int epi, float* ws, long ws_elems,
                        int M, int N, int K, int ntw, int S, bool reduce, hipStream_t s);
// large-M GEMM on the pre-shuffled layout (256 x bn x 64 LDS-DMA tiles, 8 waves; split-K via ws)
// four-wave tile of 256 columns (gemm_w4.hip; tile code 4256 of launch_gemm_big): N % 256 == 0, K % 128 == 0; rows 128 ..
// 256 in steps of 32, 0: by the kernel's own rule
int launch_gemm_w4(const uint16_t* X, int ldx, const uint16_t* W, const uint16_t* bias, const uint16_t* R, int ldr,
                   void* Y, int ldy, bool out_f32, int epi, float* ws, int M, int N, int K, int S, int rows, int group_m,
                   float epi_arg, hipStream_t st);
// the same tile on token-major operands (weight gradients): Y [M, N] (+)= Xt^T . Wt, Xt [K, M], Wt [K, N]
int launch_gemm_w4_tn(const uint16_t* Xt, int ldx, const uint16_t* Wt, int ldw, const uint16_t* R, int ldr, void* Y,
                      int ldy, bool out_f32, int epi, int M, int N, int K, int group_m, hipStream_t st);
int gemm_big_group_m();  // grouped raster width of tall grids (XOT_GEMM_GROUP_M)
int launch_gemm_big(const uint16_t* X, int ldx, const uint16_t* W, const uint16_t* bias, const uint16_t* R, int ldr,
                    void* Y, int ldy, bool out_f32, int epi, float* ws, long ws_elems, int M, int N, int K, int bn,
                    int S, bool reduce, float epi_arg, hipStream_t s);
// B independent GEMMs Y_e = X_e . W_e^T (pre-shuffled W [B][N][K]; X_e = X + e*xbat, Y_e = Y + e*ybat)
// training-GEMM layouts (csrc/layout.hip): src [R, C] row-major with row stride ld
int launch_shuffle(const uint16_t* src, long ld, uint16_t* dst, int R, int C, hipStream_t s);
int launch_shuffle_t(const uint16_t* src, long ld, uint16_t* dst, int R, int C, hipStream_t s);
int launch_transpose(const uint16_t* src, long ld, uint16_t* dst, int R, int C, hipStream_t s);
int launch_gemm_kgroup(const uint16_t* X, int ldx, const uint16_t* W, uint16_t* Y, int ldy, bool resid,
                       const int* koff, int E, int M, int N, int K, hipStream_t st);
int launch_gemm_batched(const uint16_t* X, int ldx, long xbat, const uint16_t* W, void* Y, int ldy, long ybat,
                        bool out_f32, int B, int M, int N, int K, hipStream_t s);
// h += bias + sum of S fp32 split-K slabs [S][rows][D] (in place, bf16), out = rmsnorm(h) * w
void launch_splitk_resid_rmsnorm(const float* ws, int S, const uint16_t* bias, uint16_t* h, const uint16_t* w,
                                 uint16_t* out, int rows, int D, float eps, hipStream_t s);
// grouped expert GEMM on gemm_big tiles (bm = 128 or 256 rows per tile; large per-expert row counts)
int launch_gemm_moe_big(const uint16_t* X, int ldx, const uint16_t* W, void* Y, int ldy, bool out_f32, int epi,
                        const int* off, const int* gather, int E, int max_rows, int N, int K, int S, long ysplit,
                        int bm, float epi_arg, hipStream_t s);
// grouped decode GEMM of routed experts on pre-shuffled weights (gemm_group.hip); X has xrows rows.  Wsh: nsh shared experts of all
// max_rows tokens, one matrix [nsh N, K], or (sh_cols) [N, nsh K]; their slots are slot0 ...
int launch_gemm_group(const uint16_t* X, int ldx, int xrows, const uint16_t* W, void* Y, int ldy, bool out_f32, int epi, const int* off,
                      const int* gather, int E, int max_rows, int N, int K, int S, long ysplit, float epi_arg, const uint16_t* Wsh,
                      int nsh, bool sh_cols, int slot0, hipStream_t st);
// grouped GEMM over experts: rows of expert e are off[e]..off[e+1] (slot order), W is [E][N][K]
int launch_gemm_moe(const uint16_t* X, int ldx, const uint16_t* W, void* Y, int ldy, bool out_f32, int epi,
                    const int* off, const int* gather, int E, int max_rows, int N, int K, bool wshuf, int S,
                    long ysplit, float epi_arg, hipStream_t s);
void launch_splitk_silu(const float* ws, int S, int M, int N, uint16_t* y, hipStream_t s);
int launch_moe_combine_norm(const float* y, const int32_t* slot_of, const float* topw, uint16_t* h,
                            const uint16_t* lnw, uint16_t* out, int T, int k, int nsh, int D, int S, long ysplit, float eps,
                            hipStream_t s);
int launch_router_logits(const uint16_t* x, const uint16_t* w, float* out, int T, int E, int D, hipStream_t s);
void launch_moe_route(const float* logits, int T, int E, int k, float* topw, int32_t* topi, int32_t* slot_of,
                      int32_t* sorted_tok, int32_t* off, hipStream_t s);
void launch_moe_combine(const float* y, const int32_t* slot_of, const float* topw, uint16_t* h, int T, int k, int nsh,
                        int D, int S, long ysplit, hipStream_t s);
// DeepSeekMoE routing: method 0 greedy, 1 group max (V2 group_limited_greedy), 2 group top-2 sum (V3 noaux_tc)
// cnt: [E] int32 counters, zero on entry and left zero on exit
int launch_moe_route_ds(const float* logits, const float* bias, int T, int E, int k, int n_group, int topk_group,
                        int method, bool sigmoid, bool norm, float scale, int* cnt, float* topw, int32_t* topi,
                        int32_t* slot_of, int32_t* sorted_tok, int32_t* off, hipStream_t s);
// DeepSeek MLA: latent norm + rope + latent cache write (q_pe rotated in place), and the absorbed attention
int launch_mla_prep_slabs(const float* P, int S, long ss, int N, int nope, const uint16_t* kv_ln, uint16_t* q, long ldq,
                          const int32_t* pos, const float* cos_sin, const int64_t* slots, uint16_t* cache, int T, int H, int DL,
                          int DR, int max_pos, long nslots, float eps, hipStream_t s);
void launch_mla_prep(const uint16_t* ckv, long ldc, const uint16_t* kv_ln, uint16_t* q, long ldq, long qpe_off,
                     const int32_t* pos, const float* cos_sin, const int64_t* slots, uint16_t* cache, int T, int H,
                     int DL, int DR, int max_pos, long nslots, float eps, hipStream_t s);
int launch_mla_attn(const uint16_t* q_lat, const uint16_t* q_pe, long ldqpe, const uint16_t* cache,
                    const int32_t* block_tables, int max_blocks, const int32_t* cu_q, const int32_t* ctx_lens, int B,
                    int T, int H, int DL, int DR, uint16_t* out, float* ws_o, float* ws_ml, int pages_per_part,
                    int nparts, float scale, int num_pages, int wide, int even, hipStream_t s);
int launch_gemm_tiled(const uint16_t* X, int ldx, const uint16_t* W, int ldw, const uint16_t* bias,
                      const uint16_t* R, int ldr, void* Y, int ldy, bool out_f32, int epi, int M, int N, int K,
                      hipStream_t s);

// one unit of a decode step's attention for every KV head: pages first .. last of sequence b, one of its `parts` parts (0: none), the
// first of which has place `place`
struct __attribute__((aligned(32))) DecodePart {
  int b, first, last, parts, place, ctx, pad0, pad1;
};
// A part holds at most ppp pages, ppp at least MIN_PAGES (a page for each of a unit's four waves); the parts of a sequence are equal to a
// page, so they have at least half of that (5 pages: 3 + 2).  Over all KV heads there are at most B Hkv + UNITS units: one a sequence,
// and what cutting adds (two workgroups on each of 256 CUs).
constexpr int DECODE_MIN_PAGES = 4, DECODE_UNITS = 512;
// places of a plan: sum over the sequences of max(1, ceil(pages / ppp)) < B + total / ppp + 1, and ppp >= total Hkv / UNITS
inline int decode_split_places(int B, int Hkv, int max_blocks) {
  const int64_t wide = (int64_t)B * ((max_blocks + DECODE_MIN_PAGES - 1) / DECODE_MIN_PAGES);
  const int64_t n = (int64_t)B + DECODE_UNITS / Hkv;
  return (int)(n < wide ? n : wide);
}
// Pages of a part of a lone sequence, which every workgroup cuts by itself: 0.63 sqrt(pages), for a page costs 0.75 us and a further part
// to merge about 0.3 (8000 tokens in parts of 4 / 6 / 8 pages 19.1 / 16.9 / 16.0 us).
__device__ __forceinline__ int decode_lone_pages(int pages, int Hkv) {
  const int p = max(DECODE_MIN_PAGES, (int)(0.63f * sqrtf((float)pages) + 0.5f));
  return max(p, (pages * Hkv + DECODE_UNITS - 1) / DECODE_UNITS);
}
int launch_decode_plan(const int32_t* ctx_lens, int B, int Hkv, int Dh, int max_blocks, DecodePart* plan, hipStream_t s);
// ws_o [places][H][Dh], ws_ml [places][H][2], tickets [B][Hkv] (zero before and after); plan none: one sequence of ctx_lens[0] tokens,
// whose parts stay in ws_o / ws_ml with defer
int launch_attn_decode_split(const uint16_t* q, const uint16_t* kc, const uint16_t* vc, const int32_t* block_tables, int max_blocks,
                             const DecodePart* plan, int places, const int32_t* ctx_lens, int* tickets, uint16_t* out, float* ws_o,
                             float* ws_ml, int H, int Hkv, int Dh, float scale, int num_pages, bool nt, bool defer, hipStream_t s);
int launch_attn_decode(const uint16_t* q, const uint16_t* kc, const uint16_t* vc, const int32_t* block_tables,
                       int max_blocks, const int32_t* ctx_lens, uint16_t* out, float* ws_o, float* ws_ml, int B,
                       int H, int Hkv, int Dh, int pages_per_part, int nparts, float scale, int num_pages, int algo,
                       hipStream_t s);
int launch_attn_prefill(const uint16_t* q, const uint16_t* kc, const uint16_t* vc, const int32_t* block_tables,
                        int max_blocks, const int32_t* cu_q, const int32_t* ctx_lens, uint16_t* out, int B,
                        int max_qlen, int H, int Hkv, int Dh, float scale, int num_pages, int algo, hipStream_t s);

// causal self-attention for training (token-major Q / K / V slices, GQA); lse2 [B, H, L] fp32 (log2 domain);
// *t arguments are [B, heads, Dh, Lp] transposed images from launch_attn_train_transpose (zero past L)
int launch_attn_train_transpose(const uint16_t* x, long ldx, uint16_t* xt, int B, int L, int Lp, int n, int Dh,
                                hipStream_t s);
int launch_attn_train_fwd(const uint16_t* q, long ldq, const uint16_t* k, long ldk, const uint16_t* vt, int Lp,
                          uint16_t* o, long ldo, float* lse2, int B, int L, int H, int Hkv, int Dh, float scale,
                          bool causal, hipStream_t s);
int launch_attn_train_bwd(const uint16_t* q, long ldq, const uint16_t* k, long ldk, const uint16_t* v, long ldv,
                          const uint16_t* o, long ldo, const uint16_t* dout, long lddo, int Lp, const float* lse2,
                          float* delta, uint16_t* dq, long lddq, uint16_t* dk, long lddk, uint16_t* dv, long lddv,
                          float* ws, long ws_elems, int B, int L, int H, int Hkv, int Dh, float scale, hipStream_t s);

void launch_sample(const float* logits, long ld, int B, int V, const float* temps, int top_k,
                   const int64_t* seed_off, int32_t* out, uint32_t* cand_key, int32_t* cand_idx, hipStream_t s, int algo = -1);
int launch_topk_cand(const float* logits, long ld, int B, int V, int top_k, float* cval, int32_t* cidx, int kc,
                     hipStream_t s);
constexpr int SAMPLE_CAND_PER_ROW = 64 * 64;  // split path scratch: chunks x max top-k

void launch_ce_fwd(const void* x, bool x_f32, long ld, int T, int V, const int32_t* tgt, float* loss, float* lse,
                   hipStream_t s);
void launch_ce_bwd(const void* x, bool x_f32, long ld, int T, int V, const int32_t* tgt, const float* lse,
                   const float* gscale, uint16_t* dx, long ldd, hipStream_t s);
// multi-tensor sum of squares (gradient clipping): batches of up to SUMSQ_MAXT tensors passed by value
constexpr int SUMSQ_MAXT = 64;
struct SumsqBatch {
  const void* p[SUMSQ_MAXT];
  long n[SUMSQ_MAXT];
  int f32[SUMSQ_MAXT];
  int count;
};
int multi_sumsq_chunk();
long multi_sumsq_scratch(int nbatch, int maxc);  // floats of `part`
void launch_multi_sumsq(const SumsqBatch* batches, int nbatch, int maxc, float* part, float* out, hipStream_t s);
int launch_adamw_tiled(float* p, const void* g, bool g_f32, float* m, float* v, uint16_t* pb, uint16_t* ws,
                       uint16_t* wts, int N, int K, float lr, float b1, float b2, float eps, float wd, int step,
                       float gscale, hipStream_t s);
void launch_adamw(float* p, const void* g, bool g_f32, float* m, float* v, uint16_t* p_bf16, long n, float lr,
                  float b1, float b2, float eps, float wd, int step, float gscale, hipStream_t s);

}  // namespace xot
