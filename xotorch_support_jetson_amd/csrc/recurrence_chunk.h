// linear_recurrence over chunks of 16 tokens (recurrence_chunk.hip); arguments checked by linear_recurrence (mixers.hip).
#pragma once
#include <cstdint>

namespace xot {

// Decays per key channel that chunk_prep_k makes itself: the plain write's from a low-rank product, sigmoid(P[:, p_off : +rank] w^T + b)
// to the power of 1 / tau (w [H d, rank], A_log null), or the delta rule's exp(-exp(A_log) softplus(w + b)) of finished products w
// [T, >= H d], with sigmoid(P[:, p_off : +H]) as the write strengths.
struct DecaySource {
  const float* P;
  int ldp, p_off;
  const float *w, *b;
  int ldw;  // rank, or the row stride of the finished products
  float inv_tau;
  const float* A_log;
};

struct ChunkRecurrence {
  const float *q, *k, *v, *decay, *beta;  // beta: the delta rule's write strength, or (not delta) an input scale, may be null
  int ldq, ldk, ldv, dstride;             // dstride: decays of consecutive tokens (0: one fixed decay per head)
  float q_scale;
  float* state;
  const int *state_slots, *cu_q;
  int T, B, H, G, d, dv, dvin, longest;  // longest: tokens of the longest sequence, or (not known) what is taken for it
  bool known;
  bool chan, delta;  // a decay per key channel; the delta rule
  float *ws, *out;
  DecaySource src;  // (P null: decay and beta hold them)
};

// takes d 64 or 128, rows of q, k, the decays (chan) and the state on 16-byte boundaries
void chunk_recurrence(const ChunkRecurrence& a);
int64_t chunk_recurrence_ws(int64_t T, int64_t B, int64_t H, int64_t d, bool chan, bool delta, int64_t max_qlen);  // floats, at most 128 M

}  // namespace xot
