// online_seal.hpp — the InfLLM online seal on the device (the reference's
// P1.3c.4, cpp/src/online_seal_main.cpp:41-44): when a decode step seals a
// 32-token block, the representative of query head h is
// build_local_causal_representatives (cpp/src/selection.cpp:12-94) applied to
// that block alone, with the block's 32 keys (KV head h / G) and the 32
// decode queries of head h issued with those tokens, block_tokens 32, a local
// window and a top-k: the mean of the top-k keys ranked by the softmax mass
// they received from the block's queries.  Same arithmetic as the reference,
// bit for bit: sequential fp32 dots (no fused multiply-add; the including
// file is compiled with -ffp-contract=off), logits scaled, the row maximum,
// glibc's expf (expf_glibc.hpp), the denominator summed in key order,
// probabilities divided, each key's mass summed in query order, a stable
// descending rank (ties keep token order) and the chosen keys summed in rank
// order, divided by top-k.
//
// The decode queries live in a ring in HBM: the query of head h issued with
// the token at position p is kept at slot p % ring_tokens of
// ring[b][h][slot][128], written by the decode step that appends the token.
#pragma once

#include "expf_glibc.hpp"
#include "sa_device.hpp"
#include "sa_internal.hpp"

namespace sa {
namespace online {

constexpr int kT = kPageTokens;           // tokens of a sealed block
constexpr int kDim = kHeadDim;
constexpr int kQStride = kDim + 1;        // padded query rows (floats): no bank conflicts
constexpr int kKStride = kDim / 2 + 1;    // padded key rows (dwords of two FP16 values)
constexpr int kLStride = kT + 1;          // padded logit rows
// LDS floats the seal of one (sequence, query head, block) borrows
constexpr int kSmemFloats = kT * kQStride + kT * kKStride + kT * kLStride + 3 * kT;

struct Args {
  float* ring;          // [batch][query_heads][ring_tokens][128] decode queries
  int32_t ring_tokens;
  int32_t window;       // local causal window of the builder (>= 1)
  int32_t topk;         // keys averaged per representative (1..32)
  int32_t query_heads;
  float scale;          // 1 / sqrt(128), as the reference computes it
};

// Keep the decode query rows of heads [h0, h0 + heads) of sequence b for the
// token at position pos (ring slot pos % ring_tokens).  Any thread layout.
__device__ inline void store_queries(const Args& a, const float* query, int b, int h0, int heads, int64_t pos,
                                     int tid, int threads) {
  const int64_t slot = pos % a.ring_tokens;
  for (int e = tid; e < heads * kDim; e += threads) {
    const int h = h0 + e / kDim;
    const int d = e % kDim;
    a.ring[((static_cast<int64_t>(b) * a.query_heads + h) * a.ring_tokens + slot) * kDim + d] =
        query[(static_cast<int64_t>(b) * a.query_heads + h) * kDim + d];
  }
}

// Representative of one sealed block for query head h.  keys: the block's
// key row of its KV head for token 0 (token t at keys + t * token_elems);
// first_pos: the position of the block's token 0; rep: the representative's
// value of d = 0 (d at rep + d * rep_stride).  Every thread of the workgroup
// calls it (workgroup barriers inside); smem: kSmemFloats floats of LDS.
// Bound by its chain of latencies (two loads' round trips, the 128-step dots,
// then folds over 32 entries between barriers), not by bytes or arithmetic.
template <int kThreads>
__device__ inline void seal_head(const Args& a, int b, int h, const uint16_t* keys, int64_t token_elems,
                                 int64_t first_pos, float* rep, int64_t rep_stride, float* smem) {
  const int tid = threadIdx.x;
  float* qs = smem;                                                     // [32][129]
  uint32_t* ks = reinterpret_cast<uint32_t*>(smem + kT * kQStride);     // [32][65]
  float* ls = smem + kT * kQStride + kT * kKStride;                     // [32][33]
  float* received = ls + kT * kLStride;                                 // [32]
  float* row = received + kT;                                           // [32] max, then denominator
  int* order = reinterpret_cast<int*>(row + kT);                        // [32]

  const float* ring_h = a.ring + (static_cast<int64_t>(b) * a.query_heads + h) * a.ring_tokens * kDim;
  // every load of the queries and keys is issued before the first is used
  constexpr int kQLoads = kT * kDim / kThreads;
  constexpr int kKLoads = kT * kDim / 2 / kThreads;
  const int slot0 = static_cast<int>(first_pos % a.ring_tokens);
  float qv[kQLoads];
  uint32_t kv[kKLoads];
#pragma unroll
  for (int i = 0; i < kQLoads; ++i) {
    const int e = tid + i * kThreads;
    int slot = slot0 + e / kDim;  // the ring holds the whole block: at most one wrap
    if (slot >= a.ring_tokens) slot -= a.ring_tokens;
    qv[i] = ring_h[static_cast<int64_t>(slot) * kDim + e % kDim];
  }
#pragma unroll
  for (int i = 0; i < kKLoads; ++i) {
    const int e = tid + i * kThreads;
    kv[i] = *reinterpret_cast<const uint32_t*>(keys + e / (kDim / 2) * token_elems + 2 * (e % (kDim / 2)));
  }
#pragma unroll
  for (int i = 0; i < kQLoads; ++i) {
    const int e = tid + i * kThreads;
    qs[e / kDim * kQStride + e % kDim] = qv[i];
  }
#pragma unroll
  for (int i = 0; i < kKLoads; ++i) {
    const int e = tid + i * kThreads;
    ks[e / (kDim / 2) * kKStride + e % (kDim / 2)] = kv[i];
  }
  __syncthreads();

  // Pairs (query i, key j <= i): rows r and 31 - r together hold 33 of them,
  // so the 528 pairs are numbered with no gaps (a 32 x 32 grid would leave
  // half the lanes without a pair).
  auto pair = [](int e, int& i, int& j) {
    const int r = e / (kT + 1);
    const int c = e % (kT + 1);
    i = c <= r ? r : kT - 1 - r;
    j = c <= r ? c : c - r - 1;
  };
  constexpr int kPairs = kT * (kT + 1) / 2;

  // logits of query i over keys j in [i + 1 - window, i] (selection.cpp:36-48)
  for (int e = tid; e < kPairs; e += kThreads) {
    int i, j;
    pair(e, i, j);
    if (i - j >= a.window) continue;
    const float* q = qs + i * kQStride;
    const uint32_t* k = ks + j * kKStride;
    float dot = 0.0f;
#pragma unroll 16
    for (int w = 0; w < kDim / 2; ++w) {
      const uint32_t kw = k[w];
      dot = dot + q[2 * w] * lo_h2f(kw);
      dot = dot + q[2 * w + 1] * hi_h2f(kw);
    }
    ls[i * kLStride + j] = dot * a.scale;
  }
  __syncthreads();
  // The serial folds over a row or column of logits read all 32 entries first
  // (LDS reads in flight together) and skip those outside the window.  Each
  // fold's row index is opaque to the compiler, which would otherwise keep 32
  // lane masks from one fold to the next in scalar registers.
  const uint32_t window = static_cast<uint32_t>(a.window);
  auto in_window = [window](int back) { return static_cast<uint32_t>(back) < window; };  // 0 <= back < window
  auto opaque = [](int x) {
    asm("" : "+v"(x));
    return x;
  };
  if (tid < kT) {
    const int i = opaque(tid);
    float x[kT];
#pragma unroll
    for (int j = 0; j < kT; ++j) x[j] = ls[i * kLStride + j];
    float maximum = -__builtin_huge_valf();
#pragma unroll
    for (int j = 0; j < kT; ++j) maximum = in_window(i - j) ? fmaxf(maximum, x[j]) : maximum;
    row[i] = maximum;
  }
  __syncthreads();
  // exponentials (selection.cpp:51-52)
  for (int e = tid; e < kPairs; e += kThreads) {
    int i, j;
    pair(e, i, j);
    if (i - j >= a.window) continue;
    ls[i * kLStride + j] = expf_glibc(ls[i * kLStride + j] - row[i]);
  }
  __syncthreads();
  if (tid < kT) {  // denominators in key order (selection.cpp:53)
    const int i = opaque(tid);
    float x[kT];
#pragma unroll
    for (int j = 0; j < kT; ++j) x[j] = ls[i * kLStride + j];
    float denominator = 0.0f;
#pragma unroll
    for (int j = 0; j < kT; ++j) denominator = in_window(i - j) ? denominator + x[j] : denominator;
    row[i] = denominator;
  }
  __syncthreads();
  for (int e = tid; e < kPairs; e += kThreads) {
    int i, j;
    pair(e, i, j);
    if (i - j >= a.window) continue;
    ls[i * kLStride + j] = ls[i * kLStride + j] / row[i];
  }
  __syncthreads();
  if (tid < kT) {  // the mass key j received, in query order (selection.cpp:55-58)
    const int j = opaque(tid);
    float x[kT];
#pragma unroll
    for (int i = 0; i < kT; ++i) x[i] = ls[i * kLStride + j];
    float r = 0.0f;
#pragma unroll
    for (int i = 0; i < kT; ++i) r = in_window(i - j) ? r + x[i] : r;
    received[j] = r;
  }
  __syncthreads();
  if (tid < kT) {  // stable descending rank (selection.cpp:71-76)
    const int j = tid;
    const float rj = received[j];
    float x[kT];
#pragma unroll
    for (int k = 0; k < kT; ++k) x[k] = received[k];
    int rank = 0;
#pragma unroll
    for (int k = 0; k < kT; ++k) rank += (mass_before(x[k], rj) || (k < j && mass_tied(x[k], rj))) ? 1 : 0;
    order[rank] = j;
  }
  __syncthreads();
  for (int d = tid; d < kDim; d += kThreads) {  // top-k keys in rank order (selection.cpp:80-89)
    float value = 0.0f;
    for (int r = 0; r < a.topk; ++r) {
      const uint32_t kw = ks[order[r] * kKStride + d / 2];
      value = value + ((d & 1) ? hi_h2f(kw) : lo_h2f(kw));
    }
    rep[d * rep_stride] = value / static_cast<float>(a.topk);
  }
  __syncthreads();  // the LDS is free again
}

}  // namespace online
}  // namespace sa
