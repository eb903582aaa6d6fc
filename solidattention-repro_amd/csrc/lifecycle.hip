// lifecycle.hip — decode-token append, 32-token seal with mean-key
// representative, page gather, synthetic data and the output consumer
// (gfx950).
//
// Append follows the reference's append_fp16_kv (cpp/src/qwen_layer_main.cpp
// :270-281): one token's K and V, converted fp32 -> FP16 round-to-nearest-
// even, written at the token's slot of the token-major page.  The seal
// follows the tail lifecycle of cpp/src/kv_lifecycle_main.cpp:92-113: while
// the tail holds at least local_tokens + 32 tokens the oldest tail block is
// sealed and the generation advances.  With paging, "erase" is only the
// sealed-count advance: the block stays in its page.  The representative is
// the mean key of the block (sum of its 32 keys in token order, divided by
// 32), i.e. the reference's build_local_causal_representatives with window 1
// and top-k 32 (cpp/src/selection.cpp:12-94), bit-exact; or, for the InfLLM
// online seal, the builder itself over the sealed block and the decode
// queries issued with its tokens (online_seal.hpp).
#include "online_seal.hpp"
#include "sa_device.hpp"
#include "sa_internal.hpp"

namespace sa {
namespace {

constexpr int D = kHeadDim;
constexpr int kThreads = 256;

struct Params {
  uint16_t* pool;
  const int32_t* table;
  int32_t* seq_len;
  int32_t* sealed;
  int32_t* generation;
  float* reps;
  int32_t* status;
  const float* k;
  const float* v;
  const uint16_t* k16;
  const uint16_t* v16;
  int64_t num_pages;
  int64_t page_elems;
  int32_t token_elems;
  int32_t width;          // kv_heads * head_dim
  int32_t table_stride;
  int32_t rep_heads;
  int32_t rep_stride;
  int32_t group;
  int32_t local_tokens;
  int32_t append;
  int32_t head_dim;       // D, or another multiple of 8 (not the online seal)
  const float* query;     // online seal: this step's decode queries [batch][query_heads][D]
  online::Args online;
};

__device__ inline int64_t table_page(const Params& p, int b, int64_t logical) {
  if (logical < 0 || logical >= p.table_stride) return -1;
  const int64_t page = p.table[static_cast<int64_t>(b) * p.table_stride + logical];
  return (page >= 0 && page < p.num_pages) ? page : -1;
}

__global__ __launch_bounds__(kThreads) void append_seal_kernel(const Params p) {
  const int b = blockIdx.x;
  const int tid = threadIdx.x;
  int64_t len = p.seq_len[b];

  if (p.append) {
    const int64_t page = table_page(p, b, len / kPageTokens);
    if (page < 0) {
      if (tid == 0) flag_status(p.status, kStatusCapacity);
      return;
    }
    uint16_t* dst = p.pool + page * p.page_elems + (len % kPageTokens) * p.token_elems;
    const int64_t src = static_cast<int64_t>(b) * p.width;
    // 4 consecutive values per thread and half: 8-byte stores, coalesced.
    for (int e = tid * 4; e < p.width; e += kThreads * 4) {
      ushort4 kk, vv;
      if (p.k16) {
        kk = *reinterpret_cast<const ushort4*>(p.k16 + src + e);
        vv = *reinterpret_cast<const ushort4*>(p.v16 + src + e);
      } else {
        const float4 kf = *reinterpret_cast<const float4*>(p.k + src + e);
        const float4 vf = *reinterpret_cast<const float4*>(p.v + src + e);
        kk = make_ushort4(f2h_rne(kf.x), f2h_rne(kf.y), f2h_rne(kf.z), f2h_rne(kf.w));
        vv = make_ushort4(f2h_rne(vf.x), f2h_rne(vf.y), f2h_rne(vf.z), f2h_rne(vf.w));
      }
      *reinterpret_cast<ushort4*>(dst + e) = kk;
      *reinterpret_cast<ushort4*>(dst + p.width + e) = vv;
    }
    len += 1;
    // The seal below may read the token just written by other threads.
    __syncthreads();
    if (tid == 0) p.seq_len[b] = static_cast<int32_t>(len);
  }

  int64_t s = p.sealed[b];
  int added = 0;
  while (len >= (s + 1) * kPageTokens + p.local_tokens) {
    const int64_t page = s < p.rep_stride ? table_page(p, b, s) : -1;
    if (page < 0) {
      if (tid == 0) flag_status(p.status, kStatusCapacity);
      break;
    }
    const uint16_t* src = p.pool + page * p.page_elems;
    const int hd = p.head_dim;
    for (int o = tid; o < p.width; o += kThreads) {  // o = kv_head * head_dim + d
      float sum = 0.0f;
#pragma unroll 8
      for (int t = 0; t < kPageTokens; ++t) sum = sum + h2f(src[t * p.token_elems + o]);
      const float rep = sum / static_cast<float>(kPageTokens);
      const int g = o / hd;
      const int d = o % hd;
      // group == 1 for per-KV-head representatives; otherwise every query
      // head of the group receives the (identical) mean key.
      for (int j = 0; j < p.group; ++j)
        p.reps[((static_cast<int64_t>(b) * p.rep_heads + g * p.group + j) * hd + d) * p.rep_stride + s] =
            rep;
    }
    ++s;
    ++added;
  }
  if (tid == 0) {
    p.sealed[b] = static_cast<int32_t>(s);
    if (p.generation) p.generation[b] += added;
  }
}

// ---- append + InfLLM online seal ------------------------------------------------
// Workgroup (query head h, sequence b) appends the token of h's KV head (the
// group's workgroups write the same bytes, so that each reads only what it
// wrote), keeps head h's query in the ring and, where the tail rule seals a
// block, writes head h's representative of it.  A seal is a chain of
// latencies (8-20 us a head); with one workgroup for a sequence's heads in
// turn a step that seals took 308-326 us at 16 heads, with a workgroup per
// head 15-16 us (4 sequences of 4-8K tokens; a step that seals nothing 4.5 us
// either way).
//
// The counters move only once every workgroup of the sequence has read them:
// the last of them to arrive at arrive[b] (zero between launches) writes
// them, or, for a caller without counters (arrive null), online_commit_kernel
// behind this launch.
constexpr int kOnlineThreads = 512;

// Sealed blocks after the tail rule has run on `len` tokens from block s on
// (it stops at a block without a representative slot or a page: *full).
__device__ inline int64_t sealed_after(const Params& p, int b, int64_t len, int64_t s, bool* full) {
  while (len >= (s + 1) * kPageTokens + p.local_tokens) {
    if (s >= p.rep_stride || table_page(p, b, s) < 0) {
      *full = true;
      break;
    }
    ++s;
  }
  return s;
}

__global__ __launch_bounds__(kOnlineThreads) void append_seal_online_kernel(const Params p, int32_t* arrive) {
  const int h = blockIdx.x;
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  __shared__ float smem[online::kSmemFloats];
  const int64_t pos = p.seq_len[b];
  const int64_t s0 = p.sealed[b];
  const int64_t page = table_page(p, b, pos / kPageTokens);
  int arrived = -1;
  if (arrive) {
    // every wave reads the counters for itself: all of them have them in
    // registers before the workgroup counts as arrived
    asm volatile("" ::"s"(s0), "s"(page) : "memory");
    __syncthreads();
    if (tid == 0) arrived = __hip_atomic_fetch_add(arrive + b, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const bool last = arrived == static_cast<int>(gridDim.x) - 1;  // (thread 0)
  if (page < 0) {
    if (h == 0 && tid == 0) flag_status(p.status, kStatusCapacity);
    if (last) __hip_atomic_store(arrive + b, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  const int g = h / (p.online.query_heads / (p.width / D));
  if (tid < kWave) {  // 4 consecutive values per lane: K in lanes 0..31, V in 32..63
    const int is_v = tid / 32;
    const int e = tid % 32 * 4;
    const float4 f = *reinterpret_cast<const float4*>((is_v ? p.v : p.k) + static_cast<int64_t>(b) * p.width + g * D + e);
    *reinterpret_cast<ushort4*>(p.pool + page * p.page_elems + (pos % kPageTokens) * p.token_elems + is_v * p.width +
                                g * D + e) = make_ushort4(f2h_rne(f.x), f2h_rne(f.y), f2h_rne(f.z), f2h_rne(f.w));
  }
  online::store_queries(p.online, p.query, b, h, 1, pos, tid, kOnlineThreads);
  __syncthreads();  // the token and its query, written by other waves, before the seal reads them
  bool full = false;
  const int64_t s1 = sealed_after(p, b, pos + 1, s0, &full);
  for (int64_t s = s0; s < s1; ++s)
    online::seal_head<kOnlineThreads>(p.online, b, h, p.pool + table_page(p, b, s) * p.page_elems + g * D,
                                      p.token_elems, s * kPageTokens,
                                      p.reps + (static_cast<int64_t>(b) * p.rep_heads + h) * D * p.rep_stride + s,
                                      p.rep_stride, smem);
  if (full && h == 0 && tid == 0) flag_status(p.status, kStatusCapacity);
  if (last) {
    p.seq_len[b] = static_cast<int32_t>(pos + 1);
    p.sealed[b] = static_cast<int32_t>(s1);
    if (p.generation) p.generation[b] += static_cast<int32_t>(s1 - s0);
    __hip_atomic_store(arrive + b, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The counters after append_seal_online_kernel without arrival counters: one
// thread per sequence.
__global__ __launch_bounds__(kWave) void online_commit_kernel(const Params p, int batch) {
  const int b = blockIdx.x * kWave + threadIdx.x;
  if (b >= batch) return;
  const int64_t pos = p.seq_len[b];
  if (table_page(p, b, pos / kPageTokens) < 0) return;
  const int64_t s0 = p.sealed[b];
  bool full = false;
  const int64_t s1 = sealed_after(p, b, pos + 1, s0, &full);
  p.seq_len[b] = static_cast<int32_t>(pos + 1);
  p.sealed[b] = static_cast<int32_t>(s1);
  if (p.generation) p.generation[b] += static_cast<int32_t>(s1 - s0);
}

// ---- bulk seal (no append): a prefill's whole pages sealed at once ----------
// The tail rule of append_seal_kernel seals blocks sealed, sealed + 1, ...
// while seq_len >= (block + 1) * 32 + local_tokens, and stops at the first
// block without a representative slot or a page (a capacity error).  The
// bulk form computes the same block range up front: the last block to seal
// from seq_len, the stopping block by a scan of the table.  Workgroup
// (chunk, KV head, sequence) sums kSealBlocks consecutive blocks of one KV
// head; a second launch of one wave per sequence commits sealed and
// generation, so that no workgroup reads a counter another has moved.
// 32 blocks per workgroup: the representatives leave as whole 128-byte lines
// (64 sequences of 16K tokens, 2.15 GB of keys and 134 MB written: 16 blocks
// 482 us, 32 blocks 456 us; KV heads as the fastest grid index 480 and 473 us).
// With fewer workgroups of 32 than compute units, 16 blocks: the seal is then
// as long as one workgroup (14.3 us against 14.5, one draw's 16.3 against 17.0).
constexpr int kSealPieces = D / 8;  // 16-byte pieces of one head's key row

// Blocks sealed once the tail rule has run to its end, ignoring capacity.
__device__ inline int64_t seal_target(int64_t len, int64_t local, int64_t s0) {
  if (len < local) return s0;
  const int64_t t = (len - local) / kPageTokens;
  return t > s0 ? t : s0;
}

// The first block of [from, to) that cannot be sealed (no representative
// slot or no page), or `to`; strided over `threads` threads, the caller
// takes the minimum.
__device__ inline int64_t first_unsealable(const Params& p, int b, int64_t from, int64_t to, int tid, int threads) {
  for (int64_t s = from + tid; s < to; s += threads)
    if (s >= p.rep_stride || table_page(p, b, s) < 0) return s;
  return to;
}

template <int kSealBlocks>
__global__ __launch_bounds__(kSealBlocks * kSealPieces) void seal_blocks_kernel(const Params p) {
  constexpr int kSealThreads = kSealBlocks * kSealPieces;  // one per (block, piece)
  const int g = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x;
  const int64_t s0 = p.sealed[b];
  const int64_t target = seal_target(p.seq_len[b], p.local_tokens, s0);
  const int64_t first = s0 + static_cast<int64_t>(blockIdx.x) * kSealBlocks;
  if (first >= target) return;
  __shared__ int32_t s_stop;
  __shared__ float tile[D][kSealBlocks + 1];
  // blocks past a capacity error stay unsealed, as in the tail rule
  const int64_t end = target < first + kSealBlocks ? target : first + kSealBlocks;
  if (tid == 0) s_stop = static_cast<int32_t>(end - first);
  __syncthreads();
  const int64_t bad = first_unsealable(p, b, s0, end, tid, kSealThreads);
  if (bad < end) atomicMin(&s_stop, static_cast<int32_t>(bad > first ? bad - first : 0));
  __syncthreads();
  const int n = s_stop;
  if (n <= 0) return;

  // thread = (block j, 16-byte piece q of head g's key row); 32 loads in
  // flight, then the 32 keys summed in token order
  const int j = tid / kSealPieces, q = tid % kSealPieces;
  if (j < n) {
    const int64_t page = table_page(p, b, first + j);
    const uint16_t* src = p.pool + page * p.page_elems + g * D + q * 8;
    uint4 w[kPageTokens];
#pragma unroll
    for (int t = 0; t < kPageTokens; ++t) w[t] = load_stream16(src + static_cast<int64_t>(t) * p.token_elems);
    float sum[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[i] = 0.0f;
#pragma unroll
    for (int t = 0; t < kPageTokens; ++t) {
      const uint32_t h[4] = {w[t].x, w[t].y, w[t].z, w[t].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sum[2 * i] = sum[2 * i] + lo_h2f(h[i]);
        sum[2 * i + 1] = sum[2 * i + 1] + hi_h2f(h[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) tile[q * 8 + i][j] = sum[i] / static_cast<float>(kPageTokens);
  }
  __syncthreads();
  // rows d of the representative: kSealBlocks consecutive floats each
  for (int e = tid; e < D * kSealBlocks; e += kSealThreads) {
    const int d = e / kSealBlocks, jj = e % kSealBlocks;
    if (jj >= n) continue;
    const float rep = tile[d][jj];
    for (int r = 0; r < p.group; ++r)
      p.reps[((static_cast<int64_t>(b) * p.rep_heads + g * p.group + r) * D + d) * p.rep_stride + first + jj] = rep;
  }
}

// The bulk seal at a head_dim other than 128: thread = (block j, 16-byte
// piece q of head g's key row) with head_dim / 8 pieces and 256 / pieces
// blocks per workgroup (the row tile in dynamic LDS: head_dim x (blocks + 1)
// floats), the same sums in token order and the same capacity rule as
// seal_blocks_kernel.
__global__ __launch_bounds__(kThreads) void seal_blocks_any_kernel(const Params p, int blocks_per_wg) {
  extern __shared__ float any_tile[];  // [head_dim][blocks_per_wg + 1]
  const int g = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x;
  const int hd = p.head_dim;
  const int pieces = hd / 8;
  const int64_t s0 = p.sealed[b];
  const int64_t target = seal_target(p.seq_len[b], p.local_tokens, s0);
  const int64_t first = s0 + static_cast<int64_t>(blockIdx.x) * blocks_per_wg;
  if (first >= target) return;
  __shared__ int32_t s_stop;
  const int64_t end = target < first + blocks_per_wg ? target : first + blocks_per_wg;
  if (tid == 0) s_stop = static_cast<int32_t>(end - first);
  __syncthreads();
  const int64_t bad = first_unsealable(p, b, s0, end, tid, kThreads);
  if (bad < end) atomicMin(&s_stop, static_cast<int32_t>(bad > first ? bad - first : 0));
  __syncthreads();
  const int n = s_stop;
  if (n <= 0) return;
  const int tile_stride = blocks_per_wg + 1;
  const int j = tid / pieces, q = tid % pieces;
  if (j < n) {
    const int64_t page = table_page(p, b, first + j);
    const uint16_t* src = p.pool + page * p.page_elems + static_cast<int64_t>(g) * hd + q * 8;
    uint4 w[kPageTokens];
#pragma unroll
    for (int t = 0; t < kPageTokens; ++t) w[t] = load_stream16(src + static_cast<int64_t>(t) * p.token_elems);
    float sum[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sum[i] = 0.0f;
#pragma unroll
    for (int t = 0; t < kPageTokens; ++t) {
      const uint32_t h[4] = {w[t].x, w[t].y, w[t].z, w[t].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sum[2 * i] = sum[2 * i] + lo_h2f(h[i]);
        sum[2 * i + 1] = sum[2 * i + 1] + hi_h2f(h[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) any_tile[(q * 8 + i) * tile_stride + j] = sum[i] / static_cast<float>(kPageTokens);
  }
  __syncthreads();
  for (int e = tid; e < hd * blocks_per_wg; e += kThreads) {
    const int d = e / blocks_per_wg, jj = e % blocks_per_wg;
    if (jj >= n) continue;
    const float rep = any_tile[d * tile_stride + jj];
    for (int r = 0; r < p.group; ++r)
      p.reps[((static_cast<int64_t>(b) * p.rep_heads + g * p.group + r) * hd + d) * p.rep_stride + first + jj] = rep;
  }
}

// One wave per sequence: the counters after the bulk seal.
__global__ __launch_bounds__(kWave) void seal_commit_kernel(const Params p) {
  const int b = blockIdx.x;
  const int lane = threadIdx.x;
  const int64_t s0 = p.sealed[b];
  const int64_t target = seal_target(p.seq_len[b], p.local_tokens, s0);
  int64_t stop = first_unsealable(p, b, s0, target, lane, kWave);
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    const int64_t o = __shfl_xor(stop, off, kWave);
    stop = o < stop ? o : stop;
  }
  if (lane == 0) {
    if (stop < target) flag_status(p.status, kStatusCapacity);
    p.sealed[b] = static_cast<int32_t>(stop);
    if (p.generation) p.generation[b] += static_cast<int32_t>(stop - s0);
  }
}

__global__ __launch_bounds__(kThreads) void gather_pages_kernel(const uint4* pool, int64_t page_vecs,
                                                                int64_t num_pages, const int32_t* pages,
                                                                uint4* out, int32_t* status) {
  const int i = blockIdx.y;
  const int64_t page = pages[i];
  if (page < 0 || page >= num_pages) {
    if (threadIdx.x == 0 && blockIdx.x == 0) flag_status(status, kStatusBadPage);
    return;
  }
  const uint4* src = pool + page * page_vecs;
  uint4* dst = out + static_cast<int64_t>(i) * page_vecs;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; e < page_vecs;
       e += static_cast<int64_t>(gridDim.x) * kThreads)
    dst[e] = src[e];
}

// A read-only pass over the bytes one decode step reads for each (sequence,
// KV head): the fp32 representative rows of its sealed blocks, the K/V
// slices of its selected pages and the K/V of its unsealed tail.  Nothing is
// computed but an XOR of every 32-bit word read (one value per (sequence, KV
// head), so that no load is dead).  It times the memory system on the decode
// step's own access pattern, the reference point for the attention kernels'
// bandwidth.  Workgroup (h, b) as in the decode-step kernels; 8 waves.
constexpr int kReadThreads = 512;
constexpr int kReadWaves = kReadThreads / kWave;

__global__ __launch_bounds__(kReadThreads) void read_step_bytes_kernel(const ReadStepLaunch p) {
  __shared__ uint32_t red[kReadWaves];
  const int h = blockIdx.x, b = blockIdx.y;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  uint32_t x = 0;
  const int64_t sealed = p.sealed[b];
  const int64_t len = p.seq_len[b];
  if (sealed < 0 || sealed > p.table_stride || len < sealed * kPageTokens ||
      len > static_cast<int64_t>(p.table_stride) * kPageTokens) {
    if (tid == 0) flag_status(p.status, kStatusBadLength);
    return;
  }

  // representative rows: rep heads h, h + kv_heads, ...; wave w takes rows
  // d = w + 8 u, 16 loads in flight per lane
  const int64_t quads = sealed / 4;
  for (int r = h; r < p.rep_heads; r += p.kv_heads) {
    const float* rows = p.reps + (static_cast<int64_t>(b) * p.rep_heads + r) * D * p.rep_stride;
    for (int64_t j = lane; j < quads; j += kWave) {
      u32x4_t v[D / kReadWaves];
#pragma unroll
      for (int u = 0; u < D / kReadWaves; ++u)
        v[u] = __builtin_nontemporal_load(
            reinterpret_cast<const u32x4_t*>(rows + static_cast<int64_t>(wave + kReadWaves * u) * p.rep_stride) + j);
#pragma unroll
      for (int u = 0; u < D / kReadWaves; ++u) x ^= v[u][0] ^ v[u][1] ^ v[u][2] ^ v[u][3];
    }
    const int rem = static_cast<int>(sealed % 4);
    if (tid < D * rem) {
      const int d = tid / rem, w = tid % rem;
      x ^= __float_as_uint(rows[static_cast<int64_t>(d) * p.rep_stride + 4 * quads + w]);
    }
  }

  // selected pages: wave w takes list entries w + 8 i; its lanes resolve 64
  // entries at a time (id, then page), then every lane reads 16 of the
  // page's 1024 16-byte pieces of head h (64 segments of 256 bytes: token
  // t = segment / 2, K or V = segment % 2)
  const int per_sel = p.kv_heads / p.select_groups;
  const int64_t list = static_cast<int64_t>(b) * p.select_groups + h / per_sel;
  const int count = min(p.counts[list], p.sel_stride);
  const int32_t* ids = p.selected + list * p.sel_stride;
  const int32_t* table = p.table + static_cast<int64_t>(b) * p.table_stride;
  const int64_t tok_vecs = 2 * p.kv_heads * D * 2 / 16;  // 16-byte pieces per token row
  const int64_t page_vecs = kPageTokens * tok_vecs;
  const u32x4_t* pool = reinterpret_cast<const u32x4_t*>(p.pool);
  for (int first = wave; first < count; first += kReadWaves * kWave) {
    const int mine = first + kReadWaves * lane;
    int64_t page = -1;
    if (mine < count) {
      const int blk = ids[mine];
      if (blk < 0 || blk >= sealed) {
        flag_status(p.status, kStatusBadBlock);
      } else {
        page = table[blk];
        if (page < 0 || page >= p.num_pages) {
          flag_status(p.status, kStatusBadPage);
          page = -1;
        }
      }
    }
    const int n = min(kWave, (count - first + kReadWaves - 1) / kReadWaves);
    for (int i = 0; i < n; ++i) {
      const int64_t pg = __shfl(page, i, kWave);
      if (pg < 0) continue;
      const u32x4_t* base = pool + pg * page_vecs + h * (D * 2 / 16);
      u32x4_t v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int piece = j * kWave + lane;
        const int seg = piece / 16;
        v[j] = __builtin_nontemporal_load(base + (seg / 2) * tok_vecs + (seg % 2) * (tok_vecs / 2) + piece % 16);
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) x ^= v[j][0] ^ v[j][1] ^ v[j][2] ^ v[j][3];
    }
  }

  // the unsealed tail: 32 pieces (K then V of head h) per token
  const int64_t tail = len - sealed * kPageTokens;
  for (int64_t i = tid; i < tail * 32; i += kReadThreads) {
    const int64_t t = sealed * kPageTokens + i / 32;
    const int q = static_cast<int>(i % 32);
    const int64_t page = table[t / kPageTokens];
    if (page < 0 || page >= p.num_pages) {
      flag_status(p.status, kStatusBadPage);
      continue;
    }
    const u32x4_t v = pool[page * page_vecs + (t % kPageTokens) * tok_vecs + (q / 16) * (tok_vecs / 2) +
                           h * (D * 2 / 16) + q % 16];
    x ^= v[0] ^ v[1] ^ v[2] ^ v[3];
  }

#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) x ^= __shfl_xor(x, off, kWave);
  if (lane == 0) red[wave] = x;
  __syncthreads();
  if (tid == 0) {
    uint32_t t = 0;
#pragma unroll
    for (int w = 0; w < kReadWaves; ++w) t ^= red[w];
    p.out[static_cast<int64_t>(b) * p.kv_heads + h] = t;
  }
}

// Pages whose ids travel in the kernel arguments (no device-side list):
// page i of the launch goes to out + i * page_vecs; out may be pinned host
// memory (seal writeback staging), written through its device mapping.
struct PageIdsArg {
  int32_t ids[kPagesPerHostCopy];
};

// A few workgroups, each copying whole pages in turn: the copy runs beside
// the decode kernels and is bound by the host link, so it holds only a few
// compute units (every workgroup of a grid sized to the pages would sit on
// a CU for the length of its link transfer).
constexpr int kHostCopyGroups = 16;

__global__ __launch_bounds__(kThreads) void pages_to_host_kernel(const uint4* pool, int64_t page_vecs, int count,
                                                                 const PageIdsArg pages, uint4* out) {
  for (int i = blockIdx.x; i < count; i += gridDim.x) {
    const uint4* src = pool + static_cast<int64_t>(pages.ids[i]) * page_vecs;
    uint4* dst = out + static_cast<int64_t>(i) * page_vecs;
    for (int64_t e = threadIdx.x; e < page_vecs; e += kThreads) dst[e] = src[e];
  }
}

__global__ __launch_bounds__(kThreads) void fill_synthetic_f16_kernel(uint16_t* dst, int64_t count,
                                                                      uint64_t seed_mixed,
                                                                      uint64_t first) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < count;
       i += static_cast<int64_t>(gridDim.x) * kThreads)
    dst[i] = f2h_rne(synth_normal(seed_mixed, first + static_cast<uint64_t>(i)));
}

__global__ __launch_bounds__(kThreads) void fill_synthetic_f32_kernel(float* dst, int64_t count,
                                                                      uint64_t seed_mixed,
                                                                      uint64_t first) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < count;
       i += static_cast<int64_t>(gridDim.x) * kThreads)
    dst[i] = synth_normal(seed_mixed, first + static_cast<uint64_t>(i));
}

// C1.4 consumer: a serial weighted checksum, the reference's consume_attention
// (cpp/src/cuda_backend.cpp:160-168).  One lane, sequential order.
__global__ void consume_checksum_kernel(const float* input, int32_t elements, float* checksum) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  float value = 0.0f;
  for (int i = 0; i < elements; ++i)
    value = value + input[i] * (1.0f + static_cast<float>(i % 17) * 0.001f);
  checksum[0] = value;
}

// Miss-correction fill from pinned host memory mapped into the device
// address space: one workgroup-row per missing page reads its 128 KiB over
// PCIe with 16-byte loads and writes the slot.  One launch replaces one
// hipMemcpyAsync per page.
__global__ __launch_bounds__(kThreads) void fill_from_host_kernel(uint4* pool, int64_t page_vecs, int64_t num_pages,
                                                                  const int32_t* dst_pages, const uint4* src,
                                                                  int64_t src_total, const int64_t* src_blocks,
                                                                  int32_t* status) {
  const int i = blockIdx.y;
  const int64_t page = dst_pages[i];
  const int64_t blk = src_blocks[i];
  if (page < 0 || page >= num_pages || blk < 0 || blk >= src_total) {
    if (threadIdx.x == 0 && blockIdx.x == 0) flag_status(status, kStatusBadPage);
    return;
  }
  const uint4* s = src + blk * page_vecs;
  uint4* d = pool + page * page_vecs;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; e < page_vecs;
       e += static_cast<int64_t>(gridDim.x) * kThreads)
    d[e] = s[e];
}

// C0 transport smoke transform: out[i] = in[i] ^ mask (the reference's
// kv_transform, cpp/src/cuda_backend.cpp:40-46), 16 bytes per lane.
__global__ __launch_bounds__(kThreads) void xor_bytes_kernel(const uint8_t* in, uint8_t* out, uint64_t bytes,
                                                             uint8_t mask) {
  const uint32_t m4 = 0x01010101u * mask;
  const uint64_t vecs = bytes / 16;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x; i < vecs;
       i += static_cast<uint64_t>(gridDim.x) * kThreads) {
    uint4 v = reinterpret_cast<const uint4*>(in)[i];
    v.x ^= m4;
    v.y ^= m4;
    v.z ^= m4;
    v.w ^= m4;
    reinterpret_cast<uint4*>(out)[i] = v;
  }
  if (blockIdx.x == 0)
    for (uint64_t i = vecs * 16 + threadIdx.x; i < bytes; i += kThreads) out[i] = in[i] ^ mask;
}

int grid_for(int64_t items, int per_block) {
  const int64_t g = (items + per_block - 1) / per_block;
  return static_cast<int>(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}

}  // namespace

hipError_t launch_append_seal(const LifecycleLaunch& l, hipStream_t stream) {
  Params p{};
  p.pool = l.pool;
  p.table = l.table;
  p.seq_len = l.seq_len;
  p.sealed = l.sealed;
  p.generation = l.generation;
  p.reps = l.reps;
  p.status = l.status;
  p.k = l.k;
  p.v = l.v;
  p.k16 = l.k16;
  p.v16 = l.v16;
  p.num_pages = l.num_pages;
  p.head_dim = general_head_dim(l.head_dim) ? l.head_dim : D;
  p.token_elems = 2 * l.kv_heads * p.head_dim;
  p.page_elems = static_cast<int64_t>(kPageTokens) * p.token_elems;
  p.width = l.kv_heads * p.head_dim;
  p.table_stride = l.table_stride;
  p.rep_heads = l.rep_heads;
  p.rep_stride = l.rep_stride;
  p.group = l.rep_heads == l.kv_heads ? 1 : l.query_heads / l.kv_heads;
  p.local_tokens = l.local_tokens;
  p.append = l.append;
  if (p.head_dim != D) {
    // another head_dim (no ring: checked by the API): a decode step's append
    // and seal in one workgroup per sequence; the bulk seal spread over
    // blocks and KV heads
    if (l.ring) return hipErrorInvalidValue;
    if (l.append) {
      hipLaunchKernelGGL(append_seal_kernel, dim3(l.batch), dim3(kThreads), 0, stream, p);
    } else {
      const int per_wg = kThreads / (p.head_dim / 8);  // head_dim <= 512: at least 4
      const int64_t blocks = l.table_stride < l.rep_stride ? l.table_stride : l.rep_stride;
      const dim3 grid(static_cast<unsigned>((blocks + per_wg - 1) / per_wg), l.kv_heads, l.batch);
      const size_t smem = static_cast<size_t>(p.head_dim) * (per_wg + 1) * sizeof(float);
      hipLaunchKernelGGL(seal_blocks_any_kernel, grid, dim3(kThreads), smem, stream, p, per_wg);
      if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
      hipLaunchKernelGGL(seal_commit_kernel, dim3(l.batch), dim3(kWave), 0, stream, p);
    }
  } else if (l.ring) {
    p.query = l.query;
    p.online = online::Args{l.ring, l.ring_tokens, l.window, l.topk, l.query_heads, l.seal_scale};
    hipLaunchKernelGGL(append_seal_online_kernel, dim3(l.query_heads, l.batch), dim3(kOnlineThreads), 0, stream, p,
                       l.arrive);
    if (!l.arrive) {
      if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
      hipLaunchKernelGGL(online_commit_kernel, dim3((l.batch + kWave - 1) / kWave), dim3(kWave), 0, stream, p, l.batch);
    }
  } else if (!l.append) {
    // bulk seal: every block of a sequence's range in its own workgroup
    const int64_t blocks = l.table_stride < l.rep_stride ? l.table_stride : l.rep_stride;
    const int64_t wide = (blocks + 31) / 32 * l.kv_heads * l.batch;
    if (wide >= compute_units()) {
      const dim3 grid(static_cast<unsigned>((blocks + 31) / 32), l.kv_heads, l.batch);
      hipLaunchKernelGGL(seal_blocks_kernel<32>, grid, dim3(32 * kSealPieces), 0, stream, p);
    } else {
      const dim3 grid(static_cast<unsigned>((blocks + 15) / 16), l.kv_heads, l.batch);
      hipLaunchKernelGGL(seal_blocks_kernel<16>, grid, dim3(16 * kSealPieces), 0, stream, p);
    }
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    hipLaunchKernelGGL(seal_commit_kernel, dim3(l.batch), dim3(kWave), 0, stream, p);
  } else {
    hipLaunchKernelGGL(append_seal_kernel, dim3(l.batch), dim3(kThreads), 0, stream, p);
  }
  return hipGetLastError();
}

hipError_t launch_gather_pages(const uint16_t* pool, int64_t page_bytes, int64_t num_pages,
                               const int32_t* pages, int32_t count, uint16_t* out,
                               int32_t* status, hipStream_t stream) {
  if (count <= 0) return hipSuccess;
  const int64_t vecs = page_bytes / 16;
  const dim3 grid(grid_for(vecs, kThreads * 4), count);
  hipLaunchKernelGGL(gather_pages_kernel, grid, dim3(kThreads), 0, stream,
                     reinterpret_cast<const uint4*>(pool), vecs, num_pages, pages,
                     reinterpret_cast<uint4*>(out), status);
  return hipGetLastError();
}

hipError_t launch_read_step_bytes(const ReadStepLaunch& l, hipStream_t stream) {
  hipLaunchKernelGGL(read_step_bytes_kernel, dim3(l.kv_heads, l.batch), dim3(kReadThreads), 0, stream, l);
  return hipGetLastError();
}

hipError_t launch_pages_to_host(const uint16_t* pool, int64_t page_bytes, const int32_t* pages, int32_t count,
                                void* out, hipStream_t stream) {
  const int64_t vecs = page_bytes / 16;
  for (int32_t first = 0; first < count; first += kPagesPerHostCopy) {
    const int n = count - first < kPagesPerHostCopy ? count - first : kPagesPerHostCopy;
    PageIdsArg ids{};
    for (int i = 0; i < n; ++i) ids.ids[i] = pages[first + i];
    const dim3 grid(n < kHostCopyGroups ? n : kHostCopyGroups);
    hipLaunchKernelGGL(pages_to_host_kernel, grid, dim3(kThreads), 0, stream, reinterpret_cast<const uint4*>(pool),
                       vecs, n, ids, reinterpret_cast<uint4*>(static_cast<uint8_t*>(out) + first * page_bytes));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_fill_synthetic_f16(uint16_t* dst, int64_t count, uint64_t seed,
                                     uint64_t first_index, hipStream_t stream) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_synthetic_f16_kernel, dim3(grid_for(count, kThreads * 8)), dim3(kThreads), 0,
                     stream, dst, count, mix64(seed), first_index);
  return hipGetLastError();
}

hipError_t launch_fill_synthetic_f32(float* dst, int64_t count, uint64_t seed, uint64_t first_index,
                                     hipStream_t stream) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_synthetic_f32_kernel, dim3(grid_for(count, kThreads * 8)), dim3(kThreads), 0,
                     stream, dst, count, mix64(seed), first_index);
  return hipGetLastError();
}

hipError_t launch_fill_from_host(uint16_t* pool, int64_t page_bytes, int64_t num_pages, const int32_t* dst_pages,
                                 const uint8_t* src_dev, int64_t src_total, const int64_t* src_blocks, int32_t count,
                                 int32_t* status, hipStream_t stream) {
  if (count <= 0) return hipSuccess;
  const int64_t vecs = page_bytes / 16;
  const dim3 grid(grid_for(vecs, kThreads * 8), count);
  hipLaunchKernelGGL(fill_from_host_kernel, grid, dim3(kThreads), 0, stream, reinterpret_cast<uint4*>(pool), vecs,
                     num_pages, dst_pages, reinterpret_cast<const uint4*>(src_dev), src_total, src_blocks, status);
  return hipGetLastError();
}

hipError_t launch_xor_bytes(const uint8_t* input, uint8_t* output, uint64_t bytes, uint8_t mask,
                            hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  hipLaunchKernelGGL(xor_bytes_kernel, dim3(grid_for(static_cast<int64_t>(bytes / 16 + 1), kThreads * 4)),
                     dim3(kThreads), 0, stream, input, output, bytes, mask);
  return hipGetLastError();
}

hipError_t launch_consume_checksum(const float* input, int32_t elements, float* checksum,
                                   hipStream_t stream) {
  hipLaunchKernelGGL(consume_checksum_kernel, dim3(1), dim3(64), 0, stream, input, elements, checksum);
  return hipGetLastError();
}

}  // namespace sa
