// Token embedding forward (row gather) and a deterministic backward
// (scatter-add without floating-point atomics).
//
// Reference: the embedding of the first pipeline stage
// (femtotron/model/llama_partial_model.py:181-184) is an nn.Embedding, which
// femtotron's TP plan replaces by VocabParallelEmbedding
// (femtotron/parallel/tensor_parallel/embedding.py:57-79).  At one rank that
// module is: ids outside [0, V) are masked to row 0, looked up with
// F.embedding, and their output rows zeroed; the backward of F.embedding sums
// the output gradients of all tokens with the same id into that id's row
// (nothing for masked tokens, nothing for nn.Embedding's padding_idx).
//
// Forward: one wave per token row, 128-bit loads/stores.  Backward:
//   1. the token numbers grouped by id, in ascending token order within an id,
//      and each id's [start, end) range in that order.  Up to kGroupTokens
//      tokens one launch does it (k_embed_group); else a stable LSD radix
//      sort of (id, token): 8-bit digits, 1024-key tiles, per-tile digit
//      histograms, one exclusive scan over (digit, tile), a scatter whose
//      in-tile ranks come from wave ballots (peers with the same digit) plus
//      per-wave digit counts in LDS; keys are V for masked / padding tokens;
//   2. a vocabulary row's gradient is the fp32 sum of its tokens'
//      output-gradient rows in token order, rounded once; rows with no token
//      are written as zeros (no separate clear).
// Integer atomics appear only in LDS histograms, whose counts do not depend on
// order; no float is ever summed in a run-dependent order.
#include <type_traits>

#include "fh_common.hpp"

namespace fh {
namespace {

constexpr int kEmbThreads = 256;
constexpr int kRowsPerBlock = kEmbThreads / kWave;  // one row per wave
constexpr int kTile = 1024;                         // keys per sort block
constexpr int kRounds = kTile / kEmbThreads;
constexpr int kBins = 256;                          // 8-bit digits

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// ------------------------------------------------------------- forward
template <typename T>
__global__ __launch_bounds__(kEmbThreads) void k_embed_fwd(const T* __restrict__ w,
                                                           const int64_t* __restrict__ ids,
                                                           T* __restrict__ out, int64_t n_tokens,
                                                           int64_t vocab, int64_t hidden) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + (threadIdx.x >> 6);
  if (t >= n_tokens) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t id = ids[t];
  const bool ok = id >= 0 && id < vocab;
  T* dst = out + t * hidden;
  if (ok) {
    const T* src = w + id * hidden;
    for (int64_t c = lane * 8; c < hidden; c += kWave * 8)
      Elem<T>::straw(dst + c, Elem<T>::ldraw(src + c));
  } else {
    const float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int64_t c = lane * 8; c < hidden; c += kWave * 8) Elem<T>::store8(dst + c, z);
  }
}

// ------------------------------------------------------------- backward
// Sort keys and values; clears the per-id ranges (threads i < vocab).
__global__ __launch_bounds__(kEmbThreads) void k_embed_keys(const int64_t* __restrict__ ids,
                                                            int64_t n_tokens, int64_t vocab,
                                                            int64_t padding_idx,
                                                            uint32_t* __restrict__ keys,
                                                            uint32_t* __restrict__ vals,
                                                            uint32_t* __restrict__ seg_start,
                                                            uint32_t* __restrict__ seg_end) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kEmbThreads + threadIdx.x;
  if (i < n_tokens) {
    const int64_t id = ids[i];
    const bool ok = id >= 0 && id < vocab && id != padding_idx;
    keys[i] = static_cast<uint32_t>(ok ? id : vocab);
    vals[i] = static_cast<uint32_t>(i);
  }
  if (i < vocab) {
    seg_start[i] = 0;
    seg_end[i] = 0;
  }
}

// Per-tile digit histogram, stored digit-major: hist[d * n_tiles + tile].
__global__ __launch_bounds__(kEmbThreads) void k_radix_hist(const uint32_t* __restrict__ keys,
                                                            int64_t n, int shift,
                                                            uint32_t* __restrict__ hist,
                                                            int n_tiles) {
  __shared__ uint32_t cnt[kBins];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile;
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    const int64_t i = base + r * kEmbThreads + threadIdx.x;
    if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & (kBins - 1)], 1u);
  }
  __syncthreads();
  hist[static_cast<int64_t>(threadIdx.x) * n_tiles + blockIdx.x] = cnt[threadIdx.x];
}

// Exclusive scan of hist[0, m) in place by one block of 1024 threads: each
// thread owns one contiguous span; span totals are scanned in LDS.
__global__ __launch_bounds__(1024) void k_radix_scan(uint32_t* __restrict__ hist, int64_t m) {
  __shared__ uint32_t part[1024];
  const int64_t span = (m + 1023) / 1024;
  const int64_t lo = threadIdx.x * span;
  const int64_t hi = lo + span < m ? lo + span : m;
  uint32_t s = 0;
  for (int64_t i = lo; i < hi; ++i) s += hist[i];
  part[threadIdx.x] = s;
  __syncthreads();
  // Hillis-Steele inclusive scan of the 1024 span totals.
  for (int off = 1; off < 1024; off <<= 1) {
    const uint32_t add = threadIdx.x >= static_cast<unsigned>(off) ? part[threadIdx.x - off] : 0u;
    __syncthreads();
    part[threadIdx.x] += add;
    __syncthreads();
  }
  uint32_t run = threadIdx.x ? part[threadIdx.x - 1] : 0u;
  for (int64_t i = lo; i < hi; ++i) {
    const uint32_t c = hist[i];
    hist[i] = run;
    run += c;
  }
}

// Stable scatter of one tile.  Keys are taken in rounds of 256 (index order =
// (round, thread)); a key's position = scanned offset of (digit, tile) + keys
// of its digit in earlier rounds + in lower waves of this round + in lower
// lanes of its wave.
__global__ __launch_bounds__(kEmbThreads) void k_radix_scatter(
    const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out, int64_t n, int shift,
    const uint32_t* __restrict__ offsets, int n_tiles) {
  __shared__ uint32_t run[kBins];
  __shared__ uint32_t wcnt[kRowsPerBlock][kBins];
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x >> 6;
  const uint64_t lt_mask = (uint64_t(1) << lane) - 1;
  run[threadIdx.x] = 0;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kTile;
  for (int r = 0; r < kRounds; ++r) {
#pragma unroll
    for (int w = 0; w < kRowsPerBlock; ++w) wcnt[w][threadIdx.x] = 0;
    __syncthreads();
    const int64_t i = base + r * kEmbThreads + threadIdx.x;
    const bool valid = i < n;
    const uint32_t key = valid ? keys_in[i] : 0u;
    const uint32_t d = valid ? (key >> shift) & (kBins - 1) : kBins;  // kBins: no key
    uint64_t peers = ~uint64_t(0);
#pragma unroll
    for (int b = 0; b < 9; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const uint32_t rank = __popcll(peers & lt_mask);
    if (valid && rank == 0) wcnt[wv][d] = __popcll(peers);
    __syncthreads();
    if (valid) {
      uint32_t pos = run[d] + rank;
      for (int w = 0; w < wv; ++w) pos += wcnt[w][d];
      const uint64_t dst = static_cast<uint64_t>(offsets[static_cast<int64_t>(d) * n_tiles + blockIdx.x]) + pos;
      keys_out[dst] = key;
      vals_out[dst] = vals_in[i];
    }
    __syncthreads();
    uint32_t add = 0;
#pragma unroll
    for (int w = 0; w < kRowsPerBlock; ++w) add += wcnt[w][threadIdx.x];
    run[threadIdx.x] += add;
    // the next round's clear of wcnt is ordered after this read by its barrier
    __syncthreads();
  }
}

// [start, end) of every id's run in the sorted keys (sentinel key = vocab skipped).
__global__ __launch_bounds__(kEmbThreads) void k_embed_bounds(const uint32_t* __restrict__ keys,
                                                              int64_t n, uint32_t vocab,
                                                              uint32_t* __restrict__ seg_start,
                                                              uint32_t* __restrict__ seg_end) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kEmbThreads + threadIdx.x;
  if (i >= n) return;
  const uint32_t k = keys[i];
  if (k >= vocab) return;
  if (i == 0 || keys[i - 1] != k) seg_start[k] = static_cast<uint32_t>(i);
  if (i == n - 1 || keys[i + 1] != k) seg_end[k] = static_cast<uint32_t>(i + 1);
}

// The grouping in one launch: workgroup b owns ids [b R, (b + 1) R) and reads
// every token's id twice (n_tokens * 8 bytes from L2), each of its 16 waves one
// contiguous share of the tokens in order.  Pass 1 counts, per wave, the
// tokens of each owned id and those of lower ids (the sum is where the
// workgroup's tokens start, so workgroups need nothing from each other); the
// counts become offsets, id by id and wave by wave; pass 2 writes each token's
// number at its offset, ranked among the equal ids of its 64 lanes.  Against
// the sort's eight launches over the same 128 KB of ids (16384 tokens,
// V = 32000): 37 -> 17 us of kernel time and seven launches fewer.  The reads
// grow with n_tokens times the workgroups, so longer batches (and vocabularies
// of more than kGroupBlocks * kGroupMaxIds ids) keep the sort.
constexpr int kGroupThreads = 1024;
constexpr int kGroupWaves = kGroupThreads / kWave;
constexpr int64_t kGroupTokens = 65536;
constexpr int64_t kGroupBlocks = 512;   // two workgroups per CU
constexpr int64_t kGroupMaxIds = 1024;  // ids per workgroup: 64 KB of LDS counts

__global__ __launch_bounds__(kGroupThreads) void k_embed_group(const int64_t* __restrict__ ids, int n_tokens,
                                                               int64_t vocab, int64_t padding_idx, int R,
                                                               uint32_t* __restrict__ tok,
                                                               uint32_t* __restrict__ seg_start,
                                                               uint32_t* __restrict__ seg_end) {
  extern __shared__ uint32_t cnt[];  // [wave][R]: counts, then offsets
  __shared__ uint32_t part[kGroupWaves], below[kGroupWaves];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const uint64_t lt_mask = (uint64_t(1) << lane) - 1;
  const int64_t lo = static_cast<int64_t>(blockIdx.x) * R;
  const int n_ids = static_cast<int>(vocab - lo < R ? vocab - lo : R);
  const int per = (n_tokens + kGroupThreads - 1) / kGroupThreads * kWave;  // tokens of a wave, whole rounds
  const int beg = wave * per, end = min(n_tokens, beg + per);
  for (int i = threadIdx.x; i < kGroupWaves * R; i += kGroupThreads) cnt[i] = 0;
  __syncthreads();

  uint32_t lower = 0;
#pragma unroll 8
  for (int i = beg + lane; i < end; i += kWave) {
    const int64_t id = ids[i];
    if (id >= 0 && id < vocab && id != padding_idx) {
      if (id < lo) ++lower;
      else if (id < lo + n_ids) atomicAdd(&cnt[wave * R + static_cast<int>(id - lo)], 1u);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lower += __shfl_xor(lower, off, kWave);
  if (lane == 0) below[wave] = lower;
  __syncthreads();

  // Thread t: id lo + t.  Exclusive scan of the ids' totals (R <= 1024).
  const int t = threadIdx.x;
  uint32_t total = 0;
  if (t < n_ids)
    for (int w = 0; w < kGroupWaves; ++w) total += cnt[w * R + t];
  uint32_t incl = total;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t up = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += up;
  }
  if (lane == kWave - 1) part[wave] = incl;
  __syncthreads();
  uint32_t pos = incl - total;
  for (int w = 0; w < kGroupWaves; ++w) pos += below[w] + (w < wave ? part[w] : 0u);
  if (t < n_ids) {
    seg_start[lo + t] = pos;
    seg_end[lo + t] = pos + total;
    for (int w = 0; w < kGroupWaves; ++w) {
      const uint32_t c = cnt[w * R + t];
      cnt[w * R + t] = pos;
      pos += c;
    }
  }
  __syncthreads();

  for (int r0 = beg; r0 < end; r0 += kWave) {  // uniform per wave
    const int i = r0 + lane;
    const int64_t id = i < end ? ids[i] : -1;
    const bool mine = id >= lo && id < lo + n_ids && id != padding_idx;
    const int local = mine ? static_cast<int>(id - lo) : -1;
    for (uint64_t todo = __ballot(mine); todo != 0;) {
      const int cur = __shfl(local, __builtin_ctzll(todo), kWave);
      const uint64_t same = __ballot(local == cur);
      const uint32_t at = cnt[wave * R + cur];
      if (local == cur) tok[at + __popcll(same & lt_mask)] = static_cast<uint32_t>(i);
      cnt[wave * R + cur] = at + __popcll(same);  // every lane the same value
      todo &= ~same;
    }
  }
}

// The rows of dw.  A wave sums one vocabulary row of fewer than kHotTokens
// tokens: columns in groups of kRowChunks x 512 (8 per lane per chunk), so that
// one token's loads for the whole group are in flight together.
//
// A frequent id's row is one long chain of additions per column (text is
// Zipf-distributed: the first id of 16384 tokens has ~1100), and with one
// token's loads in flight at a time it took 1.3 us per token: 1489 us at
// V = 32000, H = 2048, whose bytes take 38 us.  So the grid's first workgroups
// take the rows of kHotTokens and more: a wave sums 128 columns of such a row
// (2 per lane) with the rows of up to kHotDepth tokens in flight, the additions
// still one after the other in token order: 58-62 us there.  (One wave per row and
// 1024 threads per workgroup, the tokens read as scalars: 132 us.)
//
// A hot workgroup looks through hot_ids consecutive ids and sums its frequent ones
// one after the other: 64 of them where the vocabulary gives workgroups enough, as
// few of whose ids are frequent, fewer (down to one) in a small vocabulary, whose
// ids may all be: fh_embedding_bwd halves them until there are kHotWaves waves.
// With 64 throughout, uniform ids of a small vocabulary were 32 waves' work at
// V = 1024, H = 256 (16384 tokens: 91 us, now 17; one wave per row 40) and 64 at
// V = 64, H = 2048 (4096 tokens: 203 us, now 11; one wave per row 64).
constexpr int kRowChunks = 4;
constexpr int kHotTokens = 8;
constexpr int kHotCols = 2 * kWave;  // columns that a wave sums of a hot row
constexpr int64_t kHotWaves = 4096;  // 16 per CU
template <typename T>
constexpr int kHotDepth = sizeof(T) == 2 ? 64 : 32;

// dst[c], dst[c + 1] of a row whose tokens are tok[0 .. n), n >= kHotTokens.
// Lane l holds the row offset of token j + l of the current 64 (the next 64
// token numbers are loaded meanwhile); readlane hands each to a load's scalar
// base, so a token costs two readlanes, a scalar add and a load.
template <typename T>
__device__ __forceinline__ void hot_columns(const T* __restrict__ dy, const uint32_t* __restrict__ tok, int n,
                                            T* __restrict__ dst, int64_t c, int64_t hidden, int lane) {
  using Pair = typename std::conditional<sizeof(T) == 2, uint32_t, float2>::type;
  const bool ok = c < hidden;  // hidden % 8 == 0: a pair is wholly in or out
  const char* col = reinterpret_cast<const char*>(dy + (ok ? c : 0));
  float a0 = 0.f, a1 = 0.f;
  int64_t off = 0;
  // Tokens k0 .. k0 + D - 1 of the current 64, those before `valid` added.
  auto sum = [&](auto depth, int k0, int valid) {
    constexpr int D = decltype(depth)::value;
    Pair v[D];
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(off), k0 + k);
      const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(off >> 32), k0 + k);
      v[k] = *reinterpret_cast<const Pair*>(col + (static_cast<int64_t>(hi) << 32 | lo));
    }
#pragma unroll
    for (int k = 0; k < D; ++k) {
      if (k0 + k >= valid) continue;  // uniform
      if constexpr (sizeof(T) == 2) {
        a0 += __uint_as_float(v[k] << 16);
        a1 += __uint_as_float(v[k] & 0xffff0000u);
      } else {
        a0 += v[k].x;
        a1 += v[k].y;
      }
    }
  };
  uint32_t next = tok[min(lane, n - 1)];
  for (int j = 0; j < n; j += kWave) {
    off = static_cast<int64_t>(next) * hidden * static_cast<int64_t>(sizeof(T));
    const int left = n - j;
    if (left > kWave) next = tok[min(j + kWave + lane, n - 1)];  // past the end: the last token again, not added
    if (left >= kWave) {
#pragma unroll
      for (int k0 = 0; k0 < kWave; k0 += kHotDepth<T>) sum(std::integral_constant<int, kHotDepth<T>>{}, k0, kWave);
    } else {
      int k0 = 0;
      for (; k0 + 16 <= left; k0 += 16) sum(std::integral_constant<int, 16>{}, k0, left);
      for (; k0 < left; k0 += 8) sum(std::integral_constant<int, 8>{}, k0, left);
    }
  }
  if (!ok) return;
  if constexpr (sizeof(T) == 2) *reinterpret_cast<uint32_t*>(dst + c) = pk_bf16(a0, a1);
  else *reinterpret_cast<float2*>(dst + c) = make_float2(a0, a1);
}

// Workgroups [0, hot_blocks): hot_blocks / hot_parts groups of hot_ids (at most 64)
// ids, and for each group hot_parts workgroups of kRowsPerBlock column slices; then
// one wave per row.
template <typename T>
__global__ __launch_bounds__(kEmbThreads) void k_embed_rows(const T* __restrict__ dy,
                                                            const uint32_t* __restrict__ tok,
                                                            const uint32_t* __restrict__ seg_start,
                                                            const uint32_t* __restrict__ seg_end,
                                                            T* __restrict__ dw, int64_t vocab,
                                                            int64_t hidden, int hot_blocks, int hot_parts,
                                                            int hot_ids) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int block = blockIdx.x;
  if (block < hot_blocks) {
    const int64_t v0 = static_cast<int64_t>(block / hot_parts) * hot_ids;
    const int64_t c0 = static_cast<int64_t>(block % hot_parts * kRowsPerBlock + wave) * kHotCols;
    if (c0 >= hidden) return;
    uint32_t lo = 0, len = 0;
    if (lane < hot_ids && v0 + lane < vocab) {
      lo = seg_start[v0 + lane];
      len = seg_end[v0 + lane] - lo;
    }
    for (uint64_t hot = __ballot(len >= kHotTokens); hot != 0; hot &= hot - 1) {
      const int l = __builtin_ctzll(hot);
      hot_columns<T>(dy, tok + __builtin_amdgcn_readlane(lo, l), __builtin_amdgcn_readlane(len, l),
                     dw + (v0 + l) * hidden, c0 + 2 * lane, hidden, lane);
    }
    return;
  }
  const int64_t v = static_cast<int64_t>(block - hot_blocks) * kRowsPerBlock + wave;
  if (v >= vocab) return;
  const uint32_t lo = seg_start[v], hi = seg_end[v];
  if (hi - lo >= kHotTokens) return;
  T* dst = dw + v * hidden;
  for (int64_t c0 = lane * 8; c0 < hidden; c0 += kRowChunks * kWave * 8) {
    float acc[kRowChunks][8];
#pragma unroll
    for (int k = 0; k < kRowChunks; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[k][e] = 0.f;
    for (uint32_t j = lo; j < hi; ++j) {
      const T* src = dy + static_cast<int64_t>(tok[j]) * hidden + c0;
      float g[kRowChunks][8];
#pragma unroll
      for (int k = 0; k < kRowChunks; ++k)
        if (c0 + k * kWave * 8 < hidden) Elem<T>::load8(src + k * kWave * 8, g[k]);
#pragma unroll
      for (int k = 0; k < kRowChunks; ++k)
        if (c0 + k * kWave * 8 < hidden)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[k][e] += g[k][e];
    }
#pragma unroll
    for (int k = 0; k < kRowChunks; ++k)
      if (c0 + k * kWave * 8 < hidden) Elem<T>::store8(dst + c0 + k * kWave * 8, acc[k]);
  }
}

int radix_passes(int64_t vocab) {
  int bits = 0;
  while ((int64_t(1) << bits) <= vocab) ++bits;  // keys take values 0..vocab
  return (bits + 7) / 8;
}

struct BwdLayout {
  size_t keys_a, vals_a, keys_b, vals_b, hist, seg_start, seg_end, total;
};

BwdLayout bwd_layout(int64_t n_tokens, int64_t vocab) {
  const int64_t tiles = (n_tokens + kTile - 1) / kTile;
  BwdLayout l{};
  size_t off = 0;
  const size_t keyb = align256(static_cast<size_t>(n_tokens) * 4);
  l.keys_a = off; off += keyb;
  l.vals_a = off; off += keyb;
  l.keys_b = off; off += keyb;
  l.vals_b = off; off += keyb;
  l.hist = off; off += align256(static_cast<size_t>(tiles) * kBins * 4);
  l.seg_start = off; off += align256(static_cast<size_t>(vocab) * 4);
  l.seg_end = off; off += align256(static_cast<size_t>(vocab) * 4);
  l.total = off;
  return l;
}

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" int fh_embedding_fwd(fh_dtype dt, const void* weight, const int64_t* ids, void* out,
                                int64_t n_tokens, int64_t vocab, int64_t hidden,
                                hipStream_t stream) {
  FH_REQUIRE(dt == FH_BF16 || dt == FH_F32, "embedding_fwd: dtype must be FH_BF16 or FH_F32");
  FH_REQUIRE(n_tokens >= 0 && vocab > 0 && hidden > 0, "embedding_fwd: bad sizes");
  FH_REQUIRE(hidden % 8 == 0, "embedding_fwd: hidden must be a multiple of 8");
  if (n_tokens == 0) return FH_OK;
  FH_REQUIRE(weight && ids && out, "embedding_fwd: null pointer");
  FH_REQUIRE(aligned16(weight) && aligned16(out), "embedding_fwd: weight/out must be 16-byte aligned");
  FH_REQUIRE((n_tokens + kRowsPerBlock - 1) / kRowsPerBlock <= 0x7fffffff, "embedding_fwd: too many tokens");
  const dim3 grid(static_cast<unsigned>((n_tokens + kRowsPerBlock - 1) / kRowsPerBlock));
  if (dt == FH_BF16)
    hipLaunchKernelGGL(k_embed_fwd<uint16_t>, grid, dim3(kEmbThreads), 0, stream,
                       static_cast<const uint16_t*>(weight), ids, static_cast<uint16_t*>(out),
                       n_tokens, vocab, hidden);
  else
    hipLaunchKernelGGL(k_embed_fwd<float>, grid, dim3(kEmbThreads), 0, stream,
                       static_cast<const float*>(weight), ids, static_cast<float*>(out), n_tokens,
                       vocab, hidden);
  return check_launch("fh_embedding_fwd");
}

extern "C" size_t fh_embedding_bwd_workspace_size(int64_t n_tokens, int64_t vocab) {
  if (n_tokens < 0 || vocab <= 0) return 0;
  return bwd_layout(n_tokens, vocab).total;
}

extern "C" int fh_embedding_bwd(fh_dtype dt, const void* dy, const int64_t* ids, void* dweight,
                                int64_t n_tokens, int64_t vocab, int64_t hidden,
                                int64_t padding_idx, void* workspace, hipStream_t stream) {
  FH_REQUIRE(dt == FH_BF16 || dt == FH_F32, "embedding_bwd: dtype must be FH_BF16 or FH_F32");
  FH_REQUIRE(n_tokens >= 0 && vocab > 0 && hidden > 0, "embedding_bwd: bad sizes");
  FH_REQUIRE(hidden % 8 == 0, "embedding_bwd: hidden must be a multiple of 8");
  FH_REQUIRE(vocab < 0x7fffffff && n_tokens < 0x7fffffff, "embedding_bwd: sizes must fit 31 bits");
  FH_REQUIRE(dweight && workspace && (n_tokens == 0 || (dy && ids)), "embedding_bwd: null pointer");
  FH_REQUIRE(aligned16(dweight) && (n_tokens == 0 || aligned16(dy)) && aligned16(workspace),
             "embedding_bwd: dy/dweight/workspace must be 16-byte aligned");
  const BwdLayout l = bwd_layout(n_tokens, vocab);
  char* ws = static_cast<char*>(workspace);
  uint32_t* keys[2] = {reinterpret_cast<uint32_t*>(ws + l.keys_a), reinterpret_cast<uint32_t*>(ws + l.keys_b)};
  uint32_t* vals[2] = {reinterpret_cast<uint32_t*>(ws + l.vals_a), reinterpret_cast<uint32_t*>(ws + l.vals_b)};
  uint32_t* hist = reinterpret_cast<uint32_t*>(ws + l.hist);
  uint32_t* seg_start = reinterpret_cast<uint32_t*>(ws + l.seg_start);
  uint32_t* seg_end = reinterpret_cast<uint32_t*>(ws + l.seg_end);
  int cur = 0;
  if (n_tokens <= kGroupTokens && vocab <= kGroupBlocks * kGroupMaxIds) {
    // As many ids per workgroup as give kGroupBlocks workgroups.
    const int64_t per = (vocab + kGroupBlocks - 1) / kGroupBlocks;
    const int R = static_cast<int>(per);
    hipLaunchKernelGGL(k_embed_group, dim3(static_cast<unsigned>((vocab + R - 1) / R)), dim3(kGroupThreads),
                       static_cast<size_t>(kGroupWaves) * R * 4, stream, ids, static_cast<int>(n_tokens), vocab,
                       padding_idx, R, vals[0], seg_start, seg_end);
  } else {
    const int64_t wide = n_tokens > vocab ? n_tokens : vocab;
    hipLaunchKernelGGL(k_embed_keys, dim3(static_cast<unsigned>((wide + kEmbThreads - 1) / kEmbThreads)),
                       dim3(kEmbThreads), 0, stream, ids, n_tokens, vocab, padding_idx, keys[0], vals[0],
                       seg_start, seg_end);
    if (n_tokens > 0) {
      const int tiles = static_cast<int>((n_tokens + kTile - 1) / kTile);
      const int passes = radix_passes(vocab);
      for (int p = 0; p < passes; ++p) {
        hipLaunchKernelGGL(k_radix_hist, dim3(tiles), dim3(kEmbThreads), 0, stream, keys[cur], n_tokens,
                           8 * p, hist, tiles);
        hipLaunchKernelGGL(k_radix_scan, dim3(1), dim3(1024), 0, stream, hist,
                           static_cast<int64_t>(tiles) * kBins);
        hipLaunchKernelGGL(k_radix_scatter, dim3(tiles), dim3(kEmbThreads), 0, stream, keys[cur],
                           vals[cur], keys[cur ^ 1], vals[cur ^ 1], n_tokens, 8 * p, hist, tiles);
        cur ^= 1;
      }
      hipLaunchKernelGGL(k_embed_bounds, dim3(static_cast<unsigned>((n_tokens + kEmbThreads - 1) / kEmbThreads)),
                         dim3(kEmbThreads), 0, stream, keys[cur], n_tokens, static_cast<uint32_t>(vocab),
                         seg_start, seg_end);
    }
  }
  // A row of kHotTokens tokens needs that many.
  const int64_t hot_parts = (hidden + kRowsPerBlock * kHotCols - 1) / (kRowsPerBlock * kHotCols);
  int64_t hot_ids = kWave;
  while (hot_ids > 1 && (vocab + hot_ids - 1) / hot_ids * hot_parts * kRowsPerBlock < kHotWaves) hot_ids /= 2;
  const int64_t hot_blocks = n_tokens >= kHotTokens ? (vocab + hot_ids - 1) / hot_ids * hot_parts : 0;
  const int64_t blocks = hot_blocks + (vocab + kRowsPerBlock - 1) / kRowsPerBlock;
  FH_REQUIRE(blocks <= 0x7fffffff, "embedding_bwd: vocab * hidden too large");
  auto rows = [&](auto tag) {
    using T = decltype(tag);
    hipLaunchKernelGGL(k_embed_rows<T>, dim3(static_cast<unsigned>(blocks)), dim3(kEmbThreads), 0, stream,
                       static_cast<const T*>(dy), vals[cur], seg_start, seg_end, static_cast<T*>(dweight), vocab,
                       hidden, static_cast<int>(hot_blocks), static_cast<int>(hot_parts), static_cast<int>(hot_ids));
  };
  if (dt == FH_BF16) rows(uint16_t{});
  else rows(float{});
  return check_launch("fh_embedding_bwd");
}
