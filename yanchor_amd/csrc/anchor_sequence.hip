// Anchor memory, prefill continuation: the block-wise Top-K scan and the
// state rewrite of IndependentGQAMemory._sequence with a state
// (modeling_yanchor.py:178-275), for prefill chunks that continue a memory
// state (the CausalLM's bounded prefill chunks, modeling_yanchor.py:981-1012;
// the vLLM / SGLang per-request prefill, vllm_yanchor.py:85-96,
// sglang_models/yanchor.py:70-83).
//
// The sequence a row sees is its old pending tokens (count of them) followed
// by its valid new tokens, cut into blocks of C.  Queries of block j read the
// memory committed before block j: the Top-K of the initial committed slots
// and every complete block before j.  The reference computes those prefixes
// with an up-sweep / down-sweep tree of merge_topk (exclusive_prefix_topk,
// modeling_yanchor.py:65-78) and merges the initial state in afterwards
// (217-219).  Top-K under one strict order is a selection of the best K of a
// union, so a left-to-right scan -- memory_{j+1} = TopK(memory_j u block_j) --
// gives the same sets in the same (rank) order, and that is what the decode
// commit does one chunk at a time.  It also means that memory j is the first K
// of ALL candidates in rank order that come before block j, so the blocks need
// no scan: a workgroup per (row, group) sorts the committed slots and a segment
// of blocks once and every wave reads off the memories of its own blocks.
// (Equal keys keep candidate order: committed slots first, then tokens, as the
// scan's merges leave them.)
//
// Source rows (per batch row, shared by its groups) number the candidates:
//   [0, K)          the committed slots of the state
//   [K, K + C)      the old pending slots
//   [K + C, K + C + L)  the new tokens, in order
// anchor_prefix_kernel writes, per block, the source rows of the memory in
// force (the `read_refs` of modeling_yanchor.py:248), and rewrites the scores,
// positions and pending scores of the state in place; anchor_seq_commit_kernel
// then copies the key / value rows of the final memory and of the new pending
// tokens from where they are (modeling_yanchor.py:256-274) and advances count /
// total.
#include "anchor_source.h"

namespace yh {
namespace {

constexpr int kSeqThreads = 256;
constexpr int kSeqMaxCand = 2048;  // capacity + chunk
constexpr int kSeqMaxChunk = 1024;
constexpr int kSortThreads = 1024;
constexpr int kSortMax = 4096;     // candidates sorted at once
constexpr int kSortPer = kSortMax / kSortThreads;
constexpr int kRun = 16;           // length of the runs ranked by counting

struct PrefixArgs {
  const float* new_scores;  // [.., G]     token i of row b at row (bases ? bases[b] : b L) + (order ? order[b L + i] : i)
  const int64_t* bases;
  const int32_t* order;     // [B, L]      valid tokens first
  const int64_t* counts;    // [B]         valid new tokens per row
  float* scores;            // [B, G, KC]  committed scores (in place)
  int32_t* pos;             // [B, G, KC]  committed positions (in place)
  float* pscores;           // [B, G, PC]  pending scores (in place)
  const int64_t* count;     // [B]
  const int64_t* total;     // [B]
  int32_t* block_refs;      // [B, NB, G, KC]
  int32_t* final_refs;      // [B, G, KC]
  int32_t* pending_refs;    // [B, G, PC]
  int L, G, KC, PC, C, NB;
  int64_t groups;           // B * G
};

// Sort the n candidates key[0][0, n) (and idx[0]) into rank order: runs of
// kRun by counting, then merges in which an element's place is its place in
// its own run plus the number of the other run's elements before it (a binary
// search; the left run's candidates come first on equal keys).  Returns which
// of the two buffers holds the result.  Starts and ends with a workgroup
// barrier.
__device__ __forceinline__ int sort_candidates(uint64_t (*key)[kSortMax], uint16_t (*idx)[kSortMax], int n, int tid) {
  __syncthreads();
  int from = 0;
  for (int i = tid; i < n; i += kSortThreads) {
    const int r0 = i & ~(kRun - 1), r1 = min(r0 + kRun, n);
    const uint64_t mine = key[0][i];
    int rank = 0;
    for (int m = r0; m < r1; ++m) {
      const uint64_t o = key[0][m];
      rank += (o < mine) | ((o == mine) & (m < i));
    }
    key[1][r0 + rank] = mine;
    idx[1][r0 + rank] = idx[0][i];
  }
  from = 1;
  for (int len = kRun; len < n; len *= 2) {
    __syncthreads();
    const uint64_t* src = key[from];
    uint64_t mine[kSortPer];
    int lo[kSortPer], hi[kSortPer], other[kSortPer];
    bool right[kSortPer];
#pragma unroll
    for (int k = 0; k < kSortPer; ++k) {
      const int i = tid + k * kSortThreads;
      lo[k] = hi[k] = other[k] = 0;
      right[k] = false;
      mine[k] = 0;
      if (i < n) {
        right[k] = (i & len) != 0;
        other[k] = (i & ~(2 * len - 1)) + (right[k] ? 0 : len);   // start of the other run
        hi[k] = max(0, min(len, n - other[k]));
        mine[k] = src[i];
      }
    }
    for (int step = len; step > 0; step >>= 1) {   // log2(len) + 1 halvings close every [lo, hi]
#pragma unroll
      for (int k = 0; k < kSortPer; ++k) {
        if (lo[k] < hi[k]) {
          const int mid = (lo[k] + hi[k]) >> 1;
          const uint64_t o = src[other[k] + mid];
          if (o < mine[k] || (right[k] && o == mine[k])) lo[k] = mid + 1;
          else hi[k] = mid;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kSortPer; ++k) {
      const int i = tid + k * kSortThreads;
      if (i < n) {
        const int at = (i & ~(2 * len - 1)) + (i & (len - 1)) + lo[k];
        key[from ^ 1][at] = mine[k];
        idx[from ^ 1][at] = idx[from][i];
      }
    }
    from ^= 1;
  }
  __syncthreads();
  return from;
}

// Bound by LDS latency (about ten dependent reads a merge level) at one
// workgroup a CU.  32 rows x 8 groups of 2048 tokens: 38 us, where merging one
// block after the other into the memory took 195.
__global__ void __launch_bounds__(kSortThreads) anchor_prefix_kernel(PrefixArgs a) {
  __shared__ uint64_t key[2][kSortMax];
  __shared__ uint16_t idx[2][kSortMax];
  __shared__ float mscore[kSeqMaxCand];   // the memory before the segment
  __shared__ int32_t mpos[kSeqMaxCand];
  __shared__ int32_t mref[kSeqMaxCand];
  __shared__ float opend[kSeqMaxChunk];

  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t bg = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
  if (bg >= a.groups) return;
  const int64_t b = bg / a.G;
  const int g = static_cast<int>(bg % a.G);
  const int KC = a.KC, C = a.C, G = a.G;
  int32_t* brefs = a.block_refs + (b * a.NB * G + g) * KC;  // block j at + j * G * KC
  const int64_t old_count = a.count[b];
  if (old_count < 0 || old_count >= C) {
    // corrupt counter: the row reads nothing and its state is left untouched
    for (int j = 0; j < a.NB; ++j)
      for (int s = tid; s < KC; s += kSortThreads) brefs[static_cast<int64_t>(j) * G * KC + s] = -1;
    return;
  }
  const int64_t n_new = min(max(a.counts[b], static_cast<int64_t>(0)), static_cast<int64_t>(a.L));
  const int64_t n_all = old_count + n_new;
  const int64_t full = n_all / C, rem = n_all - full * C;
  const int64_t base_pos = a.total[b] - old_count;
  float* scores = a.scores + bg * KC;
  int32_t* pos = a.pos + bg * KC;
  float* pscores = a.pscores + bg * a.PC;
  const int64_t row0 = a.bases ? a.bases[b] : b * a.L;
  // sequence index q: the old pending tokens, then the new ones
  auto token_score = [&](int64_t q) -> float {
    if (q < old_count) return opend[q];
    const int64_t i = q - old_count;
    return a.new_scores[(row0 + (a.order ? a.order[b * a.L + i] : i)) * G + g];
  };
  auto token_ref = [&](int64_t q) { return static_cast<int32_t>(q < old_count ? KC + q : KC + C + (q - old_count)); };

  for (int s = tid; s < KC; s += kSortThreads) {
    const int32_t p = pos[s];
    mscore[s] = scores[s];
    mpos[s] = p >= 0 ? p : -1;
    mref[s] = p >= 0 ? s : -1;
  }
  for (int t = tid; t < old_count; t += kSortThreads) opend[t] = pscores[t];

  // The committed slots are ranked also when no block completes (the merge of
  // the initial state into an empty prefix, modeling_yanchor.py:217-219).
  const int64_t seg_blocks = (kSortMax - KC) / C;
  int64_t done = 0;
  do {
    const int nb = static_cast<int>(min(full - done, seg_blocks));
    const int n = KC + nb * C;
    __syncthreads();  // the memory and opend
    for (int i = tid; i < n; i += kSortThreads) {
      const int64_t q = done * C + (i - KC);
      key[0][i] = i < KC ? topk_key(mscore[i], mpos[i]) : topk_key(token_score(q), static_cast<int32_t>(base_pos + q));
      idx[0][i] = static_cast<uint16_t>(i);
    }
    const uint16_t* order = idx[sort_candidates(key, idx, n, tid)];
    // wave w: the memories of blocks done + w, done + w + 16, ...
    for (int j = w; j < nb; j += kSortThreads / 64) {
      int32_t* out = brefs + (done + j) * G * KC;
      const int limit = KC + j * C;   // candidates before the block
      for (int i0 = 0, have = 0; have < KC; i0 += 64) {
        const int c = i0 + lane < n ? order[i0 + lane] : kSortMax;
        const bool take = c < limit;
        const uint64_t m = __ballot(take);
        const int at = have + __popcll(m & ((1ull << lane) - 1));
        if (take && at < KC) out[at] = c < KC ? mref[c] : token_ref(done * C + (c - KC));
        have += __popcll(m);
      }
    }
    // the first KC of all are the memory after the segment
    float ns[kSeqMaxCand / kSortThreads];
    int32_t np[kSeqMaxCand / kSortThreads], nr[kSeqMaxCand / kSortThreads];
#pragma unroll
    for (int k = 0; k < kSeqMaxCand / kSortThreads; ++k) {
      const int s = tid + k * kSortThreads;
      if (s < KC) {
        const int c = order[s];
        const int64_t q = done * C + (c - KC);
        ns[k] = c < KC ? mscore[c] : token_score(q);
        np[k] = c < KC ? mpos[c] : static_cast<int32_t>(base_pos + q);
        nr[k] = c < KC ? mref[c] : token_ref(q);
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSeqMaxCand / kSortThreads; ++k) {
      const int s = tid + k * kSortThreads;
      if (s < KC) {
        mscore[s] = ns[k];
        mpos[s] = np[k];
        mref[s] = nr[k];
      }
    }
    done += nb;
  } while (done < full);
  __syncthreads();

  // the blocks past the last full one, the final memory, the pending tail
  for (int64_t j = full + w; j < a.NB; j += kSortThreads / 64)
    for (int s = lane; s < KC; s += 64) brefs[j * G * KC + s] = mref[s];
  int32_t* frefs = a.final_refs + bg * KC;
  for (int s = tid; s < KC; s += kSortThreads) {
    scores[s] = mscore[s];
    pos[s] = mpos[s];
    frefs[s] = mref[s];
  }
  int32_t* prefs = a.pending_refs + bg * a.PC;
  for (int t = tid; t < a.PC; t += kSortThreads) {
    float sc = -INFINITY;
    int32_t ref = -1;
    if (t < rem) {
      const int64_t q = full * C + t;
      sc = token_score(q);
      ref = token_ref(q);
    }
    pscores[t] = sc;
    prefs[t] = ref;
  }
}

struct SeqCommitArgs {
  AnchorSource src;
  const int32_t* final_refs;  // [B, G, KC]
  const int32_t* pending_refs;  // [B, G, PC]
  const int64_t* counts;      // [B]
  char* out[2];               // keys, values [B, G, KC, D]
  char* pout[2];              // pending [B, G, PC, D]
  int64_t* count;             // [B]
  int64_t* total;             // [B]
  int G, KC, PC, C, L;
  int pending;                // pending slots that can hold a row; the others are zeroed
  int64_t rowbytes;
};

constexpr int kStage = 4096;  // 16-byte pieces staged at once

// One workgroup per (row, group) and tensor: the committed slots and the
// pending slots take their rows from the sources (zeros where no row is
// referenced, as the masked copies of the reference).  The sources may be the
// state itself: a slice of every row's 16-byte pieces is read into LDS before
// any row of that slice is written (with more rows than the stage holds the
// sources are another tensor).  The first workgroup of a row advances its count
// and total; the others only ask whether count is in range, which it is before
// and after.  A corrupt count leaves the row untouched.
__global__ void __launch_bounds__(kSeqThreads) anchor_seq_commit_kernel(SeqCommitArgs a) {
  __shared__ uint4 stage[kStage];
  const int tid = threadIdx.x;
  const int64_t bg = blockIdx.x;
  const int64_t b = bg / a.G;
  const int g = static_cast<int>(bg % a.G);
  const int64_t old_count = a.count[b];
  if (old_count < 0 || old_count >= a.C) return;
  const int which = blockIdx.y;
  const int pieces = static_cast<int>(a.rowbytes / 16);
  const int all = a.KC + a.pending, rows = min(all, kStage);
  char* out = a.out[which] + bg * a.KC * a.rowbytes;
  char* pout = a.pout[which] + bg * a.PC * a.rowbytes;
  const int width = min(pieces, kStage / rows);
  for (int r0 = 0; r0 < all; r0 += rows)
    for (int c0 = 0; c0 < pieces; c0 += width) {
      const int wd = min(width, pieces - c0), n = min(rows, all - r0) * wd;
      for (int i = tid; i < n; i += kSeqThreads) {
        const int slot = r0 + i / wd, c = c0 + i % wd;
        const int32_t ref = slot < a.KC ? a.final_refs[bg * a.KC + slot] : a.pending_refs[bg * a.PC + (slot - a.KC)];
        uint4 x = make_uint4(0, 0, 0, 0);
        if (ref >= 0 && ref < a.src.S) x = static_cast<const uint4*>(a.src.row(which, b, ref, g))[c];
        stage[i] = x;
      }
      __syncthreads();
      for (int i = tid; i < n; i += kSeqThreads) {
        const int slot = r0 + i / wd, c = c0 + i % wd;
        char* dst = slot < a.KC ? out + slot * a.rowbytes : pout + (slot - a.KC) * a.rowbytes;
        reinterpret_cast<uint4*>(dst)[c] = stage[i];
      }
      __syncthreads();
    }
  for (int64_t i = tid; i < static_cast<int64_t>(a.PC - a.pending) * pieces; i += kSeqThreads)
    reinterpret_cast<uint4*>(pout + a.pending * a.rowbytes)[i] = make_uint4(0, 0, 0, 0);
  if (g == 0 && which == 0 && tid == 0) {
    const int64_t n = min(max(a.counts[b], static_cast<int64_t>(0)), static_cast<int64_t>(a.L));
    a.count[b] = (old_count + n) % a.C;
    a.total[b] += n;
  }
}

int launch_commit(SeqCommitArgs a, int64_t B, yh_stream_t stream, const char* what) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(anchor_seq_commit_kernel, dim3(static_cast<unsigned>(B * a.G), 2), dim3(kSeqThreads), 0, st, a);
  YH_CHECK_LAUNCH(what);
  return YH_OK;
}

int launch_prefix(PrefixArgs a, int64_t B, int64_t L, int64_t G, int64_t capacity, int64_t pending_capacity,
                  int64_t chunk, int64_t NB, yh_stream_t stream, const char* what) {
  YH_CHECK_ARG(B >= 0 && L >= 0 && G > 0 && capacity > 0 && NB >= 0, "%s: bad sizes", what);
  YH_CHECK_ARG(chunk >= 1 && chunk <= pending_capacity && chunk <= kSeqMaxChunk,
               "%s: chunk must be in [1, min(pending capacity, %d)]", what, kSeqMaxChunk);
  YH_CHECK_ARG(capacity + chunk <= kSeqMaxCand, "%s: capacity + chunk must be <= %d", what, kSeqMaxCand);
  YH_CHECK_ARG(NB * chunk >= L + chunk - 1, "%s: %lld blocks of %lld cannot hold %lld pending + new tokens", what,
               (long long)NB, (long long)chunk, (long long)(L + chunk - 1));
  YH_CHECK_ARG(capacity + chunk + L < (1LL << 31) && B * G < (1LL << 31), "%s: too large", what);
  if (B == 0) return YH_OK;
  YH_CHECK_ARG(a.counts && a.scores && a.pos && a.pscores && a.count && a.total && a.final_refs && a.pending_refs &&
                   (L == 0 || a.new_scores) && (NB == 0 || a.block_refs),
               "%s: null pointer", what);
  a.L = static_cast<int>(L);
  a.G = static_cast<int>(G);
  a.KC = static_cast<int>(capacity);
  a.PC = static_cast<int>(pending_capacity);
  a.C = static_cast<int>(chunk);
  a.NB = static_cast<int>(NB);
  a.groups = B * G;
  const int64_t wide = a.groups < (1 << 20) ? a.groups : 1 << 20;   // a grid's row holds less than 2^32 threads
  const dim3 grid(static_cast<unsigned>(wide), static_cast<unsigned>((a.groups + wide - 1) / wide));
  hipLaunchKernelGGL(anchor_prefix_kernel, grid, dim3(kSortThreads), 0, static_cast<hipStream_t>(stream), a);
  YH_CHECK_LAUNCH(what);
  return YH_OK;
}

}  // namespace
}  // namespace yh

extern "C" int yh_anchor_prefix(const float* new_scores, const int64_t* counts, float* scores, int32_t* positions,
                                float* pending_scores, const int64_t* count, const int64_t* total,
                                int32_t* block_refs, int32_t* final_refs, int32_t* pending_refs, int64_t B, int64_t L,
                                int64_t G, int64_t capacity, int64_t pending_capacity, int64_t chunk, int64_t NB,
                                yh_stream_t stream) {
  using namespace yh;
  return launch_prefix(PrefixArgs{new_scores, nullptr, nullptr, counts, scores, positions, pending_scores, count,
                                  total, block_refs, final_refs, pending_refs},
                       B, L, G, capacity, pending_capacity, chunk, NB, stream, "anchor_prefix");
}

extern "C" int yh_anchor_tokens_prefix(const float* new_scores, const int64_t* bases, const int32_t* order,
                                       const int64_t* counts, float* scores, int32_t* positions,
                                       float* pending_scores, const int64_t* count, const int64_t* total,
                                       int32_t* block_refs, int32_t* final_refs, int32_t* pending_refs, int64_t B,
                                       int64_t L, int64_t G, int64_t capacity, int64_t pending_capacity,
                                       int64_t chunk, int64_t NB, yh_stream_t stream) {
  using namespace yh;
  return launch_prefix(PrefixArgs{new_scores, bases, order, counts, scores, positions, pending_scores, count, total,
                                  block_refs, final_refs, pending_refs},
                       B, L, G, capacity, pending_capacity, chunk, NB, stream, "anchor_tokens_prefix");
}

extern "C" int yh_anchor_sequence_commit(const void* src_keys, const void* src_values, const int32_t* final_refs,
                                         const int32_t* pending_refs, const int64_t* counts, void* keys, void* values,
                                         void* pending_keys, void* pending_values, int64_t* count, int64_t* total,
                                         int64_t B, int64_t S, int64_t L, int64_t G, int64_t capacity,
                                         int64_t pending_capacity, int64_t chunk, int64_t D, int dtype,
                                         yh_stream_t stream) {
  using namespace yh;
  YH_CHECK_ARG(B >= 0 && S >= 0 && L >= 0 && G > 0 && capacity > 0 && pending_capacity > 0 && D > 0,
               "anchor_sequence_commit: bad sizes");
  YH_CHECK_ARG(chunk >= 1 && chunk <= pending_capacity, "anchor_sequence_commit: chunk outside [1, pending capacity]");
  YH_CHECK_ARG(is_float_dtype(dtype), "anchor_sequence_commit: unsupported dtype %d", dtype);
  const int64_t rowbytes = D * (dtype == YH_F32 ? 4 : 2);
  YH_CHECK_ARG(rowbytes % 16 == 0, "anchor_sequence_commit: a row must be a multiple of 16 bytes");
  YH_CHECK_ARG(S < (1LL << 31) && B * G < (1LL << 32) / kSeqThreads, "anchor_sequence_commit: too large");
  if (B == 0) return YH_OK;
  YH_CHECK_ARG(src_keys && src_values && final_refs && pending_refs && counts && keys && values && pending_keys &&
                   pending_values && count && total,
               "anchor_sequence_commit: null pointer");
  YH_CHECK_ARG(((reinterpret_cast<uintptr_t>(src_keys) | reinterpret_cast<uintptr_t>(src_values) |
                 reinterpret_cast<uintptr_t>(keys) | reinterpret_cast<uintptr_t>(values) |
                 reinterpret_cast<uintptr_t>(pending_keys) | reinterpret_cast<uintptr_t>(pending_values)) & 15) == 0,
               "anchor_sequence_commit: key/value tensors must be 16-byte aligned");
  SeqCommitArgs a{assembled_source(src_keys, src_values, S, S, G, rowbytes), final_refs, pending_refs, counts,
                  {static_cast<char*>(keys), static_cast<char*>(values)},
                  {static_cast<char*>(pending_keys), static_cast<char*>(pending_values)}, count, total, (int)G,
                  (int)capacity, (int)pending_capacity, (int)chunk, (int)L, (int)pending_capacity, rowbytes};
  return launch_commit(a, B, stream, "anchor_sequence_commit");
}

extern "C" int yh_anchor_tokens_commit(const void* key, int64_t key_stride, const void* value, int64_t value_stride,
                                       const int32_t* final_refs, const int32_t* pending_refs, const int64_t* counts,
                                       const int64_t* bases, const int32_t* order, void* keys, void* values,
                                       void* pending_keys, void* pending_values, int64_t* count, int64_t* total,
                                       int64_t B, int64_t L, int64_t G, int64_t capacity, int64_t pending_capacity,
                                       int64_t chunk, int64_t D, int dtype, yh_stream_t stream) {
  using namespace yh;
  const char* what = "anchor_tokens_commit";
  YH_CHECK_ARG(B >= 0 && L >= 0 && G > 0 && capacity > 0 && D > 0, "%s: bad sizes", what);
  YH_CHECK_ARG(chunk >= 1 && chunk <= pending_capacity, "%s: chunk outside [1, pending capacity]", what);
  YH_CHECK_ARG(is_float_dtype(dtype), "%s: unsupported dtype %d", what, dtype);
  const int64_t size = dtype == YH_F32 ? 4 : 2, rowbytes = D * size;
  YH_CHECK_ARG(rowbytes % 16 == 0 && key_stride * size % 16 == 0 && value_stride * size % 16 == 0 &&
                   key_stride >= G * D && value_stride >= G * D,
               "%s: rows must be multiples of 16 bytes and hold whole heads", what);
  YH_CHECK_ARG(capacity + chunk + L < (1LL << 31) && B * G < (1LL << 32) / kSeqThreads && capacity + chunk <= kStage,
               "%s: too large", what);
  if (B == 0) return YH_OK;
  YH_CHECK_ARG((L == 0 || (key && value)) && final_refs && pending_refs && counts && keys && values && pending_keys &&
                   pending_values && count && total,
               "%s: null pointer", what);
  YH_CHECK_ARG(((reinterpret_cast<uintptr_t>(key) | reinterpret_cast<uintptr_t>(value) |
                 reinterpret_cast<uintptr_t>(keys) | reinterpret_cast<uintptr_t>(values) |
                 reinterpret_cast<uintptr_t>(pending_keys) | reinterpret_cast<uintptr_t>(pending_values)) & 15) == 0,
               "%s: key/value tensors must be 16-byte aligned", what);
  SeqCommitArgs a{state_source(keys, values, pending_keys, pending_values, key, key_stride * size, value,
                               value_stride * size, bases, order, L, chunk, G, capacity, pending_capacity, rowbytes),
                  final_refs, pending_refs, counts, {static_cast<char*>(keys), static_cast<char*>(values)},
                  {static_cast<char*>(pending_keys), static_cast<char*>(pending_values)}, count, total, (int)G,
                  (int)capacity, (int)pending_capacity, (int)chunk, (int)L, (int)chunk, rowbytes};
  return launch_commit(a, B, stream, what);
}
