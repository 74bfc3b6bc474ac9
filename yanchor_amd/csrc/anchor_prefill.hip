// Anchor-memory prefill read: every query of a C-token block attends over the
// source tokens its block references (the block's prefix Top-K), with the
// zero-logit sink.  Replaces _indexed_forward / indexed_gqa
// (runtime/model/independent_memory.py:6-45) and indexed_gqa_torch / _gqa_tile
// (modeling_yanchor.py:22-42), called from IndependentGQAMemory._sequence
// (modeling_yanchor.py:249).
//
//   query       [B, NB, C, H, D]   bf16 / fp16
//   key, value  [KB, S, G, D]      KB == B, or 1 (one source shared by all rows)
//   references  [B, NB, G, CAP]    int32 / int64 index into S, -1 = none
//   out         [B, NB, C, H, D]
//
// Query head h belongs to group h / (H / G).  Per (b, block, g) the C * H/G
// query rows share one gathered set of CAP key/value rows, so the read is a
// small dense attention: S^T = K Q^T and O^T = V^T P^T on MFMA, with an
// online softmax whose running max starts at 0 and denominator at 1 (the
// sink logit 0 with value 0).  As in the reference, P enters the PV product as
// a hi + lo pair of 16-bit values, so the product keeps fp32 accuracy.
//
// A workgroup of 4 waves takes 128 of a block's C * H/G query rows (attn_tile.h);
// reference rows are gathered 64 at a time, straight into LDS.
//
// Source rows come in up to three parts (a state's committed slots, its
// pending slots, the new tokens), so a prefill that continues a state reads
// them where they are.
#include "anchor_source.h"
#include "attn_tile.h"

namespace yh {
namespace {

using attn::kD;

struct IdxArgs {
  const uint16_t* q;
  int64_t q_ts;
  AnchorSource src;
  const void* refs;
  uint16_t* out;   // [.., H, D]
  int64_t NB;
  int C, H, G, CAP, ref64;
  int per;         // blocks a workgroup walks
  float scale;
  // tokens in place (first != null): the query at block position
  // p = nb * C + t of row b is token p - first[b] of the row (src.token_row);
  // no token, no read, for p outside [first[b], first[b] + L); tokens past
  // counts[b] read nothing and get zeros (packed rows have none)
  const int64_t* first;
  const int64_t* counts;
};

// A workgroup walks `per` consecutive blocks of one (row, group) and one chunk
// of their query rows: a block has only a few tiles, so the first gather and
// the queries of the next block are in flight while the last tile of this one
// is computed (one block a workgroup left the chip waiting for both; the whole
// call at 32 rows of 2048 tokens, 256 slots: 794 us then, 743 us so).
//
// Workgroup id: group fastest, then the row chunk, so the chunks of a block
// gather their common rows through one XCD's L2 one after the other.
template <int DT, int NW>
__global__ void __launch_bounds__(NW * 64, 2) indexed_gqa_kernel(IdxArgs a) {
  static_assert(NW == 4, "the output stages in the 32 KB of one tile");
  __shared__ attn::Rows ktile[2], vtile[2];

  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int R = a.H / a.G, rows = a.C * R, chunks = (rows + NW * attn::kRows - 1) / (NW * attn::kRows);
  const int g = blockIdx.x % a.G;
  unsigned rest = blockIdx.x / a.G;
  const int m0 = (rest % chunks) * NW * attn::kRows + w * attn::kRows;
  rest /= chunks;
  const unsigned segs = static_cast<unsigned>((a.NB + a.per - 1) / a.per);
  const int64_t b = rest / segs;
  int64_t nb = static_cast<int64_t>(rest % segs) * a.per;
  const int blocks = static_cast<int>(min(a.NB - nb, static_cast<int64_t>(a.per)));

  // query row m of block n -> its row of q / out, -1 for none; live: it reads
  auto query_row = [&](int64_t n, int m, bool& live) -> int64_t {
    asm volatile("" : "+v"(m));   // its quotients are formed where used, not kept over the blocks in registers
    live = m < rows;
    if (!live) return -1;
    const int t = static_cast<unsigned>(m) % static_cast<unsigned>(a.C);
    if (a.first == nullptr) return (b * a.NB + n) * a.C + t;
    const int64_t i = n * a.C + t - a.first[b];
    live = i >= 0 && i < a.src.L;
    if (!live) return -1;
    if (a.counts != nullptr && i >= a.counts[b]) live = false;
    if (!live && a.src.bases != nullptr) return -1;   // packed: the next row's tokens
    return a.src.token_row(b, static_cast<int>(i));
  };
  attn::State<DT, true> st;
  auto load_queries = [&](int64_t n) -> bool {   // whether any query of the wave reads
    int m = m0 + (lane & 31);
    asm volatile("" : "+v"(m));
    bool live;
    const int64_t qrow = query_row(n, m, live);
    st.load_q(a.q + (live ? qrow * a.q_ts + (g * R + static_cast<unsigned>(m) / static_cast<unsigned>(a.C)) * kD : 0),
              live);
    return __any(live);
  };

  const int tiles = max(1, (a.CAP + attn::kTile - 1) / attn::kTile);   // of a block
  const int64_t ref_base = (b * a.NB * a.G + g) * a.CAP, ref_block = static_cast<int64_t>(a.G) * a.CAP;
  // this lane's reference of a tile, -1 for none; the tiles one after the other
  int64_t ref_nb = nb;
  int ref_left = blocks, ref_start = 0;
  auto next_ref = [&]() -> int {
    int64_t r = -1;
    if (ref_left > 0 && ref_start + lane < a.CAP) {
      const int64_t at = ref_base + ref_nb * ref_block + ref_start + lane;
      r = a.ref64 ? static_cast<const int64_t*>(a.refs)[at] : static_cast<const int32_t*>(a.refs)[at];
    }
    ref_start += attn::kTile;
    if (ref_start >= a.CAP) {
      ref_start = 0;
      ++ref_nb;
      --ref_left;
    }
    return r >= 0 && r < a.src.S ? static_cast<int>(r) : -1;
  };
  auto gather = [&](int buf, int ref) {     // lane l's reference is row l of the tile
    const uint16_t *kp = reinterpret_cast<const uint16_t*>(attn::zero_row), *vp = kp;
    if (ref >= 0) {
      kp = static_cast<const uint16_t*>(a.src.row(0, b, ref, g));
      vp = static_cast<const uint16_t*>(a.src.row(1, b, ref, g));
    }
    const uint64_t ka = reinterpret_cast<uint64_t>(kp), va = reinterpret_cast<uint64_t>(vp);
    attn::load_rows<NW>(ktile[buf], [&](int row, int e, const void* l) {
      attn::copy16(reinterpret_cast<const uint16_t*>(__shfl(ka, row, 64)) + e, l);
    });
    attn::load_rows<NW>(vtile[buf], [&](int row, int e, const void* l) {
      attn::copy16(reinterpret_cast<const uint16_t*>(__shfl(va, row, 64)) + e, l);
    });
  };
  const float k2 = a.scale * 1.4426950408889634f;
  int ref = next_ref();
  st.init(true);
  bool wave_live = load_queries(nb);
  uint64_t have = __ballot(ref >= 0), next = 0;
  if (have) gather(0, ref);
  ref = next_ref();
  int buf = 0, tile = 0;
  for (int left = blocks; left > 0; buf ^= 1) {
    attn::copy_wait();
    attn::tile_barrier();
    next = __ballot(ref >= 0);   // the same in every wave
    if (next) gather(buf ^ 1, ref);
    ref = next_ref();
    const bool last = ++tile == tiles;
    bool live_after = false;
    if (have && wave_live) {
      attn::f32x16 c[2];
      st.scores(ktile[buf], c);
      if (last && left > 1) live_after = load_queries(nb + 1);   // the scores are the last use of this block's
      if (have != ~0ull)
        st.mask(c, [&](int key, int half) { return (have >> (key + 4 * half)) & 1; });
      st.template step<true, false>(c, vtile[buf], k2);
    } else if (last && left > 1) {
      live_after = load_queries(nb + 1);
    }
    have = next;
    if (!last) continue;
    attn::tile_barrier();   // the tile is consumed: its LDS stages the output
    st.store((w < 2 ? &ktile[buf][0] : &vtile[buf][0]) + (w & 1) * attn::kRows * 16, [&](int row, int d0, uint4 o) {
      bool lv;
      int m = m0 + row;
      asm volatile("" : "+v"(m));
      const int64_t orow = query_row(nb, m, lv);
      if (orow < 0) return;
      if (!lv) o = make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(a.out + (orow * a.H + g * R + static_cast<unsigned>(m) / static_cast<unsigned>(a.C)) * kD + d0) = o;
    });
    st.init(true);
    wave_live = live_after;
    tile = 0;
    ++nb;
    --left;
  }
  attn::copy_wait();
}

int launch_indexed(IdxArgs a, int64_t B, int dtype, yh_stream_t stream, const char* what) {
  constexpr int kWaves = 4;
  const int64_t groups = B * a.NB * a.G;
  if (groups == 0) return YH_OK;
  const int64_t chunks = (static_cast<int64_t>(a.C) * (a.H / a.G) + kWaves * attn::kRows - 1) / (kWaves * attn::kRows);
  // blocks a workgroup: as many as leave four workgroups for each of the 512
  // that the chip holds
  const int64_t per = groups * chunks / 2048;
  a.per = static_cast<int>(per < 1 ? 1 : per > 8 ? 8 : per);
  const int64_t wgs = B * ((a.NB + a.per - 1) / a.per) * a.G * chunks;
  YH_CHECK_ARG(groups < (1ll << 31) && wgs < (1ll << 32) / (kWaves * 64), "%s: grid too large", what);
  const dim3 grid(static_cast<unsigned>(wgs)), block(kWaves * 64);
  a.scale = 1.f / sqrtf(static_cast<float>(kD));
  if (dtype == YH_BF16)
    hipLaunchKernelGGL((indexed_gqa_kernel<YH_BF16, kWaves>), grid, block, 0, static_cast<hipStream_t>(stream), a);
  else
    hipLaunchKernelGGL((indexed_gqa_kernel<YH_F16, kWaves>), grid, block, 0, static_cast<hipStream_t>(stream), a);
  YH_CHECK_LAUNCH(what);
  return YH_OK;
}

int check_indexed(const void* query, const void* key, const void* value, const void* references, int ref_dtype,
                  const void* out, int64_t B, int64_t NB, int64_t C, int64_t H, int64_t G, int64_t D, int64_t KB,
                  int64_t S, int64_t CAP, int64_t L, int dtype, const char* what) {
  YH_CHECK_ARG(B >= 0 && NB >= 0 && C > 0 && H > 0 && G > 0 && H % G == 0 && S >= 0 && CAP >= 0 && L >= 0,
               "%s: bad sizes", what);
  YH_CHECK_ARG(D == kD, "%s: head dim must be %d", what, kD);
  YH_CHECK_ARG(KB == 1 || KB == B, "%s: key batch must be 1 or B", what);
  YH_CHECK_ARG(ref_dtype == YH_I32 || ref_dtype == YH_I64, "%s: references must be int32 or int64", what);
  if (dtype != YH_BF16 && dtype != YH_F16) {
    set_error("%s: dtype must be bf16 or fp16", what);
    return YH_ERR_UNSUPPORTED;
  }
  if (B * NB * G == 0) return YH_OK;
  YH_CHECK_ARG(query && key && value && out && (CAP == 0 || references), "%s: null pointer", what);
  YH_CHECK_ARG(((reinterpret_cast<uintptr_t>(query) | reinterpret_cast<uintptr_t>(key) |
                 reinterpret_cast<uintptr_t>(value) | reinterpret_cast<uintptr_t>(out)) & 15) == 0,
               "%s: tensors must be 16-byte aligned", what);
  YH_CHECK_ARG(C * (H / G) < (1ll << 20) && L < (1ll << 31) && S < (1ll << 31) && CAP < (1ll << 30),
               "%s: grid too large", what);
  return YH_OK;
}

}  // namespace
}  // namespace yh

extern "C" int yh_indexed_gqa(const void* query, const void* key, const void* value, const void* references,
                              int ref_dtype, void* out, int64_t B, int64_t NB, int64_t C, int64_t H, int64_t G,
                              int64_t D, int64_t KB, int64_t S, int64_t CAP, int dtype, yh_stream_t stream) {
  using namespace yh;
  const int rc = check_indexed(query, key, value, references, ref_dtype, out, B, NB, C, H, G, D, KB, S, CAP, 0, dtype,
                               "indexed_gqa");
  if (rc != YH_OK || B * NB * G == 0) return rc;
  IdxArgs a{static_cast<const uint16_t*>(query), H * D, assembled_source(key, value, KB == 1 ? 0 : S, S, G, D * 2),
            references, static_cast<uint16_t*>(out), NB, (int)C, (int)H, (int)G, (int)CAP,
            ref_dtype == YH_I64 ? 1 : 0, 1, 0.f, nullptr, nullptr};
  return launch_indexed(a, B, dtype, stream, "indexed_gqa");
}

extern "C" int yh_anchor_sequence_read(const void* query, const void* key, const void* value,
                                       const void* references, int ref_dtype, const int64_t* first, void* out,
                                       int64_t B, int64_t L, int64_t NB, int64_t C, int64_t H, int64_t G, int64_t D,
                                       int64_t S, int64_t CAP, int dtype, yh_stream_t stream) {
  using namespace yh;
  YH_CHECK_ARG(first != nullptr || B == 0, "anchor_sequence_read: null pointer");
  const int rc = check_indexed(query, key, value, references, ref_dtype, out, B, NB, C, H, G, D, B, S, CAP, L, dtype,
                               "anchor_sequence_read");
  if (rc != YH_OK || B * NB * G == 0) return rc;
  IdxArgs a{static_cast<const uint16_t*>(query), H * D, assembled_source(key, value, S, S, G, D * 2), references,
            static_cast<uint16_t*>(out), NB, (int)C, (int)H, (int)G, (int)CAP, ref_dtype == YH_I64 ? 1 : 0, 1, 0.f,
            first, nullptr};
  a.src.L = (int)L;        // query rows: token i of row b at b * L + i
  a.src.batch_rows = L;
  return launch_indexed(a, B, dtype, stream, "anchor_sequence_read");
}

extern "C" int yh_anchor_tokens_read(const void* query, int64_t query_stride, const void* key, int64_t key_stride,
                                     const void* value, int64_t value_stride, const void* keys, const void* values,
                                     const void* pending_keys, const void* pending_values, const int32_t* references,
                                     const int64_t* first, const int64_t* counts, const int64_t* bases,
                                     const int32_t* order, void* out, int64_t B, int64_t L, int64_t NB, int64_t C,
                                     int64_t H, int64_t G, int64_t D, int64_t capacity, int64_t pending_capacity,
                                     int dtype, yh_stream_t stream) {
  using namespace yh;
  const char* what = "anchor_tokens_read";
  YH_CHECK_ARG(capacity > 0 && pending_capacity >= C, "%s: bad sizes", what);
  const int rc = check_indexed(query, key, value, references, YH_I32, out, B, NB, C, H, G, D, B, capacity + C + L,
                               capacity, L, dtype, what);
  if (rc != YH_OK || B * NB * G == 0) return rc;
  YH_CHECK_ARG(keys && values && pending_keys && pending_values && first && counts, "%s: null pointer", what);
  YH_CHECK_ARG(((reinterpret_cast<uintptr_t>(keys) | reinterpret_cast<uintptr_t>(values) |
                 reinterpret_cast<uintptr_t>(pending_keys) | reinterpret_cast<uintptr_t>(pending_values)) & 15) == 0 &&
                   query_stride % 8 == 0 && key_stride % 8 == 0 && value_stride % 8 == 0 && query_stride >= H * D &&
                   key_stride >= G * D && value_stride >= G * D,
               "%s: rows must be 16-byte aligned and hold whole heads", what);
  IdxArgs a{static_cast<const uint16_t*>(query), query_stride,
            state_source(keys, values, pending_keys, pending_values, key, key_stride * 2, value, value_stride * 2, bases,
                         order, L, C, G, capacity, pending_capacity, D * 2),
            references, static_cast<uint16_t*>(out), NB, (int)C, (int)H, (int)G, (int)capacity, 0, 1, 0.f, first, counts};
  return launch_indexed(a, B, dtype, stream, what);
}
