// Refill prefill of a packed, ragged set of prompt pieces (cu_seqlens), each
// piece continuing its sequence's caches:
//
//   conv_prefill_kernel   the GDN layer's causal conv1d + SiLU over every token
//                         of every piece, the first K-1 taps of a piece taken
//                         from the sequence's conv window (the causal-conv1d
//                         prefill call of the CUDA backend, modeling_yanchor.py:
//                         392-407; torch form wheel transformers/models/qwen3_5/
//                         modeling_qwen3_5.py:455-470).  One rounding: fp32
//                         taps in the decode prologue's order, SiLU, bf16.
//   conv_window_kernel    the conv window left behind: the last K-1 inputs of
//                         [window | piece].
//   swa_prefill_kernel    sliding-window causal attention of every query over
//                         the W keys ending at its own position (flash_swa /
//                         reference_swa, modeling_yanchor.py:412-449), the keys
//                         before the piece read from the sequence's physical
//                         ring (slot = position mod W), GQA, and the output
//                         gate read * sigmoid(gate) of Qwen3_5FixedWindowAttention
//                         (modeling_yanchor.py:871-875) in the store.
//   ring_fill_kernel      the last min(W, L) keys / values / positions of each
//                         piece into its ring slots (the chronological ring of
//                         runtime/model/inference_kernels.py:1799-1856, built
//                         in place).
//
// swa_prefill_kernel: a tile is 64 query rows, 64 / R consecutive tokens x the
// R query heads of a KV group.  A workgroup of NW waves takes NW / 2 tiles that
// follow each other in the list, two waves each; tiles of one piece whose windows
// meet share their key tiles (attn_tile.h).
#include <type_traits>

#include "attn_tile.h"

namespace yh {
namespace {

__device__ __forceinline__ float silu(float x) { return x / (1.f + expf(-x)); }

// Sequence of packed token n: the last r with cu[r] <= n (cu ascending,
// empty pieces allowed).
__device__ __forceinline__ int seq_of(const int32_t* cu, int nseq, int64_t n) {
  int lo = 0, hi = nseq - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= n) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// ---------------------------------------------------------------------------
// conv: x = proj[:, :C] of the packed tokens; window [R, 3, C] time-major
// (oldest first); w [C, 4].  y[n, c] = bf16(silu(sum_j x(t - 3 + j) w[c, j]))
// with x(u < 0) = window[r, 3 + u].
struct ConvArgs {
  const uint16_t* proj;
  int64_t P;
  const uint16_t* window;
  const uint16_t* w;
  const int32_t* cu;
  uint16_t* y;         // [C / Cp, total, Cp]
  int64_t C, Cp;
  int nseq;
};

// VEC consecutive bf16 channels of a row: 16 bytes in one access (VEC = 8),
// or one element where a row does not keep 16-byte alignment (VEC = 1).
template <int VEC>
struct Chan;
template <>
struct Chan<8> {
  typedef uint4 T;
  static __device__ __forceinline__ float f32(const T& x, int i) {
    const uint32_t w = i < 2 ? x.x : i < 4 ? x.y : i < 6 ? x.z : x.w;
    return __uint_as_float((i & 1) ? (w & 0xffff0000u) : (w << 16));
  }
  static __device__ __forceinline__ T pack(const float (&y)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = attn::Mfma<YH_BF16>::round2(y[2 * i], y[2 * i + 1]);
    return make_uint4(w[0], w[1], w[2], w[3]);
  }
};
template <>
struct Chan<1> {
  typedef uint16_t T;
  static __device__ __forceinline__ float f32(const T& x, int) { return bf16_to_f32(x); }
  static __device__ __forceinline__ T pack(const float (&y)[1]) { return f32_to_bf16(y[0]); }
};

constexpr int kConvBatch = 4;  // rows in flight per thread

// Bound by the VALU, which issues in 86 % of the cycles: 35 issue slots an
// element, most of them the SiLU's exact exp and division (HBM would take 140 us
// of the 240 below).  A thread owns VEC channels and walks a run of `run` tokens
// with the three earlier inputs and the four taps in registers, so a row is
// loaded once (plus three halo rows a run) in 16-byte accesses, four rows ahead
// of their use.  One token and one channel a thread (2-byte accesses, every row
// loaded four times, a sequence search a workgroup) took 976 us at 64 pieces of
// 17,400 tokens x 12288 channels (871 MB); this takes 247 us with the host's
// checks.
template <int VEC>
__global__ void __launch_bounds__(256) conv_prefill_kernel(ConvArgs a, int64_t total, int run) {
  using Ch = Chan<VEC>;
  typedef typename Ch::T T;
  const int64_t c = (static_cast<int64_t>(blockIdx.y) * 256 + threadIdx.x) * VEC;
  if (c >= a.C) return;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * run;
  const int64_t n1 = n0 + run < total ? n0 + run : total;
  int r = seq_of(a.cu, a.nseq, n0);
  int64_t s = a.cu[r], e = a.cu[r + 1];
  if (n0 >= e) return;   // tokens outside every piece
  const T* src = reinterpret_cast<const T*>(a.proj + c);
  const int64_t sp = a.P / VEC, sc = a.C / VEC, yc = a.Cp / VEC, plane = c / a.Cp;
  T* dst = reinterpret_cast<T*>(a.y + plane * total * a.Cp + (c - plane * a.Cp));

  float wt[4][VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    if constexpr (VEC == 8) {
      const uint2 w4 = *reinterpret_cast<const uint2*>(a.w + (c + i) * 4);
      wt[0][i] = __uint_as_float(w4.x << 16);
      wt[1][i] = __uint_as_float(w4.x & 0xffff0000u);
      wt[2][i] = __uint_as_float(w4.y << 16);
      wt[3][i] = __uint_as_float(w4.y & 0xffff0000u);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) wt[j][i] = bf16_to_f32(a.w[(c + i) * 4 + j]);
    }
  }
  // the inputs of kConvBatch tokens behind the three before them: token i of a
  // batch reads h[i .. i + 3], so nothing moves but the last three a batch
  float h[kConvBatch + 3][VEC];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int64_t u = n0 - s - 3 + j;
    T x{};
    if (n0 > s)
      x = u >= 0 ? src[(n0 - 3 + j) * sp]
                 : reinterpret_cast<const T*>(a.window + c)[(static_cast<int64_t>(r) * 3 + 3 + u) * sc];
#pragma unroll
    for (int i = 0; i < VEC; ++i) h[j][i] = Ch::f32(x, i);
  }
  for (int64_t nb = n0; nb < n1; nb += kConvBatch) {
    T x[kConvBatch];
#pragma unroll
    for (int i = 0; i < kConvBatch; ++i) x[i] = src[(nb + i < n1 ? nb + i : n1 - 1) * sp];
#pragma unroll
    for (int i = 0; i < kConvBatch; ++i) {
      const int64_t n = nb + i;
      if (n >= n1) break;
      if (n >= e) {   // the next piece that is not empty
        do ++r;
        while (r < a.nseq && a.cu[r + 1] <= n);
        if (r >= a.nseq) return;
        s = a.cu[r];
        e = a.cu[r + 1];
      }
#pragma unroll
      for (int v = 0; v < VEC; ++v) h[i + 3][v] = Ch::f32(x[i], v);
      if (n < s) continue;
      if (n == s) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          const T x0 = reinterpret_cast<const T*>(a.window + c)[(static_cast<int64_t>(r) * 3 + j) * sc];
#pragma unroll
          for (int v = 0; v < VEC; ++v) h[i + j][v] = Ch::f32(x0, v);
        }
      }
      float y[VEC];
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        float acc = h[i][v] * wt[0][v];
        acc = fmaf(h[i + 1][v], wt[1][v], acc);
        acc = fmaf(h[i + 2][v], wt[2][v], acc);
        acc = fmaf(h[i + 3][v], wt[3][v], acc);
        y[v] = silu(acc);
      }
      dst[n * yc] = Ch::pack(y);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int v = 0; v < VEC; ++v) h[j][v] = h[kConvBatch + j][v];
  }
}

// window[r, m] <- input at relative time L - 3 + m (m = 0, 1, 2): from the
// piece, or, for pieces shorter than 3 tokens, the old window shifted.  One
// thread owns VEC channels of a row and goes in ascending m, so every old
// entry is read before it is overwritten.
template <int VEC>
__global__ void __launch_bounds__(256) conv_window_kernel(ConvArgs a) {
  typedef typename Chan<VEC>::T T;
  const int r = blockIdx.x;
  const int64_t c = (static_cast<int64_t>(blockIdx.y) * 256 + threadIdx.x) * VEC;
  if (c >= a.C) return;
  const int64_t s0 = a.cu[r], len = a.cu[r + 1] - s0, sp = a.P / VEC, sc = a.C / VEC;
  T* win = reinterpret_cast<T*>(const_cast<uint16_t*>(a.window) + static_cast<int64_t>(r) * 3 * a.C + c);
  const T* src = reinterpret_cast<const T*>(a.proj + c);
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int64_t u = len - 3 + m;
    win[m * sc] = u >= 0 ? src[(s0 + u) * sp] : win[(3 + u) * sc];
  }
}

// ---------------------------------------------------------------------------
using attn::kD;

struct SwaArgs {
  const uint16_t* q;      // [N, H, D]
  int64_t q_ts;
  const uint16_t* k;      // [N, G, D] normed, rotated piece keys
  int64_t k_ts;
  const uint16_t* v;      // [N, G, D] piece values
  int64_t v_ts;
  const uint16_t* ring_k; // [RB, G, W, D]
  const uint16_t* ring_v;
  const int64_t* ring_row;  // [R], -1 = no ring context
  const int64_t* start;     // [R] position of each piece's first token
  const int32_t* cu;        // [R + 1]
  const int32_t* tiles;     // [n_tiles, 2] (piece, first token)
  const uint16_t* gate;   // [N, H, D] (token / head strides) or null
  int64_t g_ts, g_hs;
  uint16_t* out;          // [N, H, D]
  int64_t n_tiles;
  int H, G, W;
  int gate16;             // gate rows keep 16-byte alignment
  int off32;              // a tile's and a ring's byte offsets fit 31 bits
  float scale;
};

// Workgroup id: the KV group is the fastest index, so with 8 groups every XCD
// keeps one group's keys and values in its L2 while neighbouring tiles, whose
// windows overlap by all but a tile, run on it.  (A grid's row holds less than
// 2^32 threads: longer lists take further rows.)
template <int DT, int NW>
__global__ void __launch_bounds__(NW * 64, 2) swa_prefill_kernel(SwaArgs a) {
  using M = attn::Mfma<DT>;
  constexpr int kTiles = NW / 2;
  __shared__ attn::Rows stage[4];   // two buffers of key rows, two of value rows; then the output
  attn::Rows *ktile = stage, *vtile = stage + 2;

  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = blockIdx.x % a.G;
  const int64_t first = (static_cast<int64_t>(blockIdx.y) * (gridDim.x / a.G) + blockIdx.x / a.G) * kTiles;
  if (first >= a.n_tiles) return;
  const int count = static_cast<int>(a.n_tiles - first < kTiles ? a.n_tiles - first : kTiles);
  const int32_t* list = a.tiles + 2 * first;
  const int R = a.H / a.G, TT = attn::kTile / R, W = a.W;
  const int tshift = 31 - __builtin_clz(TT);

  // this wave's tile and this lane's query
  const bool active = (w >> 1) < count;
  const int mine = active ? w >> 1 : 0;
  const int r = list[2 * mine], t0 = list[2 * mine + 1];
  const int64_t s0 = a.cu[r];
  const int len = a.cu[r + 1] - a.cu[r];
  const int m0 = (w & 1) * attn::kRows, m = m0 + (lane & 31);
  const int tok = t0 + (m & (TT - 1));
  const int head = g * R + (m >> tshift);
  const bool mvalid = active && tok < len;

  attn::State<DT> st;
  st.init(false);
  st.load_q(a.q + (s0 + (mvalid ? tok : 0)) * a.q_ts + head * kD, mvalid);
  const float k2 = a.scale * 1.4426950408889634f;

  for (int i0 = 0; i0 < count;) {
    // the tiles i0 .. i1 - 1 of one piece whose windows meet: the union of their key ranges
    const int pr = list[2 * i0];
    int lo = list[2 * i0 + 1], hi = lo, i1 = i0 + 1;
    for (; i1 < count && list[2 * i1] == pr; ++i1) {
      const int t = list[2 * i1 + 1];
      if (max(hi, t) - min(lo, t) > W) break;   // nothing to share, and the keys between would be copied for nobody
      lo = min(lo, t);
      hi = max(hi, t);
    }
    const int64_t ps = a.cu[pr];
    const int plen = a.cu[pr + 1] - a.cu[pr];
    const int64_t start = a.start[pr], rrow = a.ring_row[pr];
    const int nctx = rrow < 0 ? 0 : static_cast<int>(start < W - 1 ? start : W - 1);
    const int j_hi = nctx + min(hi + TT, plen) - 1;   // inclusive, in [ring context | piece]
    const int j_lo = max(nctx + lo - W + 1, 0);
    const int64_t ring_base = rrow < 0 ? 0 : (rrow * a.G + g) * W;
    const int slot0 = static_cast<int>((start - nctx) % W);  // ring slot of key index 0
    // A tile's key (src = k, ring_k) or value rows into LDS.  A tile that lies
    // in the piece or in the ring goes through a buffer resource with 32-bit
    // offsets; the one across the seam by addresses.
    auto load = [&](attn::Rows& t, int j0, const uint16_t* src, int64_t ts, const uint16_t* ring) {
      if (j0 > j_hi) return;
      if (j0 >= nctx && a.off32) {
        const int left = min(j_hi - j0, attn::kTile - 1), bytes = static_cast<int>(ts) * 2;
        const auto rb = attn::buffer(src + (ps + j0 - nctx) * ts + g * kD, left * bytes + kD * 2);
        attn::load_rows<NW>(t, [&](int row, int e, const void* l) { attn::copy16(rb, row * bytes + e * 2, l); });
      } else if (j0 + attn::kTile <= nctx && a.off32) {
        const auto rb = attn::buffer(ring + ring_base * kD, W * kD * 2);
        attn::load_rows<NW>(t, [&](int row, int e, const void* l) {
          const unsigned slot = slot0 + j0 + row, wrapped = slot - W;   // j < W - 1
          attn::copy16(rb, static_cast<int>(min(slot, wrapped)) * (kD * 2) + e * 2, l);
        });
      } else {
        attn::load_rows<NW>(t, [&](int row, int e, const void* l) {
          const int j = j0 + row;
          const uint16_t* p = reinterpret_cast<const uint16_t*>(attn::zero_row);
          if (j < nctx)
            p = ring + (ring_base + (slot0 + j < W ? slot0 + j : slot0 + j - W)) * kD;
          else if (j <= j_hi)
            p = src + (ps + j - nctx) * ts + g * kD;
          attn::copy16(p + e, l);
        });
      }
    };
    // this wave's tokens: key tiles outside their windows are passed over
    const int self = nctx + tok;
    const int wtok = t0 + (m0 & (TT - 1)), wspan = min(TT, attn::kRows);
    const int wlo = nctx + wtok, whi = nctx + min(wtok + wspan, len) - 1;
    const bool in = active && mine >= i0 && mine < i1 && wtok < len;
    auto sees = [&](int j0) { return in && j0 <= whi && j0 + attn::kTile - 1 > wlo - W; };
    // the keys of such a tile that any of them sees: the others are a later
    // tile's, or the oldest of an earlier one
    auto seen = [&](int j0) {
      const int lo = max(wlo - W + 1 - j0, 0), hi = min(whi - j0, attn::kTile - 1);
      return (~0ull << (lo & 63)) & (~0ull >> ((attn::kTile - 1 - hi) & 63));
    };
    load(ktile[0], j_lo, a.k, a.k_ts, a.ring_k);
    load(vtile[0], j_lo, a.v, a.v_ts, a.ring_v);
    int buf = 0, j0 = j_lo;
    auto tile = [&](auto edge, uint64_t keep) {
      attn::copy_wait();      // this wave's part of the tile has arrived
      attn::tile_barrier();   // everyone's has, and the other buffers are consumed
      load(ktile[buf ^ 1], j0 + attn::kTile, a.k, a.k_ts, a.ring_k);
      load(vtile[buf ^ 1], j0 + attn::kTile, a.v, a.v_ts, a.ring_v);
      if (sees(j0)) {
        attn::f32x16 c[2];
        st.scores(ktile[buf], c);
        if constexpr (edge.value)
          st.mask(c, [&](int key, int half) {
            const int j = j0 + key + 4 * half;
            return j <= self && j > self - W;
          });
        st.template step<false, edge.value>(c, vtile[buf], k2, keep);
      }
      j0 += attn::kTile;
      buf ^= 1;
    };
    // Every key of an inner tile is live for every query of the wave.  The two
    // kinds take a loop each (the waves of a workgroup change over on their own:
    // both pass one barrier a tile): as branches of one loop they spill 97
    // registers, and a branch at each value operand costs 9 % of the kernel.
    auto inner = [&]() { return j0 + attn::kTile - 1 <= wlo && j0 > whi - W; };
    while (j0 <= j_hi) {
#pragma unroll 1
      while (j0 <= j_hi && inner()) tile(std::false_type{}, ~0ull);
#pragma unroll 1
      while (j0 <= j_hi && !inner()) tile(std::true_type{}, seen(j0));
    }
    attn::copy_wait();
    attn::tile_barrier();     // the buffers are consumed
    i0 = i1;
  }

  if (!active) return;
  static_assert(NW * attn::kRows * 16 <= sizeof(stage) / 16, "output staging");
  st.store(&stage[0][0] + w * attn::kRows * 16, [&](int row, int d0, uint4 o) {
    const int mm = m0 + row, tk = t0 + (mm & (TT - 1)), hd = g * R + (mm >> tshift);
    if (tk >= len) return;
    if (a.gate) {   // read * sigmoid(gate), each product rounded as the torch ops round it
      const uint16_t* grow = a.gate + (s0 + tk) * a.g_ts + hd * a.g_hs + d0;
      uint32_t gw[4], ow[4] = {o.x, o.y, o.z, o.w};
      if (a.gate16) {
        const uint4 x = *reinterpret_cast<const uint4*>(grow);
        gw[0] = x.x;
        gw[1] = x.y;
        gw[2] = x.z;
        gw[3] = x.w;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) gw[i] = attn::pack2(grow[2 * i], grow[2 * i + 1]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        uint16_t y[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const uint16_t sg = M::round(1.f / (1.f + __expf(-M::widen(static_cast<uint16_t>(gw[i] >> (16 * e))))));
          y[e] = M::round(M::widen(static_cast<uint16_t>(ow[i] >> (16 * e))) * M::widen(sg));
        }
        ow[i] = attn::pack2(y[0], y[1]);
      }
      o = make_uint4(ow[0], ow[1], ow[2], ow[3]);
    }
    *reinterpret_cast<uint4*>(a.out + ((s0 + tk) * a.H + hd) * kD + d0) = o;
  });
}

// ---------------------------------------------------------------------------
// ring_fill: block per packed token; the last min(W, L) tokens of each piece
// write their key / value rows (all G heads, 16 B per thread) and position.
struct FillArgs {
  const uint16_t* k;
  int64_t k_ts;
  const uint16_t* v;
  int64_t v_ts;
  const int64_t* ring_row;
  const int64_t* start;
  const int32_t* cu;
  uint16_t* ring_k;
  uint16_t* ring_v;
  int32_t* ring_pos;
  int G, W, nseq;
};

__global__ void __launch_bounds__(256) ring_fill_kernel(FillArgs a) {
  const int64_t n = blockIdx.x;
  const int r = seq_of(a.cu, a.nseq, n);
  const int64_t t = n - a.cu[r], len = a.cu[r + 1] - a.cu[r];
  const int64_t rrow = a.ring_row[r];
  if (t < 0 || t >= len) return;           // a token outside every piece
  if (rrow < 0 || t < len - a.W) return;   // overwritten by a later token of the piece
  const int64_t pos = a.start[r] + t;
  const int64_t slot = pos % a.W;
  for (int e = threadIdx.x; e < a.G * (kD / 8); e += blockDim.x) {
    const int g = e / (kD / 8), c8 = (e % (kD / 8)) * 8;
    const int64_t dst = ((rrow * a.G + g) * a.W + slot) * kD + c8;
    *reinterpret_cast<uint4*>(a.ring_k + dst) = *reinterpret_cast<const uint4*>(a.k + n * a.k_ts + g * kD + c8);
    *reinterpret_cast<uint4*>(a.ring_v + dst) = *reinterpret_cast<const uint4*>(a.v + n * a.v_ts + g * kD + c8);
    if (c8 == 0) a.ring_pos[(rrow * a.G + g) * a.W + slot] = static_cast<int32_t>(pos);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace yh

extern "C" int yh_conv_prefill(const void* proj, int64_t proj_stride, void* window, const void* conv_w,
                               const int32_t* cu_seqlens, int64_t n_seqs, int64_t total_tokens, int64_t channels,
                               void* out, int dtype, yh_stream_t stream) {
  using namespace yh;
  YH_CHECK_ARG(n_seqs >= 0 && total_tokens >= 0 && channels > 0 && proj_stride >= channels,
               "conv_prefill: bad sizes");
  YH_CHECK_ARG(dtype >= 0 && (dtype & 0xff) == YH_BF16, "conv_prefill: activations must be bfloat16");
  const int64_t planes = dtype >> 8 > 0 ? dtype >> 8 : 1;
  YH_CHECK_ARG(channels % planes == 0, "conv_prefill: planes must divide the channels");
  if (n_seqs == 0) return YH_OK;
  YH_CHECK_ARG(proj && window && conv_w && cu_seqlens && (out || total_tokens == 0), "conv_prefill: null pointer");
  YH_CHECK_ARG(total_tokens < (1ll << 31) && n_seqs < (1ll << 31), "conv_prefill: sizes too large");
  hipStream_t st = static_cast<hipStream_t>(stream);
  ConvArgs c{static_cast<const uint16_t*>(proj), proj_stride, static_cast<const uint16_t*>(window),
             static_cast<const uint16_t*>(conv_w), cu_seqlens, static_cast<uint16_t*>(out), channels,
             channels / planes, (int)n_seqs};
  // 16-byte channel groups where every row of every tensor keeps them aligned
  const bool vec = channels / planes % 8 == 0 && proj_stride % 8 == 0 && aligned16(proj) && aligned16(window) &&
                   aligned16(out) && (reinterpret_cast<uintptr_t>(conv_w) & 7) == 0;
  const int64_t per_block = 256 * (vec ? 8 : 1);
  const unsigned cb = static_cast<unsigned>((channels + per_block - 1) / per_block);
  if (total_tokens > 0) {
    // run: tokens a thread walks.  Long runs save the three halo rows; short
    // ones keep 8 workgroups a CU in flight when there are few tokens.
    const int64_t want = total_tokens * cb / 2048 / kConvBatch * kConvBatch;
    const int run = static_cast<int>(want < kConvBatch ? kConvBatch : want > 64 ? 64 : want);
    const dim3 grid(static_cast<unsigned>((total_tokens + run - 1) / run), cb);
    if (vec)
      hipLaunchKernelGGL(conv_prefill_kernel<8>, grid, dim3(256), 0, st, c, total_tokens, run);
    else
      hipLaunchKernelGGL(conv_prefill_kernel<1>, grid, dim3(256), 0, st, c, total_tokens, run);
    YH_CHECK_LAUNCH("conv_prefill");
  }
  const dim3 wgrid(static_cast<unsigned>(n_seqs), cb);
  if (vec)
    hipLaunchKernelGGL(conv_window_kernel<8>, wgrid, dim3(256), 0, st, c);
  else
    hipLaunchKernelGGL(conv_window_kernel<1>, wgrid, dim3(256), 0, st, c);
  YH_CHECK_LAUNCH("conv_prefill window");
  return YH_OK;
}

extern "C" int yh_swa_prefill(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                              int64_t v_stride, const void* ring_k, const void* ring_v, const int64_t* ring_rows,
                              const int64_t* starts, const int32_t* cu_seqlens, const int32_t* tiles,
                              int64_t n_tiles, const void* gate, int64_t gate_token_stride,
                              int64_t gate_head_stride, void* out, int64_t n_seqs, int64_t ring_batch, int64_t H,
                              int64_t G, int64_t D, int64_t window, int dtype, yh_stream_t stream) {
  using namespace yh;
  YH_CHECK_ARG(n_seqs >= 0 && n_tiles >= 0 && H > 0 && G > 0 && H % G == 0 && window > 0 && ring_batch >= 0,
               "swa_prefill: bad sizes");
  YH_CHECK_ARG(D == kD, "swa_prefill: head dim must be %d", kD);
  YH_CHECK_ARG(64 % (H / G) == 0, "swa_prefill: query heads per KV head must divide 64");
  if (dtype != YH_BF16 && dtype != YH_F16) {
    set_error("swa_prefill: dtype must be bf16 or fp16");
    return YH_ERR_UNSUPPORTED;
  }
  if (n_tiles == 0) return YH_OK;
  YH_CHECK_ARG(q && k && v && out && starts && ring_rows && cu_seqlens && tiles, "swa_prefill: null pointer");
  YH_CHECK_ARG(ring_batch == 0 || (ring_k && ring_v), "swa_prefill: null ring");
  YH_CHECK_ARG(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out) && (!ring_k || aligned16(ring_k)) &&
                   (!ring_v || aligned16(ring_v)),
               "swa_prefill: tensors must be 16-byte aligned");
  YH_CHECK_ARG(q_stride % 8 == 0 && k_stride % 8 == 0 && v_stride % 8 == 0 && q_stride >= H * D && k_stride >= G * D &&
                   v_stride >= G * D,
               "swa_prefill: token strides must hold whole heads and keep 16-byte rows");
  YH_CHECK_ARG(!gate || (gate_head_stride >= D && gate_token_stride >= H * gate_head_stride),
               "swa_prefill: bad gate strides");
  YH_CHECK_ARG(n_tiles < (1ll << 31) && G < 65536 && window < (1ll << 30), "swa_prefill: grid too large");
  const bool off32 = k_stride < (1ll << 23) && v_stride < (1ll << 23) && window < (1ll << 22);
  const bool gate16 = gate && aligned16(gate) && gate_token_stride % 8 == 0 && gate_head_stride % 8 == 0;
  SwaArgs a{static_cast<const uint16_t*>(q), q_stride, static_cast<const uint16_t*>(k), k_stride,
            static_cast<const uint16_t*>(v), v_stride, static_cast<const uint16_t*>(ring_k),
            static_cast<const uint16_t*>(ring_v), ring_rows, starts, cu_seqlens, tiles,
            static_cast<const uint16_t*>(gate), gate_token_stride, gate_head_stride, static_cast<uint16_t*>(out),
            n_tiles, (int)H, (int)G, (int)window, gate16 ? 1 : 0, off32 ? 1 : 0, 1.f / sqrtf(static_cast<float>(D))};
  // Two tiles a workgroup: with four, fewer copies a tile gain nothing on long
  // prompts (385 and 390 us at 16 pieces of 15,465 tokens with context) and
  // short ones leave the chip emptier (45 and 38 us for 1000 tokens).
  constexpr int kWaves = 4;
  const int64_t pairs = (n_tiles + kWaves / 2 - 1) / (kWaves / 2), row = ((1ll << 32) / (kWaves * 64) - 1) / G;
  const int64_t wide = pairs < row ? pairs : row;
  const dim3 grid(static_cast<unsigned>(wide * G), static_cast<unsigned>((pairs + wide - 1) / wide));
  const dim3 block(kWaves * 64);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == YH_BF16)
    hipLaunchKernelGGL((swa_prefill_kernel<YH_BF16, kWaves>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((swa_prefill_kernel<YH_F16, kWaves>), grid, block, 0, st, a);
  YH_CHECK_LAUNCH("swa_prefill");
  return YH_OK;
}

extern "C" int yh_ring_fill(const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                            const int64_t* ring_rows, const int64_t* starts, const int32_t* cu_seqlens,
                            int64_t n_seqs, int64_t total_tokens, void* ring_k, void* ring_v, int32_t* ring_pos,
                            int64_t G, int64_t D, int64_t window, int dtype, yh_stream_t stream) {
  using namespace yh;
  YH_CHECK_ARG(n_seqs >= 0 && total_tokens >= 0 && G > 0 && window > 0, "ring_fill: bad sizes");
  YH_CHECK_ARG(D == kD, "ring_fill: head dim must be %d", kD);
  YH_CHECK_ARG(dtype == YH_BF16 || dtype == YH_F16, "ring_fill: dtype must be bf16 or fp16");
  if (total_tokens == 0 || n_seqs == 0) return YH_OK;
  YH_CHECK_ARG(k && v && ring_rows && starts && cu_seqlens && ring_k && ring_v && ring_pos, "ring_fill: null pointer");
  YH_CHECK_ARG(aligned16(k) && aligned16(v) && aligned16(ring_k) && aligned16(ring_v) && k_stride % 8 == 0 &&
                   v_stride % 8 == 0 && k_stride >= G * D && v_stride >= G * D,
               "ring_fill: rows must be 16-byte aligned");
  YH_CHECK_ARG(total_tokens < (1ll << 31), "ring_fill: sizes too large");
  FillArgs a{static_cast<const uint16_t*>(k), k_stride, static_cast<const uint16_t*>(v), v_stride, ring_rows, starts,
             cu_seqlens, static_cast<uint16_t*>(ring_k), static_cast<uint16_t*>(ring_v), ring_pos, (int)G,
             (int)window, (int)n_seqs};
  hipLaunchKernelGGL(ring_fill_kernel, dim3(static_cast<unsigned>(total_tokens)), dim3(128), 0,
                     static_cast<hipStream_t>(stream), a);
  YH_CHECK_LAUNCH("ring_fill");
  return YH_OK;
}
