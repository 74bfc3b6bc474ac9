// Dense attention over key / value rows staged through LDS on 32x32x16 MFMA,
// shared by the sliding-window prefill and the anchor-memory prefill read.
//
// A wave owns 32 query rows; a workgroup of NW waves shares the key tiles.
// Per 64-key tile and wave:
//   S^T = K Q^T      lane (query lane % 32, half lane / 32) ends with the
//                    scores of 32 of the 64 keys of its query
//   O^T += V^T P^T   P is already where the B operand wants it: reduction slot
//                    e of half h in step s stands for key
//                    16 s + 8 (e / 4) + 4 h + e % 4, and the V operand is read
//                    in that order by transposing LDS reads
// so neither P nor O leaves registers.
//
// What bounds it: the softmax's vector work (a fma, a quarter-rate exp2, half a
// conversion and an addition a score, and a rescaling of the accumulators a
// tile).  A wave's tile costs a SIMD 3460 cycles in window attention over 16
// pieces of 15,465 tokens with full rings: vector instructions issue in 1970 of
// them, the MFMAs take 1024, and two waves a SIMD overlap the two only in part;
// the rest is waits on LDS and on the tile's barrier.  Hence: key tiles by direct
// global-to-LDS copies, double buffered, one barrier a tile; 16-byte pieces
// swizzled so that the 16-byte K reads and the transposing V reads hit distinct
// banks; a few operands read ahead of their MFMA; the exponentials of one step of
// the value product between the MFMAs of the step before; a raised wave priority
// around the MFMAs, so that they run under the other wave's vector work; no mask
// code on tiles where every key is live.  Six waves a workgroup (three a SIMD,
// 168 registers) take 1.4 times as long even with the addresses re-formed a
// tile.  The denominator sums P in float32, before the rounding that the value
// product sees.  (A running maximum that lags the scores by up to 2^8 and leaves
// out most rescalings was 10 % faster and 2 % further from float64: a row's
// largest probability is exact only while the maximum is.)
#pragma once
#include "common.h"

namespace yh {
namespace attn {

constexpr int kD = 128;      // head dim
constexpr int kTile = 64;    // keys per tile
constexpr int kRows = 32;    // query rows per wave

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4v lds_s16x4v;

template <int DT>
struct Mfma;
template <>
struct Mfma<YH_BF16> {
  typedef bf16x8_t vec;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t round2(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, bf16x2_t));
  }
  static __device__ __forceinline__ uint16_t round(float x) { return f32_to_bf16(x); }
  static __device__ __forceinline__ float widen(uint16_t h) { return bf16_to_f32(h); }
};
template <>
struct Mfma<YH_F16> {
  typedef f16x8_t vec;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t round2(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, f16x2_t));
  }
  static __device__ __forceinline__ uint16_t round(float x) { return f32_to_f16(x); }
  static __device__ __forceinline__ float widen(uint16_t h) { return f16_to_f32(h); }
};

__device__ __forceinline__ uint32_t pack2(uint16_t lo, uint16_t hi) {
  return static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16);
}

// 64 key or value rows of 16 pieces, piece p of row r at p ^ swz(r).  K reads
// take one piece of 32 consecutive rows, V reads four pieces of four rows:
// swz maps both to distinct pieces of a 256-byte row.
typedef uint4 Rows[kTile * 16];
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// 16 bytes a lane from global memory into LDS at `lds` (wave-uniform) + 16 l.
// Inline assembly, because the compiler would make every later LDS read wait
// for a copy that it can see; copy_wait() (then a barrier) is the wait.  (The
// LDS offset is the low half of the flat address of an LDS object.)
__device__ __forceinline__ void copy16(const void* src, const void* lds) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m0v), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ void copy_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void tile_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The same through a buffer resource (wave-uniform) at byte offset `voff`;
// bytes past the resource arrive as zeros.
__device__ __forceinline__ void copy16(__amdgpu_buffer_rsrc_t r, int voff, const void* lds) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>(lds)));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(m0v), "v"(voff), "s"(r)
               : "memory", "m0");
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const uint16_t* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), 0, bytes, 0x00020000);
}

// A row of zeros for keys that do not exist (their probability is 0, and 0
// times their value has to be 0).
__device__ const uint4 zero_row[kD / 8] = {};

// The 64 rows of a tile into LDS by all NW waves, 4 rows an instruction:
// copy(row of the tile, first element of the piece, its LDS).
template <int NW, class CopyFn>
__device__ __forceinline__ void load_rows(Rows& t, CopyFn copy) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int it = 0; it < 16 / NW; ++it) {
    const int bl = it * NW + w, r = 4 * bl + (lane >> 4);
    copy(r, ((lane & 15) ^ swz(r)) * 8, &t[64 * bl]);
  }
}

// FRESH: LDS addresses are formed in every tile instead of staying in registers
// over the tile loop, where a kernel's own invariants leave no room for them (a
// spilled one is reloaded behind the copies in flight).
template <int DT, bool FRESH = false>
struct State {
  static __device__ __forceinline__ int lane_id() {
    int lane = threadIdx.x & 63;
    if constexpr (FRESH) asm volatile("" : "+v"(lane));
    return lane;
  }
  typename Mfma<DT>::vec q[8];  // Q^T: dims 16 s + 8 half .. + 7 of the lane's query
  f32x16 acc[4];                // O^T: dim 32 t + 8 (i / 4) + 4 half + i % 4
  float base;                   // running maximum, log2 units
  float den;                    // this half's share of the denominator

  // sink: a logit 0 with value 0 takes part in the softmax
  __device__ __forceinline__ void init(bool sink) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
    base = sink ? 0.f : -3.0e38f;
    den = sink && (threadIdx.x & 32) == 0 ? 1.f : 0.f;
  }
  __device__ __forceinline__ void load_q(const uint16_t* row, bool valid) {
    const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      uint4 x = make_uint4(0, 0, 0, 0);
      if (valid) x = *reinterpret_cast<const uint4*>(row + s * 16 + half * 8);
      q[s] = __builtin_bit_cast(typename Mfma<DT>::vec, x);
    }
  }
  // Raw scores of a tile: c[kt][i] is key 32 kt + 8 (i / 4) + 4 half + i % 4.
  __device__ __forceinline__ void scores(const Rows& k, f32x16 (&c)[2]) {
    using M = Mfma<DT>;
    using vec = typename M::vec;
    const int lane = lane_id(), half = lane >> 5;
    constexpr int kAhead = 4;   // K operands in flight
    vec kf[kAhead];
    auto read_k = [&](int n) {  // n = 2 s + kt
      const int r = (n & 1) * 32 + (lane & 31);
      return __builtin_bit_cast(vec, k[r * 16 + (((n & ~1) + half) ^ swz(lane & 15))]);
    };
#pragma unroll
    for (int n = 0; n < kAhead; ++n) kf[n] = read_k(n);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) c[kt][i] = 0.f;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      __builtin_amdgcn_sched_barrier(0);
      c[n & 1] = M::run(kf[n % kAhead], q[n >> 1], c[n & 1]);
      if (n + kAhead < 16) kf[n % kAhead] = read_k(n + kAhead);
    }
    __builtin_amdgcn_s_setprio(0);
  }
  // live(key of the tile, half): whether the lane's query sees it
  template <class LiveFn>
  static __device__ __forceinline__ void mask(f32x16 (&c)[2], LiveFn live) {
    const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) c[kt][i] = live(kt * 32 + 8 * (i >> 2) + (i & 3), half) ? c[kt][i] : -INFINITY;
  }
  // The softmax of a tile's scores c and its value product.  HILO: P enters the
  // product as a hi + lo pair.  k2 = scale * log2(e).  EDGE: keep (wave-uniform)
  // has a bit for each key of the tile; the others' values count as zeros, since
  // a weight of 0 does not take out a value that is not finite.
  template <bool HILO, bool EDGE>
  __device__ __forceinline__ void step(const f32x16 (&c)[2], const Rows& v, float k2, uint64_t keep = ~0ull) {
    using M = Mfma<DT>;
    using vec = typename M::vec;
    const int lane = lane_id(), half = lane >> 5;
    float mx = c[0][0];
#pragma unroll
    for (int i = 1; i < 32; ++i) mx = fmaxf(mx, c[i >> 4][i & 15]);
    mx *= k2;
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float nb = fmaxf(base, mx);
    const float alpha = __builtin_amdgcn_exp2f(base - nb);
    base = nb;
    den *= alpha;
    // V operands: lane 4 j + m of a 16-lane group reads the 8 bytes at columns
    // 4 m .. + 3 (of the group's 16) of row 16 ks + 8 u + 4 half + j
    const int j = (lane & 15) >> 2, m = lane & 3, gi = (lane >> 4) & 1;
    const int low = 2 * gi + (m >> 1);
    auto read_v = [&](int n) {   // n = 4 ks + d
      const int d = n & 3, ks = n >> 2;
      s16x4v x[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int row = 16 * ks + 8 * u + 4 * half + j;
        const int pc = ((4 * d + low) ^ ((j << 2) | (2 * u + half))) & 15;
        x[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4v*)(reinterpret_cast<const uint2*>(&v[row * 16 + pc]) + (m & 1)));
      }
      return __builtin_bit_cast(vec, __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // P of the 16 keys of step ks, a quarter (two scores) at a time: the next
    // step's between this one's MFMAs
    uint32_t ph[2][4], pl[2][4];
    auto quarter = [&](int ks, int e) {
      const float p0 = __builtin_amdgcn_exp2f(fmaf(c[ks >> 1][8 * (ks & 1) + 2 * e], k2, -base));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(c[ks >> 1][8 * (ks & 1) + 2 * e + 1], k2, -base));
      const uint32_t h = M::round2(p0, p1);
      ph[ks & 1][e] = h;
      den += p0 + p1;
      if constexpr (HILO)
        pl[ks & 1][e] =
            M::round2(p0 - M::widen(static_cast<uint16_t>(h)), p1 - M::widen(static_cast<uint16_t>(h >> 16)));
    };
    // word e of a V operand of step ks holds keys 16 ks + 8 (e / 2) + 4 half + 2 (e % 2) and the next
    uint32_t kept[4];
    auto find_kept = [&](int ks) {
      const uint32_t live = static_cast<uint32_t>(keep >> (32 * (ks >> 1))) >> (4 * half);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int bit = 16 * (ks & 1) + 8 * (e >> 1) + 2 * (e & 1);
        const uint32_t even = static_cast<int32_t>(live << (31 - bit)) >> 31;
        const uint32_t odd = static_cast<int32_t>(live << (30 - bit)) >> 31;
        kept[e] = (even & 0xffffu) | (odd & 0xffff0000u);
      }
    };
    constexpr int kAhead = 3;   // V operands in flight
    vec vf[kAhead];
#pragma unroll
    for (int n = 0; n < kAhead; ++n) vf[n] = read_v(n);
#pragma unroll
    for (int e = 0; e < 4; ++e) quarter(0, e);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      __builtin_amdgcn_sched_barrier(0);
      const int d = n & 3, ks = n >> 2;
      const uint32_t* h = ph[ks & 1];
      if (ks == 0) acc[d] *= alpha;
      if constexpr (EDGE) {
        if (d == 0) find_kept(ks);
        const uint4 x = __builtin_bit_cast(uint4, vf[n % kAhead]);
        vf[n % kAhead] =
            __builtin_bit_cast(vec, make_uint4(x.x & kept[0], x.y & kept[1], x.z & kept[2], x.w & kept[3]));
      }
      acc[d] = M::run(vf[n % kAhead], __builtin_bit_cast(vec, make_uint4(h[0], h[1], h[2], h[3])), acc[d]);
      if constexpr (HILO) {
        const uint32_t* l = pl[ks & 1];
        acc[d] = M::run(vf[n % kAhead], __builtin_bit_cast(vec, make_uint4(l[0], l[1], l[2], l[3])), acc[d]);
      }
      if (n + kAhead < 16) vf[n % kAhead] = read_v(n + kAhead);
      if (ks < 3) quarter(ks + 1, d);
    }
    __builtin_amdgcn_s_setprio(0);
  }
  // The wave's 32 rows, normalised and rounded, row-major through its 8 KB of
  // LDS: store(row of the wave, first dim, 8 packed elements) for each 16-byte
  // piece, 16 lanes a row.  After the last tile and a barrier.
  template <class StoreFn>
  __device__ __forceinline__ void store(uint4* lds, StoreFn put) {
    using M = Mfma<DT>;
    const int lane = lane_id(), half = lane >> 5, qn = lane & 31;
    const float inv = 1.f / (den + __shfl_xor(den, 32, 64));
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const uint2 o = make_uint2(M::round2(acc[d][4 * rr] * inv, acc[d][4 * rr + 1] * inv),
                                   M::round2(acc[d][4 * rr + 2] * inv, acc[d][4 * rr + 3] * inv));
        (reinterpret_cast<uint2*>(&lds[qn * 16 + ((4 * d + rr) ^ (qn & 15))]))[half] = o;
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave's writes, read by its other lanes
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int r = it * 4 + (lane >> 4), p = lane & 15;
      put(r, p * 8, lds[r * 16 + (p ^ (r & 15))]);
    }
  }
};

}  // namespace attn
}  // namespace yh
