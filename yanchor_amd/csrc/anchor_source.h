// Where the key / value rows of an anchor-memory prefill are.  Source rows of
// row b: [0, end0) the committed slots, [end0, end1) the old pending slots,
// [end1, S) the new tokens, each part with its own strides, so that nothing is
// assembled first (copying the parts into one tensor took 390 us of 1770 at 32
// rows of 2048 tokens).
#pragma once
#include "common.h"

namespace yh {

struct AnchorSource {
  const char* base[2][3];        // [keys, values][part]
  int64_t row_stride[2][3];      // bytes
  int64_t batch_stride[3];       // bytes, parts 0 and 1
  int64_t group_stride[3];       // bytes
  int end0, end1, S, L;
  // new token i of row b is row (bases ? bases[b] : b * batch_rows) +
  // (order ? order[b * L + i] : i) of the token tensors
  int64_t batch_rows;
  const int64_t* bases;
  const int32_t* order;

  __device__ __forceinline__ int64_t token_row(int64_t b, int i) const {
    return (bases ? bases[b] : b * batch_rows) + (order ? order[b * L + i] : i);
  }
  // start of source row ref (in [0, S)) of group g; which: 0 keys, 1 values
  __device__ __forceinline__ const void* row(int which, int64_t b, int ref, int g) const {
    if (ref < end0) return base[which][0] + b * batch_stride[0] + ref * row_stride[which][0] + g * group_stride[0];
    if (ref < end1)
      return base[which][1] + b * batch_stride[1] + (ref - end0) * row_stride[which][1] + g * group_stride[1];
    return base[which][2] + token_row(b, ref - end1) * row_stride[which][2] + g * group_stride[2];
  }
};

// One tensor [KB, S, G, row]: batch_rows S, or 0 where all rows share one source.
inline AnchorSource assembled_source(const void* key, const void* value, int64_t batch_rows, int64_t S, int64_t G,
                                     int64_t rowbytes) {
  AnchorSource s{};
  s.base[0][0] = static_cast<const char*>(key);
  s.base[1][0] = static_cast<const char*>(value);
  s.row_stride[0][0] = s.row_stride[1][0] = G * rowbytes;
  s.batch_stride[0] = batch_rows * G * rowbytes;
  s.group_stride[0] = rowbytes;
  s.end0 = s.end1 = s.S = static_cast<int>(S);
  s.batch_rows = batch_rows;
  return s;
}

// A state's tensors [B, G, slots, row] and the new tokens [.., G, row] with
// their token strides in bytes.
inline AnchorSource state_source(const void* keys, const void* values, const void* pkeys, const void* pvalues,
                                 const void* key, int64_t key_stride, const void* value, int64_t value_stride,
                                 const int64_t* bases, const int32_t* order, int64_t L, int64_t C, int64_t G,
                                 int64_t capacity, int64_t pending_capacity, int64_t rowbytes) {
  AnchorSource s{};
  const void* b[2][3] = {{keys, pkeys, key}, {values, pvalues, value}};
  for (int x = 0; x < 2; ++x) {
    for (int p = 0; p < 3; ++p) s.base[x][p] = static_cast<const char*>(b[x][p]);
    s.row_stride[x][0] = s.row_stride[x][1] = rowbytes;
    s.row_stride[x][2] = x == 0 ? key_stride : value_stride;
  }
  s.batch_stride[0] = G * capacity * rowbytes;
  s.batch_stride[1] = G * pending_capacity * rowbytes;
  s.group_stride[0] = capacity * rowbytes;
  s.group_stride[1] = pending_capacity * rowbytes;
  s.group_stride[2] = rowbytes;
  s.end0 = static_cast<int>(capacity);
  s.end1 = static_cast<int>(capacity + C);
  s.S = static_cast<int>(capacity + C + L);
  s.L = static_cast<int>(L);
  s.batch_rows = L;
  s.bases = bases;
  s.order = order;
  return s;
}

}  // namespace yh
