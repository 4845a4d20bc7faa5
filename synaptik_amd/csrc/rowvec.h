// A float row of any start and width as aligned 16-byte groups: group q covers the four floats
// at base + 4 q, base being the row's start rounded down to 16 bytes. The first group holds
// `lead` floats before the row and the last one may run past its end; only a group's floats that
// belong to the row are ever read or written, so every interior access is one aligned 16-byte
// access whatever the row's width, and nothing outside the row is touched.
#pragma once
#include "common.h"

namespace shk {

struct RowGroups {
  int lead;    // floats of group 0 that precede the row
  int groups;  // groups that hold a float of the row
  int width;   // floats of the row
  __device__ __forceinline__ RowGroups(const float* row, int C) {
    lead = (int)((reinterpret_cast<uintptr_t>(row) >> 2) & 3u);
    groups = (lead + C + 3) >> 2;
    width = C;
  }
  // Ordinal in the row of the group's first float (negative inside group 0's lead).
  __device__ __forceinline__ int first(int q) const { return 4 * q - lead; }
  __device__ __forceinline__ bool whole(int q) const {
    return first(q) >= 0 && first(q) + 4 <= width;
  }
  // Group q of the row, or of another tensor's row of the same width; floats outside it read as
  // `fill`. q < groups.
  __device__ __forceinline__ float4 load(const float* row, int q, float fill) const {
    const int c = first(q);
    if (whole(q)) {
      const float4u t = __builtin_nontemporal_load(reinterpret_cast<const float4u*>(row + c));
      return make_float4(t[0], t[1], t[2], t[3]);
    }
    float4 v;
    v.x = c >= 0 && c < width ? row[c] : fill;
    v.y = c + 1 >= 0 && c + 1 < width ? row[c + 1] : fill;
    v.z = c + 2 >= 0 && c + 2 < width ? row[c + 2] : fill;
    v.w = c + 3 < width ? row[c + 3] : fill;
    return v;
  }
  // Whether float j of group q belongs to the row.
  __device__ __forceinline__ bool holds(int q, int j) const {
    return first(q) + j >= 0 && first(q) + j < width;
  }
  // Writes group q likewise. (Another tensor's row need not share the alignment of this one.)
  __device__ __forceinline__ void store(float* row, int q, const float4& v) const {
    const int c = first(q);
    if (whole(q)) {
      __builtin_nontemporal_store(float4u{v.x, v.y, v.z, v.w}, reinterpret_cast<float4u*>(row + c));
      return;
    }
    if (c >= 0 && c < width) row[c] = v.x;
    if (c + 1 >= 0 && c + 1 < width) row[c + 1] = v.y;
    if (c + 2 >= 0 && c + 2 < width) row[c + 2] = v.z;
    if (c + 3 < width) row[c + 3] = v.w;
  }
};

}  // namespace shk
