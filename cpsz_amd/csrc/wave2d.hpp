// Lorenzo wavefronts of the 2D codec (kernels in wave2d.hip).
#pragma once
#include <cstdint>
#include <vector>

#include "common.hpp"
#include "ctx.hpp"
#include "lorenzo2d_step.hpp"

namespace cpsz {

// Where the codec's own per-element arrays (eb codes and stream ids for the
// wavefront, quantization codes, unpredictable values) keep element (i, j):
// tiles of one 64-row strip by one 16-step chunk of its wavefront (row l of
// the strip takes column t - l at step t), row by row, so that a chunk is one
// contiguous 1024-element piece. The elements of a tile outside the field hold
// anything in the arrays the wavefront reads and code 0 in the codes it writes.
// A field of one column is kept as one row (its values precede each other the
// same way).
constexpr int kTileSteps = 16;
struct Tile2d {
  uint32_t row_len = 2;  // r2, or r1 of a one-column field
  uint32_t nch = 0;      // chunks of a strip
  uint32_t mul = 0, shift = 0;  // division by row_len
  bool column = false;
  Tile2d() = default;
  Tile2d(size_t r1, size_t r2) {
    column = r2 == 1;
    row_len = (uint32_t)(column ? r1 : r2);
    nch = (uint32_t)((row_len + 63 + kTileSteps - 1) / kTileSteps);
    // n / d = (((n - q) >> 1) + q) >> (L - 1) with q = the high word of mul n
    // (Granlund and Montgomery 1994): exact for every 32-bit n, d >= 2
    uint32_t L = 0;
    while ((1ull << L) < row_len) L++;
    if (L) {
      mul = (uint32_t)((((1ull << L) - row_len) << 32) / row_len + 1);
      shift = L - 1;
    }
  }
  __host__ __device__ size_t strips(size_t r1) const { return column ? 1 : (r1 + 63) / 64; }
  __host__ __device__ size_t elems(size_t r1) const { return strips(r1) * nch * (64 * kTileSteps); }
  __host__ __device__ size_t at(int i, int j) const {
    if (column) {
      j = i;
      i = 0;
    }
    const uint32_t l = (uint32_t)i & 63, t = (uint32_t)j + l;
    return ((size_t)((uint32_t)i >> 6) * nch + t / kTileSteps) * (64 * kTileSteps) + l * kTileSteps + t % kTileSteps;
  }
  // n / row_len
  __host__ __device__ uint32_t rows_in(uint32_t n) const {
    const uint32_t q = (uint32_t)(((uint64_t)mul * n) >> 32);
    return row_len > 1 ? (((n - q) >> 1) + q) >> shift : n;
  }
  // element e of the row-major field
  __host__ __device__ size_t at_linear(uint64_t e) const {
    uint32_t i, j;
    if (e < (1ull << 32)) {
      const uint32_t n = (uint32_t)e;
      i = rows_in(n);
      j = n - i * row_len;
    } else {
      i = (uint32_t)(e / row_len);
      j = (uint32_t)(e - (uint64_t)i * row_len);
    }
    const uint32_t l = i & 63, t = j + l;
    return ((size_t)(i >> 6) * nch + t / kTileSteps) * (64 * kTileSteps) + l * kTileSteps + t % kTileSteps;
  }
};

// 64-row strips that one workgroup carries (double fields: half as many,
// their staged elements are twice as wide)
constexpr int kStrips = 4, kStrips64 = 2;

// One field's wavefront. T: the field's value type.
template <typename T>
struct Strip2dT {
  const T* x[2];         // compress: the values, row-major
  const uint16_t* c[2];  // compress: eb codes; decompress: stream ids (tiles, as q and raw)
  uint16_t* q[2];        // quant codes (written by compress, read by decompress)
  const T* raw[2];       // decompress: unpredictable value per element
  T* out[2];             // decompress output, row-major
  uint64_t* bnd;         // [2][ngroups][r2] last row of every strip group, published value by value
  int* ticket;           // the item ticket of a single field's launch
  int r1, r2, ngroups;
  int wide;              // float fields with ids above 81: double-precision step
  int shift;             // log2 of the eb base: 2 (offline, 4^id eps) or 1 (offline_log, 2^id eps)
  // compress of a batch: the eb pass's flags, read in place of `wide`
  // ([1]); a field with [0] set (non-finite input) is skipped as a whole
  const int* flags;
};
using Strip2d = Strip2dT<float>;
using Strip2d64 = Strip2dT<double>;

template <typename T>
inline int strip_groups(size_t r1) {
  return (int)div_up(r1, (size_t)64 * (sizeof(T) == 8 ? kStrips64 : kStrips));
}
// The wavefront addresses a strip's elements by 32-bit byte offsets from its
// first one, unless the strip spans 4 GiB: row-major it takes 64 rows of r2
// values, in tiles up to 78 steps a row more.
inline bool far_strip(size_t r2, size_t value_bytes) {
  return div_up(r2 + 63, (size_t)kTileSteps) * (64 * kTileSteps) * value_bytes >= (1ull << 32);
}
// A word of a field's boundary rows: a float with a tag, or a double in place of
// a NaN pattern (kBndEmpty). A corrupt stream's unpredictable values can hold
// any pattern: that one is published as the NaN next to it, or the reader would
// wait for it without end (the output keeps its own; what is predicted from
// either is a NaN).
constexpr uint64_t kBndTag = 1ull << 32;
constexpr uint64_t kBndEmpty = 0x7FF4DEADBEEF0000ull;
__host__ __device__ inline bool bnd_ready(uint64_t v, float) { return (v >> 32) != 0; }
__host__ __device__ inline bool bnd_ready(uint64_t v, double) { return v != kBndEmpty; }
__host__ __device__ inline uint64_t bnd_word(float x) { return kBndTag | l2d_bits(x); }
__host__ __device__ inline uint64_t bnd_word(double x) {
  const uint64_t b = l2d_bits(x);
  return b == kBndEmpty ? b + 1 : b;
}
__host__ __device__ inline float bnd_value(uint64_t v, float) { return l2d_float((uint32_t)v); }
__host__ __device__ inline double bnd_value(uint64_t v, double) { return l2d_double(v); }

// 64-bit words of a field's boundary rows (enough for either type)
inline size_t bnd_words(size_t r1, size_t r2) { return 2 * div_up(r1, (size_t)64 * kStrips64) * r2; }

// The wavefronts of fields f[0..nf) in one launch.
void wavefront2d_compress(Ctx& ctx, std::vector<Strip2d>& f, int grid_cap);
void wavefront2d_decompress(Ctx& ctx, std::vector<Strip2d>& f, int grid_cap);
void wavefront2d_compress64(Ctx& ctx, Strip2d64& f, int grid_cap);
void wavefront2d_decompress64(Ctx& ctx, Strip2d64& f, int grid_cap);

}  // namespace cpsz
