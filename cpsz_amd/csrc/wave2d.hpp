// Lorenzo wavefronts of the 2D codec (kernels in wave2d.hip).
#pragma once
#include <cstdint>
#include <vector>

#include "common.hpp"
#include "ctx.hpp"
#include "lorenzo2d_step.hpp"

namespace cpsz {

// A field of fewer than 64 columns and more rows is taken with rows and columns
// exchanged: as one strip instead of many that wait for each other, and in tiles
// that it fills. (The sum that predicts a value is the same with its left and upper
// neighbours exchanged, bit for bit.) Compress / decompress of 62501 x 16: 5.6 /
// 8.7 ms in strips of 64 rows, 3.9 / 3.2 flipped; of 29411 x 34: 3.2 / 4.0 and 2.2 /
// 1.8; from 64 columns on a strip's steps outnumber the lag to the next one.
__host__ __device__ inline bool flipped_2d(size_t r1, size_t r2) { return r2 < 64 && r2 < r1; }

// Where the codec's own per-element arrays (eb codes and stream ids for the
// wavefront, quantization codes, unpredictable values) keep element (i, j):
// tiles of one 64-row strip by one 16-step chunk of its wavefront (row l of
// the strip takes column t - l at step t), row by row, so that a chunk is one
// contiguous 1024-element piece. The elements of a tile outside the field hold
// anything in the arrays the wavefront reads and code 0 in the codes it writes.
// The tiles of a field of fewer than 64 rows (or columns, flipped) have the next
// power of two: at most two slots a value, but for the 63 + 15 steps more than
// columns that each strip has (64 slots a value in a single row or column, and
// 40 in two columns, before: 2^28 values in a row took 275 GB to decompress).
constexpr int kTileSteps = 16;
struct Tile2d {
  uint32_t row_len = 2;   // r2
  uint32_t strips = 0;
  uint32_t nch = 0;       // chunks of a strip
  uint32_t rows_log = 6;  // log2 of a tile's rows
  uint32_t mul = 0, shift = 0;  // division by row_len
  bool flip = false;
  Tile2d() = default;
  Tile2d(size_t r1, size_t r2) {
    row_len = (uint32_t)r2;
    flip = flipped_2d(r1, r2);
    const size_t rows = flip ? r2 : r1, cols = flip ? r1 : r2;
    strips = (uint32_t)((rows + 63) / 64);
    while (rows_log && rows <= (1u << (rows_log - 1))) rows_log--;
    nch = (uint32_t)((cols + (1u << rows_log) - 1 + kTileSteps - 1) / kTileSteps);
    // n / d = (((n - q) >> 1) + q) >> (L - 1) with q = the high word of mul n
    // (Granlund and Montgomery 1994): exact for every 32-bit n, d >= 2
    uint32_t L = 0;
    while ((1ull << L) < row_len) L++;
    if (L) {
      mul = (uint32_t)((((1ull << L) - row_len) << 32) / row_len + 1);
      shift = L - 1;
    }
  }
  // elements of an array
  __host__ __device__ size_t elems() const { return (size_t)strips * nch << (rows_log + 4); }
  // step t of row l of a strip
  __host__ __device__ size_t at_step(uint32_t strip, uint32_t l, uint32_t t) const {
    return (((size_t)strip * nch + t / kTileSteps) << (rows_log + 4)) + (l * kTileSteps + t % kTileSteps);
  }
  __host__ __device__ size_t at(int i, int j) const {
    const uint32_t y = (uint32_t)(flip ? j : i), x = (uint32_t)(flip ? i : j), l = y & 63;
    return at_step(y >> 6, l, x + l);
  }
  // n / row_len
  __host__ __device__ uint32_t rows_in(uint32_t n) const {
    const uint32_t q = (uint32_t)(((uint64_t)mul * n) >> 32);
    return row_len > 1 ? (((n - q) >> 1) + q) >> shift : n;
  }
  // element e of the row-major field
  __host__ __device__ size_t at_linear(uint64_t e) const {
    if (e < (1ull << 32)) {
      const uint32_t n = (uint32_t)e, i = rows_in(n);
      return at((int)i, (int)(n - i * row_len));
    }
    const uint64_t i = e / row_len;
    return at((int)i, (int)(e - i * row_len));
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
  Tile2d t;
  int cs;                // values from one column to the next (set by the launch, which exchanges r1 and r2 of a flipped field)
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
// first one, unless 64 rows span 4 GiB: of cols values in the row-major arrays (a
// flipped field's are among 64 rows of r1), in tiles up to 78 steps a row more.
inline bool far_strip(size_t cols, size_t value_bytes) {
  return div_up(cols + 63, (size_t)kTileSteps) * (64 * kTileSteps) * value_bytes >= (1ull << 32);
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

// 64-bit words of a field's boundary rows (enough for either type); a single
// group publishes none
inline size_t bnd_words(size_t r1, size_t r2) {
  const size_t groups = div_up(r1, (size_t)64 * kStrips64);
  return flipped_2d(r1, r2) || groups == 1 ? 0 : 2 * groups * r2;
}

// The wavefronts of fields f[0..nf) in one launch.
void wavefront2d_compress(Ctx& ctx, std::vector<Strip2d>& f, int grid_cap);
void wavefront2d_decompress(Ctx& ctx, std::vector<Strip2d>& f, int grid_cap);
void wavefront2d_compress64(Ctx& ctx, Strip2d64& f, int grid_cap);
void wavefront2d_decompress64(Ctx& ctx, Strip2d64& f, int grid_cap);

}  // namespace cpsz
