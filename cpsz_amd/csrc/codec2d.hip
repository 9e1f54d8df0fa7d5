// 2D critical-point-preserving codec on gfx950 (the drop-in for
// sz_compress_cp_preserve_2d_offline / sz_decompress_cp_preserve_2d_offline).
//
// Device pipeline (compress), all inputs resident in HBM:
//   k_eb2d*       per-cell triangle bounds in LDS (16x32 vertex tiles + 1-cell
//                 halo), ordered per-vertex min, |U|,|V| scaling and the base-4
//                 eb id -> eb code per vertex and component (row-major for the id
//                 encoder, in tiles for the wavefront), id histogram
//   k_wave2d      strip-pipelined wavefront Lorenzo + linear quantization (wave2d.hip)
//   Huffman       histogram -> tree on the host or, in batches, the device
//                 (reference tie-break) -> encode, with the unpredictable
//                 values compacted in 12x12 block-major order
// Decompress mirrors it: parallel Huffman decode of ids and codes, block-major
// unpredictable scatter, wavefront reconstruction.
//
// Bit-exactness: every float/double operation follows the reference's types
// and order (src/sz_compress_cp_preserve_2d.cpp:17-172, quantize in
// include/sz_compression_utils.hpp:50-65); the Lorenzo step runs in FP32, which
// reproduces the reference's double arithmetic exactly (the argument is in the
// comments of lorenzo2d_step.hpp).
#include <algorithm>
#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "codec2d.hpp"
#include "pool.hpp"
#include "stream_reader.hpp"
#include "huff_gpu.hpp"
#include "libm_math.hpp"
#include "lorenzo2d_step.hpp"
#include "bounds2d_fast.hpp"
#include "wave2d.hpp"

namespace cpsz {

// ----------------------------------------------------------------- eb bound --
namespace {

__device__ __forceinline__ double dminf(double a, double b) { return (a < b) ? a : b; }
__device__ __forceinline__ double dmaxm(double a, double b) { return (a > b) ? a : b; }

template <typename V>
__device__ __forceinline__ void dacc(V v, double& p, double& n) {
  if (v >= 0) p += v;
  else n += -v;
}

// max_eb_to_keep_sign (include/sz_cp_preserve_utils.hpp:59-90), degrees 1, 2
__device__ __forceinline__ double dsign_bound(double p, double n, int deg) {
  if (n == 0 || p == 0) return 1;
  double P = p, N = n;
  if (deg == 2) {
    P = sqrt(p);
    N = sqrt(n);
  }
  return fabs(P - N) / (P + N);
}

__device__ __forceinline__ double dbound2(double a, double b) {
  double p = 0, n = 0;
  dacc(a, p, n);
  dacc(b, p, n);
  return dsign_bound(p, n, 2);
}
__device__ __forceinline__ double dbound4(double a, double b, double c, double d) {
  double p = 0, n = 0;
  dacc(a, p, n);
  dacc(b, p, n);
  dacc(c, p, n);
  dacc(d, p, n);
  return dsign_bound(p, n, 2);
}

// max_eb_to_keep_sign_eigen_delta_2 (:75-123); rarely taken (CP triangles).
// T is the field's value type: the reference computes c[], m, C and the
// coefficients in T.
template <typename T>
__device__ __noinline__ double deigen(T u0, T u1, T u2, T v0, T v1, T v2, T x0, T x1, T x2, T y0, T y1, T y2) {
  double eb = 1;
  T c[4];
  {
    const T det = (x0 - x2) * (y1 - y2) - (x1 - x2) * (y0 - y2);
    c[0] = (y1 - y2) / det;
    c[1] = -(y0 - y2) / det;
    c[2] = -(x1 - x2) / det;
    c[3] = (x0 - x2) / det;
    double p = 0, n = 0;
    dacc(c[0] * u0, p, n);
    dacc(c[1] * u1, p, n);
    dacc(-(c[0] + c[1]) * u2, p, n);
    dacc(c[2] * v0, p, n);
    dacc(c[3] * v1, p, n);
    dacc(-(c[2] + c[3]) * v2, p, n);
    eb = dsign_bound(p, n, 1);
    double p2 = 0, n2 = 0;
    dacc(u0 * v1, p2, n2);
    dacc(-u0 * v2, p2, n2);
    dacc(u1 * v2, p2, n2);
    dacc(-u1 * v0, p2, n2);
    dacc(u2 * v0, p2, n2);
    dacc(-u2 * v1, p2, n2);
    eb = dminf(eb, dsign_bound(p2, n2, 2));
  }
  const T m = c[1] * c[2] - c[0] * c[3];
  const T C = (-m) * (u0 * v1 - u0 * v2 + u1 * v2 - u1 * v0 + u2 * v0 - u2 * v1);
  if (C == 0) return 0;
  if (C < 0) return eb;
  const T co[6] = {c[0] * u0, c[1] * u1, -(c[1] + c[0]) * u2, c[2] * v0, c[3] * v1, -(c[3] + c[2]) * v2};
  double p = 0, n = 0;
  for (int i = 0; i < 6; i++)
    for (int j = 0; j < 6; j++) dacc(co[i] * co[j], p, n);
  dacc(-4 * m * u1 * v0, p, n);
  dacc(4 * m * u2 * v0, p, n);
  dacc(4 * m * u0 * v1, p, n);
  dacc(-4 * m * u2 * v1, p, n);
  dacc(-4 * m * u0 * v2, p, n);
  dacc(4 * m * u1 * v2, p, n);
  return dminf(eb, dsign_bound(p, n, 2));
}

// max_eb_to_keep_position_and_type (src/sz_compress_cp_preserve_2d.cpp:125-172)
// for the two triangle shapes of a cell (coordinates passed "reversed", :187-206).
template <typename T>
__device__ double dtri(T u0, T u1, T u2, T v0, T v1, T v2, int lower) {
  const double u0v1 = u0 * v1, u1v0 = u1 * v0, u0v2 = u0 * v2, u2v0 = u2 * v0, u1v2 = u1 * v2,
               u2v1 = u2 * v1;
  const double det = u0v1 - u1v0 + u1v2 - u2v1 + u2v0 - u0v2;
  if (!(det != 0)) return 0;
  const bool f1 = (det / (u2v0 - u0v2) >= 1);
  const bool f2 = (det / (u1v2 - u2v1) >= 1);
  const bool f3 = (det / (u0v1 - u1v0) >= 1);
  if (f1 && f2 && f3) {
    const double e1 = dminf(dbound2(u2v0, -u0v2), dbound4(u0v1, -u1v0, u1v2, -u2v1));
    const double e2 = dminf(dbound2(u1v2, -u2v1), dbound4(u0v1, -u1v0, u2v0, -u0v2));
    const double e3 = dminf(dbound2(u0v1, -u1v0), dbound4(u1v2, -u2v1, u2v0, -u0v2));
    // X_upper = {{0,0},{1,0},{1,1}}, X_lower = {{0,0},{0,1},{1,1}}; x = X[.][1], y = X[.][0]
    const T o = 0, l = 1;
    const double e4 = lower ? dminf(e3, deigen<T>(u0, u1, u2, v0, v1, v2, o, l, l, o, o, l))
                            : dminf(e3, deigen<T>(u0, u1, u2, v0, v1, v2, o, o, l, o, l, l));
    double eb = dminf(e1, e2);
    return dminf(eb, e4);
  }
  double eb = 0;
  if (!f1) eb = dmaxm(eb, dminf(dbound2(u2v0, -u0v2), dbound4(u0v1, -u1v0, u1v2, -u2v1)));
  if (!f2) eb = dmaxm(eb, dminf(dbound2(u1v2, -u2v1), dbound4(u0v1, -u1v0, u2v0, -u0v2)));
  if (!f3) eb = dmaxm(eb, dminf(dbound2(u0v1, -u1v0), dbound4(u1v2, -u2v1, u2v0, -u0v2)));
  return eb;
}

// The FP32-approximated triangle bound (tri_fast) and its constants are in
// bounds2d_fast.hpp, shared with the host check.
struct DeviceRoots {
  __device__ static float sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
  __device__ static float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
};

// eb code: 0 = zero precision; c >= 1: reference id c-1 with precision
// 4^(c-1) * DBL_EPSILON (id 0 keeps precision eps in the compressor).
__device__ __forceinline__ uint32_t eb_code_2d(double x, const double* __restrict__ q2d, int nq) {
  if (!(x > 2.220446049250313080847263336181640625e-16)) return 0;
  const int e = (int)((__double_as_longlong(x) >> 52) & 0x7FF) - 1023 + 52;  // exponent of x/eps
  int k = e >> 1;
  if (k + 1 < nq && x >= q2d[k + 1]) k++;
  return (uint32_t)k + 1;
}

// Eb code from a threshold table q[1..nq-2] (q[nq-1] = +inf): the largest k
// with x >= q[k], 0 below q[1].
__device__ __forceinline__ uint32_t code_from_table(double x, const double* __restrict__ q, int nq) {
  if (!(x >= q[1])) return 0;
  int lo = 1, hi = nq - 2;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (x >= q[mid]) lo = mid;
    else hi = mid - 1;
  }
  return (uint32_t)lo;
}

// The eb codes once more, where the wavefront reads them (the id encoder reads
// them in row-major order).
struct CodeTiles {
  uint16_t* u;
  uint16_t* v;
  Tile2d t;
};

constexpr int kTH = 16, kTW = 32;  // vertex tile (17x33 cells: 9 wave rounds of triangles per 512 vertices)

template <typename T>
__device__ __forceinline__ void eb2d_tile(const T* __restrict__ U, const T* __restrict__ V, int r1, int r2,
                                          double max_pwr_eb, const double* __restrict__ q2d, int nq,
                                          uint16_t* __restrict__ cu, uint16_t* __restrict__ cv,
                                          uint32_t* __restrict__ hist, int* __restrict__ flags, const EbOverride& ov,
                                          const double* __restrict__ qlog, int nqlog, const CodeTiles& ct, int bx,
                                          int by) {
  __shared__ T su[kTH + 2][kTW + 2];
  __shared__ T sv[kTH + 2][kTW + 2];
  __shared__ double tb[kTH + 1][kTW + 1][2];
  __shared__ uint32_t sh_hist[kMaxEbCode];
  const int tid = threadIdx.x;
  const int i0 = by * kTH, j0 = bx * kTW;
  for (int k = tid; k < kMaxEbCode; k += 256) sh_hist[k] = 0;
  for (int k = tid; k < (kTH + 2) * (kTW + 2); k += 256) {
    const int r = k / (kTW + 2), c = k % (kTW + 2);
    const int gi = i0 - 1 + r, gj = j0 - 1 + c;
    T a = 0, b = 0;
    if (gi >= 0 && gi < r1 && gj >= 0 && gj < r2) {
      a = U[(size_t)gi * r2 + gj];
      b = V[(size_t)gi * r2 + gj];
    }
    su[r][c] = a;
    sv[r][c] = b;
  }
  __syncthreads();
  for (int k = tid; k < (kTH + 1) * (kTW + 1); k += 256) {
    const int cr = k / (kTW + 1), cc = k % (kTW + 1);
    const int ci = i0 - 1 + cr, cj = j0 - 1 + cc;
    double up = INFINITY, lo = INFINITY;
    if (ci >= 0 && ci < r1 - 1 && cj >= 0 && cj < r2 - 1) {
      // upper: (i,j),(i+1,j),(i+1,j+1); lower: (i,j),(i,j+1),(i+1,j+1)
      up = dtri<T>(su[cr][cc], su[cr + 1][cc], su[cr + 1][cc + 1], sv[cr][cc], sv[cr + 1][cc],
                   sv[cr + 1][cc + 1], 0);
      lo = dtri<T>(su[cr][cc], su[cr][cc + 1], su[cr + 1][cc + 1], sv[cr][cc], sv[cr][cc + 1],
                   sv[cr + 1][cc + 1], 1);
    }
    tb[cr][cc][0] = up;
    tb[cr][cc][1] = lo;
  }
  __syncthreads();
  int bad = 0;
  for (int k = tid; k < kTH * kTW; k += 256) {
    const int vr = k / kTW, vc = k % kTW;
    const int i = i0 + vr, j = j0 + vc;
    if (i >= r1 || j >= r2) continue;
    const T u = su[vr + 1][vc + 1], v = sv[vr + 1][vc + 1];
    // incident triangles in the reference's visiting order (cells row-major, upper first)
    double eb = max_pwr_eb;
    eb = dminf(eb, tb[vr][vc][0]);
    eb = dminf(eb, tb[vr][vc][1]);
    eb = dminf(eb, tb[vr][vc + 1][0]);
    eb = dminf(eb, tb[vr + 1][vc][1]);
    eb = dminf(eb, tb[vr + 1][vc + 1][0]);
    eb = dminf(eb, tb[vr + 1][vc + 1][1]);
    const size_t vix = (size_t)i * r2 + j;
    if (ov.eb_out) ov.eb_out[vix] = eb;
    if (ov.gain && !(ov.fallback && ov.fallback[vix]) && ov.gain[vix])
      eb = dminf(max_pwr_eb, ldexp(eb, (int)ov.gain[vix]));
    if (ov.fallback && ov.fallback[vix] == 2) eb = 0;  // stored exactly
    if (!isfinite(u) || !isfinite(v) || !(eb == eb)) bad = 1;
    if (qlog) {
      // offline_log: one code per vertex for both components, from the bound
      // itself (src/sz_compress_cp_preserve_2d.cpp:327-331)
      const uint32_t a = code_from_table(eb, qlog, nqlog);
      cu[(size_t)i * r2 + j] = (uint16_t)a;
      ct.u[ct.t.at(i, j)] = (uint16_t)a;
      atomicAdd(&sh_hist[a ? a - 1 : 0], 1u);
      continue;
    }
    // the reference's eb/DBL_EPSILON overflows from 2^972 on (undefined id)
    // eb_u = fabs(U[i]) * eb[i] (src/sz_compress_cp_preserve_2d.cpp:231)
    const double au = (double)fabs(u) * eb, av = (double)fabs(v) * eb;
    if (au >= 0x1p972 || av >= 0x1p972) bad = 1;
    const uint32_t a = eb_code_2d(au, q2d, nq);
    const uint32_t b = eb_code_2d(av, q2d, nq);
    cu[(size_t)i * r2 + j] = (uint16_t)a;
    cv[(size_t)i * r2 + j] = (uint16_t)b;
    const size_t te = ct.t.at(i, j);
    ct.u[te] = (uint16_t)a;
    ct.v[te] = (uint16_t)b;
    atomicAdd(&sh_hist[a ? a - 1 : 0], 1u);
    atomicAdd(&sh_hist[b ? b - 1 : 0], 1u);
    if (a > 82 || b > 82) atomicOr(&flags[1], 1);  // beyond the FP32 Lorenzo path
  }
  if (bad) atomicOr(&flags[0], 1);
  __syncthreads();
  for (int k = tid; k < kMaxEbCode; k += 256)
    if (sh_hist[k]) atomicAdd(&hist[k], sh_hist[k]);
}

// code(x) >= c for the eb code function above (c = code(y) for some y >= x):
// the codes step at eps and at the thresholds q2d[1..]
__device__ __forceinline__ bool code_reaches(uint32_t c, double x, const double* __restrict__ q2d) {
  if (c == 0) return true;
  if (c == 1) return x > 2.220446049250313080847263336181640625e-16;
  return x >= q2d[c - 1];
}

// Marks, in cu, a vertex whose bound the fix-up pass computes in FP64 (eb
// codes stay far below).
constexpr uint16_t kFixCode = 0xFFFF;

// Every field of a batch in one launch (float fields): a job per field, its
// tiles numbered from blk0 row by row.
struct Eb2dJob {
  const float* U;
  const float* V;
  int r1, r2, gx;  // gx: tiles per tile row
  uint16_t* cu;
  uint16_t* cv;
  uint32_t* hist;
  int* flags;
  EbOverride ov;
  CodeTiles ct;
  uint32_t blk0;
};

__device__ __forceinline__ const Eb2dJob& eb_job_of(const Eb2dJob* __restrict__ jobs, int nj, uint32_t tile) {
  int lo = 0, hi = nj - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].blk0 <= tile) lo = mid;
    else hi = mid - 1;
  }
  return jobs[lo];
}

// eb2d_tile for float fields without overrides or log bounds: the cell table
// holds tri_fast entries and each vertex takes its eb codes from the
// enclosure of its bound. Vertices that need the FP64 bound get kFixCode, and
// the tile goes on the fix-up list (fix_tiles, counted by fix_n) for
// k_eb2d_fix, which also counts them in the histogram.
__device__ __forceinline__ void eb2d_tile_fast(const float* __restrict__ U, const float* __restrict__ V, int r1,
                                               int r2, double max_pwr_eb, const double* __restrict__ q2d, int nq,
                                               uint16_t* __restrict__ cu, uint16_t* __restrict__ cv,
                                               uint32_t* __restrict__ hist, int* __restrict__ flags,
                                               const CodeTiles& ct, int bx, int by, uint32_t tile, uint32_t* __restrict__ fix_tiles,
                                               uint32_t* __restrict__ fix_n) {
  __shared__ float su[kTH + 2][kTW + 2];
  __shared__ float sv[kTH + 2][kTW + 2];
  __shared__ float tb[kTH + 1][kTW + 1][2];
  __shared__ uint32_t sh_hist[kMaxEbCode];
  __shared__ int sh_fix;
  const int tid = threadIdx.x;
  const int i0 = by * kTH, j0 = bx * kTW;
  for (int k = tid; k < kMaxEbCode; k += 256) sh_hist[k] = 0;
  if (tid == 0) sh_fix = 0;
  int in_range = 1;
  for (int k = tid; k < (kTH + 2) * (kTW + 2); k += 256) {
    const int r = k / (kTW + 2), c = k % (kTW + 2);
    const int gi = i0 - 1 + r, gj = j0 - 1 + c;
    float a = 0, b = 0;
    if (gi >= 0 && gi < r1 && gj >= 0 && gj < r2) {
      a = U[(size_t)gi * r2 + gj];
      b = V[(size_t)gi * r2 + gj];
    }
    su[r][c] = a;
    sv[r][c] = b;
    in_range &= (int)(value_ok(a) && value_ok(b));
  }
  const bool checked = __syncthreads_and(in_range) != 0;
  // one triangle per item: upper (i,j),(i+1,j),(i+1,j+1); lower (i,j),(i,j+1),(i+1,j+1)
  for (int k = tid; k < 2 * (kTH + 1) * (kTW + 1); k += 256) {
    const int cell = k >> 1, lower = k & 1;
    const int cr = cell / (kTW + 1), cc = cell % (kTW + 1);
    const int ci = i0 - 1 + cr, cj = j0 - 1 + cc;
    float t = INFINITY;
    if (ci >= 0 && ci < r1 - 1 && cj >= 0 && cj < r2 - 1) {
      const int mr = lower ? cr : cr + 1, mc = lower ? cc + 1 : cc;
      t = tri_fast<DeviceRoots>(su[cr][cc], su[mr][mc], su[cr + 1][cc + 1], sv[cr][cc], sv[mr][mc], sv[cr + 1][cc + 1],
                                   checked);
    }
    tb[cr][cc][lower] = t;
  }
  __syncthreads();
  int bad = 0, fix = 0;
  for (int k = tid; k < kTH * kTW; k += 256) {
    const int vr = k / kTW, vc = k % kTW;
    const int i = i0 + vr, j = j0 + vc;
    if (i >= r1 || j >= r2) continue;
    const float u = su[vr + 1][vc + 1], v = sv[vr + 1][vc + 1];
    // the six incident triangles (for the reference, in the order cells
    // row-major, upper first; the order matters only through NaN bounds,
    // which go to the fix-up pass)
    const float m = fminf(fminf(fminf(tb[vr][vc][0], tb[vr][vc][1]), fminf(tb[vr][vc + 1][0], tb[vr + 1][vc][1])),
                          fminf(tb[vr + 1][vc + 1][0], tb[vr + 1][vc + 1][1]));
    uint32_t a, b;
    if (m > 0 && m < kExact1) {
      // the smallest bound is an approximation: exact 1s and missing cells do not matter
      const double am = m;
      const double lo = dminf(max_pwr_eb, enclosure_lo(am));
      const double hi = dminf(max_pwr_eb, enclosure_hi(am));
      const double uh = (double)fabsf(u) * hi, vh = (double)fabsf(v) * hi;
      a = eb_code_2d(uh, q2d, nq);
      b = eb_code_2d(vh, q2d, nq);
      if (!(uh < 0x1p972 && vh < 0x1p972 && code_reaches(a, (double)fabsf(u) * lo, q2d) &&
            code_reaches(b, (double)fabsf(v) * lo, q2d))) {
        cu[(size_t)i * r2 + j] = kFixCode;
        fix = 1;
        continue;
      }
    } else if (m >= 0) {
      // exact: 0, 1 or no triangle
      const double eb = m == 0 ? 0.0 : (m == kExact1 ? dminf(max_pwr_eb, 1.0) : max_pwr_eb);
      // eb_u = fabs(U[i]) * eb[i] (src/sz_compress_cp_preserve_2d.cpp:231); the
      // reference's eb/DBL_EPSILON overflows from 2^972 on (undefined id)
      const double au = (double)fabsf(u) * eb, av = (double)fabsf(v) * eb;
      if (au >= 0x1p972 || av >= 0x1p972 || !isfinite(u) || !isfinite(v)) bad = 1;
      a = eb_code_2d(au, q2d, nq);
      b = eb_code_2d(av, q2d, nq);
    } else {
      cu[(size_t)i * r2 + j] = kFixCode;
      fix = 1;
      continue;
    }
    cu[(size_t)i * r2 + j] = (uint16_t)a;
    cv[(size_t)i * r2 + j] = (uint16_t)b;
    const size_t te = ct.t.at(i, j);
    ct.u[te] = (uint16_t)a;
    ct.v[te] = (uint16_t)b;
    atomicAdd(&sh_hist[a ? a - 1 : 0], 1u);
    atomicAdd(&sh_hist[b ? b - 1 : 0], 1u);
    if (a > 82 || b > 82) atomicOr(&flags[1], 1);  // beyond the FP32 Lorenzo path
  }
  if (bad) atomicOr(&flags[0], 1);
  if (fix) sh_fix = 1;
  __syncthreads();
  for (int k = tid; k < kMaxEbCode; k += 256)
    if (sh_hist[k]) atomicAdd(&hist[k], sh_hist[k]);
  if (tid == 0 && sh_fix) fix_tiles[atomicAdd(fix_n, 1u)] = tile;
}

// The FP64 bounds of the vertices eb2d_tile_fast marked, tile by tile from the
// fix-up list: the six incident triangles in the reference's order, from
// global memory (missing cells contribute +inf, as in eb2d_tile).
__global__ void __launch_bounds__(256) k_eb2d_fix(const Eb2dJob* __restrict__ jobs, int nj,
                                                  const uint32_t* __restrict__ fix_tiles,
                                                  const uint32_t* __restrict__ fix_n, double max_pwr_eb,
                                                  const double* __restrict__ q2d, int nq) {
  const uint32_t n = *fix_n;
  for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
    const uint32_t tile = fix_tiles[e];
    const Eb2dJob& J = eb_job_of(jobs, nj, tile);
    const uint32_t t = tile - J.blk0;
    const int i0 = (int)(t / (uint32_t)J.gx) * kTH, j0 = (int)(t % (uint32_t)J.gx) * kTW;
    const int r1 = J.r1, r2 = J.r2;
    int bad = 0;
    for (int k = threadIdx.x; k < kTH * kTW; k += blockDim.x) {
      const int i = i0 + k / kTW, j = j0 + k % kTW;
      if (i >= r1 || j >= r2) continue;
      const size_t vix = (size_t)i * r2 + j;
      if (J.cu[vix] != kFixCode) continue;
      auto tri = [&](int ci, int cj, int lower) -> double {
        if (ci < 0 || ci >= r1 - 1 || cj < 0 || cj >= r2 - 1) return INFINITY;
        const size_t c0 = (size_t)ci * r2 + cj, c2 = c0 + r2 + 1, c1 = lower ? c0 + 1 : c0 + r2;
        return dtri<float>(J.U[c0], J.U[c1], J.U[c2], J.V[c0], J.V[c1], J.V[c2], lower);
      };
      double eb = max_pwr_eb;
      eb = dminf(eb, tri(i - 1, j - 1, 0));
      eb = dminf(eb, tri(i - 1, j - 1, 1));
      eb = dminf(eb, tri(i - 1, j, 0));
      eb = dminf(eb, tri(i, j - 1, 1));
      eb = dminf(eb, tri(i, j, 0));
      eb = dminf(eb, tri(i, j, 1));
      const float u = J.U[vix], v = J.V[vix];
      const double au = (double)fabsf(u) * eb, av = (double)fabsf(v) * eb;
      if (au >= 0x1p972 || av >= 0x1p972 || !(eb == eb) || !isfinite(u) || !isfinite(v)) bad = 1;
      const uint32_t a = eb_code_2d(au, q2d, nq), b = eb_code_2d(av, q2d, nq);
      J.cu[vix] = (uint16_t)a;
      J.cv[vix] = (uint16_t)b;
      const size_t te = J.ct.t.at(i, j);
      J.ct.u[te] = (uint16_t)a;
      J.ct.v[te] = (uint16_t)b;
      atomicAdd(&J.hist[a ? a - 1 : 0], 1u);
      atomicAdd(&J.hist[b ? b - 1 : 0], 1u);
      if (a > 82 || b > 82) atomicOr(&J.flags[1], 1);
    }
    if (bad) atomicOr(&J.flags[0], 1);
  }
}

template <typename T>
__global__ void __launch_bounds__(256) k_eb2d(const T* __restrict__ U, const T* __restrict__ V,
                                              int r1, int r2, double max_pwr_eb,
                                              const double* __restrict__ q2d, int nq,
                                              uint16_t* __restrict__ cu, uint16_t* __restrict__ cv,
                                              uint32_t* __restrict__ hist, int* __restrict__ flags,
                                              EbOverride ov, const double* __restrict__ qlog, int nqlog,
                                              CodeTiles ct) {
  eb2d_tile<T>(U, V, r1, r2, max_pwr_eb, q2d, nq, cu, cv, hist, flags, ov, qlog, nqlog, ct, blockIdx.x, blockIdx.y);
}

// APPROX: eb2d_tile_fast (jobs without overrides), with its fix-up list
template <bool APPROX>
__global__ void __launch_bounds__(256) k_eb2d_multi(const Eb2dJob* __restrict__ jobs, int nj, double max_pwr_eb,
                                                    const double* __restrict__ q2d, int nq,
                                                    uint32_t* __restrict__ fix_tiles, uint32_t* __restrict__ fix_n) {
  const Eb2dJob& J = eb_job_of(jobs, nj, blockIdx.x);
  const uint32_t t = blockIdx.x - J.blk0;
  const int bx = (int)(t % (uint32_t)J.gx), by = (int)(t / (uint32_t)J.gx);
  if constexpr (APPROX)
    eb2d_tile_fast(J.U, J.V, J.r1, J.r2, max_pwr_eb, q2d, nq, J.cu, J.cv, J.hist, J.flags, J.ct, bx, by,
                   blockIdx.x, fix_tiles, fix_n);
  else
    eb2d_tile<float>(J.U, J.V, J.r1, J.r2, max_pwr_eb, q2d, nq, J.cu, J.cv, J.hist, J.flags, J.ov, nullptr, 0,
                     J.ct, bx, by);
}

__global__ void k_zero_i32(int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ------------------------------------------------------- huffman sources ----
// The ids: the u codes then the v codes (offline), or the one code per vertex
// of offline_log.
struct SrcIds2d {
  const uint16_t* cu;  // 256-byte aligned, and padded to that
  const uint16_t* cv;
  size_t n, per;       // chunks of one component
  // 16 ids a lane, two 16-byte loads: each component starts a chunk of its own,
  // so that these are aligned whatever its length
  static constexpr int kRun = 16, kLds = 8, kChunk = 64 * kRun;
  SrcIds2d(const uint16_t* u, const uint16_t* v, size_t n_) : cu(u), cv(v), n(n_), per((n_ + kChunk - 1) / kChunk) {}
  size_t chunks(bool both) const { return both ? 2 * per : per; }
  __device__ void stage(size_t, uint16_t*) const {}
  __device__ int load(size_t c, const uint16_t*, uint32_t* sym) const {
    const bool v = c >= per;
    const size_t p = (v ? c - per : c) * kChunk + kRun * (threadIdx.x & 63);
    const auto s = glob(reinterpret_cast<const u32x4*>((v ? cv : cu) + min(p, (n - 1) & ~(size_t)(kRun - 1))));
    const u32x4 a = s[0], b = s[1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < kRun; k++) {
      const uint32_t x = k & 1 ? w[k / 2] >> 16 : w[k / 2] & 0xFFFFu;
      sym[k] = x ? min(x, (uint32_t)kMaxEbCode) - 1 : 0;  // (the padding may hold anything)
    }
    return (int)max((long long)0, min((long long)kRun, (long long)n - (long long)p));
  }
};

// The codes of 8 consecutive 12x12 blocks of a block row. Their 12 row pieces
// lie in the tiles as runs of 16 codes: the wave copies them to LDS by 16-byte
// loads (3 a lane) and reads 18 codes a lane from there, in the blocks' order.
// Row ii of the chunk lands one code later than row ii - 1 (the tiles are
// skewed by a step a row), so row ii, column j is at first + ii (kPitch + 1) + j.
// A flipped field's columns lie in the tiles as runs: a chunk, the whole of a block
// row, takes the 24 codes from a multiple of 8 on that hold 12 rows of each.
template <typename T>
struct SrcCodes2dT {
  const uint16_t* q;  // tiles
  Tile2d t;
  int r1, r2, nby, per;  // per: chunks of a block row
  // optional: the values the codec ran on, the exclusive scan of the chunks'
  // zero counts at this component's first chunk, and where the encoder
  // gathers the unpredictable values
  const T* x = nullptr;
  const uint64_t* uoff = nullptr;
  T* unp = nullptr;
  static constexpr bool kUnpred = true;
  bool flip;
  static constexpr int kBlocks = 8, kRun = 18, kPitch = 128, kSegs = 15, kLds = kBlock2d * kPitch;
  static constexpr int kFlipPitch = 24, kFlipSegs = 3;
  static_assert(kBlocks * kBlock2d * kBlock2d == 64 * kRun && kSegs * 8 >= 7 + kBlock2d - 1 + kBlocks * kBlock2d);
  static_assert(kFlipPitch >= 7 + kBlock2d && 64 * kFlipPitch <= kLds && 63 * kFlipSegs <= 3 * 64 && kBlocks * kBlock2d >= 63);
  // a one-column field is laid out, and has its codes in the order of, a one-row field
  SrcCodes2dT(const uint16_t* q_, const Tile2d& t_, size_t r1_, size_t r2_, const T* x_ = nullptr)
      : q(q_), t(t_), r1((int)(r2_ == 1 ? 1 : r1_)), r2((int)(r2_ == 1 ? r1_ : r2_)),
        nby((int)div_up((size_t)r2, (size_t)kBlock2d)), per((int)div_up((size_t)nby, (size_t)kBlocks)), x(x_),
        flip(t_.flip && r2_ > 1) {}
  size_t chunks() const { return div_up((size_t)r1, (size_t)kBlock2d) * per; }
  __device__ bool flipped() const { return __builtin_amdgcn_readfirstlane((int)flip) != 0; }  // (a scalar branch)
  // first block of chunk c
  __device__ void first(size_t c, int& bi, int& bj) const {
    if (c < (1ull << 32)) {
      bi = (int)((uint32_t)c / (uint32_t)per);
      bj = (int)((uint32_t)c - (uint32_t)bi * (uint32_t)per) * kBlocks;
    } else {
      bi = (int)(c / per);
      bj = (int)(c - (size_t)bi * per) * kBlocks;
    }
  }
  __device__ void stage(size_t c, uint16_t* lds) const {
    int bi, bj;
    first(c, bi, bj);
    const uint32_t i0 = (uint32_t)bi * kBlock2d, sx = (uint32_t)min(kBlock2d, r1 - (int)i0);
    u32x4 v[3];
    if (flipped()) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const uint32_t s = (threadIdx.x & 63) + 64 * k, col = s / kFlipSegs, seg = s % kFlipSegs;
        const uint32_t step = ((i0 + col) & ~7u) + 8 * seg;
        // (8 steps that hold none of the rows are not read)
        const bool in = col < (uint32_t)r2 && step < i0 + sx + col;
        v[k] = *glob(reinterpret_cast<const u32x4*>(q + t.at_step(0, in ? col : 0u, in ? step : 0u)));
      }
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const uint32_t s = (threadIdx.x & 63) + 64 * k;
        *reinterpret_cast<u32x4*>(lds + s / kFlipSegs * kFlipPitch + 8 * (s % kFlipSegs)) = v[k];
      }
      return;
    }
    const uint32_t t0 = ((uint32_t)bj * kBlock2d + (i0 & 63)) & ~7u;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const uint32_t s = (threadIdx.x & 63) + 64 * k, row = s / kSegs, seg = s % kSegs;
      const uint32_t i = i0 + row, l = i & 63;
      // the step within the row's own strip (the next one's steps start over)
      const int step = (int)(t0 + 8 * seg) - (l < (i0 & 63) ? 64 : 0);
      // (8 steps that hold none of the row's columns are not read)
      const bool in = row < sx && step >= 0 && step < r2 + (int)l;
      v[k] = *glob(reinterpret_cast<const u32x4*>(q + t.at_step(in ? i >> 6 : 0u, in ? l : 0u, in ? (uint32_t)step : 0u)));
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const uint32_t s = (threadIdx.x & 63) + 64 * k, row = s / kSegs, seg = s % kSegs;
      if (row < kBlock2d) *reinterpret_cast<u32x4*>(lds + row * kPitch + 8 * seg) = v[k];
    }
  }
  // row and column (from the chunk's first) of the lane's first symbol, its
  // block's width and the symbols left in the chunk from there
  __device__ int place(size_t c, int& bi, int& bj, int& sx, int& b, int& ii, int& jj, int& w, int& last_w) const {
    first(c, bi, bj);
    sx = min(kBlock2d, r1 - bi * kBlock2d);
    const int nblk = min(kBlocks, nby - bj);
    last_w = min(kBlock2d, r2 - (bj + nblk - 1) * kBlock2d);
    const int m0 = kRun * (int)(threadIdx.x & 63), area = sx * kBlock2d;
    const int total = (nblk - 1) * area + sx * last_w;
    b = min((int)((uint32_t)m0 / (uint32_t)area), nblk - 1);
    w = b == nblk - 1 ? last_w : kBlock2d;
    const int r = m0 - b * area;
    ii = (int)((uint32_t)r / (uint32_t)w);
    jj = r - ii * w;
    return total - m0;
  }
  __device__ int load(size_t c, const uint16_t* lds, uint32_t* sym) const {
    int bi, bj, sx, b, ii, jj, w, last_w;
    first(c, bi, bj);
    const uint32_t rem = ((uint32_t)bj * kBlock2d + ((uint32_t)(bi * kBlock2d) & 63)) & 7u;
    if (!flipped() && bi * kBlock2d + kBlock2d <= r1 && (bj + kBlocks) * kBlock2d <= r2) {
      // whole blocks: three half rows a lane, eight lanes a block
      const uint32_t lane = threadIdx.x & 63, s = lane & 7, odd = s & 1;
      const uint16_t* p = lds + rem + ((3 * s) >> 1) * (kPitch + 1) + (lane >> 3) * kBlock2d + 6 * odd;
      const uint16_t* p2 = p + (odd ? kPitch + 1 - 6 : 6);
#pragma unroll
      for (int k = 0; k < 6; k++) {
        sym[k] = p[k];
        sym[6 + k] = p2[k];
        sym[12 + k] = p[kPitch + 1 + k];
      }
      return kRun;
    }
    const int left = place(c, bi, bj, sx, b, ii, jj, w, last_w);
    auto walk = [&](auto at) {
#pragma unroll
      for (int k = 0; k < kRun; k++) {
        const bool in = k < left;
        sym[k] = lds[in ? at(ii, b * kBlock2d + jj) : (int)rem];
        if (++jj == w) {
          jj = 0;
          if (++ii == sx) {
            ii = 0;
            b++;
            w = bj + b == nby - 1 ? last_w : kBlock2d;
          }
        }
      }
    };
    if (flipped()) walk([&](int i, int col) { return col * kFlipPitch + ((bi * kBlock2d + col) & 7) + i; });
    else walk([&](int i, int col) { return (int)rem + i * (kPitch + 1) + col; });
    return max(0, min(kRun, left));
  }
  __device__ size_t elem(size_t c, int k) const {
    int bi, bj, sx, b, ii, jj, w, last_w;
    place(c, bi, bj, sx, b, ii, jj, w, last_w);
    for (jj += k; jj >= w;) {
      jj -= w;
      if (++ii == sx) {
        ii = 0;
        b++;
        w = bj + b == nby - 1 ? last_w : kBlock2d;
      }
    }
    return (size_t)(bi * kBlock2d + ii) * r2 + (bj + b) * kBlock2d + jj;
  }
};
using SrcCodes2d = SrcCodes2dT<float>;

struct SinkIds2d {
  static constexpr int kBytes = 2;
  uint16_t* su;  // tiles
  uint16_t* sv;
  size_t n;
  Tile2d t;
  __device__ void put(uint64_t p, uint32_t s) const {
    if (p < n) su[t.at_linear(p)] = (uint16_t)s;
    else sv[t.at_linear(p - n)] = (uint16_t)s;
  }
};

// The id streams when every id symbol is below 256 (the float codec's ids
// stay below 90): staged as bytes, so a block's whole output fits its LDS
// stage and leaves in coalesced stores, and decoded up to 3 codes per step.
struct SinkIds2dB {
  static constexpr int kBytes = 1;
  uint16_t* su;  // tiles
  uint16_t* sv;
  size_t n;
  Tile2d t;
  __device__ void put(uint64_t p, uint32_t s) const {
    if (p < n) su[t.at_linear(p)] = (uint16_t)s;
    else sv[t.at_linear(p - n)] = (uint16_t)s;
  }
};

// block-major position -> element
struct SinkCodes2d {
  static constexpr int kBytes = 2;
  uint16_t* q;  // tiles
  Tile2d t;
  int r1, r2, nby;
  // optional: zero-filled per-block counts of code 0 (the unpredictable
  // marker), added up while the codes are written
  uint32_t* zc = nullptr;
  // optional: zero-filled per-block masks of the code-0 positions (three
  // words per block, bit k for the block's k-th element in row-major order)
  uint64_t* zm = nullptr;
  __device__ void put(uint64_t p, uint32_t s) const {
    const uint64_t rowblk = (uint64_t)kBlock2d * r2;
    int bi, bj, ii, jj;
    uint32_t k;  // position within the block
    if (p < (1ull << 32) && rowblk < (1ull << 32)) {
      // divisions by multiplication, but in the field's last blocks (a
      // division is some 30 instructions, of 32 bits): p / (12 r2) is
      // (p / 12) / r2
      const uint32_t p32 = (uint32_t)p, rb = (uint32_t)rowblk;
      const uint32_t b = t.rows_in(p32 / kBlock2d), rem = p32 - b * rb;
      bi = (int)b;
      const uint32_t sx = (uint32_t)min(kBlock2d, r1 - bi * kBlock2d);
      bj = min((int)(sx == kBlock2d ? rem / (kBlock2d * kBlock2d) : rem / (sx * kBlock2d)), nby - 1);
      const uint32_t rem2 = rem - (uint32_t)bj * sx * kBlock2d;
      const uint32_t sy = (uint32_t)min(kBlock2d, r2 - bj * kBlock2d);
      ii = (int)(sy == kBlock2d ? rem2 / kBlock2d : rem2 / sy);
      jj = (int)(rem2 - (uint32_t)ii * sy);
      k = rem2;
    } else {
      bi = (int)(p / rowblk);
      const uint64_t rem = p - (uint64_t)bi * rowblk;
      const int sx = min(kBlock2d, r1 - bi * kBlock2d);
      bj = (int)(rem / ((uint64_t)sx * kBlock2d));
      if (bj > nby - 1) bj = nby - 1;
      const uint32_t rem2 = (uint32_t)(rem - (uint64_t)bj * sx * kBlock2d);
      const int sy = min(kBlock2d, r2 - bj * kBlock2d);
      ii = rem2 / sy;
      jj = rem2 - ii * sy;
      k = rem2;
    }
    q[t.at(bi * kBlock2d + ii, bj * kBlock2d + jj)] = (uint16_t)s;
    if (zm && s == 0)
      atomicOr((unsigned long long*)&zm[3 * ((size_t)bi * nby + bj) + (k >> 6)], 1ull << (k & 63));
    if (zc) {
      // one atomic per block among the active lanes' zeros: consecutive
      // positions (the staged writes) fall in one or two blocks
      const uint32_t b = (uint32_t)bi * (uint32_t)nby + (uint32_t)bj;
      const bool z = s == 0;
      uint64_t m = __ballot(z);
      while (m) {
        const int leader = __ffsll((long long)m) - 1;
        const uint32_t bl = (uint32_t)__shfl((int)b, leader);
        const uint64_t same = __ballot(z && b == bl);
        if ((int)(threadIdx.x & 63) == leader) atomicAdd(&zc[bl], (uint32_t)__popcll(same));
        m &= ~same;
      }
    }
  }
};

// Unpredictable values in block-major order. One wave per 12x12 block (4
// blocks per 256-thread workgroup); its lanes take the block's elements in
// row-major order, 64 at a time, so a row's 12 codes are read by consecutive
// lanes, and the ranks of the zero codes come from a ballot.
constexpr int kUnpWaves = 4;
inline int unp_grid(size_t nb) { return (int)div_up(nb, (size_t)kUnpWaves); }

struct BlockView {
  int i0, j0, sy, m;
  __device__ BlockView(size_t b, int r1, int r2, int nby) {
    const int bi = (int)(b / nby), bj = (int)(b - (size_t)bi * nby);
    i0 = bi * kBlock2d;
    j0 = bj * kBlock2d;
    const int sx = min(kBlock2d, r1 - i0);
    sy = min(kBlock2d, r2 - j0);
    m = sx * sy;
  }
  __device__ size_t tile_elem(int k, const Tile2d& t) const {
    const int ii = k / sy, jj = k - ii * sy;
    return t.at(i0 + ii, j0 + jj);
  }
};

__global__ void __launch_bounds__(256) k_block_zeros(const uint16_t* __restrict__ q, Tile2d t, int r1, int r2,
                                                     int nby, size_t nb, uint32_t* __restrict__ cnt) {
  const size_t b = (size_t)blockIdx.x * kUnpWaves + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= nb) return;  // uniform across the wave
  const BlockView v(b, r1, r2, nby);
  uint32_t z = 0;
  for (int k0 = 0; k0 < v.m; k0 += 64) {
    const int k = k0 + lane;
    const bool zero = k < v.m && q[v.tile_elem(k, t)] == 0;
    z += (uint32_t)__popcll(__ballot(zero));
  }
  if (lane == 0) cnt[b] = z;
}

template <typename T>
__global__ void __launch_bounds__(256) k_scatter_unpred(const uint16_t* __restrict__ q, Tile2d t,
                                                        const T* __restrict__ vals, int r1, int r2, int nby, size_t nb,
                                                        const uint64_t* __restrict__ off, uint64_t count,
                                                        T* __restrict__ raw, int* __restrict__ err) {
  const size_t b = (size_t)blockIdx.x * kUnpWaves + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (b >= nb) return;
  const BlockView v(b, r1, r2, nby);
  uint64_t o = off[b];
  const uint64_t below = (1ull << lane) - 1;
  for (int k0 = 0; k0 < v.m; k0 += 64) {
    const int k = k0 + lane;
    const size_t e = k < v.m ? v.tile_elem(k, t) : 0;
    const bool zero = k < v.m && q[e] == 0;
    const uint64_t mask = __ballot(zero);
    if (zero) {
      const uint64_t r = o + __popcll(mask & below);
      if (r < count) raw[e] = vals[r];
      else *err = 1;
    }
    o += __popcll(mask);
  }
}

// offline_log transform (include/sz_cp_preserve_utils.hpp:205-221): host-libm
// log2f of |x| (-100 for 0) and the MSB-first sign bitmaps (1 = positive):
// one wave per 64 values; reversing the ballot's 64 bits and then its byte
// order puts value 8k+j at bit 7-j of byte k. Block y = component.
__global__ void __launch_bounds__(256) k_log2d(const float* __restrict__ U, const float* __restrict__ V, size_t n,
                                               size_t nq, LibmView lv, float* __restrict__ LU,
                                               float* __restrict__ LV, uint64_t* __restrict__ smap) {
  const int c = blockIdx.y, lane = threadIdx.x & 63;
  const float* X = c ? V : U;
  float* L = c ? LV : LU;
  const size_t q = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (q >= nq) return;  // uniform across the wave
  const size_t e = q * 64 + lane;
  const float x = e < n ? X[e] : 0.f;
  if (e < n) L[e] = x != 0 ? host_log2f(lv, fabsf(x)) : -100.f;
  const uint64_t m = __ballot(x > 0);
  if (lane == 0) smap[c * nq + q] = __builtin_bswap64(__builtin_bitreverse64(m));
}

// offline_log decode, in place (src/sz_decompress_cp_preserve_2d.cpp:80-92):
// 0 below -99, else +-exp2f (host libm) by the sign bitmap.
__global__ void __launch_bounds__(256) k_finish2d(float* __restrict__ U, float* __restrict__ V, size_t n,
                                                  const uint8_t* __restrict__ signs, size_t smap, LibmView ev) {
  const int c = blockIdx.y;
  float* X = c ? V : U;
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float lx = X[e];
  const bool pos = (signs[c * smap + e / 8] >> (7 - (e % 8))) & 1;
  float y = 0.f;
  if (!(lx < -99)) {
    const float t = host_exp2f(ev, lx);
    y = pos ? t : -t;
  }
  X[e] = y;
}

// The quantization codes as a tile array, padding and all: the histogram's
// count of code 0 leaves the pads out.
struct U16Hist {
  const uint16_t* p;  // 8-byte aligned (the code arrays are 256-byte aligned)
  size_t n;
  uint32_t pads;
  static constexpr int kChunk = 1024;
  // four codes per item, one 8-byte load
  static constexpr int kMaxItems = kChunk / 4, kPer = 4;
  __device__ int get(size_t c, int idx, uint32_t* sym) const {
    const uint2 w = *reinterpret_cast<const uint2*>(p + c * kChunk + 4 * (size_t)idx);
    sym[0] = w.x & 0xFFFFu;
    sym[1] = w.x >> 16;
    sym[2] = w.y & 0xFFFFu;
    sym[3] = w.y >> 16;
    return 4;
  }
  static constexpr bool kPads = true;  // code-0 pads, counted out of bin 0
  __device__ uint32_t at(size_t i) const { return p[i]; }
};

// ---- batched entropy stage: many fields' streams per launch -----------------
// One component of one field for the batched unpredictable scatter.
struct UnpJob {
  Tile2d t;
  const float* x;        // the stream's unpredictable values
  int r1, r2, nby;
  size_t nb;
  const uint64_t* off;   // global exclusive scan of the blocks' zero counts, at this component's first block
  float* out;            // per-element values (tiles)
  uint64_t count;        // values in the stream
  int* err;              // set when the codes ask for more values than the stream holds
  uint32_t blk0;
  const uint64_t* zm;    // per-block code-0 masks (SinkCodes2d::zm)
};

inline uint32_t unp_blocks(size_t nb) { return (uint32_t)div_up(3 * nb, (size_t)256); }

// A lane takes a 64-bit word of a block's mask (three a block) and goes through
// its bits; a wave in which some word holds many (land, noise) takes its words
// one after the other instead, a lane per bit, so that loads and stores stay
// together. A wave per block, a lane per code, took 1.20 of the 12.08 ms of
// decompressing 96 fields; now 11.01 in all.
__global__ void __launch_bounds__(256) k_scatter_unpred_multi(const UnpJob* __restrict__ jobs, int nj) {
  const UnpJob& J = jobs[job_of(jobs, nj, blockIdx.x)];
  const Tile2d t = J.t;
  const auto x = glob(J.x);
  const auto out = glob(J.out);
  const auto zm = glob(J.zm);
  const uint64_t count = J.count;
  const size_t idx = (size_t)(blockIdx.x - J.blk0) * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool in = idx < 3 * J.nb;
  const size_t b = in ? idx / 3 : 0;
  const int w = in ? (int)(idx - 3 * b) : 0;
  const uint64_t m = in ? zm[3 * b + w] : 0;
  if (!__any(m != 0)) return;
  uint64_t o = 0;
  if (m) {
    o = glob(J.off)[b] - glob(J.off)[0];
    for (int p = 0; p < w; p++) o += (uint64_t)__popcll(zm[3 * b + p]);
  }
  bool lacking = false;
  auto put = [&](const BlockView& v, int k, uint64_t r) {
    if (r < count) out[v.tile_elem(k, t)] = x[r];
    else lacking = true;
  };
  if (!__any(__popcll(m) > 8)) {
    const BlockView v(b, J.r1, J.r2, J.nby);
    for (uint64_t q = m; q; q &= q - 1) put(v, 64 * w + __ffsll((long long)q) - 1, o++);
  } else {
    for (int l = 0; l < 64; l++) {
      const uint64_t q = __shfl((unsigned long long)m, l);
      if (!q) continue;
      const size_t bl = (size_t)__shfl((unsigned long long)b, l);
      const BlockView v(bl, J.r1, J.r2, J.nby);
      const uint64_t ol = __shfl((unsigned long long)o, l);
      const int k = 64 * __shfl(w, l) + lane;
      if ((q >> lane) & 1) put(v, k, ol + __popcll(q & ((1ull << lane) - 1)));
    }
  }
  if (lacking) *J.err = 1;
}

// The present symbols of each histogram (one 1024-thread workgroup per
// histogram), in symbol order, packed into one list: histogram h gets
// count[h] entries from base[h].
struct CompactJob {
  const uint32_t* hist;
  uint32_t nbins;
};

__global__ void __launch_bounds__(1024) k_compact_hist(const CompactJob* __restrict__ jobs, uint32_t* __restrict__ count,
                                                       uint64_t* __restrict__ base,
                                                       unsigned long long* __restrict__ total,
                                                       uint32_t* __restrict__ syms, uint32_t* __restrict__ freqs) {
  __shared__ uint32_t wsum[16];
  __shared__ uint64_t b0;
  const CompactJob J = jobs[blockIdx.x];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint32_t c = 0;
  for (uint32_t i = threadIdx.x; i < J.nbins; i += 1024) c += J.hist[i] != 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  if (lane == 0) wsum[wv] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t k = 0;
    for (int x = 0; x < 16; x++) k += wsum[x];
    const uint64_t at = atomicAdd(total, (unsigned long long)k);
    count[blockIdx.x] = k;
    base[blockIdx.x] = at;
    b0 = at;
  }
  __syncthreads();
  uint64_t pos = b0;
  const uint64_t below = (1ull << lane) - 1;
  for (uint32_t i0 = 0; i0 < J.nbins; i0 += 1024) {
    const uint32_t i = i0 + threadIdx.x;
    const uint32_t f = i < J.nbins ? J.hist[i] : 0u;
    const uint64_t m = __ballot(f != 0);
    if (lane == 0) wsum[wv] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int x = 0; x < 16; x++) {
      const uint32_t y = wsum[x];
      before += x < wv ? y : 0u;
      all += y;
    }
    if (f) {
      const uint64_t at = pos + before + (uint32_t)__popcll(m & below);
      syms[at] = i;
      freqs[at] = f;
    }
    pos += all;
    __syncthreads();
  }
}

// Codebooks of many trees into their dense tables (one workgroup per tree).
struct CbJob {
  const uint32_t* syms;
  const uint64_t* codes;
  const uint8_t* lens;
  uint32_t k;
  uint64_t* code;
  uint8_t* len;
};

__global__ void __launch_bounds__(256) k_scatter_codebooks(const CbJob* __restrict__ jobs) {
  const CbJob& J = jobs[blockIdx.x];
  for (uint32_t i = threadIdx.x; i < J.k; i += blockDim.x) {
    J.code[J.syms[i]] = J.codes[i];
    J.len[J.syms[i]] = J.lens[i];
  }
}

// A host-built tree moved to where the device tree builder puts its results:
// codebook scattered into the dense tables, serialized bytes, info words.
struct HostTreeJob {
  CbJob cb;
  const uint8_t* tree_src;
  uint8_t* tree_dst;
  uint64_t tree_n;
  uint64_t* info_dst;
  uint64_t info[4];
};

__global__ void __launch_bounds__(256) k_host_trees_in(const HostTreeJob* __restrict__ jobs) {
  const HostTreeJob& J = jobs[blockIdx.x];
  for (uint32_t i = threadIdx.x; i < J.cb.k; i += blockDim.x) {
    J.cb.code[J.cb.syms[i]] = J.cb.codes[i];
    J.cb.len[J.cb.syms[i]] = J.cb.lens[i];
  }
  for (uint64_t i = threadIdx.x; i < J.tree_n; i += blockDim.x) J.tree_dst[i] = J.tree_src[i];
  if (threadIdx.x < 4) J.info_dst[threadIdx.x] = J.info[threadIdx.x];
}

// out[j] = a[j].hi - a[j].lo: per-stream sums read off global exclusive scans.
struct ScanDiff {
  const uint64_t* lo;
  const uint64_t* hi;
};

__global__ void k_scan_diffs(const ScanDiff* __restrict__ d, int n, uint64_t* __restrict__ out) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) out[j] = *d[j].hi - *d[j].lo;
}

// Stream assembly: one workgroup per piece (at most 64 KiB) copies len bytes
// to out + dst. The destination's aligned words are stored whole, each built
// from the two source words that cover it (alignbyte); the at most 3 bytes
// before and after them go byte by byte, so neighbouring pieces never share a
// word store.
struct CopyPiece {
  uint64_t dst;
  const uint8_t* src;
  uint32_t len;
  uint32_t pad;
};

__device__ __forceinline__ void copy_piece(uint8_t* __restrict__ d, const uint8_t* __restrict__ s, uint32_t n) {
  const uint32_t head = min(n, (uint32_t)((4u - ((uint32_t)(uintptr_t)d & 3u)) & 3u));
  const uint32_t nw = (n - head) >> 2, tail0 = head + 4 * nw;
  if (threadIdx.x < head) d[threadIdx.x] = s[threadIdx.x];
  if (threadIdx.x < n - tail0) d[tail0 + threadIdx.x] = s[tail0 + threadIdx.x];
  uint32_t* dw = (uint32_t*)(d + head);
  const uint8_t* sp = s + head;
  const uint32_t mis = (uint32_t)(uintptr_t)sp & 3u;
  const uint32_t* sw = (const uint32_t*)(sp - mis);
  if (mis == 0) {
    for (uint32_t k = threadIdx.x; k < nw; k += blockDim.x) dw[k] = sw[k];
  } else {
    for (uint32_t k = threadIdx.x; k < nw; k += blockDim.x)
      dw[k] = __builtin_amdgcn_alignbyte(sw[k + 1], sw[k], mis);
  }
}

__global__ void __launch_bounds__(256) k_assemble(const CopyPiece* __restrict__ pieces, uint8_t* __restrict__ out) {
  const CopyPiece P = pieces[blockIdx.x];
  copy_piece(out + P.dst, P.src, P.len);
}

// ---- device-side layout of a batch's streams: every size and offset follows
// from the per-stream totals and the device-built trees, so no host round trip
// sits between the scans and the assembled streams.
struct Layout2d {
  // set by the host
  uint64_t off;              // stream offset in the batch output
  uint64_t cap;              // bytes available there
  uint64_t nb;               // 12x12 blocks
  const uint64_t* tot;       // bits of the eb/u/v streams, unpredictable u/v counts
  const uint64_t* tinfo[3];  // device tree info of the eb/u/v trees (node count, tree bytes, ...)
  const uint8_t* tree[3];
  EncJob<SrcIds2d>* ej_ids;  // jobs whose word arrays k_layout2d fills in
  EncJob<SrcCodes2d>* ej_codes;  // [2], also their unpredictable-value arrays
  // set by k_layout2d
  uint32_t* words;  // eb, u, v word arrays, consecutive
  float* unp;       // u then v unpredictable values
  uint64_t bytes[3], wn[3], unp_n[2], size;
  uint64_t at[11];  // hdr, h_eb, eb bits, hu1, unp u, hu2, u bits, hv1, unp v, hv2, v bits
};

__device__ __forceinline__ uint64_t wave_incl_scan64(uint64_t x) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up((unsigned long long)x, o);
    if ((int)(threadIdx.x & 63) >= o) x += y;
  }
  return x;
}

// One wave, a lane per field: sizes, offsets, the word and value arrays of
// every field (in the preallocated pools: *err set when they would overflow),
// sizes[k]. One thread going through the fields measured 1.3 us a field, the
// latency of its loads.
__global__ void __launch_bounds__(64) k_layout2d(Layout2d* __restrict__ L, int nf, uint32_t* words, uint64_t words_cap,
                                                 float* unp, uint64_t unp_cap, uint64_t* __restrict__ sizes,
                                                 uint64_t* __restrict__ words_used, int* __restrict__ err) {
  const int lane = threadIdx.x;
  uint64_t wpos = 0, upos = 0;
  for (int k0 = 0; k0 < nf; k0 += 64) {
    const int k = k0 + lane;
    const bool in = k < nf;
    Layout2d& F = L[in ? k : 0];
    uint64_t wneed = 0, uneed = 0, wn[3], un[2], size = 0;
    if (in) {
      uint64_t tb[3], bytes[3];
      for (int t = 0; t < 3; t++) {
        bytes[t] = (F.tot[t] + 7) / 8;
        wn[t] = (bytes[t] + 3) / 4 + 2;
        F.bytes[t] = bytes[t];
        F.wn[t] = wn[t];
        tb[t] = F.tinfo[t][1];
      }
      for (int c = 0; c < 2; c++) F.unp_n[c] = un[c] = F.tot[3 + c];
      const uint64_t ind = (F.nb - 1) / 8 + 1;
      const uint64_t h_eb = 8 + 4 + tb[0] + 8, h1 = 4 + 1 + 4 + 8 + 8 + 8;
      const uint64_t hu2 = ind + 8 + 4 + tb[1] + 8, hv2 = ind + 8 + 4 + tb[2] + 8;
      uint64_t p = F.off;
      const uint64_t sec[11] = {36, h_eb, bytes[0], h1, 4 * un[0], hu2, bytes[1], h1, 4 * un[1], hv2, bytes[2]};
      for (int q = 0; q < 11; q++) {
        F.at[q] = p;
        p += sec[q];
      }
      size = p - F.off;
      F.size = size;
      sizes[k] = size;
      wneed = (wn[0] + wn[1] + wn[2] + 63) & ~63ull;
      uneed = (un[0] + un[1] + 63) & ~63ull;
    }
    const uint64_t wi = wave_incl_scan64(wneed), ui = wave_incl_scan64(uneed);
    const uint64_t wp = wpos + wi - wneed, up = upos + ui - uneed;
    const uint64_t bad = __ballot(in && (size > F.cap || wp + wneed > words_cap || up + uneed > unp_cap));
    const int first_bad = bad ? __ffsll((long long)bad) - 1 : 64;
    if (in && lane < first_bad) {
      F.words = words + wp;
      F.unp = unp + up;
      F.ej_ids->words = F.words;
      F.ej_codes[0].words = F.words + wn[0];
      F.ej_codes[1].words = F.words + wn[0] + wn[1];
      F.ej_codes[0].src.unp = F.unp;
      F.ej_codes[1].src.unp = F.unp + un[0];
    }
    if (bad) {
      // this and the remaining fields keep null arrays: the passes that
      // follow skip them, and the host reports the error
      if (lane == first_bad) {
        *err = 1;
        *words_used = wp;
      }
      return;
    }
    wpos += (uint64_t)__shfl((unsigned long long)wi, 63);
    upos += (uint64_t)__shfl((unsigned long long)ui, 63);
  }
  if (lane == 0) *words_used = wpos;
}

__global__ void k_fill_words(uint32_t* __restrict__ w, const uint64_t* __restrict__ n) {
  const uint64_t m = *n;
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < m; i += (uint64_t)gridDim.x * blockDim.x)
    w[i] = 0;
}

__device__ __forceinline__ void put_bytes(uint8_t* p, uint64_t v, int nbytes) {
  for (int b = 0; b < nbytes; b++) p[b] = (uint8_t)(v >> (8 * b));
}

// One workgroup per field: the stream header, the id tree head, the two
// compressor heads and the two code tree heads (all-zero block indicators
// first), trees copied from the device builds (the host layout of
// src/sz_compress_cp_preserve_2d.cpp:258-269, src/sz_compress_3d.cpp:219-228).
__global__ void __launch_bounds__(256) k_write_heads2d(const Layout2d* __restrict__ L, uint8_t* __restrict__ out) {
  const Layout2d& F = L[blockIdx.x];
  if (!F.words) return;  // not laid out (an overflow the host reports)
  const uint64_t ind = (F.nb - 1) / 8 + 1;
  if (threadIdx.x == 0) {
    uint8_t* h = out + F.at[0];
    put_bytes(h, 4, 4);
    put_bytes(h + 4, 0x3CB0000000000000ull, 8);  // DBL_EPSILON
    put_bytes(h + 12, F.bytes[0] + 8 + 4 + F.tinfo[0][1] + 8, 8);
    put_bytes(h + 20, F.at[7] - F.at[3], 8);
    put_bytes(h + 28, F.off + F.size - F.at[7], 8);
    for (int c = 0; c < 2; c++) {
      uint8_t* q = out + F.at[c ? 7 : 3];
      put_bytes(q, kBlock2d, 4);
      q[4] = 0;
      put_bytes(q + 5, kRadius, 4);
      put_bytes(q + 9, 0, 8);   // meanInfo<float>{false, 0}
      put_bytes(q + 17, 0, 8);  // reg_count
      put_bytes(q + 25, F.unp_n[c], 8);
    }
  }
  for (int t = 0; t < 3; t++) {
    uint8_t* q = out + (t == 0 ? F.at[1] : F.at[t == 1 ? 5 : 9] + ind);
    const uint64_t tb = F.tinfo[t][1];
    if (threadIdx.x == 0) {
      put_bytes(q, F.tinfo[t][0], 8);
      put_bytes(q + 8, tb, 4);
      put_bytes(q + 12 + tb, F.bytes[t], 8);
    }
    for (uint64_t b = threadIdx.x; b < tb; b += blockDim.x) q[12 + b] = F.tree[t][b];
  }
  for (uint64_t b = threadIdx.x; b < ind; b += blockDim.x) {
    out[F.at[5] + b] = 0;
    out[F.at[9] + b] = 0;
  }
}

// The five device sections of every field (bitstreams and unpredictable
// values) into place, 64 KiB pieces spread over the workgroups of the
// field's grid row.
__global__ void __launch_bounds__(256) k_assemble2d(const Layout2d* __restrict__ L, uint8_t* __restrict__ out) {
  const Layout2d& F = L[blockIdx.y];
  if (!F.words) return;
  constexpr uint64_t kP = 65536;
  const uint8_t* src[5] = {(const uint8_t*)F.words, (const uint8_t*)F.unp, (const uint8_t*)(F.words + F.wn[0]),
                           (const uint8_t*)(F.unp + F.unp_n[0]), (const uint8_t*)(F.words + F.wn[0] + F.wn[1])};
  const uint64_t len[5] = {F.bytes[0], 4 * F.unp_n[0], F.bytes[1], 4 * F.unp_n[1], F.bytes[2]};
  const uint64_t dst[5] = {F.at[2], F.at[4], F.at[6], F.at[8], F.at[10]};
  uint64_t p = blockIdx.x;
  for (int q = 0; q < 5; q++) {
    const uint64_t np = (len[q] + kP - 1) / kP;
    for (; p < np; p += gridDim.x) {
      const uint64_t o = p * kP;
      copy_piece(out + dst[q] + o, src[q] + o, (uint32_t)min(kP, len[q] - o));
    }
    p -= np;
  }
}

}  // namespace

// ---------------------------------------------------------------- host ----
namespace {

template <typename V>
void put(std::vector<uint8_t>& o, const V& v) {
  const size_t at = o.size();
  o.resize(at + sizeof(V));
  std::memcpy(o.data() + at, &v, sizeof(V));
}

struct Piece {  // a contiguous part of the output stream
  size_t off;
  const void* src;  // host (staging) or device pointer
  size_t len;
  bool device;
};

// Host-written parts of a 2D stream (src/sz_compress_cp_preserve_2d.cpp:258-269,
// src/sz_compress_3d.cpp:219-228): the id section's tree head, the two
// components' compressor heads (block size, radius, meanInfo<T>, unpredictable
// count) and tree heads (the all-zero block indicator bytes first), and the
// stream header with the three section sizes. vb: bytes of T.
// One pinned staging area mirrored on the device: tables are filled on the
// host and sent with one copy; take() returns the device address of a slot and
// its host address through `host`.
struct Arena {
  uint8_t* h = nullptr;
  uint8_t* d = nullptr;
  size_t used = 0, cap = 0;
  template <class T>
  T* take(size_t count, T** host) {
    used = (used + 15) & ~(size_t)15;
    CPSZ_REQUIRE(used + count * sizeof(T) <= cap, kErrInternal, "staging table overflow");
    *host = (T*)(h + used);
    T* dp = (T*)(d + used);
    used += count * sizeof(T);
    return dp;
  }
};

struct Heads2d {
  std::vector<uint8_t> hdr, h_eb, hu1, hu2, hv1, hv2;
  size_t eb_size = 0, u_size = 0, v_size = 0;
};

void heads_2d(const HuffEncodeTable& t_eb, const HuffEncodeTable& t_u, const HuffEncodeTable& t_v, size_t bytes_eb,
              size_t bytes_u, size_t bytes_v, uint64_t unp_u, uint64_t unp_v, size_t nb, bool log, size_t vb,
              Heads2d& H) {
  const size_t ind_bytes = (nb - 1) / 8 + 1;
  auto huff_head = [](std::vector<uint8_t>& h, const HuffEncodeTable& t, size_t nbytes) {
    put(h, (size_t)t.node_count);
    put(h, (uint32_t)t.tree.size());
    h.insert(h.end(), t.tree.begin(), t.tree.end());
    put(h, (size_t)nbytes);
  };
  auto comp_head = [&](std::vector<uint8_t>& h, uint64_t unp_count) {
    put(h, (int)kBlock2d);
    put(h, (char)0);
    put(h, (int)kRadius);
    put(h, (uint64_t)0);  // meanInfo<T>{false, 0}: flag byte, padding bytes, T 0 (8 or 16 bytes)
    if (vb == 8) put(h, (uint64_t)0);
    put(h, (size_t)0);    // reg_count
    put(h, (size_t)unp_count);
  };
  H.hdr.clear();
  H.h_eb.clear();
  H.hu1.clear();
  H.hv1.clear();
  huff_head(H.h_eb, t_eb, bytes_eb);
  comp_head(H.hu1, unp_u);
  comp_head(H.hv1, unp_v);
  H.hu2.assign(ind_bytes, 0);
  H.hv2.assign(ind_bytes, 0);
  huff_head(H.hu2, t_u, bytes_u);
  huff_head(H.hv2, t_v, bytes_v);
  H.eb_size = H.h_eb.size() + bytes_eb;
  H.u_size = H.hu1.size() + vb * unp_u + H.hu2.size() + bytes_u;
  H.v_size = H.hv1.size() + vb * unp_v + H.hv2.size() + bytes_v;
  put(H.hdr, (int)(log ? 2 : 4));
  put(H.hdr, (double)DBL_EPSILON);
  put(H.hdr, H.eb_size);
  put(H.hdr, H.u_size);
  put(H.hdr, H.v_size);
}

size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace

// ------------------------------------------------------------- staged form --
size_t c2_scratch_bytes(size_t r1, size_t r2) {
  const size_t n = r1 * r2, te = Tile2d(r1, r2).elems();
  return 2 * al256(2 * n) + 4 * al256(2 * te) + al256((kMaxEbCode + 2 * 65536) * 4) + al256(16) + al256(8 * bnd_words(r1, r2)) + al256(4);
}

void c2_bind(C2Work& w, uint8_t* p) {
  w.t = Tile2d(w.r1, w.r2);
  const size_t n = w.r1 * w.r2, te = w.t.elems();
  auto take = [&](size_t bytes) {
    uint8_t* q = p;
    p += al256(bytes);
    return q;
  };
  w.cu = (uint16_t*)take(2 * n);
  w.cv = (uint16_t*)take(2 * n);
  w.tu = (uint16_t*)take(2 * te);
  w.tv = (uint16_t*)take(2 * te);
  w.qu = (uint16_t*)take(2 * te);
  w.qv = (uint16_t*)take(2 * te);
  w.hist = (uint32_t*)take((kMaxEbCode + 2 * 65536) * 4);
  w.flags = (int*)take(16);
  w.bnd = (uint64_t*)take(8 * bnd_words(w.r1, w.r2));
  w.ticket = (int*)take(4);
}

namespace {
std::atomic<bool> g_exact_bounds{false};
}
void set_exact_2d_bounds(bool on) { g_exact_bounds.store(on); }
bool exact_2d_bounds() { return g_exact_bounds.load(); }

namespace {
// The fast bounds pass over a job table already on its way to the device
// (blk tiles), then the FP64 fix-up of the vertices it marked. Graph-capture
// safe: the list counter is cleared by a kernel and nothing waits.
void launch_eb_fast(Ctx& ctx, const Eb2dJob* dj, int nj, uint32_t blk, double max_pwr_eb) {
  hipStream_t st = ctx.stream();
  uint32_t* fx = ctx.buf<uint32_t>("eb.fix", (size_t)blk + 1);  // [0] count, [1..] tiles
  k_fill_u32<<<1, 64, 0, st>>>(fx, 1, 0);
  k_eb2d_multi<true><<<blk, 256, 0, st>>>(dj, nj, max_pwr_eb, ctx.d_q2d(), ctx.q2d_size(), fx + 1, fx);
  // a listed tile costs a few dependent global loads per marked vertex: enough
  // blocks to keep every CU's slots filled (72 VGPRs: 7 blocks per CU)
  k_eb2d_fix<<<std::min<uint32_t>(blk, 2048), 256, 0, st>>>(dj, nj, fx + 1, fx, max_pwr_eb, ctx.d_q2d(),
                                                            ctx.q2d_size());
}
}  // namespace

void c2_eb(Ctx& ctx, C2Work& w, double max_pwr_eb, const EbOverride& ov) {
  CPSZ_REQUIRE((w.f64 ? w.dU64 && w.dV64 : w.dU && w.dV) && w.r1 >= 1 && w.r2 >= 1, kErrArg,
               "compress_2d: bad arguments");
  CPSZ_REQUIRE(w.r1 < (1u << 30) && w.r2 < (1u << 30) && w.r1 * w.r2 < (1ull << 40), kErrUnsupported,
               "compress_2d: field too large");
  hipStream_t st = ctx.stream();
  CPSZ_HIP(hipMemsetAsync(w.hist, 0, (kMaxEbCode + 2 * 65536) * sizeof(uint32_t), st));
  CPSZ_HIP(hipMemsetAsync(w.flags, 0, 4 * sizeof(int), st));
  dim3 grid((unsigned)div_up(w.r2, kTW), (unsigned)div_up(w.r1, kTH));
  if (w.f64) {
    k_eb2d<double><<<grid, 256, 0, st>>>(w.dU64, w.dV64, (int)w.r1, (int)w.r2, max_pwr_eb, ctx.d_q2d(),
                                         ctx.q2d_size(), w.cu, w.cv, w.hist, w.flags, ov, nullptr, 0,
                                         CodeTiles{w.tu, w.tv, w.t});
  } else if (!w.log && !has_override(ov) && !exact_2d_bounds()) {
    Eb2dJob J{};
    J.U = w.dU;
    J.V = w.dV;
    J.r1 = (int)w.r1;
    J.r2 = (int)w.r2;
    J.gx = (int)grid.x;
    J.cu = w.cu;
    J.cv = w.cv;
    J.hist = w.hist;
    J.flags = w.flags;
    J.ct = CodeTiles{w.tu, w.tv, w.t};
    J.blk0 = 0;
    const size_t tiles = (size_t)grid.x * grid.y;
    CPSZ_REQUIRE(tiles < (1ull << 31), kErrUnsupported, "compress_2d: field too large");
    Eb2dJob* dj = ctx.buf<Eb2dJob>("c2eb.job", 1);
    Eb2dJob* hj = (Eb2dJob*)ctx.host_table("c2eb.job", sizeof(Eb2dJob));
    *hj = J;
    ctx.upload_table("c2eb.job", dj, hj, sizeof(Eb2dJob));
    launch_eb_fast(ctx, dj, 1, (uint32_t)tiles, max_pwr_eb);
  } else {
    k_eb2d<float><<<grid, 256, 0, st>>>(w.dU, w.dV, (int)w.r1, (int)w.r2, max_pwr_eb, ctx.d_q2d(), ctx.q2d_size(),
                                        w.cu, w.cv, w.hist, w.flags, ov, w.log ? ctx.d_q2l() : nullptr,
                                        ctx.q2l_size(), CodeTiles{w.tu, w.tv, w.t});
  }
  CPSZ_HIP(hipGetLastError());
}

// Bounds of every field (plain offline, float) in one launch: the fields'
// histograms and flags move to two contiguous arrays, cleared at once. The
// flags stay on the device (the wavefront reads them there).
void c2_eb_batch(Ctx& ctx, C2Work* const* w, size_t nf, double max_pwr_eb, const std::vector<EbOverride>* ov) {
  hipStream_t st = ctx.stream();
  constexpr size_t HN = kMaxEbCode + 2 * 65536;
  uint32_t* hist = ctx.buf<uint32_t>("b2eb.hist", nf * HN);
  int* flags = ctx.buf<int>("b2eb.flags", 4 * nf);
  std::vector<Eb2dJob> jobs(nf);
  uint32_t blk = 0;
  bool approx = !exact_2d_bounds();
  for (size_t k = 0; k < nf; k++) {
    C2Work& W = *w[k];
    CPSZ_REQUIRE(W.dU && W.dV && W.r1 >= 1 && W.r2 >= 1 && !W.log && !W.f64, kErrArg, "compress_2d: bad arguments");
    CPSZ_REQUIRE(W.r1 < (1u << 30) && W.r2 < (1u << 30) && W.r1 * W.r2 < (1ull << 40), kErrUnsupported,
                 "compress_2d: field too large");
    W.hist = hist + k * HN;
    W.flags = flags + 4 * k;
    W.flags_on_device = true;
    Eb2dJob& J = jobs[k];
    J.U = W.dU;
    J.V = W.dV;
    J.r1 = (int)W.r1;
    J.r2 = (int)W.r2;
    J.gx = (int)div_up(W.r2, kTW);
    J.cu = W.cu;
    J.cv = W.cv;
    J.hist = W.hist;
    J.flags = W.flags;
    J.ct = CodeTiles{W.tu, W.tv, W.t};
    J.ov = ov ? (*ov)[k] : EbOverride();
    approx = approx && !has_override(J.ov);
    J.blk0 = blk;
    const size_t tiles = div_up(W.r2, kTW) * div_up(W.r1, kTH);
    CPSZ_REQUIRE(blk + tiles < (1ull << 31), kErrUnsupported, "2D batch: too many tiles in one call");
    blk += (uint32_t)tiles;
  }
  Eb2dJob* dj = ctx.buf<Eb2dJob>("b2eb.jobs", nf);
  const double* q2d = ctx.d_q2d();
  Eb2dJob* hj = (Eb2dJob*)ctx.host_table("b2eb.jobs", nf * sizeof(Eb2dJob));
  std::memcpy(hj, jobs.data(), nf * sizeof(Eb2dJob));
  ctx.upload_table("b2eb.jobs", dj, hj, nf * sizeof(Eb2dJob));
  k_fill_u32<<<1024, 256, 0, st>>>(hist, nf * HN, 0);
  k_fill_u32<<<(unsigned)div_up(4 * nf, 256), 256, 0, st>>>((uint32_t*)flags, 4 * nf, 0);
  if (approx)
    launch_eb_fast(ctx, dj, (int)nf, blk, max_pwr_eb);
  else
    k_eb2d_multi<false><<<blk, 256, 0, st>>>(dj, (int)nf, max_pwr_eb, q2d, ctx.q2d_size(), nullptr, nullptr);
  CPSZ_HIP(hipGetLastError());
}

void c2_check(Ctx& ctx, C2Work* const* w, size_t nf) {
  hipStream_t st = ctx.stream();
  int* hf = (int*)ctx.host_buf("c2.hflags", std::max<size_t>(nf, 1) * 16);
  for (size_t k = 0; k < nf; k++)
    CPSZ_HIP(hipMemcpyAsync(hf + 4 * k, w[k]->flags, 16, hipMemcpyDeviceToHost, st));
  CPSZ_HIP(hipStreamSynchronize(st));
  for (size_t k = 0; k < nf; k++) {
    CPSZ_REQUIRE(hf[4 * k] == 0, kErrNonFinite,
                 "compress_2d: non-finite input or bound (the reference cannot encode it)");
    w[k]->wide = hf[4 * k + 1] != 0;
  }
}

void c2_wavefront(Ctx& ctx, C2Work* const* w, size_t nf, int grid_cap) {
  if (nf == 1 && w[0]->f64) {
    Strip2d64 sa{};
    sa.x[0] = w[0]->dU64;
    sa.x[1] = w[0]->dV64;
    sa.c[0] = w[0]->tu;
    sa.c[1] = w[0]->tv;
    sa.q[0] = w[0]->qu;
    sa.q[1] = w[0]->qv;
    sa.bnd = w[0]->bnd;
    sa.ticket = w[0]->ticket;
    sa.r1 = (int)w[0]->r1;
    sa.r2 = (int)w[0]->r2;
    sa.ngroups = strip_groups<double>(w[0]->r1);
    sa.t = w[0]->t;
    sa.shift = 2;
    wavefront2d_compress64(ctx, sa, grid_cap);
    return;
  }
  for (size_t k = 0; k < nf; k++)
    CPSZ_REQUIRE(!w[k]->f64, kErrUnsupported, "compress_2d: double fields go one at a time");
  std::vector<Strip2d> f(nf);
  for (size_t k = 0; k < nf; k++) {
    Strip2d& sa = f[k];
    sa = Strip2d{};
    const bool lg = w[k]->log;
    sa.x[0] = lg ? w[k]->lu : w[k]->dU;
    sa.x[1] = lg ? w[k]->lv : w[k]->dV;
    sa.c[0] = w[k]->tu;
    sa.c[1] = lg ? w[k]->tu : w[k]->tv;
    sa.shift = lg ? 1 : 2;
    sa.q[0] = w[k]->qu;
    sa.q[1] = w[k]->qv;
    sa.ngroups = strip_groups<float>(w[k]->r1);
    sa.bnd = w[k]->bnd;
    sa.ticket = w[k]->ticket;
    sa.r1 = (int)w[k]->r1;
    sa.r2 = (int)w[k]->r2;
    sa.t = w[k]->t;
    sa.wide = w[k]->wide;
    sa.flags = w[k]->flags_on_device ? w[k]->flags : nullptr;
    CPSZ_REQUIRE(!(lg && (sa.wide || sa.flags)), kErrInternal, "compress_2d_log: eb id beyond the base-2 range");
  }
  wavefront2d_compress(ctx, f, grid_cap);
}

namespace {
template <bool F64>
void c2_entropy_of(Ctx& ctx, const C2Work& w, DeviceStream& out) {
  hipStream_t st = ctx.stream();
  const size_t r1 = w.r1, r2 = w.r2, n = r1 * r2;
  // the values the codec ran on (unpredictable ones are stored as they are)
  const float *dU = w.log ? w.lu : w.dU, *dV = w.log ? w.lv : w.dV;
  const uint16_t *cu = w.cu, *cv = w.cv, *qu = w.qu, *qv = w.qv;
  uint32_t* hist = w.hist;
  // ---- histograms of the quant codes
  {
    const uint32_t win_lo = 32768 - 8192, win_n = 16384;
    const size_t te = w.t.elems();
    U16Hist hu{qu, te, (uint32_t)(te - n)}, hv{qv, te, (uint32_t)(te - n)};
    const size_t nch = te / U16Hist::kChunk;
    const int grid = (int)std::min<size_t>(std::max<size_t>(encode_blocks(nch), 1), 512);
    k_hist<<<grid, 256, win_n * 4, st>>>(hu, nch, hist + kMaxEbCode, win_lo, win_n);
    k_hist<<<grid, 256, win_n * 4, st>>>(hv, nch, hist + kMaxEbCode + 65536, win_lo, win_n);
    CPSZ_HIP(hipGetLastError());
  }
  ctx.mark("hist");
  // ---- host trees
  const size_t hist_n = kMaxEbCode + 2 * 65536;
  uint32_t* hh = (uint32_t*)ctx.host_buf("c2.hist", hist_n * 4);
  CPSZ_HIP(hipMemcpyAsync(hh, hist, hist_n * 4, hipMemcpyDeviceToHost, st));
  const hipEvent_t hist_done = ctx.record_point();
  // the job table needs no tree: it travels while the host builds them
  const size_t nb = div_up(r1, kBlock2d) * div_up(r2, kBlock2d);
  using SrcV = std::conditional_t<F64, SrcCodes2dT<double>, SrcCodes2d>;
  using V = std::conditional_t<F64, double, float>;
  const V* xs[2];
  if constexpr (F64) xs[0] = w.dU64, xs[1] = w.dV64;
  else xs[0] = dU, xs[1] = dV;
  const SrcIds2d s_ids(cu, cv, n);
  const SrcV s_q[2] = {SrcV(qu, w.t, r1, r2, xs[0]), SrcV(qv, w.t, r1, r2, xs[1])};
  const size_t nch_ids = s_ids.chunks(!w.log), ncc = s_q[0].chunks();
  uint64_t* bits = ctx.buf<uint64_t>("c2.bits", nch_ids + 2 * ncc);
  uint64_t* offs = ctx.buf<uint64_t>("c2.offs", nch_ids + 2 * ncc + 8);
  uint32_t* zc = ctx.buf<uint32_t>("c2.zc", 2 * ncc);
  uint64_t* zoff = ctx.buf<uint64_t>("c2.zoff", 2 * ncc + 4);
  uint64_t* totals = ctx.buf<uint64_t>("c2.totals", 8);
  uint64_t* cb_code = ctx.buf<uint64_t>("c2.cbcode", 3 * 65536);
  uint8_t* cb_len = ctx.buf<uint8_t>("c2.cblen", 3 * 65536);
  struct Jobs {
    EncJob<SrcIds2d> ids;
    EncJob<SrcV> q[2];
  };
  Jobs* d_jobs = (Jobs*)ctx.buf<uint8_t>("c2.jobs", sizeof(Jobs));
  const uint32_t iblk = (uint32_t)encode_blocks(nch_ids), cblk = (uint32_t)encode_blocks(ncc);
  // words, unp: null before the encode
  auto send_jobs = [&](uint32_t* const (&words)[3], V* const (&unp)[2]) {
    Jobs* j = (Jobs*)ctx.host_table("c2.jobs", sizeof(Jobs));
    j->ids = {s_ids, nch_ids, cb_code, cb_len, offs, bits, words[0], 0, nullptr};
    for (int c = 0; c < 2; c++) {
      const size_t at = nch_ids + c * ncc;
      j->q[c] = {s_q[c], ncc, cb_code + (c + 1) * 65536, cb_len + (c + 1) * 65536, offs + at, bits + at, words[c + 1],
                 c * cblk, zc + c * ncc};
      j->q[c].src.uoff = zoff + c * ncc;
      j->q[c].src.unp = unp[c];
    }
    ctx.upload_table("c2.jobs", d_jobs, j, sizeof(Jobs));
  };
  send_jobs({nullptr, nullptr, nullptr}, {nullptr, nullptr});
  CPSZ_HIP(hipEventSynchronize(hist_done));
  // the v tree is built on the helper thread beside the eb and u trees, and
  // the id stream's bit counts run on the device meanwhile; the tables are
  // kept per thread so their storage is reused from call to call (the helper
  // reaches the calling thread's objects through references: a thread_local
  // named in the job would be the helper thread's own)
  thread_local HuffEncodeTable t_eb, t_u, t_v_keep;
  thread_local std::vector<uint64_t> f, fv_keep;
  HuffEncodeTable& t_v = t_v_keep;
  std::vector<uint64_t>& fv = fv_keep;
  f.resize(65536);
  fv.resize(65536);
  for (int k = 0; k < 65536; k++) fv[k] = hh[kMaxEbCode + 65536 + k];
  {
    HelperJob v_tree([&] { huff_build(fv.data(), 65536, 2 * kCapacity, t_v); }, !ctx.batch_worker);
    for (int k = 0; k < kMaxEbCode; k++) f[k] = hh[k];
    huff_build(f.data(), kMaxEbCode, 2 * 1024, t_eb);
    upload_codebook(ctx, t_eb, cb_code, cb_len, "c2.eb");
    k_run_bits<SrcIds2d><<<iblk, kEncThreads, 0, st>>>(&d_jobs->ids, 1);
    CPSZ_HIP(hipGetLastError());
    scan_u64(ctx, bits, offs, nch_ids, totals + 0);
    for (int k = 0; k < 65536; k++) f[k] = hh[kMaxEbCode + k];
    huff_build(f.data(), 65536, 2 * kCapacity, t_u);
    v_tree.join();
  }
  ctx.mark("tree");
  // ---- codebooks and encode pass A (bits per chunk)
  upload_codebook(ctx, t_u, cb_code + 65536, cb_len + 65536, "c2.u");
  upload_codebook(ctx, t_v, cb_code + 2 * 65536, cb_len + 2 * 65536, "c2.v");
  k_run_bits<SrcV><<<2 * cblk, kEncThreads, 0, st>>>(d_jobs->q, 2);
  CPSZ_HIP(hipGetLastError());
  // one scan for both components: the second one's first offset is the first one's total
  scan_u64(ctx, bits + nch_ids, offs + nch_ids, 2 * ncc, totals + 1);
  scan_u32_to_u64(ctx, zc, zoff, 2 * ncc, totals + 2);
  uint64_t* ht = (uint64_t*)ctx.host_buf("c2.totals", 8 * 8);
  CPSZ_HIP(hipMemcpyAsync(ht, totals, 3 * 8, hipMemcpyDeviceToHost, st));
  CPSZ_HIP(hipMemcpyAsync(ht + 3, offs + nch_ids + ncc, 8, hipMemcpyDeviceToHost, st));
  CPSZ_HIP(hipMemcpyAsync(ht + 4, zoff + ncc, 8, hipMemcpyDeviceToHost, st));
  CPSZ_HIP(hipStreamSynchronize(st));
  const uint64_t bits_eb = ht[0], bits_u = ht[3], bits_v = ht[1] - ht[3], unp_u = ht[4], unp_v = ht[2] - ht[4];
  ctx.mark("scan");
  // ---- encode pass B into aligned scratch
  const size_t bytes_eb = div_up(bits_eb, 8), bytes_u = div_up(bits_u, 8), bytes_v = div_up(bits_v, 8);
  const size_t w_eb = div_up(bytes_eb, 4) + 2, w_u = div_up(bytes_u, 4) + 2, w_v = div_up(bytes_v, 4) + 2;
  uint32_t* words = ctx.buf<uint32_t>("c2.words", w_eb + w_u + w_v);
  k_fill_u32<<<1024, 256, 0, st>>>(words, w_eb + w_u + w_v, 0);
  // unpredictable values in the field's own type (T = double: 8 bytes each)
  constexpr size_t vb = sizeof(V);
  V* unp = ctx.buf<V>("c2.unp", unp_u + unp_v + 1);
  send_jobs({words, words + w_eb, words + w_eb + w_u}, {unp, unp + unp_u});
  k_run_encode<SrcIds2d><<<iblk, kEncThreads, 0, st>>>(&d_jobs->ids, 1);
  k_run_encode<SrcV><<<2 * cblk, kEncThreads, 0, st>>>(d_jobs->q, 2);
  CPSZ_HIP(hipGetLastError());
  ctx.mark("encode");
  // ---- stream layout
  Heads2d H;
  heads_2d(t_eb, t_u, t_v, bytes_eb, bytes_u, bytes_v, unp_u, unp_v, nb, w.log, vb, H);
  const std::vector<uint8_t>&hdr = H.hdr, &h_eb = H.h_eb, &hu1 = H.hu1, &hu2 = H.hu2, &hv1 = H.hv1, &hv2 = H.hv2;
  const size_t eb_size = H.eb_size, u_size = H.u_size, v_size = H.v_size;
  // offline_log: the two sign bitmaps follow the id section
  // (src/sz_compress_cp_preserve_2d.cpp:358-366)
  const size_t smap = w.log ? (n - 1) / 8 + 1 : 0;
  const size_t total = hdr.size() + eb_size + 2 * smap + u_size + v_size;
  uint8_t* dout = ctx.buf<uint8_t>("c2.out", total + 16);
  // host pieces go through one pinned staging buffer
  std::vector<const std::vector<uint8_t>*> hp = {&hdr, &h_eb, &hu1, &hu2, &hv1, &hv2};
  size_t hbytes = 0;
  for (auto* p : hp) hbytes += p->size();
  uint8_t* stage = (uint8_t*)ctx.host_buf("c2.stage", hbytes);
  std::vector<Piece> pieces;
  size_t pos = 0, spos = 0;
  auto host_piece = [&](const std::vector<uint8_t>& v) {
    std::memcpy(stage + spos, v.data(), v.size());
    pieces.push_back({pos, stage + spos, v.size(), false});
    pos += v.size();
    spos += v.size();
  };
  auto dev_piece = [&](const void* src, size_t len) {
    pieces.push_back({pos, src, len, true});
    pos += len;
  };
  host_piece(hdr);
  host_piece(h_eb);
  dev_piece(words, bytes_eb);
  if (w.log) {
    const size_t nq = div_up(n, 64);
    if (nq * 8 == smap) dev_piece(w.smap, 2 * smap);  // the two bitmaps are already contiguous
    else
      for (int c = 0; c < 2; c++) dev_piece(w.smap + c * nq, smap);
  }
  host_piece(hu1);
  dev_piece(unp, vb * unp_u);
  host_piece(hu2);
  dev_piece(words + w_eb, bytes_u);
  host_piece(hv1);
  dev_piece(unp + unp_u, vb * unp_v);
  host_piece(hv2);
  dev_piece(words + w_eb + w_u, bytes_v);
  CPSZ_REQUIRE(pos == total, kErrInternal, "stream layout mismatch");
  for (const Piece& p : pieces) {
    if (!p.len) continue;
    CPSZ_HIP(hipMemcpyAsync(dout + p.off, p.src, p.len,
                            p.device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, st));
  }
  ctx.mark("assemble");
  out.data = dout;
  out.size = total;
  CPSZ_HIP(hipStreamSynchronize(st));
}

}  // namespace

void c2_entropy(Ctx& ctx, const C2Work& w, DeviceStream& out) {
  if (w.f64) c2_entropy_of<true>(ctx, w, out);
  else c2_entropy_of<false>(ctx, w, out);
}

// Batched entropy stage (plain offline, float), on the device from the codes
// to the finished streams: every field's histograms, block zero counts and
// their scan, the present symbols of every histogram, the Huffman trees (one
// wave per tree, huff_tree.hip), chunk bit counts and one scan for every
// stream, then the layout (sizes, offsets, word arrays) computed by a kernel
// from the per-stream totals, the encodes, the unpredictable gathers, the
// headers and the assembly. The host only fills the job tables up front and
// reads the sizes at the end. Each field's stream is byte-identical to
// c2_entropy's.
void c2_entropy_batch(Ctx& ctx, C2Work* const* w, size_t nf, uint8_t* dout, const std::vector<size_t>& off,
                      const std::vector<size_t>& cap, std::vector<size_t>& size, int workers, bool device_trees) {
  hipStream_t st = ctx.stream();
  constexpr size_t HN = kMaxEbCode + 2 * 65536;  // dense codebook entries per field
  constexpr uint32_t kMaxCodeLeaves = 65536, kMaxIdLeaves = kMaxEbCode;
  struct G {
    size_t n, nb, nch_ids, ncc, zb, cb;  // ncc: chunks of one component's codes
  };
  std::vector<G> g(nf);
  size_t Z = 0, CB = 0, words_cap = 0, unp_cap = 0;
  for (size_t k = 0; k < nf; k++) {
    const C2Work& W = *w[k];
    CPSZ_REQUIRE(!W.log && !W.f64, kErrInternal, "batched entropy: plain float fields only");
    G& x = g[k];
    x.n = W.r1 * W.r2;
    x.nb = div_up(W.r1, kBlock2d) * div_up(W.r2, kBlock2d);
    x.nch_ids = SrcIds2d(W.cu, W.cv, x.n).chunks(true);
    x.ncc = SrcCodes2d(W.qu, W.t, W.r1, W.r2).chunks();
    x.zb = Z;
    Z += 2 * x.ncc;
    x.cb = CB;
    CB += x.nch_ids + 2 * x.ncc;
    words_cap += cap[k] / 4 + 6 + 64;
    unp_cap += 2 * x.n + 64;
  }
  const size_t ntree = 3 * nf;
  // ---- device pools (fixed per batch shape)
  uint32_t* zc = ctx.buf<uint32_t>("b2e.zc", Z + 1);
  uint64_t* zoff = ctx.buf<uint64_t>("b2e.zoff", Z + 1);
  uint64_t* bits = ctx.buf<uint64_t>("b2e.bits", CB + 1);
  uint64_t* offs = ctx.buf<uint64_t>("b2e.offs", CB + 1);
  uint64_t* cb_code = ctx.buf<uint64_t>("b2e.cbcode", nf * HN);
  uint8_t* cb_len = ctx.buf<uint8_t>("b2e.cblen", nf * HN);
  uint32_t* d_syms = ctx.buf<uint32_t>("b2e.syms", nf * (kMaxIdLeaves + 2 * (size_t)kMaxCodeLeaves));
  uint32_t* d_freqs = ctx.buf<uint32_t>("b2e.freqs", nf * (kMaxIdLeaves + 2 * (size_t)kMaxCodeLeaves));
  // per tree: heap (code trees only: id trees fit LDS), tree bytes, info
  const size_t heap_n = kMaxCodeLeaves + 2;
  const size_t tb_code = 13 * (2 * (size_t)kMaxCodeLeaves - 1) + 1, tb_id = 13 * (2 * (size_t)kMaxIdLeaves - 1) + 1;
  const size_t tb_field = (tb_id + 2 * tb_code + 3 * 255) & ~(size_t)255;
  uint64_t* t_heap = ctx.buf<uint64_t>("b2e.theap", 2 * nf * heap_n);
  uint8_t* t_tree = ctx.buf<uint8_t>("b2e.ttree", nf * tb_field);
  uint8_t* meta = ctx.buf<uint8_t>("b2e.meta", ntree * (12 + 32) + nf * 8 + 5 * nf * 8 + 64);
  unsigned long long* d_total = (unsigned long long*)meta;        // present symbols, all trees
  uint64_t* d_words_used = (uint64_t*)(meta + 8);
  int* d_err = (int*)(meta + 16);                                  // layout pool overflow
  uint64_t* d_base = (uint64_t*)(meta + 64);
  uint64_t* d_info = d_base + ntree;                               // 4 per tree
  uint64_t* d_sizes = d_info + 4 * ntree;
  uint64_t* d_tot = d_sizes + nf;
  uint32_t* d_count = (uint32_t*)(d_tot + 5 * nf);
  uint32_t* words = ctx.buf<uint32_t>("b2e.words", words_cap);
  float* unp = ctx.buf<float>("b2e.unp", unp_cap);
  // ---- job tables, filled on the host and sent in one copy
  for (size_t k = 0; k < nf; k++)
    CPSZ_REQUIRE(w[k]->flags == w[0]->flags + 4 * k, kErrInternal, "batched entropy: eb flags not contiguous");
  Arena A;
  const size_t abytes = 2 * nf * sizeof(HistJob<U16Hist>) + ntree * sizeof(CompactJob) +
                        ntree * sizeof(TreeJob) + nf * sizeof(EncJob<SrcIds2d>) + 2 * nf * sizeof(EncJob<SrcCodes2d>) +
                        5 * nf * sizeof(ScanDiff) + nf * sizeof(Layout2d) + 16 * 64;
  A.d = ctx.buf<uint8_t>("b2e.tab", abytes);
  A.h = (uint8_t*)ctx.host_table("b2e.tab", abytes);
  A.cap = abytes;
  HistJob<U16Hist>* hj;
  HistJob<U16Hist>* d_hj = A.take(2 * nf, &hj);
  CompactJob* cj;
  CompactJob* d_cj = A.take(ntree, &cj);
  TreeJob* tj;
  TreeJob* d_tj = A.take(ntree, &tj);
  EncJob<SrcIds2d>* ej_i;
  EncJob<SrcIds2d>* d_ej_i = A.take(nf, &ej_i);
  EncJob<SrcCodes2d>* ej_c;
  EncJob<SrcCodes2d>* d_ej_c = A.take(2 * nf, &ej_c);
  ScanDiff* sd;
  ScanDiff* d_sd = A.take(5 * nf, &sd);
  Layout2d* lj;
  Layout2d* d_lj = A.take(nf, &lj);
  uint32_t hblk = 0, iblk = 0, cblk = 0;
  for (size_t k = 0; k < nf; k++) {
    const C2Work& W = *w[k];
    const G& x = g[k];
    const size_t te = W.t.elems(), nch = te / U16Hist::kChunk;
    for (int c = 0; c < 2; c++) {
      HistJob<U16Hist>& h = hj[2 * k + c];
      h.src = U16Hist{c ? W.qv : W.qu, te, (uint32_t)(te - x.n)};
      h.nchunks = nch;
      h.hist = W.hist + kMaxEbCode + c * 65536;
      // 128 chunks per block: a block clears and flushes its 16384-bin window once per 131072 codes
      h.nblk = (uint32_t)std::min<size_t>(std::max<size_t>(div_up(nch, 128), 1), 512);
      h.blk0 = hblk;
      hblk += h.nblk;
    }
    for (int t = 0; t < 3; t++) {
      const size_t tt = 3 * k + t;
      cj[tt] = CompactJob{W.hist + (t == 0 ? 0 : kMaxEbCode + (t - 1) * 65536), t == 0 ? (uint32_t)kMaxEbCode : 65536u};
      TreeJob& T = tj[tt];
      T = TreeJob{};
      T.syms = d_syms;
      T.freqs = d_freqs;
      T.count = d_count + tt;
      T.base = d_base + tt;
      T.state_num = t == 0 ? 2 * 1024 : 2 * kCapacity;
      T.max_leaves = t == 0 ? kMaxIdLeaves : kMaxCodeLeaves;
      T.heap = t == 0 ? nullptr : t_heap + (2 * k + t - 1) * heap_n;
      T.tree = t_tree + k * tb_field + (t == 0 ? 0 : ((tb_id + 255) & ~(size_t)255) + (t - 1) * ((tb_code + 255) & ~(size_t)255));
      const size_t at = k * HN + (t == 0 ? 0 : kMaxEbCode + (t - 1) * 65536);
      T.code = cb_code + at;
      T.len = cb_len + at;
      T.info = d_info + 4 * tt;
    }
    EncJob<SrcIds2d>& e = ej_i[k];
    e.src = SrcIds2d(W.cu, W.cv, x.n);
    e.nchunks = x.nch_ids;
    e.code = cb_code + k * HN;
    e.len = cb_len + k * HN;
    e.bits = bits + x.cb;
    e.off = offs + x.cb;
    e.words = nullptr;
    e.blk0 = iblk;
    e.zc = nullptr;
    iblk += (uint32_t)encode_blocks(x.nch_ids);
    for (int c = 0; c < 2; c++) {
      EncJob<SrcCodes2d>& f = ej_c[2 * k + c];
      // the chunks' zero counts come with their bit counts; the encoder
      // gathers the unpredictable values (its array comes from k_layout2d)
      f.src = SrcCodes2d(c ? W.qv : W.qu, W.t, W.r1, W.r2, c ? W.dV : W.dU);
      f.src.uoff = zoff + x.zb + c * x.ncc;
      f.zc = zc + x.zb + c * x.ncc;
      f.nchunks = x.ncc;
      f.code = cb_code + k * HN + kMaxEbCode + c * 65536;
      f.len = cb_len + k * HN + kMaxEbCode + c * 65536;
      f.bits = bits + x.cb + x.nch_ids + c * x.ncc;
      f.off = offs + x.cb + x.nch_ids + c * x.ncc;
      f.words = nullptr;
      f.blk0 = cblk;
      cblk += (uint32_t)encode_blocks(x.ncc);
    }
    const size_t c0 = x.cb, c1 = c0 + x.nch_ids, c2 = c1 + x.ncc, c3 = c2 + x.ncc;
    sd[5 * k + 0] = ScanDiff{offs + c0, offs + c1};
    sd[5 * k + 1] = ScanDiff{offs + c1, offs + c2};
    sd[5 * k + 2] = ScanDiff{offs + c2, offs + c3};
    sd[5 * k + 3] = ScanDiff{zoff + x.zb, zoff + x.zb + x.ncc};
    sd[5 * k + 4] = ScanDiff{zoff + x.zb + x.ncc, zoff + x.zb + 2 * x.ncc};
    Layout2d& l = lj[k];
    l = Layout2d{};
    l.off = off[k];
    l.cap = cap[k];
    l.nb = x.nb;
    l.tot = d_tot + 5 * k;
    for (int t = 0; t < 3; t++) {
      l.tinfo[t] = d_info + 4 * (3 * k + t);
      l.tree[t] = tj[3 * k + t].tree;
    }
    l.ej_ids = d_ej_i + k;
    l.ej_codes = d_ej_c + 2 * k;
  }
  ctx.upload_table("b2e.tab", A.d, A.h, A.used);
  // ---- histograms, present symbols, trees
  const uint32_t win_lo = 32768 - 4096, win_n = 8192;
  k_hist_multi<U16Hist><<<hblk, 256, win_n * 4, st>>>(d_hj, (int)(2 * nf), win_lo, win_n);
  CPSZ_HIP(hipGetLastError());
  k_zero_i32<<<1, 64, 0, st>>>((int*)meta, 16);  // total, words used, error flag
  k_compact_hist<<<(unsigned)ntree, 1024, 0, st>>>(d_cj, d_count, d_base, d_total, d_syms, d_freqs);
  CPSZ_HIP(hipGetLastError());
  if (device_trees) {
    ctx.mark("hist");
    build_trees_device(ctx, d_tj, (int)ntree);
  } else {
    // present symbols to the host, trees on the worker pool, results moved to
    // where the device builder would have put them
    CPSZ_REQUIRE(!ctx.capturing, kErrInternal, "batched entropy: host trees cannot be captured");
    const size_t cm = 12 * ntree;
    uint8_t* hc = (uint8_t*)ctx.host_buf("b2e.hcnt", cm + 16 * nf + 64);
    CPSZ_HIP(hipMemcpyAsync(hc, d_total, 8, hipMemcpyDeviceToHost, st));
    CPSZ_HIP(hipMemcpyAsync(hc + 64, d_base, 8 * ntree, hipMemcpyDeviceToHost, st));
    CPSZ_HIP(hipMemcpyAsync(hc + 64 + 8 * ntree, d_count, 4 * ntree, hipMemcpyDeviceToHost, st));
    CPSZ_HIP(hipMemcpyAsync(hc + 64 + cm, w[0]->flags, 16 * nf, hipMemcpyDeviceToHost, st));
    CPSZ_HIP(hipStreamSynchronize(st));
    for (size_t k = 0; k < nf; k++)  // a skipped field's codes are not the codec's: report it before its trees
      CPSZ_REQUIRE(((const int*)(hc + 64 + cm))[4 * k] == 0, kErrNonFinite,
                   "compress_2d: non-finite input or bound (the reference cannot encode it)");
    const uint64_t present = *(const uint64_t*)hc;
    const uint64_t* h_base = (const uint64_t*)(hc + 64);
    const uint32_t* h_count = (const uint32_t*)(hc + 64 + 8 * ntree);
    uint32_t* h_sf = (uint32_t*)ctx.host_buf("b2e.sf", 8 * present + 8);
    CPSZ_HIP(hipMemcpyAsync(h_sf, d_syms, 4 * present, hipMemcpyDeviceToHost, st));
    CPSZ_HIP(hipMemcpyAsync(h_sf + present, d_freqs, 4 * present, hipMemcpyDeviceToHost, st));
    CPSZ_HIP(hipStreamSynchronize(st));
    ctx.mark("hist");
    // kept per calling thread so their storage is reused; the pool threads
    // reach them through a reference (a thread_local named inside a job would
    // be the worker's own)
    thread_local std::vector<HuffEncodeTable> tabs_keep;
    std::vector<HuffEncodeTable>& tabs = tabs_keep;
    if (tabs.size() < ntree) tabs.resize(ntree);
    // the upload table's layout follows from the leaf counts alone, so each
    // worker writes its tree's results straight into it
    auto tree_bytes_of = [](size_t k) {
      const size_t N = 2 * k - 1, w = N <= 256 ? 1 : (N <= 65536 ? 2 : 4);
      return 1 + 2 * N * w + 5 * N;
    };
    size_t tbytes = 0;
    for (size_t t = 0; t < ntree; t++) tbytes += h_count[t] * 13 + tree_bytes_of(h_count[t] ? h_count[t] : 1) + 64;
    Arena B;
    const size_t bbytes = tbytes + ntree * sizeof(HostTreeJob) + 64;
    B.d = ctx.buf<uint8_t>("b2e.tabB", bbytes);
    B.h = (uint8_t*)ctx.host_table("b2e.tabB", bbytes);
    B.cap = bbytes;
    HostTreeJob* hj2;
    HostTreeJob* d_hj2 = B.take(ntree, &hj2);
    std::vector<uint8_t*> hdst(4 * ntree);
    for (size_t t = 0; t < ntree; t++) {
      const size_t kk = h_count[t];
      HostTreeJob& J = hj2[t];
      J.cb.codes = B.take(kk, (uint64_t**)&hdst[4 * t]);
      J.cb.syms = B.take(kk, (uint32_t**)&hdst[4 * t + 1]);
      J.cb.lens = B.take(kk, &hdst[4 * t + 2]);
      J.tree_src = B.take(tree_bytes_of(kk ? kk : 1), &hdst[4 * t + 3]);
      J.cb.k = (uint32_t)kk;
      J.cb.code = tj[t].code;
      J.cb.len = tj[t].len;
      J.tree_dst = tj[t].tree;
      J.info_dst = tj[t].info;
    }
    {
      std::vector<std::function<void(Ctx&)>> jobs(ntree);
      for (size_t t = 0; t < ntree; t++)
        jobs[t] = [&, t](Ctx&) {
          CPSZ_REQUIRE(h_count[t] > 0, kErrInternal, "batched entropy: empty histogram");
          HuffEncodeTable& T = tabs[t];
          huff_build_sparse(h_sf + h_base[t], h_sf + present + h_base[t], h_count[t], tj[t].state_num, T);
          const size_t kk = T.syms.size();
          CPSZ_REQUIRE(kk == h_count[t] && T.tree.size() == tree_bytes_of(kk), kErrInternal,
                       "batched entropy: tree size mismatch");
          std::memcpy(hdst[4 * t], T.codes.data(), 8 * kk);
          std::memcpy(hdst[4 * t + 1], T.syms.data(), 4 * kk);
          std::memcpy(hdst[4 * t + 2], T.lens.data(), kk);
          std::memcpy(hdst[4 * t + 3], T.tree.data(), T.tree.size());
          HostTreeJob& J = hj2[t];
          J.tree_n = T.tree.size();
          J.info[0] = T.node_count;
          J.info[1] = T.tree.size();
          J.info[2] = (uint64_t)T.max_len;
          J.info[3] = 0;
        };
      pool_run(pool_for(ctx.device()), jobs, std::max(workers, 1));
    }
    ctx.upload_table("b2e.tabB", B.d, B.h, B.used);
    k_host_trees_in<<<(unsigned)ntree, 256, 0, st>>>(d_hj2);
    CPSZ_HIP(hipGetLastError());
  }
  ctx.mark("tree");
  // ---- chunk bit counts (and the code chunks' zero counts), one scan for
  // every stream, per-stream totals
  k_run_bits<SrcIds2d><<<iblk, kEncThreads, 0, st>>>(d_ej_i, (int)nf);
  k_run_bits<SrcCodes2d><<<cblk, kEncThreads, 0, st>>>(d_ej_c, (int)(2 * nf));
  CPSZ_HIP(hipGetLastError());
  scan_u64(ctx, bits, offs, CB, offs + CB);
  scan_u32_to_u64(ctx, zc, zoff, Z, zoff + Z);
  k_scan_diffs<<<(unsigned)div_up(5 * nf, 256), 256, 0, st>>>(d_sd, (int)(5 * nf), d_tot);
  CPSZ_HIP(hipGetLastError());
  ctx.mark("scan");
  // ---- layout, encode (with the unpredictable gather), headers, assembly
  k_layout2d<<<1, 64, 0, st>>>(d_lj, (int)nf, words, words_cap, unp, unp_cap, d_sizes, d_words_used, d_err);
  k_fill_words<<<2048, 256, 0, st>>>(words, d_words_used);
  k_run_encode<SrcIds2d><<<iblk, kEncThreads, 0, st>>>(d_ej_i, (int)nf);
  k_run_encode<SrcCodes2d><<<cblk, kEncThreads, 0, st>>>(d_ej_c, (int)(2 * nf));
  CPSZ_HIP(hipGetLastError());
  ctx.mark("encode");
  k_write_heads2d<<<(unsigned)nf, 256, 0, st>>>(d_lj, dout);
  k_assemble2d<<<dim3(64, (unsigned)nf), 256, 0, st>>>(d_lj, dout);
  CPSZ_HIP(hipGetLastError());
  ctx.mark("assemble");
  // ---- tree infos, sizes and error flags back to the host
  const size_t mb = ntree * 32 + nf * 8;
  uint8_t* hm = (uint8_t*)ctx.host_buf("b2e.hmeta", mb + 16 * nf + 64);
  CPSZ_HIP(hipMemcpyAsync(hm, d_info, mb, hipMemcpyDeviceToHost, st));
  CPSZ_HIP(hipMemcpyAsync(hm + mb, d_err, 4, hipMemcpyDeviceToHost, st));
  CPSZ_HIP(hipMemcpyAsync(hm + mb + 64, w[0]->flags, 16 * nf, hipMemcpyDeviceToHost, st));
  if (!ctx.capturing) c2_entropy_batch_finish(ctx, nf, cap, size);
}

void c2_entropy_batch_finish(Ctx& ctx, size_t nf, const std::vector<size_t>& cap, std::vector<size_t>& size) {
  const size_t ntree = 3 * nf, mb = ntree * 32 + nf * 8;
  const uint8_t* hm = (const uint8_t*)ctx.host_buf("b2e.hmeta", mb + 16 * nf + 64);
  CPSZ_HIP(hipStreamSynchronize(ctx.stream()));
  const int* hflags = (const int*)(hm + mb + 64);
  for (size_t k = 0; k < nf; k++)
    CPSZ_REQUIRE(hflags[4 * k] == 0, kErrNonFinite,
                 "compress_2d: non-finite input or bound (the reference cannot encode it)");
  const uint64_t* hinfo = (const uint64_t*)hm;
  const uint64_t* hsizes = hinfo + 4 * ntree;
  for (size_t t = 0; t < ntree; t++) {
    const uint64_t e = hinfo[4 * t + 3];
    CPSZ_REQUIRE(e != 3, kErrUnsupported, "symbol beyond the coder's state count");
    CPSZ_REQUIRE(e == 0, kErrInternal, "device huffman tree failed (code " + std::to_string(e) + ")");
  }
  CPSZ_REQUIRE(*(const int*)(hm + mb) == 0, kErrInternal, "batched entropy: layout pools overflowed");
  for (size_t k = 0; k < nf; k++) {
    CPSZ_REQUIRE(hsizes[k] <= cap[k], kErrInternal, "batch stream bound exceeded");
    size[k] = hsizes[k];
  }
}

void eb_2d_device(Ctx& ctx, const float* dU, const float* dV, size_t r1, size_t r2, double max_pwr_eb,
                  double* dE) {
  CPSZ_REQUIRE(dU && dV && dE && r1 >= 1 && r2 >= 1, kErrArg, "eb_2d: bad arguments");
  C2Work w;
  w.dU = dU;
  w.dV = dV;
  w.r1 = r1;
  w.r2 = r2;
  c2_bind(w, ctx.buf<uint8_t>("c2.scratch", c2_scratch_bytes(r1, r2)));
  EbOverride ov;
  ov.eb_out = dE;
  c2_eb(ctx, w, max_pwr_eb, ov);
}

void compress_2d_device(Ctx& ctx, const float* dU, const float* dV, size_t r1, size_t r2,
                        double max_pwr_eb, DeviceStream& out, const EbOverride& ov) {
  ctx.stages.clear();
  ctx.mark("start");
  C2Work w;
  w.dU = dU;
  w.dV = dV;
  w.r1 = r1;
  w.r2 = r2;
  CPSZ_REQUIRE(r1 >= 1 && r2 >= 1 && r1 < (1u << 30) && r2 < (1u << 30), kErrArg, "compress_2d: bad shape");
  c2_bind(w, ctx.buf<uint8_t>("c2.scratch", c2_scratch_bytes(r1, r2)));
  c2_eb(ctx, w, max_pwr_eb, ov);
  ctx.mark("eb");
  C2Work* wp = &w;
  c2_check(ctx, &wp, 1);
  c2_wavefront(ctx, &wp, 1, 4096);
  ctx.mark("lorenzo");
  c2_entropy(ctx, w, out);
  ctx.finish_marks();
}

void compress_2d_log_device(Ctx& ctx, const float* dU, const float* dV, size_t r1, size_t r2,
                            double max_pwr_eb, DeviceStream& out) {
  ctx.stages.clear();
  ctx.mark("start");
  CPSZ_REQUIRE(dU && dV && r1 >= 1 && r2 >= 1 && r1 < (1u << 30) && r2 < (1u << 30), kErrArg,
               "compress_2d_log: bad arguments");
  hipStream_t st = ctx.stream();
  C2Work w;
  w.dU = dU;
  w.dV = dV;
  w.r1 = r1;
  w.r2 = r2;
  w.log = true;
  const size_t n = r1 * r2, nq = div_up(n, 64);
  c2_bind(w, ctx.buf<uint8_t>("c2.scratch", c2_scratch_bytes(r1, r2)));
  float* L = ctx.buf<float>("c2l.log", 2 * n);
  uint64_t* sm = ctx.buf<uint64_t>("c2l.smap", 2 * nq);
  w.lu = L;
  w.lv = L + n;
  w.smap = sm;
  c2_eb(ctx, w, max_pwr_eb, EbOverride());
  k_log2d<<<dim3((unsigned)div_up(nq, 4), 2), 256, 0, st>>>(dU, dV, n, nq, ctx.libm_dev().log2f, L, L + n, sm);
  CPSZ_HIP(hipGetLastError());
  ctx.mark("eb");
  C2Work* wp = &w;
  c2_check(ctx, &wp, 1);
  c2_wavefront(ctx, &wp, 1, 4096);
  ctx.mark("lorenzo");
  c2_entropy(ctx, w, out);
  ctx.finish_marks();
}

namespace {
// Reads stream bytes either from a host copy or from device memory.
struct HuffSection {
  size_t node_count;
  uint32_t tree_size;
  std::vector<uint8_t> tree;
  size_t nbytes;
  size_t bits_off;  // absolute offset of the bitstream
  size_t end;
};

HuffSection parse_huff(StreamReader& r, size_t off) {
  HuffSection h;
  h.node_count = r.get<size_t>(off);
  h.tree_size = r.get<uint32_t>(off + 8);
  CPSZ_REQUIRE(h.node_count >= 1 && h.node_count < (1u << 24), kErrStream, "bad huffman node count");
  const uint8_t* t = r.read(off + 12, h.tree_size);
  h.tree.assign(t, t + h.tree_size);
  h.nbytes = r.get<size_t>(off + 12 + h.tree_size);
  h.bits_off = off + 20 + h.tree_size;
  CPSZ_REQUIRE(h.nbytes <= r.size && h.bits_off + h.nbytes <= r.size, kErrStream,
               "huffman bitstream truncated");
  h.end = h.bits_off + h.nbytes;
  return h;
}

// The header fields and section positions of a 2D stream.
struct D2Plan {
  HuffSection h_eb;
  struct Comp {
    size_t off = 0, unp_count = 0, unp_off = 0;
    HuffSection h;
  } comp[2];
  int nby = 0;
  size_t nb = 0;
  size_t sign_off = 0;  // offline_log: the two sign bitmaps
};

// log: the offline_log layout (base 2, the sign bitmaps between the id
// section and the u section, src/sz_decompress_cp_preserve_2d.cpp:60-79).
void d2_parse(StreamReader& rd, size_t r1, size_t r2, D2Plan& p, bool log = false, size_t vb = 4) {
  const size_t n = r1 * r2;
  const int base = rd.get<int>(0);
  const double thr = rd.get<double>(4);
  const size_t u_size = rd.get<size_t>(20);
  CPSZ_REQUIRE(base == (log ? 2 : 4) && thr == DBL_EPSILON, kErrUnsupported,
               log ? "decompress_2d_log: stream base/threshold differ from the offline_log 2D format"
                   : "decompress_2d: stream base/threshold differ from the offline 2D format");
  p.h_eb = parse_huff(rd, 36);
  // components follow the id section (and the sign bitmaps) directly; the u
  // section spans u_size bytes
  p.nby = (int)div_up(r2, kBlock2d);
  p.nb = div_up(r1, kBlock2d) * p.nby;
  size_t off = p.h_eb.end;
  if (log) {
    const size_t smap = (n - 1) / 8 + 1;
    p.sign_off = off;
    rd.read(off, 2 * smap);  // bounds check
    off += 2 * smap;
  }
  for (int c = 0; c < 2; c++) {
    D2Plan::Comp& k = p.comp[c];
    k.off = off;
    const int bs = rd.get<int>(off);
    const int radius = rd.get<int>(off + 5);
    // meanInfo<T> is 2 * sizeof(T) bytes: bool, padding, T mean
    const uint8_t use_mean = rd.get<uint8_t>(off + 9);
    const size_t reg = rd.get<size_t>(off + 9 + 2 * vb);
    k.unp_count = rd.get<size_t>(off + 17 + 2 * vb);
    CPSZ_REQUIRE(bs == kBlock2d && radius == kRadius && use_mean == 0 && reg == 0, kErrUnsupported,
                 "decompress_2d: stream uses block settings the offline compressor never writes");
    CPSZ_REQUIRE(k.unp_count <= n, kErrStream, "bad unpredictable count");
    k.unp_off = off + 25 + 2 * vb;
    const size_t ind = k.unp_off + vb * k.unp_count;
    const size_t ind_bytes = (p.nb - 1) / 8 + 1;
    const uint8_t* ib = rd.read(ind, ind_bytes);
    for (size_t b = 0; b < ind_bytes; b++)
      CPSZ_REQUIRE(ib[b] == 0, kErrUnsupported, "regression blocks are not produced by the 2D codec");
    k.h = parse_huff(rd, ind + ind_bytes);
    off = c == 0 ? off + u_size : k.h.end;
  }
}

// Largest symbol of a parsed tree (ids above 81 need the wide wavefront path).
uint32_t max_symbol(const HuffDecodeTree& t) {
  uint32_t m = 0;
  for (size_t i = 0; i < t.node_count; i++)
    if ((t.leaf[i] || (i == 0 && t.root_leaf)) && t.sym[i] > m) m = t.sym[i];
  return m;
}

// Unpredictable values to per-element raw arrays (block-major order).
void d2_unpred(Ctx& ctx, const uint8_t* d_in, const D2Plan& p, D2Work& w) {
  hipStream_t st = ctx.stream();
  const size_t r1 = w.r1, r2 = w.r2, n = r1 * r2, nb = p.nb;
  uint32_t* zc = ctx.buf<uint32_t>("d2.zc", 2 * nb);
  uint64_t* zoff = ctx.buf<uint64_t>("d2.zoff", 2 * nb + 4);
  CPSZ_HIP(hipMemsetAsync(w.err, 0, 8, st));
  uint16_t* qs[2] = {w.qu, w.qv};
  const size_t vb = w.f64 ? 8 : 4;
  for (int c = 0; c < 2; c++) {
    uint8_t* vals = ctx.buf<uint8_t>(c ? "d2.unpv" : "d2.unpu", vb * (p.comp[c].unp_count + 1));
    if (p.comp[c].unp_count)
      CPSZ_HIP(hipMemcpyAsync(vals, d_in + p.comp[c].unp_off, vb * p.comp[c].unp_count, hipMemcpyDeviceToDevice,
                              st));
    k_block_zeros<<<unp_grid(nb), 256, 0, st>>>(qs[c], w.t, (int)r1, (int)r2, p.nby, nb, zc + c * nb);
    scan_u32_to_u64(ctx, zc + c * nb, zoff + c * (nb + 1), nb, zoff + c * (nb + 1) + nb);
    if (w.f64)
      k_scatter_unpred<double><<<unp_grid(nb), 256, 0, st>>>(qs[c], w.t, (const double*)vals, (int)r1, (int)r2, p.nby,
                                                             nb, zoff + c * (nb + 1), p.comp[c].unp_count,
                                                             (double*)w.raw + c * w.t.elems(), w.err);
    else
      k_scatter_unpred<float><<<unp_grid(nb), 256, 0, st>>>(qs[c], w.t, (const float*)vals, (int)r1, (int)r2, p.nby, nb,
                                                            zoff + c * (nb + 1), p.comp[c].unp_count,
                                                            w.raw + c * w.t.elems(), w.err);
    CPSZ_HIP(hipGetLastError());
  }
}

}  // namespace

size_t d2_scratch_bytes(size_t r1, size_t r2, bool f64) {
  // (the kernels' rows, columns and steps are ints)
  CPSZ_REQUIRE(r1 < kMaxSide2d && r2 < kMaxSide2d && r1 * r2 < (1ull << 40), kErrUnsupported,
               "decompress_2d: field too large");
  const size_t te = Tile2d(r1, r2).elems();
  return 4 * al256(2 * te) + al256((f64 ? 16 : 8) * te) + al256(8 * bnd_words(r1, r2)) + al256(4) + al256(16);
}

void d2_bind(D2Work& w, uint8_t* p) {
  w.t = Tile2d(w.r1, w.r2);
  const size_t te = w.t.elems();
  auto take = [&](size_t bytes) {
    uint8_t* q = p;
    p += al256(bytes);
    return q;
  };
  w.sid_u = (uint16_t*)take(2 * te);
  w.sid_v = (uint16_t*)take(2 * te);
  w.qu = (uint16_t*)take(2 * te);
  w.qv = (uint16_t*)take(2 * te);
  w.raw = (float*)take((w.f64 ? 16 : 8) * te);  // T = double: doubles
  w.bnd = (uint64_t*)take(8 * bnd_words(w.r1, w.r2));
  w.ticket = (int*)take(4);
  w.err = (int*)take(16);
}

void d2_entropy(Ctx& ctx, const uint8_t* d_in, const uint8_t* h_in, size_t in_size, D2Work& w) {
  CPSZ_REQUIRE(d_in && w.r1 >= 1 && w.r2 >= 1, kErrArg, "decompress_2d: bad arguments");
  hipStream_t st = ctx.stream();
  const size_t r1 = w.r1, r2 = w.r2, n = r1 * r2;
  uint16_t *sid_u = w.sid_u, *sid_v = w.sid_v, *qu = w.qu, *qv = w.qv;
  const bool log = w.log;
  const Tile2d tile = w.t;
  StreamReader rd(ctx, h_in, d_in, in_size);
  D2Plan p;
  d2_parse(rd, r1, r2, p, w.log, w.f64 ? 8 : 4);
  if (w.log) w.signs = d_in + p.sign_off;
  const HuffSection& h_eb = p.h_eb;
  const int nby = p.nby;
  ctx.mark("parse");
  // ---- bitstreams into aligned scratch
  BitsCopy bc[3] = {{d_in + h_eb.bits_off, h_eb.nbytes, nullptr, 0},
                    {d_in + p.comp[0].h.bits_off, p.comp[0].h.nbytes, nullptr, 0},
                    {d_in + p.comp[1].h.bits_off, p.comp[1].h.nbytes, nullptr, 0}};
  // The code trees are parsed and tabulated while the device decodes the id
  // stream (the u tree on the helper thread, the v tree on this one after
  // queuing the id decode); then the u and v streams decode together, and the
  // host looks at what all three held. The tables are kept per calling thread (their storage is
  // reused); the helper fills them through the pointer (a thread_local named
  // in the job would be the helper thread's own).
  thread_local HostDecoder hc_keep[2];
  HostDecoder* hc = hc_keep;
  auto prep = [&](int c) {
    prepare_decoder(p.comp[c].h.tree.data(), p.comp[c].h.tree.size(), p.comp[c].h.node_count, hc[c]);
  };
  uint32_t id_max = 0;
  {
    HuffDecodeTree t;
    CPSZ_REQUIRE(huff_parse_tree(h_eb.tree.data(), h_eb.tree.size(), h_eb.node_count, t), kErrStream,
                 "malformed id tree");
    id_max = max_symbol(t);
  }
  DecodeResult ids;
  const SettleOnThrow settle{st};
  {
    HelperJob u_ready([&] { prep(0); }, !ctx.batch_worker);
    stage_bits_multi(ctx, bc, 3, "d2.bits");
    DeviceDecoder dd = upload_decoder(ctx, h_eb.tree.data(), h_eb.tree.size(), h_eb.node_count, "d2.eb");
    if (id_max < 256)
      ids = decode_stream(ctx, dd, bc[0].dst, h_eb.nbytes, log ? n : 2 * n, SinkIds2dB{sid_u, sid_v, n, tile}, "d2.eb");
    else
      ids = decode_stream(ctx, dd, bc[0].dst, h_eb.nbytes, log ? n : 2 * n, SinkIds2d{sid_u, sid_v, n, tile}, "d2.eb");
    prep(1);
    u_ready.join();  // rethrows a malformed code tree
  }
  const DeviceDecoder du = upload_decoder(ctx, hc[0], "d2.u");
  const DeviceDecoder dv = upload_decoder(ctx, hc[1], "d2.v");
  const DecJob<SinkCodes2d> jobs[2] = {
      {&du, bc[1].dst, p.comp[0].h.nbytes, n, SinkCodes2d{qu, tile, (int)r1, (int)r2, nby}},
      {&dv, bc[2].dst, p.comp[1].h.nbytes, n, SinkCodes2d{qv, tile, (int)r1, (int)r2, nby}}};
  const DecodeResult codes = decode_streams(ctx, jobs, 2, "d2.codes");
  CPSZ_HIP(hipStreamSynchronize(st));
  ids.check();
  codes.check();
  ctx.mark("huffman");
  d2_unpred(ctx, d_in, p, w);
  w.wide = id_max > 81;
  ctx.mark("unpred");
}

// Unpredictable values of every field of a batch (float): the stream's
// values copied to aligned arrays in one assembly launch, the per-block zero
// counts of every component, one global scan, one scatter launch.
void d2_unpred_batch(Ctx& ctx, const std::vector<const uint8_t*>& d_in, const std::vector<D2Plan>& plan,
                     D2Work* const* w, size_t nf, const uint64_t* zmask) {
  hipStream_t st = ctx.stream();
  size_t Z = 0, V = 0, npieces = 0;
  constexpr size_t kPiece = 65536;
  std::vector<size_t> zb(nf), vb(2 * nf);
  for (size_t k = 0; k < nf; k++) {
    CPSZ_REQUIRE(!w[k]->f64 && !w[k]->log, kErrInternal, "batched unpredictable scatter: plain float fields only");
    zb[k] = Z;
    Z += 2 * plan[k].nb;
    for (int c = 0; c < 2; c++) {
      vb[2 * k + c] = V;
      V += (plan[k].comp[c].unp_count + 63) & ~(size_t)63;
      npieces += div_up(4 * plan[k].comp[c].unp_count, kPiece);
    }
  }
  uint32_t* zc = ctx.buf<uint32_t>("b2u.zc", Z + 1);
  uint64_t* zoff = ctx.buf<uint64_t>("b2u.zoff", Z + 1);
  float* vals = ctx.buf<float>("b2u.vals", V + 1);
  int* errs = ctx.buf<int>("b2u.err", 4 * nf);
  Arena A;
  const size_t bytes = 2 * nf * sizeof(UnpJob) + npieces * sizeof(CopyPiece) + 64;
  A.h = (uint8_t*)ctx.host_buf("b2u.tab", bytes);
  A.d = ctx.buf<uint8_t>("b2u.tab", bytes);
  A.cap = bytes;
  UnpJob* uj;
  UnpJob* d_uj = A.take(2 * nf, &uj);
  CopyPiece* cp;
  CopyPiece* d_cp = A.take(npieces, &cp);
  size_t np = 0;
  uint32_t blk = 0;
  for (size_t k = 0; k < nf; k++) {
    const D2Plan& p = plan[k];
    D2Work& W = *w[k];
    W.err = errs + 4 * k;
    for (int c = 0; c < 2; c++) {
      UnpJob& u = uj[2 * k + c];
      u = UnpJob{};
      u.t = W.t;
      u.x = vals + vb[2 * k + c];
      u.r1 = (int)W.r1;
      u.r2 = (int)W.r2;
      u.nby = p.nby;
      u.nb = p.nb;
      u.off = zoff + zb[k] + c * p.nb;
      u.out = W.raw + c * W.t.elems();
      u.count = p.comp[c].unp_count;
      u.err = W.err;
      u.blk0 = blk;
      u.zm = zmask + 3 * (zb[k] + c * p.nb);
      blk += unp_blocks(p.nb);
      const size_t len = 4 * p.comp[c].unp_count;
      for (size_t o = 0; o < len; o += kPiece)
        cp[np++] = CopyPiece{4 * vb[2 * k + c] + o, d_in[k] + p.comp[c].unp_off + o,
                             (uint32_t)std::min(kPiece, len - o), 0};
    }
  }
  CPSZ_HIP(hipMemcpyAsync(A.d, A.h, A.used, hipMemcpyHostToDevice, st));
  k_fill_u32<<<1, 256, 0, st>>>((uint32_t*)errs, 4 * nf, 0);
  if (np) k_assemble<<<(unsigned)np, 256, 0, st>>>(d_cp, (uint8_t*)vals);
  CPSZ_HIP(hipGetLastError());
  scan_u32_to_u64(ctx, zc, zoff, Z, zoff + Z);
  k_scatter_unpred_multi<<<blk, 256, 0, st>>>(d_uj, (int)(2 * nf));
  CPSZ_HIP(hipGetLastError());
  // the pinned table is reused by the next call only after the stream passes here
  CPSZ_HIP(hipStreamSynchronize(st));
}

// Batched form: every field's headers parsed and trees tabulated on the
// workers; all decoders uploaded in one copy and all bitstreams staged in one
// launch; the id streams of every field decoded together, then the u and v
// streams of every field together (one grid per pass, one look at the results);
// one unpredictable scatter.
void d2_entropy_batch(Ctx& ctx, const std::vector<const uint8_t*>& d_in, const std::vector<size_t>& in_size,
                      D2Work* const* w, size_t nf, int workers) {
  hipStream_t st = ctx.stream();
  std::vector<D2Plan> plan(nf);
  std::vector<HostDecoder> hd(3 * nf);
  // Every stream's header pieces come to the host in four batched rounds (a
  // gather of the pieces on the device, one copy, one wait each): the start of
  // the stream (header, id tree), the u and v section heads, their indicator
  // bytes and tree heads, then their trees. The offsets follow the layout
  // d2_parse reads; a piece outside what was fetched is read from the device
  // by the parser itself.
  for (size_t k = 0; k < nf; k++)
    CPSZ_REQUIRE(d_in[k] && w[k]->r1 >= 1 && w[k]->r2 >= 1, kErrArg, "decompress_2d: bad arguments");
  std::vector<std::vector<StreamReader::Range>> pre(nf);
  {
    struct Want {
      size_t k, off, len;
    };
    // one round: gathers the wanted pieces into a device staging buffer, copies
    // it to pinned host memory and records the ranges; returns their host copies
    int round = 0;
    auto fetch = [&](const std::vector<Want>& want) {
      std::vector<const uint8_t*> where(want.size(), nullptr);
      size_t total = 0, npc = 0;
      for (const Want& x : want) {
        total += (x.len + 15) & ~(size_t)15;
        npc += div_up(x.len, (size_t)65536);
      }
      if (!total) return where;
      const std::string tag = "b2d.pre" + std::to_string(round++);
      uint8_t* dst = ctx.buf<uint8_t>(tag.c_str(), total);
      uint8_t* hst = (uint8_t*)ctx.host_buf(tag.c_str(), total);
      CopyPiece* hp = (CopyPiece*)ctx.host_table((tag + "t").c_str(), npc * sizeof(CopyPiece));
      CopyPiece* dp = ctx.buf<CopyPiece>((tag + "t").c_str(), npc);
      size_t at = 0, np = 0;
      for (size_t i = 0; i < want.size(); i++) {
        const Want& x = want[i];
        for (size_t o = 0; o < x.len; o += 65536)
          hp[np++] = CopyPiece{at + o, d_in[x.k] + x.off + o, (uint32_t)std::min<size_t>(65536, x.len - o), 0};
        where[i] = hst + at;
        pre[x.k].push_back({x.off, x.len, hst + at});
        at += (x.len + 15) & ~(size_t)15;
      }
      ctx.upload_table((tag + "t").c_str(), dp, hp, np * sizeof(CopyPiece));
      k_assemble<<<(unsigned)np, 256, 0, st>>>(dp, dst);
      CPSZ_HIP(hipGetLastError());
      CPSZ_HIP(hipMemcpyAsync(hst, dst, at, hipMemcpyDeviceToHost, st));
      CPSZ_HIP(hipStreamSynchronize(st));
      return where;
    };
    constexpr size_t kStart = 32u << 10;  // header + id tree (at most 1024 leaves: < 27 KiB)
    std::vector<Want> w1(nf);
    for (size_t k = 0; k < nf; k++) w1[k] = {k, 0, std::min(kStart, in_size[k])};
    const std::vector<const uint8_t*> h1 = fetch(w1);
    // section starts: u after the id section, v u_size bytes later
    std::vector<Want> w2;
    for (size_t k = 0; k < nf; k++) {
      const uint8_t* h = h1[k];
      if (!h || w1[k].len < 48) continue;
      uint64_t u_size, nbytes;
      uint32_t tsz;
      std::memcpy(&u_size, h + 20, 8);
      std::memcpy(&tsz, h + 44, 4);
      if ((uint64_t)48 + tsz + 8 > w1[k].len) continue;
      std::memcpy(&nbytes, h + 48 + tsz, 8);
      const uint64_t u0 = 56 + (uint64_t)tsz + nbytes;
      if (nbytes > in_size[k] || u0 > in_size[k]) continue;
      // section head: block size, radius, meanInfo, regression count, then
      // the unpredictable count (at +25) and values (from +33)
      if (in_size[k] - u0 >= 33) {
        w2.push_back({k, u0, 33});
      }
      if (u_size <= in_size[k] - u0 && in_size[k] - u0 - u_size >= 33) {
        w2.push_back({k, u0 + u_size, 33});
      }
    }
    const std::vector<const uint8_t*> h2 = fetch(w2);
    std::vector<Want> w3;
    for (size_t i = 0; i < w2.size(); i++) {
      const size_t k = w2[i].k;
      uint64_t unp;
      std::memcpy(&unp, h2[i] + 25, 8);
      const size_t nb = div_up(w[k]->r1, kBlock2d) * div_up(w[k]->r2, kBlock2d);
      const uint64_t ind = w2[i].off + 33 + 4 * (uint64_t)std::min<uint64_t>(unp, w[k]->r1 * w[k]->r2);
      const uint64_t len = (nb - 1) / 8 + 1 + 12;  // indicator bytes, tree head
      if (ind > in_size[k] || len > in_size[k] - ind) continue;
      w3.push_back({k, ind, len});
    }
    const std::vector<const uint8_t*> h3 = fetch(w3);
    std::vector<Want> w4;
    for (size_t i = 0; i < w3.size(); i++) {
      const size_t k = w3[i].k;
      uint32_t tsz;
      std::memcpy(&tsz, h3[i] + w3[i].len - 4, 4);
      const uint64_t t0 = w3[i].off + w3[i].len;
      if ((uint64_t)tsz + 8 > in_size[k] - t0) continue;
      w4.push_back({k, t0, (size_t)tsz + 8});  // tree and bitstream size
    }
    fetch(w4);
  }
  {
    std::vector<std::function<void(Ctx&)>> jobs(nf);
    for (size_t k = 0; k < nf; k++)
      jobs[k] = [&, k](Ctx& wc) {
        StreamReader rd(wc, nullptr, d_in[k], in_size[k]);
        rd.pre = pre[k];
        d2_parse(rd, w[k]->r1, w[k]->r2, plan[k]);
        const D2Plan& p = plan[k];
        prepare_decoder(p.h_eb.tree.data(), p.h_eb.tree.size(), p.h_eb.node_count, hd[3 * k]);
        for (int c = 0; c < 2; c++)
          prepare_decoder(p.comp[c].h.tree.data(), p.comp[c].h.tree.size(), p.comp[c].h.node_count,
                          hd[3 * k + 1 + c]);
        w[k]->wide = max_symbol(hd[3 * k].d) > 81;
      };
    pool_run(pool_for(ctx.device()), jobs, workers);
  }
  ctx.mark("parse");
  std::vector<const HostDecoder*> hp(3 * nf);
  for (size_t k = 0; k < 3 * nf; k++) hp[k] = &hd[k];
  std::vector<DeviceDecoder> dd(3 * nf);
  upload_decoders(ctx, hp.data(), (int)(3 * nf), dd.data(), "b2d.dec", &pool_for(ctx.device()), workers);
  ctx.mark("upload");
  std::vector<BitsCopy> bc(3 * nf);
  for (size_t k = 0; k < nf; k++) {
    const D2Plan& p = plan[k];
    bc[3 * k] = BitsCopy{d_in[k] + p.h_eb.bits_off, p.h_eb.nbytes, nullptr, 0};
    for (int c = 0; c < 2; c++)
      bc[3 * k + 1 + c] = BitsCopy{d_in[k] + p.comp[c].h.bits_off, p.comp[c].h.nbytes, nullptr, 0};
  }
  stage_bits_multi(ctx, bc.data(), (int)(3 * nf), "b2d.bits");
  ctx.mark("stage");
  std::vector<DecJob<SinkIds2d>> ji(nf);
  std::vector<DecJob<SinkIds2dB>> ji8(nf);
  std::vector<DecJob<SinkCodes2d>> jc(2 * nf);
  // the code decoders count each 12x12 block's zero codes as they write them
  // (the unpredictable scatter's offsets), in the array d2_unpred_batch scans
  size_t Z = 0;
  for (size_t k = 0; k < nf; k++) Z += 2 * plan[k].nb;
  uint32_t* zc = ctx.buf<uint32_t>("b2u.zc", Z + 1);
  k_fill_u32<<<(unsigned)std::min<size_t>(div_up(Z, 256), 2048), 256, 0, st>>>(zc, Z, 0);
  // and record where the zeros are, so that the scatter reads 24 bytes of masks per
  // block instead of the block's codes
  uint64_t* zm = ctx.buf<uint64_t>("b2u.zm", 3 * Z + 1);
  k_fill_u32<<<(unsigned)std::min<size_t>(div_up(6 * Z, 256), 2048), 256, 0, st>>>((uint32_t*)zm, 6 * Z, 0);
  CPSZ_HIP(hipGetLastError());
  size_t zb = 0;
  bool ids8 = true;
  for (size_t k = 0; k < nf; k++) ids8 = ids8 && max_symbol(hd[3 * k].d) < 256;
  for (size_t k = 0; k < nf; k++) {
    const size_t r1 = w[k]->r1, r2 = w[k]->r2, n = r1 * r2;
    const D2Plan& p = plan[k];
    ji[k] = {&dd[3 * k], bc[3 * k].dst, p.h_eb.nbytes, 2 * n, SinkIds2d{w[k]->sid_u, w[k]->sid_v, n, w[k]->t}};
    ji8[k] = {&dd[3 * k], bc[3 * k].dst, p.h_eb.nbytes, 2 * n, SinkIds2dB{w[k]->sid_u, w[k]->sid_v, n, w[k]->t}};
    uint16_t* qs[2] = {w[k]->qu, w[k]->qv};
    for (int c = 0; c < 2; c++)
      jc[2 * k + c] = {&dd[3 * k + 1 + c], bc[3 * k + 1 + c].dst, p.comp[c].h.nbytes, n,
                       SinkCodes2d{qs[c], w[k]->t, (int)r1, (int)r2, p.nby, zc + zb + c * p.nb, zm + 3 * (zb + c * p.nb)}};
    zb += 2 * p.nb;
  }
  const SettleOnThrow settle{st};
  const DecodeResult ids = ids8 ? decode_streams(ctx, ji8.data(), (int)nf, "b2d.ids")
                                : decode_streams(ctx, ji.data(), (int)nf, "b2d.ids");
  const DecodeResult codes = decode_streams(ctx, jc.data(), (int)(2 * nf), "b2d.codes");
  CPSZ_HIP(hipStreamSynchronize(st));
  ids.check();
  codes.check();
  ctx.mark("huffman");
  d2_unpred_batch(ctx, d_in, plan, w, nf, zm);
  ctx.mark("unpred");
}

void d2_wavefront(Ctx& ctx, D2Work* const* w, size_t nf, int grid_cap) {
  if (nf == 1 && w[0]->f64) {
    const size_t n = w[0]->t.elems();
    Strip2d64 sa{};
    sa.c[0] = w[0]->sid_u;
    sa.c[1] = w[0]->sid_v;
    sa.q[0] = w[0]->qu;
    sa.q[1] = w[0]->qv;
    sa.raw[0] = (const double*)w[0]->raw;
    sa.raw[1] = (const double*)w[0]->raw + n;
    sa.out[0] = w[0]->dU64;
    sa.out[1] = w[0]->dV64;
    sa.bnd = w[0]->bnd;
    sa.ticket = w[0]->ticket;
    sa.r1 = (int)w[0]->r1;
    sa.r2 = (int)w[0]->r2;
    sa.ngroups = strip_groups<double>(w[0]->r1);
    sa.t = w[0]->t;
    sa.shift = 2;
    wavefront2d_decompress64(ctx, sa, grid_cap);
    return;
  }
  for (size_t k = 0; k < nf; k++)
    CPSZ_REQUIRE(!w[k]->f64, kErrUnsupported, "decompress_2d: double fields go one at a time");
  std::vector<Strip2d> f(nf);
  for (size_t k = 0; k < nf; k++) {
    Strip2d& sa = f[k];
    sa = Strip2d{};
    const size_t n = w[k]->t.elems();
    sa.c[0] = w[k]->sid_u;
    sa.c[1] = w[k]->log ? w[k]->sid_u : w[k]->sid_v;
    sa.shift = w[k]->log ? 1 : 2;
    sa.q[0] = w[k]->qu;
    sa.q[1] = w[k]->qv;
    sa.raw[0] = w[k]->raw;
    sa.raw[1] = w[k]->raw + n;
    sa.out[0] = w[k]->dU;
    sa.out[1] = w[k]->dV;
    sa.ngroups = strip_groups<float>(w[k]->r1);
    sa.bnd = w[k]->bnd;
    sa.ticket = w[k]->ticket;
    sa.r1 = (int)w[k]->r1;
    sa.r2 = (int)w[k]->r2;
    sa.t = w[k]->t;
    sa.wide = w[k]->wide;
    CPSZ_REQUIRE(!(w[k]->log && sa.wide), kErrStream, "decompress_2d_log: eb id beyond the base-2 range");
  }
  wavefront2d_decompress(ctx, f, grid_cap);
}

void d2_check(Ctx& ctx, D2Work* const* w, size_t nf) {
  hipStream_t st = ctx.stream();
  int* he = (int*)ctx.host_buf("d2.herr", std::max<size_t>(nf, 1) * 16);
  for (size_t k = 0; k < nf; k++) CPSZ_HIP(hipMemcpyAsync(he + 4 * k, w[k]->err, 8, hipMemcpyDeviceToHost, st));
  CPSZ_HIP(hipStreamSynchronize(st));
  for (size_t k = 0; k < nf; k++)
    CPSZ_REQUIRE(he[4 * k] == 0, kErrStream, "decompress_2d: more unpredictable codes than values");
}

void decompress_2d_device(Ctx& ctx, const uint8_t* d_in, const uint8_t* h_in, size_t in_size,
                          size_t r1, size_t r2, float* dU, float* dV) {
  CPSZ_REQUIRE(d_in && dU && dV && r1 >= 1 && r2 >= 1, kErrArg, "decompress_2d: bad arguments");
  ctx.stages.clear();
  ctx.mark("start");
  D2Work w;
  w.r1 = r1;
  w.r2 = r2;
  w.dU = dU;
  w.dV = dV;
  d2_bind(w, ctx.buf<uint8_t>("d2.scratch", d2_scratch_bytes(r1, r2)));
  CPSZ_HIP(hipMemsetAsync(w.err, 0, 16, ctx.stream()));
  d2_entropy(ctx, d_in, h_in, in_size, w);
  D2Work* wp = &w;
  d2_wavefront(ctx, &wp, 1, 4096);
  ctx.mark("lorenzo");
  d2_check(ctx, &wp, 1);
  ctx.finish_marks();
}

void decompress_2d_log_device(Ctx& ctx, const uint8_t* d_in, const uint8_t* h_in, size_t in_size, size_t r1,
                              size_t r2, float* dU, float* dV) {
  CPSZ_REQUIRE(d_in && dU && dV && r1 >= 1 && r2 >= 1, kErrArg, "decompress_2d_log: bad arguments");
  ctx.stages.clear();
  ctx.mark("start");
  D2Work w;
  w.r1 = r1;
  w.r2 = r2;
  w.dU = dU;
  w.dV = dV;
  w.log = true;
  d2_bind(w, ctx.buf<uint8_t>("d2.scratch", d2_scratch_bytes(r1, r2)));
  CPSZ_HIP(hipMemsetAsync(w.err, 0, 16, ctx.stream()));
  d2_entropy(ctx, d_in, h_in, in_size, w);
  D2Work* wp = &w;
  d2_wavefront(ctx, &wp, 1, 4096);
  ctx.mark("lorenzo");
  const size_t n = r1 * r2;
  k_finish2d<<<dim3((unsigned)div_up(n, 256), 2), 256, 0, ctx.stream()>>>(dU, dV, n, w.signs, (n - 1) / 8 + 1,
                                                                         ctx.libm_dev().exp2f);
  CPSZ_HIP(hipGetLastError());
  ctx.mark("finish");
  d2_check(ctx, &wp, 1);
  ctx.finish_marks();
}

void compress_2d_f64_device(Ctx& ctx, const double* dU, const double* dV, size_t r1, size_t r2,
                            double max_pwr_eb, DeviceStream& out) {
  ctx.stages.clear();
  ctx.mark("start");
  CPSZ_REQUIRE(dU && dV && r1 >= 1 && r2 >= 1 && r1 < (1u << 30) && r2 < (1u << 30), kErrArg,
               "compress_2d (double): bad arguments");
  C2Work w;
  w.f64 = true;
  w.dU64 = dU;
  w.dV64 = dV;
  w.r1 = r1;
  w.r2 = r2;
  c2_bind(w, ctx.buf<uint8_t>("c2.scratch", c2_scratch_bytes(r1, r2)));
  c2_eb(ctx, w, max_pwr_eb, EbOverride());
  ctx.mark("eb");
  C2Work* wp = &w;
  c2_check(ctx, &wp, 1);
  c2_wavefront(ctx, &wp, 1, 4096);
  ctx.mark("lorenzo");
  c2_entropy(ctx, w, out);
  ctx.finish_marks();
}

void decompress_2d_f64_device(Ctx& ctx, const uint8_t* d_in, const uint8_t* h_in, size_t in_size, size_t r1,
                              size_t r2, double* dU, double* dV) {
  CPSZ_REQUIRE(d_in && dU && dV && r1 >= 1 && r2 >= 1, kErrArg, "decompress_2d (double): bad arguments");
  ctx.stages.clear();
  ctx.mark("start");
  D2Work w;
  w.r1 = r1;
  w.r2 = r2;
  w.f64 = true;
  w.dU64 = dU;
  w.dV64 = dV;
  d2_bind(w, ctx.buf<uint8_t>("d2.scratch", d2_scratch_bytes(r1, r2, true)));
  CPSZ_HIP(hipMemsetAsync(w.err, 0, 16, ctx.stream()));
  d2_entropy(ctx, d_in, h_in, in_size, w);
  D2Work* wp = &w;
  d2_wavefront(ctx, &wp, 1, 4096);
  ctx.mark("lorenzo");
  d2_check(ctx, &wp, 1);
  ctx.finish_marks();
}

// Host emulation of the wavefront kernels' arithmetic (row-major order; any
// order that respects the Lorenzo dependencies yields the same values).
void lorenzo2d_emulate(const float* x, const uint16_t* c, size_t r1, size_t r2, bool wide,
                       uint16_t* q, float* recon) {
  std::vector<float> R((r1 + 1) * (r2 + 1), 0.f);
  const size_t W = r2 + 1;
  for (size_t i = 0; i < r1; i++)
    for (size_t j = 0; j < r2; j++) {
      float* rp = &R[(i + 1) * W + j + 1];
      const float pred = (rp[-1] + rp[-(ptrdiff_t)W]) - rp[-(ptrdiff_t)W - 1];
      float qs;
      const size_t e = i * r2 + j;
      *rp = wide ? l2d_quantize_wide(pred, x[e], c[e], qs) : l2d_quantize(pred, x[e], l2d_prep(c[e], 2), qs);
      q[e] = l2d_code(qs);
      if (recon) recon[e] = *rp;
    }
}

void lorenzo2d_emulate_decode(const uint16_t* q, const uint16_t* sid, const float* raw, size_t r1,
                              size_t r2, bool wide, float* out) {
  std::vector<float> R((r1 + 1) * (r2 + 1), 0.f);
  const size_t W = r2 + 1;
  for (size_t i = 0; i < r1; i++)
    for (size_t j = 0; j < r2; j++) {
      float* rp = &R[(i + 1) * W + j + 1];
      const float pred = (rp[-1] + rp[-(ptrdiff_t)W]) - rp[-(ptrdiff_t)W - 1];
      const size_t e = i * r2 + j;
      *rp = wide ? l2d_restore_wide(pred, q[e], sid[e], raw[e])
                 : (q[e] == 0 ? raw[e] : pred + l2d_step(q[e], sid[e], 2));
      out[e] = *rp;
    }
}

}  // namespace cpsz
