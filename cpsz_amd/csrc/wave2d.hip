// Lorenzo wavefronts of the 2D codec.
//
// Every value is predicted from the reconstructions of its left, upper and
// upper-left neighbours, so a field is one chain of r1 + r2 dependent steps
// that no reordering shortens. What bounds a single field is the latency of
// one step; what bounds a batch is that latency times the steps of its
// largest field, then the issue slots of the waves.
//
// A strip is 64 rows of one component: lane l of its recurrence wave holds row
// l and takes column t - l at step t, so the value above arrives from lane
// l - 1 through DPP wave_shr:1. A workgroup carries S strips that follow each
// other down the field, kLag chunks of kC steps apart, and hands the rows
// between them through LDS. Its waves are specialised:
//   S recurrence waves   one per strip: the prediction and what depends on it,
//                        nothing else. Each step reads one staged element from
//                        LDS and writes one result (compress 17 vector
//                        instructions a step and 22 in all, decompress 6 and 9).
//   2S input waves       two per strip: load a chunk's tile of codes and its
//                        values (16 columns of 4 rows per instruction), prepare
//                        what depends on the element alone, and stage it in
//                        step order. Loads run kAhead chunks ahead of their use.
//   S output waves       one per strip: results from LDS to the field's rows;
//                        the last one publishes the group's last row.
// All waves meet at one barrier per chunk (which orders LDS only: the loads in
// flight stay in flight). Row pitch kPitch = 68: the recurrence wave's rows
// are contiguous, and 16 steps of 4 rows spread over all banks.
//
// Why tiles (Tile2d) for the codec's own arrays: with row-major codes a chunk is
// 64 pieces of 32 bytes, which the L1 (32 KB for 4 strips' 64 rows) loses
// before the rest of their lines is used; the stores left the CU as requests of
// 21 bytes. Measured on 96 uneven fields (220M vertices) with one wave per
// strip doing everything / specialised waves / and tiles: compress 3.96 / 2.72
// / 1.47 ms, decompress 5.55 / 2.90 / 2.18 ms; one 2400x3600 field 1.57 / 0.94
// / 0.62 and 2.39 / 0.83 / 0.64 ms. (Compress is at 1.35 and 0.55 since no copy
// of the field's descriptor is in scratch memory, see group_item.) One strip alone
// takes 0.56 us a chunk (decompress) to 0.86 us (compress), where the recurrence
// binds; four on one CU 1.4 us, where the values' row-major accesses and the issue
// slots of 16 waves bind.
//
// The row below a group travels through global memory value by value: each
// 64-bit word is a published value or empty (bnd_word), so that the reader
// needs no counter and the writer no wait for its stores. Groups are taken
// from a ticket counter in dependency order: every wait targets an earlier
// ticket, whose workgroup is resident or done.
#include "wave2d.hpp"

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "lorenzo2d_step.hpp"

namespace cpsz {
namespace {

constexpr int kC = kTileSteps;  // steps per chunk
constexpr int kPitch = 68;   // staged elements per step
constexpr int kLag = 5;      // chunks between two strips: 63 steps + 1, rounded up, + 1 for the barrier
constexpr int kAhead = 4;    // chunks between an input wave's loads and their use
constexpr int kRing = 128;   // ring of a strip's last-row values (> kLag * kC + kC)

// Global address space: the pointers of a batch's table are generic, and flat
// accesses would count with the LDS accesses that the barrier waits for.
#define GLB __attribute__((address_space(1)))
#define CST __attribute__((address_space(4)))

__device__ __forceinline__ uint64_t ld_coh64(const GLB uint64_t* p) {
  return __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_coh64(GLB uint64_t* p, uint64_t v) {
  __hip_atomic_store((uint64_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// lane l takes lane l - 1's src, lane 0 keeps lane0
__device__ __forceinline__ float shr1(float src, float lane0) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(lane0), __float_as_int(src),
                                                    0x138 /* wave_shr:1 */, 0xF, 0xF, false));
}
__device__ __forceinline__ double shr1(double src, double lane0) {
  const uint64_t b = l2d_bits(src), z = l2d_bits(lane0);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)z, (int)(uint32_t)b, 0x138, 0xF, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)(z >> 32), (int)(uint32_t)(b >> 32), 0x138,
                                                            0xF, 0xF, false);
  return l2d_double(((uint64_t)hi << 32) | lo);
}

// Orders the waves' LDS accesses only: global loads stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A staged element. Compress: the value and l2d_prep of its eb code (wide: the
// code's bits). Decompress: the step and an all-ones mask where the
// unpredictable value stands in its place (wide: the value or the id's bits,
// and the code's bits).
template <typename T>
struct alignas(2 * sizeof(T)) Elem {
  T a, b;
};

template <typename T, int S, bool COMPRESS>
struct WaveLds {
  using Out = typename std::conditional<COMPRESS, float, T>::type;  // quanta or reconstructions
  Elem<T> in[S][2][kC][kPitch];
  Out out[S][2][kC][kPitch];
  T up[S + 1][kRing];  // up[w]: the row above strip w, column j at (j + 63) % kRing
};

__device__ __forceinline__ float restore(float pred, const Elem<float>& e) {
  const uint32_t m = __float_as_uint(e.b), s = __float_as_uint(pred + e.a);
  return __uint_as_float((m & __float_as_uint(e.a)) | (~m & s));
}
__device__ __forceinline__ double restore(float pred, const Elem<double>& e) {
  return e.b != 0 ? e.a : (double)pred + e.a;
}

// A strip's part of one array. Elements are addressed by their offset from the
// strip's first one; an access whose lane is not `on` reads 0 or writes
// nothing. Buffer accesses do that in the address unit (offsets past the
// resource's range), so every load and store is issued without a branch, and
// the compiler can count the loads in flight. FAR: strips that span 4 GiB and
// more (far_strip) take 64-bit addresses and masks.
template <typename V, bool FAR>
struct Part;

template <typename V>
struct Part<V, false> {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ Part(const V* base, size_t elems)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(uint32_t)min(elems * sizeof(V), (size_t)0xFFFFFFF0u),
                                               0x00020000)) {}
  __device__ __forceinline__ V load(uint32_t e, bool on) const {
    const uint32_t o = on ? e * (uint32_t)sizeof(V) : 0xFFFFFFFFu;
    if constexpr (sizeof(V) == 4) {
      return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, o, 0, 0));
    } else {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, o, 0, 0);
      return l2d_double((uint64_t)v[1] << 32 | v[0]);
    }
  }
  __device__ __forceinline__ void store(uint32_t e, bool on, V v) const {
    const uint32_t o = on ? e * (uint32_t)sizeof(V) : 0xFFFFFFFFu;
    if constexpr (sizeof(V) == 4) {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc, o, 0, 0);
    } else {
      typedef uint32_t __attribute__((ext_vector_type(2))) u32x2;
      const uint64_t b = l2d_bits(v);
      __builtin_amdgcn_raw_buffer_store_b64(u32x2{(uint32_t)b, (uint32_t)(b >> 32)}, rsrc, o, 0, 0);
    }
  }
};

template <typename V>
struct Part<V, true> {
  GLB V* base;
  size_t elems;
  __device__ Part(const V* b, size_t n) : base((GLB V*)b), elems(n) {}
  __device__ V load(size_t e, bool on) const { return on && e < elems ? base[e] : (V)0; }
  __device__ void store(size_t e, bool on, V v) const {
    if (on && e < elems) base[e] = v;
  }
};

// One item: S consecutive strips of one component (group g). `wave` is
// uniform: 0..S-1 recurrence, S..3S-1 input, 3S..4S-1 output. FAR: a strip
// spans 4 GiB or more (64-bit offsets within it). FLIP: the field may be flipped
// (in decompression, masking the rows that such a field lacks costs a single
// strip 10%: 0.54 against 0.60 ms for 64 rows of 15627). The field's descriptor is read
// by scalar loads where a role needs it: members held since the kernel's beginning
// would spill, and a copy to choose the component from would be in scratch memory.
template <typename T, int S, bool COMPRESS, bool FAR, bool FLIP>
__device__ __forceinline__ void group_item(const CST Strip2dT<T>& a, bool wide, int comp, int g, int wave, int lane,
                                           WaveLds<T, S, COMPRESS>& sh) {
  constexpr bool kMayWide = sizeof(T) == 4;  // double fields have one step for all ids
  const int r1 = a.r1, r2 = a.r2;
  const int nstrips = (r1 + 63) >> 6;
  const int ns = min(S, nstrips - g * S);        // strips of this group
  const int nch = a.t.nch;                       // chunks of a strip
  // strip w computes chunk e - 1 in iteration it = e + kLag w: its input waves
  // stage chunk e, its output wave stores chunk e - 2 (iterations rounded up
  // to the input waves' rotation of kAhead sets)
  const int it_end = (nch + 2 + kLag * (ns - 1) + kAhead - 1) / kAhead * kAhead;
  const int role = wave < S ? 0 : (wave < 3 * S ? 1 : 2);
  const int w = role == 0 ? wave : (role == 1 ? (wave - S) >> 1 : wave - 3 * S);
  const int row0 = (g * S + w) * 64;             // first row of the wave's strip
  const int e0 = -kLag * w;                      // e = it + e0
  if (w >= ns) {
    for (int it = -kAhead; it < it_end; it++) lds_barrier();
    return;
  }
  // a chunk whose columns lie inside the row for every lane
  auto columns_inside = [&](int c) { return c * kC >= 63 && c * kC + kC <= r2; };

  if (role == 0) {
    __builtin_amdgcn_s_setprio(3);
    // the first strip fetches the row above the group, one chunk ahead of its
    // use (this wave has no other global accesses to wait for)
    const bool fetch = w == 0 && g > 0;
    const GLB uint64_t* bin = (const GLB uint64_t*)a.bnd + ((size_t)comp * a.ngroups + (g > 0 ? g - 1 : 0)) * r2;
    const uint64_t none = bnd_word((T)0);
    uint64_t next = none;  // lane k: column c kC + k of the chunk to come
    auto peek = [&](int c) {
      const int j = c * kC + lane;
      return lane < kC && j < r2 ? ld_coh64(bin + j) : none;
    };
    T Rp = 0, Up = 0;  // the previous step's value and the one above it
    for (int it = -kAhead; it < it_end; it++) {
      const int c = it + e0 - 1;
      if (c >= 0 && c < nch) {
        const Elem<T>(*in)[kPitch] = sh.in[w][c & 1];
        auto(*out)[kPitch] = sh.out[w][c & 1];
        const int t0 = c * kC;
        const T* up0 = &sh.up[w][(t0 + 63) & (kRing - 1)];
        const T* up1 = &sh.up[w][(t0 + 64) & (kRing - 1)];
        T* last = &sh.up[w + 1][t0 & (kRing - 1)];
        if (kMayWide && wide) {
          if constexpr (kMayWide) {
#pragma unroll 1
            for (int k = 0; k < kC; k++) {
              const Elem<T> e = in[k][lane];
              const T Uv = shr1(Rp, k == 0 ? up0[0] : up1[k - 1]);
              const float pred = (Rp + Uv) - Up;
              if constexpr (COMPRESS) {
                Rp = l2d_quantize_wide(pred, e.a, l2d_bits(e.b), out[k][lane]);
              } else {
                Rp = l2d_restore_wide(pred, l2d_bits(e.b), l2d_bits(e.a), e.a);
                out[k][lane] = Rp;
              }
              Up = Uv;
              if (lane == 63) last[k] = Rp;
            }
          }
        } else {
          // the chunk's inputs first: the compiler would not move the reads
          // above the results' writes
          Elem<T> e[kC];
          T u[kC];
#pragma unroll
          for (int k = 0; k < kC; k++) {
            e[k] = in[k][lane];
            u[k] = k == 0 ? up0[0] : up1[k - 1];
          }
#pragma unroll
          for (int k = 0; k < kC; k++) {
            const T Uv = shr1(Rp, u[k]);
            const float pred = (float)((Rp + Uv) - Up);
            if constexpr (COMPRESS) {
              Rp = l2d_quantize(pred, e[k].a, e[k].b, out[k][lane]);
            } else {
              Rp = restore(pred, e[k]);
              out[k][lane] = Rp;
            }
            Up = Uv;
            u[k] = Rp;
          }
          if (lane == 63) {
#pragma unroll
            for (int k = 0; k < kC; k++) last[k] = u[k];
          }
        }
      }
      if (fetch && c + 1 >= 0) {
        if ((c + 1) * kC < r2) {  // chunk c + 1 is computed in the next iteration
          if (c + 1 == 0) next = peek(0);
          while (!__all(bnd_ready(next, (T)0))) {
            __builtin_amdgcn_s_sleep(1);
            if (!bnd_ready(next, (T)0)) next = ld_coh64(bin + (c + 1) * kC + lane);
          }
          if (lane < kC) sh.up[0][((c + 1) * kC + lane + 63) & (kRing - 1)] = bnd_value(next, (T)0);
        }
        next = peek(c + 2);
      }
      lds_barrier();
    }
    __builtin_amdgcn_s_setprio(0);
  } else if (role == 1) {
    const int half = (wave - S) & 1, shift = a.shift;
    using Off = typename std::conditional<FAR, size_t, uint32_t>::type;
    // The code arrays are tiles: chunk c of the strip is one contiguous piece,
    // and a lane takes 8 consecutive steps (from k8) of row lt of it.
    const int rows_log = a.t.rows_log, tile_log = rows_log + 4;
    const size_t strip_at = (size_t)(g * S + w) * nch << tile_log;
    // The row-major arrays: row l, column t - l is at l * ls + t * cs
    const int cs = FLIP ? a.cs : 1, ls = cs == 1 ? r2 - 1 : 1 - cs;
    const int lt = 32 * half + (lane >> 1), k8 = 8 * (lane & 1);
    const uint32_t lane_at = (uint32_t)(min(lt, (1 << rows_log) - 1) * kC + k8);  // (rows past a short tile's last: any)
    const GLB uint16_t* C = (const GLB uint16_t*)a.c[comp] + strip_at;
    const GLB uint16_t* Q = (const GLB uint16_t*)a.q[comp] + strip_at;
    // The values of a compression are row-major: 16 columns of 4 rows per
    // instruction; chunk c, group i: row lx + 4 i, column c kC + kx - row.
    // (one element per lane: a load of two floats costs three times a load of
    // one here, and at 2-byte alignment a load of two codes four times)
    const int kx = lane & 15, lx = 32 * half + (lane >> 4);
    const size_t first = (size_t)row0 * r2;
    const Part<T, FAR> X(COMPRESS ? a.x[comp] + first : a.raw[comp] + strip_at,
                         COMPRESS ? (size_t)r1 * r2 - first : (size_t)nch << tile_log);
    Off lane0 = (Off)lx * (Off)ls + (Off)kx * (Off)cs;
    const Off istep = 4 * (Off)ls, cstep = kC * (Off)cs;
    int lane_col = kx - lx;
    // What a wave holds of a chunk on its way from memory to LDS: eb codes
    // and values, or stream ids, quantization codes and unpredictable values.
    // Every load is issued in every iteration, and with no branch around it:
    // with loads that may be skipped, the wait for a set would have to be a
    // wait for all of them.
    struct Codes {
      uint32_t c[4], q[COMPRESS ? 1 : 4];  // 8 codes each
    };
    struct Values {
      T v[8];
    };
    auto ld16 = [&](const GLB uint16_t* p, uint32_t* d) {
      typedef uint32_t __attribute__((ext_vector_type(4))) u32x4;
      const u32x4 x = *(const GLB u32x4*)p;
      d[0] = x[0];
      d[1] = x[1];
      d[2] = x[2];
      d[3] = x[3];
    };
    auto nth = [](const uint32_t* d, int m) { return (m & 1) ? d[m >> 1] >> 16 : d[m >> 1] & 0xFFFFu; };
    // element (lt, k8 + m) of chunk c lies in the field
    const bool row_in = row0 + lt < r1;
    auto inside = [&](int c, int m) { return row_in && (uint32_t)(c * kC + k8 + m - lt) < (uint32_t)r2; };
    auto load = [&](int c, Values& x, Codes& s) {
      const size_t at = (size_t)min(max(c, 0), nch - 1) << tile_log;
      ld16(C + at + lane_at, s.c);
      if constexpr (!COMPRESS) {
        ld16(Q + at + lane_at, s.q);
      } else {
        // (a row past the field's last lies past the array's end; chunks
        // before the first and after the last one are outside the row)
#pragma unroll
        for (int i = 0; i < 8; i++)
          x.v[i] = X.load(lane0 + ((Off)c * cstep + i * istep), (uint32_t)(lane_col + (c * kC - 4 * i)) < (uint32_t)r2);
      }
    };
    // decompress: the unpredictable values, where the code is 0
    auto load_raw = [&](int c, Values& x, const Codes& s) {
      if constexpr (!COMPRESS) {
        const Off at = ((Off)min(max(c, 0), nch - 1) << tile_log) + lane_at;
#pragma unroll
        for (int m = 0; m < 8; m++) x.v[m] = X.load(at + m, nth(s.q, m) == 0);
      }
    };
    // Outside the field the staged elements are (0, code 0) or an
    // unpredictable 0, which keeps the recurrence at 0 there.
    auto stage = [&](int c, const Values& x, const Codes& s, auto at_edge, auto is_wide) {
      Elem<T>(*in)[kPitch] = sh.in[w][c & 1];
      if constexpr (COMPRESS) {
#pragma unroll
        for (int i = 0; i < 8; i++) in[kx][lx + 4 * i].a = x.v[i];
      }
#pragma unroll
      for (int m = 0; m < 8; m++) {
        uint32_t cc = nth(s.c, m);
        Elem<T>& e = in[k8 + m][lt];
        if constexpr (COMPRESS) {
          if (decltype(at_edge)::value) cc = inside(c, m) ? cc : 0;
          if constexpr (sizeof(T) == 8) e.b = l2d_prep64(cc);
          else if constexpr (decltype(is_wide)::value) e.b = l2d_float(cc);
          else e.b = l2d_prep(cc, shift);
        } else {
          uint32_t q = nth(s.q, m);
          T v = x.v[m];
          if (decltype(at_edge)::value) {
            const bool in_field = inside(c, m);
            q = in_field ? q : 0;
            v = in_field ? v : (T)0;
          }
          Elem<T> y;
          if constexpr (sizeof(T) == 8) {
            const double step = l2d_step64(q, cc);
            y.a = q ? step : v;
            y.b = q ? 0.0 : 1.0;
          } else if constexpr (decltype(is_wide)::value) {
            y.a = q ? l2d_float(cc) : v;
            y.b = l2d_float(q);
          } else {
            const float step = l2d_step(q, cc, shift);
            y.a = q ? step : v;
            y.b = __uint_as_float(q ? 0u : 0xFFFFFFFFu);
          }
          e = y;
        }
      }
    };
    const bool full_rows = row0 + 64 <= r1;
    // iteration it: stage chunk e (loaded kAhead iterations ago into the same
    // set), fetch chunk e + 2's unpredictable values, load chunk e + kAhead
    auto iteration = [&](int it, Codes& s0, const Codes& s2, Values& x) {
      const int e = it + e0;
      // opaque per iteration: the lanes' parts of the 8 groups' offsets and
      // columns, kept in registers across the loop, would spill
      asm volatile("" : "+v"(lane0), "+v"(lane_col));
      if (e >= 0 && e < nch) {
        if (kMayWide && wide) {
          if constexpr (kMayWide) stage(e, x, s0, std::true_type{}, std::true_type{});
        } else if (full_rows && columns_inside(e)) {
          stage(e, x, s0, std::false_type{}, std::false_type{});
        } else {
          stage(e, x, s0, std::true_type{}, std::false_type{});
        }
      }
      load_raw(e + 2, x, s2);
      load(e + kAhead, x, s0);
      lds_barrier();
    };
    Codes ca{}, cb{}, cc{}, cd{};
    Values xa, xb, xc, xd;
    for (int it = -kAhead; it < it_end; it += kAhead) {
      iteration(it, ca, cc, xa);
      iteration(it + 1, cb, cd, xb);
      if constexpr (COMPRESS) {
        iteration(it + 2, cc, ca, xc);
        iteration(it + 3, cd, cb, xd);
      } else {
        iteration(it + 2, cc, ca, xa);
        iteration(it + 3, cd, cb, xb);
      }
    }
  } else {
    const bool publish = w == S - 1 && g + 1 < a.ngroups;
    GLB uint64_t* bout = (GLB uint64_t*)a.bnd + ((size_t)comp * a.ngroups + g) * r2;
    // compress: the chunk's codes are one tile, 8 steps of a row per lane and half;
    // decompress: values, 16 columns of 4 rows per instruction
    const int lt = lane >> 1, k8 = 8 * (lane & 1);
    const int tile_log = a.t.rows_log + 4, tile_rows = 1 << a.t.rows_log;
    GLB uint16_t* Q = (GLB uint16_t*)a.q[comp] + ((size_t)(g * S + w) * nch << tile_log);
    const int k = lane & 15, rs = lane >> 4;
    using Off = typename std::conditional<FAR, size_t, uint32_t>::type;
    const size_t first = (size_t)row0 * r2;
    const Part<T, FAR> O(a.out[comp] + first, (size_t)r1 * r2 - first);
    const int cs = FLIP ? a.cs : 1, ls = cs == 1 ? r2 - 1 : 1 - cs;
    const Off lane0 = (Off)rs * (Off)ls + (Off)k * (Off)cs, istep = 4 * (Off)ls, cstep = kC * (Off)cs;
    // (row-major, a row past the field's last lies past the array's end)
    const int rows = cs == 1 ? 64 : r1;
    for (int it = -kAhead; it < it_end; it++) {
      const int c = it + e0 - 2;
      if (c >= 0 && c < nch) {
        if (publish && lane < kC) {
          const int t = c * kC + lane, j = t - 63;
          if (j >= 0 && j < r2) st_coh64(bout + j, bnd_word(sh.up[S][t & (kRing - 1)]));
        }
        const auto(*out)[kPitch] = sh.out[w][c & 1];
        // all reads first: the compiler would not move them above the stores
        typename WaveLds<T, S, COMPRESS>::Out v[16];
        if constexpr (COMPRESS) {
#pragma unroll
          for (int m = 0; m < 16; m++) v[m] = out[k8 + (m & 7)][lt + 32 * (m >> 3)];
#pragma unroll
          for (int h = 0; h < 2; h++) {
            typedef uint32_t __attribute__((ext_vector_type(4))) u32x4;
            u32x4 p;
#pragma unroll
            for (int m = 0; m < 4; m++)
              p[m] = l2d_code(v[8 * h + 2 * m]) | (uint32_t)l2d_code(v[8 * h + 2 * m + 1]) << 16;
            const int l = lt + 32 * h;
            if (l < tile_rows) *(GLB u32x4*)(Q + (((size_t)c << tile_log) + l * kC + k8)) = p;
          }
        } else {
#pragma unroll
          for (int i = 0; i < 16; i++) v[i] = out[k][4 * i + rs];
#pragma unroll
          for (int i = 0; i < 16; i++)
            O.store(lane0 + ((Off)c * cstep + i * istep),
                    (!FLIP || rs + 4 * i < rows) && (uint32_t)(c * kC + k - rs - 4 * i) < (uint32_t)r2, v[i]);
        }
      }
      lds_barrier();
    }
  }
}

// Fields of one launch: a single field travels in the kernel arguments (one),
// several through a device table f[0..nf) with start[k] = first item of field
// k. Items are (group, component) pairs in group order, numbered field by
// field and taken from one ticket counter.
template <typename T>
struct StripBatch {
  Strip2dT<T> one;  // (first: the kernel finds it at the beginning of its arguments)
  const Strip2dT<T>* f;  // null: the single field `one`
  const int* start;
  int nf, items;
  int* ticket;
};

template <typename T, int S, bool COMPRESS, bool FAR, bool FLIP>
__global__ void __launch_bounds__(256 * S) k_wave2d(StripBatch<T> b) {
  __shared__ WaveLds<T, S, COMPRESS> sh;
  __shared__ int s_item;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  for (;;) {
    if (threadIdx.x == 0) s_item = atomicAdd(b.ticket, 1);
    // the first group of a component has zeros above it; the other rings are
    // written before they are read
    for (int i = threadIdx.x; i < kRing; i += blockDim.x) sh.up[0][i] = 0;
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(s_item);
    if (item >= b.items) return;
    int lo = 0, at = item;
    if (b.f) {
      int hi = b.nf - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (((const CST int*)b.start)[mid] <= item) lo = mid;
        else hi = mid - 1;
      }
      at = item - ((const CST int*)b.start)[lo];
    }
    // (constant address space: neither is written while the kernel runs)
    const CST Strip2dT<T>* const f = b.f ? (const CST Strip2dT<T>*)b.f + lo
                                         : (const CST Strip2dT<T>*)__builtin_amdgcn_kernarg_segment_ptr();  // b.one
    bool skip = false, wide = f->wide;
    if (f->flags) {
      skip = __builtin_amdgcn_readfirstlane(f->flags[0]) != 0;  // every item of the field skips: no group waits on another
      wide = __builtin_amdgcn_readfirstlane(f->flags[1]) != 0;
    }
    if (!skip) group_item<T, S, COMPRESS, FAR, FLIP>(*f, wide, at & 1, at >> 1, wave, lane, sh);
    __syncthreads();
  }
}

// 64-bit words of a field's published rows: none when one group carries all
// its rows (which is so for every flipped field).
template <typename T>
__host__ __device__ size_t published_words(const Strip2dT<T>& f) {
  return f.ngroups > 1 ? (size_t)2 * f.ngroups * f.r2 : 0;
}

// Empties every field's published rows (block row y = field) and clears the
// launch's ticket.
template <typename T>
__global__ void __launch_bounds__(256) k_wave2d_clear(StripBatch<T> b) {
  const Strip2dT<T>& f = b.f ? b.f[blockIdx.y] : b.one;
  uint64_t* bnd = f.bnd;
  const size_t n = published_words(f);
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += step) bnd[i] = sizeof(T) == 8 ? kBndEmpty : 0;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *b.ticket = 0;
}

// The kernel's rows and columns: a flipped field's are exchanged, one strip.
template <typename T>
void orient(Strip2dT<T>& f) {
  f.cs = 1;
  if (!f.t.flip) return;
  f.cs = f.r2;
  std::swap(f.r1, f.r2);
  f.ngroups = 1;
}

// The kernel for the fields of one launch: the plainest that takes them all
// (compression and 64-bit offsets always take flipped fields).
template <typename T, int S, bool COMPRESS>
void launch_wave(Ctx& ctx, const StripBatch<T>& b, int grid_cap, bool far, bool flip) {
  const int grid = std::min(b.items, grid_cap);
  if (far) k_wave2d<T, S, COMPRESS, true, true><<<grid, 256 * S, 0, ctx.stream()>>>(b);
  else if (COMPRESS || flip) k_wave2d<T, S, COMPRESS, false, true><<<grid, 256 * S, 0, ctx.stream()>>>(b);
  else k_wave2d<T, S, COMPRESS, false, COMPRESS><<<grid, 256 * S, 0, ctx.stream()>>>(b);
  CPSZ_HIP(hipGetLastError());
}

template <typename T, int S, bool COMPRESS>
void launch_one(Ctx& ctx, Strip2dT<T> f, int grid_cap) {
  hipStream_t st = ctx.stream();
  orient(f);
  StripBatch<T> b{};
  b.one = f;
  b.nf = 1;
  b.items = 2 * f.ngroups;
  b.ticket = f.ticket;
  const size_t words = published_words(f);
  k_wave2d_clear<T><<<(unsigned)std::min<size_t>(div_up(words, 256) + 1, 1024), 256, 0, st>>>(b);
  launch_wave<T, S, COMPRESS>(ctx, b, grid_cap, far_strip(f.r2, sizeof(T)), f.t.flip);
}

template <bool COMPRESS>
void launch_many(Ctx& ctx, std::vector<Strip2d>& f, int grid_cap) {
  if (f.size() == 1 && !f[0].flags) {
    launch_one<float, kStrips, COMPRESS>(ctx, f[0], grid_cap);
    return;
  }
  // Tickets go out field by field, the fields with the longest wavefront (a
  // strip's lag per strip plus the row length) first: the launch ends when its
  // longest chain does.
  hipStream_t st = ctx.stream();
  const size_t nf = f.size();
  CPSZ_REQUIRE(nf <= 65535, kErrUnsupported, "2D batch: at most 65535 fields per call");
  std::vector<Strip2d> g(f);
  for (Strip2d& x : g) orient(x);
  auto steps = [](const Strip2d& a) { return (int64_t)div_up((size_t)a.r1, (size_t)64) * kLag * kC + a.r2; };
  std::stable_sort(g.begin(), g.end(), [&](const Strip2d& a, const Strip2d& b) { return steps(a) > steps(b); });
  std::vector<int> start(nf + 1, 0);
  size_t max_words = 0;
  for (size_t k = 0; k < nf; k++) {
    start[k + 1] = start[k] + 2 * g[k].ngroups;
    max_words = std::max(max_words, published_words(g[k]));
  }
  const size_t tbytes = nf * sizeof(Strip2d), sbytes = (nf + 1) * sizeof(int);
  uint8_t* d = ctx.buf<uint8_t>("w2b.tab", tbytes + sbytes + 64);
  uint8_t* h = (uint8_t*)ctx.host_table("w2b.tab", tbytes + sbytes);
  std::memcpy(h, g.data(), tbytes);
  std::memcpy(h + tbytes, start.data(), sbytes);
  ctx.upload_table("w2b.tab", d, h, tbytes + sbytes);
  StripBatch<float> b{};
  b.f = (const Strip2d*)d;
  b.start = (const int*)(d + tbytes);
  b.nf = (int)nf;
  b.items = start[nf];
  b.ticket = (int*)(d + ((tbytes + sbytes + 15) & ~(size_t)15));
  k_wave2d_clear<float><<<dim3((unsigned)std::min<size_t>(div_up(max_words, 256 * 8) + 1, 64), (unsigned)nf), 256, 0, st>>>(b);
  launch_wave<float, kStrips, COMPRESS>(
      ctx, b, grid_cap, std::any_of(g.begin(), g.end(), [](const Strip2d& x) { return far_strip(x.r2, sizeof(float)); }),
      std::any_of(g.begin(), g.end(), [](const Strip2d& x) { return x.t.flip; }));
}

}  // namespace

void wavefront2d_compress(Ctx& ctx, std::vector<Strip2d>& f, int grid_cap) { launch_many<true>(ctx, f, grid_cap); }
void wavefront2d_decompress(Ctx& ctx, std::vector<Strip2d>& f, int grid_cap) { launch_many<false>(ctx, f, grid_cap); }
void wavefront2d_compress64(Ctx& ctx, Strip2d64& f, int grid_cap) { launch_one<double, kStrips64, true>(ctx, f, grid_cap); }
void wavefront2d_decompress64(Ctx& ctx, Strip2d64& f, int grid_cap) {
  launch_one<double, kStrips64, false>(ctx, f, grid_cap);
}

}  // namespace cpsz
