// GPU Huffman stage shared by the 2D and 3D codecs.
//
// Symbols are produced by a "source" that exposes one chunk as items in
// stream order (`get(chunk, item, sym[])`), so the block-major
// (2D) or predictable-vertex (3D) orders of the reference stream are walked in
// place without materializing a permuted copy. One wave takes one chunk, its
// lanes consecutive items.
//
//   histogram : LDS-privatized window + global atomics outside the window
//   encode    : per-chunk bit counts -> exclusive scan -> each wave packs its
//               chunk's codes MSB-first in LDS (lane offsets from a wave
//               prefix sum) and stores 32-bit big-endian words coalesced; only
//               the first and last (shared) word of a chunk use atomicOr
//   decode    : parallel decode of the single unchunked bitstream: every code
//               boundary that a segment can start on, given nothing but the
//               bits before it; the exit and count from each; then the one true
//               chain through them, and the final decode
#pragma once
#include <hip/hip_runtime.h>

#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/transform_iterator.hpp>
#include <cstring>
#include <exception>
#include <functional>
#include <string>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "ctx.hpp"
#include "huff_host.hpp"

namespace cpsz {

constexpr int kLutBits = 11;
constexpr int kLut2Bits = 12;  // width cap of the level-2 decode tables
constexpr uint32_t kSegBits = 256;   // bits per decode segment
constexpr uint32_t kWarmBits = 256;  // bits before a segment from which its possible starts are worked out
constexpr int kCand = 16;            // possible starts kept per segment

__device__ __forceinline__ uint32_t bswap32(uint32_t x) { return __builtin_bswap32(x); }

// --------------------------------------------------------------- histogram --
// One wave per chunk (sources as for the encode kernels below), grid-stride
// over chunks; symbols in [win_lo, win_lo + win_n) count in LDS, the rest in
// global memory directly.
template <class Src>
__global__ void __launch_bounds__(256) k_hist(Src src, size_t nchunks, uint32_t* __restrict__ hist,
                                              uint32_t win_lo, uint32_t win_n);

// ------------------------------------------------------------------ encode --
// The encode-side kernels run one wave per chunk (4 chunks per 256-thread
// block). A source exposes its chunk (of the 3D streams; the 2D ones follow below) as items taken by lanes in stream order:
//   Src::kMaxItems            items per chunk at most
//   Src::kPer                 symbols per item at most
//   int get(c, idx, sym[])    the symbols of item idx, in stream order, and
//                             their count; idx in [0, kMaxItems), 0 symbols
//                             past the chunk's end (branch-free, so that a
//                             wave issues every round's loads together)
constexpr int kEncWaves = 4;
constexpr int kEncThreads = kEncWaves * 64;  // block size of the chunk-bits and encode kernels

inline size_t encode_blocks(size_t nchunks) { return (nchunks + kEncWaves - 1) / kEncWaves; }

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  return x;
}

// A source may also carry the stream's unpredictable values (kUnpred): the
// values at its symbol-0 items, gathered in stream order while encoding.
template <class S, class = void>
struct HasUnpred : std::false_type {};
template <class S>
struct HasUnpred<S, std::void_t<decltype(S::kUnpred)>> : std::bool_constant<S::kUnpred> {};

template <class Src>
__device__ __forceinline__ void chunk_bits_wave(const Src& src, size_t c, const uint8_t* __restrict__ len,
                                                uint64_t* __restrict__ bits) {
  constexpr int kRounds = (Src::kMaxItems + 63) / 64;
  const int lane = threadIdx.x & 63;
  // every round's symbols are fetched before any is used (overlapped latency)
  uint32_t sym[kRounds][Src::kPer];
  int ns[kRounds];
#pragma unroll
  for (int r = 0; r < kRounds; r++) ns[r] = src.get(c, r * 64 + lane, sym[r]);
  uint32_t b = 0;
#pragma unroll
  for (int r = 0; r < kRounds; r++)
#pragma unroll
    for (int q = 0; q < Src::kPer; q++)
      if (q < ns[r]) b += len[sym[r][q]];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) b += __shfl_xor(b, o);
  if (lane == 0) bits[c] = b;
}

template <class Src>
__global__ void __launch_bounds__(kEncThreads) k_chunk_bits(Src src, size_t nchunks,
                                                    const uint8_t* __restrict__ len,
                                                    uint64_t* __restrict__ bits) {
  const size_t c = (size_t)xcd_block(blockIdx.x, gridDim.x) * kEncWaves + (threadIdx.x >> 6);
  if (c >= nchunks) return;  // whole wave
  chunk_bits_wave(src, c, len, bits);
}

// ---- many streams per launch: a job table sorted by first block; block b
// belongs to the job with the largest blk0 <= b.
template <class Job>
__device__ __forceinline__ int job_of(const Job* __restrict__ jobs, int nj, uint32_t b) {
  int lo = 0, hi = nj - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].blk0 <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

template <class Src>
struct EncJob {
  Src src;
  size_t nchunks;
  const uint64_t* code;  // dense codebook of this stream's tree
  const uint8_t* len;
  const uint64_t* off;   // global exclusive scan of chunk bits, at this stream's first chunk
  uint64_t* bits;        // chunk bits, at this stream's first chunk
  uint32_t* words;       // this stream's zero-filled word array
  uint32_t blk0;         // first block (kEncWaves chunks per block)
  uint32_t* zc;          // optional: per-chunk symbol-0 counts (with the bits), for the offsets of gathered values
};

// A source whose n symbols include `pads` extra symbols 0 (kPads), which the
// histogram does not count. (Those past the last whole chunk, fewer than one, are
// counted one by one.)
template <class S, class = void>
struct HasPads : std::false_type {};
template <class S>
struct HasPads<S, std::void_t<decltype(S::kPads)>> : std::bool_constant<S::kPads> {};

template <class Src>
__device__ __forceinline__ void hist_block(const Src& src, size_t nchunks, uint32_t* __restrict__ hist,
                                           uint32_t win_lo, uint32_t win_n, uint32_t blk, uint32_t nblk,
                                           uint32_t* sh) {
  constexpr int kRounds = (Src::kMaxItems + 63) / 64;
  for (uint32_t i = threadIdx.x; i < win_n; i += blockDim.x) sh[i] = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  // symbol 0 (the unpredictable marker of the 2D code streams, often frequent)
  // counts in a register when it lies outside the window: one global atomic
  // per wave instead of one per occurrence on a single address
  const bool zero_out = win_lo > 0;
  uint32_t zeros = 0;
  const uint32_t waves = blockDim.x >> 6;
  for (size_t c = (size_t)blk * waves + (threadIdx.x >> 6); c < nchunks; c += (size_t)nblk * waves) {
    uint32_t sym[kRounds][Src::kPer];
    int ns[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) ns[r] = src.get(c, r * 64 + lane, sym[r]);
#pragma unroll
    for (int r = 0; r < kRounds; r++)
#pragma unroll
      for (int q = 0; q < Src::kPer; q++) {
        if (q < ns[r]) {
          const uint32_t o = sym[r][q] - win_lo;
          if (o < win_n) atomicAdd(&sh[o], 1u);
          else if (zero_out && sym[r][q] == 0) zeros++;
          else atomicAdd(&hist[sym[r][q]], 1u);
        }
      }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) zeros += __shfl_xor(zeros, o);
  if (lane == 0 && zeros) atomicAdd(&hist[0], zeros);
  if constexpr (HasPads<Src>::value) {
    if (blk == 0) {
      if (threadIdx.x == 0) atomicSub(&hist[0], src.pads);
      for (size_t i = nchunks * Src::kChunk + threadIdx.x; i < src.n; i += blockDim.x) atomicAdd(&hist[src.at(i)], 1u);
    }
  }
  __syncthreads();
  // blocks start their flush at different bins so that their global atomics
  // on the popular bins do not all arrive together
  const uint32_t rot = (uint32_t)(((uint64_t)blk * 2654435761u) % win_n);
  for (uint32_t i = threadIdx.x; i < win_n; i += blockDim.x) {
    const uint32_t b = i + rot < win_n ? i + rot : i + rot - win_n;
    if (sh[b]) atomicAdd(&hist[win_lo + b], sh[b]);
  }
}

template <class Src>
__global__ void __launch_bounds__(256) k_hist(Src src, size_t nchunks, uint32_t* __restrict__ hist,
                                              uint32_t win_lo, uint32_t win_n) {
  extern __shared__ uint32_t sh[];
  hist_block(src, nchunks, hist, win_lo, win_n, xcd_block(blockIdx.x, gridDim.x), gridDim.x, sh);
}

template <class Src>
struct HistJob {
  Src src;
  size_t nchunks;
  uint32_t* hist;
  uint32_t blk0, nblk;
};

template <class Src>
__global__ void __launch_bounds__(256) k_hist_multi(const HistJob<Src>* __restrict__ jobs, int nj, uint32_t win_lo,
                                                    uint32_t win_n) {
  extern __shared__ uint32_t sh[];
  const HistJob<Src>& J = jobs[job_of(jobs, nj, blockIdx.x)];
  hist_block(J.src, J.nchunks, J.hist, win_lo, win_n, blockIdx.x - J.blk0, J.nblk, sh);
}

// Writes the MSB-aligned code cw (L bits) at bit p of an MSB-first word array.
__device__ __forceinline__ void put_bits(uint32_t* st, uint32_t p, uint64_t cw, uint32_t L) {
  const uint32_t wi = p >> 5, o = p & 31;
  atomicOr(&st[wi], (uint32_t)(cw >> (32 + o)));
  if (L > 32 - o) atomicOr(&st[wi + 1], (uint32_t)((cw << (32 - o)) >> 32));
  if (L > 64 - o) atomicOr(&st[wi + 2], (uint32_t)((cw << (64 - o)) >> 32));  // o > 0 here
}

// Each wave assembles its chunk's bits in LDS (lanes place consecutive
// symbols at offsets from a wave prefix sum) and then stores the chunk's
// words with consecutive lanes on consecutive words. The words a chunk
// shares with its neighbours (a partial first or last word) are merged with
// atomicOr into the zero-filled output; the others are plain stores. b0 is
// the chunk's first bit within its stream. Called by whole blocks: the
// block's waves (adjacent chunks, whose rows share cache lines) stay in step
// at its barriers, which measured faster than letting them drift apart.
template <class Src>
__device__ __forceinline__ void encode_wave(const Src& src, size_t c, bool live, uint64_t b0, uint64_t nbits,
                                            const uint64_t* __restrict__ code, const uint8_t* __restrict__ len,
                                            uint32_t* __restrict__ words, uint32_t* st) {
  const int lane = threadIdx.x & 63;
  const uint32_t sh = (uint32_t)(b0 & 31), nw = (uint32_t)((sh + nbits + 31) >> 5);
  for (uint32_t k = lane; k < nw; k += 64) st[k] = 0;
  __syncthreads();
  if (live) {
    constexpr int kRounds = (Src::kMaxItems + 63) / 64;
    // every round's symbols, lengths and codes are fetched before any is used
    uint32_t sym[kRounds][Src::kPer], L[kRounds][Src::kPer];
    uint64_t cw[kRounds][Src::kPer];
    int ns[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) ns[r] = src.get(c, r * 64 + lane, sym[r]);
#pragma unroll
    for (int r = 0; r < kRounds; r++)
#pragma unroll
      for (int q = 0; q < Src::kPer; q++) {
        const uint32_t l = len[sym[r][q]];  // symbols are always valid table indices
        L[r][q] = q < ns[r] ? l : 0u;
        cw[r][q] = code[sym[r][q]];
      }
    uint32_t pos = sh;
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
      uint32_t b = 0;
#pragma unroll
      for (int q = 0; q < Src::kPer; q++) b += L[r][q];
      const uint32_t incl = wave_incl_scan(b);
      uint32_t p = pos + incl - b;
#pragma unroll
      for (int q = 0; q < Src::kPer; q++) {
        if (L[r][q]) put_bits(st, p, cw[r][q], L[r][q]);
        p += L[r][q];
      }
      pos += __shfl(incl, 63);
    }
  }
  __syncthreads();
  if (live) {
    const size_t w0 = b0 >> 5;
    const bool tail_shared = ((b0 + nbits) & 31) != 0;
    for (uint32_t k = lane; k < nw; k += 64) {
      const uint32_t word = bswap32(st[k]);
      if ((k == 0 && sh != 0) || (k == nw - 1 && tail_shared)) atomicOr(&words[w0 + k], word);
      else words[w0 + k] = word;
    }
  }
}

template <class Src>
__global__ void __launch_bounds__(kEncThreads) k_encode(Src src, size_t nchunks,
                                                const uint64_t* __restrict__ code,
                                                const uint8_t* __restrict__ len,
                                                const uint64_t* __restrict__ off,
                                                const uint64_t* __restrict__ bits,
                                                uint32_t* __restrict__ words) {
  constexpr int kStage = Src::kMaxItems * Src::kPer * 2 + 2;  // 64-bit codes at most
  __shared__ uint32_t stage[kEncWaves][kStage];
  const int wv = threadIdx.x >> 6;
  const size_t c = (size_t)xcd_block(blockIdx.x, gridDim.x) * kEncWaves + wv;
  const bool live = c < nchunks;  // uniform per wave
  encode_wave(src, c, live, live ? off[c] : 0, live ? bits[c] : 0, code, len, words, stage[wv]);
}

// ---- chunks that give every lane a run of consecutive symbols (the 2D
// streams). A source exposes
//   Src::kRun                 symbols per lane at most
//   Src::kLds                 16-bit words of LDS that a wave's chunk takes
//   void stage(c, lds)        the wave brings chunk c's symbols into LDS
//   int load(c, lds, sym)     the lane's symbols, in stream order, and their
//                             count (the others are valid table indices)
// and, with kUnpred, elem(c, k): where the value of the lane's k-th symbol is.
// One scan per chunk places the lanes; a lane packs its codes into words by
// itself and merges each finished word into the wave's LDS words: an OR per 32
// bits in place of one or two per code. Bound by instruction issue and the
// gathers of lengths and codes. 96 fields of 256 to 4096 a side (220 million
// vertices), against one symbol per lane and a scan per 64 of them: bit counts
// and scans 2.02 -> 0.60 ms, encode with the unpredictable values 4.35 -> 2.25.
//
// (Pointers that come out of a job table are generic to the compiler, and a
// load through one waits for LDS as well: glob() says that they are global.)
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T* glob(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kRunWords = 580;  // words of a chunk kept in LDS: 16 bits a symbol and more

template <class Src>
__device__ __forceinline__ void run_bits_wave(const Src& src, size_t c, const uint8_t* __restrict__ len,
                                              uint64_t* __restrict__ bits, uint32_t* __restrict__ zc,
                                              const uint16_t* lds) {
  uint32_t sym[Src::kRun];
  const int ns = src.load(c, lds, sym);
  uint32_t l[Src::kRun];
#pragma unroll
  for (int k = 0; k < Src::kRun; k++) l[k] = glob(len)[sym[k]];
  uint32_t b = 0;  // bits, and in the upper 12 bits the symbols 0
#pragma unroll
  for (int k = 0; k < Src::kRun; k++) b += k < ns ? l[k] + (sym[k] == 0 ? 1u << 20 : 0u) : 0u;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) b += __shfl_xor(b, o);
  if ((threadIdx.x & 63) == 0) {
    bits[c] = b & 0xFFFFFu;
    if (zc) zc[c] = b >> 20;
  }
}

template <class Src>
__device__ __forceinline__ void run_encode_wave(const Src& src, size_t c, bool live, uint64_t b0, uint64_t nbits,
                                                const uint64_t* __restrict__ code, const uint8_t* __restrict__ len,
                                                uint32_t* __restrict__ words, uint32_t* st, uint16_t* lds) {
  static_assert(64 * Src::kRun * 64 < 1 << 20 && 64 * Src::kRun < 1 << 12, "bits and zeros share a word");
  const int lane = threadIdx.x & 63;
  const uint32_t sh = (uint32_t)(b0 & 31), nw = (uint32_t)((sh + nbits + 31) >> 5);
  const bool direct = nw > kRunWords;
  if (!direct)
    for (uint32_t k = lane; k < nw; k += 64) st[k] = 0;
  if (live) src.stage(c, lds);
  __syncthreads();
  uint32_t* const w0 = words + (b0 >> 5);
  if (live) {
    uint32_t sym[Src::kRun], l[Src::kRun], hi[Src::kRun];
    const int ns = src.load(c, lds, sym);
    const auto code32 = glob((const uint32_t*)code);
#pragma unroll
    for (int k = 0; k < Src::kRun; k++) {
      l[k] = glob(len)[sym[k]];
      hi[k] = code32[2 * (size_t)sym[k] + 1];
    }
    uint32_t b = 0;
#pragma unroll
    for (int k = 0; k < Src::kRun; k++) {
      l[k] = k < ns ? l[k] : 0u;
      b += l[k];
      if constexpr (HasUnpred<Src>::value) b += k < ns && sym[k] == 0 ? 1u << 20 : 0u;
    }
    const uint32_t before = wave_incl_scan(b) - b;
    if constexpr (HasUnpred<Src>::value) {
      if (src.unp) {
        // the chunk's unpredictable values, at its offset among the stream's
        uint64_t o = glob(src.uoff)[c] - glob(src.uoff)[0] + (before >> 20);
        if (b >> 20) {
#pragma unroll
          for (int k = 0; k < Src::kRun; k++)
            if (k < ns && sym[k] == 0) glob(src.unp)[o++] = glob(src.x)[src.elem(c, k)];
        }
      }
    }
    const uint32_t pos = sh + (before & 0xFFFFFu);
    uint32_t wi = pos >> 5, fill = pos & 31, acc = 0;
    auto out = [&](uint32_t x) {
      if (direct) atomicOr(&w0[wi], bswap32(x));
      else atomicOr(&st[wi], x);
    };
    // n <= 32 bits from the top of x
    auto push = [&](uint32_t x, uint32_t n) {
      acc |= x >> fill;
      const uint32_t f = fill + n;
      if (f >= 32) {
        out(acc);
        wi++;
        acc = __builtin_amdgcn_alignbit(x, 0u, fill);  // what did not fit
      }
      fill = f & 31;
    };
#pragma unroll
    for (int k = 0; k < Src::kRun; k++) {
      push(l[k] ? hi[k] : 0u, min(l[k], 32u));
      if (l[k] > 32) push(code32[2 * (size_t)sym[k]], l[k] - 32);
    }
    if (fill) out(acc);
  }
  __syncthreads();
  if (live && !direct) {
    const bool tail_shared = ((b0 + nbits) & 31) != 0;
    for (uint32_t k = lane; k < nw; k += 64) {
      const uint32_t word = bswap32(st[k]);
      if ((k == 0 && sh != 0) || (k == nw - 1 && tail_shared)) atomicOr(&w0[k], word);
      else glob(w0)[k] = word;
    }
  }
}

template <class Src>
__global__ void __launch_bounds__(kEncThreads) k_run_bits(const EncJob<Src>* __restrict__ jobs, int nj) {
  __shared__ __align__(16) uint16_t lds[kEncWaves][Src::kLds];
  const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
  const EncJob<Src>& J = jobs[job_of(jobs, nj, b)];
  const int wv = threadIdx.x >> 6;
  const size_t c = (size_t)(b - J.blk0) * kEncWaves + wv;
  const bool live = c < J.nchunks;  // uniform per wave
  const Src src = J.src;  // (LDS stores may alias what a reference reaches)
  if (live) src.stage(c, lds[wv]);
  __syncthreads();
  if (live) run_bits_wave(src, c, J.len, J.bits, J.zc, lds[wv]);
}

template <class Src>
__global__ void __launch_bounds__(kEncThreads) k_run_encode(const EncJob<Src>* __restrict__ jobs, int nj) {
  __shared__ __align__(16) uint16_t lds[kEncWaves][Src::kLds];
  __shared__ uint32_t stage[kEncWaves][kRunWords];
  const uint32_t b = xcd_block(blockIdx.x, gridDim.x);
  const EncJob<Src>& J = jobs[job_of(jobs, nj, b)];
  if (!J.words) return;  // a stream without an output array is skipped (whole block)
  const int wv = threadIdx.x >> 6;
  const size_t c = (size_t)(b - J.blk0) * kEncWaves + wv;
  const bool live = c < J.nchunks;
  const Src src = J.src;
  run_encode_wave(src, c, live, live ? J.off[c] - J.off[0] : 0, live ? J.bits[c] : 0, J.code, J.len, J.words,
                  stage[wv], lds[wv]);
}

// One Huffman tree built on the device (huff_tree.hip) from a histogram's
// present symbols: syms/freqs + *base hold *count (symbol, count) pairs in
// increasing symbol order. Outputs: the serialized tree (13 * (2k - 1) + 1
// bytes at most), the dense codebook code[sym] / len[sym], and info = {node
// count, tree bytes, longest code, error (0 = none)}. heap (max_leaves + 1
// words) is scratch for trees too large for LDS (more than 8190 leaves).
// Errors: 1 empty, 2 more leaves than max_leaves (or beyond 2^23), 3 a symbol
// at or beyond state_num, 4 a code longer than 64 bits, 5 internal.
struct TreeJob {
  const uint32_t* syms;
  const uint32_t* freqs;
  const uint32_t* count;
  const uint64_t* base;
  uint32_t state_num, max_leaves;
  uint64_t* heap;
  uint8_t* tree;
  uint64_t* code;
  uint8_t* len;
  uint64_t* info;
};
__global__ void k_huff_tree(const TreeJob* jobs);
void build_trees_device(Ctx& ctx, const TreeJob* d_jobs, int ntrees);

__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t v);
__global__ void k_scatter_codebook(const uint32_t* syms, const uint64_t* codes, const uint8_t* lens,
                                   int k, uint64_t* code, uint8_t* len);

// ------------------------------------------------------------------ decode --
struct DecTree {
  const uint32_t* lut;    // 2^kLutBits entries
  const uint32_t* lut2;   // level-2 tables (huff_build_lut)
  const uint32_t* left;   // node arrays (preorder numbering)
  const uint32_t* right;
  const uint32_t* sym;
  const uint8_t* leaf;
  uint32_t nodes;
};

typedef __attribute__((address_space(3))) const uint32_t lds_u32;  // an LDS word

// A block decodes 256 segments: their 2048 words, the words before them (the
// first segment's warm-up) and a few past them (the last code's overrun, 64
// bits, and one window) are staged in LDS, zeros beyond the stream. A staged
// word is bit-reversed, the stream's first bit lowest, so that the 32 bits
// from any position are one funnel shift of two neighbouring words: no bit
// buffer to refill, 32-bit positions counted from the first staged bit, and no
// read outside LDS.
constexpr uint32_t kPreWords = kWarmBits / 32;
constexpr uint32_t kStageWords = kPreWords + 256 * (kSegBits / 32) + 8;

struct BlockBits {
  lds_u32* w;
  __device__ __forceinline__ uint32_t window(uint32_t p) const {
    return __builtin_amdgcn_alignbit(w[(p >> 5) + 1], w[p >> 5], p & 31);
  }
};

// Stages the words of segments [b0, b0 + 256); returns the position of the
// first of them. Callers synchronize.
__device__ __forceinline__ uint32_t stage_words(uint32_t* sw, const uint32_t* __restrict__ w, uint64_t nbits,
                                                uint32_t b0) {
  const uint32_t pre = b0 ? kPreWords : 0;
  const uint64_t base = (uint64_t)b0 * (kSegBits / 32) - pre, have = (nbits + 31) / 32;
  for (uint32_t k = threadIdx.x; k < kStageWords; k += blockDim.x)
    sw[k] = base + k < have ? __brev(bswap32(w[base + k])) : 0u;
  return pre * 32;
}

// The level-1 table in the order of the windows' low bits. Callers synchronize.
__device__ __forceinline__ void stage_lut(uint32_t* slut, const uint32_t* __restrict__ lut) {
  for (uint32_t k = threadIdx.x; k < (1u << kLutBits); k += blockDim.x) slut[__brev(k) >> (32 - kLutBits)] = lut[k];
}

constexpr uint32_t kLutMask = (1u << kLutBits) - 1;

// A level-1 entry is sym << 8 | length for short codes, off << 8 | 0x80 | K for
// prefixes continued by a level-2 table (t.lut2, global memory) over the next
// K bits; codes longer still continue bit by bit down the tree.
__device__ __forceinline__ bool short_code(uint32_t e) { return (e & 0xFF) - 1 < 0x7F; }

// The rest of the code whose level-1 entry at p is e: its symbol, or
// 0xFFFFFFFF for a bad code. p moves past it, 64 bits at most.
__device__ __forceinline__ uint32_t long_code(const DecTree& t, const BlockBits& bits, uint32_t e, uint32_t& p) {
  uint32_t node = e >> 8;
  p += kLutBits;
  if (e & 0x80u) {
    const int K = (int)(e & 0x7F);
    const uint32_t e2 = t.lut2[node + (__brev(bits.window(p)) >> (32 - K))];
    const uint32_t L2 = e2 & 0xFF;
    if (L2) {
      p += L2;
      return e2 >> 8;
    }
    node = e2 >> 8;
    p += (uint32_t)K;
  }
  for (int d = 0; d < 64; d++) {
    const uint32_t b = bits.window(p) & 1;
    p++;
    node = b ? t.right[node] : t.left[node];
    if (node == 0 || node >= t.nodes) return 0xFFFFFFFFu;
    if (t.leaf[node]) return t.sym[node];
  }
  return 0xFFFFFFFFu;
}

// Decodes one symbol (0xFFFFFFFF: a bad code).
__device__ __forceinline__ uint32_t dec_one(const DecTree& t, const uint32_t* slut, const BlockBits& bits, uint32_t& p) {
  const uint32_t e = slut[bits.window(p) & kLutMask];
  if (short_code(e)) {
    p += e & 0xFF;
    return e >> 8;
  }
  return long_code(t, bits, e, p);
}

// Multi-code steps for the passes that only locate code boundaries: for each
// kLutBits-bit window, the number n of whole codes (each at most kLutBits
// bits, decoded greedily from the window's start) and their total length,
// stored as n << 8 | length (0 when the first code is longer). Built from the
// level-1 table in LDS by the whole block; callers synchronize before use.
__device__ __forceinline__ void build_mstep(const uint32_t* slut, uint16_t* ms) {
  for (uint32_t w = threadIdx.x; w <= kLutMask; w += blockDim.x) {
    uint32_t pos = 0, n = 0;
    for (;;) {
      const uint32_t e = slut[w >> pos];
      if (!short_code(e) || pos + (e & 0xFF) > (uint32_t)kLutBits) break;
      pos += e & 0xFF;
      n++;
    }
    ms[w] = (uint16_t)(n << 8 | pos);
  }
}

// Decodes from p up to the first code boundary at or after `stop`, adding the
// number of codes to c: a window's run of short codes at a time (two from one
// fetch) while the run ends at or before `stop` (so no boundary at or after
// `stop` is stepped over), one code at a time otherwise. False on a bad code.
__device__ __forceinline__ bool dec_until(const DecTree& t, const uint32_t* slut, const uint16_t* ms,
                                          const BlockBits& bits, uint32_t& p, uint32_t stop, uint32_t& c) {
  while (p < stop) {
    const uint32_t win = bits.window(p);
    const uint32_t m = ms[win & kLutMask], len = m & 0xFF;
    if (len && p + len <= stop) {
      p += len;
      c += m >> 8;
      const uint32_t m2 = ms[(win >> len) & kLutMask], len2 = m2 & 0xFF;
      if (p + len2 <= stop) {  // (nothing to add if the next code is a long one)
        p += len2;
        c += m2 >> 8;
      }
      continue;
    }
    const uint32_t e = slut[win & kLutMask];
    if (short_code(e)) p += e & 0xFF;
    else if (long_code(t, bits, e, p) == 0xFFFFFFFFu) return false;
    c++;
  }
  return true;
}

// Multi-code decode for streams whose symbols fit a byte: for each window,
// up to 3 whole short codes: length | n << 4 | sym0 << 8 | sym1 << 16 | sym2 << 24
// (n = 0 when the first code is longer than the window).
__device__ __forceinline__ void build_mdec8(const uint32_t* slut, uint32_t* md) {
  for (uint32_t w = threadIdx.x; w <= kLutMask; w += blockDim.x) {
    uint32_t pos = 0, n = 0, syms = 0;
    while (n < 3) {
      const uint32_t e = slut[w >> pos];
      if (!short_code(e) || pos + (e & 0xFF) > (uint32_t)kLutBits || (e >> 8) > 0xFFu) break;
      syms |= (e >> 8) << (8 * n);
      pos += e & 0xFF;
      n++;
    }
    md[w] = pos | n << 4 | syms << 8;
  }
}

// ---- finding the code boundaries. A segment's start (its first code boundary)
// depends on everything before it, but only a few starts are possible: those
// that some path reaches from one of the max_len bit positions kWarmBits
// earlier. Paths merge within a few codes, so mostly one is left; where codes of
// one length follow each other (runs of one symbol, near-uniform alphabets) up
// to that length stay apart, however far back one begins, and a guessed start
// would be wrong for the whole run.
//   k_dec_cand    per segment: its possible starts, and from each the exit (first
//                 boundary at or past the segment's end) and the code count
//   k_dec_serial  streams in which some segment has more than kCand starts: the
//                 true chain, one segment after the other
//   k_dec_follow  per block of 256 segments: where each start of its first
//                 segment leads, and the counts on the way
//   k_dec_chain   per stream: the true start and output offset of every block
// No pass waits for the host, and the result does not depend on how fast the
// codes resynchronize.
struct MDecJob {
  DecTree t;
  const uint32_t* w;
  uint64_t nbits, n;
  uint32_t nseg, nblk, blk0, max_len;
  uint64_t* mask;   // per segment: possible starts (bit o: o bits past its beginning)
  uint8_t* st;      // [kCand][nseg] the same as offsets
  uint8_t* ex;      // [kCand][nseg] exit, bits past the segment's end
  uint16_t* cnt;    // [kCand][nseg] codes
  uint64_t* sel;    // per segment: the start (4 bits) that each start of its block's first segment leads to
  uint64_t* bmap;   // per block: the next block's start for each of its own (4 bits each)
  uint32_t* btot;   // [nblk][kCand] codes from each
  uint32_t* bsel;   // per block: the true start; bit 31: all its segments have one start
  uint64_t* boff;   // per block: the first code's position
};
template <class Sink>
struct MDecJobS {
  MDecJob j;
  Sink sink;
};
// A table of MDecJob at the start of larger elements.
struct MDecTable {
  const char* base;
  size_t stride;
  const uint32_t* blk0;  // first block of each job, nj + 1 entries
  int nj;
  __device__ __forceinline__ const MDecJob& operator[](int j) const { return *(const MDecJob*)(base + (size_t)j * stride); }
  __device__ __forceinline__ int of_block(uint32_t b) const {
    int lo = 0, hi = nj - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (blk0[mid] <= b) lo = mid;
      else hi = mid - 1;
    }
    return lo;
  }
};
__global__ void k_dec_cand(MDecTable jobs, int* err, int* over);
__global__ void k_dec_serial(MDecTable jobs, int* err, const int* over);
__global__ void k_dec_follow(MDecTable jobs);
__global__ void k_dec_chain(MDecTable jobs, uint64_t* totals);

// Decode every segment into its final position. The symbols of a
// block's 256 consecutive segments are contiguous in the output: they are
// gathered in LDS and written out by consecutive threads (coalesced), instead
// of each thread storing its own run one symbol at a time (64 scattered
// 2-byte stores per instruction, which reach HBM as ~15x the bytes), a
// stage's worth after the other. Sink::kBytes (1 or 2)
// is the width of a staged symbol. Bound by the decode's LDS latency, then by
// the sinks' index arithmetic. 96 fields' ids 1.85 -> 1.56 ms and codes
// 2.97 -> 2.38 ms with several codes from one fetched window in place of a bit
// buffer refilled under a branch; 1.25 and 2.22 ms with stages small enough for
// three blocks a CU, taken in turn (ids at 1.5 bits a code make 44000 symbols a
// block, which a stage of 32768 left to scattered stores).
template <int kBytes>
struct DecStage {
  using T = typename std::conditional<kBytes == 1, uint8_t, uint16_t>::type;
  static constexpr uint32_t kCap = kBytes == 1 ? 24576 : 12288;  // symbols at a time: three blocks a CU
};

// Exclusive scan of the block's 256 values (x of thread 255 is the last);
// tot receives the sum.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, uint32_t* wsum, uint32_t& tot) {
  const uint32_t incl = wave_incl_scan(x);
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 63) wsum[wv] = incl;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t v = wsum[k];
    before += k < wv ? v : 0u;
    all += v;
  }
  tot = all;
  return before + incl - x;
}

template <class Sink>
__device__ __forceinline__ void dec_write_block(const MDecJob& J, const Sink& sink, uint32_t blk, uint32_t* slut,
                                                uint32_t* sw, typename DecStage<Sink::kBytes>::T* stage, uint32_t* md,
                                                uint32_t* wsum) {
  using Stage = DecStage<Sink::kBytes>;
  const DecTree t = J.t;  // (and the sink below: LDS stores may alias what a reference reaches)
  const Sink out = sink;
  stage_lut(slut, t.lut);
  const uint32_t b0 = blk * 256, i = b0 + threadIdx.x;
  const BlockBits bits{(lds_u32*)sw};
  const uint32_t pre = stage_words(sw, J.w, J.nbits, b0);
  // the segment's start, exit and count on the true chain
  uint32_t p = 0, end = 0, codes = 0;
  const uint32_t bs = J.bsel[blk];
  if (i < J.nseg) {
    const uint32_t c = bs >> 31 ? 0u : (uint32_t)(J.sel[i] >> (4 * bs)) & 15u;
    const size_t at = (size_t)c * J.nseg + i;
    p = pre + threadIdx.x * kSegBits + J.st[at];
    end = pre + (uint32_t)(min((uint64_t)(i + 1) * kSegBits, J.nbits) - (uint64_t)b0 * kSegBits) + J.ex[at];
    codes = J.cnt[at];
  }
  const uint64_t n = J.n, first = J.boff[blk];
  uint32_t tot;
  uint32_t o = block_excl_scan(codes, wsum, tot);  // synchronizes
  if (first >= n) return;
  if (Sink::kBytes == 1) {
    build_mdec8(slut, md);
    __syncthreads();
  }
  const uint32_t limit = (uint32_t)min((uint64_t)tot, n - first);
  using S = typename Stage::T;
  // (o0 and o1 are uniform; a lane's run may span two stages)
  for (uint32_t o0 = 0; o0 < limit; o0 += Stage::kCap) {
    const uint32_t o1 = min(limit, o0 + Stage::kCap);
    if (Sink::kBytes == 1) {
      // up to 6 codes per fetch while they all start before `end` and fit
      while (p < end && o < o1) {
        uint32_t win = bits.window(p);
        bool none = true;
#pragma unroll
        for (int r = 0; r < 2; r++) {
          const uint32_t m = md[win & kLutMask];
          const uint32_t len = m & 0xF, k = (m >> 4) & 3;
          if (!k || p + len > end || o + k > o1) break;
          S* d = stage + (o - o0);
          d[0] = (S)(m >> 8);
          if (k > 1) d[1] = (S)(m >> 16);
          if (k > 2) d[2] = (S)(m >> 24);
          o += k;
          p += len;
          win >>= len;
          none = false;
        }
        if (none) stage[o++ - o0] = (S)dec_one(t, slut, bits, p);
      }
    } else {
      // up to 3 codes per fetch
      while (p < end && o < o1) {
        const uint32_t win = bits.window(p);
        uint32_t e = slut[win & kLutMask];
        if (!short_code(e)) {
          stage[o++ - o0] = (S)long_code(t, bits, e, p);
          continue;
        }
        uint32_t used = e & 0xFF;
        stage[o++ - o0] = (S)(e >> 8);
        p += used;
#pragma unroll
        for (int r = 0; r < 2; r++) {
          e = slut[(win >> used) & kLutMask];
          if (p >= end || o >= o1 || !short_code(e) || used > 32 - kLutBits) break;
          stage[o++ - o0] = (S)(e >> 8);
          used += e & 0xFF;
          p += e & 0xFF;
        }
      }
    }
    __syncthreads();
    for (uint32_t x = o0 + threadIdx.x; x < o1; x += blockDim.x) out.put(first + x, stage[x - o0]);
    __syncthreads();
  }
}

template <class Sink>
__global__ void __launch_bounds__(256) k_dec_write(MDecTable jobs) {
  __shared__ uint32_t slut[1 << kLutBits];
  __shared__ uint32_t sw[kStageWords];
  __shared__ typename DecStage<Sink::kBytes>::T stage[DecStage<Sink::kBytes>::kCap];
  __shared__ uint32_t md[Sink::kBytes == 1 ? (1 << kLutBits) : 1];
  __shared__ uint32_t wsum[4];
  const int j = jobs.of_block(blockIdx.x);
  const MDecJobS<Sink>& J = *(const MDecJobS<Sink>*)&jobs[j];
  dec_write_block(J.j, J.sink, blockIdx.x - J.j.blk0, slut, sw, stage, md, wsum);
}

template <class Sink>
__global__ void k_dec_const(uint64_t n, uint32_t s, Sink sink) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    sink.put(i, s);
}

// --------------------------------------------------------- host helpers ----
// Exclusive scan of u64 counts (rocPRIM), writing the total to *d_total.
void scan_u64(Ctx& ctx, const uint64_t* in, uint64_t* out, size_t n, uint64_t* d_total);
void scan_u32_to_u64(Ctx& ctx, const uint32_t* in, uint64_t* out, size_t n, uint64_t* d_total);

// Uploads an encode table into dense device tables (code, len) over nbins.
void upload_codebook(Ctx& ctx, const HuffEncodeTable& t, uint64_t* d_code, uint8_t* d_len,
                     const char* tag);

struct DeviceDecoder {
  DecTree tree{};
  uint32_t max_len = 0;  // longest code
  bool single = false;
  uint32_t single_sym = 0;
};
// Parses a serialized tree and uploads the decode tables (tag names the buffers).
// The host half of a decoder: the parsed tree and the level-1 / level-2
// tables. prepare_decoder makes no HIP call, so it can run on another thread
// while the device works.
struct HostDecoder {
  HuffDecodeTree d;
  std::vector<uint32_t> lut, pfx;
  size_t n2 = 0;  // level-2 entries
};
void prepare_decoder(const uint8_t* tree, size_t tree_size, size_t node_count, HostDecoder& h);
DeviceDecoder upload_decoder(Ctx& ctx, const HostDecoder& h, const char* tag);
DeviceDecoder upload_decoder(Ctx& ctx, const uint8_t* tree, size_t tree_size, size_t node_count,
                             const char* tag);

// Many decoders in one packed copy and one level-2 fill launch (out[k] for
// hd[k]); `tag` names the buffers.
// pool (optional): host workers that share the table copies (the caller must
// not itself be running on that pool)
class WorkerPool;
void upload_decoders(Ctx& ctx, const HostDecoder* const* hd, int n, DeviceDecoder* out, const char* tag,
                     WorkerPool* pool = nullptr, int workers = 0);

// Bitstreams at arbitrary byte offsets copied into aligned word arrays with
// zero slack (the decoder's input form), all in one launch. Fills dst/nwords.
struct BitsCopy {
  const uint8_t* src;
  uint64_t nbytes;
  uint32_t* dst;
  uint64_t nwords;
};
constexpr uint32_t kStageBlockWords = 2048;
void stage_bits_multi(Ctx& ctx, BitsCopy* c, int n, const char* tag);

// One bitstream to decode: n symbols of words already copied to aligned
// device words (padded with at least 8 zero words) into `sink`.
template <class Sink>
struct DecJob {
  const DeviceDecoder* dd;
  const uint32_t* words;
  uint64_t nbytes, n;
  Sink sink;
};

// What a decode found, to be looked at once the stream has passed it.
struct DecodeResult {
  const uint64_t* totals = nullptr;  // pinned: codes found per stream
  const int* err = nullptr;          // pinned
  std::vector<uint64_t> want;
  void check() const {
    for (size_t k = 0; k < want.size(); k++) {
      CPSZ_REQUIRE(err[k] == 0, kErrStream, "invalid huffman code in stream");
      CPSZ_REQUIRE(totals[k] >= want[k], kErrStream, "huffman bitstream holds fewer symbols than expected");
    }
  }
};

// Waits for the stream when a call is left by an exception, so that nothing
// queued still reads the caller's buffers after it.
struct SettleOnThrow {
  hipStream_t st;
  int before = std::uncaught_exceptions();
  ~SettleOnThrow() {
    if (std::uncaught_exceptions() > before) (void)hipStreamSynchronize(st);
  }
};

// Decodes many independent bitstreams, every stream's segments in one grid per
// pass. Queues all passes on the context's stream and returns without waiting;
// whatever the streams hold, the sinks get positions below n only. `tag` names
// the buffers: one decode per tag until its result has been checked.
template <class Sink>
DecodeResult decode_streams(Ctx& ctx, const DecJob<Sink>* jobs, int nj, const char* tag) {
  hipStream_t st = ctx.stream();
  DecodeResult res;
  std::vector<int> act;
  for (int k = 0; k < nj; k++) {
    const DecJob<Sink>& j = jobs[k];
    if (j.n == 0) continue;
    if (j.dd->single) {
      k_dec_const<<<(unsigned)std::min<uint64_t>(div_up(j.n, (uint64_t)256), 1024), 256, 0, st>>>(
          j.n, j.dd->single_sym, j.sink);
      CPSZ_HIP(hipGetLastError());
      continue;
    }
    CPSZ_REQUIRE(j.nbytes > 0, kErrStream, "empty huffman bitstream for a multi-symbol tree");
    act.push_back(k);
  }
  const int na = (int)act.size();
  if (!na) return res;
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  const std::string t(tag);
  // the job table, block starts and (zero) flags travel in one copy
  const size_t tb = al(na * sizeof(MDecJobS<Sink>)), bb = al((na + 1) * 4), fb = al(2 * na * 4), ob = na * 8;
  uint8_t* hh = (uint8_t*)ctx.host_table((t + ".tab").c_str(), tb + bb + fb);
  uint8_t* dt = ctx.buf<uint8_t>((t + ".tab").c_str(), tb + bb + fb + ob);
  MDecJobS<Sink>* h = (MDecJobS<Sink>*)hh;
  uint32_t* blk0 = (uint32_t*)(hh + tb);
  blk0[0] = 0;
  size_t arena = 0;
  for (int a = 0; a < na; a++) {
    const DecJob<Sink>& j = jobs[act[a]];
    MDecJob& m = h[a].j;
    m = MDecJob{};
    m.t = j.dd->tree;
    m.max_len = j.dd->max_len;
    m.w = j.words;
    m.nbits = j.nbytes * 8;
    m.n = j.n;
    const uint64_t nseg = div_up(m.nbits, (uint64_t)kSegBits);
    CPSZ_REQUIRE(nseg < (1ull << 31) && (uint64_t)blk0[a] + div_up(nseg, (uint64_t)256) < (1ull << 31), kErrUnsupported,
                 "huffman decode: too many segments");
    m.nseg = (uint32_t)nseg;
    m.nblk = (uint32_t)div_up(m.nseg, 256u);
    m.blk0 = blk0[a];
    blk0[a + 1] = blk0[a] + m.nblk;
    h[a].sink = j.sink;
    res.want.push_back(j.n);
    arena += 2 * al(8 * (size_t)m.nseg) + 2 * al(kCand * (size_t)m.nseg) + al(2 * kCand * (size_t)m.nseg) +
             2 * al(8 * (size_t)m.nblk) + al(4 * kCand * (size_t)m.nblk) + al(4 * (size_t)m.nblk);
  }
  uint8_t* d = ctx.buf<uint8_t>((t + ".arena").c_str(), arena);
  for (int a = 0; a < na; a++) {
    MDecJob& m = h[a].j;
    auto take = [&](size_t bytes) {
      uint8_t* q = d;
      d += al(bytes);
      return q;
    };
    m.mask = (uint64_t*)take(8 * (size_t)m.nseg);
    m.sel = (uint64_t*)take(8 * (size_t)m.nseg);
    m.st = (uint8_t*)take(kCand * (size_t)m.nseg);
    m.ex = (uint8_t*)take(kCand * (size_t)m.nseg);
    m.cnt = (uint16_t*)take(2 * kCand * (size_t)m.nseg);
    m.bmap = (uint64_t*)take(8 * (size_t)m.nblk);
    m.boff = (uint64_t*)take(8 * (size_t)m.nblk);
    m.btot = (uint32_t*)take(4 * kCand * (size_t)m.nblk);
    m.bsel = (uint32_t*)take(4 * (size_t)m.nblk);
  }
  std::memset(hh + tb + bb, 0, fb);
  const uint32_t nblocks = blk0[na];
  ctx.upload_table((t + ".tab").c_str(), dt, hh, tb + bb + fb);
  const MDecTable tab{(const char*)dt, sizeof(MDecJobS<Sink>), (const uint32_t*)(dt + tb), na};
  int* err = (int*)(dt + tb + bb);
  int* over = err + na;
  uint64_t* totals = (uint64_t*)(dt + tb + bb + fb);
  k_dec_cand<<<nblocks, 256, 0, st>>>(tab, err, over);
  k_dec_serial<<<na, 64, 0, st>>>(tab, err, over);
  ctx.mark((t + ".cand").c_str());
  k_dec_follow<<<nblocks, 256, 0, st>>>(tab);
  k_dec_chain<<<na, 1024, 0, st>>>(tab, totals);
  ctx.mark((t + ".chain").c_str());
  k_dec_write<Sink><<<nblocks, 256, 0, st>>>(tab);
  CPSZ_HIP(hipGetLastError());
  ctx.mark((t + ".write").c_str());
  uint8_t* hr = (uint8_t*)ctx.host_buf((t + ".res").c_str(), fb + ob);
  CPSZ_HIP(hipMemcpyAsync(hr, dt + tb + bb, fb + ob, hipMemcpyDeviceToHost, st));
  res.err = (const int*)hr;
  res.totals = (const uint64_t*)(hr + fb);
  return res;
}

// Decodes n symbols of one bitstream (see decode_streams).
template <class Sink>
DecodeResult decode_stream(Ctx& ctx, const DeviceDecoder& dd, const uint32_t* d_words, uint64_t nbytes, uint64_t n,
                           Sink sink, const char* tag) {
  DecJob<Sink> j{&dd, d_words, nbytes, n, sink};
  return decode_streams(ctx, &j, 1, tag);
}

}  // namespace cpsz
