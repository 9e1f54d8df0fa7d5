#include "huff_gpu.hpp"
#include "pool.hpp"

#include <cstring>
#include <functional>

namespace cpsz {

__global__ void k_fill_u32(uint32_t* p, size_t n, uint32_t v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_scatter_codebook(const uint32_t* syms, const uint64_t* codes, const uint8_t* lens,
                                   int k, uint64_t* code, uint8_t* len) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k) return;
  code[syms[i]] = codes[i];
  len[syms[i]] = lens[i];
}

namespace {

// Length of the code at p. (A parsed tree is full, so there always is one.)
__device__ __forceinline__ uint32_t code_len(const DecTree& t, const uint32_t* slut, const BlockBits& bits, uint32_t p) {
  const uint32_t e = slut[bits.window(p) & kLutMask];
  if (short_code(e)) return e & 0xFF;
  uint32_t q = p;
  long_code(t, bits, e, q);
  return q - p;
}

}  // namespace

// Bound by the lanes' serial walks (two LDS reads and some ten instructions a
// step). Paths are followed as a bit set of the positions that some path
// reaches, lowest first: the set spans max_len bits, and while it holds one
// position the walk goes on by runs of codes. Measured in ms, on the ids of 96
// fields of 256 to 4096 a side (1.5 bits a code): a guessed start after a
// 2048-bit warm-up 2.61, its fix-up rounds 0.80 (22 on smoother fields, whose
// runs of one id keep wrong phases alive); here 0.94, and 0.12 for the chain.
// Codes of the same fields: 2.0 and 0.3 before, 1.77 and 0.20 here. One
// 601 x 1203 log field, both decodes in all: 3.9 before, 0.4 here.
__global__ void __launch_bounds__(256) k_dec_cand(MDecTable jobs, int* __restrict__ err, int* __restrict__ over) {
  __shared__ uint32_t slut[1 << kLutBits];
  __shared__ uint32_t sw[kStageWords];
  __shared__ uint16_t ms[1 << kLutBits];
  const int j = jobs.of_block(blockIdx.x);
  const MDecJob& J = jobs[j];
  const DecTree t = J.t;
  const uint32_t b0 = (blockIdx.x - J.blk0) * 256, i = b0 + threadIdx.x;
  stage_lut(slut, t.lut);
  const BlockBits bits{(lds_u32*)sw};
  const uint32_t pre = stage_words(sw, J.w, J.nbits, b0);
  __syncthreads();
  build_mstep(slut, ms);
  __syncthreads();
  const uint32_t nseg = J.nseg;
  if (i >= nseg) return;
  const uint32_t a = pre + threadIdx.x * kSegBits;
  const uint32_t end = a + (uint32_t)min((uint64_t)kSegBits, J.nbits - (uint64_t)i * kSegBits);
  uint32_t p = i ? a - kWarmBits : a;
  uint64_t m = i > 1 ? ~0ull >> (64 - J.max_len) : 1;  // positions from p on (max_len is 1 to 64)
  while (p < a) {
    if (m == 1) {
      uint32_t skipped = 0;
      dec_until(t, slut, ms, bits, p, a, skipped);
      break;
    }
    m = m >> 1 | 1ull << (code_len(t, slut, bits, p) - 1);
    const uint32_t s = (uint32_t)__ffsll((long long)m);  // on to the next position, 64 at most
    m >>= s - 1;
    p += s;
  }
  // every position is now in [a, a + max_len)
  m <<= p - a;
  uint32_t n = (uint32_t)__popcll(m);
  if (n > (uint32_t)kCand) {
    over[j] = 1;
    n = kCand;
  }
  J.mask[i] = m;
  uint8_t* const st = J.st;
  uint8_t* const ex = J.ex;
  uint16_t* const cnt = J.cnt;
  for (uint32_t k = 0; k < n; k++) {
    const uint32_t o = (uint32_t)__ffsll((long long)m) - 1;
    m &= m - 1;
    p = a + o;
    uint32_t c = 0;
    if (!dec_until(t, slut, ms, bits, p, end, c)) err[j] = 1;
    const size_t at = (size_t)k * nseg + i;
    st[at] = (uint8_t)o;
    ex[at] = (uint8_t)(p > end ? p - end : 0);
    cnt[at] = (uint16_t)c;
  }
}

// One wave per stream; leaves at once unless the stream needs it. Lane 0 walks
// the whole stream, so each of its segments has its one true start, at 1.7 us a
// code (1744 ms for 10^6 codes of 17 bits; of 16 bits, without it, 1.2). It takes
// runs of codes above 16 bits and of one length: streams made for it, as uniform
// noise (2400 x 3600, at bounds from 0.1 down to 1e-5) does not come to it.
__global__ void __launch_bounds__(64) k_dec_serial(MDecTable jobs, int* __restrict__ err, const int* __restrict__ over) {
  __shared__ uint32_t slut[1 << kLutBits];
  __shared__ uint32_t sw[kStageWords];
  const int j = blockIdx.x;
  const MDecJob& J = jobs[j];
  if (!over[j]) return;
  stage_lut(slut, J.t.lut);
  const BlockBits bits{(lds_u32*)sw};
  uint32_t o = 0;  // the next code, bits past the block's beginning
  for (uint32_t b0 = 0; b0 < J.nseg; b0 += 256) {
    const uint32_t pre = stage_words(sw, J.w, J.nbits, b0);
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t p = pre + o;
      for (uint32_t i = b0; i < min(b0 + 256, J.nseg); i++) {
        const uint32_t a = pre + (i - b0) * kSegBits;
        const uint32_t end = a + (uint32_t)min((uint64_t)kSegBits, J.nbits - (uint64_t)i * kSegBits);
        J.mask[i] = 1;
        J.st[i] = (uint8_t)(p - a);
        uint32_t c = 0;
        while (p < end) {
          if (dec_one(J.t, slut, bits, p) == 0xFFFFFFFFu) {  // a bad code: the call fails, the walk ends
            err[j] = 1;
            p = end;
          }
          c++;
        }
        J.ex[i] = (uint8_t)(p - end);
        J.cnt[i] = (uint16_t)c;
      }
      o = p - (pre + 256 * kSegBits);
    }
    __syncthreads();
  }
}

// Where each possible start of a block's first segment leads. Most blocks hold
// one start per segment: their counts are a sum. In the others lane k of the
// first wave follows start k through the 256 segments, a table look-up each.
__global__ void __launch_bounds__(256) k_dec_follow(MDecTable jobs) {
  __shared__ uint64_t nx[256];            // the next segment's start for each of the segment's (4 bits each)
  __shared__ uint16_t cn[kCand][256];
  __shared__ uint8_t path[256][kCand];    // [segment][start of the block]
  __shared__ uint8_t leads[kCand];
  __shared__ int n_first;
  __shared__ uint32_t wsum[4];
  const MDecJob& J = jobs[jobs.of_block(blockIdx.x)];
  const uint32_t blk = blockIdx.x - J.blk0, i = blk * 256 + threadIdx.x;
  const uint32_t last = min(255u, J.nseg - 1 - blk * 256);  // last segment of the block
  const bool valid = i < J.nseg;
  const uint64_t m = valid ? J.mask[i] : 1, m1 = valid && i + 1 < J.nseg ? J.mask[i + 1] : 1;
  const int n = min(__popcll(m), kCand);
  auto next = [&](uint32_t e) { return m1 & (m1 - 1) ? (uint64_t)min(__popcll(m1 & ((1ull << e) - 1)), kCand - 1) : 0; };
  uint64_t nxt = 0;
  for (int k = 0; k < n; k++)
    if (valid) nxt |= next(min((uint32_t)J.ex[(size_t)k * J.nseg + i], 63u)) << (4 * k);
  if (!__syncthreads_or(n > 1)) {
    uint32_t tot;
    block_excl_scan(valid ? J.cnt[i] : 0u, wsum, tot);
    if (threadIdx.x == last) J.bmap[blk] = nxt;
    if (threadIdx.x == 0) {
      J.btot[(size_t)blk * kCand] = tot;
      J.bsel[blk] = 1u << 31;
    }
    return;
  }
  nx[threadIdx.x] = nxt;
  for (int k = 0; k < n; k++) cn[k][threadIdx.x] = valid ? J.cnt[(size_t)k * J.nseg + i] : 0;
  if (threadIdx.x == 0) n_first = n;
  __syncthreads();
  if (threadIdx.x < (uint32_t)n_first) {
    uint32_t cur = threadIdx.x, tot = 0;
    for (uint32_t s = 0; s <= last; s++) {
      path[s][threadIdx.x] = (uint8_t)cur;
      tot += cn[cur][s];
      cur = (uint32_t)(nx[s] >> (4 * cur)) & 15u;
    }
    J.btot[(size_t)blk * kCand + threadIdx.x] = tot;
    leads[threadIdx.x] = (uint8_t)cur;
  }
  __syncthreads();
  uint64_t p = 0;
  if (valid) {
    for (int k = 0; k < n_first; k++) p |= (uint64_t)path[threadIdx.x][k] << (4 * k);
    J.sel[i] = p;
  }
  if (threadIdx.x == 0) {
    p = 0;
    for (int k = 0; k < n_first; k++) p |= (uint64_t)leads[k] << (4 * k);
    J.bmap[blk] = p;
    J.bsel[blk] = 0;
  }
}

// The true chain over a stream's blocks, 64 to a wave and 1024 at a time. Each
// wave first composes its blocks' maps (lane e follows entry e, the maps come
// by lane reads), the waves' maps then give every wave its entry, and it
// follows its blocks once more from there; the lanes fetch the chosen totals
// and sum them. One wave alone, 64 blocks after the other, took 0.19 ms for the
// codes of a 256^3 field.
__global__ void __launch_bounds__(1024) k_dec_chain(MDecTable jobs, uint64_t* __restrict__ totals) {
  __shared__ uint32_t leads[16][16];  // [wave][entry]
  __shared__ uint64_t sum[16];
  const MDecJob& J = jobs[blockIdx.x];
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6, nblk = J.nblk;
  uint32_t cur = 0;
  uint64_t pos = 0;
  for (uint32_t b0 = 0; b0 < nblk; b0 += 1024) {
    const uint32_t b = b0 + threadIdx.x;
    // lanes past the last block lead nowhere and hold nothing
    const uint32_t one = b < nblk ? J.bsel[b] : 1u << 31;
    const uint64_t map = b < nblk ? J.bmap[b] : 0;
    const uint32_t lo = (uint32_t)map, hi = (uint32_t)(map >> 32);
    const bool all_one = __all(one >> 31);
    auto map_of = [&](uint32_t k) {
      return (uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, k) << 32 | (uint32_t)__builtin_amdgcn_readlane(lo, k);
    };
    uint32_t c = lane & 15;
    if (all_one) {
      c = __builtin_amdgcn_readlane(lo, 63) & 15u;
    } else {
#pragma unroll
      for (uint32_t k = 0; k < 64; k++) c = (uint32_t)(map_of(k) >> (4 * c)) & 15u;
    }
    if (lane < 16) leads[w][lane] = c;
    __syncthreads();
    uint32_t entry = 0;
    for (uint32_t q = 0; q < 16; q++) {
      entry = q == w ? cur : entry;
      cur = leads[q][cur];
    }
    uint32_t mine = 0;
    if (!all_one) {
      uint32_t e = __builtin_amdgcn_readfirstlane(entry);
#pragma unroll
      for (uint32_t k = 0; k < 64; k++) {
        mine = lane == k ? e : mine;
        e = (uint32_t)(map_of(k) >> (4 * e)) & 15u;
      }
    }
    const uint32_t tot = b < nblk ? J.btot[(size_t)b * kCand + mine] : 0u;
    const uint32_t incl = wave_incl_scan(tot);
    if (lane == 63) sum[w] = incl;
    __syncthreads();
    uint64_t before = 0, all = 0;
    for (uint32_t q = 0; q < 16; q++) {
      before += q < w ? sum[q] : 0;
      all += sum[q];
    }
    if (b < nblk) {
      J.bsel[b] = one | mine;
      J.boff[b] = pos + before + incl - tot;
    }
    pos += all;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = pos;
}

// Level-2 entry for the K bits u below `node`: sym << 8 | length of the leaf
// reached, or the node reached after K bits, node << 8.
__host__ __device__ inline uint32_t lut2_entry(const uint32_t* left, const uint32_t* right, const uint32_t* sym,
                                               const uint8_t* leaf, uint32_t node, int K, uint32_t u) {
  for (int len = 0; len < K; len++) {
    node = ((u >> (K - 1 - len)) & 1) ? right[node] : left[node];
    if (leaf[node]) return (sym[node] << 8) | (uint32_t)(len + 1);
  }
  return node << 8;
}

// Level-2 decode tables: entry e of prefix p (pfx triples (node, K, off),
// offsets ascending) walks the K bits of e - off down from node.
__global__ void k_fill_lut2(const uint32_t* __restrict__ left, const uint32_t* __restrict__ right,
                            const uint32_t* __restrict__ sym, const uint8_t* __restrict__ leaf,
                            const uint32_t* __restrict__ pfx, uint32_t npfx, uint32_t n2,
                            uint32_t* __restrict__ lut2) {
  const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n2) return;
  uint32_t lo = 0, hi = npfx - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (pfx[3 * mid + 2] <= e) lo = mid;
    else hi = mid - 1;
  }
  lut2[e] = lut2_entry(left, right, sym, leaf, pfx[3 * lo], (int)pfx[3 * lo + 1], e - pfx[3 * lo + 2]);
}

void decode_host(const uint8_t* tree, size_t tree_size, size_t node_count, const uint8_t* bits, size_t nbytes,
                 size_t n, uint32_t* out) {
  HuffDecodeTree d;
  CPSZ_REQUIRE(huff_parse_tree(tree, tree_size, node_count, d), kErrStream, "malformed huffman tree");
  if (d.root_leaf) {
    for (size_t i = 0; i < n; i++) out[i] = d.root_sym;
    return;
  }
  std::vector<uint32_t> lut, pfx;
  const size_t n2 = huff_build_lut(d, kLutBits, kLut2Bits, lut, pfx);
  std::vector<uint32_t> lut2(n2);
  for (size_t p = 0; p < pfx.size() / 3; p++)
    for (uint32_t u = 0; u < (1u << pfx[3 * p + 1]); u++)
      lut2[pfx[3 * p + 2] + u] = lut2_entry(d.left.data(), d.right.data(), d.sym.data(), d.leaf.data(),
                                            pfx[3 * p], (int)pfx[3 * p + 1], u);
  const uint64_t nbits = 8 * (uint64_t)nbytes;
  uint64_t pos = 0;
  auto peek = [&](int k) -> uint32_t {  // next k <= 32 bits, zeros past the end
    uint32_t v = 0;
    for (int b = 0; b < k; b++) {
      const uint64_t q = pos + b;
      v = (v << 1) | (q < nbits ? (bits[q >> 3] >> (7 - (q & 7))) & 1u : 0u);
    }
    return v;
  };
  for (size_t i = 0; i < n; i++) {
    const uint32_t e = lut[peek(kLutBits)];
    const uint32_t L = e & 0xFF;
    if (L && !(L & 0x80u)) {
      pos += L;
      out[i] = e >> 8;
      continue;
    }
    uint32_t node = e >> 8;
    pos += kLutBits;
    if (L & 0x80u) {
      const int K = (int)(L & 0x7F);
      const uint32_t e2 = lut2[node + peek(K)];
      if (e2 & 0xFF) {
        pos += e2 & 0xFF;
        out[i] = e2 >> 8;
        continue;
      }
      node = e2 >> 8;
      pos += K;
    }
    for (;;) {
      CPSZ_REQUIRE(pos < nbits, kErrStream, "huffman bitstream exhausted");
      node = peek(1) ? d.right[node] : d.left[node];
      pos++;
      if (d.leaf[node]) break;
    }
    out[i] = d.sym[node];
  }
}

namespace {
__global__ void k_total(const uint64_t* out, const uint64_t* in, size_t n, uint64_t* total) {
  *total = n ? out[n - 1] + in[n - 1] : 0;
}
__global__ void k_total32(const uint64_t* out, const uint32_t* in, size_t n, uint64_t* total) {
  *total = n ? out[n - 1] + in[n - 1] : 0;
}
struct U32ToU64 {
  __device__ uint64_t operator()(uint32_t x) const { return x; }
};
}  // namespace

void scan_u64(Ctx& ctx, const uint64_t* in, uint64_t* out, size_t n, uint64_t* d_total) {
  if (n == 0) {
    CPSZ_HIP(hipMemsetAsync(d_total, 0, 8, ctx.stream()));
    return;
  }
  size_t tmp = 0;
  CPSZ_HIP(rocprim::exclusive_scan(nullptr, tmp, in, out, (uint64_t)0, n, rocprim::plus<uint64_t>(),
                                   ctx.stream()));
  void* d_tmp = ctx.raw_buf("scan.tmp", tmp);
  CPSZ_HIP(rocprim::exclusive_scan(d_tmp, tmp, in, out, (uint64_t)0, n, rocprim::plus<uint64_t>(),
                                   ctx.stream()));
  k_total<<<1, 1, 0, ctx.stream()>>>(out, in, n, d_total);
  CPSZ_HIP(hipGetLastError());
}

void scan_u32_to_u64(Ctx& ctx, const uint32_t* in, uint64_t* out, size_t n, uint64_t* d_total) {
  if (n == 0) {
    CPSZ_HIP(hipMemsetAsync(d_total, 0, 8, ctx.stream()));
    return;
  }
  auto it = rocprim::make_transform_iterator(in, U32ToU64());
  size_t tmp = 0;
  CPSZ_HIP(rocprim::exclusive_scan(nullptr, tmp, it, out, (uint64_t)0, n, rocprim::plus<uint64_t>(),
                                   ctx.stream()));
  void* d_tmp = ctx.raw_buf("scan.tmp", tmp);
  CPSZ_HIP(rocprim::exclusive_scan(d_tmp, tmp, it, out, (uint64_t)0, n, rocprim::plus<uint64_t>(),
                                   ctx.stream()));
  k_total32<<<1, 1, 0, ctx.stream()>>>(out, in, n, d_total);
  CPSZ_HIP(hipGetLastError());
}

void upload_codebook(Ctx& ctx, const HuffEncodeTable& t, uint64_t* d_code, uint8_t* d_len,
                     const char* tag) {
  const int k = (int)t.syms.size();
  std::string s(tag);
  const size_t bytes = k * (4 + 8 + 1);
  uint8_t* h = (uint8_t*)ctx.host_buf((s + ".cb").c_str(), bytes);
  std::memcpy(h, t.syms.data(), 4 * k);
  std::memcpy(h + 4 * k, t.codes.data(), 8 * k);
  std::memcpy(h + 12 * k, t.lens.data(), k);
  uint8_t* d = ctx.buf<uint8_t>((s + ".cb").c_str(), bytes + 16);
  // keep the u64 array 8-byte aligned on the device: place codes first
  uint64_t* dc = (uint64_t*)d;
  uint32_t* ds = (uint32_t*)(d + 8 * (size_t)k);
  uint8_t* dl = d + 12 * (size_t)k;
  CPSZ_HIP(hipMemcpyAsync(dc, h + 4 * k, 8 * (size_t)k, hipMemcpyHostToDevice, ctx.stream()));
  CPSZ_HIP(hipMemcpyAsync(ds, h, 4 * (size_t)k, hipMemcpyHostToDevice, ctx.stream()));
  CPSZ_HIP(hipMemcpyAsync(dl, h + 12 * k, (size_t)k, hipMemcpyHostToDevice, ctx.stream()));
  k_scatter_codebook<<<(int)div_up(k, 256), 256, 0, ctx.stream()>>>(ds, dc, dl, k, d_code, d_len);
  CPSZ_HIP(hipGetLastError());
}

void prepare_decoder(const uint8_t* tree, size_t tree_size, size_t node_count, HostDecoder& h) {
  CPSZ_REQUIRE(huff_parse_tree(tree, tree_size, node_count, h.d), kErrStream,
               "malformed huffman tree in stream");
  h.n2 = h.d.root_leaf ? 0 : huff_build_lut(h.d, kLutBits, kLut2Bits, h.lut, h.pfx);
}

DeviceDecoder upload_decoder(Ctx& ctx, const HostDecoder& hd, const char* tag) {
  const HuffDecodeTree& d = hd.d;
  DeviceDecoder out;
  if (d.root_leaf) {
    out.single = true;
    out.single_sym = d.root_sym;
    return out;
  }
  out.max_len = (uint32_t)d.max_len;
  const std::vector<uint32_t>& lut = hd.lut;
  const std::vector<uint32_t>& pfx = hd.pfx;
  const size_t n2 = hd.n2;
  const size_t N = d.node_count;
  const uint32_t npfx = (uint32_t)(pfx.size() / 3);
  std::string s(tag);
  const size_t lut_b = lut.size() * 4, pfx_b = pfx.size() * 4, arr_b = N * 4;
  const size_t bytes = lut_b + pfx_b + 3 * arr_b + N;
  uint8_t* h = (uint8_t*)ctx.host_buf((s + ".dec").c_str(), bytes);
  std::memcpy(h, lut.data(), lut_b);
  if (pfx_b) std::memcpy(h + lut_b, pfx.data(), pfx_b);
  uint8_t* q = h + lut_b + pfx_b;
  std::memcpy(q, d.left.data(), arr_b);
  std::memcpy(q + arr_b, d.right.data(), arr_b);
  std::memcpy(q + 2 * arr_b, d.sym.data(), arr_b);
  std::memcpy(q + 3 * arr_b, d.leaf.data(), N);
  uint8_t* dv = ctx.buf<uint8_t>((s + ".dec").c_str(), bytes);
  CPSZ_HIP(hipMemcpyAsync(dv, h, bytes, hipMemcpyHostToDevice, ctx.stream()));
  out.tree.lut = (const uint32_t*)dv;
  const uint32_t* dpfx = (const uint32_t*)(dv + lut_b);
  const uint8_t* dq = dv + lut_b + pfx_b;
  out.tree.left = (const uint32_t*)dq;
  out.tree.right = (const uint32_t*)(dq + arr_b);
  out.tree.sym = (const uint32_t*)(dq + 2 * arr_b);
  out.tree.leaf = dq + 3 * arr_b;
  uint32_t* lut2 = ctx.buf<uint32_t>((s + ".lut2").c_str(), n2 + 1);
  out.tree.lut2 = lut2;
  if (n2) {
    k_fill_lut2<<<(int)div_up(n2, 256), 256, 0, ctx.stream()>>>(out.tree.left, out.tree.right, out.tree.sym,
                                                                 out.tree.leaf, dpfx, npfx, (uint32_t)n2, lut2);
    CPSZ_HIP(hipGetLastError());
  }
  out.tree.nodes = (uint32_t)N;
  // The pinned staging buffer is reused by the next decoder upload of the same
  // tag only after the stream has consumed it (callers synchronize per call).
  return out;
}

// ---- many decoders at once: one packed host-to-device copy and one level-2
// fill launch for all of them
namespace {
struct Lut2Fill {
  const uint32_t *left, *right, *sym, *pfx;
  const uint8_t* leaf;
  uint32_t* lut2;
  uint32_t npfx, n2;
  uint64_t e0;  // first entry of this decoder in the launch
};

__global__ void k_fill_lut2_multi(const Lut2Fill* __restrict__ f, int nf, uint64_t total) {
  const uint64_t g = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  if (g >= total) return;
  int lo = 0, hi = nf - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (f[mid].e0 <= g) lo = mid;
    else hi = mid - 1;
  }
  const Lut2Fill& d = f[lo];
  const uint32_t e = (uint32_t)(g - d.e0);
  uint32_t a = 0, b = d.npfx - 1;
  while (a < b) {
    const uint32_t mid = (a + b + 1) >> 1;
    if (d.pfx[3 * mid + 2] <= e) a = mid;
    else b = mid - 1;
  }
  d.lut2[e] = lut2_entry(d.left, d.right, d.sym, d.leaf, d.pfx[3 * a], (int)d.pfx[3 * a + 1], e - d.pfx[3 * a + 2]);
}

__global__ void k_stage_bits_multi(const BitsCopy* __restrict__ c, const uint32_t* __restrict__ blk0, int nc) {
  int lo = 0, hi = nc - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (blk0[mid] <= blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  const BitsCopy& j = c[lo];
  const uint64_t k0 = (uint64_t)(blockIdx.x - blk0[lo]) * kStageBlockWords;
  for (uint32_t t = threadIdx.x; t < kStageBlockWords; t += blockDim.x) {
    const uint64_t k = k0 + t;
    if (k >= j.nwords) break;
    const uint64_t b = 4 * k;
    uint32_t v = 0;
    if (b + 4 <= j.nbytes) {
      v = (uint32_t)j.src[b] | (uint32_t)j.src[b + 1] << 8 | (uint32_t)j.src[b + 2] << 16 |
          (uint32_t)j.src[b + 3] << 24;
    } else {
      for (int q = 0; q < 4; q++)
        if (b + q < j.nbytes) v |= (uint32_t)j.src[b + q] << (8 * q);
    }
    j.dst[k] = v;
  }
}
}  // namespace

void upload_decoders(Ctx& ctx, const HostDecoder* const* hd, int n, DeviceDecoder* out, const char* tag,
                     WorkerPool* pool, int workers) {
  hipStream_t st = ctx.stream();
  auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
  std::vector<size_t> base(n + 1, 0), l2base(n + 1, 0);
  for (int k = 0; k < n; k++) {
    const HostDecoder& h = *hd[k];
    const size_t N = h.d.root_leaf ? 0 : h.d.node_count;
    base[k + 1] = base[k] + (h.d.root_leaf ? 0 : al(h.lut.size() * 4 + h.pfx.size() * 4 + 13 * N));
    l2base[k + 1] = l2base[k] + (h.d.root_leaf ? 0 : al(4 * (h.n2 + 1)));
  }
  const std::string t(tag);
  const size_t nfill = sizeof(Lut2Fill) * (size_t)(n ? n : 1);
  uint8_t* hbuf = (uint8_t*)ctx.host_buf((t + ".h").c_str(), base[n] + nfill);
  uint8_t* dbuf = ctx.buf<uint8_t>((t + ".d").c_str(), base[n] + nfill);
  uint32_t* dl2 = ctx.buf<uint32_t>((t + ".lut2").c_str(), l2base[n] / 4 + 1);
  Lut2Fill* hf = (Lut2Fill*)(hbuf + base[n]);
  // a decoder's tables into its slot of the pinned staging buffer
  auto copy_one = [&](int k) {
    const HostDecoder& h = *hd[k];
    if (h.d.root_leaf) return;
    const size_t N = h.d.node_count, lut_b = h.lut.size() * 4, pfx_b = h.pfx.size() * 4, arr_b = N * 4;
    uint8_t* q = hbuf + base[k];
    std::memcpy(q, h.lut.data(), lut_b);
    if (pfx_b) std::memcpy(q + lut_b, h.pfx.data(), pfx_b);
    uint8_t* a = q + lut_b + pfx_b;
    std::memcpy(a, h.d.left.data(), arr_b);
    std::memcpy(a + arr_b, h.d.right.data(), arr_b);
    std::memcpy(a + 2 * arr_b, h.d.sym.data(), arr_b);
    std::memcpy(a + 3 * arr_b, h.d.leaf.data(), N);
  };
  if (pool) {
    // the copies of many decoders (megabytes) split over the host workers
    const int parts = std::max(1, std::min(workers, n));
    std::vector<std::function<void(Ctx&)>> jobs(parts);
    for (int j = 0; j < parts; j++)
      jobs[j] = [&, j](Ctx&) {
        for (int k = j; k < n; k += parts) copy_one(k);
      };
    pool_run(*pool, jobs, parts);
  }
  int nf = 0;
  uint64_t total2 = 0;
  for (int k = 0; k < n; k++) {
    const HostDecoder& h = *hd[k];
    DeviceDecoder& o = out[k];
    o = DeviceDecoder();
    if (h.d.root_leaf) {
      o.single = true;
      o.single_sym = h.d.root_sym;
      continue;
    }
    const size_t N = h.d.node_count, lut_b = h.lut.size() * 4, pfx_b = h.pfx.size() * 4, arr_b = N * 4;
    if (!pool) copy_one(k);
    const uint8_t* dq = dbuf + base[k];
    const uint8_t* da = dq + lut_b + pfx_b;
    o.tree.lut = (const uint32_t*)dq;
    o.tree.left = (const uint32_t*)da;
    o.tree.right = (const uint32_t*)(da + arr_b);
    o.tree.sym = (const uint32_t*)(da + 2 * arr_b);
    o.tree.leaf = da + 3 * arr_b;
    o.tree.lut2 = dl2 + l2base[k] / 4;
    o.tree.nodes = (uint32_t)N;
    o.max_len = (uint32_t)h.d.max_len;
    if (h.n2) {
      Lut2Fill& f = hf[nf++];
      f.left = o.tree.left;
      f.right = o.tree.right;
      f.sym = o.tree.sym;
      f.leaf = o.tree.leaf;
      f.pfx = (const uint32_t*)(dq + lut_b);
      f.lut2 = dl2 + l2base[k] / 4;
      f.npfx = (uint32_t)(h.pfx.size() / 3);
      f.n2 = (uint32_t)h.n2;
      f.e0 = total2;
      total2 += h.n2;
    }
  }
  CPSZ_HIP(hipMemcpyAsync(dbuf, hbuf, base[n] + sizeof(Lut2Fill) * nf, hipMemcpyHostToDevice, st));
  if (total2) {
    k_fill_lut2_multi<<<(unsigned)div_up(total2, (uint64_t)256), 256, 0, st>>>((const Lut2Fill*)(dbuf + base[n]),
                                                                                nf, total2);
    CPSZ_HIP(hipGetLastError());
  }
}

void stage_bits_multi(Ctx& ctx, BitsCopy* c, int n, const char* tag) {
  hipStream_t st = ctx.stream();
  std::vector<uint32_t> blk0(n + 1, 0);
  size_t words = 0;
  for (int k = 0; k < n; k++) {
    c[k].nwords = div_up(c[k].nbytes, (uint64_t)4) + 8;  // zero slack past the last bit
    words += (c[k].nwords + 63) & ~(uint64_t)63;
  }
  const std::string t(tag);
  uint32_t* dw = ctx.buf<uint32_t>((t + ".words").c_str(), words + 1);
  size_t w0 = 0;
  for (int k = 0; k < n; k++) {
    c[k].dst = dw + w0;
    w0 += (c[k].nwords + 63) & ~(uint64_t)63;
    blk0[k + 1] = blk0[k] + (uint32_t)div_up(c[k].nwords, (uint64_t)kStageBlockWords);
  }
  const size_t tb = sizeof(BitsCopy) * n, bb = 4 * (size_t)(n + 1);
  uint8_t* h = (uint8_t*)ctx.host_buf((t + ".tab").c_str(), tb + bb);
  std::memcpy(h, c, tb);
  std::memcpy(h + tb, blk0.data(), bb);
  uint8_t* d = ctx.buf<uint8_t>((t + ".tab").c_str(), tb + bb);
  CPSZ_HIP(hipMemcpyAsync(d, h, tb + bb, hipMemcpyHostToDevice, st));
  if (blk0[n]) {
    k_stage_bits_multi<<<blk0[n], 256, 0, st>>>((const BitsCopy*)d, (const uint32_t*)(d + tb), n);
    CPSZ_HIP(hipGetLastError());
  }
}

DeviceDecoder upload_decoder(Ctx& ctx, const uint8_t* tree, size_t tree_size, size_t node_count,
                             const char* tag) {
  thread_local HostDecoder hd;  // keeps its allocations from call to call
  prepare_decoder(tree, tree_size, node_count, hd);
  return upload_decoder(ctx, hd, tag);
}

}  // namespace cpsz
