// Bit-packed attention masks for the attention layers' tree verify:
//   dft_packbits        flashinfer.packbits / segment_packbits as
//                       fc1_plan.py:26 calls it (numpy.packbits semantics)
//   dft_tree_mask_pack  the packed tree mask itself: fc1_branch64.py:39
//                       builds [ones(n, plen) | Anc] row-major and
//                       fc1_plan.py:26 packs it; here it is built straight
//                       from the ancestry bits, with no boolean mask.
//
// Both are HBM-bound byte work.  A segment (one packbits segment, one
// request's mask) starts at the byte offset sum_{s' < s} ceil(bits_s' / 8);
// every workgroup of a segment computes that sum itself (a block reduction
// over the earlier segments' sizes), so one launch suffices and nothing is
// read back by the host.  A thread produces an aligned word of the output.
#include <stdint.h>

#include "dft_device.h"

namespace dft {
namespace {

constexpr int kThreads = 256;
constexpr int kBlocksPerSegment = 8, kSegmentBlocks = 6144;  // launch_packbits
constexpr int64_t kMaskBlocks = 768, kMaskWide = 1024;  // launch_tree_mask

__device__ __forceinline__ uint32_t low_mask(int bits) { return bits >= 32 ? 0xffffffffu : ((1u << bits) - 1u); }

// little order: element 8j + k -> bit k of byte j; big: bit 7 - k
__device__ __forceinline__ uint32_t to_order(uint32_t w, int order) {
  return order == DFT_BITS_BIG ? __builtin_bswap32(__builtin_bitreverse32(w)) : w;
}

// Sum over threads of a block (int64), once per kernel; every thread gets the
// total.
__device__ __forceinline__ int64_t block_sum(int64_t v, int64_t* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  int64_t t = 0;
  for (int i = 0; i < kThreads / 64; ++i) t += red[i];
  return t;
}

// Bytes j .. j + 3 of a segment of `nbytes` bytes at byte `off` of out, where
// out + off + j is 4-byte aligned (j may be negative: a word that starts in
// front of the segment); nothing outside the segment, nothing at or past
// `cap`.  Returns false if a byte of the segment was dropped.
__device__ __forceinline__ bool store_word(uint8_t* out, int64_t cap, int64_t off, int64_t nbytes, int64_t j,
                                           uint32_t word) {
  if (j >= 0 && j + 4 <= nbytes && off + j + 4 <= cap) {
    *reinterpret_cast<uint32_t*>(out + off + j) = word;
    return true;
  }
  bool ok = true;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (j + b >= 0 && j + b < nbytes) {
      if (off + j + b < cap)
        out[off + j + b] = (uint8_t)(word >> (8 * b));
      else
        ok = false;
    }
  }
  return ok;
}

__device__ __forceinline__ void store_indptr(void* p, int dt, int64_t i, int64_t v) {
  if (dt == DFT_I64)
    static_cast<int64_t*>(p)[i] = v;
  else
    static_cast<int32_t*>(p)[i] = (int32_t)v;
}

// ---- generic packbits ------------------------------------------------------
__device__ __forceinline__ int64_t seg_begin(const dft_packbits_args& a, int s) {
  return a.indptr ? ld_i(a.indptr, s, a.indptr_dtype) : 0;
}
__device__ __forceinline__ int64_t seg_len(const dft_packbits_args& a, int s) {
  if (!a.indptr) return a.n;
  const int64_t l = ld_i(a.indptr, s + 1, a.indptr_dtype) - ld_i(a.indptr, s, a.indptr_dtype);
  return l < 0 ? 0 : l;
}

// 4 elements (bytes) of a dword to 0 / 1 each
__device__ __forceinline__ uint32_t nonzero4(uint32_t w) {
  return ((((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w) >> 7) & 0x01010101u;
}

// 32 elements (bytes, 8 dwords) to 32 bits, element t at bit t: a dot product
// of each 4 flags with their bits' weights
__device__ __forceinline__ uint32_t pack32(const uint32_t (&d)[8]) {
  uint32_t word = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const uint32_t lo = __builtin_amdgcn_udot4(nonzero4(d[2 * b]), 0x08040201u, 0u, false);
    word |= __builtin_amdgcn_udot4(nonzero4(d[2 * b + 1]), 0x80402010u, lo, false) << (8 * b);
  }
  return word;
}

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// A thread packs the 32 elements of one aligned word of the output.  They
// come as whole dwords (two 16-byte loads; where the elements start inside a
// dword one more, and the bytes are shifted into place: every dword read
// holds at least one of the elements), one by one only in a word that the
// segment's ends cut (16 loads at once: 500 segments of 77 elements 11.6 ->
// 9.2 us; 32 at once take 76 registers and 6% more on a large mask).  Read one
// by one, the 32 elements of every word were 32 loads of one byte, 32 apart
// between lanes: 6.9 us per launch for a 64 x 32795 mask (2.1 MB), now 2.6.
__global__ void __launch_bounds__(kThreads) packbits_kernel(const dft_packbits_args a) {
  __shared__ int64_t red[kThreads / 64];
  const int s = blockIdx.y;
  int64_t off = 0;
  if (s > 0) {  // uniform
    int64_t part = 0;
    for (int q = threadIdx.x; q < s; q += kThreads) part += (seg_len(a, q) + 7) >> 3;
    off = block_sum(part, red);
  }
  const int64_t len = seg_len(a, s), nbytes = (len + 7) >> 3;
  if (a.out_indptr && blockIdx.x == 0 && threadIdx.x == 0) {
    store_indptr(a.out_indptr, a.out_indptr_dtype, s, off);
    if (s + 1 == (int)gridDim.y) store_indptr(a.out_indptr, a.out_indptr_dtype, s + 1, off + nbytes);
  }
  const int lead = (int)(reinterpret_cast<uintptr_t>(a.out + off) & 3);  // bytes of word 0 in front of the segment
  const int64_t nwords = nbytes > 0 ? (lead + nbytes + 3) >> 2 : 0;
  const uint8_t* x = a.x + seg_begin(a, s);
  bool ok = true;
  for (int64_t w = (int64_t)blockIdx.x * kThreads + threadIdx.x; w < nwords; w += (int64_t)gridDim.x * kThreads) {
    const int64_t j = 4 * w - lead, e0 = 8 * j;
    uint32_t word = 0;
    if (e0 >= 0 && e0 + 32 <= len) {
      const int mis = (int)(reinterpret_cast<uintptr_t>(x + e0) & 3);
      const uint32_t* src = reinterpret_cast<const uint32_t*>(x + e0 - mis);
      const u32x4_a4 u = *reinterpret_cast<const u32x4_a4*>(src), v = *reinterpret_cast<const u32x4_a4*>(src + 4);
      uint32_t d[9] = {u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3], 0u};
      if (mis) {  // uniform over the segment (e0 is a multiple of 8)
        d[8] = src[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) d[t] = __builtin_amdgcn_alignbyte(d[t + 1], d[t], mis);
      }
      const uint32_t el[8] = {d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7]};
      word = pack32(el);
    } else {  // elements lo .. hi of the word: clamped, always valid addresses, 16 loads at once
      const int lo = e0 < 0 ? (int)-e0 : 0, hi = len - e0 < 32 ? (int)(len - e0) - 1 : 31;
#pragma unroll 1
      for (int h = 0; h < 32; h += 16) {
        uint8_t v[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) v[t] = x[e0 + min(max(h + t, lo), hi)];
#pragma unroll
        for (int t = 0; t < 16; ++t) word |= (uint32_t)(v[t] != 0) << (h + t);
      }
      word &= low_mask(hi + 1) & ~low_mask(lo);
    }
    ok &= store_word(a.out, a.out_capacity, off, nbytes, j, to_order(word, a.bit_order));
  }
  if (!ok && a.status) *a.status = 1;
}

// ---- packed tree mask -------------------------------------------------------
struct MaskSeg {
  int64_t row0;  // row of node 0
  int64_t plen;  // committed prefix tokens
  int n;         // nodes (<= 64)
};

__device__ __forceinline__ MaskSeg mask_seg(const dft_mask_args& a, int b) {
  MaskSeg m;
  if (a.cu_seqlens) {
    m.row0 = a.cu_seqlens[b];
    m.n = a.cu_seqlens[b + 1] - a.cu_seqlens[b];
  } else {
    m.row0 = (int64_t)b * a.n_nodes;
    m.n = a.n_nodes;
  }
  m.n = m.n < 0 ? 0 : (m.n > 64 ? 64 : m.n);
  const int64_t pl = ld_i(a.prefix_len, b, a.prefix_len_dtype);
  m.plen = pl < 0 ? 0 : pl;
  return m;
}

__device__ __forceinline__ int64_t mask_bits(const MaskSeg& m) { return (int64_t)m.n * (m.plen + m.n); }

// columns c .. c + take - 1 (take <= 32, within one row) of the row whose
// ancestor-or-self bits are `anc`: ones below plen, then the ancestry bits
__device__ __forceinline__ uint32_t row_bits(uint64_t anc, int64_t plen, int64_t c, int take) {
  if (c + take <= plen) return low_mask(take);
  if (c >= plen) return (uint32_t)(anc >> (c - plen)) & low_mask(take);  // c - plen < n <= 64
  const int k = (int)(plen - c);                                          // 1 .. take - 1
  return low_mask(k) | ((uint32_t)(anc << k) & low_mask(take));
}

// A thread produces aligned words of the output (a word that the segment's
// ends or the capacity cut is stored byte by byte).  Most words lie inside one
// row's prefix: all ones.  The ancestry rows are read once per workgroup, and
// come in while it sums the earlier segments' sizes.
__global__ void __launch_bounds__(kThreads) tree_mask_kernel(const dft_mask_args a) {
  __shared__ int64_t red[kThreads / 64];
  __shared__ uint64_t anc[64];
  const int b = blockIdx.y;
  const MaskSeg m = mask_seg(a, b);
  const int64_t L = m.plen + m.n, nbits = mask_bits(m), nbytes = (nbits + 7) >> 3;
  // No word falls to this workgroup (at most 3 bytes of the first lie in front
  // of the segment): said before the sum over the requests ahead.  Workgroup 0
  // also writes the offsets.
  if (blockIdx.x > 0 && (int64_t)blockIdx.x * kThreads >= (nbytes + 6) >> 2) return;  // uniform
  // (the rows come in while the sum runs)
  const uint64_t mine = (int)threadIdx.x < m.n ? a.anc_bits[m.row0 + threadIdx.x] : 0;
  int64_t part = 0;
  for (int q = threadIdx.x; q < b; q += kThreads) part += (mask_bits(mask_seg(a, q)) + 7) >> 3;
  if (threadIdx.x < 64) anc[threadIdx.x] = mine;
  const int64_t off = block_sum(part, red);  // (its barrier covers the ancestry rows)
  if (a.out_indptr && blockIdx.x == 0 && threadIdx.x == 0) {
    store_indptr(a.out_indptr, a.out_indptr_dtype, b, off);
    if (b + 1 == (int)gridDim.y) store_indptr(a.out_indptr, a.out_indptr_dtype, b + 1, off + nbytes);
  }
  const int lead = (int)(reinterpret_cast<uintptr_t>(a.out + off) & 3);  // bytes of word 0 in front of the segment
  const int64_t nwords = nbytes > 0 ? (lead + nbytes + 3) >> 2 : 0;
  bool ok = true;
  for (int64_t w = (int64_t)blockIdx.x * kThreads + threadIdx.x; w < nwords; w += (int64_t)gridDim.x * kThreads) {
    const int64_t j = 4 * w - lead;       // byte of the segment
    int done = j < 0 ? (int)(-8 * j) : 0;  // bits of the word in front of the segment
    const int64_t q0 = j < 0 ? 0 : 8 * j;
    int64_t r, c;
    if (nbits <= 0x7fffffff) {  // 32-bit division (uniform per request)
      r = (uint32_t)q0 / (uint32_t)L;
      c = q0 - r * L;
    } else {
      r = q0 / L;
      c = q0 - r * L;
    }
    uint32_t word = 0;
    if (done == 0 && c + 32 <= m.plen) {
      word = ~0u;
    } else {
      while (done < 32 && r < m.n) {  // at most 32 rows (rows are >= 1 bit long)
        const int take = (int)(L - c < 32 - done ? L - c : 32 - done);
        word |= row_bits(anc[r], m.plen, c, take) << done;
        done += take;
        ++r;
        c = 0;
      }
      word = to_order(word, a.bit_order);
    }
    ok &= store_word(a.out, a.out_capacity, off, nbytes, j, word);
  }
  if (!ok && a.status) *a.status = 1;
}

}  // namespace

int launch_packbits(const dft_packbits_args* a, hipStream_t stream) {
  const int segs = a->indptr ? a->n_segments : 1;
  // Segments (their sizes stay on the device): 8 workgroups each that stride
  // over its words, fewer where there are so many that starting them is the
  // launch's time.  us with 8 for each and the cut words' elements one after
  // another / now (in brackets the form that read every word so):
  //   1000 segments of 77 elements         19.0 /  11.6   [17.5]
  //   3000                                 58.4 /  17.8   [54.5]
  //   9000                                273.8 /  41.2  [264.1]
  //   3000, one of them of 2^21            59.1 /  54.0  [145.3]
  // One segment of known length: enough workgroups to cover it once.
  int bx = segs <= kSegmentBlocks / kBlocksPerSegment ? kBlocksPerSegment
                                                      : (segs < kSegmentBlocks ? kSegmentBlocks / segs : 1);
  if (!a->indptr) {
    const int64_t words = ((a->n + 31) >> 5) + 1, need = (words + kThreads - 1) / kThreads;  // (+ 1: an unaligned out)
    bx = (int)(need < 1 ? 1 : (need > 4096 ? 4096 : need));
  }
  hipLaunchKernelGGL(packbits_kernel, dim3((unsigned)bx, (unsigned)segs), dim3(kThreads), 0, stream, *a);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

int launch_tree_mask(const dft_mask_args* a, hipStream_t stream) {
  // The sizes stay on the device, so the grid goes by what is known here.  The
  // capacity bounds the words, one per thread, but is no measure of them where
  // the buffer is a reserve: no more workgroups for it than kMaskBlocks in all
  // (one that finds no words costs about 2 ns of launch).  A request may hold
  // most of the words, and a workgroup alone takes 0.25 us per 256 of them: at
  // least 8 each up to kMaskWide requests, and 8 kMaskWide in all beyond.  us
  // per launch, back to back, with 8 workgroups per request that walked its
  // words by a division and an ancestry read each, with a thread per word of
  // the capacity up to 2048 workgroups in all, and now (exact buffer / 64 MiB):
  //   64 requests x 32 nodes, 4096 tokens       3.7    3.8 / 4.6    3.7 / 3.7
  //   64 x 16-64 nodes, 6000 tokens             6.4    5.2 / 5.4    4.7 / 4.7
  //   1 x 64 nodes, 32768 tokens               12.2    2.7 / 3.3    2.7 / 2.7
  //   8 x 64 nodes, 100 tokens                  3.0    3.1 / 4.5    3.1 / 3.2
  //   128 x 8-64 nodes, 300 tokens              4.0    3.8 / 4.8    3.9 / 3.9
  //   256 x 8-64 nodes, 2000 tokens             6.8    6.4 / 6.3    6.5 / 6.5
  //   300 of 100 tokens, one of 64 x 32768     12.4   35.1 /13.1   12.0 /12.0
  //   2100 of 100 tokens, one of 64 x 32768    33.2   62.3 /62.2   23.3 /23.4
  const int64_t least = a->batch <= kMaskWide ? 8 : (a->batch < 8 * kMaskWide ? 8 * kMaskWide / a->batch : 1);
  const int64_t most = a->batch * least < kMaskBlocks ? kMaskBlocks / a->batch : least;
  const int64_t need = (a->out_capacity / a->batch + 4 * kThreads - 1) / (4 * kThreads);
  const int64_t bx = need < least ? least : (need > most ? most : need);
  hipLaunchKernelGGL(tree_mask_kernel, dim3((unsigned)bx, (unsigned)a->batch), dim3(kThreads), 0, stream, *a);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

}  // namespace dft
