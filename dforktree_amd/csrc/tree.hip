// Tree structure from parent indices (tree_ops.py:68-89, fc1_builder.py:38-47).
// Four waves per request, or one (n <= 64 nodes, lane i = node i):
//   - ancestor-or-self set of i as a uint64 (exact closure by pointer
//     doubling: after k rounds the set holds the ancestors at distances below
//     2^k and p the 2^k-th one, so six rounds cover any tree; the reference's
//     five squarings stop at 31 edges, tree_ops.py:75-79),
//   - depth, conv gather columns cidx[i][kc-1-r] = kc-1 + (r-th ancestor)
//     if r <= depth else kc-1-(r-depth) (tree_ops.py:81-88),
//   - first child / next sibling links (fc1_builder.py:41-47), from the set of
//     every node's children.
// Node 0 is the root; for i >= 1 the parent is max(parent[i], 0), the clamp
// of tree_ops.py:73.  Integer work; results are bit-exact.
//
// Bound by the chain of one request: every wave forms the sets (registers
// and lane shuffles), then wave 0 writes the sets, depths and status, wave 1
// cidx, wave 2 the links, and all four the dense rows (one wave does it all
// where there is little to share out: launch_tree_struct).  128 requests of
// 8-64 nodes with every output: 19.9 us with one wave per request that walked
// the parents one LDS read at a time (63 for a chain) and searched the links
// by a loop over the nodes, now 4.2 us, 4.6 with what no tree covers zeroed
// too (23.6 with two fill launches ahead).
#include "dft_device.h"

namespace dft {

// One request.  A request whose parents form a cycle keeps what a walk of n
// steps sees: the nodes it visits, depth n, status 2.
// W: waves that take part (w: this one's number), each with a share of the
// outputs.
// FILL: also zeroes the dense matrix outside the tree (n_nodes x n_nodes; a
// tree cut to 64 rows is cut to n_nodes there) and the ancestry rows between
// this request's last node and the next request.
template <bool FILL, int W>
__device__ __forceinline__ void tree_of_request(const dft_tree_args& p, int b, int64_t rows_all, int w,
                                                unsigned long long* kids) {
  constexpr int kCidxWave = 1 % W, kLinkWave = 2 % W;
  const int lane = threadIdx.x & 63;
  int64_t row0;
  int n;
  if (p.cu_seqlens) {
    row0 = p.cu_seqlens[b];
    n = p.cu_seqlens[b + 1] - p.cu_seqlens[b];
  } else {
    row0 = (int64_t)b * p.n_nodes;
    n = p.n_nodes;
  }
  const int span = n;
  n = n < 0 ? 0 : (n > 64 ? 64 : n);
  const int i = lane;
  const bool in = i < n;

  bool bad = false;
  int par = 0;  // (the root's: itself)
  if (in && i > 0) {
    const int64_t raw = ld_i(p.parent, row0 + i, p.parent_dtype);
    par = raw < 0 ? 0 : (int)raw;
    if (par >= n) {  // out of range: treated as a child of the root
      par = 0;
      bad = true;
    }
    bad |= par >= i;  // not topologically ordered
  }

  // (every lane takes part in the shuffles; lanes past the tree are no one's parent)
  uint64_t bits = 1ull << i;
  int up = par;
#pragma unroll 1
  for (int k = 0; k < 6 && __ballot(up != 0); ++k) {
    bits |= __shfl(bits, up);
    up = __shfl(up, up);
  }
  const bool cycle = up != 0;  // no root among 64 ancestors
  if (!cycle) bits |= 1ull;
  const int depth = cycle ? n : __popcll(bits) - 1;

  if (w == 0) {
    if (in) {
      if (p.anc_bits) p.anc_bits[row0 + i] = bits;
      if (p.depth) st_i(p.depth, row0 + i, p.depth_dtype, depth);
    }
    if (p.status) {
      const uint64_t any_cycle = __ballot(in && cycle), any_bad = __ballot(in && bad);
      if (lane == 0) p.status[b] = any_cycle ? 2 : (any_bad ? 1 : 0);
    }
  }
  if (w == kCidxWave && p.cidx) {
    int cur = i;  // the r-th ancestor
    for (int r = 0; r < p.kc; ++r) {
      const int v = r <= depth ? (p.kc - 1 + cur) : (p.kc - 1 - (r - depth));
      if (in) st_i(p.cidx, (row0 + i) * p.kc + (p.kc - 1 - r), p.cidx_dtype, v);
      cur = __shfl(par, cur);
    }
  }
  if (w == kLinkWave && (p.nxt || p.sib)) {
    // (one wave: its LDS operations run in order)
    volatile unsigned long long* k = kids;
    k[i] = 0;
    asm volatile("" ::: "memory");
    if (in && i > 0) atomicOr(&kids[par], 1ull << i);
    asm volatile("" ::: "memory");
    const uint64_t own = k[i], later = k[par] & ~mask_upto(i);
    if (in) {
      if (p.nxt) st_i(p.nxt, row0 + i, p.link_dtype, own ? __ffsll((unsigned long long)own) - 1 : -1);
      if (p.sib) st_i(p.sib, row0 + i, p.link_dtype, (i > 0 && later) ? __ffsll((unsigned long long)later) - 1 : -1);
    }
  }
  if (p.anc_f32) {
    // row r of the dense matrix: lane = column, coalesced
    float* base = p.anc_f32 + (int64_t)b * p.anc_req_stride;
    const uint32_t lo = (uint32_t)bits, hi = (uint32_t)(bits >> 32);
    const int rows = FILL ? p.n_nodes : n, cols = rows;
    for (int r = w; r < rows; r += W) {  // (uniform)
      uint64_t rb = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, r) << 32) |
                    (uint32_t)__builtin_amdgcn_readlane(lo, r);
      if (FILL && r >= n) rb = 0;
      if (lane < cols) base[(int64_t)r * p.anc_row_stride + lane] = (float)((rb >> lane) & 1ull);
    }
  }
  if (FILL && p.anc_bits)
    for (int64_t r = row0 + 64 + 64 * w + lane; r < row0 + span && r < rows_all; r += 64 * W) p.anc_bits[r] = 0;
}

// The smallest and the largest of the batch's cu_seqlens (every request's
// rows lie between them), reduced in registers (one LDS atomic per request
// was 15 us at 1024 requests, 129 at 8192, ahead of what it is for).
__device__ __forceinline__ void packed_ends(const dft_tree_args& p, int& lo, int& hi) {
  __shared__ int ends[2][4];
  const int wave = threadIdx.x >> 6;
  lo = hi = p.cu_seqlens[0];
#pragma unroll 8
  for (int q = threadIdx.x; q <= p.batch; q += 256) {
    const int c = p.cu_seqlens[q];
    lo = min(lo, c);
    hi = max(hi, c);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
  }
  ends[0][wave] = lo;
  ends[1][wave] = hi;
  __syncthreads();
  lo = min(min(ends[0][0], ends[0][1]), min(ends[0][2], ends[0][3]));
  hi = max(max(ends[1][0], ends[1][1]), max(ends[1][2], ends[1][3]));
}

// FILL: the grid's last workgroup zeroes the ancestry rows (of `rows`) in
// front of the first request and behind the last.
template <bool FILL, int W>
__global__ void __launch_bounds__(256) tree_struct_kernel(const dft_tree_args p, int64_t rows) {
  __shared__ unsigned long long kids[4 / W][64];
  const int blocks = (int)gridDim.x - (FILL ? 1 : 0);
  if (FILL && (int)blockIdx.x == blocks) {
    if (!p.anc_bits) return;
    int64_t lo = 0, hi = (int64_t)p.batch * p.n_nodes;
    if (p.cu_seqlens) {
      int first, last;
      packed_ends(p, first, last);
      lo = first;
      hi = last < 0 ? 0 : last;
    }
    for (int64_t r = threadIdx.x; r < lo && r < rows; r += 256) p.anc_bits[r] = 0;
    for (int64_t r = hi + threadIdx.x; r < rows; r += 256) p.anc_bits[r] = 0;
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int b = blockIdx.x * (4 / W) + wave / W; b < p.batch; b += blocks * (4 / W))
    tree_of_request<FILL, W>(p, b, rows, wave % W, kids[wave / W]);
}

// Dense 0/1 ancestry rows -> the uint64 rows the verify and commit read.
// A wave per 16 rows, W of them per request (one wave with all 64: 2 to 3 us
// more per batch-1 step): lane j loads column j of every one of its rows
// first (coalesced rows, all loads in flight at once), then the wave's ballot
// of each row is that row's mask; bits above the diagonal are dropped, as the
// kernels that read dense rows drop them.  Lane i keeps the wave's row i and
// writes it at the end.
// The loads take clamped, always valid addresses (row and column min(., n-1))
// and the ballots mask what lies outside the n x n matrix: with the bounds in
// a condition around each load, every load sat in its own branch and was
// waited for at once (batch 1: 7.4 us per launch at 32 nodes).
__device__ __forceinline__ void anc_pack_rows(const dft_anc_pack_args& p, int b, int r0) {
  const int lane = threadIdx.x & 63;
  const int n = p.n_nodes;
  if (r0 >= n) return;  // (uniform over the wave) no rows
  const float* base = p.anc + (int64_t)b * p.anc_req_stride + (lane < n ? lane : n - 1);
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = base[(int64_t)(r0 + i < n ? r0 + i : n - 1) * p.anc_row_stride];
  const bool col_in = lane < n;
  uint64_t mine = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const uint64_t row = __ballot(col_in && v[i] > 0.5f) & mask_upto(r0 + i);
    if (lane == i) mine = row;
  }
  if (lane < 16 && r0 + lane < n) p.anc_bits[(int64_t)b * n + r0 + lane] = mine;
}

template <int W>
__global__ void __launch_bounds__(256) anc_pack_kernel(const dft_anc_pack_args p) {
  const int wave = threadIdx.x >> 6;  // (as a scalar: 16 scalar row addresses, 0.2 us more at batch 1)
  for (int b = blockIdx.x * (4 / W) + wave / W; b < p.batch; b += gridDim.x * (4 / W))
    anc_pack_rows(p, b, 16 * (wave % W));
}

template <int W>
void launch_anc_rows(const dft_anc_pack_args* a, hipStream_t stream) {
  const int64_t need = ((int64_t)a->batch * W + 3) / 4;
  const dim3 grid((unsigned)(need < 65536 ? need : 65536));  // workgroups stride over further requests
  hipLaunchKernelGGL(anc_pack_kernel<W>, grid, dim3(256), 0, stream, *a);
}

// As many waves per request as its rows need (8192 trees of 8 nodes 13.7 us
// with four, one of them with rows).
int launch_anc_pack(const dft_anc_pack_args* a, hipStream_t stream) {
  if (a->n_nodes <= 16)
    launch_anc_rows<1>(a, stream);
  else if (a->n_nodes <= 32)
    launch_anc_rows<2>(a, stream);
  else
    launch_anc_rows<4>(a, stream);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

// One wave per request, four to a workgroup, where there is nothing to share
// out (the sets, depths and status are wave 0's) or the requests alone fill the
// chip.  us with four waves / one, for the sets alone and for every output:
//   1 request of 64 nodes      2.6 / 2.5    4.1 / 7.9
//   128 of 8-64                3.0 / 3.0    4.7 / 8.6
//   2048 of 8-64               4.8 / 3.3   11.5 / 11.8
//   4096 of 8-64               6.8 / 3.7   16.6 / 16.5
//   8192 of 4-8               10.3 / 4.5   13.4 / 8.1
constexpr int kTreeOneWave = 4096;

template <int W>
void launch_trees(const dft_tree_args* a, int64_t rows, hipStream_t stream) {
  const int64_t need = ((int64_t)a->batch * W + 3) / 4;
  const unsigned grid = (unsigned)(need < 65536 ? need : 65536);  // workgroups stride over further requests
  if (rows >= 0)
    hipLaunchKernelGGL((tree_struct_kernel<true, W>), dim3(grid + 1), dim3(256), 0, stream, *a, rows);
  else
    hipLaunchKernelGGL((tree_struct_kernel<false, W>), dim3(grid), dim3(256), 0, stream, *a, rows);
}

// rows >= 0: the filling form over that many ancestry rows
int launch_tree_struct(const dft_tree_args* a, int64_t rows, hipStream_t stream) {
  const bool shared = a->cidx || a->nxt || a->sib || a->anc_f32;
  if (shared && a->batch < kTreeOneWave)
    launch_trees<4>(a, rows, stream);
  else
    launch_trees<1>(a, rows, stream);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

}  // namespace dft
