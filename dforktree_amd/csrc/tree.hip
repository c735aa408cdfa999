// Tree structure from parent indices (tree_ops.py:68-89, fc1_builder.py:38-47).
// One workgroup of four waves per request (n <= 64 nodes, lane i = node i):
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
// cidx, wave 2 the links, and all four the dense rows.  128 requests of 8-64
// nodes with every output: 20.4 us with one wave per request that walked the
// parents one LDS read at a time (63 for a chain) and searched the links by
// a loop over the nodes, now 4.7 us, 6.4 with what no tree covers zeroed too
// (two fill launches fewer).
#include "dft_device.h"

namespace dft {

// One request.  A request whose parents form a cycle keeps what a walk of n
// steps sees: the nodes it visits, depth n, status 2.
// FILL: also zeroes the dense matrix outside the tree (n_nodes x n_nodes; a
// tree cut to 64 rows is cut to n_nodes there) and the ancestry rows between
// this request's last node and the next request.
template <bool FILL>
__device__ __forceinline__ void tree_of_request(const dft_tree_args& p, int b, int64_t rows_all, unsigned long long* kids) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
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
  } else if (w == 1) {
    if (p.cidx) {
      int cur = i;  // the r-th ancestor
      for (int r = 0; r < p.kc; ++r) {
        const int v = r <= depth ? (p.kc - 1 + cur) : (p.kc - 1 - (r - depth));
        if (in) st_i(p.cidx, (row0 + i) * p.kc + (p.kc - 1 - r), p.cidx_dtype, v);
        cur = __shfl(par, cur);
      }
    }
  } else if (w == 2 && (p.nxt || p.sib)) {
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
    for (int r = w; r < rows; r += 4) {  // (uniform)
      uint64_t rb = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(hi, r) << 32) | (uint32_t)__builtin_amdgcn_readlane(lo, r);
      if (FILL && r >= n) rb = 0;
      if (lane < cols) base[(int64_t)r * p.anc_row_stride + lane] = (float)((rb >> lane) & 1ull);
    }
  }
  if (FILL && p.anc_bits)
    for (int64_t r = row0 + 64 + threadIdx.x; r < row0 + span && r < rows_all; r += 256) p.anc_bits[r] = 0;
}

// FILL: the grid's last workgroup zeroes the ancestry rows (of `rows`) in
// front of the first request and behind the last.
template <bool FILL>
__global__ void __launch_bounds__(256) tree_struct_kernel(const dft_tree_args p, int64_t rows) {
  __shared__ unsigned long long kids[64];  // wave 2's
  const int stride = (int)gridDim.x - (FILL ? 1 : 0);
  if (FILL && (int)blockIdx.x == stride) {
    if (!p.anc_bits) return;
    int64_t lo = 0, hi = (int64_t)p.batch * p.n_nodes;
    if (p.cu_seqlens) {
      __shared__ int ends[2];
      if (threadIdx.x == 0) ends[0] = ends[1] = p.cu_seqlens[0];
      __syncthreads();
      for (int q = 1 + threadIdx.x; q <= p.batch; q += 256) {
        atomicMin(&ends[0], p.cu_seqlens[q]);
        atomicMax(&ends[1], p.cu_seqlens[q]);
      }
      __syncthreads();
      lo = ends[0];
      hi = ends[1] < 0 ? 0 : ends[1];
    }
    for (int64_t r = threadIdx.x; r < lo && r < rows; r += 256) p.anc_bits[r] = 0;
    for (int64_t r = hi + threadIdx.x; r < rows; r += 256) p.anc_bits[r] = 0;
    return;
  }
  for (int b = blockIdx.x; b < p.batch; b += stride) tree_of_request<FILL>(p, b, rows, kids);
}

// Dense 0/1 ancestry rows -> the uint64 rows the verify and commit read.
// Four waves per request, each with 16 of the rows (one wave with all 64: 2 to
// 3 us more per batch-1 step): lane j loads column j of
// every one of them first (coalesced rows, all loads in flight at once), then
// the wave's ballot of each row is that row's mask; bits above the diagonal
// are dropped, as the kernels that read dense rows drop them.  Lane i keeps
// the wave's row i and writes it at the end.
// The loads take clamped, always valid addresses (row and column min(., n-1))
// and the ballots mask what lies outside the n x n matrix: with the bounds in
// a condition around each load, every load sat in its own branch and was
// waited for at once (batch 1: 7.4 us per launch at 32 nodes).
__device__ __forceinline__ void anc_pack_request(const dft_anc_pack_args& p, int b) {
  const int lane = threadIdx.x & 63, r0 = 16 * (threadIdx.x >> 6);
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

__global__ void __launch_bounds__(256) anc_pack_kernel(const dft_anc_pack_args p) {
  for (int b = blockIdx.x; b < p.batch; b += gridDim.x) anc_pack_request(p, b);
}

int launch_anc_pack(const dft_anc_pack_args* a, hipStream_t stream) {
  const dim3 grid((unsigned)(a->batch < 65536 ? a->batch : 65536));  // workgroups stride over further requests
  hipLaunchKernelGGL(anc_pack_kernel, grid, dim3(256), 0, stream, *a);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

// rows >= 0: the filling form over that many ancestry rows
int launch_tree_struct(const dft_tree_args* a, int64_t rows, hipStream_t stream) {
  const unsigned grid = (unsigned)(a->batch < 65536 ? a->batch : 65536);  // workgroups stride over further requests
  if (rows >= 0)
    hipLaunchKernelGGL(tree_struct_kernel<true>, dim3(grid + 1), dim3(256), 0, stream, *a, rows);
  else
    hipLaunchKernelGGL(tree_struct_kernel<false>, dim3(grid), dim3(256), 0, stream, *a, rows);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

}  // namespace dft
