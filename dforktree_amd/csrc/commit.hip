// Closed-form accepted-path state commit (tree_kernels.py:111-127 in place,
// fc1_fused.py:26-49 into a snapshot slot):
//   S_u = e^{G_u} S0 + sum_{t in path, t anc-or-self of u} e^{G_u - G_t} k_t vn_t^T
// One workgroup per (layer, request, head, end) rewrites one 128x128 fp32
// state: a rank-T update (T <= 64 accepted nodes) that is read-modify-write
// HBM traffic at ~4 flop/B, so plain fp32 FMAs from registers, the state
// streamed with 16-byte loads.
//
// The state is addressed as rows x cols.  Pool layout [.., V, K] (k
// contiguous): rows = v, cols = k, so S[v][k] += (w_t vn_t[v]) k_t[k].
// With DFT_COMMIT_KV the rows are k and the update is k_t[k] (w_t vn_t[v]).
#include <initializer_list>

#include "dft_device.h"

namespace dft {

constexpr int kCD = 128;

struct CommitParams {
  dft_commit_args a;
  int src_vec, dst_vec;  // 16-byte vector path usable
  int path_vec;          // key and value rows 16-byte aligned
};

// global -> LDS, lane l's 16 bytes at lds + 16 l
__device__ __forceinline__ void lds_copy16(const float* g, float* lds) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// Element i (uniform) of an int32 or int64 array that the launch does not
// write, as two scalar loads with no branch between them: behind a branch on
// the type, each of a workgroup's five index reads was a round trip of its
// own ahead of the tile.
__device__ __forceinline__ int64_t uniform_index(const void* idx, int64_t i, int dt) {
  typedef const __attribute__((address_space(4))) int32_t* Words;
  const Words w = (Words)(uintptr_t)idx;
  const bool wide = dt == DFT_I64;
  const int32_t lo = w[wide ? 2 * i : i], hi = w[wide ? 2 * i + 1 : i];
  return wide ? (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo) : (int64_t)lo;
}

// path entries of request b that count (path_len, or all path_cols)
__device__ __forceinline__ int path_entries(const dft_commit_args& p, int b) {
  int len = p.path_cols;
  if (p.path_len) {
    len = (int)uniform_index(p.path_len, b, p.path_len_dtype);
    if (p.flags & DFT_COMMIT_LEN_IS_LAST) len += 1;
    len = len < 0 ? 0 : (len > p.path_cols ? p.path_cols : len);
  }
  return len;
}

// The status word of request b (wave 0 of its first workgroup): a row span
// past n_nodes, and path entries or ends at or past its n nodes.
__device__ __forceinline__ void commit_status(const dft_commit_args& p, int b, int n, bool span_bad, int lane) {
  const int len = path_entries(p, b);
  bool bad = false;
  for (int c = lane; c < len; c += 64) bad |= ld_i(p.path, (int64_t)b * p.path_req_stride + c, p.path_dtype) >= n;
  if (p.ends && lane < p.n_ends) bad |= ld_i(p.ends, (int64_t)b * p.ends_req_stride + lane, p.ends_dtype) >= n;
  const bool any = __ballot(bad) != 0;
  if (lane == 0) p.status[b] = (span_bad ? DFT_STATUS_SPAN : 0) | (any ? DFT_STATUS_PATH : 0);
}

// Bound by the tile's traffic (a read and a write of 64 KiB per workgroup),
// if nothing but the tile is waited for.  So the index reads are scalar and
// come in one batch, the path's entries are loaded ahead of the tile, every
// wave decodes them by itself, and the path's rows follow the tile straight
// into LDS, all at once.  Staged by a loop of up to 8 dependent rounds per
// thread behind the tile, a path of 16 nodes cost as much again as the tile.
// us for 1 / 4 / 16 nodes, before and now:
//   4 layers x 128 requests x 32 heads (2.1 GB)  368 / 380 / 584   367 / 366 / 374
//   12 x 12 x 16 (302 MB)                         52 /  59 /  98    51 /  52 /  58
//   batch 1, 24 x 32, into 2 snapshots, 16 nodes  65                34
// Two corners are slower: one path node on a state that is in cache (24 layers
// of batch 1 in place: 14.7 -> 15.8, where 4 nodes take 17.9 -> 16.6 and 16 38.8
// -> 17.8), and tiles read element by element, whose kernel holds three
// registers too many (the same with strided columns: 156 / 153 / 160 -> 162 /
// 157 / 158; four waves per SIMD spill nothing and take 24% more at batch 32).
// Five waves per SIMD (64 KiB of state in flight for each of five workgroups
// per CU; four measured 4% slower); six leave 80 registers, spilled 2 and
// took 381 us for the first row.
// VEC: every tile and path row takes 16-byte accesses, so that no branch
// joins two ways of loading (after such a join the wait counts are not known
// and the path's entries would be waited for with the whole tile).
template <bool VEC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5)))
tree_commit_kernel(const CommitParams P) {
  const dft_commit_args& p = P.a;
  extern __shared__ float cshm[];  // the path's keys [path_cols, even][128], then its values
  __shared__ int s_nodes[4][64];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // block id -> (layer, request, head) unit and end.  The ends of one unit
  // read the same source tile: their blocks sit 8 ids apart, so that they
  // land on one XCD (blocks are dealt to the 8 XCDs in turn) and the later
  // reads of the tile hit that XCD's L2.  Units past the last whole group
  // of 8 take their ends from consecutive ids.
  int id = blockIdx.x, e;
  {
    const int units = p.n_layers * p.batch * p.hv;
    const int full = (units / 8) * 8 * p.n_ends;
    if (id < full) {
      const int grp = id / (8 * p.n_ends), rem = id - grp * 8 * p.n_ends;
      e = rem >> 3;
      id = grp * 8 + (rem & 7);
    } else {
      const int t = id - full;
      e = t % p.n_ends;
      id = (units / 8) * 8 + t / p.n_ends;
    }
  }
  const int h = id % p.hv;
  id /= p.hv;
  const int b = id % p.batch;
  const int l = id / p.batch;

  // nodes of the request: its row span cut to [0, n_nodes]
  int64_t row0;
  int span;
  if (p.cu_seqlens) {
    row0 = uniform_index(p.cu_seqlens, b, DFT_I32);
    span = (int)(uniform_index(p.cu_seqlens, b + 1, DFT_I32) - row0);
  } else {
    row0 = (int64_t)b * p.n_nodes;
    span = p.n_nodes;
  }
  const int n = span < 0 ? 0 : (span > p.n_nodes ? p.n_nodes : span);
  if (p.status && l == 0 && h == 0 && e == 0 && tid < 64) commit_status(p, b, n, span < 0 || span > p.n_nodes, lane);

  int u_end = -1;
  if (p.ends) {
    u_end = (int)uniform_index(p.ends, (int64_t)b * p.ends_req_stride + e, p.ends_dtype);
    if (u_end < 0 || u_end >= n) return;  // nothing to commit for this end
  }

  // A negative destination slot (in place: a negative source slot), e.g. a
  // padded request, commits nothing; a negative source slot with a separate
  // destination reads slot 0, as the verify reads its S0.
  int64_t slot = b;
  if (p.src_slots) slot = uniform_index(p.src_slots, b, p.src_slots_dtype);
  int64_t dslot = slot;
  if (p.dst_slots) dslot = uniform_index(p.dst_slots, b, p.dst_slots_dtype);
  if (dslot < 0) return;
  if (slot < 0) slot = 0;
  const int len = path_entries(p, b);

  // this lane's path entry, ahead of the tile (vector memory returns in order)
  // (the low word of an int64 entry: nodes are small, and a negative one's is negative)
  const int64_t entry = (int64_t)b * p.path_req_stride + (lane < p.path_cols ? lane : 0);
  const int node = static_cast<const int32_t*>(p.path)[entry * (p.path_dtype == DFT_I64 ? 2 : 1)];
  asm volatile("" ::: "memory");

  // ---- state tile: thread owns rows 16*rg .. 16*rg+15, cols 4*c4 .. 4*c4+3
  const int c4 = tid & 31, rg = tid >> 5;
  const float* srcp = p.src + (int64_t)l * p.src_layer_stride + slot * p.src_slot_stride + (int64_t)h * p.src_h_stride;
  f32x4 st[16];
  // (a lane's offset within the tile in 32 bits, checked by the caller: the
  // accesses then take a scalar row base, and no row address is held in a
  // vector register pair)
  if (VEC || P.src_vec) {
    const uint32_t at = 4u * (16u * (uint32_t)rg * (uint32_t)p.src_row_stride + 4u * (uint32_t)c4);
#pragma unroll
    for (int m = 0; m < 16; ++m)
      st[m] = __builtin_nontemporal_load(
          reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(srcp + m * p.src_row_stride) + at));
  } else {  // element loads, walking the rows (no per-row index is kept live)
    const float* rowp = srcp + (int64_t)(16 * rg) * p.src_row_stride + (int64_t)(4 * c4) * p.src_col_stride;
#pragma unroll
    for (int m = 0; m < 16; ++m, rowp += p.src_row_stride)
#pragma unroll
      for (int q = 0; q < 4; ++q) st[m][q] = rowp[(int64_t)q * p.src_col_stride];
  }

  // ---- the path, in every wave (its entries were loaded ahead of the tile
  // and arrive ahead of it): the entries that count, in path order, and the
  // node u whose state is written
  const bool valid = lane < len && node >= 0 && node < n;
  const uint64_t vmask = __ballot(valid);
  int u = u_end;
  if (!p.ends) u = vmask ? __shfl(node, 63 - __builtin_clzll(vmask)) : -1;
  if (u < 0) return;  // no accepted node: the state stays as it is (uniform over the workgroup)
  u = __builtin_amdgcn_readfirstlane(u);
  const int T = __builtin_popcountll(vmask);
  int* nodes = s_nodes[wave];  // (one wave: its LDS operations run in order)
  if (valid) nodes[__builtin_popcountll(vmask & mask_below(lane))] = node;
  asm volatile("" ::: "memory");

  // the nodes of lane t's entry and of the rows this wave copies: read ahead
  // of the copies, as every LDS read behind one is made to wait for it
  const int half = lane >> 5;
  const int mine = nodes[lane < T ? lane : 0];
  const int copy0 = nodes[T > 0 ? min(2 * wave + half, T - 1) : 0];
  const int copy1 = nodes[T > 0 ? min(2 * wave + 8 + half, T - 1) : 0];

  // lane t: the weight of entry t, and whether it counts (an ancestor of u)
  const float* gl = p.gains + (int64_t)l * p.g_layer_stride + (int64_t)h * p.g_h_stride;
  const float Gu = gl[(row0 + u) * p.g_row_stride];
  const float Gt = gl[(row0 + (T > 0 ? mine : u)) * p.g_row_stride];
  const bool check = (p.flags & DFT_COMMIT_CHECK_ANC) != 0;
  uint64_t abits = ~0ull;
  if (check && p.anc_bits) abits = p.anc_bits[row0 + u];
  if (check && !p.anc_bits) {
    const float av = lane < n ? p.anc_f32[(int64_t)b * p.anc_req_stride + (int64_t)u * p.anc_row_stride + lane] : 0.f;
    abits = __ballot(av > 0.5f);
  }

  // their rows straight into LDS (two per 1 KiB copy), behind the tile
  const float* kl = p.keys + (int64_t)l * p.k_layer_stride + (int64_t)(h / p.k_head_div) * p.k_h_stride;
  const float* vl = p.values + (int64_t)l * p.v_layer_stride + (int64_t)h * p.v_h_stride;
  float* ks = cshm;
  float* vs = cshm + (p.path_cols + (p.path_cols & 1)) * kCD;
  if (VEC || P.path_vec) {
    const auto copy = [&](int t, int nd) {  // rows t and t + 1
      const int64_t r = row0 + nd;
      lds_copy16(kl + r * p.k_row_stride + 4 * (lane & 31), ks + t * kCD);
      lds_copy16(vl + r * p.v_row_stride + 4 * (lane & 31), vs + t * kCD);
    };
    if (2 * wave < T) copy(2 * wave, copy0);  // (uniform)
    if (2 * wave + 8 < T) copy(2 * wave + 8, copy1);
    for (int t = 2 * wave + 16; t < T; t += 8) copy(t, nodes[min(t + half, T - 1)]);
  } else {
    for (int c = tid; c < T * kCD; c += 256) {
      const int64_t r = row0 + nodes[c >> 7];
      ks[c] = kl[r * p.k_row_stride + (c & (kCD - 1))];
      vs[c] = vl[r * p.v_row_stride + (c & (kCD - 1))];
    }
  }
  const uint64_t onmask = __ballot(lane < T && ((abits >> mine) & 1ull));
  const float weight = __expf(Gu - Gt);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the row copies
  __syncthreads();

  const float* rv = (p.flags & DFT_COMMIT_KV) ? ks : vs;
  const float* cv = (p.flags & DFT_COMMIT_KV) ? vs : ks;
  const float eGu = __expf(Gu);
#pragma unroll
  for (int m = 0; m < 16; ++m) st[m] *= eGu;
  for (int t = 0; t < T; ++t) {
    if (!((onmask >> t) & 1ull)) continue;  // uniform
    const float w = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), t));
    const f32x4 cc = *reinterpret_cast<const f32x4*>(&cv[t * kCD + 4 * c4]) * w;
    const f32x4* rp = reinterpret_cast<const f32x4*>(&rv[t * kCD + 16 * rg]);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 r = rp[q];
#pragma unroll
      for (int m = 0; m < 4; ++m) st[4 * q + m] += r[m] * cc;
    }
  }

  float* dstp = p.dst + (int64_t)l * p.dst_layer_stride + dslot * p.dst_slot_stride + (int64_t)u * p.dst_node_stride +
                (int64_t)h * p.dst_h_stride;
  if (VEC || P.dst_vec) {
    const uint32_t at = 4u * (16u * (uint32_t)rg * (uint32_t)p.dst_row_stride + 4u * (uint32_t)c4);
#pragma unroll
    for (int m = 0; m < 16; ++m)
      __builtin_nontemporal_store(st[m], reinterpret_cast<f32x4*>(reinterpret_cast<char*>(dstp + m * p.dst_row_stride) + at));
  } else {
    float* rowp = dstp + (int64_t)(16 * rg) * p.dst_row_stride + (int64_t)(4 * c4) * p.dst_col_stride;
#pragma unroll
    for (int m = 0; m < 16; ++m, rowp += p.dst_row_stride)
#pragma unroll
      for (int q = 0; q < 4; ++q) rowp[(int64_t)q * p.dst_col_stride] = st[m][q];
  }
}

// a tile's 128 rows within 32 bits of bytes
static bool rows_ok(int64_t row_stride) { return row_stride >= 0 && row_stride < (1 << 22); }

static bool vec_ok(const float* base, int64_t col, std::initializer_list<int64_t> strides) {
  if (col != 1 || (reinterpret_cast<uintptr_t>(base) % 16) != 0) return false;
  for (int64_t s : strides)
    if (s % 4 != 0) return false;
  return true;
}

int launch_tree_commit(const dft_commit_args* a, hipStream_t stream) {
  CommitParams P;
  P.a = *a;
  P.src_vec = rows_ok(a->src_row_stride) &&
              vec_ok(a->src, a->src_col_stride,
                     {a->src_layer_stride, a->src_slot_stride, a->src_h_stride, a->src_row_stride});
  P.dst_vec = rows_ok(a->dst_row_stride) &&
              vec_ok(a->dst, a->dst_col_stride,
                     {a->dst_layer_stride, a->dst_slot_stride, a->dst_node_stride, a->dst_h_stride,
                      a->dst_row_stride});
  P.path_vec = vec_ok(a->keys, 1, {a->k_layer_stride, a->k_h_stride, a->k_row_stride}) &&
               vec_ok(a->values, 1, {a->v_layer_stride, a->v_h_stride, a->v_row_stride});
  const int64_t blocks = (int64_t)a->n_layers * a->batch * a->hv * a->n_ends;
  const size_t shm = (size_t)2 * (a->path_cols + (a->path_cols & 1)) * kCD * sizeof(float);
  if (P.src_vec && P.dst_vec && P.path_vec)
    hipLaunchKernelGGL(tree_commit_kernel<true>, dim3((unsigned)blocks), dim3(256), shm, stream, P);
  else
    hipLaunchKernelGGL(tree_commit_kernel<false>, dim3((unsigned)blocks), dim3(256), shm, stream, P);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

}  // namespace dft
