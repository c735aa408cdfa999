// Tree-parent causal conv1d (fc1_conv.py:7-27, tree_kernels.py:17-33).
//
// For node n of request b and channel c:
//   xt[col] = col < W-1 ? conv_state[slot][c][col] : x[b][col-(W-1)][c]
//   y[b][n][c] = act(sum_j w[c][j] * xt[cidx[b][n][j]] + bias[c])
//   iw[dst][n][c][j-1] = xt[cidx[b][n][j]]            (j >= 1, optional)
// The gather columns are per node, so every thread of a block reads the
// same W indices (scalar loads) and streams channels: block = 256 channels
// x one node, loads and stores coalesced along c.  HBM-bound byte work.
#include "dft_device.h"

namespace dft {

constexpr int kMaxTaps = 8;

__global__ void __launch_bounds__(256) tree_conv_kernel(const dft_conv_args p) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int n = blockIdx.y, b = blockIdx.z;
  if (c >= p.channels) return;
  const int W = p.width;

  // A negative state slot (a padded request) reads slot 0; a negative window
  // slot writes no window.
  int64_t slot = b, dst = b;
  if (p.cs_indices) slot = ld_i(p.cs_indices, b, p.cs_indices_dtype);
  if (p.iw_indices) dst = ld_i(p.iw_indices, b, p.iw_indices_dtype);
  if (slot < 0) slot = 0;

  const int64_t cbase = (int64_t)b * p.cidx_req_stride + (int64_t)n * p.cidx_node_stride;
  float acc = 0.f;
#pragma unroll
  for (int j = 0; j < kMaxTaps; ++j) {
    if (j >= W) break;
    const int64_t col = ld_i(p.cidx, cbase + j, p.cidx_dtype);
    float val;
    if (col < 0 || col >= W - 1 + p.n_nodes)  // outside [conv_state || x]: reads as zero
      val = 0.f;
    else if (col < W - 1)
      val = ld_f(p.conv_state, slot * p.cs_slot_stride + (int64_t)c * p.cs_chan_stride + col * p.cs_col_stride,
                 p.cs_dtype);
    else
      val = ld_f(p.x, (int64_t)b * p.x_req_stride + (col - (W - 1)) * p.x_node_stride + (int64_t)c * p.x_chan_stride,
                 p.x_dtype);
    const float w = ld_f(p.weight, (int64_t)c * p.w_chan_stride + (int64_t)j * p.w_tap_stride, p.w_dtype);
    acc += val * w;
    if (j > 0 && p.iw && dst >= 0)
      st_f(p.iw,
           dst * p.iw_slot_stride + (int64_t)n * p.iw_node_stride + (int64_t)c * p.iw_chan_stride +
               (int64_t)(j - 1) * p.iw_col_stride,
           p.iw_dtype, val);
  }
  if (p.bias) acc += ld_f(p.bias, c, p.bias_dtype);
  const float out = p.silu ? acc / (1.f + expf(-acc)) : acc;
  st_f(p.y, (int64_t)b * p.y_req_stride + (int64_t)n * p.y_node_stride + c, p.y_dtype, out);
}

// The plugin's layout (width 4, bf16 tokens / weights / output / window,
// channel-contiguous rows) where the conv state is of another type or a tree
// has more than 64 nodes (tree_conv4_rows_kernel below takes the rest).  A
// workgroup of one wave covers 512 channels of one node; a thread owns 8
// consecutive channels, so every gathered token row, the weights (8 channels x
// 4 taps) and the output are 16-byte accesses.  The gather columns are uniform
// over the workgroup: the four come in one batch of scalar loads (the index
// width is a template parameter, so no load waits behind a dtype branch), the
// weights go out meanwhile, and the four token loads are issued
// unconditionally (a tap outside the tokens reads row 0 and is discarded).
// The node's window over the channels is one contiguous run (iw[n][c][0..2]):
// the threads' 48-byte pieces go through LDS so that each store instruction
// writes 1 KiB of consecutive bytes (whole lines) instead of 16 bytes every 48.
// The grid is 1-D and XCD-aware: workgroups are dealt to the 8 XCDs round
// robin, so ids that agree mod 8 (one XCD, one L2) cover every node of one
// (request, channel block) and the parents' rows re-read by the children
// stay in that L2.
// us at 8192 channels with the window, here and on the per-channel kernel
// above: 64 requests x 32 nodes with an fp32 conv state 44.0 / 160.2, 32 x 65
// with a bf16 one 32.4 / 163.2, 1 x 96 5.8 / 10.6.
// Request b's index (a slot) from an int32 or int64 array as two 32-bit
// loads with no branch between them; idx NULL reads nothing (returns 0).
__device__ __forceinline__ int64_t req_index(const void* idx, int dt, int b) {
  if (!idx) return 0;
  const int32_t* w = static_cast<const int32_t*>(idx);
  const bool wide = dt == DFT_I64;
  const int32_t lo = w[wide ? 2 * b : b];
  const int32_t hi = w[wide ? 2 * b + 1 : b];
  return wide ? (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo) : (int64_t)lo;
}

template <bool CIDX64>
__global__ void __launch_bounds__(64) tree_conv4_bf16_kernel(const dft_conv_args p, int cblocks) {
  __shared__ u32x4 stage[64 * 3];
  const int id = blockIdx.x;
  const int k = id >> 3;
  const int n = k % p.n_nodes;
  const int pair = (k / p.n_nodes) * 8 + (id & 7);
  if (pair >= p.batch * cblocks) return;  // uniform over the block
  const int cb = pair % cblocks, b = pair / cblocks;
  const int nact = min(64, (p.channels - cb * 512) / 8);  // threads with channels
  const bool active = (int)threadIdx.x < nact;
  const int c0 = (cb * 64 + threadIdx.x) * 8;

  // the node's four tap columns: independent loads, one wait
  const int64_t cbase = (int64_t)b * p.cidx_req_stride + (int64_t)n * p.cidx_node_stride;
  int64_t col[4];
  if constexpr (CIDX64) {
    const int64_t* ci = static_cast<const int64_t*>(p.cidx) + cbase;
#pragma unroll
    for (int j = 0; j < 4; ++j) col[j] = ci[j];
  } else {
    const int32_t* ci = static_cast<const int32_t*>(p.cidx) + cbase;
#pragma unroll
    for (int j = 0; j < 4; ++j) col[j] = ci[j];
  }
  // The request's conv-state slot and window slot come in the same batch:
  // read where they are used (behind a dtype branch, and the window slot
  // after the arithmetic), each was one more dependent round trip, which a
  // batch-1 launch waits out in full.  Branch-free: the index's low word, and
  // its high word for 64-bit indices (for 32-bit ones the same word again).
  const int64_t slot_raw = req_index(p.cs_indices, p.cs_indices_dtype, b);
  const int64_t dst_raw = req_index(p.iw_indices, p.iw_indices_dtype, b);
  // the weights (8 channels x 4 taps) do not depend on them
  const int cw = active ? c0 : 0;
  const u32x4* wp = reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.weight) + (int64_t)cw * 4);
  uint16_t w[32];  // w[4 e + j]: channel c0 + e, tap j
#pragma unroll
  for (int q = 0; q < 4; ++q) *reinterpret_cast<u32x4*>(&w[8 * q]) = wp[q];
  int64_t slot = p.cs_indices ? slot_raw : b;
  const int64_t dst = p.iw_indices ? dst_raw : b;

  if (active) {
    const uint16_t* xb = static_cast<const uint16_t*>(p.x) + (int64_t)b * p.x_req_stride + c0;
    // the state slot (needed by conv-state taps only); a negative one reads slot 0
    if (slot < 0) slot = 0;
    // Token rows: every load is issued (a tap outside the tokens reads row 0
    // and is discarded), so none waits on a branch.  A tap on a bf16 conv-state
    // column (a node within two edges of the root) gathers the column's 8
    // values into the same registers instead, issued with the token loads
    // (the per-element path below waits for 8 two-byte loads per tap in turn).
    const bool cs_bf16 = p.cs_dtype == DFT_BF16;
    u32x4 raw[4];
    bool tok[4], csg[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      tok[j] = col[j] >= 3 && col[j] < 3 + p.n_nodes;
      csg[j] = cs_bf16 && col[j] >= 0 && col[j] < 3;  // uniform
      if (csg[j]) {
        const uint16_t* cs = static_cast<const uint16_t*>(p.conv_state) + slot * p.cs_slot_stride +
                             (int64_t)c0 * p.cs_chan_stride + col[j] * p.cs_col_stride;
        uint16_t h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = cs[(int64_t)e * p.cs_chan_stride];
        raw[j] = *reinterpret_cast<const u32x4*>(h);
      } else {
        raw[j] = *reinterpret_cast<const u32x4*>(xb + (tok[j] ? col[j] - 3 : 0) * p.x_node_stride);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (!tok[j] && !csg[j]) raw[j] = u32x4{0u, 0u, 0u, 0u};

    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = p.bias ? ld_f(p.bias, c0 + e, p.bias_dtype) : 0.f;
    uint16_t win[24];  // win[3 e + j - 1]
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v[8];
      if (col[j] >= 0 && col[j] < 3 && !csg[j]) {  // a conv-state column of another dtype
#pragma unroll
        for (int e = 0; e < 8; ++e)
          v[e] = ld_f(p.conv_state,
                      slot * p.cs_slot_stride + (int64_t)(c0 + e) * p.cs_chan_stride + col[j] * p.cs_col_stride,
                      p.cs_dtype);
      } else {  // a token row, a gathered bf16 state column, or zero outside [conv_state || x]
        const uint16_t* h = reinterpret_cast<const uint16_t*>(&raw[j]);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = bf16_bits_to_f32(h[e]);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        acc[e] += v[e] * bf16_bits_to_f32(w[4 * e + j]);
        if (j > 0) win[3 * e + j - 1] = f32_to_bf16_bits(v[e]);
      }
    }
    uint16_t out[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) out[e] = f32_to_bf16_bits(p.silu ? acc[e] / (1.f + expf(-acc[e])) : acc[e]);
    *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p.y) + (int64_t)b * p.y_req_stride + (int64_t)n * p.y_node_stride +
                              c0) = *reinterpret_cast<const u32x4*>(out);
    if (p.iw) {
#pragma unroll
      for (int q = 0; q < 3; ++q) stage[threadIdx.x * 3 + q] = *reinterpret_cast<const u32x4*>(&win[8 * q]);
    }
  }
  if (p.iw) {
    __syncthreads();
    if (dst >= 0) {  // uniform over the block (one request); a negative slot writes no window
      u32x4* iw = reinterpret_cast<u32x4*>(static_cast<uint16_t*>(p.iw) + dst * p.iw_slot_stride +
                                           (int64_t)n * p.iw_node_stride + (int64_t)cb * 512 * 3);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int i = threadIdx.x + 64 * q;
        if (i < nact * 3) iw[i] = stage[i];
      }
    }
  }
}

// The fast path's main form, for a bf16 conv state and trees of up to 64
// nodes: a workgroup of W waves takes 256 channels of one request and holds
// every column of [conv_state || x] in LDS (and a row of zeros for taps
// outside it), 512 bytes each.  The token rows are copied in (two per 1 KiB
// copy) without waiting for the tap columns and are read from memory once
// instead of once per tap; a lane owns 4 channels, whose weights stay in
// registers; a wave takes every W-th node of the workgroup's share and reads
// the next node's columns ahead.
//
// A node's window over the slice (iw[n][c][0..2], 1.5 KiB) goes through LDS
// and leaves as 16-byte pieces of whole lines, non-temporal: it is read back
// for the accepted nodes only, and kept out of the caches it does not push
// out the tokens and y (40 -> 37 us per launch; y is read by the verify that
// follows, and stored past the caches too it made that pair slower: 83 -> 86
// us at batch 64, although the conv alone took 30).
//
// 64 requests x 32 nodes x 8192 channels, six layers in turn (168 MB each):
// 54.8 us per launch with a one-wave workgroup per node that gathered its
// four rows from memory, 37.2 here, 4.5 TB/s; a streaming probe moves 5.2
// TB/s at this mix of reads and writes.  The same rows in cache: 42.0 -> 32.8.
// Batch 4: 8.2 -> 5.6, batch 1 (plugin step, 24 layers): 354 -> 334, and 330
// -> 318 once no load of the prologue waited for another.  8 waves; 4 took 1.2
// us longer, 16 4 us (small trees: launch_conv4_rows).
constexpr int kConvNodes = 64, kConvSlice = 256;

// rows of the workgroup's LDS: zeros, 3 state columns, the tokens (an odd
// count's last copy fills one more)
__host__ __device__ constexpr int conv_rows(int n) { return 4 + n + (n & 1); }

// Request b's index (b itself without an array) by scalar loads: the array is
// not written by the launch.
__device__ __forceinline__ int64_t uniform_req_index(const void* idx, int dt, int b) {
  if (!idx) return b;
  typedef const __attribute__((address_space(4))) int32_t* Words;
  const Words w = (Words)(uintptr_t)idx;
  const bool wide = dt == DFT_I64;
  const int half = wide ? 0 : 1;  // (shifts: selected addresses become a branch)
  const int32_t lo = w[(2 * b) >> half], hi = w[(2 * b + 1) >> half];
  return wide ? (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo) : (int64_t)lo;
}

// 4 channels (of lane l) of the four rows at these byte offsets
__device__ __forceinline__ void tap_rows(const uint16_t* rows, const int* taps, int n, int lane, uint2 (&r)[4]) {
  const int4 t = *reinterpret_cast<const int4*>(&taps[4 * n]);
  const char* base = reinterpret_cast<const char*>(rows) + 8 * lane;
  r[0] = *reinterpret_cast<const uint2*>(base + t.x);
  r[1] = *reinterpret_cast<const uint2*>(base + t.y);
  r[2] = *reinterpret_cast<const uint2*>(base + t.z);
  r[3] = *reinterpret_cast<const uint2*>(base + t.w);
}

template <bool CIDX64, int W>
__global__ void __launch_bounds__(64 * W) tree_conv4_rows_kernel(const dft_conv_args p, int cblocks, int splits) {
  // Every load of the prologue goes out before anything waits for one of
  // them: read where they are used, the tap columns were waited for (and with
  // them the row copies ahead of them) before the weights and the state were
  // asked for.  The arguments are forced into scalar registers first, for the
  // same reason.
  asm volatile("" ::"s"(p.batch), "s"(p.n_nodes), "s"(p.channels), "s"(p.x), "s"(p.x_req_stride),
               "s"(p.x_node_stride), "s"(p.conv_state), "s"(p.cs_slot_stride), "s"(p.cs_chan_stride), "s"(p.cs_col_stride), "s"(p.cs_indices), "s"(p.cs_indices_dtype), "s"(p.weight),
               "s"(p.cidx), "s"(p.cidx_req_stride), "s"(p.cidx_node_stride), "s"(p.iw_indices), "s"(p.iw_indices_dtype),
               "s"(cblocks), "s"(splits));
  extern __shared__ u32x4 conv_lds[];
  const int N = p.n_nodes;
  uint16_t* rows = reinterpret_cast<uint16_t*>(conv_lds);                // [conv_rows(N)][256]
  int* taps = reinterpret_cast<int*>(rows + conv_rows(N) * kConvSlice);  // [N][4] byte offsets into rows
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint16_t* stage = reinterpret_cast<uint16_t*>(taps + 4 * N) + wave * 3 * kConvSlice;  // the wave's window

  // ids that agree mod 8 (one XCD) hold the node shares of a (request, slice)
  const int id = blockIdx.x, k = id >> 3;
  const int split = k % splits, pair = (k / splits) * 8 + (id & 7);
  if (pair >= p.batch * cblocks) return;  // uniform over the workgroup
  const int cb = pair % cblocks, b = pair / cblocks;
  const int cbase = cb * kConvSlice, nch = min(kConvSlice, p.channels - cbase);  // a multiple of 8

  // the slots (a negative state slot reads slot 0, a negative window slot writes no window)
  const int64_t slot_raw = uniform_req_index(p.cs_indices, p.cs_indices_dtype, b);
  const int64_t dst = uniform_req_index(p.iw_indices, p.iw_indices_dtype, b);
  {
    // (channels past the last read channel 0 of the slice instead)
    const uint16_t* xb = static_cast<const uint16_t*>(p.x) + (int64_t)b * p.x_req_stride + cbase;
    const int c8 = 8 * (lane & 31), half = lane >> 5;
    for (int r = 2 * wave; r < N; r += 2 * W)
      __builtin_amdgcn_global_load_lds(xb + min(r + half, N - 1) * p.x_node_stride + (c8 < nch ? c8 : 0),
                                       (__attribute__((address_space(3))) void*)(rows + (4 + r) * kConvSlice), 16, 0, 0);
  }
  // one tap column per thread (the low and the high word of a 64-bit one)
  const int tap = min(tid, 4 * N - 1);
  const int64_t tap_at = (int64_t)b * p.cidx_req_stride + (int64_t)(tap >> 2) * p.cidx_node_stride + (tap & 3);
  const int32_t* ci = static_cast<const int32_t*>(p.cidx) + (CIDX64 ? 2 * tap_at : tap_at);
  const int32_t col_lo = ci[0], col_hi = CIDX64 ? ci[1] : 0;
  const int c0 = 4 * lane;
  const bool active = c0 < nch;
  const u32x4* wp = reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.weight) +
                                                   (int64_t)(cbase + (active ? c0 : 0)) * 4);
  const u32x4 wraw[2] = {wp[0], wp[1]};
  // the state: a channel per thread, or every 64 W-th
  constexpr int SC = W < 4 ? 4 / W : 1;
  const uint16_t* cs = static_cast<const uint16_t*>(p.conv_state) + (slot_raw < 0 ? 0 : slot_raw) * p.cs_slot_stride +
                       (int64_t)cbase * p.cs_chan_stride;
  uint16_t state[SC][3];
#pragma unroll
  for (int q = 0; q < SC; ++q) {
    const uint16_t* col = cs + (int64_t)min(tid + 64 * W * q, nch - 1) * p.cs_chan_stride;
#pragma unroll
    for (int j = 0; j < 3; ++j) state[q][j] = col[j * p.cs_col_stride];
  }
  __builtin_amdgcn_sched_barrier(0);

  if (tid < 4 * N) {
    const int64_t col = CIDX64 ? (int64_t)(((uint64_t)(uint32_t)col_hi << 32) | (uint32_t)col_lo) : (int64_t)col_lo;
    taps[tid] = col >= 0 && col < 3 + N ? 2 * kConvSlice * (1 + (int)col) : 0;
  }
  float w[16];  // w[4 e + j]: channel c0 + e, tap j
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      w[8 * q + 2 * e] = __uint_as_float(wraw[q][e] << 16);
      w[8 * q + 2 * e + 1] = __uint_as_float(wraw[q][e] & 0xffff0000u);
    }
#pragma unroll
  for (int q = 0; q < SC; ++q) {
    const int c = tid + 64 * W * q;
    if (c < nch) {
#pragma unroll
      for (int j = 0; j < 3; ++j) rows[(1 + j) * kConvSlice + c] = state[q][j];
    }
  }
  float bias[4] = {0.f, 0.f, 0.f, 0.f};
  if (p.bias) {  // uniform
#pragma unroll
    for (int e = 0; e < 4; ++e) bias[e] = active ? ld_f(p.bias, cbase + c0 + e, p.bias_dtype) : 0.f;
  }
  if (tid < 64) *reinterpret_cast<uint2*>(rows + 4 * tid) = uint2{0u, 0u};
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the row copies
  __syncthreads();

  uint16_t* yb = static_cast<uint16_t*>(p.y) + (int64_t)b * p.y_req_stride + cbase + c0;
  const bool window = p.iw && dst >= 0;
  uint16_t* iwb = static_cast<uint16_t*>(p.iw) + dst * p.iw_slot_stride + 3 * cbase;
  const int pieces = 3 * nch / 8;  // of a node's window
  const int share = (N + splits - 1) / splits, n_end = min(N, (split + 1) * share);
  int n = split * share + wave;
  uint2 next[4] = {};
  if (n < n_end) tap_rows(rows, taps, n, lane, next);
  for (; n < n_end; n += W) {
    const uint2 r[4] = {next[0], next[1], next[2], next[3]};
    if (n + W < n_end) tap_rows(rows, taps, n + W, lane, next);
    float acc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = bias[e];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[0] += __uint_as_float(r[j].x << 16) * w[j];
      acc[1] += __uint_as_float(r[j].x & 0xffff0000u) * w[4 + j];
      acc[2] += __uint_as_float(r[j].y << 16) * w[8 + j];
      acc[3] += __uint_as_float(r[j].y & 0xffff0000u) * w[12 + j];
    }
    if (p.silu) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = acc[e] / (1.f + expf(-acc[e]));
    }
    if (active) {
      const bf16x2 lo = __builtin_convertvector((f32x2{acc[0], acc[1]}), bf16x2);  // round to nearest even
      const bf16x2 hi = __builtin_convertvector((f32x2{acc[2], acc[3]}), bf16x2);
      uint2 o;
      __builtin_memcpy(&o.x, &lo, 4);
      __builtin_memcpy(&o.y, &hi, 4);
      *reinterpret_cast<uint2*>(yb + n * p.y_node_stride) = o;
    }
    if (window) {
      // [channel][tap 1 .. 3]; a pair of channels is three words: (t1 t2) (t3 t1') (t2' t3')
      uint2* st = reinterpret_cast<uint2*>(stage + 12 * lane);
      const uint32_t a1 = r[1].x, a2 = r[2].x, a3 = r[3].x, b1 = r[1].y, b2 = r[2].y, b3 = r[3].y;
      st[0] = uint2{__builtin_amdgcn_perm(a2, a1, 0x05040100u), __builtin_amdgcn_perm(a1, a3, 0x07060100u)};
      st[1] = uint2{__builtin_amdgcn_perm(a3, a2, 0x07060302u), __builtin_amdgcn_perm(b2, b1, 0x05040100u)};
      st[2] = uint2{__builtin_amdgcn_perm(b1, b3, 0x07060100u), __builtin_amdgcn_perm(b3, b2, 0x07060302u)};
      asm volatile("" ::: "memory");  // (one wave: its LDS operations run in order)
      const u32x4* sv = reinterpret_cast<const u32x4*>(stage);
      const u32x4 v0 = sv[lane], v1 = sv[64 + (lane & 31)];
      u32x4* iw = reinterpret_cast<u32x4*>(iwb + n * p.iw_node_stride);
      if (lane < pieces) __builtin_nontemporal_store(v0, iw + lane);
      if (lane < 32 && 64 + lane < pieces) __builtin_nontemporal_store(v1, iw + 64 + lane);
      asm volatile("" ::: "memory");
    }
  }
}

static bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

// The fast path needs the plugin's layout; anything else takes the
// per-channel kernel above.
static bool conv4_bf16_ok(const dft_conv_args* a) {
  if (a->width != 4 || a->channels % 8) return false;
  if (a->x_dtype != DFT_BF16 || a->w_dtype != DFT_BF16 || a->y_dtype != DFT_BF16) return false;
  if (a->x_chan_stride != 1 || a->x_node_stride % 8 || a->x_req_stride % 8 || !aligned16(a->x)) return false;
  if (a->w_chan_stride != 4 || a->w_tap_stride != 1 || !aligned16(a->weight)) return false;
  if (a->y_node_stride % 8 || a->y_req_stride % 8 || !aligned16(a->y)) return false;
  if (a->iw && (a->iw_dtype != DFT_BF16 || a->iw_col_stride != 1 || a->iw_chan_stride != 3 || a->iw_node_stride % 8 ||
                a->iw_slot_stride % 8 || !aligned16(a->iw)))
    return false;
  return true;
}

// A launch of few (request, slice) pairs divides each pair's nodes over
// several workgroups, which each copy all rows in, until there is one per CU
// or a wave has one node (batch 1: 334 us per plugin step, 375 undivided).
template <int W>
static void launch_rows_kernel(const dft_conv_args* a, int cblocks, int64_t pairs8, hipStream_t stream) {
  int splits = 1;
  while (splits * W < a->n_nodes && pairs8 * 8 * splits < 256) splits *= 2;
  const size_t lds = 2 * kConvSlice * (size_t)conv_rows(a->n_nodes) + 16 * a->n_nodes + 6 * kConvSlice * W;
  const dim3 grid((unsigned)(pairs8 * 8 * splits)), block(64 * W);
  if (a->cidx_dtype == DFT_I64)
    hipLaunchKernelGGL((tree_conv4_rows_kernel<true, W>), grid, block, lds, stream, *a, cblocks, splits);
  else
    hipLaunchKernelGGL((tree_conv4_rows_kernel<false, W>), grid, block, lds, stream, *a, cblocks, splits);
}

// 8 waves per workgroup, or fewer where they would have no node to take: a
// launch of many pairs is then bound by the waves it starts.  Beyond 4 nodes a
// launch below kConvPairs is not, and the 8 share the copies.  us for 8192
// channels (32 pairs per request), without and with the window, 8 waves / fewer
// (in brackets a one-wave workgroup per node, the kernel above):
//   batch 64, 1 node    7.3 / 4.5   [5.2]    7.8 / 5.0   [5.9]
//   batch 64, 3         9.0 / 6.4   [7.9]    9.9 / 7.3   [9.7]
//   batch 512, 1       38.9 / 17.1 [18.4]   39.1 / 18.0 [20.8]
//   batch 512, 5       56.8 / 37.9 [47.4]   61.4 / 44.9 [58.4]
//   batch 64, 12       13.4 / 11.0 [17.2]   14.5 / 13.0 [20.7]
//   batch 8, 8          3.9 / 4.0   [5.2]    4.3 / 4.6   [5.9]   (8 waves taken)
//   batch 8, 3          3.7 / 3.6   [4.6]    3.9 / 3.8   [5.1]
// More nodes than the LDS rows hold, or a conv state of another type, take the
// per-node kernel.
constexpr int64_t kConvPairs = 1024;
static bool launch_conv4_rows(const dft_conv_args* a, hipStream_t stream) {
  if (a->cs_dtype != DFT_BF16 || a->n_nodes > kConvNodes) return false;
  const int cblocks = (a->channels + kConvSlice - 1) / kConvSlice;
  const int64_t pairs8 = ((int64_t)a->batch * cblocks + 7) / 8;
  if (pairs8 * 8 > (int64_t)0xffffffffll / (64 * 8)) return false;  // work-items in 32 bits
  if (a->n_nodes <= 2)
    launch_rows_kernel<2>(a, cblocks, pairs8, stream);
  else if (a->n_nodes <= 4 || (a->n_nodes <= 12 && pairs8 * 8 >= kConvPairs))
    launch_rows_kernel<4>(a, cblocks, pairs8, stream);
  else
    launch_rows_kernel<8>(a, cblocks, pairs8, stream);
  return true;
}

int launch_tree_conv(const dft_conv_args* a, hipStream_t stream) {
  if (conv4_bf16_ok(a) && launch_conv4_rows(a, stream)) {
  } else if (conv4_bf16_ok(a)) {
    const int cblocks = (a->channels + 511) / 512;
    const int64_t pairs8 = ((int64_t)a->batch * cblocks + 7) / 8;
    const dim3 grid((unsigned)(pairs8 * 8 * a->n_nodes));
    if (a->cidx_dtype == DFT_I64)
      hipLaunchKernelGGL(tree_conv4_bf16_kernel<true>, grid, dim3(64), 0, stream, *a, cblocks);
    else
      hipLaunchKernelGGL(tree_conv4_bf16_kernel<false>, grid, dim3(64), 0, stream, *a, cblocks);
  } else {
    const dim3 grid((unsigned)((a->channels + 255) / 256), (unsigned)a->n_nodes, (unsigned)a->batch);
    hipLaunchKernelGGL(tree_conv_kernel, grid, dim3(256), 0, stream, *a);
  }
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

}  // namespace dft
