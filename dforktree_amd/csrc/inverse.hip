// Standalone in-place (I+A)^-1 (fc1_block_inverse.py): one wave per matrix.
//
// The matrix (n <= NP = 16, 32 or 64) sits in LDS, NP x NP floats, and is
// replaced there 16-row block by 16-row block, top down.  With X held as
// 16 x 16 tiles, xt[i][j][r] of lane (n, g) = X[16i + n][16j + 4g + r]:
//   X_ij <- E_ij - sum_{m = j}^{i-1} A_im X_mj   (fp32 MFMA 16x16x4, formed
//           transposed, so that the product comes out in this layout)
//   X_ij <- (I + A_ii)^-1 X_ij                   (forward substitution)
// Step m of the substitution takes row m of every column from lane m of each
// 16-lane row (one DPP row broadcast, fused into the multiply-add) and each
// lane's own A[16i + n][16i + m], so the tiles of a block row share one
// register per step and run side by side.  The sums are the forward
// substitution's own, with no product by an inverted diagonal block, and a
// non-finite value goes where it goes there: into its own row of X and the
// rows below that use it, never into the rows above (subst_step).  An element
// A[i][c] that is itself not finite takes in every column of row i up to the
// end of c's 16-column block, as 0 * NaN.
//
// Bound by memory: 2 n^2 floats per matrix.  2048 64 x 64 matrices (67 MB),
// with the copy that keeps the input (about 8 us): 44.5 us with one column
// per lane (each lane read its own 256-byte row, element by element, and ran
// 2016 dependent multiply-adds), 23.0 us here.  16 KiB of LDS at 64 nodes
// holds 10 waves per CU, so 2048 matrices are resident at once, and would
// load, compute and store in step: so every load goes out first, a block row
// is solved as soon as its own rows are in and leaves while the next one is
// solved (4% against copies straight into LDS, waited for at once).
#include "dft_device.h"

namespace dft {
namespace {

// 16-byte chunk c / 4 of row i at chunk position (c / 4) ^ i (mod the row's
// chunks): rows stay contiguous, so a wave's 1 KiB is whole rows, and the
// 16-byte reads of 16 rows at one column hit distinct banks (at 64; 2- and
// 4-way conflicts at 32 and 16, where there are few reads).
template <int NP>
__device__ __forceinline__ int mat_at(int i, int c) {
  return i * NP + ((((c >> 2) ^ i) & (NP / 4 - 1)) << 2) + (c & 3);
}

// Step M of the substitution on the J tiles of a block row: x += na * (x of
// lane M of the 16-lane row), on the lanes from M on.  The lanes below M are
// masked off and lane M's own na is the smallest normal number (x + 2^-126 x
// is x, also for infinities), where zeros would do for finite values: 0 * inf
// and 0 * NaN would carry a bad row M back into the finished rows above it.
// The compiler keeps the broadcast as a move of its own (with two wait states
// after each multiply-add), hence the statement; the two wait states a DPP
// read needs after a vector write are the two moves to the lane mask for the
// first instruction and lie in the three others for the rest.  Every lane of
// the wave is active here.  x must not come straight from an MFMA: the backend
// does not see the reads in here.
#define DFT_STEP4(a, b, c, d) DFT_STEP1(a) DFT_STEP1(b) DFT_STEP1(c) DFT_STEP1(d)
#define DFT_STEP1(k) "v_fmac_f32_dpp %" #k ", %" #k ", %[na] row_newbcast:%c[m] row_mask:0xf bank_mask:0xf\n\t"
#define DFT_STEP_OUT(j) "+v"(t[j][0]), "+v"(t[j][1]), "+v"(t[j][2]), "+v"(t[j][3])
#define DFT_STEP(text, ...)                                                                      \
  asm("s_mov_b32 exec_lo, %[lanes]\n\ts_mov_b32 exec_hi, %[lanes]\n\t" text "s_mov_b64 exec, -1" \
      : __VA_ARGS__                                                                              \
      : [na] "v"(na), [m] "i"(M), [lanes] "i"((int32_t)kLanes))
template <int M, int J>
__device__ __forceinline__ void subst_step(float na, f32x4 (&x)[J]) {
  constexpr uint32_t kLanes = ((0xffffu << M) & 0xffffu) * 0x00010001u;  // of each half wave
  float t[J][4];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) t[j][r] = x[j][r];
  if constexpr (J == 1)
    DFT_STEP(DFT_STEP4(0, 1, 2, 3), DFT_STEP_OUT(0));
  else if constexpr (J == 2)
    DFT_STEP(DFT_STEP4(0, 1, 2, 3) DFT_STEP4(4, 5, 6, 7), DFT_STEP_OUT(0), DFT_STEP_OUT(1));
  else if constexpr (J == 3)
    DFT_STEP(DFT_STEP4(0, 1, 2, 3) DFT_STEP4(4, 5, 6, 7) DFT_STEP4(8, 9, 10, 11), DFT_STEP_OUT(0), DFT_STEP_OUT(1),
             DFT_STEP_OUT(2));
  else
    DFT_STEP(DFT_STEP4(0, 1, 2, 3) DFT_STEP4(4, 5, 6, 7) DFT_STEP4(8, 9, 10, 11) DFT_STEP4(12, 13, 14, 15),
             DFT_STEP_OUT(0), DFT_STEP_OUT(1), DFT_STEP_OUT(2), DFT_STEP_OUT(3));
#pragma unroll
  for (int j = 0; j < J; ++j) x[j] = f32x4{t[j][0], t[j][1], t[j][2], t[j][3]};
}
#undef DFT_STEP
#undef DFT_STEP_OUT
#undef DFT_STEP1
#undef DFT_STEP4

// steps M .. 14 on tiles 0 .. J - 1 of a block row
template <int M, int J>
__device__ __forceinline__ void subst_steps(const float (&na)[16], f32x4 (&x)[J]) {
  if constexpr (M < 15) {
    subst_step<M>(na[M], x);
    subst_steps<M + 1, J>(na, x);
  }
}

// block row I; xr[m][j]: X_mj of the block rows above as MFMA operands
// (element s of lane (n, g): X[16m + 4g + s][16j + n])
// before(I) runs ahead of block row I, after(I) behind it.
template <int NP, int I, class Before, class After>
__device__ __forceinline__ void block_rows(float* a, int n16, int g4, f32x4 (&xr)[NP / 16][NP / 16], Before before,
                                           After after) {
  if constexpr (I < NP / 16) {
    before(I);
    f32x4 x[I + 1];
    if constexpr (I > 0) {
      f32x4 am[I];  // A[16I + n][16m + 4g ..]
#pragma unroll
      for (int m = 0; m < I; ++m)
        am[m] = *reinterpret_cast<const f32x4*>(&a[mat_at<NP>(16 * I + n16, 16 * m + 4 * g4)]);
#pragma unroll
      for (int j = 0; j < I; ++j) {
        x[j] = f32x4{};
#pragma unroll
        for (int m = j; m < I; ++m)
#pragma unroll
          for (int s = 0; s < 4; ++s) x[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xr[m][j][s], am[m][s], x[j], 0, 0, 0);
        x[j] = -x[j];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) x[I][r] = (n16 == 4 * g4 + r) ? 1.f : 0.f;
    float na[16];  // row n of A_II, negated, and subst_step's diagonal (what lies above that meets no active lane)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(&a[mat_at<NP>(16 * I + n16, 16 * I + 4 * c)]);
#pragma unroll
      for (int e = 0; e < 4; ++e) na[4 * c + e] = 4 * c + e == n16 ? 0x1p-126f : -v[e];
    }
    subst_steps<0, I + 1>(na, x);
    // over A's rows 16I .., which nothing reads any more (one wave: its LDS
    // operations run in order)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j <= I; ++j) *reinterpret_cast<f32x4*>(&a[mat_at<NP>(16 * I + n16, 16 * j + 4 * g4)]) = x[j];
    asm volatile("" ::: "memory");
    if constexpr (I + 1 < NP / 16) {
#pragma unroll
      for (int j = 0; j <= I; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s) xr[I][j][s] = a[mat_at<NP>(16 * I + 4 * g4 + s, 16 * j + n16)];
    }
    after(I);
    block_rows<NP, I + 1>(a, n16, g4, xr, before, after);
  }
}

// 16 bytes of a matrix: its floats are aligned, its rows need not be
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// WHOLE: n == NP, the matrix moves as 16-byte pieces; else as 64 / NP rows of
// NP floats per load, the elements past n left out.  us for 2048 matrices in
// cache, a row per load and store in turn (which an unaligned whole matrix
// took too) and now: 20 x 20 8.3 / 5.0, 33 x 33 16.1 / 12.9, 48 x 48 18.7 /
// 14.0; unaligned 16 x 16 6.2 / 3.4, 32 x 32 10.6 / 4.7, 64 x 64 23.6 / 10.9.
template <int NP, bool WHOLE>
__global__ void __launch_bounds__(64) block_inverse_kernel(float* x, int n, int64_t mat_stride) {
  __shared__ alignas(16) float a[NP * NP];
  constexpr int CH = NP / 4;  // 16-byte chunks of a row
  float* m = x + (int64_t)blockIdx.x * mat_stride;
  const int lane = threadIdx.x;
  f32x4 xr[NP / 16][NP / 16];
  if constexpr (WHOLE) {
    constexpr int PB = NP / 16;  // 1 KiB pieces of whole rows per block row
    f32x4 ld[PB * PB];
#pragma unroll
    for (int b = 0; b < PB * PB; ++b) {
      const int i = (64 / CH) * b + lane / CH;
      ld[b] = *reinterpret_cast<const f32x4_a4*>(m + i * NP + 4 * ((lane ^ i) & (CH - 1)));
    }
    block_rows<NP, 0>(
        a, lane & 15, lane >> 4, xr,
        [&](int bi) {
#pragma unroll
          for (int b = 0; b < PB; ++b) *reinterpret_cast<f32x4*>(&a[256 * (PB * bi + b) + 4 * lane]) = ld[PB * bi + b];
          asm volatile("" ::: "memory");
        },
        [&](int bi) {  // (tiles above the diagonal still hold A: zeros)
#pragma unroll
          for (int b = 0; b < PB; ++b) {
            const int i = (64 / CH) * (PB * bi + b) + lane / CH, c = (lane ^ i) & (CH - 1);
            const f32x4 v = *reinterpret_cast<const f32x4*>(&a[256 * (PB * bi + b) + 4 * lane]);
            *reinterpret_cast<f32x4_a4*>(m + i * NP + 4 * c) = (c >> 2) > (i >> 4) ? f32x4{} : v;
          }
        });
  } else {
    // (the loads take clamped, always valid addresses and go out together)
    constexpr int RL = 64 / NP, K = NP / RL, G = K < 16 ? K : 16;  // rows per load, loads, loads per group
    const int r0 = lane / NP, c = lane & (NP - 1);
    float v[K] = {};
#pragma unroll
    for (int k = 0; k < K; k += G)
      if (RL * k < n)  // uniform
#pragma unroll
        for (int e = k; e < k + G; ++e) v[e] = m[min(RL * e + r0, n - 1) * n + min(c, n - 1)];
#pragma unroll
    for (int k = 0; k < K; ++k) a[mat_at<NP>(RL * k + r0, c)] = max(RL * k + r0, c) < n ? v[k] : 0.f;
    asm volatile("" ::: "memory");
    block_rows<NP, 0>(a, lane & 15, lane >> 4, xr, [](int) {}, [](int) {});
#pragma unroll
    for (int k = 0; k < K; k += G)
      if (RL * k < n) {
#pragma unroll
        for (int e = k; e < k + G; ++e) v[e] = a[mat_at<NP>(RL * e + r0, c)];
#pragma unroll
        for (int e = k; e < k + G; ++e)
          if (max(RL * e + r0, c) < n) m[(RL * e + r0) * n + c] = (c >> 4) > ((RL * e + r0) >> 4) ? 0.f : v[e];
      }
  }
}

template <int NP>
void launch(float* x, int n_mats, int n, int64_t mat_stride, hipStream_t stream) {
  if (n == NP)
    hipLaunchKernelGGL((block_inverse_kernel<NP, true>), dim3(n_mats), dim3(64), 0, stream, x, n, mat_stride);
  else
    hipLaunchKernelGGL((block_inverse_kernel<NP, false>), dim3(n_mats), dim3(64), 0, stream, x, n, mat_stride);
}

}  // namespace

int launch_block_inverse(float* x, int n_mats, int n, int64_t mat_stride, hipStream_t stream) {
  if (n <= 16)
    launch<16>(x, n_mats, n, mat_stride, stream);
  else if (n <= 32)
    launch<32>(x, n_mats, n, mat_stride, stream);
  else
    launch<64>(x, n_mats, n, mat_stride, stream);
  return hipGetLastError() == hipSuccess ? DFT_OK : DFT_ERR_LAUNCH;
}

}  // namespace dft
