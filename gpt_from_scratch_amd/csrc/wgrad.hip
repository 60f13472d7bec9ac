// wgrad.hip — weight gradient of a projection, dW[N, K] = dY[M, N]^T X[M, K] or
// added to dW, bf16 / f16, one rounding of the fp32 sum.
//
// M (the tokens) is long and dW small, so dW's 128 x 128 tiles alone leave most
// of the chip idle: the tokens are split between workgroups, whose fp32 partial
// tiles a second launch adds up, in a fixed order, with dW.
//
// A workgroup of four waves owns a tile, a wave 64 x 64 of it (2 x 2 blocks of
// 32x32x16 products).  Both operands are read along the tokens, i.e. transposed
// from their row-major tiles by ds_read_b64_tr_b16.  Tiles of 64 tokens go
// straight from global memory into LDS, double-buffered, one barrier per step;
// the operands of 16 tokens are read while the products of the 16 before run
// (2304 x 768 of 8192 tokens: 41.8 -> 39.4 us).
//
// Bound: the matrix rate; with two workgroups per CU the LDS delivers 2/3 of what
// it can.  Reached with the sum: 690-760 TFLOP/s (8192 x 2304 x 768, 8192 x 768 x
// 3072), 410 on 8192 x 768 x 768, whose partial tiles are 33 MB.  Tiles of 32
// tokens (four workgroups per CU) took 45 and 75 us against 39 and 56.
#include "mi_device.h"
#include "mi_kernels.h"

namespace mi {

namespace {

constexpr int WT = 128;   // rows and columns of a dW tile
constexpr int WM = 64;    // tokens per step
constexpr int CPR = WT / 8;  // 16-byte chunks per staged row
constexpr int TILE = WM * WT;

// LDS: row r keeps 16-byte chunk c at position c ^ swz(r).  A row is one
// 256-byte bank line, and a transposing read covers four consecutive rows and
// four aligned chunks per 32 lanes, which then hit 16 different positions.
__device__ __forceinline__ int wg_swz(int r) { return (r & 3) << 2; }

template <typename E>
__global__ __launch_bounds__(256, 2) void wgrad_kernel(WgradArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t A0[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t A1[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t B0[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t B1[TILE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Workgroups go round-robin over the 8 XCDs: each XCD takes a contiguous run
  // of (split, tile) items, whose operand panels then meet in its L2.
  const int total = gridDim.x, x = blockIdx.x & 7, p = blockIdx.x >> 3;
  const int item = x * (total >> 3) + min(x, total & 7) + p;
  const int tiles = a.tn * a.tk;
  const int split = item / tiles, tile = item % tiles;
  const int n0 = tile / a.tk * WT, k0 = tile % a.tk * WT;
  const int steps = (a.M + WM - 1) / WM;
  const int s0 = (int)((int64_t)steps * split / a.splits);
  const int s1 = (int)((int64_t)steps * (split + 1) / a.splits);

  // Staging: 1 KB slices of four rows; lane i writes chunk position i % 16 of
  // row i / 16, i.e. fetches chunk (i % 16) ^ swz(row).  Chunks past the last
  // column take an offset past every extent and stage as zeros, rows past M
  // end the descriptor.
  uint32_t oa[4], ob[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = 4 * (wave + 4 * m) + lane / CPR;
    const int c = ((lane % CPR) ^ wg_swz(r)) * 8;
    oa[m] = n0 + c < a.N ? (uint32_t)((r * a.dys + c) * 2) : kOobOffset;
    ob[m] = k0 + c < a.K ? (uint32_t)((r * a.xs + c) * 2) : kOobOffset;
  }
  const uint16_t* const ap = (const uint16_t*)a.dy + n0;
  const uint16_t* const bp = (const uint16_t*)a.x + k0;
  const int an = min(WT, a.N - n0), bn = min(WT, a.K - k0);
  auto stage = [&](int s, uint16_t* ta, uint16_t* tb) __attribute__((always_inline)) {
    const int rows = min(WM, a.M - s * WM);
    const auto ra = tile_rsrc(ap + (int64_t)s * WM * a.dys, rows_extent(rows, a.dys, an));
    const auto rb = tile_rsrc(bp + (int64_t)s * WM * a.xs, rows_extent(rows, a.xs, bn));
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      buffer_load_lds16(ra, oa[m], ta + (wave + 4 * m) * 512);
      buffer_load_lds16(rb, ob[m], tb + (wave + 4 * m) * 512);
    }
  };

  // Byte offsets of the transposing reads: row 4 g + (l % 16) / 4, column 32
  // blk + 16 ((l / 16) % 2) + 4 (l % 4).
  const int g = lane >> 5;
  const int wn = wave >> 1, wk = wave & 1;  // the wave's 64 x 64 of the tile
  int fa[2], fb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 4 * g + ((lane & 15) >> 2);
    const int c = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    fa[i] = 2 * (r * WT + (((4 * (2 * wn + i) + c) ^ wg_swz(r)) << 3) + 4 * (lane & 1));
    fb[i] = 2 * (r * WT + (((4 * (2 * wk + i) + c) ^ wg_swz(r)) << 3) + 4 * (lane & 1));
  }
  auto operand = [&](const uint16_t* t, int off, int ks) __attribute__((always_inline)) {
    return tr_operand((const uint16_t*)((const char*)t + off + 2 * 16 * ks * WT), WT);
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
  auto step = [&](int s, const uint16_t* ta, const uint16_t* tb, uint16_t* na,
                  uint16_t* nb) __attribute__((always_inline)) {
    if (s + 1 < s1) stage(s + 1, na, nb);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      opaque(fa[i]);
      opaque(fb[i]);
    }
    u32x4 x[2][2], y[2][2];
    auto read = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        x[ks & 1][i] = operand(ta, fa[i], ks);
        y[ks & 1][i] = operand(tb, fb[i], ks);
      }
    };
    read(0);
#pragma unroll
    for (int ks = 0; ks < WM / 16; ++ks) {
      if (ks + 1 < WM / 16) read(ks + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = E::mfma(x[ks & 1][i], y[ks & 1][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
  stage(s0, A0, B0);
  __syncthreads();
  for (int s = s0; s < s1; s += 2) {
    step(s, A0, B0, A1, B1);
    if (s + 1 < s1) step(s + 1, A1, B1, A0, B0);
  }

  // Accumulator: rows 8 (r / 4) + 4 g + r % 4, column l % 32 of a 32 x 32 block.
  float* const part = a.part + (int64_t)split * a.N * a.K;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int k = k0 + 64 * wk + 32 * j + (lane & 31);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + 64 * wn + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
        if (n < a.N && k < a.K) part[(int64_t)n * a.K + k] = acc[i][j][r];
      }
    }
}

// dW = (dW +) the partial sums, rounded once.  Four adjacent elements per lane.
template <typename E>
__global__ __launch_bounds__(256) void wgrad_sum_kernel(WgradArgs a) {
  const int64_t n = (int64_t)a.N * a.K;
  const int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (i >= n) return;
  const u32x2 w = a.acc ? *(const u32x2*)((const uint16_t*)a.dw + i) : u32x2{0, 0};
  f32x4 v = *(const f32x4*)(a.part + i);
  for (int s = 1; s < a.splits; ++s) v += *(const f32x4*)(a.part + s * n + i);
  u32x2 o;
  o[0] = E::pack2(v[0] + E::to_f32((uint16_t)(w[0] & 0xffffu)),
                  v[1] + E::to_f32((uint16_t)(w[0] >> 16)));
  o[1] = E::pack2(v[2] + E::to_f32((uint16_t)(w[1] & 0xffffu)),
                  v[3] + E::to_f32((uint16_t)(w[1] >> 16)));
  *(u32x2*)((uint16_t*)a.dw + i) = o;
}

template <typename E>
hipError_t launch(const WgradArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(wgrad_kernel<E>, dim3(a.tn * a.tk * a.splits), dim3(256), 0, st, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(wgrad_sum_kernel<E>, dim3((uint32_t)(((int64_t)a.N * a.K / 4 + 255) / 256)),
                     dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace

// Token splits: as many as give every CU two workgroups, of at least 8 steps.
int wgrad_splits(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((N + WT - 1) / WT) * ((K + WT - 1) / WT);
  const int64_t steps = (M + WM - 1) / WM;
  int64_t s = 512 / tiles;
  if (s > steps / 8) s = steps / 8;
  return (int)(s < 1 ? 1 : s);
}

// Whether this takes the place of the general GEMM library (addmm_ with beta = 1,
// which splits no tokens at these sizes).  The kernels alone, us, library / this,
// bf16 (weights of t tiles):
//   M 8192:  768 x 768 (t 36) 49 / 24, 2304 x 768 (108) 65 / 39, 768 x 3072 (144)
//            80 / 51, 4096 x 768 (192) 90.8 / 78.2, 6144 x 768 (288) 113 / 141
//   M 3000:  2304 x 768 34 / 24              M 16384: 1024 x 1024 110 / 52
//   M 2560:  2304 x 768 24.6 / 23.2, 1024 x 1024 (64) 19.7 / 20.8, 768 x 768 19.2 / 16.7
//   M 2048:  2304 x 768 20.3 / 23.2, 1536 x 512 (48) 16.6 / 16.6, 768 x 768 16.5 / 15.4
//   M 1500:  1536 x 512 17.1 / 15.3, 512 x 512 (16) 16.8 / 11.6
//   M 1024:  1536 x 512 11.5 / 13.4, 512 x 512 11.3 / 10.8
//   M 640:   768 x 768 8.8 / 12.0, 768 x 256 (12) 8.6 / 11.4, 256 x 256 (4) 24 / 11
// Below 16 steps the tokens are not split, and there the library's kernel is the
// shorter one but for the smallest weights.  The host bounds such a backward,
// and it spends less on this launch than on torch's addmm_: forward and backward
// of models of 4, 3 and 2 layers on 656, 600 and 726 tokens took 1.99, 1.51 and
// 1.18 ms with this, 2.06, 1.59 and 1.20 with the library.
bool wgrad_suits(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((N + WT - 1) / WT) * ((K + WT - 1) / WT);
  return M >= 256 && tiles <= 192 && (M >= 2560 || tiles <= 48);
}

hipError_t launch_wgrad(int dtype, WgradArgs a, hipStream_t st) {
  a.tn = (a.N + WT - 1) / WT;
  a.tk = (a.K + WT - 1) / WT;
  return dtype == 2 ? launch<BF16>(a, st) : launch<F16>(a, st);
}

}  // namespace mi
