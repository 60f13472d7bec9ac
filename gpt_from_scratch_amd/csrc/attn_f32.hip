// attn_f32.hip — flash attention for fp32 tensors on the fp32 matrix cores.
//
// fp32 in, fp32 products and sums (v_mfma_f32_16x16x4_f32), fp32 out: nothing
// is rounded below fp32 anywhere.  Head dims 16, 32, 64 and 128, any sequence
// length (tails are masked), any row alignment (rows that are not 16-byte
// aligned are fetched element by element).  Counterparts: `_attn_fwd`
// (core/myFlashAttn.py:447-728), `_attn_bwd_LoopKV` (:1069-1317) and
// `_attn_bwd_LoopQ` (:795-1066).
//
// Layout.  A 16x16x4 product takes A[l % 16][l / 16] and B[l / 16][l % 16]
// from lane l and leaves C[4 * (l / 16) + r][l % 16] in its register r.  With
// i = l % 16 and g = l / 16:
//   * a wave owns 16 rows of one side (queries, or keys for dK/dV), resident
//     as B operands: lane (i, g) holds columns 16 s + 4 g + jj of row i;
//   * the other side is streamed through LDS in 64-row tiles.  Scores are
//     formed as (streamed x resident): the A operand is a 16-byte LDS read per
//     lane (row i of a 16-row block, columns 16 s + 4 g ..), which feeds the
//     four products jj;
//   * the accumulator of such a block holds streamed rows 4 g + r of resident
//     row i, which is just the B operand of the second product (its k index is
//     the lane group g): probabilities never move between lanes.  That
//     product's A operand is the streamed tile transposed: lane (i, g) reads W
//     adjacent columns W i .. of row 4 g + r, one 16-byte read for four
//     products, and row 4 g + r' of its accumulator j is then column
//     W (4 g + r') + j, so a lane ends with runs of 4 W adjacent columns of
//     its row and stores them directly.
// 16-byte chunk c of row r is kept at chunk c ^ (r mod 16) (rows of fewer than 16
// chunks: see f32_swz), which puts the lanes of either read on different banks:
// 1.4 to 1.6 conflict cycles per LDS instruction measured on large grids, of which
// there are 0.31 per 32-cycle product.
//
// Bound: the fp32 matrix rate (157 TFLOP/s).  One 16-byte LDS read per lane
// feeds four 32-cycle products, a quarter of the LDS bandwidth, so 16 rows per
// wave are enough; the softmax is 16 exponentials per 128 products at D = 64.
// Matrix cores busy 75% (forward) and 79% (backward) of a large grid's launch, 51
// and 59% at B2 H12 S1000 D64, whose last workgroups run alone.
// Reached, causal, products executed (the backward's recomputed ones counted):
// B4 H16 S2048 D64 forward 301 us (115 TFLOP/s), backward 1017 us (118); on the
// vector ALUs these took 1357 and 5500 us, B2 H12 S1000 D64 216 and 774 us (now
// 42 and 129) and B1 H12 S256 D64 38 and 105 us (8.5 and 17).  Errors against
// float64 are no larger than the vector kernels' (partial_sums); with one sum per
// product they were, and these took 298 and 979, 40 and 120, 8.5 and 16.6 us.
#include <type_traits>

#include "mi_device.h"
#include "mi_kernels.h"

namespace mi {

namespace {

constexpr int TR = 64;   // rows per streamed tile
constexpr int NT = 256;  // threads per workgroup

template <int D>
struct Cfg {
  static constexpr int CPR = D / 4;                       // 16-byte chunks per row
  static constexpr int RPL = CPR >= 16 ? 1 : 16 / CPR;    // rows per 256-byte bank line
  static constexpr int NCH = TR * CPR / NT;               // chunks a thread stages per tile
  static constexpr int KB = D / 16;                       // 16-column blocks
  static constexpr int W = KB >= 4 ? 4 : KB;              // adjacent columns per lane
  static constexpr int NH = KB / W;                       // 16 W-column spans
  // Partial sums of a score and of a dO V^T product.  Scores have the same in
  // both directions, so that the backward's P repeats the forward's rounding.
  static constexpr int NPS = D == 16 ? 2 : D == 128 ? 8 : 4;
  static constexpr int NPD = D == 16 ? 2 : 8;
};

// Chunk swizzle of a row: 16 rows of one chunk column, and the chunks of one
// row, land on 16 different 16-byte bank groups.
template <int D>
__device__ __forceinline__ int f32_swz(int r) {
  return (r / Cfg<D>::RPL) & ((Cfg<D>::CPR < 16 ? Cfg<D>::CPR : 16) - 1);
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Reductions over the four lane groups g of a row i (lanes i, i + 16, ...).
__device__ __forceinline__ float max_groups(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float sum_groups(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return sum_halves(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// Four adjacent floats of a row: one 16-byte access, or four when rows are
// not 16-byte aligned.
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* p) {
  if constexpr (VEC) return *(const f32x4*)p;
  return f32x4{p[0], p[1], p[2], p[3]};
}
template <bool VEC>
__device__ __forceinline__ void store4(float* p, f32x4 v) {
  if constexpr (VEC) {
    *(f32x4*)p = v;
  } else {
    p[0] = v[0]; p[1] = v[1]; p[2] = v[2]; p[3] = v[3];
  }
}

// A thread's chunks of the 64-row tile at row0, to be written to LDS once the
// tile before it has been used; rows past S are zeros.  The descriptor of
// aligned rows ends at row S, so its loads need no test and stay in flight.
template <int D, bool VEC>
__device__ __forceinline__ void fetch_tile(const float* p, int64_t ss, int row0, int S,
                                           f32x4 (&t)[Cfg<D>::NCH]) {
  using C = Cfg<D>;
  if constexpr (VEC) {
    const int rows = min(S - row0, TR);
    const auto rs = tile_rsrc(p + row0 * ss, (uint32_t)(((rows - 1) * ss + D) * 4));
#pragma unroll
    for (int u = 0; u < C::NCH; ++u) {
      const int idx = threadIdx.x + NT * u;
      const uint32_t off = ((uint32_t)(idx / C::CPR) * (uint32_t)ss + 4 * (idx % C::CPR)) * 4;
      t[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
    }
  } else {
#pragma unroll
    for (int u = 0; u < C::NCH; ++u) {
      const int idx = threadIdx.x + NT * u;
      const int row = row0 + idx / C::CPR;
      t[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (row < S) t[u] = load4<VEC>(p + row * ss + 4 * (idx % C::CPR));
    }
  }
}
template <int D>
__device__ __forceinline__ void put_tile(float* lds, const f32x4 (&t)[Cfg<D>::NCH]) {
#pragma unroll
  for (int u = 0; u < Cfg<D>::NCH; ++u) {
    const int idx = threadIdx.x + NT * u;
    const int r = idx / Cfg<D>::CPR;
    *(f32x4*)(lds + r * D + 4 * ((idx % Cfg<D>::CPR) ^ f32_swz<D>(r))) = t[u];
  }
}

// Resident row as B operands; a row past the end is read as the last one (its
// results are never stored).
template <int D, bool VEC>
__device__ __forceinline__ void load_resident(const float* p, int64_t ss, int row, int g,
                                              f32x4 (&f)[Cfg<D>::KB]) {
#pragma unroll
  for (int s = 0; s < Cfg<D>::KB; ++s) f[s] = load4<VEC>(p + row * ss + 16 * s + 4 * g);
}

// (rows 16 b .. of the tile) x (resident rows), over the head dim: NP partial
// sums of D / NP products each, added by halves.  One chain of D products
// rounds more: errors against float64 at S = 48, D = 128, causal, were 1.7 (O)
// and 1.6 (dQ) times those of the vector kernels, whose eight lanes' chains are
// added by halves too; with Cfg's partial sums they are 0.89 and 0.99 times.
// The scheduling barrier keeps one partial sum's products in flight at a time:
// all of them interleaved need up to 90 more registers (50 to 70 bytes of scratch
// at D = 64 and 128) and ran no faster.
template <int D, int NP, int LO = 0, int HI = NP>
__device__ __forceinline__ f32x4 partial_sums(const f32x4 (&x)[Cfg<D>::KB],
                                              const f32x4 (&f)[Cfg<D>::KB]) {
  if constexpr (HI - LO > 1) {
    const f32x4 lo = partial_sums<D, NP, LO, (LO + HI) / 2>(x, f);
    __builtin_amdgcn_sched_barrier(0);
    return lo + partial_sums<D, NP, (LO + HI) / 2, HI>(x, f);
  } else {
    constexpr int N = D / 4 / NP;  // four products each
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = N * LO; e < N * HI; ++e) acc = mfma4(x[e / 4][e % 4], f[e / 4][e % 4], acc);
    return acc;
  }
}
template <int D, int NP>
__device__ __forceinline__ f32x4 row_product(const float* tile, int b, int i, int g,
                                             const f32x4 (&f)[Cfg<D>::KB]) {
  f32x4 x[Cfg<D>::KB];
#pragma unroll
  for (int s = 0; s < Cfg<D>::KB; ++s)
    x[s] = *(const f32x4*)(tile + (16 * b + i) * D + 4 * ((4 * s + g) ^ f32_swz<D>(i)));
  return partial_sums<D, NP>(x, f);
}

// acc += (rows 16 b .. of the tile, transposed) x p, p in accumulator form.
template <int D>
__device__ __forceinline__ void col_product(const float* tile, int b, int i, int g, f32x4 p,
                                            f32x4 (&acc)[Cfg<D>::KB]) {
  using C = Cfg<D>;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int rr = 4 * g + r;
#pragma unroll
    for (int h = 0; h < C::NH; ++h) {
      const int col = 16 * C::W * h + C::W * i;
      const float* x = tile + (16 * b + rr) * D + 4 * ((col / 4) ^ f32_swz<D>(rr)) + col % 4;
      float v[C::W];
      __builtin_memcpy(v, __builtin_assume_aligned(x, 4 * C::W), sizeof(v));
#pragma unroll
      for (int j = 0; j < C::W; ++j) acc[h * C::W + j] = mfma4(v[j], p[r], acc[h * C::W + j]);
    }
  }
}

// A wave's 16 x D result (transposed in the accumulators) times `sc`, to the
// lane's row at `row`.
template <int D, bool VEC>
__device__ __forceinline__ void put_rows(float* row, int g, const f32x4 (&acc)[Cfg<D>::KB],
                                         float sc) {
  using C = Cfg<D>;
#pragma unroll
  for (int h = 0; h < C::NH; ++h)
#pragma unroll
    for (int c = 0; c < C::W; ++c) {  // the run's chunk c: elements W r' + j = 4 c ..
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * c + e;
        v[e] = acc[h * C::W + x % C::W][x / C::W] * sc;
      }
      store4<VEC>(row + 16 * C::W * h + 4 * C::W * g + 4 * c, v);
    }
}

// Workgroup -> item, items sorted longest first.  Workgroups w and w + n_cu run
// on one compute unit at a time, so every odd round of n_cu workgroups is
// taken in reverse and long items share a unit with short ones (0: keep the
// order).  A round within one XCD is every eighth workgroup.
__device__ __forceinline__ int snake(int w, int n, int n_cu) {
  if (n_cu == 0) return w;
  const int round = w / n_cu;
  if (!(round & 1) || (round + 1) * n_cu > n) return w;
  const int x = w & 7, p = (w % n_cu) >> 3;
  return round * n_cu + ((n_cu / 8 - 1 - p) << 3) + x;
}

// Forward.  A workgroup of four waves owns 64 / KS queries: KS waves share the
// same 16 queries and split the streamed blocks of 16 keys between them, each
// with its own running max and sum, merged at the end (see row_split).
template <int D, int KS, bool VEC>
__global__ __launch_bounds__(NT, 2) void attn_fwd_f32_kernel(AttnArgs a, int n_tiles, int n_cu) {
  using C = Cfg<D>;
  constexpr int BQ = TR / KS;  // queries per workgroup
  constexpr int NB = 4 / KS;   // 16-key blocks of a tile per wave
  __shared__ __attribute__((aligned(16))) float Kt[TR * D];
  __shared__ __attribute__((aligned(16))) float Vt[TR * D];
  __shared__ float red[2][TR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int slice = wave % KS, grp = wave / KS;
  const int nbh = a.B * a.H;
  const int item = snake(blockIdx.x, gridDim.x, n_cu);
  const int bh = item % nbh;
  const int q0 = (n_tiles - 1 - item / nbh) * BQ;  // longest rows first
  const int b = bh / a.H, h = bh % a.H, S = a.S;
  const int qw = q0 + 16 * grp, qi = qw + i;
  const float* qp = (const float*)a.q.ptr + b * a.q.sb + h * a.q.sh;
  const float* kp = (const float*)a.k.ptr + b * a.k.sb + h * a.k.sh;
  const float* vp = (const float*)a.v.ptr + b * a.v.sb + h * a.v.sh;
  const bool causal = a.causal;
  const float c = a.scale_log2;
  const int kv_end = causal ? min(q0 + BQ, S) : S;

  f32x4 tk[C::NCH], tv[C::NCH], qf[C::KB], acc[C::KB];
  fetch_tile<D, VEC>(kp, a.k.ss, 0, S, tk);
  fetch_tile<D, VEC>(vp, a.v.ss, 0, S, tv);
  load_resident<D, VEC>(qp, a.q.ss, min(qi, S - 1), g, qf);
#pragma unroll
  for (int s = 0; s < C::KB; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  // One tile.  Masked tiles (the diagonal and the tail) skip the blocks past
  // `last` and test every pair; the others have no branch at all.
  auto step = [&](int kv0, int last, auto masked) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked)::value;
    f32x4 st[NB];
    float mx = -INFINITY;
    // the swizzled LDS offsets are formed per tile: kept across tiles they
    // cost D = 128 its last registers
    int io = i, go = g;
    opaque(io);
    opaque(go);
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const int blk = slice + KS * n, kb = kv0 + 16 * blk;
      if (MASKED && kb > last) continue;
      st[n] = row_product<D, C::NPS>(Kt, blk, io, go, qf);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = kb + 4 * g + r;
        st[n][r] *= c;
        if (MASKED && (key >= S) | (causal & (key > qi))) st[n][r] = -INFINITY;
        mx = fmaxf(mx, st[n][r]);
      }
    }
    const float m_new = fmaxf(m, max_groups(mx));
    const float ref = m_new == -INFINITY ? 0.f : m_new;  // no finite score yet: P = 0
    const float alpha = fast_exp2(m - ref);
    m = m_new;
    l *= alpha;
#pragma unroll
    for (int s = 0; s < C::KB; ++s) acc[s] *= alpha;
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      const int blk = slice + KS * n;
      if (MASKED && kv0 + 16 * blk > last) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        st[n][r] = fast_exp2(st[n][r] - ref);
        l += st[n][r];
      }
      col_product<D>(Vt, blk, io, go, st[n], acc);
    }
  };

  for (int kv0 = 0; kv0 < kv_end; kv0 += TR) {
    if (kv0) __syncthreads();
    put_tile<D>(Kt, tk);
    put_tile<D>(Vt, tv);
    __syncthreads();
    if (kv0 + TR < kv_end) {
      fetch_tile<D, VEC>(kp, a.k.ss, kv0 + TR, S, tk);
      fetch_tile<D, VEC>(vp, a.v.ss, kv0 + TR, S, tv);
    }
    // this wave's blocks that hold a visible key (they come first)
    const int last = min(causal ? qw + 15 : S - 1, S - 1);
    if (qw >= S || kv0 + 16 * slice > last) continue;
    if (kv0 + TR <= S && (!causal || kv0 + TR - 1 <= qw))
      step(kv0, last, std::false_type{});
    else
      step(kv0, last, std::true_type{});
  }

  l = sum_groups(l);
  float* op = (float*)a.o.ptr + b * a.o.sb + h * a.o.sh;
  float* lse = a.lse + (int64_t)bh * S;
  if constexpr (KS == 1) {
    if (qi >= S) return;
    put_rows<D, VEC>(op + qi * a.o.ss, g, acc, 1.f / l);
    if (g == 0) lse[qi] = (m + log2f(l)) * kLn2;
  } else {
    // merge of the KS partial results of each row, in a fixed order
    __syncthreads();
    const int row = 16 * grp + i;
    if (g == 0) {
      red[0][slice * BQ + row] = m;
      red[1][slice * BQ + row] = l;
    }
    __syncthreads();
    float ms = -INFINITY;
#pragma unroll
    for (int s = 0; s < KS; ++s) ms = fmaxf(ms, red[0][s * BQ + row]);
    const float ref = ms == -INFINITY ? 0.f : ms;
    float lt = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) lt += red[1][s * BQ + row] * fast_exp2(red[0][s * BQ + row] - ref);
    put_rows<D, true>(Kt + (slice * BQ + row) * D, g, acc, fast_exp2(m - ref));
    if (slice == 0 && g == 0 && qi < S) lse[qi] = (ms + log2f(lt)) * kLn2;
    __syncthreads();
    if (slice == 0 && g == 0) red[0][row] = 1.f / lt;
    __syncthreads();
    for (int idx = threadIdx.x; idx < BQ * C::CPR; idx += NT) {
      const int r = idx / C::CPR, d = 4 * (idx % C::CPR);
      if (q0 + r >= S) continue;
      f32x4 v = *(const f32x4*)(Kt + r * D + d);
#pragma unroll
      for (int s = 1; s < KS; ++s) v += *(const f32x4*)(Kt + (s * BQ + r) * D + d);
      store4<VEC>(op + (q0 + r) * a.o.ss + d, v * red[0][r]);
    }
  }
}

// Sum of the KS partial results of each row (in a fixed order) times `sc`.
template <int D, int KS, bool VEC>
__device__ __forceinline__ void merge_rows(float* part, const f32x4 (&acc)[Cfg<D>::KB], int slice,
                                           int row, int g, float* out, int64_t ss, int r0, int S,
                                           float sc) {
  constexpr int BR = TR / KS;
  put_rows<D, true>(part + (slice * BR + row) * D, g, acc, 1.f);
  __syncthreads();
  for (int idx = threadIdx.x; idx < BR * Cfg<D>::CPR; idx += NT) {
    const int r = idx / Cfg<D>::CPR, d = 4 * (idx % Cfg<D>::CPR);
    if (r0 + r >= S) continue;
    f32x4 v = *(const f32x4*)(part + r * D + d);
#pragma unroll
    for (int s = 1; s < KS; ++s) v += *(const f32x4*)(part + (s * BR + r) * D + d);
    store4<VEC>(out + (r0 + r) * ss + d, v * sc);
  }
}

// Backward item: 64 / KS resident rows against the streamed tiles.  DKDV:
// resident keys, streamed queries (T0 = Q, T1 = dO), accumulators dV and dK;
// otherwise resident queries, streamed keys (T0 = K, T1 = V), accumulator dQ.
// Either way S = T0 R0^T, dP = T1 R1^T, P = exp2(S c - lse2), dS = P (dP - delta).
template <int D, int KS, bool VEC, bool DKDV>
__device__ __forceinline__ void bwd_item(const AttnArgs& a, int bh, int r0, float* T0, float* T1,
                                         float (&stat)[2][TR]) {
  using C = Cfg<D>;
  constexpr int BR = TR / KS;
  constexpr int NB = 4 / KS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = lane & 15, g = lane >> 4;
  const int slice = wave % KS, grp = wave / KS;
  const int b = bh / a.H, h = bh % a.H, S = a.S;
  const int rw = r0 + 16 * grp, ri = rw + i;
  const float* qp = (const float*)a.q.ptr + b * a.q.sb + h * a.q.sh;
  const float* kp = (const float*)a.k.ptr + b * a.k.sb + h * a.k.sh;
  const float* vp = (const float*)a.v.ptr + b * a.v.sb + h * a.v.sh;
  const float* dp = (const float*)a.dout.ptr + b * a.dout.sb + h * a.dout.sh;
  const float* lsep = a.lse + (int64_t)bh * S;
  const float* delp = a.delta + (int64_t)bh * S;
  const float* t0p = DKDV ? qp : kp;
  const float* t1p = DKDV ? dp : vp;
  const int64_t t0s = DKDV ? a.q.ss : a.k.ss, t1s = DKDV ? a.dout.ss : a.v.ss;
  const bool causal = a.causal;
  const float c = a.scale_log2;
  const int begin = DKDV && causal ? r0 / TR * TR : 0;
  const int end = !DKDV && causal ? min(r0 + BR, S) : S;

  f32x4 t0[C::NCH], t1[C::NCH], f0[C::KB], f1[C::KB], acc0[C::KB], acc1[DKDV ? C::KB : 1];
  float sl = 0.f, sd = 0.f;  // a thread's streamed lse2 / delta (DKDV)
  // D = 128 has no registers for tiles in flight beside the resident rows and
  // the accumulators (100 bytes of scratch): they are fetched when their turn
  // comes, behind the products of the CU's other workgroup.
  constexpr bool AHEAD = D < 128;
  auto fetch = [&](int row0) __attribute__((always_inline)) {
    fetch_tile<D, VEC>(t0p, t0s, row0, S, t0);
    fetch_tile<D, VEC>(t1p, t1s, row0, S, t1);
    if (DKDV && threadIdx.x < TR) {
      const int r = row0 + threadIdx.x;
      sl = r < S ? lsep[r] * kLog2e : 0.f;
      sd = r < S ? delp[r] : 0.f;
    }
  };
  if constexpr (AHEAD) fetch(begin);
  const int rc = min(ri, S - 1);
  load_resident<D, VEC>(DKDV ? kp : qp, DKDV ? a.k.ss : a.q.ss, rc, g, f0);
  load_resident<D, VEC>(DKDV ? vp : dp, DKDV ? a.v.ss : a.dout.ss, rc, g, f1);
  const float lse2 = DKDV ? 0.f : lsep[rc] * kLog2e;
  const float dl = DKDV ? 0.f : delp[rc];
#pragma unroll
  for (int s = 0; s < C::KB; ++s) {
    acc0[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (DKDV) acc1[s] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // One tile; only masked tiles (the diagonal and the tails) have branches.
  auto step = [&](int row0, auto masked) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked)::value;
#pragma unroll 2
    for (int n = 0; n < NB; ++n) {
      const int blk = slice + KS * n, s0 = row0 + 16 * blk;
      if (MASKED && (s0 >= S || (causal && (DKDV ? s0 + 15 < rw : s0 > rw + 15)))) continue;
      // the swizzled LDS offsets are formed per block: kept across blocks they
      // cost D = 128 its last registers (16 bytes of scratch)
      int io = i, go = g;
      opaque(io);
      opaque(go);
      f32x4 p = row_product<D, C::NPS>(T0, blk, io, go, f0);
      f32x4 ds = row_product<D, C::NPD>(T1, blk, io, go, f1);
      f32x4 el = {lse2, lse2, lse2, lse2}, ed = {dl, dl, dl, dl};
      if constexpr (DKDV) {
        el = *(const f32x4*)&stat[0][16 * blk + 4 * g];
        ed = *(const f32x4*)&stat[1][16 * blk + 4 * g];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int x = s0 + 4 * g + r;  // streamed row
        p[r] = fast_exp2(__builtin_fmaf(p[r], c, -el[r]));
        if (MASKED && ((x >= S) | (ri >= S) | (causal & (DKDV ? ri > x : x > ri)))) p[r] = 0.f;
        ds[r] = p[r] * (ds[r] - ed[r]);
      }
      if constexpr (DKDV) col_product<D>(T1, blk, io, go, p, acc1);
      col_product<D>(T0, blk, io, go, ds, acc0);
    }
  };

  for (int row0 = begin; row0 < end; row0 += TR) {
    if (row0 > begin) __syncthreads();
    if constexpr (!AHEAD) fetch(row0);
    put_tile<D>(T0, t0);
    put_tile<D>(T1, t1);
    if (DKDV && threadIdx.x < TR) {
      stat[0][threadIdx.x] = sl;
      stat[1][threadIdx.x] = sd;
    }
    __syncthreads();
    if (AHEAD && row0 + TR < end) fetch(row0 + TR);
    if (rw >= S) continue;
    if (row0 + TR <= S && rw + 16 <= S &&
        (!causal || (DKDV ? row0 >= rw + 15 : row0 + TR - 1 <= rw)))
      step(row0, std::false_type{});
    else
      step(row0, std::true_type{});
  }

  float* o0 = DKDV ? (float*)a.dk.ptr + b * a.dk.sb + h * a.dk.sh
                   : (float*)a.dq.ptr + b * a.dq.sb + h * a.dq.sh;
  const int64_t o0s = DKDV ? a.dk.ss : a.dq.ss;
  float* o1 = DKDV ? (float*)a.dv.ptr + b * a.dv.sb + h * a.dv.sh : nullptr;
  if constexpr (KS == 1) {
    if (ri >= S) return;
    put_rows<D, VEC>(o0 + ri * o0s, g, acc0, a.scale);
    if constexpr (DKDV) put_rows<D, VEC>(o1 + ri * a.dv.ss, g, acc1, 1.f);
  } else {
    __syncthreads();
    merge_rows<D, KS, VEC>(T0, acc0, slice, 16 * grp + i, g, o0, o0s, r0, S, a.scale);
    if constexpr (DKDV)
      merge_rows<D, KS, VEC>(T1, acc1, slice, 16 * grp + i, g, o1, a.dv.ss, r0, S, 1.f);
  }
}

// dK/dV and dQ items in one launch, each kind's longest first and the longer
// kind (four products against three) before the other; `kinds` = 1 runs the
// dK/dV items alone, 2 the dQ items alone.
// D = 64 asks for three waves per SIMD: left to itself, the compiler takes more
// registers than those leave at KS = 2 (B1 H12 S1000, not causal: 150 us, not 120).
template <int D, int KS, bool VEC>
__global__ __launch_bounds__(NT, D == 64 ? 3 : 2) void attn_bwd_f32_kernel(AttnArgs a, int n_tiles,
                                                                           int kinds, int n_cu) {
  __shared__ __attribute__((aligned(16))) float T0[TR * D];
  __shared__ __attribute__((aligned(16))) float T1[TR * D];
  __shared__ __attribute__((aligned(16))) float stat[2][TR];
  const int nbh = a.B * a.H;
  const int item = snake(blockIdx.x, gridDim.x, n_cu);
  int rank = item / nbh;
  const int bh = item % nbh;
  bool dkdv = kinds == 1;
  if (kinds == 3) {
    dkdv = !(rank & 1);
    rank >>= 1;
  }
  if (dkdv)
    bwd_item<D, KS, VEC, true>(a, bh, rank * (TR / KS), T0, T1, stat);
  else
    bwd_item<D, KS, VEC, false>(a, bh, (n_tiles - 1 - rank) * (TR / KS), T0, T1, stat);
}

template <int D, int KS, bool VEC>
hipError_t launch_fwd(const AttnArgs& a, hipStream_t st) {
  const int n = (a.S + TR / KS - 1) / (TR / KS);
  hipLaunchKernelGGL((attn_fwd_f32_kernel<D, KS, VEC>), dim3(n * a.B * a.H), dim3(NT), 0, st, a, n,
                     a.causal ? cu_count(st) : 0);
  return hipGetLastError();
}

template <int D, int KS, bool VEC>
hipError_t launch_bwd(const AttnArgs& a, int kinds, hipStream_t st) {
  const int n = (a.S + TR / KS - 1) / (TR / KS);
  hipLaunchKernelGGL((attn_bwd_f32_kernel<D, KS, VEC>),
                     dim3(n * a.B * a.H * (kinds == 3 ? 2 : 1)), dim3(NT), 0, st, a, n, kinds,
                     a.causal ? cu_count(st) : 0);
  return hipGetLastError();
}

// Waves that share 16 rows and split the streamed side: fewer, longer
// workgroups amortise each staged tile over more rows, more and shorter ones
// fill the chip and shorten the longest chain.  By the number of 64-row
// workgroups (the backward has two kinds of them in one launch, so its lines
// lie at half the count), causal, KS = 4 / 2 / 1 in us:
//   48 (B1 H12 S256 D64):    forward 8.5 / 11.1 / 15.1, backward 17.4 / 20.4 / 30.0
//   192 (B1 H12 S1000 D64):  forward 28.5 / 36.3 / 50.7, backward 79 / 75 / 111
//   384 (B2 H12 S1000 D64):  forward 43.7 / 40.7 / 57.5, backward 128 / 127 / 129
//   768 (B4 H12 S1000 D64):  forward 79 / 76 / 67, backward 247 / 222 / 221
//   2048 (B4 H16 S2048 D64): forward 384 / 336 / 300, backward 1215 / 1071 / 1016
// The gradient stages run alone (`kinds` 1 or 2) split as they do together,
// so that their sums have the same order.
int row_split(const AttnArgs& a, int line) {
  const int64_t wgs = (int64_t)((a.S + TR - 1) / TR) * a.B * a.H;
  return wgs < line ? 4 : wgs < 2 * line ? 2 : 1;
}

template <int D>
hipError_t fwd_d(const AttnArgs& a, bool vec, hipStream_t st) {
  if (!vec) return launch_fwd<D, 1, false>(a, st);
  switch (row_split(a, 256)) {
    case 4: return launch_fwd<D, 4, true>(a, st);
    case 2: return launch_fwd<D, 2, true>(a, st);
    default: return launch_fwd<D, 1, true>(a, st);
  }
}
template <int D>
hipError_t bwd_d(const AttnArgs& a, int kinds, bool vec, hipStream_t st) {
  if (!vec) return launch_bwd<D, 1, false>(a, kinds, st);
  switch (row_split(a, 128)) {
    case 4: return launch_bwd<D, 4, true>(a, kinds, st);
    case 2: return launch_bwd<D, 2, true>(a, kinds, st);
    default: return launch_bwd<D, 1, true>(a, kinds, st);
  }
}

}  // namespace

hipError_t launch_attn_fwd_f32(const AttnArgs& a, bool vec, hipStream_t st) {
  switch (a.D) {
    case 16: return fwd_d<16>(a, vec, st);
    case 32: return fwd_d<32>(a, vec, st);
    case 64: return fwd_d<64>(a, vec, st);
    default: return fwd_d<128>(a, vec, st);
  }
}

hipError_t launch_attn_bwd_f32(const AttnArgs& a, int kinds, bool vec, hipStream_t st) {
  switch (a.D) {
    case 16: return bwd_d<16>(a, kinds, vec, st);
    case 32: return bwd_d<32>(a, kinds, vec, st);
    case 64: return bwd_d<64>(a, kinds, vec, st);
    default: return bwd_d<128>(a, kinds, vec, st);
  }
}

}  // namespace mi
