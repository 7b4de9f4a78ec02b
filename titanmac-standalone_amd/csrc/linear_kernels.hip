// Dense projections (nn.Linear without bias) on MFMA for gfx950: the qkv and output
// projections around the attention kernels (attn/windowed_attention.py:295-299, :331,
// attn/block_sparse_attention.py:222-223, :340), forward and both gradients, 16-bit inputs with
// fp32 accumulation.
//
//   forward  Y[M, N]  = X[M, K] · W[N, K]ᵀ     (tmac_linear_fwd)
//   input    dX[M, K] = dY[M, N] · W[N, K]     (tmac_linear_dx)
//   weight   dW[N, K] = dY[M, N]ᵀ · X[M, K]    (tmac_linear_wgrad)
//
// Features are multiples of 64, rows any number.
//
// What bounds them, and why these tiles (MI355X, bf16, rows 17920 = 32 sequences of 560):
// the copies HBM/L2 -> LDS run at about 54 bytes per clock and CU, so a tile has to give enough MFMA
// work per byte it copies. A 192 x 128 tile needs 53 bytes per clock at the full MFMA rate and leaves
// room for two independent workgroups per CU, whose barriers, copies and epilogues cover each
// other. 640 -> 1920 forward 54 us (0.81 PFLOP/s, was 80 in the library), dX 43 us (61); 640 -> 640
// forward 19 us (36), dX 18 us (37). The weight gradients have few output tiles (75 of 128 x 128) and a
// long reduction, so the rows are split over the chip: 59 us (141) and 28 us (102). Issuing a step's
// copies between its k-steps instead of ahead of them measured 0-6 % slower; a ring of six smaller
// (64 x 128) stages 2.2x slower.

#include "tmac_device.h"

using namespace tmac;

namespace {

// 128-byte LDS rows (64 16-bit values), 16-byte chunk c of row r at c ^ ((r >> 1) & 7): the
// 16-byte operand reads of 16 consecutive rows cover the 64 banks once.
__device__ __forceinline__ int xswz(int row, int chunk) {
  return row * 64 + ((chunk ^ ((row >> 1) & 7)) << 3);
}
// the global chunk that swz64 (tmac_device.h) stores at chunk position pos of row `row`
__device__ __forceinline__ int swz64_chunk(int row, int pos) {
  const int a = (row >> 1) & 7;
  return pos ^ (((a & 1) << 2) | (a >> 1));
}

// Forward and dX: a workgroup of four waves owns a 192 x 128 output tile, wave (wm, wn) its 96 rows x
// 64 columns (3 x 2 MFMA tiles). Per 64-wide step of the reduction the 192 x 64 activation tile and
// the 128 x 64 (forward) or 64 x 128 (dX) weight tile, 40 KB in all, are copied HBM/L2 -> LDS with
// global_load_lds into one of two stages, a step ahead of the math.
constexpr int kMI = 3;
constexpr int kLM = 64 * kMI, kLN = 128;
constexpr int kLX = kLM * 64, kLW = kLN * 64;  // tiles of a stage, elements
constexpr int kLStage = kLX + kLW;
constexpr int kXI = 2 * kMI;  // 8-row activation copies per wave and step (and four of the weight)

template <int DT, bool WT>
__global__ __launch_bounds__(256, 2) void linear_gemm_kernel(
    const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ W, int64_t ldw,
    uint16_t* __restrict__ Y, int64_t ldy, int M, int N, int n_steps, int n_mt, int n_nt, int per_xcd) {
  __shared__ __attribute__((aligned(16))) uint16_t smem[2 * kLStage];

  const int logical = xcd_logical_id(per_xcd);
  if (logical >= n_mt * n_nt) return;
  const int mt = logical / n_nt;
  const int m0 = mt * kLM, n0 = (logical - mt * n_nt) * kLN;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, h = lane >> 5, grp = (lane >> 4) & 1;
  const int wm = wave & 1, wn = wave >> 1;
  const int drow = lane >> 3, dpos = lane & 7;

  // Lane L of a copy covering rows R..R+7 fills chunk position L & 7 of row R + L / 8 and fetches
  // the chunk the swizzle stores there. Rows past M (columns past N) read the last valid one
  // (the first half); their results are not stored.
  uint32_t xoff[kXI], woff[4];
#pragma unroll
  for (int j = 0; j < kXI; ++j) {
    const int row = 8 * kXI * wave + 8 * j + drow;
    xoff[j] = static_cast<uint32_t>(min(row, M - 1 - m0)) * static_cast<uint32_t>(2 * lda) +
              16u * static_cast<uint32_t>(dpos ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (WT) {
      const int row = 32 * wave + 8 * j + drow;
      woff[j] = static_cast<uint32_t>(min(row, N - 1 - n0)) * static_cast<uint32_t>(2 * ldw) +
                16u * static_cast<uint32_t>(dpos ^ ((row >> 1) & 7));
    } else {
      const int row = 32 * (wave & 1) + 8 * j + drow;
      const int sub = n0 + 64 * wn < N ? wn : 0;
      woff[j] = static_cast<uint32_t>(row) * static_cast<uint32_t>(2 * ldw) +
                static_cast<uint32_t>(128 * sub + 16 * swz64_chunk(row, dpos));
    }
  }
  const uint32_t lds0 = lds_offset(smem);
  const uint16_t* xb = A + static_cast<int64_t>(m0) * lda;
  const uint16_t* wb = WT ? W + static_cast<int64_t>(n0) * ldw : W + n0;
  const int64_t wstep = WT ? 64 : 64 * ldw;
  auto issue = [&](int i) {
    const uint32_t st = lds0 + static_cast<uint32_t>((i & 1) * kLStage * 2);
    const uint16_t* xs = xb + 64 * i;
    const uint16_t* ws = wb + wstep * i;
#pragma unroll
    for (int j = 0; j < kXI; ++j) dma_lds16(xs, xoff[j], st + (8 * kXI * wave + 8 * j) * 128);
#pragma unroll
    for (int j = 0; j < 4; ++j) dma_lds16(ws, woff[j], st + kLX * 2 + (32 * wave + 8 * j) * 128);
  };

  f32x16 acc[kMI][2];
#pragma unroll
  for (int mi = 0; mi < kMI; ++mi)
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) acc[mi][ni] = f32x16{};
  // operands of k-step kk: activation rows as B, the weight as A (plain reads where the reduction
  // is contiguous, transpose reads for dX, whose reduction runs over W's rows)
  auto read_ops = [&](u32x4(&xa)[kMI], u32x4(&wf)[2], const uint16_t* st, int kk) {
#pragma unroll
    for (int mi = 0; mi < kMI; ++mi)
      xa[mi] = lds16(st + xswz(32 * kMI * wm + 32 * mi + l32, 2 * kk + h));
#pragma unroll
    for (int ni = 0; ni < 2; ++ni) {
      if constexpr (WT)
        wf[ni] = lds16(st + kLX + xswz(64 * wn + 32 * ni + l32, 2 * kk + h));
      else
        wf[ni] = lds_read_tr4x2_swz64(st + kLX + 4096 * wn, 16 * kk + 8 * h, 16 * kk + 8 * h + 4,
                                      32 * ni + 16 * grp, lane);
    }
  };
  // reads of k-step kk + 1 go out before the MFMAs of k-step kk
  auto compute = [&](const uint16_t* st) {
    u32x4 xa[2][kMI], wf[2][2];
    read_ops(xa[0], wf[0], st, 0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (kk + 1 < 4) read_ops(xa[(kk + 1) & 1], wf[(kk + 1) & 1], st, kk + 1);
#pragma unroll
      for (int mi = 0; mi < kMI; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
          acc[mi][ni] = Mfma<DT>::run(wf[kk & 1][ni], xa[kk & 1][mi], acc[mi][ni]);
    }
    constexpr int kDs = kMI + (WT ? 2 : 4);  // LDS read instructions per k-step
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kDs, 0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      __builtin_amdgcn_sched_group_barrier(0x008, 2 * kMI, 0);
      if (kk + 2 < 4) __builtin_amdgcn_sched_group_barrier(0x100, kDs, 0);
    }
  };

  const int col0 = n0 + 64 * wn;
  const bool active = col0 < N;
  issue(0);
  for (int i = 0; i < n_steps; ++i) {
    // every wave's copies of step i are in LDS, and every wave is done with step i - 1 (its reads have
    // returned), whose stage the next copies overwrite
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    ring_barrier();
    if (i + 1 < n_steps) issue(i + 1);
    if (active) compute(smem + (i & 1) * kLStage);
  }
  if (!active) return;

  // Epilogue, 32 rows at a time through 4 KB of the stage the last step did not use: packed in the
  // accumulator's layout (four consecutive columns of one row per lane), stored as 128-byte row
  // segments. No copy is in flight and every wave is past that stage's last reads.
  uint16_t* stage = smem + (n_steps & 1) * kLStage + wave * 2048;
#pragma unroll
  for (int mi = 0; mi < kMI; ++mi) {
#pragma unroll
    for (int ni = 0; ni < 2; ++ni)
#pragma unroll
      for (int jg = 0; jg < 4; ++jg) {
        u32x2 p;
        p.x = Mfma<DT>::pack2(acc[mi][ni][4 * jg], acc[mi][ni][4 * jg + 1]);
        p.y = Mfma<DT>::pack2(acc[mi][ni][4 * jg + 2], acc[mi][ni][4 * jg + 3]);
        *reinterpret_cast<u32x2*>(stage + l32 * 64 + (((4 * ni + jg) ^ (l32 & 7)) << 3) + 4 * h) = p;
      }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int row = 8 * it + drow;
      const u32x4 v = lds16(stage + row * 64 + ((dpos ^ (row & 7)) << 3));
      const int grow = m0 + 32 * kMI * wm + 32 * mi + row;
      if (grow < M) stg16(Y + static_cast<int64_t>(grow) * ldy + col0 + 8 * dpos, v);
    }
  }
}

// Weight gradient: a workgroup of two groups of four waves owns a (64 RN) x 128 tile of dW and a range
// of the M rows. Per 64-row step group g takes rows 32g..32g+31: their dY pieces (RN of 32 x 64) and X
// pieces (two) are copied into an LDS ring, and both operands are read transposed (the reduction runs
// over the rows); wave (wr, wc) of a group sums its 32 RN x 64 part. At the end the groups' sums are
// added through LDS, each group finishing one half of the tile, so that a CU writes one partial tile
// and not two. The ranges' fp32 partial tiles go to a workspace that linear_reduce_kernel adds in
// ascending order (deterministic); a single range is rounded and stored here.
template <int RN>
struct WGrad {
  static constexpr int kTiles = RN + 2;            // 32 x 64 pieces of a group's step
  static constexpr int kHalf = kTiles * 2048;      // a group's part of a stage, elements
  static constexpr int kStage = 2 * kHalf;
  static constexpr int kStages = RN == 2 ? 4 : 3;  // 128 or 144 KB of LDS: one workgroup per CU
  // the exchange: 8 waves x (RN / 2 x 2) MFMA tiles of 16 floats per lane
  static_assert(8 * (RN / 2) * 2 * 16 * 64 * 4 <= kStages * kStage * 2, "exchange fits the ring");
};

template <int DT, int RN>
__global__ __launch_bounds__(512, 1) void linear_wgrad_kernel(
    const uint16_t* __restrict__ dY, int64_t lddy, const uint16_t* __restrict__ X, int64_t ldx,
    float* __restrict__ part, uint16_t* __restrict__ out, int M, int N, int K, int n_nt, int n_kt,
    int rows_per_split, int n_splits, int per_xcd) {
  using G = WGrad<RN>;
  __shared__ __attribute__((aligned(16))) uint16_t ring[G::kStages * G::kStage];

  const int per_split = n_nt * n_kt;
  const int logical = xcd_logical_id(per_xcd);
  if (logical >= n_splits * per_split) return;
  const int split = logical / per_split;
  const int rem = logical - split * per_split;
  const int nt = rem / n_kt;
  const int n0 = nt * 64 * RN, k0 = (rem - nt * n_kt) * 128;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = wave >> 2, w4 = wave & 3;
  const int h = lane >> 5, grp = (lane >> 4) & 1, l32 = lane & 31;
  const int wr = w4 & 1, wc = w4 >> 1;
  const int drow = lane >> 3, dpos = lane & 7;

  const int m_begin = split * rows_per_split;
  const int m_end = min(M, m_begin + rows_per_split);
  const int n_steps = (m_end - m_begin + 63) / 64;

  // Each wave copies rows 8 w4..8 w4 + 7 of every piece of its group. Pieces past N or K read the
  // first one (copied, never stored); rows past M read row M - 1 and are zeroed in LDS once landed.
  const int crow = 8 * w4 + drow;
  uint32_t coff[G::kTiles];
#pragma unroll
  for (int t = 0; t < G::kTiles; ++t) {
    const int c0 = t < RN ? n0 + 64 * t : k0 + 64 * (t - RN);
    const bool in = t < RN ? c0 < N : c0 < K;
    coff[t] = 2u * static_cast<uint32_t>((in ? c0 : (t < RN ? n0 : k0)) + 8 * swz64_chunk(crow, dpos));
  }
  const uint32_t ring0 = lds_offset(ring);
  auto issue = [&](int i) {
    const int m0 = m_begin + 64 * i;  // < M
    const uint32_t st =
        ring0 + static_cast<uint32_t>(((i % G::kStages) * G::kStage + g * G::kHalf) * 2 + 8 * w4 * 128);
    const uint16_t* yb = dY + static_cast<int64_t>(m0) * lddy;
    const uint16_t* xb = X + static_cast<int64_t>(m0) * ldx;
    const uint32_t row = static_cast<uint32_t>(min(32 * g + crow, M - 1 - m0));
    const uint32_t yrow = row * static_cast<uint32_t>(2 * lddy), xrow = row * static_cast<uint32_t>(2 * ldx);
#pragma unroll
    for (int t = 0; t < G::kTiles; ++t)
      dma_lds16(t < RN ? yb : xb, (t < RN ? yrow : xrow) + coff[t], st + t * 4096);
  };

  f32x16 acc[RN][2];
#pragma unroll
  for (int ri = 0; ri < RN; ++ri)
#pragma unroll
    for (int ci = 0; ci < 2; ++ci) acc[ri][ci] = f32x16{};

#pragma unroll
  for (int i = 0; i < G::kStages - 1; ++i)
    if (i < n_steps) issue(i);
  for (int i = 0; i < n_steps; ++i) {
    // this wave's copies of step i have landed when only those of the later steps are outstanding
    const int later = min(G::kStages - 2, n_steps - 1 - i);
    if (later == 2)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * G::kTiles) : "memory");
    else if (later == 1)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(G::kTiles) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint16_t* st = ring + (i % G::kStages) * G::kStage + g * G::kHalf;
    const int valid = m_end - (m_begin + 64 * i) - 32 * g;
    if (valid < 32) {
      // rows past the range contribute zero: each wave clears the rows it copied
      if (crow >= valid) {
#pragma unroll
        for (int t = 0; t < G::kTiles; ++t) sts16(st + t * 2048 + crow * 64 + 8 * dpos, u32x4{0u, 0u, 0u, 0u});
      }
    }
    // every wave's copies of step i are in LDS, and every wave is done with step i - 1 (its reads have
    // returned), whose stage the next copies overwrite
    ring_barrier();
    if (i + G::kStages - 1 < n_steps) issue(i + G::kStages - 1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      u32x4 yf[RN], xf[2];
      const int r0 = 16 * ks + 8 * h;
#pragma unroll
      for (int ri = 0; ri < RN; ++ri) {
        const int c = 32 * RN * wr + 32 * ri;  // first of this operand's 32 dY columns in the tile
        yf[ri] = lds_read_tr4x2_swz64(st + (c >> 6) * 2048, r0, r0 + 4, (c & 63) + 16 * grp, lane);
      }
#pragma unroll
      for (int ci = 0; ci < 2; ++ci)
        xf[ci] = lds_read_tr4x2_swz64(st + (RN + wc) * 2048, r0, r0 + 4, 32 * ci + 16 * grp, lane);
#pragma unroll
      for (int ri = 0; ri < RN; ++ri)
#pragma unroll
        for (int ci = 0; ci < 2; ++ci) acc[ri][ci] = Mfma<DT>::run(yf[ri], xf[ci], acc[ri][ci]);
    }
  }

  // Exchange: each group hands the other its sums of the other's half (tile rows ri < RN / 2 are
  // finished by group 0, the rest by group 1) and adds what it receives, group 0's sum first.
  constexpr int HR = RN / 2;
  float* red = reinterpret_cast<float*>(ring);
  __syncthreads();  // every wave is done with the ring (no copy is in flight)
#pragma unroll
  for (int r = 0; r < HR; ++r)
#pragma unroll
    for (int ci = 0; ci < 2; ++ci)
#pragma unroll
      for (int j = 0; j < 16; ++j)
        red[((wave * HR + r) * 32 + ci * 16 + j) * 64 + lane] = g ? acc[r][ci][j] : acc[HR + r][ci][j];
  __syncthreads();
  const int kc = k0 + 64 * wc;
  if (kc >= K) return;
#pragma unroll
  for (int r = 0; r < HR; ++r) {
    const int nr = n0 + 32 * RN * wr + 32 * (g * HR + r);
    if (nr >= N) continue;
#pragma unroll
    for (int ci = 0; ci < 2; ++ci)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float o = red[(((wave ^ 4) * HR + r) * 32 + ci * 16 + j) * 64 + lane];
        const float v = (g ? acc[HR + r][ci][j] : acc[r][ci][j]) + o;
        const int64_t at = static_cast<int64_t>(nr + 8 * (j >> 2) + 4 * h + (j & 3)) * K + kc + 32 * ci + l32;
        if (n_splits == 1)
          out[at] = Mfma<DT>::from_f32(v);
        else
          part[static_cast<int64_t>(split) * N * K + at] = v;
      }
  }
}

// out[i] = the sum of part[split][i] over the splits, ascending, rounded to the 16-bit type.
template <int DT>
__global__ __launch_bounds__(256) void linear_reduce_kernel(const float* __restrict__ part,
                                                            uint16_t* __restrict__ out, int64_t n_elem,
                                                            int n_splits) {
  const int64_t i4 = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i4 >= n_elem) return;
  f32x4 s = *reinterpret_cast<const f32x4*>(part + i4);
  for (int k = 1; k < n_splits; ++k) s += *reinterpret_cast<const f32x4*>(part + k * n_elem + i4);
  u32x2 p;
  p.x = Mfma<DT>::pack2(s.x, s.y);
  p.y = Mfma<DT>::pack2(s.z, s.w);
  *reinterpret_cast<u32x2*>(out + i4) = p;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int launch_status() {
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? TMAC_OK : static_cast<int>(err);
}

// Common checks: a [rows, cols] operand with the given pitch.
int check_dense(const void* p, int64_t ld, int64_t cols) {
  if (!p) return TMAC_ERR_NULL;
  if (ld < cols) return TMAC_ERR_SHAPE;
  if (!aligned16(p) || (ld % 8)) return TMAC_ERR_ALIGN;
  // the copies address a tile's rows with 32-bit byte offsets
  if (ld > (1ll << 22)) return TMAC_ERR_SHAPE;
  return TMAC_OK;
}

int check_linear(int M, int N, int K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || (N % 64) || (K % 64)) return TMAC_ERR_SHAPE;
  if (static_cast<int64_t>(N) * K > (1ll << 30)) return TMAC_ERR_SHAPE;
  if (dtype != TMAC_BF16 && dtype != TMAC_F16) return TMAC_ERR_DTYPE;
  return TMAC_OK;
}

template <bool WT>
int launch_gemm(const void* A, int64_t lda, const void* W, int64_t ldw, void* Y, int64_t ldy, int M, int N,
                int R, int dtype, void* stream) {
  const int n_mt = (M + kLM - 1) / kLM, n_nt = (N + kLN - 1) / kLN;
  const int64_t total = static_cast<int64_t>(n_mt) * n_nt;
  if (total > (1ll << 30)) return TMAC_ERR_SHAPE;
  const int per_xcd = static_cast<int>((total + 7) / 8);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto* a = static_cast<const uint16_t*>(A);
  const auto* w = static_cast<const uint16_t*>(W);
  auto* y = static_cast<uint16_t*>(Y);
  if (dtype == TMAC_BF16)
    hipLaunchKernelGGL((linear_gemm_kernel<TMAC_BF16, WT>), dim3(8 * per_xcd), dim3(256), 0, s, a, lda, w,
                       ldw, y, ldy, M, N, R / 64, n_mt, n_nt, per_xcd);
  else
    hipLaunchKernelGGL((linear_gemm_kernel<TMAC_F16, WT>), dim3(8 * per_xcd), dim3(256), 0, s, a, lda, w,
                       ldw, y, ldy, M, N, R / 64, n_mt, n_nt, per_xcd);
  return launch_status();
}

// Tile height (in 64s) and split of the weight gradient: the cheapest of a model of its time in
// microseconds, rounds of one workgroup per CU, each its 64-row steps (0.85 us at 256 x 128, 0.55 at
// 128 x 128) and a fixed part, plus writing and reading the partial tiles and the second launch.
struct WGradPlan {
  int rn, n_nt, n_kt, n_splits, rows;
};
WGradPlan wgrad_plan(int M, int N, int K) {
  WGradPlan best{};
  float best_us = 0.f;
  const int m_steps = (M + 63) / 64;
  for (int rn = 2; rn <= 4; rn += 2) {
    const int n_nt = (N + 64 * rn - 1) / (64 * rn), n_kt = (K + 127) / 128;
    const int most = 256 / (n_nt * n_kt) > 64 ? 256 / (n_nt * n_kt) : 64;
    for (int want = 1; want <= most && want <= m_steps; ++want) {
      const int steps = (m_steps + want - 1) / want;
      const int n_splits = (m_steps + steps - 1) / steps;
      const int rounds = (n_nt * n_kt * n_splits + 255) / 256;
      float us = rounds * (steps * (rn == 4 ? 0.85f : 0.55f) + 3.f);
      if (n_splits > 1) us += 3.f + static_cast<float>(n_splits) * N * K * 8.f / 5e6f;
      if (best.rn == 0 || us < best_us) {
        best = WGradPlan{rn, n_nt, n_kt, n_splits, steps * 64};
        best_us = us;
      }
    }
  }
  return best;
}

// Partial tiles (none for a single range).
size_t wgrad_ws_bytes(const WGradPlan& p, int N, int K) {
  return p.n_splits > 1 ? static_cast<size_t>(p.n_splits) * N * K * sizeof(float) : 0;
}

}  // namespace

extern "C" int tmac_linear_fwd(const void* d_X, int64_t ldx, const void* d_W, int64_t ldw, void* d_Y,
                               int64_t ldy, int M, int N, int K, int dtype, void* stream) {
  int st = check_linear(M, N, K, dtype);
  if (st == TMAC_OK) st = check_dense(d_X, ldx, K);
  if (st == TMAC_OK) st = check_dense(d_W, ldw, K);
  if (st == TMAC_OK) st = check_dense(d_Y, ldy, N);
  if (st != TMAC_OK) return st;
  return launch_gemm<true>(d_X, ldx, d_W, ldw, d_Y, ldy, M, N, K, dtype, stream);
}

extern "C" int tmac_linear_dx(const void* d_dY, int64_t lddy, const void* d_W, int64_t ldw, void* d_dX,
                              int64_t lddx, int M, int N, int K, int dtype, void* stream) {
  int st = check_linear(M, N, K, dtype);
  if (st == TMAC_OK) st = check_dense(d_dY, lddy, N);
  if (st == TMAC_OK) st = check_dense(d_W, ldw, K);
  if (st == TMAC_OK) st = check_dense(d_dX, lddx, K);
  if (st != TMAC_OK) return st;
  return launch_gemm<false>(d_dY, lddy, d_W, ldw, d_dX, lddx, M, K, N, dtype, stream);
}

extern "C" int tmac_linear_wgrad_workspace(int M, int N, int K, size_t* ws_bytes) {
  if (!ws_bytes) return TMAC_ERR_NULL;
  const int st = check_linear(M, N, K, TMAC_BF16);
  if (st != TMAC_OK) return st;
  *ws_bytes = wgrad_ws_bytes(wgrad_plan(M, N, K), N, K);
  return TMAC_OK;
}

extern "C" int tmac_linear_wgrad(const void* d_dY, int64_t lddy, const void* d_X, int64_t ldx, void* d_dW,
                                 void* d_ws, size_t ws_bytes, int M, int N, int K, int dtype, void* stream) {
  int st = check_linear(M, N, K, dtype);
  if (st == TMAC_OK) st = check_dense(d_dY, lddy, N);
  if (st == TMAC_OK) st = check_dense(d_X, ldx, K);
  if (st == TMAC_OK) st = check_dense(d_dW, K, K);
  if (st != TMAC_OK) return st;
  const WGradPlan p = wgrad_plan(M, N, K);
  if (p.n_splits > 1) {
    if (!d_ws || ws_bytes < wgrad_ws_bytes(p, N, K)) return TMAC_ERR_WORKSPACE;
    if (!aligned16(d_ws)) return TMAC_ERR_ALIGN;
  }
  const int total = p.n_splits * p.n_nt * p.n_kt;
  const int per_xcd = (total + 7) / 8;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const auto* dY = static_cast<const uint16_t*>(d_dY);
  const auto* X = static_cast<const uint16_t*>(d_X);
  auto* part = static_cast<float*>(d_ws);
#define TMAC_WG_LAUNCH(DT, RN)                                                                          \
  hipLaunchKernelGGL((linear_wgrad_kernel<DT, RN>), dim3(8 * per_xcd), dim3(512), 0, s, dY, lddy, X, ldx, \
                     part, static_cast<uint16_t*>(d_dW), M, N, K, p.n_nt, p.n_kt, p.rows, p.n_splits, per_xcd)
  if (dtype == TMAC_BF16) {
    if (p.rn == 4)
      TMAC_WG_LAUNCH(TMAC_BF16, 4);
    else
      TMAC_WG_LAUNCH(TMAC_BF16, 2);
  } else {
    if (p.rn == 4)
      TMAC_WG_LAUNCH(TMAC_F16, 4);
    else
      TMAC_WG_LAUNCH(TMAC_F16, 2);
  }
#undef TMAC_WG_LAUNCH
  st = launch_status();
  if (st != TMAC_OK || p.n_splits == 1) return st;
  const int64_t n_elem = static_cast<int64_t>(N) * K;
  const int grid = static_cast<int>((n_elem / 4 + 255) / 256);
  if (dtype == TMAC_BF16)
    hipLaunchKernelGGL(linear_reduce_kernel<TMAC_BF16>, dim3(grid), dim3(256), 0, s, part,
                       static_cast<uint16_t*>(d_dW), n_elem, p.n_splits);
  else
    hipLaunchKernelGGL(linear_reduce_kernel<TMAC_F16>, dim3(grid), dim3(256), 0, s, part,
                       static_cast<uint16_t*>(d_dW), n_elem, p.n_splits);
  return launch_status();
}
