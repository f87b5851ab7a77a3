// bfloat16 matrix product for few rows (decoding and short prompt portions: 1..128 tokens), where the weights are read
// once from HBM and everything else is small:  C[M, N] (+)= X[M, K] . W[N, K]^T.
//
// The weights are the row operand of v_mfma_f32_16x16x32_bf16 and the activations the column
// operand, so a wave produces C^T for 32 weight rows (two row tiles) and up to 32 tokens (the
// second kernel below takes 33..128 tokens).
// A lane reads 32 contiguous bytes of a weight row per step; the four lane groups of a row
// cover 128 contiguous bytes.  No LDS on the way in: activations come from L2.
// A block is four waves on the same 32 rows, each on a quarter of the block's k-range; they
// add up through LDS.  The k-range may further be split over blocks (grid.y): each block
// then writes its partial tile to a workspace and the consumer of the product adds the
// partials in split order (deterministic).
//
// Epilogues as in the many-row kernel: store bf16, store f32, add into f32, SwiGLU (gate / up
// rows interleaved by 16, so the two row tiles of a wave are the gate and the up rows of the
// same 16 features; no k-split over blocks in that case).
#include <type_traits>

#include "addressing.h"
#include "mfma.h"

enum { EPI_BF16 = 0, EPI_F32 = 1, EPI_ACCUM = 2, EPI_SWIGLU = 3 };

#define ROWS_PER_BLOCK 32
#define RANGES_ROW_TILES 4      // row tiles per wave where the key ranges are merged on the way in (fewer blocks repeat the merge)
#define KSTEP addressing::KSTEP
#define SHARED_FROM_TOKENS 32   // more tokens than this: the kernel that shares an activation tile per block
#define SHARED_FROM_ELEMENTS 20000000L    // ... and more than 16 tokens on matrices of so many elements
#define RING_MAX_STRIDE (1L << 21)  // elements between rows, and of k, up to which that kernel's byte offsets fit 31 bits

template <int EPI>
__device__ inline void epilogue_store(void* Cv, long ldc, long m, long n, float v) {
  if (EPI == EPI_BF16) reinterpret_cast<bf16_t*>(Cv)[m * ldc + n] = from_float<bf16_t>(v);
  if (EPI == EPI_F32) reinterpret_cast<float*>(Cv)[m * ldc + n] = v;
  if (EPI == EPI_ACCUM) reinterpret_cast<float*>(Cv)[m * ldc + n] += v;
}

// LDS of a block: while the k loop runs, each wave stages its activations there (the loads from
// memory follow the rows, eight lanes on a row's 128 bytes, which the cache serves at twice the
// rate of the operand's own pattern of sixteen rows per quarter wave); afterwards the same bytes
// hold the waves' partial tiles for the sum.
// Activations that are still the key ranges of a decode step's attention (one token per
// request, request r at row r): float32 [token, head, range, head_dim + 4] holding each range's
// un-normalised output, then its maximum and its sum of weights.  The product kernel merges
// them on the way in, which saves the merging kernel between attention and the o projection.
struct RangeSource {
  const float* ranges;
  int heads, head_dim, count;
};

// Merges the key ranges of tokens first, first + stride, .. (TOK of them per round) for four features of one head, rounds
// them to bfloat16 and hands them to store(token, packed).  CNT > 0: up to CNT ranges, all loads of a round asked for before
// the first is used (one trip to memory); CNT == 0: any number, in two passes.  Ranges are added
// in range order with the shared arithmetic (range_weight / range_add / range_finish).
template <int CNT, int TOK, typename Store>
__device__ inline void merge_ranges_of_tokens(const float* __restrict__ head_base, long token_stride, int count, int rec, int hd,
                                              int f0, int first, int stride, int M, Store store) {
#pragma unroll 1
  for (int t0 = first; t0 < M; t0 += stride * TOK) {
    f32x4_t sum[TOK];
    float l_tot[TOK];
    if constexpr (CNT > 0) {
      float2 ml[TOK][CNT];
      f32x4_t o[TOK][CNT];
#pragma unroll
      for (int j = 0; j < TOK; ++j) {
        const float* base = head_base + (long)min(t0 + stride * j, M - 1) * token_stride;
#pragma unroll
        for (int u = 0; u < CNT; ++u) {
          const int r = min(u, count - 1);
          ml[j][u] = *reinterpret_cast<const float2*>(base + r * rec + hd);
          o[j][u] = *reinterpret_cast<const f32x4_t*>(base + r * rec + f0);
        }
      }
#pragma unroll
      for (int j = 0; j < TOK; ++j) {
        float m_tot = -INFINITY;
#pragma unroll
        for (int u = 0; u < CNT; ++u) m_tot = fmaxf(m_tot, ml[j][u].x);
        sum[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        l_tot[j] = 0.f;
#pragma unroll
        for (int u = 0; u < CNT; ++u) {
          const float wgt = u < count ? range_weight(ml[j][u].x, m_tot) : 0.f;
          l_tot[j] = range_add(wgt, ml[j][u].y, l_tot[j]);
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[j][e] = range_add(wgt, o[j][u][e], sum[j][e]);
        }
      }
    } else {
      static_assert(CNT > 0 || TOK == 1, "the two-pass merge takes one token per round");
      const float* base = head_base + (long)t0 * token_stride;
      float m_tot = -INFINITY;
#pragma unroll 8
      for (int r = 0; r < count; ++r) m_tot = fmaxf(m_tot, base[r * rec + hd]);
      sum[0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      l_tot[0] = 0.f;
#pragma unroll 8
      for (int r = 0; r < count; ++r) {
        const float2 ml = *reinterpret_cast<const float2*>(base + r * rec + hd);
        const f32x4_t o = *reinterpret_cast<const f32x4_t*>(base + r * rec + f0);
        const float wgt = range_weight(ml.x, m_tot);
        l_tot[0] = range_add(wgt, ml.y, l_tot[0]);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[0][e] = range_add(wgt, o[e], sum[0][e]);
      }
    }
#pragma unroll
    for (int j = 0; j < TOK; ++j) {
      const int token = t0 + stride * j;
      if (token >= M) break;
      uint2 packed;
      packed.x = pack_bf16x2(range_finish(sum[j][0], l_tot[j]), range_finish(sum[j][1], l_tot[j]));
      packed.y = pack_bf16x2(range_finish(sum[j][2], l_tot[j]), range_finish(sum[j][3], l_tot[j]));
      store(token, packed);
    }
  }
}

// tokens per round x ranges per token held in registers at once: about IN_FLIGHT either way
template <int IN_FLIGHT, typename Store>
__device__ inline void merge_ranges(const float* __restrict__ head_base, long token_stride, int count, int rec, int hd, int f0, int first,
                                    int stride, int M, Store store) {
  if (count <= 4) merge_ranges_of_tokens<4, IN_FLIGHT / 4>(head_base, token_stride, count, rec, hd, f0, first, stride, M, store);
  else if (count <= 8) merge_ranges_of_tokens<8, IN_FLIGHT / 8>(head_base, token_stride, count, rec, hd, f0, first, stride, M, store);
  else if (count <= 16) merge_ranges_of_tokens<16, IN_FLIGHT / 16>(head_base, token_stride, count, rec, hd, f0, first, stride, M, store);
  else merge_ranges_of_tokens<0, 1>(head_base, token_stride, count, rec, hd, f0, first, stride, M, store);
}

// Activations of a norm whose root was left to this reader (gemm_rows_kernel made them): row m holds x * w, and the
// product of the normalised row is the product of these times 1 / sqrt(mean of x^2 + eps), a factor per row that the
// epilogue applies in float32.  sums: float32 [M][count], a row's sum of x^2 in pieces.
struct LeftNorm {
  const float* sums;
  int count, width;
  float eps;
};

// The factors of rows wave * 4 .. + 3 of a block of four waves, sixteen lanes to a row.  load() asks for the pieces (up to 512
// a row) before the weights' loop, so that they travel beside it; finish() adds them, the same way in every block, and leaves
// the factors in LDS.
struct LeftNormRows {
  f32x4_t piece[8];
  __device__ inline void load(const LeftNorm& left, int wave, int lane, int M) {
    const int m = wave * 4 + lane / 16;
    const float* row = left.sums + (long)m * left.count;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int at = u * 64 + lane % 16 * 4;
      piece[u] = m < M && at < left.count ? *reinterpret_cast<const f32x4_t*>(row + at) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }
  __device__ inline void finish(const LeftNorm& left, int wave, int lane, float* factors) {
    const f32x4_t p = ((piece[0] + piece[1]) + (piece[2] + piece[3])) + ((piece[4] + piece[5]) + (piece[6] + piece[7]));
    float sum = (p[0] + p[1]) + (p[2] + p[3]);
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) sum += __shfl_xor(sum, off, PI_WAVE);
    if (lane % 16 == 0) factors[wave * 4 + lane / 16] = 1.0f / sqrtf(sum / (float)left.width + left.eps);
  }
};

template <int MB, int RT>
union SkinnyLds {
  float red[4][RT * 16][MB * 16 + 1];
  u32x4_t xs[4][MB * 8 * 16];          // per wave: [token tile][16-byte piece of the k step][token], tokens turned by the piece
};

template <int MB, int EPI, bool RANGES = false, int RT = 2>
__global__ __launch_bounds__(256) void gemm_skinny_kernel(void* __restrict__ Cv, long ldc, const bf16_t* __restrict__ X, long ldx,
                                                          const bf16_t* __restrict__ W, long ldw, int M, int N, int K,
                                                          int k_per_block, float* __restrict__ part, RangeSource rs, int tiled) {
  constexpr int ROWS = RT * 16;          // weight rows of a block: RT row tiles per wave
  static_assert(EPI != EPI_SWIGLU || RT == 2, "the SwiGLU epilogue pairs a wave's two row tiles");
  __shared__ SkinnyLds<MB, RT> lds;
  float (*red)[ROWS][MB * 16 + 1] = lds.red;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int lr = lane % 16, lg = lane / 16;
  const long n0 = (long)blockIdx.x * ROWS;
  const int splits = gridDim.y;

  // this wave's k-range: a quarter (rounded up to whole steps) of the block's range
  const addressing::WaveRange range = addressing::skinny_wave_range(K, k_per_block, blockIdx.y, wave);
  const int k0 = range.k0, k1 = range.k1;

  // rows beyond N read the last valid row; their results are never stored.  `tiled`: W is the
  // copy in the order this kernel reads (see pi_gemm_skinny): 16 rows x 64 k are 2 KB in a row,
  // one load instruction's 1 KB after the other, so a k step of 64 moves by 1,024 elements and
  // the step's second fragment lies 512 elements behind the first.
  const bf16_t* wrow[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) wrow[t] = W + addressing::skinny_w_base(tiled, n0, t, lr, lg, N, K, ldw);

  // Activations of a k step: load instruction i brings tokens 8i .. 8i+7, lane j the 16-byte
  // piece j % 8 of token 8i + j / 8.  Tokens beyond M are not loaded: what LDS holds for them
  // only reaches columns of the result that are never stored.
  const int x_loads = __builtin_amdgcn_readfirstlane((M + 7) / 8);
  const int xt = lane / 8, xp = lane % 8;
  const bf16_t* xsrc[MB * 2];
  int xdst[MB * 2];
#pragma unroll
  for (int i = 0; i < MB * 2; ++i) {
    const int token = i * 8 + xt;
    xsrc[i] = X + addressing::skinny_x_base(token, M, ldx, xp);
    xdst[i] = ((token / 16) * 8 + xp) * 16 + ((token + 2 * xp) & 15);
  }
  u32x4_t* xs = lds.xs[wave];
  int xfrag[MB][2];                     // where this lane's operand pieces lie: piece lg*2+h of token lr
#pragma unroll
  for (int c = 0; c < MB; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) xfrag[c][h] = (c * 8 + lg * 2 + h) * 16 + ((lr + 2 * (lg * 2 + h)) & 15);

  f32x4_t acc[RT][MB];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < MB; ++c) acc[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // one k step; in a last, partial one the 8-element pieces beyond k1 count as zero
  auto step = [&](const int kk, auto whole_step) {
    constexpr bool whole = decltype(whole_step)::value;
    Frag w[RT][2];
    u32x4_t xg[MB * 2];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // a piece beyond k1 is fetched from a stand-in address inside the row and counts as zero
        w[t][h] = load_frag(wrow[t] + addressing::skinny_w_step(tiled, whole, kk, h, lg, k0, k1));
        if (!addressing::skinny_w_used(whole, kk, h, lg, k1)) w[t][h] = zero_frag();
      }
    if constexpr (RANGES) {
      // The 64 features of this step belong to one head (head_dim is a multiple of 64).  Lane
      // group lg merges tokens lg, lg + 4, ..; a lane owns four features.  Every load is asked
      // for before the first is needed; the ranges are added in range order.
      static_assert(MB == 1, "merging on the way in serves up to 16 tokens");
      const int head = kk / rs.head_dim, f0 = kk - head * rs.head_dim + lr * 4;
      const int rec = rs.head_dim + 4;
      const float* head_base = rs.ranges + (long)head * rs.count * rec;
      const long token_stride = (long)rs.heads * rs.count * rec;
      uint2* xs2 = reinterpret_cast<uint2*>(xs);
      const int piece = lr / 2;                            // the 16-byte piece of the k step the lane's features lie in
      merge_ranges<16>(head_base, token_stride, rs.count, rec, rs.head_dim, f0, lg, 4, M, [&](const int token, const uint2 packed) {
        xs2[(piece * 16 + ((token + 2 * piece) & 15)) * 2 + (lr & 1)] = packed;
      });
    } else {
      const bool x_ok = whole || kk + xp * 8 < k1;
#pragma unroll
      for (int i = 0; i < MB * 2; ++i)
        if (i == 0 || i < x_loads) {
          xg[i] = *reinterpret_cast<const u32x4_t*>(xsrc[i] + addressing::skinny_x_step(whole, kk, xp, k0, k1));
          if (!x_ok) xg[i] = u32x4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
      for (int i = 0; i < MB * 2; ++i)
        if (i == 0 || i < x_loads) xs[xdst[i]] = xg[i];
    }
    // the wave reads what its own lanes wrote: LDS serves one wave's accesses in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    Frag x[MB][2];
#pragma unroll
    for (int c = 0; c < MB; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) x[c][h].n = xs[xfrag[c][h]];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int c = 0; c < MB; ++c) {
        acc[t][c] = mfma16(w[t][0], x[c][0], acc[t][c]);
        acc[t][c] = mfma16(w[t][1], x[c][1], acc[t][c]);
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  int kk = k0;
  for (; kk + KSTEP <= k1; kk += KSTEP) step(kk, std::true_type{});
  if (kk < k1) step(kk, std::false_type{});
  __syncthreads();                      // the partial tiles take the place of the staged activations

  // acc[t][c][r] is C^T[n0 + t*16 + lg*4 + r][c*16 + lr]; add the four waves through LDS
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < MB; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][t * 16 + lg * 4 + r][c * 16 + lr] = acc[t][c][r];
  __syncthreads();

  const int cols = MB * 16;
  if (splits == 1) {
    if (EPI == EPI_SWIGLU) {
      for (int idx = tid; idx < 16 * cols; idx += 256) {
        const int j = idx % 16, m = idx / 16;
        const long n = n0 + j;                     // gate row; up row is n + 16
        if (m >= M || n + 16 >= N) continue;
        const float g = red[0][j][m] + red[1][j][m] + red[2][j][m] + red[3][j][m];
        const float u = red[0][16 + j][m] + red[1][16 + j][m] + red[2][16 + j][m] + red[3][16 + j][m];
        reinterpret_cast<bf16_t*>(Cv)[(long)m * ldc + n0 / 2 + j] = from_float<bf16_t>(g / (1.0f + expf(-g)) * u);
      }
    } else {
      for (int idx = tid; idx < ROWS * cols; idx += 256) {
        const int nl = idx % ROWS, m = idx / ROWS;
        if (m >= M || n0 + nl >= N) continue;
        epilogue_store<EPI>(Cv, ldc, m, n0 + nl, red[0][nl][m] + red[1][nl][m] + red[2][nl][m] + red[3][nl][m]);
      }
    }
    return;
  }

  // k split over blocks: this block's partial tile goes to part[split][m][n]; whoever consumes
  // the product (the reduce kernel below, or a norm / rotation kernel that folds the sum into
  // its own read) adds the splits in split order.  No block waits for or signals another:
  // on a chip of several dies a device-wide fence costs more than a kernel boundary.
  float* mine = part + (long)blockIdx.y * M * N;
  for (int idx = tid; idx < ROWS * cols; idx += 256) {
    const int nl = idx % ROWS, m = idx / ROWS;
    if (m >= M || n0 + nl >= N) continue;
    mine[(long)m * N + n0 + nl] = red[0][nl][m] + red[1][nl][m] + red[2][nl][m] + red[3][nl][m];
  }
}

// The same product for 33..128 tokens (from 17 on for large matrices, pi_gemm_skinny_shares), where the activations are as many bytes as a block's weights.  A block is eight waves
// on 64 weight rows: wave w multiplies rows 32 (w / 4) .. + 31 with T tiles of 32 tokens (v_mfma_f32_32x32x16_bf16), and of
// every step of 64 k takes the 16 of its quarter w % 4; the quarters are summed through LDS at the end.  So a step's
// activations are read from LDS twice and not once per 16 rows, and the weights go into registers past LDS.  Activations go
// from memory straight into a ring of buffers; both are asked for four steps ahead (eight: 2,048 x 8,192, 64 tokens 13.5 us
// instead of 11.6).  The one barrier per step waits for
// the loads that the step needs, not for those behind them.  Steps beyond the block's k, tokens beyond M and rows beyond N
// take offsets outside the descriptors: zeros, and no bytes.
// Bound by the weights' way from memory and, towards 128 tokens, by the activations' from L2.  In place of four waves of 16
// rows each that staged the activations through registers, at 33 / 64 / 100 / 128 tokens, weights from memory in the copy's
// order: 16,384 x 2,048 16.2 / 18.6 / 23.6 / 23.7 us -> 15.5 / 16.9 / 19.1 / 21.3, 2,048 x 8,192 in eight pieces 10.7 / 12.2 /
// 16.0 / 16.6 -> 10.8 / 11.6 / 13.7 / 14.8, 6,144 x 4,096 17.1 / 19.9 / 26.4 / 28.3 in three pieces -> 15.0 / 15.7 / 18.7 / 20.1
// in two, 28,672 x 4,096 51 / 56 / 68 / 73 -> 49 / 53 / 62 / 66.
#define RING_ROWS 64
#define RING_BUFFERS 5

template <int T, int EPI>
__global__ __launch_bounds__(512, 4) void gemm_skinny_ring_kernel(void* __restrict__ Cv, long ldc, const bf16_t* __restrict__ X, long ldx,
                                                               const bf16_t* __restrict__ W, long ldw, int M, int N, int K,
                                                               int k_per_block, float* __restrict__ part, int tiled) {
  constexpr int XROWS = T == 2 ? 64 : 128, XI = XROWS / 64;        // rows of a buffer, load instructions of a wave per step
  constexpr int NB = RING_BUFFERS, AHEAD = NB - 1, TOKENS = T * 32, PITCH = TOKENS + 1;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];   // [NB][XROWS][64], 16-byte pieces of a row turned by (row / 2) % 8
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int rows32 = wave / 4, quarter = wave % 4;
  const long n0 = (long)blockIdx.x * RING_ROWS;
  const int splits = gridDim.y;
  const int k_lo = blockIdx.y * k_per_block, k_hi = min(K, k_lo + k_per_block), k_range = k_hi - k_lo;
  const int w_rows = (int)min((long)RING_ROWS, N - n0);
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t x_src = operand_descriptor(X, addressing::tile_descriptor(0, ldx, k_lo, k_hi, M));
  const __amdgpu_buffer_rsrc_t w_src = operand_descriptor(W, addressing::ring_w_descriptor(tiled, n0, k_lo, k_hi, w_rows, K, ldw));
#endif
  unsigned x_off[XI];
  int x_piece[XI];
#pragma unroll
  for (int p = 0; p < XI; ++p) {
    const int row = (p * 8 + wave) * 8 + lane / 8;
    x_piece[p] = addressing::tile_piece(lane, row);
    x_off[p] = addressing::tile_lane_offset(row, M, ldx, x_piece[p]);
  }
  const int frow = lane % 32, piece = quarter * 2 + lane / 32;     // a fragment: row (token) frow, the 8 k of the piece
  const unsigned w_off = addressing::ring_w_lane_offset(tiled, rows32 * 32 + frow, w_rows, K, ldw, piece);
  const int place = (piece ^ ((frow >> 1) & 7)) * 8;

  Frag wq[AHEAD];
  auto fetch_x = [&](const int s, const int buf) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int p = 0; p < XI; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_src, (lds_ptr_t)(lds + (buf * XROWS + (p * 8 + wave) * 8) * KSTEP), 16,
                                               addressing::tile_slab_offset(x_off[p], s * KSTEP, x_piece[p], k_range), 0, 0, 0);
#endif
  };
  auto fetch_w = [&](const int s, const int j) {
#if defined(__HIP_DEVICE_COMPILE__)
    wq[j].n = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_src, addressing::ring_w_step_offset(tiled, w_off, s * KSTEP, piece, k_range), 0, 0));
#endif
  };

  f32x16_t acc[T];
#pragma unroll
  for (int c = 0; c < T; ++c)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[c][v] = 0.f;

  const int steps = (k_range + KSTEP - 1) / KSTEP;
#pragma unroll
  for (int j = 0; j < AHEAD; ++j) {
    fetch_x(j, j);
    fetch_w(j, j);
    __builtin_amdgcn_sched_barrier(0);      // in this order: the waits in the loop count on it
  }
  int buf = 0;
  auto step = [&](const int s, const int j) {
    // step s has landed for every wave, and everybody has left the buffer of step s - 1
    block_barrier_keeping_loads<(AHEAD - 1) * (XI + 1)>();
    const uint16_t* x_base = lds + (buf * XROWS + frow) * KSTEP + place;
    Frag x[T];
#pragma unroll
    for (int c = 0; c < T; ++c) x[c].n = *reinterpret_cast<const u32x4_t*>(x_base + c * 32 * KSTEP);
    fetch_x(s + AHEAD, buf == 0 ? NB - 1 : buf - 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < T; ++c) acc[c] = mfma32(wq[j], x[c], acc[c]);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(s + AHEAD, j);                  // behind the last use of the registers it fills: in others the loop ends with copies
    buf = buf == NB - 1 ? 0 : buf + 1;
  };
  // Whole rounds of AHEAD steps without a branch, the last steps perhaps beyond the range (zeros): with one the compiler moves
  // the weights in flight to other registers, and waits for all of them
  for (int s0 = 0; s0 < steps; s0 += AHEAD) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) step(s0 + j, j);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);       // nothing may still be on its way into LDS when the sums take it over
  __syncthreads();

  // acc[c][v] is C^T[n0 + rows32*32 + 8*(v/4) + 4*(lane/32) + v%4][c*32 + lane%32], a quarter of it: quarters 2 and 3 hand
  // theirs to 0 and 1, and what is left are two tiles [64][TOKENS] to be added
  float* red = reinterpret_cast<float*>(lds);
  auto at = [&](const int c, const int v) {
    return ((quarter % 2) * RING_ROWS + rows32 * 32 + 8 * (v / 4) + 4 * (lane / 32) + v % 4) * PITCH + c * 32 + frow;
  };
  if (quarter >= 2) {
#pragma unroll
    for (int c = 0; c < T; ++c)
#pragma unroll
      for (int v = 0; v < 16; ++v) red[at(c, v)] = acc[c][v];
  }
  __syncthreads();
  if (quarter < 2) {
#pragma unroll
    for (int c = 0; c < T; ++c)
#pragma unroll
      for (int v = 0; v < 16; ++v) red[at(c, v)] += acc[c][v];
  }
  __syncthreads();
  auto total = [&](const int n, const int m) { return red[n * PITCH + m] + red[(RING_ROWS + n) * PITCH + m]; };

  if (splits == 1 && EPI == EPI_SWIGLU) {
    // rows [gate 16 | up 16 | gate 16 | up 16]: 32 features per block
    for (int idx = tid; idx < 32 * M; idx += 512) {
      const int j = idx % 16, pair = (idx / 16) % 2, m = idx / 32;
      if (n0 + pair * 32 + 16 + j >= N) continue;
      const float g = total(pair * 32 + j, m), u = total(pair * 32 + 16 + j, m);
      reinterpret_cast<bf16_t*>(Cv)[(long)m * ldc + n0 / 2 + pair * 16 + j] = from_float<bf16_t>(g / (1.0f + expf(-g)) * u);
    }
    return;
  }
  float* mine = part + (long)blockIdx.y * M * N;
  for (int idx = tid; idx < RING_ROWS * M; idx += 512) {
    const int nl = idx % RING_ROWS, m = idx / RING_ROWS;
    if (n0 + nl >= N) continue;
    if (splits == 1) epilogue_store<EPI>(Cv, ldc, m, n0 + nl, total(nl, m));
    else mine[(long)m * N + n0 + nl] = total(nl, m);   // the consumer adds the splits in split order
  }
}

// The product of up to 16 tokens with all of k in a block, from the weights' copy.  A block takes 8, 16 or 32 rows and each of
// its four or eight waves a share of k: nothing is staged or shared, the loads of eight steps (four with 32 rows) are in flight,
// and the waves' tiles are added once, in LDS.  With 8 rows lanes 8..15 of a column hold the step's second fragment of rows
// 0..7, so a step is one load and two matrix instructions (one up to 8 tokens: columns 8..15 then hold the tokens' second
// fragment), of whose results half are of use.
// Bound by the weights' way from memory, and from 8 tokens on by the activations' from L2, which every block reads.
//
// ROWS_FINISH: X[M, N] += A . W^T of a stream, and of the stream's next norm what needs no other block: h = bfloat16(x * w) and
// the block's share of the rows' sums of x^2.  The root is left to whoever reads h (LEFT): h is rounded once and by as much as
// the normalised row would be, and the factor is applied to float32 sums.  In place of a product in pieces of k and a norm that
// adds them, the second of which does little but start.  Weights cold, with that norm, 1 / 8 / 12 tokens, us: 2,048 x 8,192
// 12.5 / 12.4 / 12.6 -> 8.6 / 9.9 / 11.6; 2,048 x 2,048 7.2 / 7.4 / 7.7 -> 3.9 / 4.3 / 4.7; 3,072 x 8,192 16.9 / 17.2 / 17.6 -> 12.4 /
// 13.4 / 14.8; 4,096 x 14,336 29.2 / 29.7 / 30.2 -> 23.7 / 24.2 / 25.6; 4,096 x 4,096 14.2 / 14.5 / 14.9 -> 8.8 / 9.3 / 10.1.
// The reader's part takes 0.2 to 0.5 us where the sums' loads go out behind the weights' (1.0 in front of them).
//
// The other epilogues take the place of gemm_skinny_kernel, four waves on 32 rows that staged the activations of a step at a
// time, where that did not cut k over blocks: 16,384 x 2,048 with the gated unit, 1 / 8 / 16 tokens 15.7 / 15.8 / 15.6 us -> 14.5 /
// 14.4 / 15.4; 28,672 x 4,096 50.4 / 50.1 / 51.1 -> 43.6 / 44.8 / 46.0; 128,256 x 2,048 93.4 / 96.3 / 102.7 -> 90.8 / 93.2 / 100.7.
enum { ROWS_FINISH = 8, ROWS_CLAMPED = 9 };      // besides EPI_BF16, EPI_F32, EPI_ACCUM and EPI_SWIGLU

// the clamped gated unit (elementwise.hip's, with its roundings) of a gate and an up value with their biases
__device__ inline float clamped_unit(float g, float u, float limit, float alpha) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
}

struct FinishTo {
  const void* weight;          // ROWS_FINISH: of the norm, bfloat16 or float32
  bf16_t* h;
  float* sums;
  const float* bias;           // ROWS_FINISH: joins the update, [N], or null; ROWS_CLAMPED: of the gate and up rows, [N]
  float limit, alpha;          // ROWS_CLAMPED: the unit's (clamped_glu)
};

// Source: nothing (A), or a RangeSource: attention's key ranges, up to FINISH_RANGES, which the block merges into LDS while its
// weights travel, a thread four features of every token.
#define FINISH_RANGES 16
template <int WAVES, int ROWS, bool WIDE, int EPI, bool LEFT, typename TW, typename... Source>
__global__ __launch_bounds__(WAVES * 64) void gemm_rows_kernel(void* __restrict__ Cv, long ldc, const bf16_t* __restrict__ A, long lda,
                                                              const bf16_t* __restrict__ W, int M, int N, int K, FinishTo fin, LeftNorm left,
                                                              Source... source) {
  constexpr bool RANGES = sizeof...(Source) > 0;
  extern __shared__ __attribute__((aligned(16))) uint2 merged[];     // RANGES: [K / 8][TOKENS], a piece's tokens turned by the piece
  static_assert(ROWS == 8 || (WIDE && (ROWS == 16 || ROWS == 32)), "8, 16 or 32 rows");
  constexpr int DEPTH = ROWS == 32 ? 4 : 8;                // steps whose loads are in flight
  constexpr int RT = ROWS == 32 ? 2 : 1;                   // tiles of 16 rows (or one of 8)
  constexpr int XF = WIDE ? 2 : 1, WF = ROWS == 8 ? 1 : 2; // fragments of a step: activations, weights of a tile
  constexpr int PARTS = ROWS == 8 ? 2 * WAVES : WAVES;     // sums to add
  constexpr bool GATED = EPI == EPI_SWIGLU || EPI == ROWS_CLAMPED;
  constexpr int OUT_ROWS = GATED ? ROWS / 2 : ROWS, TOKENS = WIDE ? 16 : 8;
  __shared__ float red[PARTS][ROWS][17];
  __shared__ float factors[LEFT ? 16 : 1];
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int lr = lane % 16, lg = lane / 16;
  // blocks go to the dies in turn: every die a run of rows, so that a line of the result is written by one die
  const int dies = gridDim.x % 8 == 0 ? 8 : 1, block = blockIdx.x % dies * (gridDim.x / dies) + blockIdx.x / dies;
  const long n0 = (long)block * ROWS;
  float x = 0.f, wn = 0.f;
  if constexpr (EPI == ROWS_FINISH) {
    if (tid / ROWS < M) {
      x = reinterpret_cast<const float*>(Cv)[(long)(tid / ROWS) * N + n0 + tid % ROWS];
      wn = to_float(reinterpret_cast<const TW*>(fin.weight)[n0 + tid % ROWS]);
      if (fin.bias) x += fin.bias[n0 + tid % ROWS];
    }
  }
  const addressing::WaveRange range = addressing::wave_share(0, K, WAVES, wave);
  const int steps = range.k1 > range.k0 ? (range.k1 - range.k0) / KSTEP : 0;
#if defined(__HIP_DEVICE_COMPILE__)
  __amdgpu_buffer_rsrc_t w_src[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) w_src[t] = operand_descriptor(W, addressing::rows_w_descriptor(n0 + t * 16, range.k0, steps, K));
  const __amdgpu_buffer_rsrc_t a_src = operand_descriptor(A, addressing::rows_a_descriptor(range.k0, steps, M, lda));
#endif
  const unsigned w_lane = addressing::rows_w_lane(ROWS == 8 ? 8 : 16, n0, lane), a_lane = addressing::rows_a_lane(WIDE, lane, M, lda);

  Frag w[DEPTH][RT][WF], a[DEPTH][XF];
  constexpr int ACCS = ROWS == 8 ? XF : RT;
  f32x4_t acc[ACCS];
#pragma unroll
  for (int f = 0; f < ACCS; ++f) acc[f] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](const int s, const int j) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int f = 0; f < WF; ++f)
        w[j][t][f].n = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_src[t], addressing::rows_step(w_lane, s, steps, 2048, f * 1024), 0, 0));
#pragma unroll
    for (int f = 0; f < (RANGES ? 0 : XF); ++f)
      a[j][f].n = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_src, addressing::rows_step(a_lane, s, steps, 2 * KSTEP, f * 16), 0, 0));
#endif
  };
#pragma unroll
  for (int j = 0; j < DEPTH; ++j) fetch(j, j);
  if constexpr (RANGES) {
    const RangeSource rs{source...};
    const int rec = rs.head_dim + 4;
    for (int quad = tid; quad < K / 4; quad += WAVES * 64) {
      const int head = quad * 4 / rs.head_dim, f0 = quad * 4 - head * rs.head_dim, piece = quad / 2;
      const float* base = rs.ranges + (long)head * rs.count * rec;
      const long token_stride = (long)rs.heads * rs.count * rec;
      auto store = [&](const int token, const uint2 packed) { merged[(piece * TOKENS + (token + piece) % TOKENS) * 2 + quad % 2] = packed; };
      if (rs.count <= 4) merge_ranges_of_tokens<4, 1>(base, token_stride, rs.count, rec, rs.head_dim, f0, 0, 1, M, store);
      else if (rs.count <= 8) merge_ranges_of_tokens<8, 1>(base, token_stride, rs.count, rec, rs.head_dim, f0, 0, 1, M, store);
      else merge_ranges_of_tokens<FINISH_RANGES, 1>(base, token_stride, rs.count, rec, rs.head_dim, f0, 0, 1, M, store);
    }
    __syncthreads();
  }
  LeftNormRows rows_left;
  if constexpr (LEFT) {
    __builtin_amdgcn_sched_barrier(0);          // behind the weights' loads, whose waits then do not include them
    if (wave < 4) rows_left.load(left, wave, lane, M);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int s0 = 0; s0 < steps; s0 += DEPTH) {
    const bool more = s0 + DEPTH < steps;
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      if constexpr (RANGES) {
        // (of tokens beyond M what LDS holds, which only reaches columns that are never stored)
#pragma unroll
        for (int f = 0; f < XF; ++f) {
          const int piece = range.k0 / 8 + (s0 + j) * 8 + lg * 2 + (WIDE ? f : lr / 8), token = WIDE ? lr : lr % 8;
          a[j][f] = zero_frag();
          if (s0 + j < steps) a[j][f].n = *reinterpret_cast<const u32x4_t*>(merged + (piece * TOKENS + (token + piece) % TOKENS) * 2);
        }
      }
#pragma unroll
      for (int f = 0; f < XF; ++f)
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          f32x4_t& sum = acc[ROWS == 8 ? f : t];
          sum = mfma16(w[j][t][f % WF], a[j][f], sum);
        }
      if (more) fetch(s0 + DEPTH + j, j);
    }
  }
  if constexpr (LEFT) {
    if (wave < 4) rows_left.finish(left, wave, lane, factors);
  }
  // row lg * 4 + i, column lr of a tile; with 8 rows the weights' fragment lg / 2 of row (lg % 2) * 4 + i
  if constexpr (ROWS != 8) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][t * 16 + lg * 4 + i][lr] = acc[t][i];
  } else if constexpr (WIDE) {
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave * 2 + lg / 2][(lg % 2) * 4 + i][lr] = lg < 2 ? acc[0][i] : acc[1][i];
  } else if (lr / 8 == lg / 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave * 2 + lg / 2][(lg % 2) * 4 + i][lr % 8] = acc[0][i];
  }
  __syncthreads();
  for (int at = tid; at < OUT_ROWS * TOKENS; at += WAVES * 64) {          // whole waves
    const int token = at / OUT_ROWS, row = at % OUT_ROWS;
    const bool mine = token < M;
    auto total = [&](const int r, float sum) {
#pragma unroll
      for (int p = 0; p < PARTS; ++p) sum += red[p][r][token];
      return sum;
    };
    if constexpr (EPI == ROWS_FINISH) {
      static_assert(OUT_ROWS * TOKENS <= WAVES * 64, "one result to a thread");
      x = total(row, x);
      float square = x * x;
#pragma unroll
      for (int off = 1; off < ROWS; off <<= 1) square += __shfl_xor(square, off, PI_WAVE);
      if (!mine) return;
      reinterpret_cast<float*>(Cv)[(long)token * N + n0 + row] = x;
      fin.h[(long)token * N + n0 + row] = from_float<bf16_t>(x * wn);
      if (row == 0) fin.sums[(long)token * gridDim.x + block] = square;
    } else if (mine) {
      const float factor = LEFT ? factors[token] : 1.f;
      if constexpr (EPI == ROWS_CLAMPED) {
        const float g = total(row, 0.f) * factor + fin.bias[n0 + row], u = total(16 + row, 0.f) * factor + fin.bias[n0 + 16 + row];
        reinterpret_cast<bf16_t*>(Cv)[(long)token * ldc + n0 / 2 + row] = from_float<bf16_t>(clamped_unit(g, u, fin.limit, fin.alpha));
      } else if constexpr (EPI == EPI_SWIGLU) {
        const float g = total(row, 0.f) * factor, u = total(16 + row, 0.f) * factor;
        reinterpret_cast<bf16_t*>(Cv)[(long)token * ldc + n0 / 2 + row] = from_float<bf16_t>(g / (1.0f + expf(-g)) * u);
      } else {
        epilogue_store<EPI>(Cv, ldc, token, n0 + row, total(row, 0.f) * factor);
      }
    }
  }
}

// Rows of a block: 8 while blocks of 16 would leave more than a quarter of the units without one (2,048 x 8,192, one token 8.6
// and 10.0 us; 3,072 x 8,192 13.0 and 12.4, eight tokens 16.9 and 13.4).
static int finish_rows(int N) { return N / 16 * 4 < 3 * compute_units() ? 8 : 16; }

// Blocks (= pieces of a row's sum of squares) with which the finishing kernel takes a product, 0 where it does not: M up to 16,
// N % 64 and K % 64, up to 512 blocks (what LeftNormRows holds), and not many tokens, whose activations every block reads, of a long
// k with 8 rows to a block (2,048 x 8,192: 12 tokens 12.6 in pieces with the norm and 11.6, 16 tokens 12.8 and 13.0; none
// measured between) or with blocks for a part of a second round (5,120 rows, 320 blocks, k of 5,120 and 13,824 in the mean with
// the norm and the gap to it: 12 tokens 27.9 and 27.8, 16 tokens 28.4 and 32.1; 8,192 rows, two whole rounds, 16 tokens 62.8 and 62.9).
extern "C" int pi_gemm_finish_blocks(int M, int N, int K) {
  if (M < 1 || M > 16 || N < 64 || N % 64 || K < KSTEP || K % KSTEP) return 0;
  const int rows = finish_rows(N), blocks = N / rows, units = compute_units();
  if (blocks > 512 || (M > 12 && ((rows == 8 && K > 4096) || (blocks > units && blocks % units)))) return 0;
  return blocks;
}

// W: the copy in the streaming order (see pi_gemm_skinny).  H bfloat16 [M, N], sums float32 [M, blocks].  `bias` (or null): float32
// [N], added to every row of X besides.
extern "C" int pi_gemm_finish(float* X, const void* A, long lda, const void* W, const void* norm_w, int norm_dtype, void* H, float* sums, long sums_elems,
                              const float* bias, int M, int N, int K, hipStream_t stream) {
  const int blocks = pi_gemm_finish_blocks(M, N, K);
  PI_REQUIRE(blocks > 0, "gemm_finish: not for M=%d N=%d K=%d", M, N, K);
  PI_REQUIRE(lda >= K && lda % 8 == 0 && lda < RING_MAX_STRIDE && ((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0), "gemm_finish: operands must be 16-byte aligned, the row stride (%ld) a multiple of 8", lda);
  PI_REQUIRE(sums_elems >= (long)M * blocks, "gemm_finish: %ld floats for %ld sums", sums_elems, (long)M * blocks);
  PI_REQUIRE(norm_dtype == PI_F32 || norm_dtype == PI_BF16, "gemm_finish: unsupported norm weight dtype %d", norm_dtype);
  // waves: eight for a long k where a unit has no more than a block's worth of loads in flight otherwise
  const int rows = N / blocks;
  const bool eight = K > 2048 && (rows == 8 || blocks < compute_units());
#define GO(WV, RW, WD, T) \
  hipLaunchKernelGGL((gemm_rows_kernel<WV, RW, WD, ROWS_FINISH, false, T>), dim3(blocks), dim3(WV * 64), 0, stream, X, (long)N, (const bf16_t*)A, lda, \
                     (const bf16_t*)W, M, N, K, FinishTo{norm_w, (bf16_t*)H, sums, bias, 0.f, 0.f}, LeftNorm{})
#define PICK(WV, T) \
  do { \
    if (rows == 16) GO(WV, 16, true, T); \
    else if (M > 8) GO(WV, 8, true, T); \
    else GO(WV, 8, false, T); \
  } while (0)
  if (eight && norm_dtype == PI_BF16) PICK(8, bf16_t);
  else if (eight) PICK(8, float);
  else if (norm_dtype == PI_BF16) PICK(4, bf16_t);
  else PICK(4, float);
#undef PICK
#undef GO
  return pi_check_launch("gemm_finish");
}

// Attention's key ranges as activations of the finishing product: blocks of 8 rows, each of which merges them all, so for one
// token only.  Decode steps of 16 layers, 32 heads of 64, by the merging kernel and inside, us: one token with 2, 4, 8 and 16
// ranges (17 to 136 KB) 761 / 748, 760 / 746, 766 / 752 and 773 / 764; two with 4 and 8 771 / 771 and 777 / 774, three with 4 782 /
// 797, four with 2 and 4 794 / 795 and 800 / 801, eight with 2 834 / 849, sixteen with 2 1,011 / 1,082; of 12 layers, 16 heads: one
// with 16 411 / 392, eight with 4 433 / 482, sixteen with 2 481 / 537.
#define FINISH_RANGE_BYTES (144 << 10)
#define FINISH_RANGE_LDS (64 << 10)

// Blocks, as pi_gemm_finish_blocks, with which the finishing kernel merges the ranges itself; 0: it does not.
extern "C" int pi_gemm_finish_ranges_blocks(int M, int N, int heads, int head_dim, int count) {
  const long K = (long)heads * head_dim;
  if (M != 1 || head_dim < 8 || head_dim % 8 || count < 1 || count > FINISH_RANGES || K > 8192 || !pi_gemm_finish_blocks(M, N, (int)K) || finish_rows(N) != 8) return 0;
  if ((long)heads * count * (head_dim + 4) * 4 > FINISH_RANGE_BYTES || K * 8 * 2 > FINISH_RANGE_LDS) return 0;
  return N / 8;
}

template <typename TW>
static int launch_finish_ranges(float* X, const RangeSource& rs, const bf16_t* W, const void* norm_w, bf16_t* H, float* sums, int M, int N, int K, hipStream_t stream) {
  const auto kernel = gemm_rows_kernel<8, 8, false, ROWS_FINISH, false, TW, RangeSource>;
  static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, FINISH_RANGE_LDS);
  if (configured != hipSuccess) return pi_fail("gemm_finish: cannot reserve %d bytes of LDS: %s", FINISH_RANGE_LDS, hipGetErrorString(configured));
  hipLaunchKernelGGL(kernel, dim3(N / 8), dim3(512), (size_t)K * 8 * 2, stream, X, (long)N, (const bf16_t*)nullptr, 0L, W, M, N, K,
                     FinishTo{norm_w, H, sums, nullptr, 0.f, 0.f}, LeftNorm{}, rs);
  return pi_check_launch("gemm_finish (key ranges merged on the way in)");
}

// pi_gemm_finish whose activations are attention's key ranges (`ranges`: float32 [M, heads, count, head_dim + 4], see RangeSource).
extern "C" int pi_gemm_finish_ranges(float* X, const void* ranges, int heads, int head_dim, int count, const void* W, const void* norm_w, int norm_dtype,
                                     void* H, float* sums, long sums_elems, int M, int N, hipStream_t stream) {
  const int blocks = pi_gemm_finish_ranges_blocks(M, N, heads, head_dim, count), K = heads * head_dim;
  PI_REQUIRE(blocks > 0, "gemm_finish: not for %d ranges of %d heads of %d, M=%d N=%d", count, heads, head_dim, M, N);
  PI_REQUIRE(((uintptr_t)ranges % 16 == 0) && ((uintptr_t)W % 16 == 0), "gemm_finish: operands must be 16-byte aligned");
  PI_REQUIRE(sums_elems >= (long)M * blocks, "gemm_finish: %ld floats for %ld sums", sums_elems, (long)M * blocks);
  PI_REQUIRE(norm_dtype == PI_F32 || norm_dtype == PI_BF16, "gemm_finish: unsupported norm weight dtype %d", norm_dtype);
  const RangeSource rs{(const float*)ranges, heads, head_dim, count};
  const bf16_t* w = (const bf16_t*)W;
  if (norm_dtype == PI_BF16) return launch_finish_ranges<bf16_t>(X, rs, w, norm_w, (bf16_t*)H, sums, M, N, K, stream);
  return launch_finish_ranges<float>(X, rs, w, norm_w, (bf16_t*)H, sums, M, N, K, stream);
}

// C[M, N] = A[M, K] . W[N, K]^T for 1..16 tokens with all of k in a block, W the copy in the streaming order: stored in
// bfloat16 or float32, added into float32, or through the gated unit (gate and up rows interleaved by 16).  `sums` (or null; not
// with the sum): A is what pi_gemm_finish left of a norm; float32 [M, count], 16-byte aligned, K the norm's width.
extern "C" int pi_gemm_rows(void* C, int epilogue, long ldc, const void* A, long lda, const void* W, int M, int N, int K, const float* sums, int count,
                            float eps, hipStream_t stream) {
  PI_REQUIRE(M > 0 && M <= 16 && N > 0 && N % 16 == 0 && K > 0 && K % KSTEP == 0, "gemm_rows: takes 1..16 tokens, N in 16 and K in 64, got M=%d N=%d K=%d", M, N, K);
  PI_REQUIRE(epilogue != EPI_SWIGLU || N % 32 == 0, "gemm_rows: the gated unit takes N (%d) in 32", N);
  PI_REQUIRE(lda >= K && lda % 8 == 0 && lda < RING_MAX_STRIDE && K < RING_MAX_STRIDE && ((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0), "gemm_rows: operands must be 16-byte aligned, the row stride (%ld) a multiple of 8", lda);
  PI_REQUIRE(!sums || (count > 0 && count <= 512 && count % 4 == 0 && (uintptr_t)sums % 16 == 0), "gemm_rows: a left norm has 4..512 sums a row, got %d", count);
  PI_REQUIRE(!sums || epilogue != EPI_ACCUM, "gemm_rows: a sum does not take a left norm");
  // 16 rows to a block while the units take them in one round (3,072 x 2,048, 8 tokens 5.0 us and 6.0; 5,120 x 3,072 11.4 and 8.7)
  const int rows = epilogue == EPI_SWIGLU || (N / 16 > compute_units() && N % 32 == 0) ? 32 : 16;
  const LeftNorm left{sums, count, K, eps};
#define GO(RW, E, L) hipLaunchKernelGGL((gemm_rows_kernel<4, RW, true, E, L, float>), dim3(N / RW), dim3(256), 0, stream, C, ldc, (const bf16_t*)A, lda, (const bf16_t*)W, M, N, K, FinishTo{}, left)
#define PICK(E) \
  do { \
    if (sums && rows == 32) GO(32, E, true); \
    else if (sums) GO(16, E, true); \
    else if (rows == 32) GO(32, E, false); \
    else GO(16, E, false); \
  } while (0)
  switch (epilogue) {
    case EPI_BF16: PICK(EPI_BF16); break;
    case EPI_F32: PICK(EPI_F32); break;
    case EPI_ACCUM:
      if (rows == 32) GO(32, EPI_ACCUM, false);
      else GO(16, EPI_ACCUM, false);
      break;
    case EPI_SWIGLU:
      if (sums) GO(32, EPI_SWIGLU, true);
      else GO(32, EPI_SWIGLU, false);
      break;
    default: return pi_fail("gemm_rows: unknown epilogue %d", epilogue);
  }
#undef PICK
#undef GO
  return pi_check_launch("gemm_rows");
}

// out[M, N / 2] = the clamped gated unit of A . W^T + bias, gate and up rows of W and bias interleaved by 16, in the product's own
// kernel (a kernel of its own behind the float32 product took 4.6 us a layer at 12 tokens).  Operands as for pi_gemm_rows.
extern "C" int pi_gemm_rows_clamped(void* C, long ldc, const void* A, long lda, const void* W, int M, int N, int K, const float* bias, float limit, float alpha,
                                    const float* sums, int count, float eps, hipStream_t stream) {
  PI_REQUIRE(M > 0 && M <= 16 && N > 0 && N % 32 == 0 && K > 0 && K % KSTEP == 0 && bias, "gemm_rows_clamped: takes 1..16 tokens, N in 32 and K in 64, got M=%d N=%d K=%d", M, N, K);
  PI_REQUIRE(lda >= K && lda % 8 == 0 && lda < RING_MAX_STRIDE && K < RING_MAX_STRIDE && ((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0), "gemm_rows_clamped: operands must be 16-byte aligned, the row stride (%ld) a multiple of 8", lda);
  PI_REQUIRE(!sums || (count > 0 && count <= 512 && count % 4 == 0 && (uintptr_t)sums % 16 == 0), "gemm_rows_clamped: a left norm has 4..512 sums a row, got %d", count);
  const FinishTo unit{nullptr, nullptr, nullptr, bias, limit, alpha};
  const LeftNorm left{sums, count, K, eps};
  if (sums)
    hipLaunchKernelGGL((gemm_rows_kernel<4, 32, true, ROWS_CLAMPED, true, float>), dim3(N / 32), dim3(256), 0, stream, C, ldc, (const bf16_t*)A, lda, (const bf16_t*)W, M, N, K, unit, left);
  else
    hipLaunchKernelGGL((gemm_rows_kernel<4, 32, true, ROWS_CLAMPED, false, float>), dim3(N / 32), dim3(256), 0, stream, C, ldc, (const bf16_t*)A, lda, (const bf16_t*)W, M, N, K, unit, left);
  return pi_check_launch("gemm_rows (clamped unit)");
}

template <int MB>
static int launch_mb(int epi, dim3 grid, hipStream_t stream, void* C, long ldc, const bf16_t* X, long ldx, const bf16_t* W,
                     long ldw, int M, int N, int K, int kpb, float* part, int tiled) {
#define GO(E) hipLaunchKernelGGL((gemm_skinny_kernel<MB, E>), grid, dim3(256), 0, stream, C, ldc, X, ldx, W, ldw, M, N, K, kpb, part, RangeSource{}, tiled)
  switch (epi) {
    case EPI_BF16: GO(EPI_BF16); break;
    case EPI_F32: GO(EPI_F32); break;
    case EPI_ACCUM: GO(EPI_ACCUM); break;
    case EPI_SWIGLU: GO(EPI_SWIGLU); break;
    default: return pi_fail("gemm_skinny: unknown epilogue %d", epi);
  }
#undef GO
  return pi_check_launch("gemm_skinny");
}

template <int T, int EPI>
static int launch_ring_of(dim3 grid, hipStream_t stream, void* C, long ldc, const bf16_t* X, long ldx, const bf16_t* W, long ldw, int M, int N, int K,
                          int kpb, float* part, int tiled) {
  constexpr size_t ring = RING_BUFFERS * (T == 2 ? 64 : 128) * KSTEP * sizeof(uint16_t), sums = 2 * RING_ROWS * (T * 32 + 1) * sizeof(float);
  constexpr size_t bytes = ring > sums ? ring : sums;        // at most 80 KB: two blocks to a unit
  static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_skinny_ring_kernel<T, EPI>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (configured != hipSuccess) return pi_fail("gemm_skinny: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(configured));
  hipLaunchKernelGGL((gemm_skinny_ring_kernel<T, EPI>), grid, dim3(512), bytes, stream, C, ldc, X, ldx, W, ldw, M, N, K, kpb, part, tiled);
  return pi_check_launch("gemm_skinny (rings)");
}

template <int T>
static int launch_ring(int epi, dim3 grid, hipStream_t stream, void* C, long ldc, const bf16_t* X, long ldx, const bf16_t* W, long ldw, int M, int N,
                       int K, int kpb, float* part, int tiled) {
  switch (epi) {
    case EPI_BF16: return launch_ring_of<T, EPI_BF16>(grid, stream, C, ldc, X, ldx, W, ldw, M, N, K, kpb, part, tiled);
    case EPI_F32: return launch_ring_of<T, EPI_F32>(grid, stream, C, ldc, X, ldx, W, ldw, M, N, K, kpb, part, tiled);
    case EPI_ACCUM: return launch_ring_of<T, EPI_ACCUM>(grid, stream, C, ldc, X, ldx, W, ldw, M, N, K, kpb, part, tiled);
    case EPI_SWIGLU: return launch_ring_of<T, EPI_SWIGLU>(grid, stream, C, ldc, X, ldx, W, ldw, M, N, K, kpb, part, tiled);
  }
  return pi_fail("gemm_skinny: unknown epilogue %d", epi);
}

// Which of the two kernels; the caller asks here, and sizes its k-split by the answer (fast.py).  For 17 to 32 tokens the one that shares
// its activations is the better one on matrices of some 40 MB and more (17 / 32 tokens, us, in the norm's or the head's place: 4,096 x 14,336
// 28.5 / 29.6 -> 26.5 / 26.7, 3,072 x 8,192 17.1 / 18.9 -> 16.0 / 16.3, 6,144 x 4,096 15.6 / 17.5 -> 15.7 / 16.1, 28,672 x 4,096 50.8 / 51.1 ->
// 46.3 / 46.9, 128,256 x 4,096 199.8 / 211.1 -> 199.3 / 201.6) and the worse one below (2,048 x 8,192 13.0 / 13.5 -> 14.0 / 14.2, 2,048 x 2,048
// 8.0 / 8.3 -> 8.4 / 8.7).  At the line, with the norm that adds the pieces: 5,120 x 4,096 17.8 / 19.1 -> 16.0 / 16.3, 2,560 x 8,192 15.8 /
// 17.5 -> 15.5 / 15.9, 10,240 x 2,048 19.0 / 20.7 -> 18.5 / 19.9, 2,048 x 10,240 14.6 / 15.9 -> 14.8 / 15.2; with the gated unit 13.0 / 13.6 ->
// 12.1 / 12.4 for 10,240 x 2,048.
extern "C" int pi_gemm_skinny_shares(int M, int N, int K, long ldx, long ldw) {
  return M > SHARED_FROM_TOKENS || (M > 16 && (long)N * K >= SHARED_FROM_ELEMENTS && ldx < RING_MAX_STRIDE && ldw < RING_MAX_STRIDE && K < RING_MAX_STRIDE);
}

// splits > 1: the partial products go to `part` (float32 [splits, M, N]) and C is not touched;
// *splits_out tells how many splits were made (no empty ones).
// `tiled` != 0: W is not [N, K] row after row but a copy in the order the kernels' loads want it,
// [N / 16][K / 64][2][4][16][8]: for 16 rows and 64 k, first the k of every lane's first
// fragment, then of its second; in each, lane group g's k = 16 g + 8 h .. + 7 of rows 0..15.
// A wave's load instruction then reads 1 KB in a row instead of 64 bytes from each of 16 rows.
// N must be a multiple of 16 and K of 64.
extern "C" int pi_gemm_skinny(void* C, int epilogue, long ldc, const void* X, long ldx, const void* W, long ldw, int M,
                              int N, int K, int splits, void* part, long part_elems, int* splits_out, int tiled,
                              hipStream_t stream) {
  PI_REQUIRE(!tiled || (N % 16 == 0 && K % 64 == 0), "gemm_skinny: a tiled weight matrix needs N (%d) a multiple of 16 and K (%d) of 64", N, K);
  PI_REQUIRE(M > 0 && M <= 128 && N > 0 && K > 0, "gemm_skinny: takes 1..128 rows, got M=%d N=%d K=%d", M, N, K);
  PI_REQUIRE(K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0, "gemm_skinny: K (%d) and row strides (%ld, %ld) must be multiples of 8", K, ldx, ldw);
  PI_REQUIRE(((uintptr_t)X % 16 == 0) && ((uintptr_t)W % 16 == 0), "gemm_skinny: operands must be 16-byte aligned");
  PI_REQUIRE(splits >= 1 && splits <= 65535, "gemm_skinny: bad split count %d", splits);
  PI_REQUIRE(epilogue != EPI_SWIGLU || (splits == 1 && N % 32 == 0), "gemm_skinny: the SwiGLU epilogue needs one split and N (%d) a multiple of 32", N);
  const bool shared = pi_gemm_skinny_shares(M, N, K, ldx, ldw);
  const int groups = ceil_div(N, shared ? RING_ROWS : ROWS_PER_BLOCK);
  const addressing::KSplit cut = addressing::cut_k(K, splits, KSTEP);
  const int kpb = cut.k_per_block;
  splits = cut.splits;                            // no empty splits
  if (splits > 1)
    PI_REQUIRE(part && part_elems >= (long)splits * M * N, "gemm_skinny: workspace too small (%ld floats for %ld)", part_elems, (long)splits * M * N);
  if (splits_out) *splits_out = splits;
  const dim3 grid(groups, splits);
  const int mb = (M + 15) / 16;
  const bf16_t *x = (const bf16_t*)X, *w = (const bf16_t*)W;
  if (shared) {
    PI_REQUIRE(ldx < RING_MAX_STRIDE && ldw < RING_MAX_STRIDE && K < RING_MAX_STRIDE, "gemm_skinny: K (%d) or row strides (%ld, %ld) are too long for 32-bit offsets", K, ldx, ldw);
    if (M <= 64) return launch_ring<2>(epilogue, grid, stream, C, ldc, x, ldx, w, ldw, M, N, K, kpb, (float*)part, tiled);
    if (M <= 96) return launch_ring<3>(epilogue, grid, stream, C, ldc, x, ldx, w, ldw, M, N, K, kpb, (float*)part, tiled);
    return launch_ring<4>(epilogue, grid, stream, C, ldc, x, ldx, w, ldw, M, N, K, kpb, (float*)part, tiled);
  }
  switch (mb) {
    case 1: return launch_mb<1>(epilogue, grid, stream, C, ldc, x, ldx, w, ldw, M, N, K, kpb, (float*)part, tiled);
    default: return launch_mb<2>(epilogue, grid, stream, C, ldc, x, ldx, w, ldw, M, N, K, kpb, (float*)part, tiled);
  }
}

// The same product for a decode step of up to 16 tokens whose activations are attention's key
// ranges not yet merged (`ranges`: float32 [M, heads, count, head_dim + 4], see RangeSource): K
// is heads * head_dim, and head_dim a multiple of the kernel's k step so that a step's features
// belong to one head.  Epilogues: store bf16, store f32, add into f32.
extern "C" int pi_gemm_skinny_ranges(void* C, int epilogue, long ldc, const void* ranges, int heads, int head_dim, int count,
                                     const void* W, long ldw, int M, int N, int splits, void* part, long part_elems,
                                     int* splits_out, int tiled, hipStream_t stream) {
  PI_REQUIRE(M > 0 && M <= 16 && N > 0 && heads > 0 && count >= 1 && count <= 64, "gemm_skinny_ranges: takes 1..16 tokens and 1..64 ranges, got M=%d N=%d heads=%d ranges=%d", M, N, heads, count);
  PI_REQUIRE(head_dim > 0 && head_dim % KSTEP == 0, "gemm_skinny_ranges: head_dim %d is no multiple of %d", head_dim, KSTEP);
  PI_REQUIRE(epilogue == EPI_BF16 || epilogue == EPI_F32 || epilogue == EPI_ACCUM, "gemm_skinny_ranges: unknown epilogue %d", epilogue);
  PI_REQUIRE(ldw % 8 == 0 && ((uintptr_t)W % 16 == 0) && ((uintptr_t)ranges % 16 == 0), "gemm_skinny_ranges: operands must be 16-byte aligned");
  PI_REQUIRE(splits >= 1 && splits <= 65535, "gemm_skinny_ranges: bad split count %d", splits);
  const long K = (long)heads * head_dim;
  PI_REQUIRE(K < (1L << 30), "gemm_skinny_ranges: k too long");
  PI_REQUIRE(!tiled || N % 16 == 0, "gemm_skinny_ranges: a tiled weight matrix needs N (%d) a multiple of 16", N);
  const addressing::KSplit cut = addressing::cut_k((int)K, splits, 4 * KSTEP);     // a block's four waves take whole steps
  const int kpb = cut.k_per_block;
  splits = cut.splits;
  if (splits > 1)
    PI_REQUIRE(part && part_elems >= (long)splits * M * N, "gemm_skinny_ranges: workspace too small (%ld floats for %ld)", part_elems, (long)splits * M * N);
  if (splits_out) *splits_out = splits;
  const dim3 grid(ceil_div(N, RANGES_ROW_TILES * 16), splits);
  const RangeSource rs{(const float*)ranges, heads, head_dim, count};
#define GO(E) hipLaunchKernelGGL((gemm_skinny_kernel<1, E, true, RANGES_ROW_TILES>), grid, dim3(256), 0, stream, C, ldc, (const bf16_t*)nullptr, 0L, \
                                 (const bf16_t*)W, ldw, M, N, (int)K, kpb, (float*)part, rs, tiled)
  switch (epilogue) {
    case EPI_BF16: GO(EPI_BF16); break;
    case EPI_F32: GO(EPI_F32); break;
    default: GO(EPI_ACCUM); break;
  }
#undef GO
  return pi_check_launch("gemm_skinny (key ranges merged on the way in)");
}
