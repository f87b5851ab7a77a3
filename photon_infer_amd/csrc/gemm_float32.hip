// float32 matrix products on the matrix cores: C[M, N] (+)= A[M, K] . W[N, K]^T with 32-bit operands and sums, by the
// instructions that take float32 (v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32; 157 TFLOP/s on this chip, twice the
// vector unit's rate without packed instructions) or, for large tiles, by six that take bfloat16 (gemm_float32_parts_kernel).
// They carry the float32 path's products; gemm_general.hip keeps mixed types, odd strides and the products of a few rows that
// it streams faster (ops/fast.py).
//
// K and the row strides are multiples of 4 and the operands 16-byte aligned.  A row of 32 floats is 128 bytes, as a row
// of 64 bfloat16 is, so both kernels move their operands exactly as the bfloat16 kernels do and share those kernels'
// address arithmetic (addressing.h), in units of two bytes: every `2 *` below turns floats into such units.
//
// Up to 32 rows (decode steps): gemm_float32_rows_kernel, bound by the weights' way from memory.  More rows:
// gemm_float32_parts_kernel, bound by the matrix cores, or, for few tiles, gemm_float32_tile_kernel; where the tiles do not
// fill the chip, k is cut over blocks and pi_splitk_reduce adds the pieces in order.
#include "addressing.h"
#include "mfma.h"

#define FSTEP 32                      // floats of k per step: 128 bytes of a row
#define ROWS_MAX_M 32                 // up to this many rows of activations the weight-streaming kernel is taken
#define ROWS_SPLIT_MIN_K 4096         // from this k on a product's pieces are worth a kernel that adds them
#define ROWS_WHOLE_K 768              // up to this k a matrix of many rows is left whole for its reader too
#define FEW_TILES_ROWS 64             // rows and columns of a tile of float32 instructions
#define FEW_TILES_BUFFERS 4           // slabs of it in LDS
#define PARTS_WIDE_MAX_STRIDE (1 << 20)  // floats between weight rows up to which 256 of them lie within a descriptor's 2 GB

// What becomes of a product in one piece: stored, added to C, or, with gate and up rows interleaved in blocks of 16 in W,
// silu(gate) * up of the same feature stored to C [M, N / 2] (a kernel of its own for it took 4.7 us at eight tokens by 8,192
// features and 27 at 1,293; the products take as long as without)
enum { EPI_STORE = 0, EPI_ADD = 1, EPI_SWIGLU = 2 };

__device__ inline float silu_mul(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// ------------------------------------------------------------------ few rows: stream the weights
// The weights are the row operand, the activations the column operand.  A block is WAVES waves on the same RT * 16
// weight rows, each on a share of k; a lane fetches 32 contiguous bytes of a weight row per step, the four lane groups
// of a row 128, and a wave keeps DEPTH steps of loads in flight.  Activations go through the wave's own patch of LDS,
// turned so that neither side has bank conflicts, as in the bfloat16 kernel.  The waves' sums meet in LDS, in pairs.
// See launch_rows() for the shapes.
template <int MB, int RT, int WAVES>
union RowsLds {
  float red[WAVES][RT * 16][MB * 16 + 1];
  u32x4_t xs[WAVES][MB * 8 * 16];
};

template <int MB, int RT, int WAVES, int DEPTH, int EPI>
__global__ __launch_bounds__(WAVES * 64) void gemm_float32_rows_kernel(float* __restrict__ C, long ldc, const float* __restrict__ X, long ldx,
                                                                       const float* __restrict__ W, long ldw, int M, int N, int K,
                                                                       int k_per_block, float* __restrict__ part) {
  constexpr int ROWS = RT * 16;
  static_assert(EPI != EPI_SWIGLU || RT == 2, "a gate's rows and its up rows lie in one block");
  __shared__ RowsLds<MB, RT, WAVES> lds;
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int lr = lane % 16, lg = lane / 16;
  const long n0 = (long)blockIdx.x * ROWS;
  const addressing::WaveRange range = addressing::wave_share(2 * (int)blockIdx.y * k_per_block, 2 * min(K, (int)(blockIdx.y + 1) * k_per_block), WAVES, wave);
  const int k0 = range.k0, k1 = range.k1;                 // in units of two bytes, as all addresses below
  const int steps = k1 > k0 ? (k1 - k0 + addressing::KSTEP - 1) / addressing::KSTEP : 0;
  const bf16_t* Wh = reinterpret_cast<const bf16_t*>(W);
  const bf16_t* Xh = reinterpret_cast<const bf16_t*>(X);

  const bf16_t* wrow[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) wrow[t] = Wh + addressing::skinny_w_base(0, n0, t, lr, lg, N, 2 * K, 2 * ldw);
  const int x_loads = __builtin_amdgcn_readfirstlane((M + 7) / 8);
  const int xt = lane / 8, xp = lane % 8;
  const bf16_t* xsrc[MB * 2];
  int xdst[MB * 2];
#pragma unroll
  for (int i = 0; i < MB * 2; ++i) {
    const int token = i * 8 + xt;
    xsrc[i] = Xh + addressing::skinny_x_base(token, M, 2 * ldx, xp);
    xdst[i] = ((token / 16) * 8 + xp) * 16 + ((token + 2 * xp) & 15);
  }
  u32x4_t* xs = lds.xs[wave];
  int xfrag[MB][2];
#pragma unroll
  for (int c = 0; c < MB; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) xfrag[c][h] = (c * 8 + lg * 2 + h) * 16 + ((lr + 2 * (lg * 2 + h)) & 15);

  f32x4_t acc[RT][MB];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < MB; ++c) acc[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // pieces beyond k1 (the last, partial step) are fetched from a stand-in inside the row and count as zero; steps beyond
  // the last fetch the last again, so that the loads in flight are a number the waits can count on
  u32x4_t wq[DEPTH][RT][2], xq[DEPTH][MB * 2];
  auto fetch = [&](const int s, const int j) {
    const int kk = k0 + min(s, steps - 1) * addressing::KSTEP;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) wq[j][t][h] = *reinterpret_cast<const u32x4_t*>(wrow[t] + addressing::skinny_w_step(0, false, kk, h, lg, k0, k1));
#pragma unroll
    for (int i = 0; i < MB * 2; ++i)
      if (i == 0 || i < x_loads) xq[j][i] = *reinterpret_cast<const u32x4_t*>(xsrc[i] + addressing::skinny_x_step(false, kk, xp, k0, k1));
  };
  auto step = [&](const int s, const int j) {
    const int kk = k0 + s * addressing::KSTEP;
    f32x4_t w[RT][2];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        w[t][h] = __builtin_bit_cast(f32x4_t, addressing::skinny_w_used(false, kk, h, lg, k1) ? wq[j][t][h] : u32x4_t{0u, 0u, 0u, 0u});
    const bool x_ok = kk + xp * 8 < k1;
#pragma unroll
    for (int i = 0; i < MB * 2; ++i)
      if (i == 0 || i < x_loads) xs[xdst[i]] = x_ok ? xq[j][i] : u32x4_t{0u, 0u, 0u, 0u};
    fetch(s + DEPTH, j);
    // the wave reads what its own lanes wrote: LDS serves one wave's accesses in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int c = 0; c < MB; ++c) {
      // a quarter of the step in an accumulator of its own, then all into the running sum: chains of 8 products and one
      // of steps instead of one of all k (at k = 2,048 off by 1e-7 of the result's norm instead of 4e-7)
      f32x4_t sum[RT][4];
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) sum[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4_t x = __builtin_bit_cast(f32x4_t, xs[xfrag[c][h]]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < RT; ++t) sum[t][h * 2 + e % 2] = mfma16_f32(w[t][h][e], x[e], sum[t][h * 2 + e % 2]);
      }
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t][c] += (sum[t][0] + sum[t][1]) + (sum[t][2] + sum[t][3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  if (steps > 0) {
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) fetch(j, j);
    int s0 = 0;
    for (; s0 + DEPTH <= steps; s0 += DEPTH) {
#pragma unroll
      for (int j = 0; j < DEPTH; ++j) step(s0 + j, j);
    }
#pragma unroll
    for (int j = 0; j < DEPTH - 1; ++j)
      if (s0 + j < steps) step(s0 + j, j);
  }
  __syncthreads();                      // the partial tiles take the place of the staged activations
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int c = 0; c < MB; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) lds.red[wave][t * 16 + lg * 4 + r][c * 16 + lr] = acc[t][c][r];
  __syncthreads();
  auto total = [&](const int nl, const int m) {
    float v[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v[w] = lds.red[w][nl][m];
#pragma unroll
    for (int gap = 1; gap < WAVES; gap *= 2)
#pragma unroll
      for (int w = 0; w < WAVES; w += 2 * gap) v[w] += v[w + gap];
    return v[0];
  };
  if (EPI == EPI_SWIGLU) {
    for (int idx = tid; idx < 16 * MB * 16; idx += WAVES * 64) {
      const int j = idx % 16, m = idx / 16;
      if (m < M && n0 + 16 + j < N) C[m * ldc + n0 / 2 + j] = silu_mul(total(j, m), total(16 + j, m));
    }
    return;
  }
  for (int idx = tid; idx < ROWS * MB * 16; idx += WAVES * 64) {
    const int nl = idx % ROWS, m = idx / ROWS;
    if (m >= M || n0 + nl >= N) continue;
    const float sum = total(nl, m);
    if (gridDim.y > 1) {
      part[((long)blockIdx.y * M + m) * N + n0 + nl] = sum;
    } else {
      float* c = C + m * ldc + n0 + nl;
      *c = EPI == EPI_ADD ? *c + sum : sum;
    }
  }
}

// ------------------------------------------------------------------ many rows: tiles
// Where the block's tile lies among tiles_m x tiles_n.
struct TilePlace {
  int m, n;
};
__device__ inline TilePlace tile_place(int tiles_n) {
  const int tiles_m = gridDim.x / tiles_n;
  if (tiles_n % 8 == 0) {                        // a die streams its own slice of W and walks the row tiles of a column first
    const int die = blockIdx.x % 8, local = blockIdx.x / 8;
    return TilePlace{local % tiles_m, die * (tiles_n / 8) + local / tiles_m};
  }
  return TilePlace{(int)blockIdx.x / tiles_n, (int)blockIdx.x % tiles_n};
}

// What becomes of a wave's WM x WN accumulators of 32 x 32, whose first row and column are m_wave and n_wave.  Values v whose bit in
// `chosen` is not set are left out.
template <int WM, int WN, int EPI>
__device__ inline void finish_tiles(const f32x16_t (&acc)[WM][WN], long m_wave, long n_wave, float* __restrict__ C, long ldc, int M, int N,
                                    float* __restrict__ part, const unsigned chosen = 0xffffu) {
  const int lane = threadIdx.x % 64, frow = lane % 32;
  // acc[i][j][v] is C[m_wave + i*32 + 8*(v/4) + 4*(lane/32) + v%4][n_wave + j*32 + lane%32]: a store
  // instruction writes 128 contiguous bytes of two rows.  Added into C, sixteen of its values are fetched before the first
  // is used (one after the other 1,600 x 16,384 x 64 took 113 us, 512 x 16,384 x 512 99; 69 and 87 so)
  if (EPI == EPI_SWIGLU) {
    // columns 0..15 of a wave's 32 are gate rows of W, 16..31 the up rows of the same features: lane l and lane l + 16 swap
    // so that the one has gate and up of row v, the other of row v + 1
    const bool up = frow >= 16;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const long n = n_wave + j * 32;                 // N is a multiple of 32
      if (n >= N) continue;
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        const long mi = m_wave + i * 32 + 4 * (lane / 32);
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
          const float own = up ? acc[i][j][v + 1] : acc[i][j][v], other = __shfl_xor(up ? acc[i][j][v] : acc[i][j][v + 1], 16);
          const long m = mi + 8 * (v / 4) + v % 4 + up;
          if (m < M && (chosen >> (v + up) & 1)) C[m * ldc + n / 2 + frow % 16] = silu_mul(up ? other : own, up ? own : other);
        }
      }
    }
    return;
  }
  const bool pieces = gridDim.y > 1;
  float* out = pieces ? part + (long)blockIdx.y * M * N : C;
  const long ld = pieces ? N : ldc;
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const long n = n_wave + j * 32 + frow;
    if (n >= N) continue;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
      const long mi = m_wave + i * 32 + 4 * (lane / 32);
      float sum[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) sum[v] = acc[i][j][v];
      if (EPI == EPI_ADD && !pieces) {           // asked for together: one wait for memory, not sixteen
        float old[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) old[v] = out[min(mi + 8 * (v / 4) + v % 4, (long)M - 1) * ld + n];
#pragma unroll
        for (int v = 0; v < 16; ++v) sum[v] = old[v] + sum[v];
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const long m = mi + 8 * (v / 4) + v % 4;
        if (m < M && (chosen >> v & 1)) out[m * ld + n] = sum[v];
      }
    }
  }
}

// Few tiles: 64 x 64, four waves in 2 x 2, slabs of 32 floats of k that go from memory straight into LDS through a ring of four
// buffers (rows of 128 bytes, their 16-byte pieces turned by (row / 2) % 8 as in gemm_mfma.hip).  A block
// of these starts and steps faster than one of gemm_float32_parts_kernel: 0.6 us per 32 floats of k alone on its unit, where 64 x 64
// in parts take 0.9 (a chain of conversion, store, barrier and six products on one accumulator).
template <int EPI>
__global__ __launch_bounds__(256) void gemm_float32_tile_kernel(float* __restrict__ C, long ldc, const float* __restrict__ A, long lda,
                                                                const float* __restrict__ W, long ldw, int M, int N, int K, int tiles_n,
                                                                int k_per_split, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  constexpr int TM = FEW_TILES_ROWS, TN = FEW_TILES_ROWS, NB = FEW_TILES_BUFFERS;
  constexpr int ROW = 64;                        // a row of a slab: 128 bytes, in units of two
  constexpr int AI = TM / 32, WI = TN / 32;      // load instructions of a wave per slab: eight rows each
  constexpr int WM = TM / 64, WN = TN / 64;      // a wave's 32 x 32 tiles
  uint16_t* As = lds;                            // [NB][TM][ROW]
  uint16_t* Ws = lds + NB * TM * ROW;            // [NB][TN][ROW]
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 2, wn = wave % 2;
  const int k_lo = 2 * (int)blockIdx.y * k_per_split, k_hi = 2 * min(K, (int)(blockIdx.y + 1) * k_per_split);
  const TilePlace place_of = tile_place(tiles_n);
  const long m0 = (long)place_of.m * TM, n0 = (long)place_of.n * TN;
  const int a_rows = (int)min((long)TM, M - m0), w_rows = (int)min((long)TN, N - n0);
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t a_src = operand_descriptor(reinterpret_cast<const bf16_t*>(A), addressing::tile_descriptor(m0, 2 * lda, k_lo, k_hi, a_rows));
  const __amdgpu_buffer_rsrc_t w_src = operand_descriptor(reinterpret_cast<const bf16_t*>(W), addressing::tile_descriptor(n0, 2 * ldw, k_lo, k_hi, w_rows));
#endif
  unsigned a_off[AI], w_off[WI];
  int a_piece[AI], w_piece[WI];
#pragma unroll
  for (int p = 0; p < AI; ++p) {
    const int row = (wave * AI + p) * 8 + lane / 8;
    a_piece[p] = addressing::tile_piece(lane, row);
    a_off[p] = addressing::tile_lane_offset(row, a_rows, 2 * lda, a_piece[p]);
  }
#pragma unroll
  for (int p = 0; p < WI; ++p) {
    const int row = (wave * WI + p) * 8 + lane / 8;
    w_piece[p] = addressing::tile_piece(lane, row);
    w_off[p] = addressing::tile_lane_offset(row, w_rows, 2 * ldw, w_piece[p]);
  }
  auto load_slab = [&](int s, int buf) {         // beyond the range: offsets outside the descriptor, zeros nobody uses
#if defined(__HIP_DEVICE_COMPILE__)
    const int k = s * ROW;
#pragma unroll
    for (int p = 0; p < AI; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_src, (lds_ptr_t)(As + (buf * TM + (wave * AI + p) * 8) * ROW), 16,
                                               addressing::tile_slab_offset(a_off[p], k, a_piece[p], k_hi - k_lo), 0, 0, 0);
#pragma unroll
    for (int p = 0; p < WI; ++p)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_src, (lds_ptr_t)(Ws + (buf * TN + (wave * WI + p) * 8) * ROW), 16,
                                               addressing::tile_slab_offset(w_off[p], k, w_piece[p], k_hi - k_lo), 0, 0, 0);
#endif
  };

  f32x16_t acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  const int slabs = (k_hi - k_lo + ROW - 1) / ROW;
  const int frow = lane % 32;
  int place[4];                                  // where the four floats of this lane's k in every 8 lie in its rows
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) place[ks] = ((ks * 2 + lane / 32) ^ ((frow >> 1) & 7)) * 8;
#pragma unroll
  for (int s = 0; s < NB - 1; ++s) load_slab(s, s);
  int buf = 0;
  for (int s = 0; s < slabs; ++s) {
    // all but the slabs asked for after this one have landed: loads return in order
    constexpr int later = (NB - 2) * (AI + WI);
    block_barrier_keeping_loads<later>();        // ... for every wave, and everybody has left the buffer before this one
    load_slab(s + NB - 1, buf == 0 ? NB - 1 : buf - 1);
    const uint16_t* a_base = As + (buf * TM + wm * (TM / 2) + frow) * ROW;
    const uint16_t* w_base = Ws + (buf * TN + wn * (TN / 2) + frow) * ROW;
    f32x4_t fa[2][WM], fb[2][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i) fa[0][i] = *reinterpret_cast<const f32x4_t*>(a_base + i * 32 * ROW + place[0]);
#pragma unroll
    for (int j = 0; j < WN; ++j) fb[0][j] = *reinterpret_cast<const f32x4_t*>(w_base + j * 32 * ROW + place[0]);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) {                              // the next eight k are read while these run
#pragma unroll
        for (int i = 0; i < WM; ++i) fa[(ks + 1) & 1][i] = *reinterpret_cast<const f32x4_t*>(a_base + i * 32 * ROW + place[(ks + 1) & 3]);
#pragma unroll
        for (int j = 0; j < WN; ++j) fb[(ks + 1) & 1][j] = *reinterpret_cast<const f32x4_t*>(w_base + j * 32 * ROW + place[(ks + 1) & 3]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j) acc[i][j] = mfma32_f32(fa[ks & 1][i][e], fb[ks & 1][j][e], acc[i][j]);
      if (ks < 3) {                              // the reads go out behind the first of these products, not behind the last
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, WM + WN, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 4 * WM * WN - 1, 0);
      } else {
        __builtin_amdgcn_sched_group_barrier(0x008, 4 * WM * WN, 0);
      }
    }
    buf = buf == NB - 1 ? 0 : buf + 1;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);            // nothing may still be on its way into LDS when the block ends
  finish_tiles<WM, WN, EPI>(acc, m0 + wm * (TM / 2), n0 + wn * (TN / 2), C, ldc, M, N, part);
}

// Large tiles, in parts: a float is the sum of three bfloat16 (the bfloat16 nearest to it, the one nearest to what is left, and the
// rest, which fits), and six of the nine products of parts reach its last bit: lo . lo, lo . mid and mid . lo lie 2^-25 below the
// product and less.  Six bfloat16 instructions (exact products, 32-bit sums) take 6 x 32 cycles for the 32 x 32 x 16 that float32
// instructions need 8 x 64 for, and a sum has a sixteenth of the roundings per instruction: 1,293 x 2,048 outputs of k = 2,048 are off
// from 64 bits by 7.0e-7 of their norm here and by 8.1e-7 with float32 instructions, of k = 8,192 by 1.44e-6 and 1.62e-6.
//
// The parts are made once per block, on the way from memory into LDS: a thread fetches 16 bytes of a row a slab (16 floats of k) ahead,
// splits them (11 instructions per two floats, between the matrix instructions) and stores 8 bytes to each of three planes.  LDS holds
// two slabs of [32 rows][plane][half of k][row][8 k]: a fragment is 1 KB in lane order, the second half's rows turned by 4 so that
// four rows' stores fall on different banks.  Four waves in 2 x 2, two blocks per unit, one barrier per slab.
// Bound by the matrix cores and the chip's power: 2,048 x 16,384 x 2,048 takes 640 us (1.29 PFLOP/s of bfloat16 products at 1.8 GHz,
// the matrix cores 70 % busy, LDS 26 %, the vector unit 41 %) in tiles of 128 x 256, 996 with float32 instructions in 128 x 128;
// 1,293 x 16,384 x 2,048 450 us (729), 1,293 x 2,048 x 8,192 235 (371), 378 x 3,072 x 2,048 35 (49).  What orders the steps between
// the matrix instructions is worth 10 to 20 % in tiles of 192 x 128 (378 x 16,384 x 2,048 184 us as the compiler had them, 148 now).  Not
// kept: sched_group_barrier for that (one matrix instruction and four or six others in turn: up to 10 % slower), slabs fetched two to
// four ahead (2 % either way), tiles of 64 x 64 and 64 x 128 in parts.
//
// An infinity has no such parts (the rest would be NaN), neither has a float that rounds to one (above 3.39e38); a row whose largest
// float, within the block's k, is below 2^-100 loses its last parts (of a larger row's small floats 2^-134 each, less than its sums
// round off unless they meet zeros wherever the row is large); and the product of two leading parts may overflow where the floats' does
// not.  Outputs of such a row of A or W, and infinite ones, are made from memory with float32 instructions, 32 x 32 at a time, in the
// order of gemm_float32_tile_kernel; the others stay as they are, so that no row's bits hang on what its neighbours hold.  (One infinity
// in A, 2,048 x 16,384 x 2,048: 620 us become 1,080; 378 x 3,072 x 2,048: 41 and 94.  A NaN needs nothing: its row or column is NaN
// either way.)
// Four floats on their way into parts, in steps of some five instructions each: step 2 q + i makes part q of floats 2 i and 2 i + 1.
struct PartsOf4 {
  float r[4];
  uint32_t part[3][2];
  __device__ inline void begin(const f32x4_t x, float& top) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = x[e];
    // fmaxf would quiet NaNs in an instruction of its own
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(r[0]), "v"(r[1]));
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(r[2]), "v"(r[3]));
  }
  __device__ inline void step(const int u) {
    const int q = u / 2, i = u % 2;
    part[q][i] = pack_bf16x2(r[2 * i], r[2 * i + 1]);
    if (q < 2) {
      r[2 * i] -= __uint_as_float(part[q][i] << 16);
      r[2 * i + 1] -= __uint_as_float(part[q][i] & 0xffff0000u);
    }
  }
};

constexpr float PARTS_LARGEST = 3.3895313892515355e38f, PARTS_SMALLEST = 0x1p-100f, PARTS_OVERFLOW = 0x1p48f;      // K < 2^29: sums of smaller floats stay below 2^126

template <int WM, int WN, int EPI>
__global__ __launch_bounds__(256, 2) void gemm_float32_parts_kernel(float* __restrict__ C, long ldc, const float* __restrict__ A, long lda,
                                                                    const float* __restrict__ W, long ldw, int M, int N, int K, int tiles_n,
                                                                    int k_per_split, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  constexpr int TM = WM * 64, TN = WN * 64, LOADS = WM + WN;   // a load covers 64 rows
  constexpr int PLANE = 512, GROUP = 3 * PLANE, BUF = (TM + TN) / 32 * GROUP;
  constexpr int JP = WN == 4 ? 2 : 1;                          // columns of tiles whose products alternate (128 x 256: 670 -> 637 us)
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 2, wn = wave % 2;
  const int k_lo = 2 * (int)blockIdx.y * k_per_split, k_hi = 2 * min(K, (int)(blockIdx.y + 1) * k_per_split), k_range = k_hi - k_lo;
  const TilePlace tile = tile_place(tiles_n);
  const long m0 = (long)tile.m * TM, n0 = (long)tile.n * TN;
  const int a_rows = (int)min((long)TM, M - m0), w_rows = (int)min((long)TN, N - n0);
#if defined(__HIP_DEVICE_COMPILE__)
  const __amdgpu_buffer_rsrc_t a_src = operand_descriptor(reinterpret_cast<const bf16_t*>(A), addressing::tile_descriptor(m0, 2 * lda, k_lo, k_hi, a_rows));
  const __amdgpu_buffer_rsrc_t w_src = operand_descriptor(reinterpret_cast<const bf16_t*>(W), addressing::tile_descriptor(n0, 2 * ldw, k_lo, k_hi, w_rows));
#endif
  const int piece = addressing::parts_piece(tid);
  unsigned offset[LOADS];
  int store[LOADS];
#pragma unroll
  for (int p = 0; p < LOADS; ++p) {
    const bool of_a = p < WM;
    const int row = addressing::parts_row(of_a ? p : p - WM, tid), among = p * 64 + tid / 4;
    offset[p] = of_a ? addressing::tile_lane_offset(row, a_rows, 2 * lda, piece) : addressing::tile_lane_offset(row, w_rows, 2 * ldw, piece);
    store[p] = among / 32 * GROUP + (piece / 2 * 32 + (among % 32 ^ piece / 2 * 4)) * 8 + piece % 2 * 4;
  }
  u32x4_t got[LOADS];
  auto fetch = [&](const int p, const int s) {   // beyond the range: zeros
#if defined(__HIP_DEVICE_COMPILE__)
    got[p] = __builtin_amdgcn_raw_buffer_load_b128(p < WM ? a_src : w_src, addressing::tile_slab_offset(offset[p], s * addressing::PARTS_SLAB, piece, k_range), 0, 0);
#endif
  };
  float top[LOADS];                              // of this thread's quarter of a row per load
#pragma unroll
  for (int p = 0; p < LOADS; ++p) top[p] = 0.f;
  PartsOf4 four;
  auto put = [&](const int p, const int u, const int buf) {      // step u of load p
    if (u == 0) four.begin(__builtin_bit_cast(f32x4_t, got[p]), top[p]);
    four.step(u);
    if (u < 5) return;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(lds + buf + store[p] + q * PLANE) = make_uint2(four.part[q][0], four.part[q][1]);
  };

  f32x16_t acc[WM][WN];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  };
  clear();
  const int slabs = (k_range + addressing::PARTS_SLAB - 1) / addressing::PARTS_SLAB;
  const int frag = (lane ^ lane / 32 * 4) * 8;
  const uint16_t* a_base = lds + wm * WM * GROUP + frag;
  const uint16_t* w_base = lds + (2 * WM + wn * WN) * GROUP + frag;
#pragma unroll
  for (int p = 0; p < LOADS; ++p) fetch(p, 0);
#pragma unroll
  for (int p = 0; p < LOADS; ++p) {
#pragma unroll
    for (int u = 0; u < 6; ++u) put(p, u, 0);
    fetch(p, 1);
  }
  int buf = 0;
  for (int s = 0; s < slabs; ++s) {
    __builtin_amdgcn_sched_barrier(0);
    block_barrier_keeping_loads<63>();           // slab s is there, and everybody has left the other buffer
    __builtin_amdgcn_sched_barrier(0);
    Frag fa[WM][3], fb[2][JP][3];
    auto read_w = [&](const int j) {
#pragma unroll
      for (int jj = 0; jj < JP; ++jj)
#pragma unroll
        for (int q = 0; q < 3; ++q) fb[j / JP & 1][jj][q].q = *reinterpret_cast<const uint4*>(w_base + buf + (j + jj) * GROUP + q * PLANE);
    };
    read_w(0);
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int q = 0; q < 3; ++q) fa[i][q].q = *reinterpret_cast<const uint4*>(a_base + buf + i * GROUP + q * PLANE);
#pragma unroll
    for (int j = 0; j < WN; j += JP) {
      if (j + JP < WN) read_w(j + JP);
      constexpr int of_a[6] = {2, 0, 1, 1, 0, 0}, of_w[6] = {0, 2, 1, 0, 1, 0};      // the smallest terms first
#pragma unroll
      for (int n = 0; n < 6 * WM * JP; ++n) {
        const int t = n / (WM * JP), i = n / JP % WM, jj = n % JP, at = j * 6 * WM + n;
        acc[i][j + jj] = mfma32(fa[i][of_a[t]], fb[j / JP & 1][jj][of_w[t]], acc[i][j + jj]);
#pragma unroll
        for (int u = at * 6 * LOADS / (6 * WM * WN); u < (at + 1) * 6 * LOADS / (6 * WM * WN); ++u) {
          put(u / 6, u % 6, BUF - buf);
          if (u % 6 == 5) fetch(u / 6, s + 2);
        }
        __builtin_amdgcn_sched_barrier(0x104);   // nothing but fragment reads and scalar work moves across: left alone, the compiler bunches the steps
      }
    }
    buf = BUF - buf;
  }

  block_barrier_keeping_loads<0>();              // everybody is done with LDS
  int* met = reinterpret_cast<int*>(lds);        // whether an element may have to be made again; then, per row of A and W, whether it has no parts
  if (tid == 0) *met = 0;
  __syncthreads();
  bool odd = false;                              // whether this thread knows of a row without parts, or of one with which a sum may overflow
#pragma unroll
  for (int p = 0; p < LOADS; ++p) {
    const float t = fmaxf(top[p], dpp_move<0xB1>(top[p])), of_row = fmaxf(t, dpp_move<0x4E>(t));      // four lanes to a row
    const bool none = !(of_row <= PARTS_LARGEST) || (of_row > 0.f && of_row < PARTS_SMALLEST);
    if (piece == 0) met[1 + p * 64 + tid / 4] = none;
    odd = odd || none || of_row >= PARTS_OVERFLOW;
  }
  if (__any(odd) && lane == 0) atomicOr(met, 1);
  __syncthreads();
  const long m_wave = m0 + wm * (TM / 2), n_wave = n0 + wn * (TN / 2);
  const bool remake = __builtin_amdgcn_readfirstlane(*met) != 0;
  static_assert((1 + TM + TN) * 4 <= 2048 && 2048 + 4 * WM * WN * 256 <= 4 * BUF, "rows without parts and elements to be made again, in LDS");
  unsigned* again = reinterpret_cast<unsigned*>(lds + 1024) + wave * WM * WN * 64 + lane;      // [wave][i][j][lane]: a bit per element
  if (remake) {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const bool column = met[1 + TM + wn * (TN / 2) + j * 32 + lane % 32];
        unsigned bits = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const bool row = met[1 + wm * (TM / 2) + i * 32 + 8 * (v / 4) + 4 * (lane / 32) + v % 4];
          const bool one = row || column || fabsf(acc[i][j][v]) == INFINITY;
          bits |= (unsigned)one << v;
          acc[i][j][v] = one ? -0.f : acc[i][j][v];              // added to C it leaves C as it is, stored it is overwritten below
        }
        if (EPI == EPI_SWIGLU) bits |= __shfl_xor(bits, 16);     // gate and up of a feature
        again[(i * WN + j) * 64] = bits;
      }
  }
  finish_tiles<WM, WN, EPI>(acc, m_wave, n_wave, C, ldc, M, N, part);
  if (!remake) return;
#pragma unroll 1
  for (int t = 0; t < WM * WN; ++t) {            // a thread's elements are those that it has just written
    const unsigned bits = again[t * 64];
    if (!__any(bits != 0)) continue;
    const long m_tile = m_wave + t / WN * 32, n_tile = n_wave + t % WN * 32;
    const float* a_row = A + min(m_tile + lane % 32, (long)M - 1) * lda;
    const float* w_row = W + min(n_tile + lane % 32, (long)N - 1) * ldw;
    f32x16_t made[1][1];
#pragma unroll
    for (int v = 0; v < 16; ++v) made[0][0][v] = 0.f;
#pragma unroll 1
    for (int k = k_lo / 2; k < k_hi / 2; k += 8) {
      const int at = k + lane / 32 * 4;          // K is a multiple of 4: the upper lanes' may lie beyond it
      f32x4_t fa = {0.f, 0.f, 0.f, 0.f}, fb = fa;
      if (at < k_hi / 2) {
        fa = *reinterpret_cast<const f32x4_t*>(a_row + at);
        fb = *reinterpret_cast<const f32x4_t*>(w_row + at);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) made[0][0] = mfma32_f32(fa[e], fb[e], made[0][0]);
    }
    finish_tiles<1, 1, EPI>(made, m_tile, n_tile, C, ldc, M, N, part, bits);
  }
}

// ------------------------------------------------------------------ which kernel, which tile, how many pieces
struct Float32Plan {
  int tm, tn;            // 0: the weight-streaming kernel
  int splits, k_per_split;
};

static Float32Plan cut(int tm, int tn, int K, int splits) {
  const addressing::KSplit c = addressing::cut_k(K, splits, FSTEP);
  return Float32Plan{tm, tn, c.splits, c.k_per_block};
}

// Tiles: the shape and the number of pieces with the least time by a model fitted to 6,800 measurements (24 row counts of 33 to 2,900,
// thirteen matrices of 512 x 1,024 to 28,672 x 4,096, weights from memory): a block's start, the k that the busiest unit walks, two blocks
// of it side by side, and the result's way out.  The plan is 0.3 % above the best of these shapes and pieces in the mean, 5.6 % at worst.
// Float32 instructions (64 x 64) where the parts' larger tiles leave units idle: 64 rows by 2,048 x 8,192 26 us and 51 in tiles of 128 x
// 128; by 16,384 x 2,048 42 and 45; 100 rows by 16,384 x 2,048 75 and 49.  Pieces that a kernel adds (`after` 0) are written and read
// once at 4 TB/s, and that takes a launch; if the gated unit then is a kernel too (`after` 2), that as well (512 features, k = 512, 33 to
// 100 rows: 15.3 us whole, 12.4 in two pieces; 1,293 rows, 1,536 features, k = 2,048 163 and 115).
// `after` 1: the pieces are left to the kernel that reads the result anyway (a norm, a rotation).  They then cost their
// way through memory and no launch, and a matrix of few rows is streamed by two blocks per unit whatever its k: eight tokens and
// the norm, 2,048 x 2,048 12.4 -> 10.3 us, 3,072 x 2,048 13.1 -> 12.0; and some 2 us less for each product whose pieces a kernel
// added.  A short k in blocks of 16 rows that nearly are the units' number stays whole (24 tokens and the norm, 3,072 x 768 10.6 us
// and 14.6 in three pieces; 4,096 x 512 10.1 and 10.9).  More pieces have to promise a hundredth: 1,050 x 6,144 x 4,096
// and the norm takes 352 us whole and 386 in two, 500 x 6,144 x 4,096 180 in four and 184 in five, which the model holds for equal.  Most
// matrices that it holds for equal would gain by more pieces (1,950 x 3,072 x 2,048 169 and 159, 570 x 4,096 x 4,096 129 in three and 124 in
// five, 490 x 4,096 x 14,336 332 in four and 315 in eight; 63 x 5,120 x 3,072 30.5 and 30.4).
static Float32Plan plan(int M, int N, int K, long part_floats, int after) {
  const int units = compute_units();
  const bool read_by_next = after == 1;
  if (M <= ROWS_MAX_M) {
    // blocks of 32 rows want to be two per unit; a matrix of fewer rows whose k is long is cut over blocks, any other
    // gets its waves in blocks of 16 rows (launch_rows)
    const bool whole = read_by_next ? K <= ROWS_WHOLE_K && 4 * ceil_div(N, 16) >= 3 * units : K < ROWS_SPLIT_MIN_K;
    int splits = whole ? 1 : 2 * units / ceil_div(N, 32);
    while (splits > 1 && (K / splits < (read_by_next ? 256 : 512) || (long)splits * M * N > part_floats)) --splits;
    return cut(0, 0, K, splits < 1 ? 1 : splits);
  }
  static const struct { int tm, tn; float start, per_k, paired, out; } shapes[] = {      // us, us per k of one block, share of that where two blocks go side by side, us per MB
      {FEW_TILES_ROWS, FEW_TILES_ROWS, 3.07f, 0.01937f, 0.871f, 0.236f}, {128, 128, 2.75f, 0.04363f, 0.790f, 0.267f}, {192, 128, 3.10f, 0.05737f, 0.838f, 0.301f}, {128, 256, 4.25f, 0.06864f, 0.889f, 0.326f}};
  Float32Plan best = {FEW_TILES_ROWS, FEW_TILES_ROWS, 1, K};
  float least = 0.f;
  const float megabytes = (float)M * N * 4e-6f;
  for (const auto& s : shapes) {
    const long tiles = (long)ceil_div(M, s.tm) * ceil_div(N, s.tn);
    for (int splits = 1; splits <= 8; ++splits) {
      const Float32Plan p = cut(s.tm, s.tn, K, splits);
      if (splits > 1 && (p.splits != splits || p.k_per_split < 256 || (long)splits * M * N > part_floats)) continue;
      const long rounds = (tiles * p.splits + units - 1) / units;
      float us = s.start + (rounds % 2 + (rounds - rounds % 2) * s.paired) * s.per_k * p.k_per_split + s.out * p.splits * megabytes;
      if (p.splits > 1) us += read_by_next ? 1.f + 1.5f * p.splits * megabytes / 4.f : 2.5f + 2.f * p.splits * megabytes / 4.f;
      if (p.splits > 1 && after == 2) us += 1.f + 1.5f * megabytes / 4.f;
      if (least == 0.f || us < (read_by_next && p.splits > best.splits ? 0.99f : 1.f) * least) { least = us; best = p; }
    }
  }
  return best;
}

// Pieces that pi_gemm_float32 makes of this product when it may leave pieces in `part_floats` floats: 1 if it writes C.  `after`: what
// becomes of pieces, see plan().
extern "C" int pi_gemm_float32_pieces(int M, int N, int K, long part_floats, int after) {
  return M > 0 && N > 0 && K > 0 ? plan(M, N, K, part_floats, after).splits : 1;
}

template <int EPI>
static int launch_few_tiles(float* C, long ldc, const float* A, long lda, const float* W, long ldw, int M, int N, int K, const Float32Plan& p, float* part,
                           hipStream_t stream) {
  constexpr size_t bytes = (size_t)FEW_TILES_BUFFERS * 2 * FEW_TILES_ROWS * 128;
  static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_float32_tile_kernel<EPI>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (configured != hipSuccess) return pi_fail("gemm_float32: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(configured));
  const int tiles_n = ceil_div(N, FEW_TILES_ROWS);
  hipLaunchKernelGGL((gemm_float32_tile_kernel<EPI>), dim3((unsigned)(ceil_div(M, FEW_TILES_ROWS) * (long)tiles_n), p.splits), dim3(256), bytes, stream, C, ldc,
                     A, lda, W, ldw, M, N, K, tiles_n, p.k_per_split, part);
  return pi_check_launch("gemm_float32 (tiles)");
}

template <int WM, int WN, int EPI>
static int launch_parts(float* C, long ldc, const float* A, long lda, const float* W, long ldw, int M, int N, int K, const Float32Plan& p, float* part,
                        hipStream_t stream) {
  constexpr size_t bytes = (size_t)2 * (WM + WN) * 2 * 3072;
  static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_float32_parts_kernel<WM, WN, EPI>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (configured != hipSuccess) return pi_fail("gemm_float32: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(configured));
  const int tiles_n = ceil_div(N, WN * 64);
  hipLaunchKernelGGL((gemm_float32_parts_kernel<WM, WN, EPI>), dim3((unsigned)(ceil_div(M, WM * 64) * (long)tiles_n), p.splits), dim3(256), bytes, stream,
                     C, ldc, A, lda, W, ldw, M, N, K, tiles_n, p.k_per_split, part);
  return pi_check_launch("gemm_float32 (tiles in parts)");
}

template <int EPI>
static int launch_tiles(float* C, long ldc, const float* A, long lda, const float* W, long ldw, int M, int N, int K, const Float32Plan& p, float* part,
                        hipStream_t stream) {
  if (p.tm == FEW_TILES_ROWS) return launch_few_tiles<EPI>(C, ldc, A, lda, W, ldw, M, N, K, p, part, stream);
  if (p.tm == 192) return launch_parts<3, 2, EPI>(C, ldc, A, lda, W, ldw, M, N, K, p, part, stream);
  if (p.tn == 256 && ldw <= PARTS_WIDE_MAX_STRIDE) return launch_parts<2, 4, EPI>(C, ldc, A, lda, W, ldw, M, N, K, p, part, stream);
  return launch_parts<2, 2, EPI>(C, ldc, A, lda, W, ldw, M, N, K, p, part, stream);
}

// Enough waves for the memory whatever the matrix' rows are: blocks of four waves on 32 rows where that gives two per
// unit, also by cutting k; else blocks of 16 rows with 8 or 16 waves.  Eight tokens, N x K: 16384 x 2048 25.8 us
// (5.2 TB/s; 35.6 before, on the vector unit), 128256 x 2048 181 us (5.8 TB/s; 197), 3072 x 2048 12.5 us and
// 2048 x 2048 10.7 us with 16 waves, 2048 x 8192 17.1 us in eight pieces and 4 to add them (with 16 waves instead: 25).
template <int MB, int EPI>
static int launch_rows(float* C, long ldc, const float* A, long lda, const float* W, long ldw, int M, int N, int K, const Float32Plan& p, float* part,
                       hipStream_t stream) {
#define ROWS_GO(RT, WAVES, DEPTH)                                                                                                              \
  hipLaunchKernelGGL((gemm_float32_rows_kernel<MB, RT, WAVES, DEPTH, EPI>), dim3(ceil_div(N, RT * 16), p.splits), dim3(WAVES * 64), 0, stream, C, ldc, \
                     A, lda, W, ldw, M, N, K, p.k_per_split, part)
  const int units = compute_units();
  if (p.splits > 1 || N >= 2 * units * 24) ROWS_GO(2, 4, 1);
  else if constexpr (EPI == EPI_SWIGLU) ROWS_GO(2, 8, 2);
  else if (MB == 1 && N <= units * 16) ROWS_GO(1, (MB == 1 ? 16 : 8), 2);     // sixteen waves have registers for 16 tokens only
  else ROWS_GO(1, 8, 2);
#undef ROWS_GO
  return pi_check_launch("gemm_float32 (few rows)");
}

template <int EPI>
static int launch_float32(float* C, long ldc, const float* A, long lda, const float* W, long ldw, int M, int N, int K, const Float32Plan& p, float* part,
                          hipStream_t stream) {
  if (p.tm) return launch_tiles<EPI>(C, ldc, A, lda, W, ldw, M, N, K, p, part, stream);
  return M <= 16 ? launch_rows<1, EPI>(C, ldc, A, lda, W, ldw, M, N, K, p, part, stream) : launch_rows<2, EPI>(C, ldc, A, lda, W, ldw, M, N, K, p, part, stream);
}

static int check_float32(int M, int N, int K, const void* A, long lda, const void* W, long ldw, long ldc, int cols) {
  PI_REQUIRE(M > 0 && N > 0 && K > 0 && K < (1 << 29), "gemm_float32: bad sizes M=%d N=%d K=%d", M, N, K);
  PI_REQUIRE(lda >= K && ldw >= K && ldc >= cols, "gemm_float32: row strides (%ld, %ld, %ld) smaller than the rows (K=%d, %d columns)", lda, ldw, ldc, K, cols);
  PI_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0, "gemm_float32: K (%d) and row strides (%ld, %ld) must be multiples of 4", K, lda, ldw);
  PI_REQUIRE(128 * lda < (1L << 28) && 128 * ldw < (1L << 28), "gemm_float32: row strides (%ld, %ld) are too long for 32-bit offsets inside a tile", lda, ldw);
  PI_REQUIRE((uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0, "gemm_float32: operands must be 16-byte aligned");
  PI_REQUIRE((long)ceil_div(M, 64) * ceil_div(N, 64) < 2147483647L, "gemm_float32: too many tiles");
  return 0;
}

// C (+)= A . W^T.  `part` (may be null): float32 [part_floats] for the pieces of a product whose k is cut; when
// pi_gemm_float32_pieces says more than one, the pieces [splits, M, N] are all that is written and C is not touched.
extern "C" int pi_gemm_float32(void* C, long ldc, const void* A, long lda, const void* W, long ldw, int M, int N, int K, int accumulate,
                               void* part, long part_floats, int read_by_next, hipStream_t stream) {
  if (check_float32(M, N, K, A, lda, W, ldw, ldc, N)) return -1;
  const Float32Plan p = plan(M, N, K, part ? part_floats : 0, read_by_next != 0);
  PI_REQUIRE(p.splits == 1 || (part && part_floats >= (long)p.splits * M * N), "gemm_float32: workspace too small (%ld floats for %ld)", part_floats, (long)p.splits * M * N);
  return accumulate ? launch_float32<EPI_ADD>((float*)C, ldc, (const float*)A, lda, (const float*)W, ldw, M, N, K, p, (float*)part, stream)
                    : launch_float32<EPI_STORE>((float*)C, ldc, (const float*)A, lda, (const float*)W, ldw, M, N, K, p, (float*)part, stream);
}

// C [M, N / 2] = silu(gate) * up of the product's columns, gate and up rows interleaved in blocks of 16 in W.
extern "C" int pi_gemm_float32_swiglu(void* C, long ldc, const void* A, long lda, const void* W, long ldw, int M, int N, int K, hipStream_t stream) {
  if (check_float32(M, N, K, A, lda, W, ldw, ldc, N / 2)) return -1;
  PI_REQUIRE(N % 32 == 0, "gemm_float32: the gated epilogue needs N (%d) to be a multiple of 32", N);
  return launch_float32<EPI_SWIGLU>((float*)C, ldc, (const float*)A, lda, (const float*)W, ldw, M, N, K, plan(M, N, K, 0, 0), nullptr, stream);
}

// ------------------------------------------------------------------ adding pieces
// C[m][n] (op)= sum over splits of part[s][m][n], in split order: store bfloat16 (0), store float32 (1), add into float32 (2).
// Bound by latency and, with many rows, by memory: a thread takes V neighbouring columns (four where 16-byte accesses are
// allowed) and has eight pieces in flight (one column and one piece at a time before: 2,048 tokens by 2,048 columns added into
// float32 14.9 -> 11.5 us, 12 tokens 3.7 -> 1.8).
template <int EPI, int V>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(void* __restrict__ Cv, long ldc, const float* __restrict__ part, int splits, int M, int N) {
  typedef float vec_t __attribute__((ext_vector_type(V)));
  const int n = (blockIdx.x * blockDim.x + threadIdx.x) * V;
  if (n >= N) return;
  for (long m = blockIdx.y; m < M; m += gridDim.y) {
    const float* p = part + m * N + n;
    vec_t old = 0.f, sum = 0.f;
    if (EPI == 2) old = *reinterpret_cast<const vec_t*>((const float*)Cv + m * ldc + n);
    for (int s0 = 0; s0 < splits; s0 += 8) {
      vec_t v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (s0 + u < splits) v[u] = *reinterpret_cast<const vec_t*>(p + (long)(s0 + u) * M * N);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (s0 + u < splits) sum += v[u];
    }
    if (EPI == 0) {
#pragma unroll
      for (int i = 0; i < V; ++i) reinterpret_cast<bf16_t*>(Cv)[m * ldc + n + i] = from_float<bf16_t>(sum[i]);
    } else {
      *reinterpret_cast<vec_t*>((float*)Cv + m * ldc + n) = EPI == 2 ? old + sum : sum;
    }
  }
}

template <int V>
static int launch_reduce(void* C, int epilogue, long ldc, const float* part, int splits, int M, int N, hipStream_t stream) {
  const int across = (N + V - 1) / V, threads = across < 256 ? (across + 63) / 64 * 64 : 256;
  const dim3 grid((across + threads - 1) / threads, M < 65535 ? M : 65535), block(threads);
  switch (epilogue) {
    case 0: hipLaunchKernelGGL((splitk_reduce_kernel<0, V>), grid, block, 0, stream, C, ldc, part, splits, M, N); break;
    case 1: hipLaunchKernelGGL((splitk_reduce_kernel<1, V>), grid, block, 0, stream, C, ldc, part, splits, M, N); break;
    case 2: hipLaunchKernelGGL((splitk_reduce_kernel<2, V>), grid, block, 0, stream, C, ldc, part, splits, M, N); break;
    default: return pi_fail("splitk_reduce: unknown epilogue %d", epilogue);
  }
  return pi_check_launch("splitk_reduce");
}

extern "C" int pi_splitk_reduce(void* C, int epilogue, long ldc, const void* part, int splits, int M, int N, hipStream_t stream) {
  PI_REQUIRE(M > 0 && N > 0 && splits >= 1 && part, "splitk_reduce: bad arguments M=%d N=%d splits=%d", M, N, splits);
  const bool wide = N % 4 == 0 && (uintptr_t)part % 16 == 0 && (epilogue == 0 || (ldc % 4 == 0 && (uintptr_t)C % 16 == 0));
  return wide ? launch_reduce<4>(C, epilogue, ldc, (const float*)part, splits, M, N, stream)
              : launch_reduce<1>(C, epilogue, ldc, (const float*)part, splits, M, N, stream);
}
