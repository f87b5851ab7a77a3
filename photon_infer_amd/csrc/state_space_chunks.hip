// The state-space recurrence of prompt portions, a chunk of 64 tokens at a time on the matrix cores, 32-bit throughout
// (recurrent.hip holds the definition and the walk, which requests with fewer tokens in the step keep, also beside longer ones).  With la_t = -exp(A_log)
// dt_t and g_t its sum from the chunk's start,
//   y_t = exp(g_t) S_0^T C_t + sum_{u <= t} exp(g_t - g_u) dt_u (C_t . B_u) x_u + D x_t
//   S_64 = exp(g_64) S_0 + sum_u exp(g_64 - g_u) dt_u B_u x_u^T
// so that only the states hang together from chunk to chunk:
//   1. chunk_states_kernel: every chunk's own share of its last state, all chunks at once;
//   2. chunk_carry_kernel: the states at the chunks' starts, element by element through a request's chunks, from and into
//      its state row;
//   3. chunk_outputs_kernel: every chunk's outputs, all at once, like attention without a softmax.
// All exponents are <= 0.  g is summed in 64 bits and kept as a pair of floats: its differences are what counts, and of two
// large sums rounded to one float each little would be left (the walk multiplies decays one by one).
//
// The walk is a serial chain of a multiply-add and a 16-lane sum per token: 380 us for 2,048 tokens, 32 heads of 64 with a
// state of 128, which leaves half the chip idle.  In chunks 90 us (30, 13 and 47).
#include "mfma.h"
#include "token_tiles.h"

#define CHUNK 64
// A token's log decay from here on is complete forgetting: exp() of it, and of its sum with any other, is zero in 32 bits.  Taken
// for what it is, a decay of -1e12 left the sums that follow it without the digits of theirs, one beyond 3.4e38 left NaN.
#define LOG_DECAY_ALL (-200.0)
#define XROW (CHUNK / 4 + 1)          // 16-byte pieces of a row of tokens in LDS: an odd number, rows fall on all banks

__device__ inline float softplus_of(float v) { return v > 20.0f ? v : log1pf(expf(v)); }

// The chunk's step sizes and its running sums of log decays, lane = token, zero steps from `tokens` on.
struct ChunkDecay {
  float dt, hi, lo;     // this lane's step; g up to and with it as hi + lo
  float total;          // exp(g) of the whole chunk
};
__device__ inline ChunkDecay chunk_decay(const float* __restrict__ dt_raw, long dt_stride, float bias, float a_log, int tokens) {
  const int lane = threadIdx.x % PI_WAVE;
  const float dt = lane < tokens ? softplus_of(dt_raw[lane * dt_stride] + bias) : 0.f;
  double g = lane < tokens ? -(double)expf(a_log) * (double)dt : 0.0;
  g = g < LOG_DECAY_ALL ? LOG_DECAY_ALL : g;     // NaN stays NaN
#pragma unroll
  for (int d = 1; d < PI_WAVE; d *= 2) {
    const double other = __shfl_up(g, d, PI_WAVE);
    if (lane >= d) g += other;
  }
  const float hi = (float)g;
  return ChunkDecay{dt, hi, (float)(g - (double)hi), expf((float)__shfl(g, PI_WAVE - 1, PI_WAVE))};
}

// rows of `floats` (a multiple of 4, at most 4 * WIDTH) of the chunk's tokens into LDS, transposed: dst[column][token],
// zeros for tokens and columns that are not there; each token's row times scale[token]
template <int WIDTH>
__device__ inline void stage_columns(float* dst, const float* __restrict__ src, long stride, int tokens, int floats, const float* scale, int* first_bad) {
  // a quarter wave takes 16 tokens and the wave four neighbouring pieces: the stores fall on all banks
  for (int idx = threadIdx.x; idx < CHUNK * WIDTH; idx += blockDim.x) {
    const int u = idx % 16 + idx / 64 % 4 * 16, c = (idx / 16 % 4 + idx / 256 * 4) * 4;
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    if (u < tokens && c < floats) v = *reinterpret_cast<const f32x4_t*>(src + u * stride + c);
    if (scale) v *= scale[u];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (first_bad && !(fabsf(v[e]) < INFINITY)) {        // see chunk_outputs_kernel
        atomicMin(first_bad + c + e, u);
        v[e] = 0.f;
      }
      dst[(c + e) * (XROW * 4) + u] = v[e];
    }
  }
}

// blockIdx: (chunk, head, slice of 64 value columns).  states [chunk][head][P][N], decays [chunk][head].
template <int N>
__global__ __launch_bounds__(256) void chunk_states_kernel(float* __restrict__ states, float* __restrict__ decays, const float* __restrict__ xbc,
                                                           long xbc_stride, const float* __restrict__ dt_raw, long dt_stride,
                                                           const float* __restrict__ dt_bias, const float* __restrict__ A_log,
                                                           const int* __restrict__ q_start, int R, int from, int H, int P, int G) {
  __shared__ f32x4_t xt[64 * XROW], bt[N * XROW];
  __shared__ float weight[CHUNK];
  const int h = blockIdx.y, p0 = blockIdx.z * 64, tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int lr = lane % 16, lg = lane / 16;
  const TokenTile at = find_token_tile(q_start, R, CHUNK, blockIdx.x, from);
  if (at.req < 0) return;
  const long t0 = q_start[at.req] + (long)at.tile * CHUNK;
  const int tokens = min(CHUNK, (int)(q_start[at.req + 1] - t0)), cols = min(64, P - p0);
  const ChunkDecay d = chunk_decay(dt_raw + t0 * dt_stride + h, dt_stride, dt_bias[h], A_log[h], tokens);
  const float end_hi = __shfl(d.hi, 63, 64), end_lo = __shfl(d.lo, 63, 64);
  if (wave == 0) weight[lane] = expf((end_hi - d.hi) + (end_lo - d.lo)) * d.dt;
  if (tid == 0 && p0 == 0) decays[(long)blockIdx.x * H + h] = d.total;
  const float* row = xbc + t0 * xbc_stride;
  stage_columns<N / 4>(reinterpret_cast<float*>(bt), row + (long)H * P + (long)(h / (H / G)) * N, xbc_stride, tokens, N, nullptr, nullptr);
  __syncthreads();
  stage_columns<16>(reinterpret_cast<float*>(xt), row + (long)h * P + p0, xbc_stride, tokens, cols, weight, nullptr);
  __syncthreads();
  float* out = states + ((long)blockIdx.x * H + h) * P * N;
  for (int nb = wave; nb < N / 16; nb += 4) {
    f32x4_t acc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < CHUNK / 16; ++k) {
      const f32x4_t y = bt[(nb * 16 + lr) * XROW + k * 4 + lg];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const f32x4_t x = xt[(b * 16 + lr) * XROW + k * 4 + lg];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b] = mfma16_f32(x[e], y[e], acc[b]);
      }
    }
    // acc[b][i]: value column b * 16 + lg * 4 + i, state row nb * 16 + lr
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = b * 16 + lg * 4 + i;
        if (p < cols) out[(long)(p0 + p) * N + nb * 16 + lr] = acc[b][i];
      }
  }
}

// A thread takes one element of a request's state through its chunks: states[chunk] becomes the state at the chunk's start.
// The state row is in the walk's order (recurrent.hip): [head][slice of four columns][i][lane], NR rows per lane.
__global__ __launch_bounds__(256) void chunk_carry_kernel(float* __restrict__ states, const float* __restrict__ decays, const int* __restrict__ q_start,
                                                          const int* __restrict__ slots, int from, float* __restrict__ state, long state_stride,
                                                          int H, int P, int N, int NR) {
  const int r = blockIdx.x, h = blockIdx.y, e = blockIdx.z * 256 + threadIdx.x;
  const int first = token_tiles_before(q_start, r, CHUNK, from), chunks = token_tiles(q_start[r + 1] - q_start[r], CHUNK, from);
  if (e >= P * N || chunks == 0) return;
  const int p = e / N, n = e % N, slices = (P + 15) / 16 * 4;
  float* mine = state + (long)slots[r] * state_stride + (((long)h * slices + p / 4) * NR + n % NR) * PI_WAVE + (p % 4) * 16 + n / NR;
  float s = *mine;
  float* at = states + ((long)first * H + h) * P * N + e;
  const float* decay = decays + (long)first * H + h;
  const long step = (long)H * P * N;
  int c = 0;
  for (; c + 8 <= chunks; c += 8) {
    float own[8], a[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) { own[j] = at[(c + j) * step]; a[j] = decay[(long)(c + j) * H]; }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      at[(c + j) * step] = s;
      s = fmaf(a[j], s, own[j]);
    }
  }
  for (; c < chunks; ++c) {
    const float own = at[c * step], a = decay[(long)c * H];
    at[c * step] = s;
    s = fmaf(a, s, own);
  }
  *mine = s;
}

// A wave takes 16 of the chunk's tokens as columns.  What a token's input weighs in the outputs before it is zero, and zero
// times an input that is not finite would not be: such inputs are taken as zero, and the outputs of their column from
// their token on are NaN, as a state that holds them is.
template <int N>
__global__ __launch_bounds__(256) void chunk_outputs_kernel(float* __restrict__ y, long y_stride, const float* __restrict__ states,
                                                            const float* __restrict__ xbc, long xbc_stride, const float* __restrict__ dt_raw,
                                                            long dt_stride, const float* __restrict__ dt_bias, const float* __restrict__ A_log,
                                                            const float* __restrict__ Dskip, const int* __restrict__ q_start, int R, int from, int H, int P, int G) {
  constexpr int NROW = N / 4 + 1, IT = 64 * (N / 4) / 256;
  __shared__ f32x4_t rows[64 * NROW];           // first the tokens' B, then the state at the chunk's start, a row per value column
  __shared__ f32x4_t xt[64 * XROW];
  __shared__ float hi[CHUNK], lo[CHUNK], step[CHUNK];
  __shared__ int first_bad[64];
  const int h = blockIdx.y, p0 = blockIdx.z * 64, tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int lr = lane % 16, lg = lane / 16;
  const TokenTile at = find_token_tile(q_start, R, CHUNK, blockIdx.x, from);
  if (at.req < 0) return;
  const long t0 = q_start[at.req] + (long)at.tile * CHUNK;
  const int tokens = min(CHUNK, (int)(q_start[at.req + 1] - t0)), cols = min(64, P - p0);
  const float* row = xbc + t0 * xbc_stride;
  const long b_col = (long)H * P + (long)(h / (H / G)) * N, c_col = b_col + (long)G * N;
  const int token = wave * 16 + lr;
  if (tid < 64) first_bad[tid] = CHUNK;
  // everything from memory is asked for before the first of it is needed
  f32x4_t b_in[IT], s_in[IT], c[N / 16];
  const float* own = states + (((long)blockIdx.x * H + h) * P + p0) * N;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int idx = tid + i * 256, u = idx / (N / 4), f = idx % (N / 4) * 4;
    b_in[i] = u < tokens ? *reinterpret_cast<const f32x4_t*>(row + u * xbc_stride + b_col + f) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    s_in[i] = u < cols ? *reinterpret_cast<const f32x4_t*>(own + (long)u * N + f) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int f = 0; f < N / 16; ++f) c[f] = *reinterpret_cast<const f32x4_t*>(row + min(token, tokens - 1) * xbc_stride + c_col + f * 16 + lg * 4);
  const ChunkDecay d = chunk_decay(dt_raw + t0 * dt_stride + h, dt_stride, dt_bias[h], A_log[h], tokens);
  if (wave == 0) { hi[lane] = d.hi; lo[lane] = d.lo; step[lane] = d.dt; }
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int idx = tid + i * 256;
    rows[idx / (N / 4) * NROW + idx % (N / 4)] = b_in[i];
  }
  __syncthreads();
  stage_columns<16>(reinterpret_cast<float*>(xt), row + (long)h * P + p0, xbc_stride, tokens, cols, nullptr, first_bad);
  __syncthreads();
  const float my_hi = hi[token], my_lo = lo[token];
  f32x4_t acc[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int kt = 0; kt <= wave; ++kt) {          // tokens after the wave's own sixteen weigh nothing
    f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < N / 16; ++f) {
      const f32x4_t b = rows[(kt * 16 + lr) * NROW + f * 4 + lg];
#pragma unroll
      for (int e = 0; e < 4; ++e) s = mfma16_f32(b[e], c[f][e], s);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int u = kt * 16 + lg * 4 + i;
      s[i] = u <= token ? s[i] * (expf((my_hi - hi[u]) + (my_lo - lo[u])) * step[u]) : 0.f;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const f32x4_t x = xt[(b * 16 + lr) * XROW + kt * 4 + lg];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[b] = mfma16_f32(x[e], s[e], acc[b]);
    }
  }
  __syncthreads();                              // the state takes the place of the tokens' B
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int idx = tid + i * 256;
    rows[idx / (N / 4) * NROW + idx % (N / 4)] = s_in[i];
  }
  __syncthreads();
  const float from_start = expf(my_hi + my_lo);
#pragma unroll
  for (int f = 0; f < N / 16; ++f) {
    const f32x4_t cf = c[f] * from_start;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const f32x4_t s = rows[(b * 16 + lr) * NROW + f * 4 + lg];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[b] = mfma16_f32(s[e], cf[e], acc[b]);
    }
  }
  // acc[b][i]: value column b * 16 + lg * 4 + i of this lane's token
  if (token >= tokens) return;
  const float skip = Dskip[h];
  const float* x = reinterpret_cast<const float*>(xt);
  float* out = y + (t0 + token) * y_stride + (long)h * P + p0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int p = b * 16 + lg * 4;
    if (p >= cols) continue;
    f32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = token >= first_bad[p + i] ? __builtin_nanf("") : fmaf(skip, x[(p + i) * (XROW * 4) + token], acc[b][i]);
    *reinterpret_cast<f32x4_t*>(out + p) = v;
  }
}

// Tokens of a chunk, for the caller's count of chunks (sum of ceil(tokens / this) over the requests that run in chunks), or
// 0: sizes that the chunked form does not take.
extern "C" int pi_state_space_chunk(int P, int N) { return P > 0 && P % 4 == 0 && (N == 16 || N == 32 || N == 64 || N == 128) ? CHUNK : 0; }

// The requests that bring `from` tokens or more.  `states`: float32 [chunks, H, P, N], `decays`: float32 [chunks, H], both
// scratch.  Arguments otherwise as for
// pi_state_space_scan; rows of x, B, C and y must be 16-byte aligned.
extern "C" int pi_state_space_chunks(float* y, long y_stride, const float* xbc, long xbc_stride, const float* dt_raw, long dt_stride,
                                     const float* dt_bias, const float* A_log, const float* Dskip, const int* q_start, const int* slots, int R,
                                     int from, int chunks, float* states, float* decays, float* state, long state_stride, int H, int P, int N, int G,
                                     hipStream_t stream) {
  PI_REQUIRE(H > 0 && H <= 65535 && P > 0 && N > 0 && G > 0 && H % G == 0, "state space: bad sizes heads=%d vdim=%d state=%d groups=%d", H, P, N, G);
  PI_REQUIRE(pi_state_space_chunk(P, N) > 0, "state space: no chunked form for heads of %d with a state of %d", P, N);
  int nr = 1;
  while (16 * nr < N) nr *= 2;
  PI_REQUIRE(R > 0 && from > 0 && chunks > 0 && states && decays && state_stride >= (long)H * ((P + 15) / 16) * 4 * nr * PI_WAVE,
             "state space: bad step (%d requests, %d chunks) or a state row of %ld floats that cannot hold %d x %d x %d", R, chunks, state_stride, H, N, P);
  PI_REQUIRE(xbc_stride % 4 == 0 && y_stride % 4 == 0 && (uintptr_t)xbc % 16 == 0 && (uintptr_t)y % 16 == 0 && (uintptr_t)states % 16 == 0,
             "state space: rows must be 16-byte aligned");
  const dim3 grid(chunks, H, (P + 63) / 64), carry(R, H, (P * N + 255) / 256), block(256);
#define GO(N_)                                                                                                                                   \
  case N_:                                                                                                                                       \
    hipLaunchKernelGGL((chunk_states_kernel<N_>), grid, block, 0, stream, states, decays, xbc, xbc_stride, dt_raw, dt_stride, dt_bias, A_log,    \
                       q_start, R, from, H, P, G);                                                                                               \
    hipLaunchKernelGGL(chunk_carry_kernel, carry, block, 0, stream, states, decays, q_start, slots, from, state, state_stride, H, P, N_, nr);    \
    hipLaunchKernelGGL((chunk_outputs_kernel<N_>), grid, block, 0, stream, y, y_stride, states, xbc, xbc_stride, dt_raw, dt_stride, dt_bias,     \
                       A_log, Dskip, q_start, R, from, H, P, G);                                                                                 \
    break
  switch (N) {
    GO(16); GO(32); GO(64); GO(128);
  }
#undef GO
  return pi_check_launch("state_space_chunks");
}
