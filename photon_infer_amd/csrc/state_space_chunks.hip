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
// state of 128, which leaves half the chip idle.  In chunks 75 us (26, 13 and 35).
#include "mfma.h"
#include "token_tiles.h"

#define CHUNK 64
// A token's log decay from here on is complete forgetting: exp() of it, and of its sum with any other, is zero in 32 bits.  Taken
// for what it is, a decay of -1e12 left the sums that follow it without the digits of theirs, one beyond 3.4e38 left NaN.
#define LOG_DECAY_ALL (-200.0)

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

// blockIdx: (chunk, head, slice of 64 value columns); behind the heads the groups, whose blocks make the products C_t . B_u that the
// group's heads share.  states [chunk][head][P][N], decays [chunk][head], scores [chunk][group][t][u], whole sixteens of u up to t's.
//
// Every operand goes from memory into the registers that the matrix instructions take it from, a step ahead of them, and no wave waits
// for another: the blocks of a step are few (four to a unit at 2,048 tokens of 32 heads), each a chain of trips to memory.
// Staged through LDS, transposed, piece after piece behind a barrier, 31 us, now 26 (2,048 tokens, 32 heads of 64, state of 128; matrix
// instructions alone 7, the states' 34 MB 6 to 8).
template <int N>
__global__ __launch_bounds__(256, 5) void chunk_states_kernel(float* __restrict__ states, float* __restrict__ decays, float* __restrict__ scores,
                                                           const float* __restrict__ xbc, long xbc_stride, const float* __restrict__ dt_raw,
                                                           long dt_stride, const float* __restrict__ dt_bias, const float* __restrict__ A_log,
                                                           const int* __restrict__ q_start, int R, int from, int H, int P, int G) {
  const int h = blockIdx.y, p0 = blockIdx.z * 64, tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int lr = lane % 16, lg = lane / 16;
  const TokenTile at = find_token_tile(q_start, R, CHUNK, blockIdx.x, from);
  if (at.req < 0) return;
  const long t0 = q_start[at.req] + (long)at.tile * CHUNK;
  const int tokens = min(CHUNK, (int)(q_start[at.req + 1] - t0)), last = tokens - 1;
  const float* row = xbc + t0 * xbc_stride;
  if (h >= H) {                                 // the wave's sixteen tokens against those up to them; rows beyond the last repeat it
    if (p0 > 0) return;
    const float* b_row = row + (long)H * P + (long)(h - H) * N + lg * 4;
    const float* c_row = b_row + (long)G * N + min(wave * 16 + lr, last) * xbc_stride;
    float* out = scores + (((long)blockIdx.x * G + (h - H)) * CHUNK + wave * 16 + lr) * CHUNK + lg * 4;
    f32x4_t c[N / 16];
#pragma unroll
    for (int f = 0; f < N / 16; ++f) c[f] = *reinterpret_cast<const f32x4_t*>(c_row + f * 16);
    for (int kt = 0; kt <= wave; ++kt) {
      f32x4_t b[N / 16], s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int f = 0; f < N / 16; ++f) b[f] = *reinterpret_cast<const f32x4_t*>(b_row + min(kt * 16 + lr, last) * xbc_stride + f * 16);
#pragma unroll
      for (int f = 0; f < N / 16; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) s = mfma16_f32(b[f][e], c[f][e], s);
      *reinterpret_cast<f32x4_t*>(out + kt * 16) = s;
    }
    return;
  }
  const int cols = min(64, P - p0);
  if (wave * 16 >= cols) return;
  const float* x_row = row + (long)h * P + p0 + min(wave * 16 + lr, cols - 1);
  const float* b_row = row + (long)H * P + (long)(h / (H / G)) * N + lr;
  // this lane's tokens are j / 4 * 16 + lg * 4 + j % 4, its value column wave * 16 + lr; one beyond the last repeats it and is not stored
  float x[CHUNK / 4], y[2][CHUNK / 4];
  auto fetch_y = [&](float (&to)[CHUNK / 4], int nb) {
#pragma unroll
    for (int j = 0; j < CHUNK / 4; ++j) to[j] = b_row[min(j / 4 * 16 + lg * 4 + j % 4, last) * xbc_stride + nb * 16];
  };
#pragma unroll
  for (int j = 0; j < CHUNK / 4; ++j) x[j] = x_row[min(j / 4 * 16 + lg * 4 + j % 4, last) * xbc_stride];
  fetch_y(y[0], 0);
  const ChunkDecay d = chunk_decay(dt_raw + t0 * dt_stride + h, dt_stride, dt_bias[h], A_log[h], tokens);
  const float end_hi = __shfl(d.hi, 63, 64), end_lo = __shfl(d.lo, 63, 64);
  const float weight = expf((end_hi - d.hi) + (end_lo - d.lo)) * d.dt;
  if (tid == 0 && p0 == 0) decays[(long)blockIdx.x * H + h] = d.total;
#pragma unroll
  for (int j = 0; j < CHUNK / 4; ++j) {
    const int u = j / 4 * 16 + lg * 4 + j % 4;
    x[j] *= __shfl(weight, u, 64);
    x[j] = u < tokens ? x[j] : 0.f;
  }
  float* out = states + ((long)blockIdx.x * H + h) * P * N + (long)(p0 + wave * 16 + lr) * N + lg * 4;
  const bool stored = wave * 16 + lr < cols;
#pragma unroll
  for (int nb = 0; nb < N / 16; ++nb) {
    if (nb + 1 < N / 16) fetch_y(y[(nb + 1) % 2], nb + 1);
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < CHUNK / 4; ++j) acc = mfma16_f32(j / 4 * 16 + lg * 4 + j % 4 < tokens ? y[nb % 2][j] : 0.f, x[j], acc);
    if (stored) *reinterpret_cast<f32x4_t*>(out + nb * 16) = acc;      // state rows nb * 16 + lg * 4 + i
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
// their token on are NaN, as a state that holds them is.  Operands as in chunk_states_kernel, each fetched a step of sixteen ahead;
// the products C_t . B_u, which each of 32 heads made for itself, are read.  47 us, now 35 (sizes as above).  A wave with 16 of the value
// columns and all tokens, its state fetched at once and the scores shared through LDS: 39.
template <int N>
__global__ __launch_bounds__(256, 4) void chunk_outputs_kernel(float* __restrict__ y, long y_stride, const float* __restrict__ states,
                                                            const float* __restrict__ scores, const float* __restrict__ xbc, long xbc_stride,
                                                            const float* __restrict__ dt_raw, long dt_stride, const float* __restrict__ dt_bias,
                                                            const float* __restrict__ A_log, const float* __restrict__ Dskip,
                                                            const int* __restrict__ q_start, int R, int from, int H, int P, int G) {
  const int h = blockIdx.y, p0 = blockIdx.z * 64, tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int lr = lane % 16, lg = lane / 16;
  const TokenTile at = find_token_tile(q_start, R, CHUNK, blockIdx.x, from);
  if (at.req < 0) return;
  const long t0 = q_start[at.req] + (long)at.tile * CHUNK;
  const int tokens = min(CHUNK, (int)(q_start[at.req + 1] - t0)), last = tokens - 1, cols = min(64, P - p0);
  if (wave * 16 >= tokens) return;
  const int g = h / (H / G), token = wave * 16 + lr;
  const float* row = xbc + t0 * xbc_stride;
  const float* x_row = row + (long)h * P + p0;
  const float* own = states + (((long)blockIdx.x * H + h) * P + p0) * N + lg * 4;
  const float* score_row = scores + (((long)blockIdx.x * G + g) * CHUNK + token) * CHUNK + lg * 4;
  const float* c_row = row + min(token, last) * xbc_stride + (long)H * P + (long)(G + g) * N + lg * 4;
  f32x4_t c, s_of, state[4];
  float x[4][4];
  auto fetch_x = [&](int kt) {                  // rows beyond the last repeat it, and so do columns
    s_of = *reinterpret_cast<const f32x4_t*>(score_row + kt * 16);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int b = 0; b < 4; ++b) x[b][e] = x_row[min(kt * 16 + lg * 4 + e, last) * xbc_stride + min(b * 16 + lr, cols - 1)];
  };
  auto fetch_state = [&](int f) {
    c = *reinterpret_cast<const f32x4_t*>(c_row + f * 16);
#pragma unroll
    for (int b = 0; b < 4; ++b) state[b] = *reinterpret_cast<const f32x4_t*>(own + (long)min(b * 16 + lr, cols - 1) * N + f * 16);
  };
  fetch_x(0);
  fetch_state(0);
  const ChunkDecay d = chunk_decay(dt_raw + t0 * dt_stride + h, dt_stride, dt_bias[h], A_log[h], tokens);
  const float my_hi = __shfl(d.hi, token, 64), my_lo = __shfl(d.lo, token, 64);
  f32x4_t acc[4];
  int bad[4];                                   // per value column of this lane: the first of its tokens whose input is not finite
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    bad[b] = CHUNK;
  }
#pragma unroll
  for (int kt = 0; kt < CHUNK / 16; ++kt) {
    if (kt > wave) break;                       // tokens after the wave's own sixteen weigh nothing
    float now[4][4];
    f32x4_t s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int u = kt * 16 + lg * 4 + i;
      const float u_hi = __shfl(d.hi, u, 64), u_lo = __shfl(d.lo, u, 64), u_dt = __shfl(d.dt, u, 64);
      s[i] = u <= token ? s_of[i] * (expf((my_hi - u_hi) + (my_lo - u_lo)) * u_dt) : 0.f;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const bool finite = fabsf(x[b][i]) < INFINITY;
        now[b][i] = finite && u < tokens ? x[b][i] : 0.f;
        bad[b] = finite || u >= tokens ? bad[b] : min(bad[b], u);
      }
    }
    if (kt < wave) fetch_x(kt + 1);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[b] = mfma16_f32(now[b][e], s[e], acc[b]);
  }
  const float from_start = expf(my_hi + my_lo);
#pragma unroll
  for (int f = 0; f < N / 16; ++f) {
    const f32x4_t cf = c * from_start;
    f32x4_t now[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) now[b] = state[b];
    if (f + 1 < N / 16) fetch_state(f + 1);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[b] = mfma16_f32(now[b][e], cf[e], acc[b]);
  }
  // acc[b][i]: value column b * 16 + lg * 4 + i of this lane's token
  if (__any(min(min(bad[0], bad[1]), min(bad[2], bad[3])) < CHUNK)) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      bad[b] = min(bad[b], __shfl_xor(bad[b], 16, 64));
      bad[b] = min(bad[b], __shfl_xor(bad[b], 32, 64));
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (token >= __shfl(bad[b], lg * 4 + i, 64)) acc[b][i] = __builtin_nanf("");
    }
  }
  if (token >= tokens) return;
  const float skip = Dskip[h];
  const float* own_x = x_row + token * xbc_stride;
  float* out = y + (t0 + token) * y_stride + (long)h * P + p0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int p = b * 16 + lg * 4;
    if (p >= cols) continue;
    const f32x4_t in = *reinterpret_cast<const f32x4_t*>(own_x + p);
    f32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = fmaf(skip, in[i], acc[b][i]);
    *reinterpret_cast<f32x4_t*>(out + p) = v;
  }
}

// Tokens of a chunk, for the caller's count of chunks (sum of ceil(tokens / this) over the requests that run in chunks), or
// 0: sizes that the chunked form does not take.
extern "C" int pi_state_space_chunk(int P, int N) { return P > 0 && P % 4 == 0 && (N == 16 || N == 32 || N == 64 || N == 128) ? CHUNK : 0; }

// The requests that bring `from` tokens or more.  `states`: float32 [chunks, H, P, N], `decays`: float32 [chunks, H], `scores`: float32
// [chunks, G, 64, 64], all scratch.  Arguments otherwise as for
// pi_state_space_scan; rows of x, B, C and y must be 16-byte aligned.
extern "C" int pi_state_space_chunks(float* y, long y_stride, const float* xbc, long xbc_stride, const float* dt_raw, long dt_stride,
                                     const float* dt_bias, const float* A_log, const float* Dskip, const int* q_start, const int* slots, int R,
                                     int from, int chunks, float* states, float* decays, float* scores, float* state, long state_stride, int H, int P, int N, int G,
                                     hipStream_t stream) {
  PI_REQUIRE(H > 0 && H + G <= 65535 && P > 0 && N > 0 && G > 0 && H % G == 0, "state space: bad sizes heads=%d vdim=%d state=%d groups=%d", H, P, N, G);
  PI_REQUIRE(pi_state_space_chunk(P, N) > 0, "state space: no chunked form for heads of %d with a state of %d", P, N);
  int nr = 1;
  while (16 * nr < N) nr *= 2;
  PI_REQUIRE(R > 0 && from > 0 && chunks > 0 && states && decays && scores && state_stride >= (long)H * ((P + 15) / 16) * 4 * nr * PI_WAVE,
             "state space: bad step (%d requests, %d chunks) or a state row of %ld floats that cannot hold %d x %d x %d", R, chunks, state_stride, H, N, P);
  PI_REQUIRE(xbc_stride % 4 == 0 && y_stride % 4 == 0 && (uintptr_t)xbc % 16 == 0 && (uintptr_t)y % 16 == 0 && (uintptr_t)states % 16 == 0 &&
                 (uintptr_t)scores % 16 == 0,
             "state space: rows must be 16-byte aligned");
  const dim3 grid(chunks, H, (P + 63) / 64), with_groups(chunks, H + G, (P + 63) / 64), carry(R, H, (P * N + 255) / 256), block(256);
#define GO(N_)                                                                                                                                   \
  case N_:                                                                                                                                       \
    hipLaunchKernelGGL((chunk_states_kernel<N_>), with_groups, block, 0, stream, states, decays, scores, xbc, xbc_stride, dt_raw, dt_stride,    \
                       dt_bias, A_log, q_start, R, from, H, P, G);                                                                                               \
    hipLaunchKernelGGL(chunk_carry_kernel, carry, block, 0, stream, states, decays, q_start, slots, from, state, state_stride, H, P, N_, nr);    \
    hipLaunchKernelGGL((chunk_outputs_kernel<N_>), grid, block, 0, stream, y, y_stride, states, scores, xbc, xbc_stride, dt_raw, dt_stride,      \
                       dt_bias, A_log, Dskip, q_start, R, from, H, P, G);                                                                                 \
    break
  switch (N) {
    GO(16); GO(32); GO(64); GO(128);
  }
#undef GO
  return pi_check_launch("state_space_chunks");
}
