// The gated delta rule of prompt portions, sixteen tokens at a time, 32-bit throughout (recurrent.hip holds the definition and the
// walk, which requests with fewer tokens in the step keep, also beside longer ones).  With g_t the decays of token t (per key
// channel, or one per head), L_t their product from the chunk's start up to and with t, and S_0 the state at the chunk's start,
//   u_t = beta_t (v_t - S_0^T (L_t k_t) - sum_{s < t} a_ts u_s),   a_ts = sum_c k_t[c] k_s[c] (g_{s+1} .. g_t)[c]
//   o_t = S_0^T (L_t q_t) + sum_{s <= t} p_ts u_s,                 p_ts = sum_c q_t[c] k_s[c] (g_{s+1} .. g_t)[c]
//   S_16 = L_15 S_0 + sum_s (g_{s+1} .. g_15) k_s u_s^T
// Products of decays are taken token after token, as the walk takes them, and never divided: a decay may be zero.  Solved for u,
// U = X - Y S_0 with (I + diag(beta) a) [X Y] = diag(beta) [V (L k)], so that only three small products per chunk wait for the state:
//   1. delta_chunk_prepare_kernel: unit vectors, decays, a, p, X, Y and the rest of every chunk, all chunks at once, in the order in
//      which the matrix cores take them;
//   2. delta_chunk_walk_kernel: U, outputs and states from chunk to chunk.
// Both take a window of the step's chunks at a time, as many as the caller's scratch memory holds.
//
// The walk of single tokens is a chain of some 500 cycles per token.  16 heads of 128 x 128, 2,048 tokens of one request: 446 us walked,
// 143 so (43 and 108 by themselves), eight requests of 375 tokens 414 and 146, 128 tokens 38 and 25, 48 tokens 20 and 19.  Against 64
// bits outputs and states are off by 1.4e-7 to 6e-7 of their norm either way.
#include "mfma.h"
#include "token_tiles.h"

#define CHUNK 16

__device__ inline float softplus_of(float v) { return v > 20.0f ? v : log1pf(expf(v)); }

// What a chunk of one head leaves for the walk, in floats; fragments are [tile of 16][lane][4].
struct ChunkShape {
  int y, q, k, x, p, decay, all;
};
__host__ __device__ inline ChunkShape chunk_shape(int d, int dv) {
  ChunkShape s;
  s.y = 0;
  s.q = 16 * d;
  s.k = 32 * d;
  s.x = 48 * d;
  s.p = s.x + 16 * dv;
  s.decay = s.p + 256;
  s.all = s.decay + d;
  return s;
}

// blockIdx: (chunk behind `first_chunk`, head).  DQ: d / 64.  Bound by issue: a thread's products over pairs of tokens and the sums over sixteen lanes (72 us
// while it kept all pairs in registers, for half the waves; 43 so).
template <int DQ>
__global__ __launch_bounds__(256, 4) void delta_chunk_prepare_kernel(float* __restrict__ scratch, const float* __restrict__ qkv, long qkv_stride,
                                                                  const float* __restrict__ a, long a_stride, const float* __restrict__ dt_bias,
                                                                  const float* __restrict__ A_log, const float* __restrict__ b, long b_stride,
                                                                  const int* __restrict__ q_start, int R, int from, int first_chunk, int H, int G, int dv,
                                                                  float q_scale, float unit_eps, int per_head) {
  constexpr int D = 64 * DQ, PADDED = D / 4 * 17 * 4;          // a fragment's four rows of lanes 17 pieces apart: their stores fall on all banks
  __shared__ f32x4_t vectors[3 * CHUNK * D / 4];               // q, k, decays; then Y and L q
  __shared__ __attribute__((aligned(16))) float pairs[2][CHUNK][CHUNK];
  __shared__ float betas[CHUNK];
  static_assert(2 * PADDED <= 3 * CHUNK * D, "Y and L q take the place of the vectors");
  const int h = blockIdx.y, g = h / (H / G), tid = threadIdx.x, at = tid / 16, part = tid % 16;
  const TokenTile where = find_token_tile(q_start, R, CHUNK, first_chunk + blockIdx.x, from);
  if (where.req < 0) return;
  const long t0 = q_start[where.req] + (long)where.tile * CHUNK;
  const int tokens = min(CHUNK, (int)(q_start[where.req + 1] - t0));
  const ChunkShape shape = chunk_shape(D, dv);
  float* out = scratch + ((long)blockIdx.x * H + h) * shape.all;
  const float* rows = qkv + t0 * qkv_stride;
  f32x4_t *qs = vectors, *ks = vectors + CHUNK * D / 4, *gs = vectors + 2 * CHUNK * D / 4;

  // a thread's first value column, asked for before everything else
  auto column = [&](float (&x)[CHUNK], int c) {
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) x[t] = t < tokens ? rows[t * qkv_stride + 2L * G * D + (long)h * dv + c] : 0.f;
  };
  float first[CHUNK];
  if (tid >= D && tid < D + dv) column(first, tid - D);

  // sixteen lanes to a token, four channels of every 64 each; a token that is not there has no key, no query and forgets nothing
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t k[DQ];
  {
    const bool there = at < tokens;
    f32x4_t q[DQ], decay[DQ];
    float q2 = 0.f, k2 = 0.f;
#pragma unroll
    for (int j = 0; j < DQ; ++j) {
      const int c = j * 64 + part * 4;
      q[j] = there ? *reinterpret_cast<const f32x4_t*>(rows + at * qkv_stride + (long)g * D + c) : zero;
      k[j] = there ? *reinterpret_cast<const f32x4_t*>(rows + at * qkv_stride + (long)(G + g) * D + c) : zero;
      if (!per_head) decay[j] = there ? *reinterpret_cast<const f32x4_t*>(a + (t0 + at) * a_stride + (long)h * D + c) : zero;
    }
    const float rate = expf(A_log[h]);
    const float whole = per_head && there ? expf(-rate * softplus_of(a[(t0 + at) * a_stride + h] + dt_bias[h])) : 1.f;
#pragma unroll
    for (int j = 0; j < DQ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        q2 = fmaf(q[j][e], q[j][e], q2);
        k2 = fmaf(k[j][e], k[j][e], k2);
        decay[j][e] = per_head || !there ? whole : expf(-rate * softplus_of(decay[j][e] + dt_bias[(long)h * D + j * 64 + part * 4 + e]));
      }
    const float qn = q_scale / sqrtf(row16_sum(q2) + unit_eps), kn = 1.0f / sqrtf(row16_sum(k2) + unit_eps);
#pragma unroll
    for (int j = 0; j < DQ; ++j) {
      k[j] = there ? k[j] * kn : zero;
      qs[at * (D / 4) + j * 16 + part] = there ? q[j] * qn : zero;
      ks[at * (D / 4) + j * 16 + part] = k[j];
      gs[at * (D / 4) + j * 16 + part] = decay[j];
    }
    if (part == 0) betas[at] = there ? 1.0f / (1.0f + expf(-b[(t0 + at) * b_stride + h])) : 0.f;
  }
  __syncthreads();

  // sixteen lanes to a key s: w = k_s with the decays since s, met by the keys and queries from s on
  {
    f32x4_t w[DQ];
#pragma unroll
    for (int j = 0; j < DQ; ++j) w[j] = zero;
#pragma unroll 4
    for (int t = 0; t < CHUNK; ++t) {
      float by_k = 0.f, by_q = 0.f;
#pragma unroll
      for (int j = 0; j < DQ; ++j) {
        const f32x4_t kt = ks[t * (D / 4) + j * 16 + part], qt = qs[t * (D / 4) + j * 16 + part], gt = gs[t * (D / 4) + j * 16 + part];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          w[j][e] = t == at ? k[j][e] : w[j][e] * gt[e];
          by_k = fmaf(w[j][e], kt[e], by_k);
          by_q = fmaf(w[j][e], qt[e], by_q);
        }
      }
      by_k = row16_sum(by_k);
      by_q = row16_sum(by_q);
      if (part == 0) {
        pairs[0][t][at] = t > at ? betas[t] * by_k : 0.f;
        pairs[1][t][at] = t >= at ? by_q : 0.f;
      }
    }
  }
  __syncthreads();

  // a thread to a column of [L k | V]
  auto solve = [&](float (&x)[CHUNK]) {
#pragma unroll
    for (int t = 1; t < CHUNK; ++t) {
#pragma unroll
      for (int s = 0; s < t; ++s) x[t] = fmaf(-pairs[0][t][s], x[s], x[t]);
      if (t % 4 == 3) asm volatile("" ::: "memory");      // no more than four rows of pairs in registers at a time
    }
  };
  auto store_columns = [&](float* to, int c, const float (&x)[CHUNK]) {        // [tile][lane = 16 (t / 4) + c % 16][t % 4]
#pragma unroll
    for (int i = 0; i < CHUNK / 4; ++i) reinterpret_cast<f32x4_t*>(to)[c / 16 * 64 + i * 16 + c % 16] = f32x4_t{x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
  };
  float y[CHUNK], lq[CHUNK];
  if (tid < D) {
    float decay[CHUNK], key[CHUNK];
    const float *qc = reinterpret_cast<const float*>(qs) + tid, *kc = reinterpret_cast<const float*>(ks) + tid, *gc = reinterpret_cast<const float*>(gs) + tid;
    float since = 1.f;
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
      decay[t] = gc[t * D];
      key[t] = kc[t * D];
      since *= decay[t];
      lq[t] = since * qc[t * D];
      y[t] = betas[t] * (since * key[t]);
    }
    out[shape.decay + tid] = since;
    float after = 1.f;
#pragma unroll
    for (int t = CHUNK - 1; t >= 0; --t) {
      key[t] *= after;
      after *= decay[t];
    }
    store_columns(out + shape.k, tid, key);
    solve(y);
  }
  for (int c = tid < D ? tid + 256 : tid; c < D + dv; c += 256) {      // threads beyond the channels start with V
    if (c >= 256) column(first, c - D);
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) first[t] = t < tokens ? betas[t] * first[t] : 0.f;
    solve(first);
    store_columns(out + shape.x, c - D, first);
  }
  if (tid < 64) reinterpret_cast<f32x4_t*>(out + shape.p)[tid] = *reinterpret_cast<const f32x4_t*>(&pairs[1][tid % 16][tid / 16 * 4]);
  __syncthreads();                               // everybody has read the vectors
  // Y and L q as the other operand: [tile][lane = 16 (c % 16 / 4) + t][c % 4]
  float* turned = reinterpret_cast<float*>(vectors);
  if (tid < D) {
    float* to = turned + (tid / 4 * 17) * 4 + tid % 4;
#pragma unroll
    for (int t = 0; t < CHUNK; ++t) {
      to[t * 4] = -y[t];
      to[PADDED + t * 4] = lq[t];
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < DQ; ++j) {
    const int i = j * 256 + tid;
    reinterpret_cast<f32x4_t*>(out + shape.y)[i] = reinterpret_cast<const f32x4_t*>(turned)[i / 16 * 17 + i % 16];
    reinterpret_cast<f32x4_t*>(out + shape.q)[i] = reinterpret_cast<const f32x4_t*>(turned + PADDED)[i / 16 * 17 + i % 16];
  }
}

// blockIdx: (head, slice of sixteen value columns, request): a head on one die, a long request on all of them.  Four waves keep the
// state, a quarter of its channels each, in the order in which a product leaves it, which is the order in which the next takes it:
// lane 16 r + c holds rows 4 r .. 4 r + 3 of a tile of 16 and column c.  Their shares of Y S_0 meet in LDS; with their sum, U, every
// wave brings its part of the state up to date.  A fifth wave makes the outputs a chunk behind.  What a chunk needs is fetched AHEAD
// chunks before.
// Bound by a chain of latencies: 24 matrix instructions of 32 cycles per chunk and wave at 128 channels are 0.32 of its 0.85 us (0.53
// without the fifth wave and without loads).  Outputs by the four waves themselves, a quarter of the rows each, and loads dealt out
// between the products were no faster (108 us as it is, 122 and 122).
template <int DQ>
__global__ __launch_bounds__(320) void delta_chunk_walk_kernel(float* __restrict__ o, long o_stride, const float* __restrict__ scratch,
                                                               const int* __restrict__ q_start, const int* __restrict__ slots, int from,
                                                               int first_chunk, int count, float* __restrict__ state, long state_stride, int H, int dv, int nr) {
  constexpr int D = 64 * DQ, AHEAD = DQ == 4 ? 2 : DQ == 3 ? 3 : 4;      // as many as there are registers for
  __shared__ f32x4_t of_u[2][4][64], of_o[2][4][64];
  const int h = blockIdx.x, z = blockIdx.y, r = blockIdx.z, lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // of the request's chunks those from `begin` on that lie in the window
  const int tokens = q_start[r + 1] - q_start[r], before = token_tiles_before(q_start, r, CHUNK, from);
  const int begin = max(first_chunk - before, 0), chunks = min(first_chunk + count - before, token_tiles(tokens, CHUNK, from)) - begin;
  if (chunks <= 0) return;
  const int n = tokens - begin * CHUNK;
  const ChunkShape shape = chunk_shape(D, dv);
  const long step = (long)H * shape.all;
  const float* mine = scratch + ((long)(before + begin - first_chunk) * H + h) * shape.all;
  auto fragment = [&](int c, int from_float, int tile) { return reinterpret_cast<const f32x4_t*>(mine + c * step + from_float)[tile * 64 + lane]; };
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};

  if (wave < 4) {
    // a state row holds its columns by sixteen, four to a slice: [head][slice of four columns][row % nr][16 (column % 4) + row / nr]
    float* kept = state + (long)slots[r] * state_stride + (((long)h * (dv / 16) + z) * 4 + lane % 16 / 4) * nr * 64 + lane % 4 * 16;
    auto place = [&](int tile, int i) {
      const int row = (wave * DQ + tile) * 16 + lane / 16 * 4 + i;
      return row % nr * 64 + row / nr;
    };
    f32x4_t s[DQ];
#pragma unroll
    for (int j = 0; j < DQ; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[j][i] = kept[place(j, i)];
    struct Fetched {
      f32x4_t y[DQ], q[DQ], k[DQ], decay[DQ], x;
    } got[AHEAD];
    auto fetch = [&](Fetched& f, int c) {
      c = min(c, chunks - 1);
#pragma unroll
      for (int j = 0; j < DQ; ++j) {
        f.y[j] = fragment(c, shape.y, wave * DQ + j);
        f.q[j] = fragment(c, shape.q, wave * DQ + j);
        f.k[j] = fragment(c, shape.k, wave * DQ + j);
        f.decay[j] = reinterpret_cast<const f32x4_t*>(mine + c * step + shape.decay)[(wave * DQ + j) * 4 + lane / 16];
      }
      f.x = fragment(c, shape.x, z);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(got[i], i);
    auto take = [&](Fetched& f, int c) {
      f32x4_t u0 = zero, u1 = zero, o0 = zero, o1 = zero;
#pragma unroll
      for (int j = 0; j < DQ; ++j)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          u0 = mfma16_f32(f.y[j][e], s[j][e], u0);
          u1 = mfma16_f32(f.y[j][e + 1], s[j][e + 1], u1);
        }
      of_u[c & 1][wave][lane] = u0 + u1;
      block_barrier_keeping_loads<63>();
      f32x4_t u = f.x, share[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) share[w] = of_u[c & 1][w][lane];
#pragma unroll
      for (int j = 0; j < DQ; ++j)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          o0 = mfma16_f32(f.q[j][e], s[j][e], o0);
          o1 = mfma16_f32(f.q[j][e + 1], s[j][e + 1], o1);
        }
      u += (share[0] + share[1]) + (share[2] + share[3]);
#pragma unroll
      for (int j = 0; j < DQ; ++j) s[j] *= f.decay[j];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < DQ; ++j) s[j] = mfma16_f32(f.k[j][e], u[e], s[j]);
      of_o[c & 1][wave][lane] = o0 + o1;
      fetch(f, c + AHEAD);
    };
    int c = 0;
    for (; c + AHEAD <= chunks; c += AHEAD) {    // without a way out in between: what is still on its way stays countable
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) take(got[i], c + i);
    }
#pragma unroll
    for (int i = 0; i < AHEAD - 1; ++i)
      if (c + i < chunks) take(got[i], c + i);
    block_barrier_keeping_loads<63>();           // the last outputs' shares are there
#pragma unroll
    for (int j = 0; j < DQ; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) kept[place(j, i)] = s[j][i];
  } else {
    f32x4_t inside = zero, p[AHEAD], x[AHEAD];
    auto fetch = [&](int i, int c) {
      c = min(c, chunks - 1);
      p[i] = fragment(c, shape.p, 0);
      x[i] = fragment(c, shape.x, z);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i, i);
    float* to = o + ((long)q_start[r] + begin * CHUNK + lane / 16 * 4) * o_stride + (long)h * dv + z * 16 + lane % 16;
    auto finish = [&](int c) {                   // the outputs of chunk c, whose shares the last barrier has brought
      f32x4_t share[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) share[w] = of_o[c & 1][w][lane];
      inside += (share[0] + share[1]) + (share[2] + share[3]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c * CHUNK + lane / 16 * 4 + e < n) to[(c * (long)CHUNK + e) * o_stride] = inside[e];
    };
    auto take = [&](int i, int c) {
      block_barrier_keeping_loads<63>();
      if (c > 0) finish(c - 1);
      f32x4_t u = x[i], share[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) share[w] = of_u[c & 1][w][lane];
      u += (share[0] + share[1]) + (share[2] + share[3]);
      inside = zero;
      bool finite = true;
#pragma unroll
      for (int e = 0; e < 4; ++e) finite = finite && fabsf(u[e]) < INFINITY;
      if (__all(finite)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) inside = mfma16_f32(p[i][e], u[e], inside);
      } else {                                   // a value that is not finite reaches no token before its own, not by way of zero either
#pragma unroll 1
        for (int s = 0; s < CHUNK; ++s) {
          float us = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float v = __shfl(u[e], s / 4 * 16 + lane % 16);
            us = s % 4 == e ? v : us;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int t = lane / 16 * 4 + e;
            float pts = 0.f;
#pragma unroll
            for (int f = 0; f < 4; ++f) {
              const float v = __shfl(p[i][f], s / 4 * 16 + t);
              pts = s % 4 == f ? v : pts;
            }
            if (s <= t) inside[e] = fmaf(pts, us, inside[e]);
          }
        }
      }
      fetch(i, c + AHEAD);
    };
    int c = 0;
    for (; c + AHEAD <= chunks; c += AHEAD) {
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) take(i, c + i);
    }
#pragma unroll
    for (int i = 0; i < AHEAD - 1; ++i)
      if (c + i < chunks) take(i, c + i);
    block_barrier_keeping_loads<63>();
    finish(chunks - 1);
  }
}

// Tokens of a chunk, for the caller's count of chunks (sum of ceil(tokens / this) over the requests that run in chunks), or
// 0: sizes that the chunked form does not take.
extern "C" int pi_delta_chunk(int d, int dv) { return d > 0 && d % 64 == 0 && d <= 256 && dv > 0 && dv % 16 == 0 ? CHUNK : 0; }

// The requests that bring `from` tokens or more, with a decay per channel or (`per_head`) per head; `chunks` of them in all, or an upper
// bound.  `scratch`: H * (49 d + 16 dv + 256) floats per chunk, for all of them or for fewer, which are then taken one window after the other.  Arguments otherwise as for pi_delta_scan; qkv, a and b are only read.  Rows of q, k and of the decays per channel must be 16-byte aligned.
extern "C" int pi_delta_chunks(float* o, long o_stride, const float* qkv, long qkv_stride, const float* a, long a_stride, const float* dt_bias,
                               const float* A_log, const float* b, long b_stride, const int* q_start, const int* slots, int R, int from, int chunks,
                               float* scratch, long scratch_floats, float* state, long state_stride, int H, int G, int d, int dv, float q_scale, float unit_eps, int per_head,
                               hipStream_t stream) {
  PI_REQUIRE(H > 0 && H <= 32767 && G > 0 && H % G == 0, "delta rule: bad sizes heads=%d kv_heads=%d", H, G);
  PI_REQUIRE(pi_delta_chunk(d, dv) > 0, "delta rule: no chunked form for keys of %d and values of %d", d, dv);
  int nr = 1;
  while (16 * nr < d) nr *= 2;
  PI_REQUIRE(R > 0 && from > 0 && chunks > 0 && scratch && state_stride >= (long)H * (dv / 16) * 4 * nr * PI_WAVE,
             "delta rule: bad step (%d requests, %d chunks) or a state row of %ld floats that cannot hold %d x %d x %d", R, chunks, state_stride, H, d, dv);
  PI_REQUIRE(qkv_stride % 4 == 0 && (uintptr_t)qkv % 16 == 0 && (uintptr_t)scratch % 16 == 0 && (per_head || (a_stride % 4 == 0 && (uintptr_t)a % 16 == 0)),
             "delta rule: rows must be 16-byte aligned");
  const long window = scratch_floats / ((long)H * chunk_shape(d, dv).all);
  PI_REQUIRE(window > 0, "delta rule: a chunk of %d heads does not fit %ld floats", H, scratch_floats);
  PI_REQUIRE(dv / 16 <= 65535 && R <= 65535, "delta rule: values of %d, %d requests", dv, R);
#define GO(DQ_)                                                                                                                                  \
  case DQ_:                                                                                                                                      \
    hipLaunchKernelGGL((delta_chunk_prepare_kernel<DQ_>), dim3(count, H), dim3(256), 0, stream, scratch, qkv, qkv_stride, a, a_stride, dt_bias,  \
                       A_log, b, b_stride, q_start, R, from, first, H, G, dv, q_scale, unit_eps, per_head);                                     \
    hipLaunchKernelGGL((delta_chunk_walk_kernel<DQ_>), dim3(H, dv / 16, R), dim3(320), 0, stream, o, o_stride, scratch, q_start, slots, from,    \
                       first, count, state, state_stride, H, dv, nr);                                                                            \
    break
  for (long at = 0; at < chunks; at += window) {
    const int first = (int)at, count = (int)(chunks - at < window ? chunks - at : window);
    switch (d / 64) {
      GO(1); GO(2); GO(3); GO(4);
    }
    if (pi_check_launch("delta_chunks")) return -1;
  }
#undef GO
  return 0;
}
