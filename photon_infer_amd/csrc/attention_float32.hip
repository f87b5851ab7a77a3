// Causal attention of prompt portions over the paged cache on the float32 path, on the matrix cores with 32-bit operands,
// products and sums (v_mfma_f32_16x16x4_f32).  The same definition, masks and options as attention_general.hip, which
// keeps single tokens, kept first keys, values of another width and head sizes this kernel does not take.
//
// A block is four waves on 16 rows each of (token, head): WH heads of one kv head times 4 / WH groups of 16 tokens.  They
// share rounds of 64 keys and values through LDS, fetched into registers a round ahead.  Everything is transposed: scores
// are keys x queries, so a lane holds 16 keys' scores of one query, the softmax needs two lane swaps per round, and the
// weights are the operand of the second product without leaving their lanes.  LDS rows are one 16-byte piece longer than
// their data, an odd number of pieces, so that the sixteen rows of a fragment lie on all banks.
//
// Bound by the matrix cores: 128 instructions of 32 cycles per round and wave at head size 64.  Three prompts of 345 to 517
// tokens, 32 heads of 64 on 8 kv heads: 64 us per layer, 462 on attention_general.hip (one wave per token and head).
//
// A query's masked keys weigh zero, and zero times a value that is not finite would not be: a round that holds such a value
// takes its second product key by key on the vector unit, where a query meets only the values it sees.  Looking out for them
// costs nothing that can be measured at head size 64 and 3.5 % at 128 (64 tokens at 8,192 keys: 582 us both ways, 909 -> 940).
#include "mfma.h"
#include "token_tiles.h"

#define KEYS 64

struct Float32AttnOptions {
  const float *slopes, *sinks, *gate;
  long gate_stride;
  float softcap, out_mult;
  int window, chunk;
};

__device__ inline int first_key(const Float32AttnOptions& o, int p) {
  int lo = (o.window > 0 && p - o.window + 1 > 0) ? p - o.window + 1 : 0;
  if (o.chunk > 0 && (p / o.chunk) * o.chunk > lo) lo = (p / o.chunk) * o.chunk;
  return lo;
}

// Waves per SIMD as without the path for values that are not finite, which by itself makes the compiler take more registers.
template <int HD>
__global__ __launch_bounds__(256, HD <= 16 ? 5 : HD <= 32 ? 4 : HD <= 64 ? 3 : 2) void attention_float32_kernel(float* __restrict__ out, long out_stride, const float* __restrict__ q, long q_stride,
                                                                const float* __restrict__ k_cache, const float* __restrict__ v_cache,
                                                                const int* __restrict__ block_table, int table_width,
                                                                const int* __restrict__ q_start, const int* __restrict__ kv_len, int R, int nh, int nkv,
                                                                int wh, int page_size, float scale, long num_pages, Float32AttnOptions o) {
  constexpr int P = HD / 16;                       // pieces of 16 bytes that a thread brings per round, of keys and of values
  constexpr int KROW = HD / 4 + 1, VROW = KEYS / 4 + 1;
  __shared__ f32x4_t ks[KEYS * KROW];              // [key][feature piece]
  __shared__ f32x4_t vs[HD * VROW];                // [feature][key piece]
  __shared__ int not_finite;                       // the last round (its first key) with a value that is not finite
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int lr = lane % 16, lg = lane / 16;

  // which request and which of its token tiles: the last tiles, with the longest walks, start first
  const int tile_tokens = 16 * (4 / wh);
  const TokenTile at = find_token_tile(q_start, R, tile_tokens, (int)gridDim.x - 1 - (int)blockIdx.x);
  const int req = at.req, tile = at.tile;
  if (req < 0) return;                             // the same in every wave of the block
  const int q0 = q_start[req], n = q_start[req + 1] - q0, before = kv_len[req] - n;
  const int t0 = tile * tile_tokens;
  const int last = before + min(t0 + tile_tokens, n) - 1;            // the tile's last position
  const int start = first_key(o, before + t0) / KEYS * KEYS;
  const int head = (int)blockIdx.y * wh + wave % wh, g = head / (nh / nkv);
  const int token = t0 + (wave / wh) * 16 + lr;                      // this lane's query
  const bool there = token < n;
  const int p = before + min(token, n - 1), lo = first_key(o, p);
  const int* bt = block_table + (long)req * table_width;

  f32x4_t qf[P];
  const float* qr = q + (long)(q0 + min(token, n - 1)) * q_stride + (long)head * HD + lg * 4;
#pragma unroll
  for (int f = 0; f < P; ++f) qf[f] = *reinterpret_cast<const f32x4_t*>(qr + f * 16);

  // Keys are fetched in tiles of 16, each in one page.  A key whose page is missing becomes a NaN score; what lies behind
  // the tile's last position counts as zero in the values, whose weight is zero there.
  auto page_of = [&](int key) {
    const int blk = key / page_size;
    return key <= last && blk < table_width ? (long)bt[blk] : -1L;
  };
  long pages[4];
  auto next_pages = [&](int k0) {
#pragma unroll
    for (int t = 0; t < 4; ++t) pages[t] = page_of(k0 + t * 16);
  };
  f32x4_t kn[P], vn[P];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int idx = tid + i * 256, kt = idx / (4 * HD);
      const long page = kt == 0 ? pages[0] : kt == 1 ? pages[1] : kt == 2 ? pages[2] : pages[3];
      const bool ok = page >= 0 && page < num_pages;
      const long base = (page * nkv + g) * (long)page_size * HD;
      const int key = k0 + idx / (HD / 4), vkey = k0 + kt * 16 + (idx % 4) * 4, d = idx % (4 * HD) / 4;
      const float bad = key <= last ? __builtin_nanf("") : 0.f;
      kn[i] = f32x4_t{bad, bad, bad, bad};
      vn[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (ok) {
        kn[i] = *reinterpret_cast<const f32x4_t*>(k_cache + base + (key % page_size) * HD + (idx % (HD / 4)) * 4);
        vn[i] = *reinterpret_cast<const f32x4_t*>(v_cache + base + (long)d * page_size + vkey % page_size);
      }
    }
  };
  auto stage = [&](int k0) {
    float probe = 0.f;                             // stays zero as long as every value is finite
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int idx = tid + i * 256, kt = idx / (4 * HD), vkey = k0 + kt * 16 + (idx % 4) * 4, d = idx % (4 * HD) / 4;
      ks[idx / (HD / 4) * KROW + idx % (HD / 4)] = kn[i];
      f32x4_t v = vn[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = vkey + e <= last ? v[e] : 0.f;
        probe = fmaf(v[e], 0.f, probe);
      }
      vs[d * VROW + kt * 4 + idx % 4] = v;
    }
    if (probe != 0.f) not_finite = k0;
  };

  const float slope = o.slopes ? o.slopes[head] : 0.f;
  float m = -INFINITY, l = 0.f;                    // l: this lane's share of the sum
  f32x4_t acc[P];
#pragma unroll
  for (int b = 0; b < P; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (tid == 0) not_finite = -1;
  next_pages(start);
  fetch(start);
  next_pages(start + KEYS);
  for (int k0 = start; k0 <= last; k0 += KEYS) {
    __syncthreads();                               // everybody has left the round before
    stage(k0);
    __syncthreads();
    if (k0 + KEYS <= last) {
      fetch(k0 + KEYS);
      next_pages(k0 + 2 * KEYS);
    }
    f32x4_t s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < P; ++f)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const f32x4_t a = ks[(t * 16 + lr) * KROW + f * 4 + lg];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t] = mfma16_f32(a[e], qf[f][e], s[t]);
      }
    // s[t][i] belongs to key k0 + t * 16 + lg * 4 + i
    float top = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k0 + t * 16 + lg * 4 + i;
        float x = s[t][i] * scale;
        if (o.softcap > 0.f) x = o.softcap * tanhf(x / o.softcap);
        if (o.slopes) x -= slope * (float)(p - key);
        s[t][i] = key <= p && key >= lo ? x : -INFINITY;
        top = fmaxf(top, s[t][i]);
      }
    const float m_new = fmaxf(m, column_max(top));
    const float ref = m_new == -INFINITY ? 0.f : m_new;      // nothing seen yet: every weight is zero
    const float corr = expf(m - ref);
    m = m_new;
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[t][i] = expf(s[t][i] - ref);
        sum += s[t][i];
      }
    l = l * corr + sum;
#pragma unroll
    for (int b = 0; b < P; ++b) acc[b] *= corr;
    if (__builtin_expect(not_finite == k0, 0)) {
      const float* values = reinterpret_cast<const float*>(vs) + lg * 4 * (VROW * 4);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll 1
          for (int from = 0; from < 4; ++from) {   // the lane group that holds the key's weights
            const int at = t * 16 + from * 4 + i;
            const float w = __shfl(s[t][i], from * 16 + lr, 64);
            if (k0 + at < lo || k0 + at > p) continue;
#pragma unroll
            for (int b = 0; b < P; ++b)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[b][e] = fmaf(w, values[(b * 16 + e) * (VROW * 4) + at], acc[b][e]);
          }
      continue;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int b = 0; b < P; ++b) {
        const f32x4_t a = vs[(b * 16 + lr) * VROW + t * 4 + lg];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b] = mfma16_f32(a[e], s[t][e], acc[b]);
      }
  }
  // acc[b][i] is feature b * 16 + lg * 4 + i of this lane's query
  l = column_sum(l);
  float factor = o.out_mult;
  const long row = q0 + token;
  if (o.sinks) {                                   // the sink joins the denominator once, against the common maximum
    const float m_all = fmaxf(m, o.sinks[head]), corr = expf(m - m_all);
    l = l * corr + expf(o.sinks[head] - m_all);
    factor *= corr;
  }
  if (!there) return;
  if (o.gate && !o.gate_stride) factor *= o.gate[row * nh + head];
  const float inv = factor / l;
  float* dst = out + row * out_stride + (long)head * HD + lg * 4;
  const float* gates = o.gate_stride ? o.gate + row * o.gate_stride + (long)head * HD + lg * 4 : nullptr;
#pragma unroll
  for (int b = 0; b < P; ++b) {
    f32x4_t y = acc[b];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] *= gates ? inv * (1.0f / (1.0f + expf(-gates[b * 16 + i]))) : inv;
    *reinterpret_cast<f32x4_t*>(dst + b * 16) = y;
  }
}

// Tokens of a block's tile for such heads (the caller counts the tiles: sum over requests of ceil(tokens / this)).
static int heads_per_block(int nh, int nkv) {
  const int group = nh / nkv;
  return group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
}
extern "C" int pi_attention_float32_tile_tokens(int nh, int nkv) { return nh > 0 && nkv > 0 && nh % nkv == 0 ? 16 * (4 / heads_per_block(nh, nkv)) : 0; }

extern "C" int pi_attention_float32(void* out, long out_stride, const void* q, long q_stride, const void* k_cache, const void* v_cache,
                                    const int* block_table, int table_width, const int* q_start, const int* kv_len, int R, int tiles, int nh, int nkv,
                                    int hd, int page_size, float scale, int window, long num_pages, const float* slopes, const float* sinks,
                                    const float* gate, long gate_stride, float softcap, float out_mult, int chunk, hipStream_t stream) {
  PI_REQUIRE(R > 0 && tiles > 0 && nh > 0 && nkv > 0 && nh % nkv == 0, "attention: bad sizes R=%d tiles=%d heads=%d kv heads=%d", R, tiles, nh, nkv);
  PI_REQUIRE(hd > 0 && hd <= 128 && hd % 16 == 0, "attention: the float32 tile kernel takes head sizes that are multiples of 16 up to 128, got %d", hd);
  PI_REQUIRE(page_size > 0 && page_size % 16 == 0 && table_width > 0 && num_pages > 0, "attention: bad cache geometry page_size=%d table_width=%d pages=%ld", page_size, table_width, num_pages);
  PI_REQUIRE(q_stride % 4 == 0 && out_stride % 4 == 0 && (uintptr_t)q % 16 == 0 && (uintptr_t)out % 16 == 0 && (uintptr_t)k_cache % 16 == 0 && (uintptr_t)v_cache % 16 == 0,
             "attention: rows and caches must be 16-byte aligned");
  PI_REQUIRE(window >= 0 && chunk >= 0 && gate_stride >= 0, "attention: window (%d), chunk (%d) and gate stride must not be negative", window, chunk);
  const int wh = heads_per_block(nh, nkv);
  PI_REQUIRE(nh / wh <= 65535, "attention: too many heads (%d)", nh);
  const dim3 grid(tiles, nh / wh), block(256);
  const Float32AttnOptions o{slopes, sinks, gate, gate_stride, softcap, out_mult, window, chunk};
#define GO(H)                                                                                                                                  \
  case H:                                                                                                                                      \
    hipLaunchKernelGGL((attention_float32_kernel<H>), grid, block, 0, stream, (float*)out, out_stride, (const float*)q, q_stride,              \
                       (const float*)k_cache, (const float*)v_cache, block_table, table_width, q_start, kv_len, R, nh, nkv, wh, page_size,     \
                       scale, num_pages, o);                                                                                                   \
    break
  switch (hd) {
    GO(16); GO(32); GO(48); GO(64); GO(80); GO(96); GO(112); GO(128);
  }
#undef GO
  return pi_check_launch("attention_float32");
}
