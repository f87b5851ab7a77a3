// Every global fetch of the matrix-product kernels, enumerated on the host from the kernels' own
// address arithmetic (csrc/addressing.h), checked to lie inside its operand.
//
//   load_bounds [old-standin] [only] [M N K splits]...
//
// Walks the built-in sweep of shapes (and any given as arguments) through the lanes, waves,
// blocks and steps of gemm_skinny_kernel, gemm_skinny_ring_kernel, gemm_mfma_kernel,
// gemm_mfma_big_kernel in its six tile shapes, gemm_rows_kernel, gemm_float32_rows_kernel, gemm_float32_tile_kernel and gemm_float32_parts_kernel exactly as the kernels
// walk them (and, in the built-in sweep, through the
// key and value fetches of the attention kernels' chunks for every head size and several page sizes), with the matrices row by row (several row
// strides) and, where the sizes allow, in the weight-streaming kernels' tiled order.  Prints
// "ok <fetches>" or the first fetch that leaves its operand (exit status 1).
// "only" leaves the built-in sweep out.  "old-standin" replaces the stand-in address of a lane beyond a partial k step by the formula
// the kernel once had (the range's start plus the lane's own offset): the sweep must then fail.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "addressing.h"

namespace A = addressing;

static bool old_standin = false;
static long fetches = 0;

struct Shape {
  int M, N, K, splits;
};

static bool fail(const char* kernel, const char* operand, const Shape& s, long ld, int tiled, long off, const char* why) {
  std::printf("out of bounds: %s %s M=%d N=%d K=%d splits=%d ld=%ld tiled=%d offset=%ld: %s\n", kernel, operand, s.M, s.N, s.K,
              s.splits, ld, tiled, off, why);
  return false;
}

// an 8-element fetch at `off` of a row-major operand [rows, cols] with row stride ld must lie in row `row`
static bool in_row(long off, long row, long ld, int cols) { return off >= row * ld && off + 8 <= row * ld + cols; }

// ------------------------------------------------------------------ 1..32 tokens
static bool skinny(const Shape& s, long ldx, long ldw, int tiled, int RT, int quantum) {
  const int M = s.M, N = s.N, K = s.K;
  const A::KSplit cut = A::cut_k(K, s.splits, quantum);
  const int rows_per_block = RT * 16, MB = (M + 15) / 16;
  const int groups = (N + rows_per_block - 1) / rows_per_block;
  const int x_loads = (M + 7) / 8;
  for (int by = 0; by < cut.splits; ++by)
    for (int bx = 0; bx < groups; ++bx)
      for (int wave = 0; wave < 4; ++wave) {
        const A::WaveRange r = A::skinny_wave_range(K, cut.k_per_block, by, wave);
        for (int lane = 0; lane < 64; ++lane) {
          const int lr = lane % 16, lg = lane / 16, xt = lane / 8, xp = lane % 8;
          const long n0 = (long)bx * rows_per_block;
          int kk = r.k0;
          for (;; kk += A::KSTEP) {
            const bool whole = kk + A::KSTEP <= r.k1;
            if (!whole && kk >= r.k1) break;
            if (tiled && !whole) return fail("gemm_skinny", "W", s, ldw, tiled, kk, "a tiled matrix met a partial step");
            for (int t = 0; t < RT; ++t)
              for (int h = 0; h < 2; ++h) {
                long off = A::skinny_w_base(tiled, n0, t, lr, lg, N, K, ldw) + A::skinny_w_step(tiled, whole, kk, h, lg, r.k0, r.k1);
                if (old_standin && !whole && !A::skinny_w_used(whole, kk, h, lg, r.k1))
                  off = A::skinny_w_base(tiled, n0, t, lr, lg, N, K, ldw) + r.k0;
                ++fetches;
                if (tiled) {
                  if (off < 0 || off + 8 > (long)N * K) return fail("gemm_skinny", "W", s, ldw, tiled, off, "outside the matrix");
                } else {
                  const long row = A::lmin(n0 + t * 16 + lr, (long)N - 1);
                  if (!in_row(off, row, ldw, K)) return fail("gemm_skinny", "W", s, ldw, tiled, off, "outside its row");
                  if (A::skinny_w_used(whole, kk, h, lg, r.k1) && off != row * ldw + kk + lg * 16 + h * 8)
                    return fail("gemm_skinny", "W", s, ldw, tiled, off, "a used fetch is not the lane's k");
                }
              }
            for (int i = 0; i < MB * 2; ++i)
              if (i == 0 || i < x_loads) {
                const int token = i * 8 + xt;
                long off = A::skinny_x_base(token, M, ldx, xp) + A::skinny_x_step(whole, kk, xp, r.k0, r.k1);
                if (old_standin && !(whole || kk + xp * 8 < r.k1)) off = A::skinny_x_base(token, M, ldx, xp) + r.k0;
                ++fetches;
                if (!in_row(off, A::imin(token, M - 1), ldx, K)) return fail("gemm_skinny", "X", s, ldx, tiled, off, "outside its row");
              }
            if (!whole) break;
          }
        }
      }
  return true;
}

// ------------------------------------------------------------------ 1..32 rows of float32, in units of two bytes
static bool float32_rows(const Shape& s, long ldx, long ldw, int RT, int waves, int depth) {
  const int M = s.M, N = s.N, K = s.K;
  const A::KSplit cut = A::cut_k(K, s.splits, 32);
  const int rows_per_block = RT * 16, MB = (M + 15) / 16;
  const int x_loads = (M + 7) / 8;
  for (int by = 0; by < cut.splits; ++by)
    for (int bx = 0; bx < (N + rows_per_block - 1) / rows_per_block; ++bx)
      for (int wave = 0; wave < waves; ++wave) {
        const A::WaveRange r = A::wave_share(2 * by * cut.k_per_block, 2 * A::imin(K, (by + 1) * cut.k_per_block), waves, wave);
        const int steps = r.k1 > r.k0 ? (r.k1 - r.k0 + A::KSTEP - 1) / A::KSTEP : 0;
        if (steps == 0) continue;
        for (int lane = 0; lane < 64; ++lane) {
          const int lr = lane % 16, lg = lane / 16, xt = lane / 8, xp = lane % 8;
          const long n0 = (long)bx * rows_per_block;
          for (int st = 0; st < steps + depth; ++st) {   // the loads in flight run past the last step
            const int kk = r.k0 + A::imin(st, steps - 1) * A::KSTEP;
            for (int t = 0; t < RT; ++t)
              for (int h = 0; h < 2; ++h) {
                const long off = A::skinny_w_base(0, n0, t, lr, lg, N, 2 * K, 2 * ldw) + A::skinny_w_step(0, false, kk, h, lg, r.k0, r.k1);
                const long row = A::lmin(n0 + t * 16 + lr, (long)N - 1);
                ++fetches;
                if (!in_row(off, row, 2 * ldw, 2 * K)) return fail("gemm_float32_rows", "W", s, ldw, 0, off, "outside its row");
                if (A::skinny_w_used(false, kk, h, lg, r.k1) && off != row * 2 * ldw + kk + lg * 16 + h * 8)
                  return fail("gemm_float32_rows", "W", s, ldw, 0, off, "a used fetch is not the lane's k");
              }
            for (int i = 0; i < MB * 2; ++i)
              if (i == 0 || i < x_loads) {
                const int token = i * 8 + xt;
                const long off = A::skinny_x_base(token, M, 2 * ldx, xp) + A::skinny_x_step(false, kk, xp, r.k0, r.k1);
                ++fetches;
                if (!in_row(off, A::imin(token, M - 1), 2 * ldx, 2 * K)) return fail("gemm_float32_rows", "X", s, ldx, 0, off, "outside its row");
              }
          }
        }
      }
  return true;
}

// ------------------------------------------------------------------ tile kernels
// A tile kernel's geometry: rows of its tiles of A and of W, waves, whether it is the larger-tile kernel, and the slabs it
// asks for past the last.  A wave fills tile / (8 * waves) times eight rows of each per slab.
struct Tiles {
  const char* kernel;
  int rows_a, rows_w, waves;
  bool big;
  int ahead;
};

// One operand of one block: rows [row0, row0 + tile) of [R, K] with stride ld, k in [k_lo, k_hi), in units of two bytes.
static bool tile_operand(const Tiles& t, const char* operand, const Shape& s, long R, int K, long ld, long row0, int tile, int k_lo, int k_hi) {
  const int rows = (int)A::lmin(tile, R - row0), loads = tile / (8 * t.waves);
  const A::Descriptor d = A::tile_descriptor(row0, ld, k_lo, k_hi, rows);
  const long operand_bytes = ((R - 1) * ld + K) * 2;
  if (d.base < 0 || d.bytes <= 0 || d.base * 2 + d.bytes > operand_bytes || d.bytes >= 0x7ffffff0L)
    return fail(t.kernel, operand, s, ld, 0, d.base, "the descriptor leaves the operand");
  const int k_range = k_hi - k_lo, slabs = (k_range + 63) / 64;
  for (int wave = 0; wave < t.waves; ++wave)
    for (int p = 0; p < loads; ++p)
      for (int lane = 0; lane < 64; ++lane) {
        const int row = (wave * loads + p) * 8 + lane / 8, piece = A::tile_piece(lane, row);
        for (int sl = 0; sl < slabs + t.ahead; ++sl) {
          ++fetches;
          long off;      // bytes inside the descriptor
          bool used;
          if (t.big) {
            off = (long)A::big_lane_offset(row, rows, ld, piece) + A::big_slab_bytes(sl, slabs);
            used = row < rows && sl < slabs;
            if (off + 16 > d.bytes) return fail(t.kernel, operand, s, ld, 0, off, "a fetch of the larger tiles leaves its descriptor");
          } else {
            off = A::tile_slab_offset(A::tile_lane_offset(row, rows, ld, piece), sl * 64, piece, k_range);
            used = row < rows && sl * 64 + piece * 8 < k_range;
            if (!used && off < d.bytes) return fail(t.kernel, operand, s, ld, 0, off, "a fetch that should read zeros lies inside the descriptor");
            if (used && off + 16 > d.bytes) return fail(t.kernel, operand, s, ld, 0, off, "a used fetch leaves its descriptor");
          }
          if (used && d.base * 2 + off != ((row0 + row) * ld + k_lo + A::imin(sl, slabs - 1) * 64 + piece * 8) * 2)
            return fail(t.kernel, operand, s, ld, 0, off, "a used fetch is not the lane's row and k");
        }
      }
  return true;
}

// per: units of two bytes per element
static bool tiles(const Shape& s, long lda, long ldw, const Tiles& t, int per) {
  if (t.big && s.K % 64) return true;                  // the larger tiles take whole slabs only
  const A::KSplit cut = A::cut_k(s.K, s.splits, 64 / per);
  for (int by = 0; by < cut.splits; ++by) {
    const int k_lo = per * by * cut.k_per_block, k_hi = per * A::imin(s.K, (by + 1) * cut.k_per_block);
    for (long m0 = 0; m0 < s.M; m0 += t.rows_a)
      if (!tile_operand(t, "A", s, s.M, per * s.K, per * lda, m0, t.rows_a, k_lo, k_hi)) return false;
    for (long n0 = 0; n0 < s.N; n0 += t.rows_w)
      if (!tile_operand(t, "W", s, s.N, per * s.K, per * ldw, n0, t.rows_w, k_lo, k_hi)) return false;
  }
  return true;
}
static const Tiles BFLOAT16_TILES[] = {
    {"gemm_mfma", 128, 128, 4, false, 0},              // asks for existing slabs only
    // the larger tiles: as many slabs past the last as their rings of buffers hold
    {"gemm_mfma_big<4, 2>", 256, 256, 8, true, 3}, {"gemm_mfma_big<3, 3>", 192, 384, 8, true, 2}, {"gemm_mfma_big<3, 2>", 192, 256, 8, true, 3},
    {"gemm_mfma_big<2, 3>", 128, 384, 8, true, 2}, {"gemm_mfma_big<2, 2>", 128, 256, 8, true, 3}, {"gemm_mfma_big<2, 1>", 128, 128, 8, true, 3},
};
static const Tiles FLOAT32_TILES[] = {                 // the rings of buffers, less the one in use
    {"gemm_float32_tile<64, 64>", 64, 64, 4, false, 3},
};

// The float32 tiles in parts: 64 rows a load, slabs of 16 floats, one more slab than there are, and one more.
static const Tiles FLOAT32_PARTS[] = {
    {"gemm_float32_parts<2, 2>", 128, 128, 4, false, 2}, {"gemm_float32_parts<3, 2>", 192, 128, 4, false, 2}, {"gemm_float32_parts<2, 4>", 128, 256, 4, false, 2},
};
static bool parts_operand(const Tiles& t, const char* operand, const Shape& s, long R, long ld, long row0, int tile, int k_lo, int k_hi) {
  const int rows = (int)A::lmin(tile, R - row0), k_range = k_hi - k_lo, slabs = (k_range + A::PARTS_SLAB - 1) / A::PARTS_SLAB;
  const A::Descriptor d = A::tile_descriptor(row0, ld, k_lo, k_hi, rows);
  if (d.base < 0 || d.bytes <= 0 || d.base * 2 + d.bytes > ((R - 1) * ld + 2 * s.K) * 2 || d.bytes >= 0x7ffffff0L)
    return fail(t.kernel, operand, s, ld, 0, d.base, "the descriptor leaves the operand");
  for (int load = 0; load < tile / 64; ++load)
    for (int tid = 0; tid < 256; ++tid) {
      const int row = A::parts_row(load, tid), piece = A::parts_piece(tid);
      for (int sl = 0; sl < slabs + t.ahead; ++sl) {
        ++fetches;
        const long off = A::tile_slab_offset(A::tile_lane_offset(row, rows, ld, piece), sl * A::PARTS_SLAB, piece, k_range);
        const int k = sl * A::PARTS_SLAB + piece * 8;
        const bool used = row < rows && k < k_range;
        if (used ? off + 16 > d.bytes : off < d.bytes) return fail(t.kernel, operand, s, ld, 0, off, "on the wrong side of its descriptor");
        if (used && d.base * 2 + off != ((row0 + row) * ld + k_lo + k) * 2) return fail(t.kernel, operand, s, ld, 0, off, "a used fetch is not the lane's row and k");
      }
    }
  return true;
}
static bool parts(const Shape& s, long lda, long ldw, const Tiles& t) {
  const A::KSplit cut = A::cut_k(s.K, s.splits, 32);
  for (int by = 0; by < cut.splits; ++by) {
    const int k_lo = 2 * by * cut.k_per_block, k_hi = 2 * A::imin(s.K, (by + 1) * cut.k_per_block);
    for (long m0 = 0; m0 < s.M; m0 += t.rows_a)
      if (!parts_operand(t, "A", s, s.M, 2 * lda, m0, t.rows_a, k_lo, k_hi)) return false;
    for (long n0 = 0; n0 < s.N; n0 += t.rows_w)
      if (!parts_operand(t, "W", s, s.N, 2 * ldw, n0, t.rows_w, k_lo, k_hi)) return false;
  }
  return true;
}

// ------------------------------------------------------------------ 33..128 tokens, 17..128 on large matrices
// The activations are a tile of 64 or 128 rows; of the weights a block's eight waves take 32 rows by a quarter of each step's
// k each.  A fetch that is used lies inside its descriptor, at the row and k that the fragment stands for, and any other
// outside (it reads zeros).
static bool ring(const Shape& s, long ldx, long ldw, int tiled) {
  const A::KSplit cut = A::cut_k(s.K, s.splits, A::KSTEP);
  const Tiles t{"gemm_skinny_ring", s.M <= 64 ? 64 : 128, 64, 8, false, 4};
  for (int by = 0; by < cut.splits; ++by) {
    const int k_lo = by * cut.k_per_block, k_hi = A::imin(s.K, k_lo + cut.k_per_block), k_range = k_hi - k_lo;
    if (!tile_operand(t, "X", s, s.M, s.K, ldx, 0, t.rows_a, k_lo, k_hi)) return false;
    const int steps = (k_range + 63) / 64, last = (steps + 3) / 4 * 4 + t.ahead;
    for (long n0 = 0; n0 < s.N; n0 += 64) {
      const int rows = (int)A::lmin(64, s.N - n0);
      const A::Descriptor d = A::ring_w_descriptor(tiled, n0, k_lo, k_hi, rows, s.K, ldw);
      const long operand_bytes = tiled ? (long)s.N * s.K * 2 : ((s.N - 1) * ldw + s.K) * 2;
      if (d.base < 0 || d.bytes <= 0 || d.base * 2 + d.bytes > operand_bytes || d.bytes >= 0x7ffffff0L)
        return fail(t.kernel, "W", s, ldw, tiled, d.base, "the descriptor leaves the operand");
      for (int wave = 0; wave < 8; ++wave)
        for (int lane = 0; lane < 64; ++lane) {
          const int row = wave / 4 * 32 + lane % 32, piece = wave % 4 * 2 + lane / 32;
          const unsigned lane_offset = A::ring_w_lane_offset(tiled, row, rows, s.K, ldw, piece);
          for (int st = 0; st < last; ++st) {
            ++fetches;
            const long off = A::ring_w_step_offset(tiled, lane_offset, st * 64, piece, k_range);
            const long k = k_lo + st * 64 + piece * 8;
            if (row >= rows || k >= k_hi) {
              if (off < d.bytes) return fail(t.kernel, "W", s, ldw, tiled, off, "a fetch that should read zeros lies inside the descriptor");
              continue;
            }
            if (off + 16 > d.bytes) return fail(t.kernel, "W", s, ldw, tiled, off, "a used fetch leaves its descriptor");
            const long n = n0 + row;
            const long at = tiled ? (n / 16 * (s.K / 64) + k / 64) * 1024 + k % 16 / 8 * 512 + k % 64 / 16 * 128 + n % 16 * 8 : n * ldw + k;
            if (d.base * 2 + off != at * 2) return fail(t.kernel, "W", s, ldw, tiled, off, "a used fetch is not the lane's row and k");
          }
        }
    }
  }
  return true;
}

// ------------------------------------------------------------------ 1..16 tokens, all of k in a block
// Every fetch of gemm_rows_kernel with 8 or 16 rows a tile (8 where N is in 64), four or eight waves: the weights' copy and the
// activations through descriptors of a wave's own k.  A used fetch is the lane's row (token) and k; any other lies outside its
// descriptor.  Of many tiles the first two and the last two.
static bool few_rows(const Shape& s, long lda) {
  for (int rows : {8, 16})
    for (int waves : {4, 8})
      for (int wide = rows == 16 || s.M > 8; wide < 2; ++wide)
        for (long n0 = rows == 8 && s.N % 64 ? s.N : 0; n0 < s.N; n0 += s.N >= 512 && n0 == rows ? s.N - 3 * rows : rows)
          for (int wave = 0; wave < waves; ++wave) {
            const A::WaveRange r = A::wave_share(0, s.K, waves, wave);
            const int steps = r.k1 > r.k0 ? (r.k1 - r.k0) / 64 : 0;
            const A::Descriptor dw = A::rows_w_descriptor(n0, r.k0, steps, s.K), da = A::rows_a_descriptor(r.k0, steps, s.M, lda);
            if (steps > 0 && (dw.base < 0 || dw.base * 2 + dw.bytes > (long)s.N * s.K * 2)) return fail("gemm_rows", "W", s, s.K, 1, dw.base, "the descriptor leaves the operand");
            if (steps > 0 && (da.base < 0 || da.base * 2 + da.bytes > ((s.M - 1) * lda + s.K) * 2)) return fail("gemm_rows", "A", s, lda, 0, da.base, "the descriptor leaves the operand");
            for (int lane = 0; lane < 64; ++lane)
              for (int st = 0; st < steps + 16; ++st)
                for (int f = 0; f < 2; ++f) {
                  ++fetches;
                  const long w = A::rows_step(A::rows_w_lane(rows, n0, lane), st, steps, 2048, rows == 16 ? f * 1024 : 0);
                  const long a = A::rows_step(A::rows_a_lane(wide, lane, s.M, lda), st, steps, 128, wide ? f * 16 : 0);
                  const int wf = rows == 16 ? f : lane % 16 / 8, af = wide ? f : lane % 16 / 8;
                  const long n = n0 + (rows == 16 ? lane % 16 : lane % 8), token = wide ? lane % 16 : lane % 8;
                  if (st >= steps ? w < dw.bytes : w + 16 > dw.bytes) return fail("gemm_rows", "W", s, s.K, 1, w, "on the wrong side of its descriptor");
                  if (st >= steps || token >= s.M ? a < da.bytes : a + 16 > da.bytes) return fail("gemm_rows", "A", s, lda, 0, a, "on the wrong side of its descriptor");
                  const long k = r.k0 + st * 64 + lane / 16 * 16;
                  if (st < steps && dw.base * 2 + w != (n / 16 * (s.K / 64) + k / 64) * 2048 + wf * 1024 + lane / 16 * 256 + n % 16 * 16)
                    return fail("gemm_rows", "W", s, s.K, 1, w, "a used fetch is not the lane's row and k");
                  if (st < steps && token < s.M && da.base * 2 + a != (token * lda + k + af * 8) * 2) return fail("gemm_rows", "A", s, lda, 0, a, "a used fetch is not the lane's token and k");
                }
          }
  return true;
}

// ------------------------------------------------------------------ attention over the paged cache
// Every fetch of a chunk's two tiles (attn_load): the keys' fragments (16 bytes) and the values'
// (8 bytes) of every lane, for a page that is there, one that is missing and one whose id is no
// page of the pool (both read page 0 instead), lie inside the (page, kv head) block of their pool.
static bool attention(int hd, int page_size, int nkv, long num_pages) {
  const long page_elems = A::kv_page_elems(nkv, page_size, hd);
  const long pool_bytes = num_pages * page_elems * 2;
  const int KS = (hd + 31) / 32;
  const long ids[] = {0, num_pages - 1, -1, num_pages, num_pages + 5};
  for (long id : ids)
    for (int g = 0; g < nkv; ++g)
      for (int slot = 0; slot + 16 <= page_size; slot += 16) {
        const long pg = A::kv_page_or_first(id, num_pages);
        if (A::kv_page_there(id, num_pages) != (id >= 0 && id < num_pages) || pg < 0 || pg >= num_pages) {
          std::printf("out of bounds: attention page id %ld of %ld pages becomes %ld\n", id, num_pages, pg);
          return false;
        }
        const long block0 = ((pg * nkv + g) * (long)page_size) * hd * 2, block1 = block0 + (long)page_size * hd * 2;   // bytes of this (page, kv head)
        for (int lane = 0; lane < 64; ++lane) {
          for (int ks = 0; ks < KS; ++ks) {
            const bool held = hd % 32 == 0 || ks + 1 < KS || A::kv_lane_holds(hd, KS - 1, lane);
            const long at = A::kv_key_tile(pg, page_elems, g, page_size, slot, hd) * 2 + (held ? A::kv_key_lane(lane, hd) + ks * 64 : A::kv_key_lane_first(lane, hd));
            ++fetches;
            if (at < block0 || at + 16 > block1 || at + 16 > pool_bytes) {
              std::printf("out of bounds: attention key fetch hd=%d page=%d kv heads=%d g=%d slot=%d lane=%d ks=%d at %ld\n", hd, page_size, nkv, g, slot, lane, ks, at);
              return false;
            }
            const long row = (at - block0) / (hd * 2);        // the key it belongs to: one of the tile's sixteen
            if (row != slot + lane % 16) {
              std::printf("out of bounds: attention key fetch of lane %d reads key %ld of the page, not %d\n", lane, row, slot + lane % 16);
              return false;
            }
          }
          for (int db = 0; db < hd / 16; ++db) {
            const long at = A::kv_value_tile(pg, page_elems, g, page_size, slot, hd) * 2 + A::kv_value_lane(lane, db, page_size);
            ++fetches;
            if (at < block0 || at + 8 > block1) {
              std::printf("out of bounds: attention value fetch hd=%d page=%d kv heads=%d g=%d slot=%d lane=%d db=%d at %ld\n", hd, page_size, nkv, g, slot, lane, db, at);
              return false;
            }
            const long col = ((at - block0) / 2) % page_size;  // its first key: four of the tile's sixteen per lane group
            if (col != slot + (lane / 16) * 4) {
              std::printf("out of bounds: attention value fetch of lane %d starts at key %ld, not %d\n", lane, col, slot + (lane / 16) * 4);
              return false;
            }
          }
        }
      }
  return true;
}

static bool check(const Shape& s) {
  for (int pad = 0; pad <= 16 && s.K % 8 == 0; pad += 8) {     // row strides K, K + 8, K + 16
    const long ld = s.K + pad;
    if (s.M <= 32) {
      if (!skinny(s, ld, ld, 0, 2, A::KSTEP)) return false;
      if (s.M <= 16 && s.K % 64 == 0 && !skinny(s, ld, ld, 0, 4, 4 * A::KSTEP)) return false;     // the form that merges key ranges
    }
    if (s.M > 16 && s.M <= 128 && !ring(s, ld, ld, 0)) return false;
    for (const Tiles& t : BFLOAT16_TILES)
      if (!tiles(s, ld, ld, t, 1)) return false;
  }
  for (int pad = 0; pad <= 12 && s.K % 4 == 0; pad += 12) {    // float32: row strides K and K + 12
    const long ld = s.K + pad;
    if (s.M <= 32) {
      if (!float32_rows(s, ld, ld, 2, 4, 1) || !float32_rows(s, ld, ld, 2, 8, 2) || !float32_rows(s, ld, ld, 1, 8, 2) || !float32_rows(s, ld, ld, 1, 16, 2)) return false;
    } else {
      for (const Tiles& t : FLOAT32_TILES)
        if (!tiles(s, ld, ld, t, 2)) return false;
      for (const Tiles& t : FLOAT32_PARTS)
        if (!parts(s, ld, ld, t)) return false;
    }
  }
  if (s.N % 16 == 0 && s.K % 64 == 0) {                // the streaming copy of the weights
    if (s.M <= 32 && !skinny(s, s.K, s.K, 1, 2, A::KSTEP)) return false;
    if (s.M <= 16 && !skinny(s, s.K, s.K, 1, 4, 4 * A::KSTEP)) return false;
    if (s.M > 16 && s.M <= 128 && !ring(s, s.K, s.K, 1)) return false;
    if (s.M <= 16 && (!few_rows(s, s.K) || !few_rows(s, s.K + 8))) return false;
  }
  return true;
}

int main(int argc, char** argv) {
  std::vector<Shape> shapes;
  int a = 1;
  bool sweep = true;
  if (a < argc && !std::strcmp(argv[a], "old-standin")) { old_standin = true; ++a; }
  if (a < argc && !std::strcmp(argv[a], "only")) { sweep = false; ++a; }
  for (; a + 3 < argc; a += 4) shapes.push_back(Shape{std::atoi(argv[a]), std::atoi(argv[a + 1]), std::atoi(argv[a + 2]), std::atoi(argv[a + 3])});
  const int Ms[] = {1, 2, 7, 8, 9, 16, 17, 31, 32, 33, 48, 64, 65, 100, 128, 129, 300};
  const int Ns[] = {1, 16, 31, 32, 33, 64, 100, 520, 2048};
  const int Ks[] = {4, 8, 16, 36, 64, 72, 96, 100, 128, 160, 200, 256, 272, 344, 512, 516, 1024, 2816};
  const int Ss[] = {1, 2, 3, 4, 8};
  for (int M : Ms)
    if (sweep)
    for (int N : Ns)
      for (int K : Ks)
        for (int S : Ss)
          if (S == 1 || K / S >= 4) shapes.push_back(Shape{M, N, K, S});
  for (const Shape& s : shapes)
    if (!check(s)) return 1;
  if (sweep)
    for (int hd = 16; hd <= 256; hd += 16)
      for (int page_size : {16, 32, 48, 64})
        for (int nkv : {1, 3, 8})
          if (!attention(hd, page_size, nkv, 7)) return 1;
  std::printf("ok %ld\n", fetches);
  return 0;
}
