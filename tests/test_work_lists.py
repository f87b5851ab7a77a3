"""Host-side work lists of the kernels (no GPU needed)."""
import random

import numpy as np
import pytest

from photon_infer_amd.ops.fast import (MAX_TILE_CUTS, AttentionPlanner, cut_count, deal_tiles, decode_length_bucket,
                                        decode_splits)


@pytest.mark.parametrize("seed", range(5))
def test_every_tile_is_dealt_exactly_once(seed):
    rng = random.Random(seed)
    walks = [rng.randint(1, 40) for _ in range(rng.randint(1, 300))]
    seats = rng.randint(1, 70)
    order = deal_tiles(walks, seats)
    assert order.shape[1] == seats and order.dtype == np.int32
    dealt = sorted(int(t) for t in order.reshape(-1) if t >= 0)
    assert dealt == list(range(len(walks)))


def test_the_deal_evens_out_the_work():
    # a causal prompt: tile i walks i + 1 key ranges
    walks = list(range(1, 129))
    order = deal_tiles(walks, 32)
    sums = [sum(walks[t] for t in order[:, seat] if t >= 0) for seat in range(32)]
    assert max(sums) - min(sums) <= 1
    # the first round holds the longest tiles
    assert sorted(walks[t] for t in order[0]) == list(range(97, 129))


def prompt_walks(lens, rows, keys):
    """What the tiles of ``rows`` tokens of whole prompts walk, in rounds of so many keys."""
    return [(min(start + rows, n) - 1) // keys + 1 for n in lens for start in range(0, n, rows)]


@pytest.mark.parametrize("lens,rows,keys,seats", [([1501, 1126], 4, 64, 256), ([2048], 32, 128, 24), ([90, 700, 31], 8, 64, 40), ([300], 4, 64, 74), ([1000, 900], 16, 128, 50)])
def test_the_longest_tile_of_a_round_goes_to_the_block_with_least(lens, rows, keys, seats):
    walks = prompt_walks(lens, rows, keys)
    order = deal_tiles(walks, seats)
    work = np.where(order >= 0, np.asarray(walks)[order], 0)
    sums = np.zeros(seats, np.int64)
    for got in work:
        for least in np.unique(sums)[:-1]:            # who has more so far gets no longer tile than who has less
            assert got[sums > least].max() <= got[sums <= least].min()
        sums += got
    assert sums.sum() == sum(walks)


def test_a_last_round_that_is_not_full_does_not_fall_to_the_blocks_with_the_longest_tiles():
    """Dealt back and forth the longest block of these prompts walked 36 rounds, 28 being the mean."""
    order = deal_tiles(walks := prompt_walks([1501, 1126], 4, 64), 256)
    assert np.where(order >= 0, np.asarray(walks)[order], 0).sum(0).max() <= 32


def test_fewer_tiles_than_seats():
    order = deal_tiles([3, 9], 8)
    assert order.shape == (1, 8)
    assert list(order[0][:2]) == [1, 0] and all(t == -1 for t in order[0][2:])


def test_decode_splits_fill_the_chip_but_respect_short_contexts():
    assert decode_splits(64, 8, 4096) < decode_splits(8, 8, 4096) <= 32
    assert decode_splits(1, 8, max_kv_len=100) == 1
    assert decode_splits(1, 8, max_kv_len=4096) > 1
    # the same key ranges anywhere inside a length bucket: eager steps and graph replays agree
    assert decode_length_bucket(129) == decode_length_bucket(256) == 256
    assert decode_splits(4, 8, 1025) == decode_splits(4, 8, 2048)


def test_key_ranges_of_tiles_are_cut_only_when_the_tiles_are_few():
    assert cut_count([], 64) == 1
    assert cut_count([20] * 64, 64) == 1 and cut_count([20] * 33, 64) == 1      # enough tiles: none is cut
    assert cut_count([64] * 16, 64) == 4                                        # 16 tiles, 64 blocks wanted
    assert cut_count([64] * 2, 64) == MAX_TILE_CUTS
    assert cut_count([5] * 16, 64) == 1 and cut_count([7] * 2, 64) == 1         # a share keeps four rounds at least
    assert cut_count([12] * 4, 64) == 3
    assert cut_count([8] * 8, 64) == 1 and cut_count([9] * 16, 64) == 1         # ... and the cut saves six rounds or it is not made
    assert cut_count([16] * 16, 64) == 4
    assert cut_count([1] * 4, 64) == 1


@pytest.mark.parametrize("seed", range(6))
def test_a_step_plan_covers_every_token_of_every_portion_once(seed):
    """The planner of the prompt-attention kernel, on the host: tiles (or the shares of a cut tile)
    cover each token of each portion exactly once; requests with one token go to the other kernel
    when the planner says so; every entry is dealt to a block exactly once."""
    rng = random.Random(seed)
    R = rng.randint(1, 6)
    q_lens = [rng.choice([1, 1, 2, 17, 64, 65, 300]) for _ in range(R)]
    if all(n == 1 for n in q_lens):
        q_lens[0] = 40
    kv_lens = [n + rng.choice([0, 5, 700, 3000]) for n in q_lens]
    apart = seed % 2 == 0
    planner = AttentionPlanner(tile_rows=rng.choice([16, 32, 64]), window=rng.choice([0, 0, 100]), num_kv_heads=2,
                               singles_apart=apart, units=rng.choice([8, 256]))
    arrays, finish = planner.plan(q_lens, kv_lens)
    assert all(a.dtype == np.int32 for a in arrays.values())
    singles = [r for r, n in enumerate(q_lens) if n == 1] if apart else []
    assert arrays["singles"].tolist() == singles
    n = len(arrays["req"])
    assert len(arrays["q0"]) == len(arrays["cut"]) == len(arrays["z0"]) == n
    covered = {}
    for r, q0, cut in zip(arrays["req"].tolist(), arrays["q0"].tolist(), arrays["cut"].tolist()):
        share, shares = cut & 0xff, cut >> 8
        assert 0 <= share < shares and r not in singles
        covered.setdefault((r, q0), []).append((share, shares))
    for (r, q0), shares in covered.items():
        assert q0 % planner.tile_rows == 0 and q0 < q_lens[r]
        assert sorted(s for s, _ in shares) == list(range(shares[0][1]))          # every share of a cut tile, once
    for r, qn in enumerate(q_lens):
        if r not in singles:
            assert sorted(q0 for (rr, q0) in covered if rr == r) == list(range(0, qn, planner.tile_rows))
    dealt = sorted(t for t in arrays["order"].tolist() if t >= 0)
    assert dealt == list(range(n))
    # rows of the cut tiles: one entry per token of every cut tile
    cut_rows = sum(min(planner.tile_rows, q_lens[r] - q0) for (r, q0), sh in covered.items() if sh[0][1] > 1)
    assert len(arrays["rows"]) == cut_rows


def test_steps_of_single_tokens_need_no_plan_unless_the_tile_kernel_serves_them():
    assert AttentionPlanner(16, 0, 2, True, 256).plan([1, 1, 1], [5, 900, 17]) is None
    arrays, _ = AttentionPlanner(16, 0, 2, False, 256).plan([1, 1, 1], [5, 900, 17])
    assert arrays["req"].tolist()[:3] == [0, 1, 2] or sorted(set(arrays["req"].tolist())) == [0, 1, 2]
    assert arrays["singles"].size == 0


def test_pieces_that_would_not_fit_the_workspace_are_refused():
    """The kernels write a split product's pieces without knowing the buffer's size: the host
    refuses a request beyond it, and the split rules never make one."""
    from photon_infer_amd.errors import KernelError
    from photon_infer_amd.ops import fast
    from photon_infer_amd.ops.workspace import GEMM_PART_FLOATS, KernelWorkspace
    with pytest.raises(KernelError, match="workspace holds"):
        fast._piece_buffer(KernelWorkspace("cpu"), GEMM_PART_FLOATS + 1, "cpu")
    for M, N, K in [(2048, 2048, 8192), (2048, 3072, 8192), (2048, 4096, 14336), (8192, 4096, 14336), (4096, 8192, 28672),
                    (512, 4096, 14336), (100000, 128, 4096), (129, 128256, 2048)]:
        assert fast._tile_splits(M, N, K) * M * N <= GEMM_PART_FLOATS or fast._tile_splits(M, N, K) == 1
    for M, N, K in [(8, 128256, 2048), (128, 128256, 8192), (64, 16384, 2048), (1, 2048, 8192)]:
        assert fast._skinny_splits(M, N, K) * M * N <= GEMM_PART_FLOATS or fast._skinny_splits(M, N, K) == 1


@pytest.mark.parametrize("M", [17, 32])
def test_k_is_cut_for_the_kernel_that_a_product_of_17_to_32_tokens_takes(monkeypatch, M):
    """On both sides of the line, and with rows so far apart that the kernel that shares activations does not take them."""
    import torch

    from photon_infer_amd.ops import fast
    monkeypatch.setattr(fast, "compute_units", lambda: 256)
    made = []
    monkeypatch.setattr(fast, "_skinny", lambda *args: made.append(args[10]))

    def pieces(N, K, lda, ldw):
        a, w = (torch.empty_strided((rows, K), (stride, 1), dtype=torch.bfloat16) for rows, stride in ((M, lda), (N, ldw)))
        assert fast.gemm(torch.empty(M, N), a, w, False, M, N, K, lda, ldw, N)
        return made.pop()

    long = fast.RING_MAX_STRIDE
    assert pieces(5120, 4096, 4096, 4096) == pieces(5120, 4096, long - 8, 4096) == 3       # 80 blocks of 64 rows: one per unit
    assert pieces(5120, 4096, long, 4096) == 4                                             # 160 blocks of 32 rows: two per unit
    assert pieces(4872, 4096, 4096, 4096) == 4                                             # 19.96 million elements
    assert pieces(8, 2560000, 2560000, 2560000) == 512                                     # k too long as well


# (requests' tokens, contexts, heads, kv heads, head size, window, microseconds on the tile kernel, on the general kernel), measured
FLOAT32_STEPS = [
    ([32], [2048], 32, 8, 64, 0, 150, 127), ([32], [32768], 32, 8, 64, 0, 2316, 1687), ([32], [32768], 24, 8, 128, 0, 3604, 2452),
    ([1] * 31 + [33], [2000] * 32, 24, 8, 128, 0, 590, 451), ([1] * 63 + [16], [4000] * 64, 24, 8, 128, 0, 2155, 1302), ([2] * 16, [4000] * 16, 24, 8, 128, 0, 732, 409),
    ([64], [8192], 32, 8, 64, 0, 581, 1076), ([256], [8192], 24, 8, 128, 0, 912, 5003), ([1] * 8 + [64], [16000] * 9, 32, 8, 64, 0, 1147, 2562),
    ([1] * 31 + [128], [2000] * 32, 32, 8, 64, 0, 234, 680), ([517, 431, 345], [517, 431, 345], 32, 8, 64, 0, 64, 462),
]


@pytest.mark.parametrize("step", FLOAT32_STEPS, ids=[f"step{i}" for i in range(len(FLOAT32_STEPS))])
def test_the_float32_path_takes_the_attention_kernel_that_was_the_faster_one(step):
    from photon_infer_amd.ops import fast
    q_lens, kv_lens, heads, kv_heads, head_dim, window, tiles, general = step
    tile_tokens = 64 if heads // kv_heads % 2 else 16
    tiles_us, general_us = fast.float32_attention_us(q_lens, kv_lens, heads, kv_heads, head_dim, tile_tokens, window)
    assert (tiles_us < fast.FLOAT32_TILES_WORTH * general_us) == (tiles < general)
    assert 0.6 < tiles_us / tiles < 1.6 and 0.5 < general_us / general < 1.6       # and the estimates are of that size


# (rows, columns, k), {pieces of k: microseconds of a float32 product with the norm that adds them}, measured (the row of 129 on the tiles in
# parts: 8 pieces took 75.9 us by float32 instructions)
FLOAT32_PIECES = [
    (8, 2048, 2048, {1: 12.4, 4: 10.2, 8: 10.3, 16: 12.8}), (24, 2048, 2048, {1: 14.8, 4: 12.4, 8: 12.3, 16: 15.8}), (24, 3072, 2048, {1: 15.5, 3: 17.6, 5: 15.7, 8: 15.6}),
    (8, 3072, 768, {1: 9.8, 3: 10.9}), (24, 3072, 768, {1: 10.6, 2: 11.6, 3: 11.7}), (32, 4096, 512, {1: 10.3, 2: 11.1}), (24, 5120, 3072, {1: 37.0, 3: 24.8}),
    (129, 2048, 8192, {5: 64.5, 8: 57.3}), (1000, 256, 512, {1: 16.7, 2: 12.5}), (1050, 6144, 4096, {1: 351.6, 2: 386.4}), (500, 6144, 4096, {4: 179.9, 5: 184.4}),
]


@pytest.mark.parametrize("M,N,K,times", FLOAT32_PIECES)
def test_a_float32_product_is_left_in_as_many_pieces_as_were_the_fastest(M, N, K, times):
    from photon_infer_amd.ops import _lib, fast
    made = _lib.load("core").pi_gemm_float32_pieces(M, N, K, fast.GEMM_PART_FLOATS, 1)
    assert times[made] <= 1.05 * min(times.values())


# (rows, features, k), microseconds of the gated unit in the float32 product, and of product and unit, measured (from 100 rows on, on the
# tiles in parts where they are taken: by float32 instructions alone 500 x 1,536 x 2,048 76.0 and 80.1, 900 x 4,096 x 512 77.6 and 83.8)
FLOAT32_GATED = [
    (64, 1024, 4096, 85.4, 21.5), (200, 1024, 4096, 86.3, 38.7), (32, 1024, 4096, 30.6, 23.0), (24, 2048, 2048, 18.5, 15.4), (33, 512, 512, 15.9, 13.0),
    (8, 8192, 4096, 65.0, 68.1), (8, 512, 512, 7.0, 7.2), (2, 1024, 2048, 12.7, 10.3), (1, 4096, 8192, 80.3, 57.9), (1, 8192, 2048, 26.9, 28.8), (1, 2048, 1024, 9.0, 10.0),
    (16, 3072, 2048, 16.1, 20.7), (32, 3072, 1024, 12.7, 17.2), (24, 256, 1024, 11.8, 10.0), (500, 1536, 2048, 75.5, 54.2), (900, 4096, 512, 59.1, 61.4), (100, 8192, 3072, 117.1, 89.0),
]


@pytest.mark.parametrize("M,I,K,whole,two", FLOAT32_GATED)
def test_the_float32_gated_unit_is_part_of_the_product_where_that_was_the_faster_way(M, I, K, whole, two):
    from photon_infer_amd.ops import fast
    took = whole if fast.float32_gate_in_product(M, 2 * I, K, 256) else two
    assert took <= 1.03 * min(whole, two)


# (rows, columns, k), {tile shape: microseconds of the product in one piece}, bfloat16 results, weights cold, measured; 0 is the faster kernel of 128 x 128
SHAPES_MEASURED = [
    (543, 28672, 4096, {0: 175.5, 42: 174.4, 33: 121.9, 32: 149.8, 23: 189.0, 22: 163.4}),
    (2048, 16384, 2048, {0: 147.4, 42: 111.8, 33: 124.7, 32: 126.0, 23: 155.1, 22: 134.6}),
    (384, 3072, 2048, {0: 17.8, 42: 38.4, 33: 44.4, 32: 32.0, 23: 34.3, 22: 25.0}),
    (2048, 2048, 8192, {0: 71.2, 42: 141.9, 33: 180.6, 32: 120.5, 23: 172.7, 22: 94.8}),
    (200, 4096, 14336, {0: 116.6, 42: 265.6, 33: 324.5, 32: 204.2, 23: 314.2, 22: 178.7}),
    (1150, 28672, 4096, {0: 272.6, 42: 277.0, 33: 232.4, 32: 239.3, 23: 294.0, 22: 244.7}),
    (1000, 5120, 3072, {0: 56.9, 42: 63.1, 33: 76.6, 32: 51.0, 23: 74.0, 22: 45.3}),
    (850, 6144, 4096, {0: 60.3, 42: 74.2, 33: 96.9, 32: 65.6, 23: 92.7, 22: 53.9}),
    (2048, 4096, 4096, {0: 68.0, 42: 78.6, 33: 97.7, 32: 69.0, 23: 93.7, 22: 62.1}),
    (200, 28672, 4096, {0: 78.7, 42: 89.1, 33: 109.5, 32: 78.0, 23: 105.2, 22: 68.3}),
    (2627, 3072, 2048, {0: 34.4, 42: 41.3, 33: 47.1, 32: 36.6, 23: 38.4, 22: 33.6}),
    (300, 16384, 3072, {0: 51.6, 42: 61.3, 33: 81.4, 32: 55.2, 23: 75.9, 22: 46.2}),
    (3000, 16384, 3072, {0: 311.1, 42: 240.0, 33: 268.8, 32: 254.4, 23: 317.5, 22: 281.9}),
]


@pytest.mark.parametrize("M,N,K,times", SHAPES_MEASURED)
def test_tile_shapes_follow_the_rounds_they_take(M, N, K, times):
    from photon_infer_amd.ops import fast
    assert times[fast._tile_shape_of(M, N, K, 1, 256)] <= 1.03 * min(times.values())


def test_a_k_that_is_no_whole_slabs_takes_the_only_kernel_for_it():
    from photon_infer_amd.ops import fast
    assert fast._tile_shape_of(300, 200, 1000, 1, 256) == 0 and fast._tile_shape_of(2048, 16384, 2040, 1, 256) == 0


# (rows, columns, k), microseconds of the product in one, two, ... pieces with the norm that adds them, each in its fastest tile shape, weights cold, measured
PIECES_MEASURED = [
    (130, 2048, 2048, [22.9, 15.8, 14.5, 14.0, 14.3, 14.4, 14.5, 14.8]), (200, 2048, 2048, [23.0, 16.5, 15.7, 15.3, 15.8, 16.3, 16.7, 17.2]),
    (300, 2048, 2048, [24.2, 18.4, 18.0, 18.3, 19.1, 19.8, 20.5, 20.7]), (130, 2048, 8192, [65.4, 37.6, 28.6, 24.8, 22.4, 21.2, 20.2, 20.7]),
    (300, 2048, 8192, [67.8, 40.6, 31.7, 28.4, 26.3, 30.4, 29.2, 28.1]), (2048, 2048, 8192, [84.2, 79.9, 81.9, 81.2]),
    (1500, 2048, 8192, [75.1, 67.1, 65.8, 64.6, 67.1]), (256, 4096, 4096, [47.4, 29.7, 25.7, 23.8, 26.4, 25.8, 26.4, 27.8]),
    (1000, 4096, 4096, [53.7, 51.9, 55.2, 57.9]), (2048, 2048, 2048, [34.7, 37.5, 41.5, 44.4]),
    (200, 4096, 14336, [124.6, 68.9, 52.7, 44.8, 53.0, 48.5, 47.8, 45.5]), (543, 4096, 14336, [119.3, 101.9, 82.7, 82.3, 77.5, 93.0, 88.3]),
    (700, 1024, 1024, [17.9, 15.3, 16.0, 16.8]), (300, 3072, 3072, [35.2, 24.7, 22.6, 24.6, 24.3, 23.9, 24.1, 26.9]),
    (1150, 3072, 3072, [42.2, 41.9, 44.3, 49.3]), (2627, 2048, 2048, [42.4, 46.2, 53.2]), (1267, 5376, 4544, [114.2, 174.3]),
    (850, 6144, 4096, [89.2, 111.1, 120.6]), (700, 3072, 2048, [30.7, 28.4, 27.6, 29.9, 31.3, 34.1, 36.4]),
    (1000, 2080, 2048, [31.1, 28.4, 27.2, 30.9, 32.0, 34.5, 36.4, 42.2]), (2627, 832, 2048, [30.5, 28.2, 28.1, 31.2, 33.4, 35.5, 41.8]),
]


@pytest.mark.parametrize("M,N,K,times", PIECES_MEASURED)
def test_a_product_is_left_in_as_many_pieces_as_were_the_fastest(M, N, K, times):
    from photon_infer_amd.ops import fast
    assert times[fast._tile_splits_of(M, N, K, 256, 1.0) - 1] <= 1.05 * min(times)


@pytest.mark.parametrize("N,K,tokens", [(3072, 2048, 1280), (5120, 3072, 1152), (6144, 4096, 1280), (2560, 1024, 1536), (4608, 3584, 1536), (4096, 2560, 1280),
                                        (9216, 4096, 896), (10240, 8192, 1536), (2048, 2048, 2048), (8256, 4096, 128), (16320, 512, 128)])
def test_queries_keys_and_values_of_some_hundred_tokens_reach_the_rotation_in_float32(N, K, tokens):
    """Cut over k or not: from 33 tokens on as long as the result has no more tiles than the chip has units, more with a longer k."""
    from photon_infer_amd.ops import fast
    for M in range(33, tokens + 1):
        cut = fast._skinny_splits_of(M, N, K, 256) if M <= fast.SKINNY_MAX_ROWS else fast._tile_splits_of(M, N, K, 256, fast.PIECES_WORTH, norm=False)
        assert cut > 1 or fast.keeps_float32(M, N, K, 256), M


def test_a_token_count_that_was_not_seen_before_costs_little_to_plan(monkeypatch):
    """In continuous batching the token count changes nearly every step.  Four products of a 1B layer, planned for counts that
    no step had: 13 microseconds in the library (135 in Python), the best of several rounds taken for a busy machine."""
    import time

    from photon_infer_amd.ops import fast
    monkeypatch.setattr(fast, "compute_units", lambda: 256)
    best, M = float("inf"), 10007
    for _ in range(8):
        start = time.perf_counter()
        for M in range(M + 1, M + 21):
            for N, K in ((3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192)):
                fast._tile_shape(M, N, K, fast._tile_splits(M, N, K))
        best = min(best, (time.perf_counter() - start) / 20)
    assert best < 60e-6


# (key ranges, requests, kv heads, longest context, head size) -> waves per block, as measured: a step of contexts of one length
# must lose nothing, so waves that replace no ranges go to two full rounds of blocks only (and, on the device, to uneven lengths)
@pytest.mark.parametrize("splits,R,kv_heads,longest,head_dim,waves", [
    (1, 64, 8, 4000, 64, 2), (1, 64, 8, 4000, 128, 2), (1, 128, 4, 4000, 64, 2), (1, 64, 8, 1000, 64, 2), (1, 64, 8, 1000, 128, 1), (1, 64, 8, 300, 64, 1),
    (1, 80, 8, 4096, 64, 1), (1, 96, 8, 4096, 128, 1), (1, 96, 8, 600, 128, 1), (1, 128, 8, 4096, 64, 1), (2, 48, 8, 4096, 64, 1), (2, 48, 8, 1024, 64, 2),
    (2, 32, 8, 4096, 128, 2), (2, 56, 8, 4096, 64, 2), (3, 24, 8, 4096, 64, 4), (2, 40, 8, 4096, 64, 1), (4, 16, 8, 4096, 64, 1)])
def test_waves_share_a_request_where_that_was_the_faster_way(splits, R, kv_heads, longest, head_dim, waves):
    from photon_infer_amd.ops import fast
    assert fast.decode_block_waves(splits, R, kv_heads, longest, head_dim) == waves


def test_uneven_lengths():
    from photon_infer_amd.ops import lengths_uneven
    assert not lengths_uneven([4096] * 64) and not lengths_uneven([4000 - 10 * i for i in range(64)])
    assert lengths_uneven([4000 - 30 * i for i in range(64)]) and lengths_uneven(np.asarray([500] * 63 + [4000], np.int32))
    assert not lengths_uneven([1, 4000])             # a small batch: its ranges may go on to the next product


def test_waves_of_bounded_contexts_and_of_steps_that_do_not_know_their_lengths():
    """Windows and chunks: the lengths do not say what is seen.  The answer is the same for a step and for its length bucket's graph."""
    from types import SimpleNamespace

    import torch

    from photon_infer_amd.ops import fast
    flag = torch.zeros(1, dtype=torch.int32)
    ctx, bare = SimpleNamespace(uneven=flag), SimpleNamespace()
    assert fast._waves_or_ranges(ctx, 1, 64, 8, 64, 3000, 0) == (1, 2, flag.data_ptr())
    assert fast._waves_or_ranges(bare, 1, 64, 8, 64, 3000, 0) == (1, 1, None)
    for bound in (1024, 2500, 3500):
        assert fast._waves_or_ranges(ctx, 1, 64, 8, 64, 3000, bound) == fast._waves_or_ranges(ctx, 1, 64, 8, 64, 4096, bound) == (1, 1, None)
    assert fast._waves_or_ranges(ctx, 1, 64, 8, 64, 3000, 4096) == (1, 2, flag.data_ptr())
    assert fast._waves_or_ranges(bare, 2, 32, 8, 64, 3000, 0) == (1, 2, None) and fast._waves_or_ranges(ctx, 2, 40, 8, 64, 3000, 0) == (2, 1, None)
    for uneven in (False, True):
        assert fast._waves_or_ranges(ctx, 1, 64, 8, 64, 3000, 0, SimpleNamespace(singles_uneven=uneven)) == (1, 1 + uneven, None)


@pytest.mark.parametrize("splits,R,kv_heads,made", [(1, 16, 8, (1, 1)), (31, 1, 8, (31, 1)), (32, 1, 8, (16, 2)), (64, 1, 8, (32, 2)), (64, 1, 9, (64, 1)), (15, 2, 8, (15, 1)),
                                                    (16, 2, 8, (8, 2)), (32, 2, 8, (16, 2)), (22, 3, 8, (22, 1)), (20, 3, 8, (10, 2)), (8, 4, 8, (4, 2)), (16, 4, 8, (8, 2)),
                                                    (16, 4, 9, (16, 1)), (8, 5, 1, (8, 1)), (8, 8, 8, (8, 1)), (4, 16, 8, (4, 1))])
def test_ranges_of_all_requests_from_which_on_two_waves_share_one(splits, R, kv_heads, made):
    """As it was the faster way: few requests, enough ranges, and one round of blocks (256 units)."""
    from photon_infer_amd.ops import fast
    assert fast.decode_range_waves(splits, R, kv_heads) == made
    assert made[0] * made[1] >= splits


def test_key_ranges_of_float32_decode_steps():
    """One range up to short buckets, then blocks that fill the chip, ranges that keep their keys, and no more than the merging
    kernel takes; the same within a length bucket."""
    from photon_infer_amd.ops import fast
    ranges = fast.float32_decode_ranges
    assert [ranges(1, 8, 64, n) for n in (1, 256, 257, 512, 513, 1024, 8192, 8193, 1 << 20)] == [1, 1, 4, 4, 8, 8, 64, 64, 64]
    assert [ranges(R, 8, 64, 4000) for R in (1, 4, 5, 8, 16, 64, 128, 129, 1000)] == [32, 32, 25, 16, 8, 2, 1, 1, 1]
    assert [ranges(R, 8, 128, 4000) for R in (1, 2, 3, 8, 64)] == [32, 32, 21, 8, 1]


def test_products_that_the_finishing_kernel_takes():
    """Sizes at the edges of its rules, of which the host side answers without a GPU (256 units)."""
    from photon_infer_amd.ops import fast
    blocks = lambda *a: fast._finish_blocks.__wrapped__(*a)
    assert [blocks(M, 2048, 2048) for M in (0, 1, 16, 17)] == [0, 256, 256, 0]
    assert [blocks(1, N, 2048) for N in (48, 64, 96, 3008, 3072, 8192, 8256)] == [0, 8, 0, 376, 192, 512, 0]
    assert [blocks(1, 2048, K) for K in (32, 64, 96, 4096, 4160)] == [0, 256, 0, 256, 256]
    assert [blocks(M, 2048, K) for M, K in ((12, 4160), (13, 4096), (13, 4160))] == [256, 256, 0] and blocks(16, 3072, 8192) == 192
    assert [blocks(M, N, 5120) for M, N in ((12, 5120), (13, 5120), (16, 4096), (16, 4160), (16, 8192))] == [320, 0, 256, 0, 512]
    ranges = lambda *a: fast._finish_ranges_blocks.__wrapped__(*a)
    # M, N, heads, head size, ranges: one token, at most 16 ranges and 144 KB, 64 KB of LDS, blocks of 8 rows
    assert [ranges(1, 2048, 32, 64, c) for c in (0, 1, 16, 17)] == [0, 256, 256, 0] and [ranges(M, 2048, 32, 64, 2) for M in (1, 2, 16)] == [256, 0, 0]
    assert [ranges(1, 2048, 32, 128, c) for c in (8, 9)] == [256, 0]
    assert ranges(1, 3072, 32, 64, 2) == 0 and ranges(1, 2048, 32, 60, 2) == 0 and [ranges(1, 2048, h, 64, 1) for h in (64, 65)] == [256, 0]
