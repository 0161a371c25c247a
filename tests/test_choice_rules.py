"""Which kernel the size rules pick for every BASELINE configuration, pinned on the CPU (the query functions are plain
integer arithmetic when the number of compute units is passed in). A change of a rule that moves a configuration onto
another kernel has to show up here, next to the GPU parity test that covers that kernel:
  1D kernels (numbering of turbofno_set_1d_algo): 1 SIMT, 2 / 3 matrix cores with 512- / 256-thread blocks, 4 matrix
  cores with 32-channel output tiles, 5 as 3 for four blocks per CU (one wavefront per item for eight channels of length
  128), 6 K split over the waves of a block, 7 K split over a cluster of blocks (only with an exchange buffer attached),
  8 as 3 with 64 or 128 output channels per block;
  2D algorithms: 1 three kernels (X axis first), 2 whole image, 3 three kernels (rows first).
GPU parity of each: tests/test_gpu_parity.py (every selector forced), tests/test_gpu_fullsize.py (the configurations at
full size), tests/test_gpu_cluster.py (7), tests/test_gpu_large_grids.py."""
import os
import subprocess

import turbofno_amd as tf

CUS = 256       # MI355X


def test_1d_kernel_of_configuration_1():
    assert tf.query_1d_kernel(128, 1, 64, 8, CUS) == 4


def test_1d_kernels_of_configuration_2():
    # 112 problems, all of them at most one block per CU: matrix cores, eight waves per block, 32-channel output tiles
    for bs in (1, 2, 4, 8, 16, 32, 64):
        for DY in (128, 256):
            for N in (64, 128):
                for K in (8, 16, 24, 32):
                    assert tf.query_1d_kernel(DY, bs, N, K, CUS) == 4, (bs, DY, N, K)


def test_1d_kernels_of_configuration_3():
    for K, without in ((64, 4), (128, 6)):
        assert tf.query_1d_kernel(256, 64, 128, K, CUS, exchange_attached=True) == 7
        assert tf.query_1d_kernel(256, 64, 128, K, CUS, exchange_attached=False) == without


def test_1d_k_split_is_named_where_it_runs():
    """more than 96 channels, blocks of 32 output channels for more than half of the CUs and at most one each; the query names the
    small-grid kernel, and its tile, everywhere else"""
    for N in (64, 128, 192, 256):
        most = CUS // (N // 32)
        for K in (104, 112, 128, 136):
            assert tf.query_1d_kernel(256, most, N, K, CUS) == 6 and tf.query_1d_tile(256, most, N, K, CUS) == 32, (N, K)
            assert tf.query_1d_kernel(256, most // 2 + 1, N, K, CUS) == 6, (N, K)
            assert tf.query_1d_kernel(256, most // 2, N, K, CUS) == 4 and tf.query_1d_tile(256, most // 2, N, K, CUS) == 16, (N, K)
            assert tf.query_1d_kernel(256, most + 1, N, K, CUS) == 2, (N, K)
        for K in (64, 72, 80, 88, 96):
            assert tf.query_1d_kernel(256, most, N, K, CUS) == 4, (N, K)
    assert tf.query_1d_kernel(256, 1, 64, 64, CUS) == 4 and tf.query_1d_tile(256, 1, 64, 64, CUS) == 16


def test_2d_algorithms_of_configurations_4_and_5():
    for D in (128, 256):
        for K in (16, 32):
            assert tf.query_2d_algo(1, D, D, K, 64) == tf.ALGO_THREE_KERNEL
            assert tf.query_2d_algo(4, D, D, K, 64) == tf.ALGO_THREE_KERNEL
            assert tf.query_2d_algo(16, D, D, K, 64) == tf.ALGO_WHOLE_IMAGE
    assert tf.query_2d_algo(16, 256, 256, 64, 64) == tf.ALGO_WHOLE_IMAGE          # the headline problem


def test_large_grids_and_long_axes():
    # the reference's own benchmark regime: thousands of signals per channel
    assert tf.query_1d_kernel(256, 4096, 64, 64, CUS) == 3
    assert tf.query_1d_kernel(256, 4096, 128, 64, CUS) == 8
    assert tf.query_1d_kernel(128, 4096, 64, 64, CUS) == 5
    assert tf.query_1d_kernel(128, 4096, 128, 128, CUS) == 8
    assert tf.query_1d_kernel(512, 4096, 64, 32, CUS) == 1
    # axes above 256, small problems: three stages, the longer axis (or, for squares with enough images, the contiguous
    # one) first
    assert tf.query_2d_algo(2, 512, 512, 64, 64) == tf.ALGO_ROWS_FIRST
    assert tf.query_2d_algo(1, 512, 512, 32, 64) == tf.ALGO_THREE_KERNEL
    assert tf.query_2d_algo(8, 256, 1024, 32, 64) == tf.ALGO_ROWS_FIRST
    assert tf.query_2d_algo(4, 1024, 256, 32, 64) == tf.ALGO_THREE_KERNEL
    assert tf.query_2d_algo(2, 1024, 1024, 32, 64) == tf.ALGO_ROWS_FIRST
    # large ones: the whole-image kernels (512 / 1024 rows as interleaved parts of 256, long rows with 32 / 64 lanes),
    # from a volume of input and output that depends on the lengths
    assert tf.query_2d_algo(16, 512, 512, 32, 64) == tf.ALGO_WHOLE_IMAGE
    assert tf.query_2d_algo(4, 512, 512, 32, 64) == tf.ALGO_WHOLE_IMAGE            # 768 MiB
    assert tf.query_2d_algo(4, 512, 512, 16, 64) == tf.ALGO_THREE_KERNEL           # 640 MiB
    assert tf.query_2d_algo(16, 512, 256, 32, 64) == tf.ALGO_WHOLE_IMAGE
    assert tf.query_2d_algo(4, 512, 256, 32, 64) == tf.ALGO_THREE_KERNEL           # 384 MiB
    assert tf.query_2d_algo(16, 512, 128, 32, 64) == tf.ALGO_WHOLE_IMAGE
    assert tf.query_2d_algo(8, 512, 128, 32, 64) == tf.ALGO_THREE_KERNEL
    assert tf.query_2d_algo(16, 256, 512, 32, 64) == tf.ALGO_WHOLE_IMAGE
    assert tf.query_2d_algo(8, 1024, 256, 32, 64) == tf.ALGO_WHOLE_IMAGE           # 1536 MiB
    assert tf.query_2d_algo(4, 1024, 256, 32, 64) == tf.ALGO_THREE_KERNEL          # 768 MiB
    assert tf.query_2d_algo(16, 256, 1024, 32, 64) == tf.ALGO_WHOLE_IMAGE          # 3072 MiB
    assert tf.query_2d_algo(8, 256, 1024, 32, 64) == tf.ALGO_ROWS_FIRST            # 1536 MiB
    assert tf.query_2d_algo(16, 1024, 1024, 32, 64) == tf.ALGO_WHOLE_IMAGE
    assert tf.query_2d_algo(4, 1024, 1024, 32, 64) == tf.ALGO_ROWS_FIRST           # 3072 MiB


def test_2d_algorithms_near_the_lines():
    """small batches with many channels, where the whole-image path is ahead earlier, and the order of the smallest three-stage problems: the last
    shape on each side of a line"""
    three, whole, rows = tf.ALGO_THREE_KERNEL, tf.ALGO_WHOLE_IMAGE, tf.ALGO_ROWS_FIRST
    for bs, DX, DY, K, N, algo in [
            (5, 128, 128, 112, 64, three), (5, 128, 128, 120, 64, whole), (6, 128, 128, 64, 128, three), (6, 128, 128, 72, 128, whole),
            (3, 128, 256, 40, 64, three), (3, 128, 256, 48, 64, whole), (2, 128, 256, 128, 64, whole), (2, 128, 256, 136, 64, three),
            (7, 256, 128, 104, 64, three), (7, 256, 128, 112, 64, whole), (3, 256, 256, 80, 64, whole), (3, 256, 256, 88, 64, three),
            (2, 256, 512, 104, 64, rows), (2, 256, 512, 112, 64, whole), (2, 512, 256, 104, 64, three), (2, 512, 256, 112, 64, whole),
            (2, 512, 512, 88, 64, rows), (2, 512, 512, 96, 64, whole), (2, 1024, 256, 104, 64, three), (2, 1024, 256, 112, 64, whole),
            (1, 1024, 512, 104, 64, three), (1, 1024, 512, 112, 64, whole),
            (1, 1024, 1024, 104, 64, rows), (1, 1024, 1024, 112, 64, whole), (1, 1024, 1024, 128, 64, whole), (1, 1024, 1024, 136, 64, rows),
            (1, 1024, 1024, 112, 192, whole), (1, 1024, 1024, 112, 256, rows), (2, 1024, 1024, 104, 128, rows), (2, 1024, 1024, 112, 128, whole),
            (1, 128, 256, 64, 64, rows), (1, 128, 256, 72, 64, three), (2, 128, 256, 24, 64, rows), (2, 128, 256, 32, 64, three),
            (2, 128, 256, 16, 128, rows), (2, 128, 256, 24, 128, three), (2, 128, 256, 8, 192, three), (2, 128, 256, 16, 256, three),
            (3, 128, 256, 8, 64, rows), (3, 128, 256, 16, 64, three),
            (1, 256, 512, 64, 64, three), (1, 256, 512, 72, 64, rows), (1, 512, 1024, 16, 64, three), (1, 512, 1024, 24, 64, rows)]:
        assert tf.query_2d_algo(bs, DX, DY, K, N) == algo, (bs, DX, DY, K, N)


def test_queries_answer_zero_for_arguments_the_calls_refuse():
    assert tf.query_1d_kernel(256, 4, 64, 12, CUS) == 0             # K not a multiple of 8
    assert tf.query_1d_kernel(2048, 4, 64, 8, CUS) == 0             # no kernel of that length
    assert tf.query_1d_kernel(200, 4, 64, 8, CUS) == 0              # not a power of two
    assert tf.query_2d_algo(1, 200, 256, 16, 64) == 0
    assert tf.query_2d_algo(1, 2048, 512, 16, 64, tf.ALGO_WHOLE_IMAGE) == 0
    assert tf.query_2d_algo(1, 256, 256, 16, 60) == 0
    assert tf.query_2d_algo(1, 256, 256, 16, 64, 9) == 0
    # an explicit algorithm is returned as it is
    assert tf.query_2d_algo(1, 256, 256, 16, 64, tf.ALGO_WHOLE_IMAGE) == tf.ALGO_WHOLE_IMAGE
    assert tf.query_2d_algo(1, 512, 1024, 16, 64, tf.ALGO_WHOLE_IMAGE) == tf.ALGO_WHOLE_IMAGE


def test_output_channels_per_block(algo_1d):
    assert tf.query_1d_tile(256, 1, 64, 8, CUS) == 16 and tf.query_1d_tile(256, 64, 64, 8, CUS) == 16
    assert tf.query_1d_tile(256, 65, 64, 8, CUS) == 32 and tf.query_1d_tile(256, 129, 64, 8, CUS) == 64
    assert tf.query_1d_tile(256, 64, 128, 128, CUS) == 32
    assert tf.query_1d_tile(256, 64, 128, 128, CUS, exchange_attached=True) == 128
    assert tf.query_1d_tile(256, 4096, 64, 64, CUS) == 64
    assert tf.query_1d_tile(256, 8192, 128, 128, CUS) == 128
    assert tf.query_1d_tile(256, 1000, 128, 16, CUS) == 64
    assert tf.query_1d_tile(256, 4, 64, 12, CUS) == 0
    for DY in (128, 256, 512, 1024):
        for S in (1, 40, 2048):
            for K in (8, 32, 128):
                algo_1d(8)                      # whatever the size
                assert tf.query_1d_tile(DY, S, 128, K, CUS) == 128 and tf.query_1d_tile(DY, S, 256, K, CUS) == 128
                assert tf.query_1d_tile(DY, S, 64, K, CUS) == 64 and tf.query_1d_tile(DY, S, 192, K, CUS) == 64
                algo_1d(3)
                assert tf.query_1d_tile(DY, S, 128, K, CUS) == 64


def test_1d_kernels_where_the_last_round_or_the_last_blocks_are_nearly_empty():
    assert tf.query_1d_kernel(128, 256, 64, 16, CUS) == 8           # one block of 64 output channels per CU
    assert tf.query_1d_kernel(128, 128, 128, 40, CUS) == 2          # eight of 32 channels in the last round
    assert tf.query_1d_kernel(128, 128, 128, 64, CUS) == 3
    assert tf.query_1d_kernel(1024, 600, 64, 40, CUS) == 1          # two to three blocks per CU, of which two fit at a time
    assert tf.query_1d_kernel(1024, 512, 64, 40, CUS) == 3
    assert tf.query_1d_kernel(1024, 1000, 64, 40, CUS) == 3
    assert tf.query_1d_kernel(1024, 512, 192, 48, CUS) == 1
    assert tf.query_1d_kernel(1024, 512, 192, 64, CUS) == 3
    assert tf.query_1d_tile(256, 400, 128, 32, CUS) == 128          # 800 blocks of 64 channels, 768 at a time
    assert tf.query_1d_tile(256, 512, 128, 32, CUS) == 64


def test_1d_kernels_with_nearly_a_block_per_cu():
    """where the small-grid kernel (2) gives way to the kernels that it was measured against: the last shape on each side of a line"""
    for N in (64, 128, 256):
        tiles = N // 64
        for K, last in ((8, 208), (16, 192)):           # DY = 256: the split kernel
            assert tf.query_1d_kernel(256, last // tiles, N, K, CUS) == 2, (N, K)
            assert tf.query_1d_kernel(256, last // tiles + 1, N, K, CUS) == 3, (N, K)
        assert tf.query_1d_kernel(256, CUS // tiles, N, 24, CUS) == 2
        # DY = 1024: the SIMT kernel, which takes what is left over as well
        assert tf.query_1d_kernel(1024, 192 // tiles, N, 8, CUS) == 2 and tf.query_1d_kernel(1024, 192 // tiles + 1, N, 8, CUS) == 1
        assert tf.query_1d_kernel(1024, CUS // tiles, N, 16, CUS) == 2


def _gemm_steps(tmp_path, lines):
    """answers of the rules in turbofno_amd/csrc/gemm_steps.h, as tuples"""
    exe = str(tmp_path / "gemm_steps_check")
    source = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host", "gemm_steps_check.cpp")
    subprocess.run(["g++", "-O1", "-std=c++17", source, "-o", exe], check=True)
    text = "".join(" ".join(map(str, line)) + "\n" for line in lines)
    out = subprocess.run([exe], input=text, check=True, capture_output=True, text=True).stdout.splitlines()
    return [tuple(map(int, ln.split())) for ln in out]


def test_mode_gemm_steps(tmp_path):
    """half steps follow the run that is walked, not the period of the weights: with R parts per image a run mostly covers all R of them"""
    wide, narrow, small = (4, 1024, 6), (4, 512, 6), (1, 512, 6)
    cases = [   # parts, channels per part, kernel -> channels per run, half steps
        (1, 8, wide, 8, 1), (1, 16, wide, 16, 1), (1, 24, wide, 24, 0), (1, 32, wide, 32, 0), (1, 72, wide, 72, 1), (1, 64, wide, 64, 0),
        (1, 72, (8, 512, 3), 72, 1), (1, 96, (8, 512, 3), 96, 0),
        (2, 16, wide, 32, 0), (2, 48, wide, 96, 0), (2, 80, wide, 160, 0),          # full steps although the period ends in a short one
        (4, 8, wide, 32, 0), (4, 16, wide, 64, 0), (4, 40, wide, 160, 0), (4, 48, wide, 192, 0),
        (2, 24, wide, 48, 1), (2, 56, wide, 112, 1), (2, 88, wide, 176, 1),         # the other way round
        (2, 104, wide, 104, 1), (4, 72, wide, 72, 1), (4, 56, wide, 56, 0), (2, 32, wide, 32, 0),   # more than the tile holds, whole periods: run by run
        (1, 48, small, 48, 1), (1, 72, small, 72, 0), (2, 24, small, 48, 1), (2, 40, small, 80, 0), (4, 72, small, 72, 0),
        (1, 112, narrow, 112, 1), (1, 136, narrow, 136, 0), (1, 136, wide, 136, 1), (1, 200, wide, 200, 0), (2, 72, narrow, 144, 0), (2, 72, wide, 144, 1),
    ]
    assert _gemm_steps(tmp_path, [(0, r * k, k) + kernel for r, k, kernel, _, _ in cases]) == [c[3:] for c in cases]


def test_mode_gemm_persistent_blocks(tmp_path):
    """blocks of columns, blocks that the CUs hold, channels -> blocks launched: whole groups of eight, unless with few channels they make two
    rounds of one"""
    cases = [(1, 256, 16, 1), (80, 85, 16, 80), (81, 85, 16, 81), (85, 85, 8, 85), (86, 85, 16, 80), (81, 85, 24, 80), (85, 85, 64, 80), (170, 85, 16, 80),
             (42, 42, 16, 42), (43, 42, 16, 40), (51, 51, 8, 51), (1000, 51, 16, 48), (256, 256, 72, 256), (300, 256, 16, 256), (7, 7, 72, 7),
             (1000, 7, 16, 7), (5, 0, 16, 1)]
    assert _gemm_steps(tmp_path, [(1,) + c[:3] for c in cases]) == [c[3:] for c in cases]
