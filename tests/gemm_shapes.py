"""Shapes of the FP8 GEMM's GPU tests with the kernels that each launch takes on 256
CUs (tests/gemm_plan_check.cpp spells the routes out). tests/test_gpu_gemm.py
runs them; tests/test_gemm_plan.py asserts the routes on the CPU, so that a change
of the launch rule cannot silently take a kernel out of the GPU tests."""

# Row/column GEMMs, (M, K, N): route. Each small tile ragged in M, the 192- and
# 256-wide ones in N too; K of 1 to 9 steps covers the pipeline's fill and
# drain, and K below 896 the GELU of the unrounded value.
SMALL_ROWCOL = {
    (100, 1024, 256): "64x64",
    (65, 128, 384): "64x64",
    (1, 128, 128): "64x64",
    (450, 1024, 3200): "64x128",
    (1000, 768, 2048): "64x128",
    (1000, 1024, 3072): "128x128",
    (1025, 896, 4224): "128x192",
    (1025, 640, 3968): "128x192",
    (2049, 896, 2944): "128x256",
    (4097, 640, 3200): "128x256",
    (3000, 896, 3072): "256x192",
    (2500, 640, 4224): "256x192",
    (2500, 896, 3200): "256x192",
}

# 256 x 256 tiles of the persistent kernel: more tiles than CUs, so that a
# workgroup walks whole and edge tiles in turn, edges in M, in N and in both, the
# smallest K it takes (896), with and without bias and GELU. Beside them, shapes
# below its range on the small tiles. (M, K, N, gelu, bias): route.
PERSISTENT = {
    (300, 896, 384, True, True): "64x64",
    (300, 768, 384, True, True): "64x64",
    (1000, 1280, 640, True, True): "64x64",
    (700, 1024, 1280, True, False): "64x64",
    (132, 12288, 3072, True, True): "64x64",
    (4500, 896, 2048, True, True): "256x256 edge",
    (4352, 896, 2176, False, False): "256x256 edge",
    (4700, 1024, 4224, True, False): "256x256 edge",
    (4700, 1024, 4224, False, True): "256x256 edge",
    # Last row tile 132 deep: waves of rows 0-127 multiply a whole block while
    # the stage rows they load (128-191) lie partly past M; the loads must
    # stay inside A.
    (4996, 1024, 4224, False, True): "256x256 edge",
}

# A last row stripe of at most 64 rows: gemm_tail_kernel beside the 256 x 256 tiles
# or, up to 64 rows in all, alone; K split over 4 waves or, from 256 column groups
# on, over 2; one and two 32-row blocks. The first rows take small tiles, which
# have no stripe. (M, K, N, gelu, bias): route.
TAIL = {
    (257, 1024, 384, True, True): "64x64",
    (288, 896, 640, False, True): "64x64",
    (289, 3072, 512, True, False): "64x64",
    (10800, 12288, 384, False, True): "128x128",
    (276, 4224, 8192, False, True): "128x128",
    (576, 4352, 8192, True, True): "128x192",
    (1, 4224, 256, True, True): "tail 4x1",
    (48, 3072, 1280, True, True): "tail 4x2",
    (20, 896, 8192, False, True): "tail 2x1",
    (64, 896, 8192, True, False): "tail 2x2",
    (2049, 896, 4096, True, True): "256x256 tail 4x1",
    (2049, 896, 4224, False, False): "256x256 edge tail 4x1",
    (2100, 896, 4096, False, True): "256x256 tail 4x2",
    (4129, 4224, 3072, False, True): "256x256 tail 4x2",
    (1300, 896, 8192, False, True): "256x256 tail 2x1",
    (2100, 896, 8192, True, True): "256x256 tail 2x2",
}

# The stripe on the persistent launch's light workgroups. (M, K, N, gelu, bias).
LIGHT = {
    (10785, 896, 4096, True, True): "256x256 light",     # 33 rows (two blocks), 96 light workgroups of 64 columns
    (10770, 1024, 2048, False, False): "256x256 light",  # 18 rows (one block)
}

# Into guarded buffers. (M, K, N, act): route.
GUARD = {
    (100, 1024, 256, 1): "64x64",
    (1000, 1280, 640, 0): "64x64",
    (450, 1024, 3200, 1): "64x128",
    (1000, 1024, 3072, 0): "128x128",
    (1025, 896, 3968, 1): "128x192",
    (2049, 896, 2944, 0): "128x256",
    (2500, 896, 3200, 1): "256x192",
    (4964, 1024, 4224, 1): "256x256 edge",  # last row tile 100 deep
    (5092, 1024, 4224, 0): "256x256 edge",  # 228 deep, its second row wave 100
}
GUARD_TAIL = {
    (300, 1024, 384, 1): "64x64",
    (289, 4352, 256, 0): "64x64",
    (276, 4224, 8192, 0): "128x128",
    (33, 896, 128, 1): "tail 4x2",
    (2049, 896, 4096, 0): "256x256 tail 4x1",
    (2100, 896, 4096, 1): "256x256 tail 4x2",
    (1300, 896, 8192, 0): "256x256 tail 2x1",
    (2100, 896, 8192, 1): "256x256 tail 2x2",
    (10785, 896, 4096, 1): "256x256 light",
}

# Blockwise GEMMs, (M, N, K): route. Small tiles, ragged in M and, 256 wide, in N.
SMALL_BLOCKWISE = {
    (129, 256, 384): "64x64",
    (1000, 1024, 2048): "64x64",
    (2200, 640, 1920): "64x64",
    (1000, 2048, 1024): "128x128",
    (450, 2944, 896): "128x128",
    (2000, 4096, 1024): "128x256",
    (1300, 3200, 640): "128x256",
}
# One shape per kernel: 64 x 64 and 128 x 128 add each K block's product by its
# factor; 128 x 256 and 256 x 256 carry the accumulators in units of the block's.
ZERO_FACTORS = {
    (300, 384, 1024): "64x64",
    (1000, 2048, 1024): "128x128",
    (2000, 4096, 1024): "128x256",
    (2816, 3072, 1024): "256x256",
}
FACTOR_JUMP = {
    (256, 256, 512): "64x64",
    (1000, 2048, 512): "128x128",
    (2000, 4096, 512): "128x256",
    (4352, 2048, 512): "256x256",
}
TAIL_BLOCKWISE = {
    (10800, 12288, 4096): "256x256 tail 2x2",
    (4116, 4096, 512): "256x256 tail 4x1",
    (4129, 4096, 512): "256x256 tail 4x2",
    (2049, 8192, 512): "256x256 tail 2x1",
    (3860, 4224, 512): "256x256 edge tail 4x1",
    (48, 512, 1024): "tail 4x2",
    (33, 256, 4096): "tail 4x2",
    (1, 256, 1024): "tail 4x1",
    (20, 8192, 512): "tail 2x1",
}
GUARD_BLOCKWISE = {
    (300, 256, 512): "64x64",
    (129, 384, 1024): "64x64",
    (4097, 128, 4096): "64x64",
    (450, 2944, 896): "128x128",
    (1300, 3200, 640): "128x256",
    (1556, 5120, 512): "256x256 edge",
    (2100, 8192, 512): "256x256 tail 2x2",
    (4116, 4096, 512): "256x256 tail 4x1",
}
DECODER = {
    (1536, 4096, 12288): "128x256",
    (1536, 12288, 4096): "128x256",
    (10800, 4096, 4096): "256x256 edge",
}

ROWCOL_TABLES = (SMALL_ROWCOL, PERSISTENT, TAIL, LIGHT, GUARD, GUARD_TAIL)
BLOCKWISE_TABLES = (SMALL_BLOCKWISE, ZERO_FACTORS, FACTOR_JUMP, TAIL_BLOCKWISE, GUARD_BLOCKWISE, DECODER)
