"""Sizes (M, N, K) that take every kernel of the packed GEMM, for its tests on the GPU and for the test that says so."""

# row counts around the 16 / 32 / 64-row tiles, one k step per wavefront and several rounds of them, few and many
# column blocks
FEW_ROWS = [(1, 32, 32), (16, 96, 256), (17, 768, 768), (33, 2304, 768), (64, 3072, 768), (65, 768, 3072),
            (130, 1024, 1024), (200, 1024, 4096), (300, 4096, 1056), (257, 320, 5120), (1, 32, 896), (1, 32, 3136),
            (1, 32, 4128), (81, 2080, 32), (20, 2080, 832), (391, 3712, 32), (17, 2304, 1344), (39, 3104, 864),
            (52, 3168, 736), (52, 2592, 1088), (70, 2848, 800), (140, 1632, 1184), (129, 1728, 1312), (429, 1216, 672),
            (455, 1088, 800), (260, 1920, 1184), (316, 1664, 1344)]

# one tile and several of them per workgroup, partial row blocks and column tiles, and rectangles of an XCD that the
# tiles do not fill
MANY_ROWS = [(1000, 3072, 768), (192, 768, 3072), (250, 1088, 2080), (1000, 768, 3072), (760, 1088, 2048),
             (1000, 1024, 1024), (8000, 3072, 768), (392, 1184, 64), (524, 1856, 64), (583, 3296, 64), (1476, 2976, 448),
             (16439, 160, 64), (10970, 352, 192), (17111, 288, 64), (16546, 672, 128), (16388, 1696, 128),
             (15479, 32, 448), (787, 2432, 256), (791, 2528, 512), (7203, 288, 1088), (2731, 1920, 384),
             (3597, 3904, 192), (1661, 2496, 320), (14739, 1120, 832), (1059, 3616, 192), (8329, 1824, 320)]

# normalised rows: a few kernels from registers (all of K at once, in rounds, one and several row blocks), every tile
NORMALISED_FEW = [(33, 2304, 768), (16, 32, 32), (70, 96, 4096), (129, 1728, 1312)]
NORMALISED_MANY = [(1000, 3072, 768), (1476, 2976, 448), (8000, 3072, 768), (787, 2432, 256), (791, 2528, 512),
                   (15479, 32, 448), (260, 1920, 1184)]

# What there is.  Tiles: (rows, cols, k of a slab) -> whether they fold a layer norm, and tiles a CU works on at a
# time; from registers: (rows, cols, k in flight, all of K at once).
TILES = {(256, 256, 32): (True, 1), (256, 128, 32): (False, 2), (256, 128, 64): (True, 1), (128, 128, 32): (False, 2),
         (128, 128, 64): (True, 1), (64, 128, 64): (True, 1), (64, 64, 64): (True, 2), (64, 192, 64): (True, 1)}
FROM_REGISTERS = {(16, 16, 96, True), (16, 16, 128, True), (16, 16, 384, True), (16, 16, 512, True), (16, 16, 384, False),
                  (32, 16, 96, True), (32, 16, 128, True), (32, 16, 192, True), (32, 16, 192, False),
                  (32, 32, 96, True), (32, 32, 128, True), (32, 32, 128, False),
                  (64, 16, 96, True), (64, 16, 128, True), (64, 16, 128, False),
                  (64, 32, 96, True), (64, 32, 128, True), (64, 32, 96, False), (64, 32, 128, False),
                  (64, 64, 96, True), (64, 64, 128, True), (64, 64, 96, False), (64, 64, 128, False)}
