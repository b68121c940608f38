"""Shapes of the GEMM tests by the kernel and tile they run with 256 CUs; the
CPU tests of the host path check that they still do."""

# (rows, strips, K groups) of a split-kernel tile: (M, K, N) of a single GEMM
# and of the first GEMM of a list (the second is SPLIT_TAIL).  The rows are
# 16-byte aligned; with K + 1 the same tile reads rows at any address.
SPLIT_TILES = {
    (64, 8, 2): ((200, 144, 5120), (200, 144, 5120)),
    (64, 4, 4): ((200, 144, 2560), (200, 144, 3072)),
    (32, 4, 4): ((33, 144, 5120), (33, 144, 5120)),
    (32, 2, 4): ((33, 144, 3072), (33, 144, 3072)),
    (32, 2, 8): ((33, 5136, 3072), (33, 5136, 3072)),
    (16, 2, 4): ((9, 144, 5120), (9, 144, 6912)),
    (16, 2, 8): ((9, 5136, 5120), (9, 5136, 6912)),
    (16, 1, 4): ((9, 144, 64), (9, 144, 64)),
    (16, 1, 8): ((9, 5136, 64), (9, 5136, 64)),
}
SPLIT_TAIL = (3, 32, 20)

# ring kernel, by its row blocks of 16: single GEMMs, and lists of n GEMMs that
# alternate between two weights (N a multiple of 4, and not).  Row counts fill
# their blocks or not; past 128 rows there are pieces, the last one short.
RING_SINGLE = [(5, 272, 32784), (16, 256, 32784), (20, 272, 65552), (32, 272, 65555), (33, 272, 65552), (64, 272, 65555),
               (100, 272, 32784), (128, 272, 32787), (130, 272, 32784), (256, 272, 32787)]
RING_LIST = {"1": [(5, 272, 1000), (16, 272, 1003)] * 12, "2": [(17, 272, 404), (32, 272, 403)] * 64,
             "4": [(33, 512, 404), (64, 272, 403)] * 32, "8": [(65, 272, 404), (128, 272, 403)] * 24,
             "pieces": [(200, 272, 404), (256, 272, 403), (3, 272, 404)] * 12}
