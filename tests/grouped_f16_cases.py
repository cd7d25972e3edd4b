"""Sizes of the grouped call that run its 64-pair tiles on f16 MFMA:
(dtype, qmm, d_model, d_ff, tokens, top_k, table entries, K parts of the down
projection).  Long down rows bring small calls there; the other rules take
many experts."""
Q4, Q8 = 4, 5

# few pairs: gate/up K of half a stage to several partial sums, tiles of one
# to several 16-pair groups, down rows inside one row tile and over several
LONG_ROWS = [
    (Q4, 0, 64, 8256, 16, 1, 1, 4),     # gate/up K of half a stage, one 16-pair group
    (Q8, 0, 64, 8256, 33, 1, 1, 4),     # one stage, one pair past a half tile
    (Q4, 0, 192, 8256, 32, 1, 1, 4),    # six blocks: one and a half stages, a half tile
    (Q8, 0, 192, 8256, 65, 1, 1, 4),    # one pair past a tile
    (Q4, 0, 320, 8256, 70, 2, 3, 4),    # a second row tile of 64 down rows
    (Q4, 0, 576, 8256, 40, 2, 2, 4),    # eighteen blocks: one partial sum of sixteen and a rest
    (Q8, 0, 1088, 8256, 17, 1, 1, 4),   # 34 blocks, seventeen stages
    (Q4, 0, 64, 8192, 50, 2, 3, 4),     # parts of 64 blocks each
    (Q8, 0, 64, 9280, 48, 1, 2, 4),     # parts of 76, 76, 76 and 62 blocks
]
LONG_ROWS_QMM = [
    (Q4, 1, 64, 8256, 16, 1, 1, 4),
    (Q4, 1, 192, 8256, 65, 1, 1, 4),
    (Q4, 1, 576, 8256, 40, 1, 1, 4),
    (Q4, 1, 128, 8256, 40, 2, 2, 4),
    (Q4, 1, 64, 16384, 33, 1, 1, 4),    # the longest rows
]
# many experts: the sums in one part or two
MANY = [
    (Q8, 0, 64, 192, 4096, 1, 128, 1),
    (Q4, 0, 192, 320, 1024, 3, 96, 1),
    (Q8, 0, 576, 192, 1280, 2, 64, 1),
    (Q4, 0, 64, 4160, 1664, 1, 64, 2),
    (Q4, 0, 512, 512, 512, 6, 256, 1),     # Q4_0 from 12 pairs an expert
    (Q4, 0, 1024, 1024, 512, 8, 416, 1),   # Q4_0 from 8
    (Q4, 0, 4096, 14336, 96, 2, 8, 4),     # the benchmark's experts: 128 and 448 blocks of K
    (Q8, 0, 4096, 14336, 96, 2, 8, 4),
]
