"""Shape lists and type tuples of the reference's own test matrix, restated.

TYPE_TUPLES: (lhs, rhs, accum, dst) of ruy/BUILD:1195-1206 (test_fast), plus
the int8 tuples that the benchmark configurations use.
Shape lists: ruy/test_fast.cc:31-107 and ruy/test_slow.cc:29-68.
"""
from ruy_amd import _structs as S

TYPE_TUPLES = [
    (S.F32, S.F32, S.F32, S.F32),
    (S.F64, S.F32, S.F64, S.F32),
    (S.F32, S.F64, S.F64, S.F64),
    (S.U8, S.U8, S.I32, S.U8),
    (S.I8, S.I8, S.I32, S.I8),
    (S.I8, S.U8, S.I32, S.I8),
    (S.U8, S.U8, S.I32, S.I16),
    (S.I8, S.I8, S.I32, S.I32),
    (S.I8, S.U8, S.I32, S.I32),
    (S.I8, S.I16, S.I32, S.I16),
    (S.I16, S.I8, S.I32, S.I16),
    # benchmark tuples (ruy/BUILD:1175-1184) not already above
    (S.I8, S.I8, S.I32, S.U8),
    (S.I8, S.I8, S.I32, S.I16),
    (S.U8, S.U8, S.I32, S.I32),
]

INT_TUPLES = [t for t in TYPE_TUPLES if t[2] == S.I32]
FP_TUPLES = [t for t in TYPE_TUPLES if t[2] != S.I32]


def tuple_name(t):
    return "x".join(S.DTYPE_NAMES[x] for x in t[:2]) + "_" + S.DTYPE_NAMES[t[2]] + "_" + S.DTYPE_NAMES[t[3]]


SQUARE_SIZES = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 16, 32, 48, 64, 15, 31, 63, 17, 33, 65]
MISC_SHAPES = [(2, 3, 4), (7, 6, 5), (12, 23, 6), (19, 3, 11), (3, 10, 17), (30, 21, 43),
               (7, 57, 9), (49, 69, 71), (38, 111, 29), (87, 98, 76), (16, 96, 16),
               (16, 88, 16), (16, 84, 16), (16, 92, 16), (16, 82, 16), (16, 81, 16),
               (16, 95, 16), (3, 128, 5)]
DEEP_SHAPES = [(1, 32767, 1), (5, 5001, 4), (9, 1025, 10)]
SHALLOW_SHAPES = [(101, 1, 103), (71, 2, 53), (51, 3, 73), (51, 4, 43)]
NARROW_SHAPES = [s for w in (1, 2, 3, 4, 5, 8)
                 for s in ((w, 12, 13), (15, 19, w), (w, 123, 137), (158, 119, w))]
GEMV_SHAPES = ([(size, depth, 1) for size in (1, 2, 4, 8, 16, 32, 64, 128, 256, 512)
                for depth in range(1, 500, 47)] + [(5, 5001, 1), (8193, 17, 1)])
SLOW_SHAPES = ([s for w in (1, 2, 3, 4, 5, 8) for s in ((w, 401, 601), (587, 443, w))] +
               [(7, 45984, 5), (512, 256, 16), (501, 1, 321), (301, 5, 403), (256, 32, 512),
                (225, 303, 199), (256, 192, 128), (70, 1024, 80), (60, 2048, 70),
                (40, 4096, 50)] +
               [(size, depth, 1) for size in (1025, 1409) for depth in range(350, 500, 47)])

ALL_ORDERS = [(a, b, c) for a in (0, 1) for b in (0, 1) for c in (0, 1)]
RCC = (S.ORDER_ROW_MAJOR, S.ORDER_COL_MAJOR, S.ORDER_COL_MAJOR)


def small_tile_problems(types):
    """(M, K, N, orders) of products that between them run on every form of the
    kernel on 32x32 and 64x64 tiles (csrc/kernels/small_gemm.h) that the planner
    chooses for these types on 256 CUs: test_host_side.py looks it up, and
    test_gpu_parity.py runs them. Every number of tiles to a CU and of waves to a
    tile, the depths at which those change, operands along the rows and across
    them, with runs that start at multiples of 16 bytes, of 4 and at any byte."""
    sizes = [(64, 32, 96), (64, 512, 96), (64, 4096, 96), (64, 6144, 96), (512, 512, 800), (512, 1200, 800),
             (800, 1200, 1200), (800, 1504, 1200), (1040, 1200, 976), (1040, 1504, 976)]
    if types[:2] == (S.F32, S.F32):
        sizes = [(64, 32, 96), (64, 128, 96), (64, 512, 96), (64, 1280, 96), (512, 256, 800)]
    elif S.I16 in types[:2]:
        sizes = [(64, 32, 96), (64, 512, 96)]
    for size in sizes:
        for more in (0, 4, 1):
            for lhs, rhs in [(1, 0), (1, 1), (0, 0), (0, 1)]:
                for dst in ((0, 1) if size[0] * size[1] * size[2] <= 4000000 else (0,)):
                    yield tuple(x + more for x in size) + ((lhs, rhs, dst),)


SMALL_TILE_TYPES = [(S.U8, S.I8, S.I32, S.U8), (S.I8, S.I8, S.I32, S.I32), (S.I8, S.I16, S.I32, S.I16),
                    (S.I16, S.I8, S.I32, S.I32), (S.F32, S.F32, S.F32, S.F32)]


# Rows that the staged form of the 64x64 tile reads (csrc/kernels/gemm_i8_staged.hip):
# depths either side of its ring of four and of eight stages and of a granule;
# (rows, columns, padded, LHS from the cache).
STAGED_DEPTHS = [16, 17, 31, 127, 128, 130, 383, 400, 511, 512, 513, 896, 1000, 1023, 1024, 1025]
STAGED_SHAPES = [(64, 64, False, False), (65, 129, True, False), (17, 63, False, True)]
STAGED_TYPES = [(S.U8, S.U8, S.I32, S.U8), (S.I8, S.I8, S.I32, S.I16), (S.I8, S.U8, S.I32, S.I32)]

# Edges of the pack kernels: depths either side of a 16-byte granule, of what a
# row's lanes hold and of a depth dealt to several workgroups.
PACK_DEPTHS = [1, 3, 15, 17, 33, 65, 145, 257, 1023, 1025, 1041, 4099, 9001]
PACK_SHAPES = [(65, 37), (19, 130)]
PACK_ORDERS = [(1, 0, 0), (0, 0, 0), (1, 1, 1), (0, 1, 0)]

# Grids of more fp32 tiles than CUs, which run on rings of two stages: (tile, rows, columns).
F32_SHALLOW_RINGS = [((64, 128), 1100, 2100), ((128, 64), 2100, 1100), ((128, 128), 2100, 2100)]
