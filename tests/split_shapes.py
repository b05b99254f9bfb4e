"""Shapes at the edges of the split-x GEMM's tiles, with the plan that each
weight kind takes there: test_plans_cpu.py holds the plans to this table,
test_gpu_split_tiles.py the kernels' results.  A plan is rows x columns of a
tile, x2 for two wave groups, + for stage sums."""
E4, I8, FP4, NF4, E5, B16, H16, F32, I4, U8 = range(10)
DTYPE = {E4: 4, I8: 9, FP4: 16, NF4: 26, E5: 5, B16: 3, H16: 2, F32: 1, I4: 14, U8: 13}
ONE, TABLES, SIX = (E4, I8, E5), (FP4, NF4), (F32, U8)
PAIRED = (E4, I8, FP4, NF4, E5, I4)  # SwiGLU's Gate and Up in one launch


def _plans(*groups):
    return {k: plan for kinds, plan in groups for k in kinds}


# (outputs, inputs, batch): batch, outputs and inputs (half a k stage) past
# whole tiles; plans of a single launch, and of a pair launch
SHAPES = [
    (1001, 2016, 20, _plans((ONE + SIX + (B16, H16), "32x128+"), (TABLES + (I4,), "32x256x2")),
     _plans((ONE, "32x128+"), (TABLES + (I4,), "32x256x2+"))),
    # an odd count of stages: no two groups
    (1001, 1952, 20, _plans((ONE + SIX + (B16, H16), "32x128+"), (TABLES + (I4,), "32x256+")),
     _plans((ONE, "32x128+"), (TABLES + (I4,), "32x256+"))),
    (4100, 2016, 20, _plans((ONE + (B16,), "32x128"), (SIX + (H16,), "32x128+"), (TABLES + (I4,), "32x256x2")), {}),
    (8205, 160, 20, _plans((ONE + TABLES + (B16, I4), "32x256"), ((H16,), "32x256+"), (SIX, "32x128+")),
     _plans((PAIRED, "32x256+"))),
    (130, 4128, 40, _plans((ONE + TABLES + (B16, H16, I4), "32x128+")), _plans((PAIRED, "32x128+"))),
    (1300, 1056, 70, _plans((ONE + TABLES + SIX + (H16,), "32x128+"), ((B16, I4), "32x128")), {}),
    (1300, 2016, 200, _plans((ONE + TABLES, "32x256x2+"), ((I4,), "32x256x2"), ((B16,), "32x128"), ((H16,), "32x128+"),
                             (SIX, "64x128")), _plans((PAIRED, "32x256x2+"))),
    (2065, 1952, 300, _plans((ONE + TABLES + (B16, H16, I4), "64x256"), (SIX, "64x128")), _plans((PAIRED, "64x256"))),
    (2065, 2016, 490, _plans((ONE + TABLES + (B16, H16, I4), "64x256x2"), (SIX, "64x128")),
     _plans((PAIRED, "64x256x2"))),
]
