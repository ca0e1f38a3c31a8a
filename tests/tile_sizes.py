"""Steering of the projections' tile kernel (tiled_gemm.hip) and the sizes that ran."""
FEW_ROWS = dict(TILED_BIG_MIN_TILES=10 ** 6)
SIZES = {"128x256": dict(TILED_BIG_MIN_TILES=1, TILED_WIDE_MIN_TILES=1),
         "128x128": dict(TILED_BIG_MIN_TILES=1, TILED_WIDE_MIN_TILES=10 ** 6, TILED_HALF_MAX_TILES=0),
         "128x64": dict(TILED_BIG_MIN_TILES=1, TILED_WIDE_MIN_TILES=10 ** 6, TILED_HALF_MAX_TILES=10 ** 6, TILED_SMALL_MAX_TILES=0),
         "64x64": dict(TILED_BIG_MIN_TILES=1, TILED_WIDE_MIN_TILES=10 ** 6, TILED_HALF_MAX_TILES=10 ** 6, TILED_SMALL_MAX_TILES=10 ** 6)}


def sizes_that_ran(hits):
    return {s for s in SIZES if hits.get("tiled_gemm_" + s)}
