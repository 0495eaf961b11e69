"""Which products take the pipelined loop of the gemm tiles (ttm_gemm.hip,
gemm_pipelined): long contractions whose blocks are mostly interior and whose
grid the pipelined kernels do not run in more rounds than the plain ones, on
both sides of each line, in both views and B orientations (256 compute units,
the planner's assumption without a device)."""
import re

import pytest


def _pipelined(ttmlib, na, q, m, b, dtype):
    pia = list(range(1, len(na) + 1))
    sym = ttmlib.plan_kernel_symbol(q, na, pia, [m, na[q - 1]], [1, 2] if b == "col" else [2, 1],
                                    is_double=dtype == "f64")
    got = re.match(r"k_gemm<(?:float|double), (true|false), ", sym)
    assert got, sym
    return got.group(1) == "true"


# (na, q, m, B, dtype, pipelined)
CASES = [
    # the contraction: 96 (128 rows), 192, 384 (float64)
    ([512, 95, 512], 2, 128, "row", "f32", False), ([512, 96, 512], 2, 128, "row", "f32", True),
    ([512, 191, 2048], 2, 64, "row", "f32", False), ([512, 192, 2048], 2, 64, "row", "f32", True),
    ([384, 65536], 1, 64, "col", "f64", True), ([383, 65536], 1, 64, "col", "f64", False),
    # rows that no vector of a column-major B ends at
    ([512, 400, 2048], 2, 17, "col", "f32", True), ([512, 400, 512], 2, 127, "col", "f32", True),
    ([512, 400, 512], 2, 451, "col", "f32", True), ([512, 400, 512], 2, 41, "col", "f64", True),
    # slab ends inside most blocks
    ([131, 400, 2000], 2, 128, "col", "f32", False), ([131, 400, 2000], 2, 128, "row", "f32", True),
    ([2051, 400, 128], 2, 128, "col", "f32", True),
    # ... but for the tiles of one row of waves where both kernels take two rounds
    ([131, 400, 900], 2, 41, "col", "f64", True), ([131, 400, 1000], 2, 41, "col", "f64", False),
    ([131, 400, 700], 2, 41, "col", "f64", False), ([131, 400, 1800], 2, 41, "col", "f32", False),
    ([131, 400, 1800], 2, 63, "col", "f32", True),
    # more than two, at most three blocks per compute unit
    ([256, 400, 512], 2, 20, "row", "f32", True), ([256, 400, 513], 2, 20, "row", "f32", False),
    ([256, 400, 768], 2, 20, "row", "f32", False), ([256, 400, 769], 2, 20, "row", "f32", True),
    ([256, 400, 600], 2, 40, "row", "f32", True), ([128, 400, 600], 2, 20, "row", "f64", False),
    ([400, 128 * 600], 1, 20, "row", "f64", False), ([400, 128 * 600 - 1], 1, 20, "row", "f64", True),
    ([200, 256 * 600], 1, 32, "col", "f32", False), ([200, 256 * 600 + 1], 1, 32, "col", "f32", True),
    ([400, 128 * 600], 1, 41, "col", "f64", True),
]


@pytest.mark.parametrize("na,q,m,b,dtype,want", CASES)
def test_rule(ttmlib, na, q, m, b, dtype, want):
    assert _pipelined(ttmlib, na, q, m, b, dtype) == want
