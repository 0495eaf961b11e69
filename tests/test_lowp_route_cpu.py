"""Which kernels a reduced-precision product takes (ttm_lowp.hip, lowp_route):
the fused tiles where its rows are whole vectors, otherwise one thread per
element or the converted planes, by the estimate of generic_faster; and the
planes in place of the tiles for few column blocks (256 compute units, the
planner's assumption without a device)."""
import pytest

from ttm_amd._lib import PRECISION_NAMES


def _kernel(ttmlib, na, q, m, prec, b="row"):
    pia = list(range(1, len(na) + 1))
    args = (q, na, pia, [m, na[q - 1]], [1, 2] if b == "col" else [2, 1])
    kw = {"precision": int(PRECISION_NAMES[prec])}
    return ttmlib.plan_kernel_symbol(*args, **kw).split("<")[0]


# odd extents: few rows of B or a short contraction on many elements leave the
# planes (written and read once, padded to 32 / 64 / 128 indices and 64 rows)
# behind one thread per element; measured on both sides of each pair
ODD = [
    ([317, 33, 38237], 2, 1, "bf16", "k_lowp_generic"), ([317, 33, 38237], 2, 16, "bf16", "k_planes"),
    ([5, 20000000], 1, 2, "bf16", "k_lowp_generic"), ([3, 10000000], 1, 4, "bf16", "k_lowp_generic"),
    ([3, 10000000], 1, 8, "bf16x3", "k_lowp_generic"), ([711, 301, 140], 2, 8, "bf16x3", "k_planes"),
    ([797, 33, 3807], 2, 1, "bf16x3", "k_lowp_generic"), ([379, 33, 23987], 2, 16, "fp16x2", "k_planes"),
    ([25, 3000001], 1, 1, "bf16", "k_planes"), ([1001, 100001], 1, 1, "bf16", "k_planes"),
    ([129, 1001, 99], 2, 1, "bf16", "k_planes"), ([129, 9, 999999], 2, 2, "fp8", "k_lowp_generic"),
    ([129, 301, 9999], 2, 32, "fp8", "k_fp8"), ([33, 9, 31], 2, 33, "bf16", "k_lowp_generic"),
    ([255, 301, 173], 2, 120, "fp16x2", "k_planes"), ([33, 43, 3], 1, 65, "bf16", "k_planes"),
]


@pytest.mark.parametrize("na,q,m,prec,want", ODD)
def test_odd_extents(ttmlib, na, q, m, prec, want):
    assert _kernel(ttmlib, na, q, m, prec) == want


# aligned, more than 64 rows of B and a long contraction: up to half a 128-column
# block per compute unit (two planes: a quarter), fewer for narrow slabs
FEW = [
    ([512, 128 * 128], 1, 100, "bf16", "k_planes"), ([512, 128 * 129], 1, 100, "bf16", "k_lowp"),
    ([512, 128 * 64], 1, 100, "fp16x2", "k_planes"), ([512, 128 * 65], 1, 100, "fp16x2", "k_lowp"),
    ([16, 512, 8 * 128], 2, 100, "fp16", "k_planes"), ([16, 512, 8 * 129], 2, 100, "fp16", "k_lowp"),
    ([8, 512, 16 * 96], 2, 100, "bf16", "k_planes"), ([8, 512, 16 * 97], 2, 100, "bf16", "k_lowp"),
    ([4, 512, 32 * 64], 2, 100, "bf16", "k_planes"), ([4, 512, 32 * 65], 2, 100, "bf16", "k_lowp"),
    ([4, 512, 32 * 32], 2, 100, "fp16x2", "k_planes"), ([4, 512, 32 * 33], 2, 100, "fp16x2", "k_lowp"),
    # at most one block per compute unit, rows and columns together
    ([512, 128 * 64], 1, 512, "bf16", "k_planes"), ([512, 128 * 65], 1, 512, "bf16", "k_lowp"),
    ([512, 128 * 64], 1, 64, "bf16", "k_lowp"), ([252, 128 * 64], 1, 100, "bf16", "k_lowp"),
    ([512, 128 * 64], 1, 100, "bf16x3", "k_lowp"),
]


@pytest.mark.parametrize("na,q,m,prec,want", FEW)
def test_few_aligned_blocks(ttmlib, na, q, m, prec, want):
    assert _kernel(ttmlib, na, q, m, prec) == want
