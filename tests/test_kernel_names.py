"""ttm_plan_kernel_symbol and ttm_last_kernel name kernels that exist: every
planned name is a template instance of the built library, over shapes that
reach every block shape, and a launched gemm tile carries the variant that its
buffers and splits chose."""
import itertools
import shutil
import subprocess

import numpy as np
import pytest

import refcases as rc
from ttm_amd._lib import PRECISION_NAMES


@pytest.fixture(scope="module")
def instances(ttmlib):
    nm = shutil.which("nm")
    if nm is None:
        pytest.skip("nm not available")
    out = subprocess.run([nm, "-C", str(ttmlib.LIB_PATH)], capture_output=True, text=True, check=True).stdout
    assert "k_gemm<" in out
    return out


def _symbol(ttmlib, na, q, m, b, prec, dbl=False):
    return ttmlib.plan_kernel_symbol(q, na, list(range(1, len(na) + 1)), [m, na[q - 1]], [1, 2] if b else [2, 1],
                                     is_double=dbl, precision=int(PRECISION_NAMES[prec]))


@pytest.mark.parametrize("prec", ["bf16x3", "fp16x2", "bf16", "fp16", "fp8"])
def test_reduced_precision_names_are_instances(ttmlib, instances, prec):
    seen = set()
    for (na, q), m, b in itertools.product((([33, 301], 1), ([301, 33], 2), ([33, 32769], 1), ([4097, 33, 8], 2),
                                            ([8192, 4096], 1), ([256, 300, 4], 2), ([512, 640, 512], 2), ([640, 90000], 1)),
                                           (3, 64, 65, 128, 129, 300, 1024), (0, 1)):
        sym = _symbol(ttmlib, na, q, m, b, prec)
        seen.add(sym)
        assert sym + "(" in instances, (na, q, m, sym)
    planes = {s for s in seen if s.startswith("k_planes<")}
    if prec != "fp8":  # each shape in both views: three for one and two planes
        assert len(planes) == (4 if prec == "bf16x3" else 6), planes
    if prec in ("bf16", "fp16"):
        assert any(", 1, 4, 8, 4, 1, 3, " in s for s in planes), planes


@pytest.mark.parametrize("dbl", [False, True])
def test_gemm_names_are_instances(ttmlib, instances, dbl):
    for (na, q), m, b in itertools.product((([100, 4000], 1), ([500, 40000], 1), ([64, 90, 100], 2), ([512, 500, 100], 2),
                                            ([131, 400, 90], 2), ([8, 700], 2)),
                                           (9, 17, 20, 33, 48, 64, 65, 96, 128, 190, 300), (0, 1)):
        sym = _symbol(ttmlib, na, q, m, b, "default", dbl)
        assert sym + "(" in instances, (na, q, m, b, sym)


@pytest.mark.gpu
def test_split_product_into_unaligned_c_names_the_unpadded_tile(gpu):
    """The blocks of a split product write aligned partials, whatever C is."""
    import torch
    import ttm_amd
    na, m, nq = [64, 4096, 2], 40, 4096
    A = torch.rand(int(np.prod(na)), device=gpu)
    B = torch.rand(m * nq, device=gpu)
    nc = [64, m, 2]
    n = int(np.prod(nc))
    buf = torch.empty(n + 4, device=gpu)
    names = []
    for off in (0, 1):
        ttm_amd.force_kernel("gemm")
        ttm_amd.ttm_raw(2, 3, A, na, rc.dense_strides(na, [1, 2, 3]), [1, 2, 3], B, [m, nq], [2, 1], buf[off:off + n], nc,
                        rc.dense_strides(nc, [1, 2, 3]))
        names.append(ttm_amd.last_kernel())
    assert names[0][1] > 1 and names[0] == names[1], names
    assert names[0][0].endswith(", false>"), names
