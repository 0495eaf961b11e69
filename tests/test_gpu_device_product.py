"""The tensor front ends' short way to the library (api.device_product): the
same bits as the checked low-level call for every layout, B orientation and
element type it accepts, and the same refusals."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tensor(torch, gpu, na, pia, dt, gen):
    slow_first = [r - 1 for r in reversed(pia)]
    store = torch.rand([na[r] for r in slow_first], generator=gen, dtype=dt, device=gpu)
    return store.permute(*[slow_first.index(k) for k in range(len(na))])


@pytest.mark.parametrize("name", ["float32", "float64"])
def test_same_bits_as_the_low_level_call(gpu, name):
    import torch
    import ttm_amd
    dt = getattr(torch, name)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(5)
    for na in ([9], [8, 12], [6, 1, 10], [4, 5, 6, 7]):
        p = len(na)
        for pia in itertools.permutations(range(1, p + 1)):
            A = _tensor(torch, gpu, na, pia, dt, gen)
            pi = ttm_amd.layout_from_strides(list(A.shape), list(A.stride()))
            for q in range(1, p + 1):
                M = torch.rand((5, 2 * na[q - 1]), generator=gen, dtype=dt, device=gpu)[:, ::2]  # not contiguous
                for b_layout in ("row", "col"):
                    got = ttm_amd.ttm(np.int64(q), A, M, b_layout=b_layout, layout=np.array(pi))
                    nc = list(na)
                    nc[q - 1] = 5
                    wc = ttm_amd.dense_strides(nc, pi)
                    B = M.contiguous() if b_layout == "row" else M.t().contiguous()
                    C = torch.empty_strided(nc, wc, dtype=dt, device=gpu)
                    ttm_amd.ttm_raw(q, p, A, na, list(A.stride()), pi, B, [5, na[q - 1]], [2, 1] if b_layout == "row"
                                    else [1, 2], C, nc, wc)
                    assert list(got.stride()) == wc and torch.equal(got, C), (na, pia, q, b_layout)


def test_same_refusals(gpu):
    import torch
    import ttm_amd
    A = torch.rand(6, 8, 10, device=gpu)
    B = torch.rand(3, 8, device=gpu)
    with pytest.raises(ValueError, match="dense block"):
        ttm_amd.ttm(2, A[:, :, ::2], B)
    with pytest.raises(ValueError, match="dense block"):
        ttm_amd.ttmpy.ttm(2, A[:, :, ::2], B)
    with pytest.raises(ttm_amd.TTMError, match="contraction dimension"):
        ttm_amd.ttm(1, A, B)
    with pytest.raises(ttm_amd.TTMError, match="stride vector of A"):
        ttm_amd.ttmpy.ttm(2, A.permute(2, 1, 0), B)
    with pytest.raises(ttm_amd.TTMError, match="precision"):
        ttm_amd.ttm(2, A.double(), B.double(), precision="bf16")
    with pytest.raises(ValueError, match="unknown precision"):
        ttm_amd.ttm(2, A, B, precision="int3")
    with pytest.raises(TypeError, match="float32 and float64"):
        ttm_amd.ttm(2, A.half(), B.half())
    with pytest.raises(ValueError, match="C must be one dense block"):  # a layout that is no permutation
        ttm_amd.ttm(2, A, B, layout=[1, 1, 2])
