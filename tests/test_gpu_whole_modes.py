"""The contraction mode and the layout are whole numbers on the device as they
are on the host: a fraction raises TypeError in both front ends and is not cut
to the mode below it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q", [2.5, 2.0, np.float64(2.0), np.float32(1.5)])
def test_fractional_modes_are_refused(gpu, q):
    import torch
    import ttm_amd
    A, B = torch.rand(6, 8, 10, device=gpu), torch.rand(3, 8, device=gpu)
    for module in (ttm_amd, ttm_amd.ttmpy):
        with pytest.raises(TypeError):
            module.ttm(q, A, B)
        with pytest.raises(TypeError):
            module.ttm(q, A.cpu().numpy(), B.cpu().numpy())


def test_fractional_layouts_are_refused(gpu):
    import torch
    import ttm_amd
    A, B = torch.rand(6, 8, 10, device=gpu), torch.rand(3, 8, device=gpu)
    for X, Y in ((A, B), (A.cpu().numpy(), B.cpu().numpy())):
        with pytest.raises(TypeError):
            ttm_amd.ttm(2, X, Y, layout=[3.0, 2.0, 1.0])


@pytest.mark.parametrize("q", [2, np.int64(2), np.uint8(2)])
def test_whole_modes_of_any_type(gpu, q):
    import torch
    import ttm_amd
    A, B = torch.rand(6, 8, 10, device=gpu), torch.rand(3, 8, device=gpu)
    want = torch.einsum("jl,ilk->ijk", B.double(), A.double())
    for got in (ttm_amd.ttm(q, A, B), ttm_amd.ttm(q, A, B, layout=np.array([3, 2, 1])), ttm_amd.ttmpy.ttm(q, A, B)):
        assert torch.allclose(got.double(), want, rtol=0, atol=1e-5)
