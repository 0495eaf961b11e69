"""Reduced-precision products over pre-converted operands (ttm_lowp.hip,
k_planes and the any-extent FP8 conversions): odd extents and base pointers one
element past 16-byte alignment, at the edges of the 64 / 128 / 256 row and
128 / 256 column blocks and of the 32 / 64 / 128 index stages, both views, both
B orientations, against the CPU emulation of each arithmetic with the bound of
check_vs_emulation."""
import numpy as np
import pytest

import refcases as rc
from test_gpu_precision import PRECS, _say, case, check_vs_emulation, folded

pytestmark = pytest.mark.gpu

# (na, pi, q, m)
SHAPES = [([31, 37, 4], [1, 2, 3], 1, 64), ([33, 43, 3], [1, 2, 3], 1, 65), ([65, 127], [1, 2], 1, 128),
          ([129, 129], [1, 2], 1, 129), ([127, 31], [1, 2], 2, 63), ([43, 33, 3], [1, 2, 3], 2, 128),
          ([3, 65, 85], [1, 2, 3], 2, 130), ([1, 257, 9], [2, 3, 1], 2, 1), ([257, 129], [1, 2], 2, 70),
          ([2, 25, 11, 6], [1, 3, 2, 4], 2, 300)]
# enough 256 x 256 blocks to fill the chip
BIG = [([33, 32769], [1, 2], 1, 257), ([4097, 33, 8], [1, 2, 3], 2, 256)]


def _run(gpu, na, pia, q, m, colmajor, prec, offset):
    import torch
    import ttm_amd
    rng = np.random.default_rng(91)
    a, wa, Bm, b, nb, pib, nc, wc = case(rng, na, pia, q, m, colmajor, "uniform")

    def up(x):
        t = torch.zeros(x.size + offset, dtype=torch.float32, device=gpu)
        t[offset:] = torch.from_numpy(np.ascontiguousarray(x)).to(gpu)
        return t[offset:]

    guard = 4096  # elements past C stay as they were
    C = up(np.full(int(np.prod(nc)) + guard, 7.0, dtype=np.float32))
    label = f"{prec} {na} {pia} q={q} m={m} col={colmajor} offset={offset}"
    _say(label)
    ttm_amd.ttm_raw(q, len(na), up(a), na, wa, pia, up(b), nb, pib, C[:int(np.prod(nc))], nc, wc, precision=prec)
    torch.cuda.synchronize()
    sym, _ = ttm_amd.last_kernel()
    c = C.cpu().numpy()
    assert np.all(c[-guard:] == 7.0), label
    check_vs_emulation(folded(c[:-guard], nc, pia, q), a, na, pia, q, Bm, prec, label)
    return sym


@pytest.mark.parametrize("prec", PRECS)
def test_odd_extents_and_offsets_match_their_emulation(gpu, prec):
    want = "k_fp8<" if prec == "fp8" else "k_planes<"
    for i, (na, pia, q, m) in enumerate(SHAPES):
        for offset in (0, 1):
            sym = _run(gpu, na, pia, q, m, bool((i + offset) % 2), prec, offset)
            assert sym.startswith(want), (na, q, m, sym)


@pytest.mark.parametrize("prec", ["bf16", "fp16", "fp16x2", "bf16x3"])
def test_few_aligned_blocks_match_their_emulation(gpu, prec):
    """Aligned products of few blocks and long contractions: the planes' kernels
    for one and two planes, the fused tiles for three."""
    for na, pia, q, m in (([256, 300], [1, 2], 1, 65), ([1000, 129], [1, 2], 1, 256), ([132, 260], [1, 2], 2, 130)):
        sym = _run(gpu, na, pia, q, m, m == 256, prec, 0)
        assert sym.startswith("k_lowp<" if prec == "bf16x3" else "k_planes<"), (na, q, m, sym)


@pytest.mark.parametrize("prec", ["bf16", "fp16x2"])
def test_chip_filling_blocks_match_their_emulation(gpu, prec):
    for na, pia, q, m in BIG:
        sym = _run(gpu, na, pia, q, m, False, prec, 1)
        assert sym.startswith("k_planes<"), sym


def test_large_workspace_goes_back_to_the_device(gpu):
    """Planes of more than 8 GiB (three of 2.0e9 elements): after a
    synchronization the pool keeps at most 8 GiB of them."""
    import torch
    import ttm_amd
    from ttm_amd import _lib
    A = torch.zeros(801, 1201, 2003, device=gpu)
    B = torch.ones(3, 1201, device=gpu)
    C = ttm_amd.ttm(2, A, B, precision="bf16x3")
    assert ttm_amd.last_kernel()[0].startswith("k_planes<")
    torch.cuda.synchronize()
    assert _lib.workspace_bytes() <= 8 << 30
    assert not C.any()
