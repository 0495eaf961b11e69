"""The guarded slices of the gemm tiles in the NN view (ttm_gemm.hip,
load_tiles without element-aligned vectors): every thread reads one vector at
an in-range address -- rows past the contraction at its last row, columns past
the last one at column 0 -- and the store keeps exactly the elements that
belong to the slice.  A CPU model of both, over every tile shape, for edge
blocks, ragged contractions and contraction splits; and on the GPU products
whose blocks are all guarded, with infinities and NaN where a masked read
lands, against the FP64 brute force."""
import itertools

import numpy as np
import pytest

import refcases as rc

# vec, NT, WM of the k_gemm tiles (the loads of A do not depend on the rows)
TILES = [(4, 4, 1), (4, 4, 2), (2, 4, 1), (2, 2, 1), (2, 4, 2)]


@pytest.mark.parametrize("vec,NT,WM", TILES)
def test_guarded_reads_and_kept_elements(vec, NT, WM):
    BK, BN = 16, (4 // WM) * 16 * NT
    for (outer, w), ld in itertools.product(((1, BN + vec), (2, vec), (3, BN // 2 + vec), (5, 3 * vec)), (1, 17, 70)):
        ncols, size = outer * w, outer * ld * w
        for l0_split, nq in ((0, ld), (ld // 2, ld - ld // 2)):  # the whole contraction, and its second half
            a_off = l0_split * w
            for n0, l0 in itertools.product({0, (ncols - 1) // BN * BN}, {0, (nq - 1) // BK * BK}):
                for v in range(BK * BN // vec):
                    row, col = v // (BN // vec), v % (BN // vec) * vec
                    n, l = n0 + col, l0 + row
                    ok = n < ncols
                    k = n // w if ok else 0
                    base = k * ld * w + (n - k * w if ok else 0)
                    start = a_off + base + min(l, nq - 1) * w
                    assert 0 <= start and start + vec <= size
                    if ok and l < nq:  # kept whole: VEC columns of row l of one slab
                        i = n - k * w
                        assert i + vec <= w and start == k * ld * w + (l0_split + l) * w + i


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_products_of_guarded_blocks(gpu, oracle, dtype):
    """Fewer columns than a block, and B column-major with ragged rows."""
    import torch
    import ttm_amd
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    rng = np.random.default_rng(81)
    for (na, m), colmajor, plant in itertools.product((([44, 37, 3], 33), ([8, 97, 5], 40), ([84, 160, 2], 9),
                                                       ([12, 400, 9], 127)), (True, False), (False, True)):
        nq, pia = na[1], [1, 2, 3]
        wa = rc.dense_strides(na, pia)
        nc = [na[0], m, na[2]]
        wc = rc.dense_strides(nc, pia)
        a = rng.uniform(-1, 1, int(np.prod(na))).astype(dtype)
        if plant:  # the last row of the contraction, which rows past it re-read, and column 0
            A3 = a.reshape(na, order="F")
            A3[1, nq - 1, 0], A3[0, 0, 0], A3[2, nq - 1, na[2] - 1] = np.inf, -np.inf, np.nan
            a = A3.reshape(-1, order="F").copy()
        Bm = rng.uniform(0.5, 1, (m, nq)).astype(dtype)
        b = (Bm.T if colmajor else Bm).reshape(-1).copy()
        label = f"{np.dtype(dtype).name} {na} m={m} col={colmajor} plant={plant}"
        print(label, flush=True)
        C = torch.full((int(np.prod(nc)),), float("nan"), dtype=tdt, device=gpu)
        ttm_amd.force_kernel("gemm")
        ttm_amd.ttm_raw(2, 3, torch.from_numpy(a).to(gpu), na, wa, pia, torch.from_numpy(b).to(gpu), [m, nq],
                        [1, 2] if colmajor else [2, 1], C, nc, wc)
        torch.cuda.synchronize()
        assert ttm_amd.last_kernel()[0].startswith("k_gemm<"), label
        got = C.cpu().numpy().reshape(nc, order="F")
        clean = a.reshape(na, order="F").copy()
        touched = [(1, 0, np.inf), (0, 0, -np.inf), (2, na[2] - 1, np.nan)] if plant else []
        for i, k, value in touched:  # the fibres that hold one: all of their results are that value
            assert np.array_equal(got[i, :, k], np.full(m, value, dtype=dtype), equal_nan=True), (label, i, k)
            clean[i, :, k] = 0
            got[i, :, k] = 0
        clean = clean.reshape(-1, order="F").copy()
        err = rc.normwise_error(got.reshape(-1, order="F"), oracle.ttm_brute_f64(2, clean, na, wa, b, m, colmajor, nc, wc),
                                clean, b)
        assert err <= 4 * nq * rc.eps(dtype), (label, err)
