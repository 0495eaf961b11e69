"""The pipelined loop of the gemm tiles in the views where its blocks are
interior although A is not aligned: padded slabs wider than a block (w not a
multiple of the vector) and slabs of whole vectors at an element-aligned A, on
both sides of the line where the loop starts; each product names the loop it
ran.  And the CPU models of the loop's ragged slice and of the C[n][j] stores
over the tiles of three rows per lane (48 and 96 rows)."""
import itertools
import re

import numpy as np
import pytest

import refcases as rc
import test_gemm_pipeline as models

THREE_ROWS = [(t, vec, 3, nt, wm, 16) for t, vec, nt, wm in (("float", 4, 4, 1), ("float", 4, 4, 2), ("double", 2, 2, 1),
                                                             ("double", 2, 4, 2))]


@pytest.mark.parametrize("tn,bcol", list(itertools.product((True, False), repeat=2)))
@pytest.mark.parametrize("cfg", THREE_ROWS, ids=lambda c: "-".join(map(str, c)))
def test_ragged_slice_of_three_row_tiles(cfg, tn, bcol):
    models.test_ragged_slice_takes_its_elements(cfg + (tn, bcol, False))


@pytest.mark.parametrize("cfg", THREE_ROWS, ids=lambda c: "-".join(map(str, c)))
def test_tn_stores_of_three_row_tiles(cfg):
    models.test_tn_stores_cover_a_block_once(cfg[1:5])


# w: more than two blocks of 256 columns, odd; and whole vectors, read one element off alignment
@pytest.mark.gpu
@pytest.mark.parametrize("w,offset", [(521, 0), (520, 1), (523, 1)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_interior_blocks_of_padded_views(gpu, oracle, dtype, w, offset):
    import torch
    import ttm_amd
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    rng = np.random.default_rng(73)
    lines = {np.float32: lambda m: 96 if m > 64 else 192, np.float64: lambda m: 384}[dtype]
    for m in (10, 20, 40, 48, 64, 96, 130):
        line = lines(m)
        for nq in (line - 1, line, line + 7):
            na, pia = [w, nq, 2], [1, 2, 3]
            wa = rc.dense_strides(na, pia)
            nc = [w, m, 2]
            wc = rc.dense_strides(nc, pia)
            a = rng.uniform(-1, 1, int(np.prod(na))).astype(dtype)
            Bm = rng.uniform(-1, 1, (m, nq)).astype(dtype)
            A = torch.empty(a.size + offset, dtype=tdt, device=gpu)[offset:]
            A.copy_(torch.from_numpy(a))
            n = int(np.prod(nc))
            for colmajor in (False, True):
                b = (Bm.T if colmajor else Bm).reshape(-1).copy()
                label = f"{np.dtype(dtype).name} w={w}+{offset} nq={nq} m={m} col={colmajor}"
                print(label, flush=True)
                C = torch.full((n + 4096,), float("nan"), dtype=tdt, device=gpu)
                ttm_amd.force_kernel("gemm")
                ttm_amd.ttm_raw(2, 3, A, na, wa, pia, torch.from_numpy(b).to(gpu), [m, nq], [1, 2] if colmajor else [2, 1],
                                C[:n], nc, wc)
                torch.cuda.synchronize()
                sym = ttm_amd.last_kernel()[0]
                pipelined, padded = re.match(r"k_gemm<\w+, (\w+), .*, (\w+)>", sym).groups()
                assert padded == "true", (label, sym)
                assert pipelined == ("true" if nq >= line else "false"), (label, sym)
                c = C.cpu().numpy()
                assert np.all(np.isnan(c[n:])), label
                err = rc.normwise_error(c[:n], oracle.ttm_brute_f64(2, a, na, wa, b, m, colmajor, nc, wc), a, b)
                assert err <= 4 * nq * rc.eps(dtype), (label, sym, err)
