"""Column-major B whose columns no vector ends at (m % VEC != 0): the last row
block of the gemm tiles (ttm_gemm.hip) keeps the unguarded loop, its vector
across row m reading on into the next column, and only the last column's slice
is guarded.  A CPU model of those reads (in bounds, and the right elements for
every row of C), and products on the GPU with infinities and NaN in the rows
that such a vector picks up, against the FP64 brute force."""
import itertools

import numpy as np
import pytest

import refcases as rc
from test_gemm_pipeline import _shift_mask


@pytest.mark.parametrize("vec,BM", [(4, 16), (4, 32), (4, 48), (4, 64), (4, 96), (4, 128), (2, 16), (2, 32), (2, 48),
                                    (2, 64), (2, 96), (2, 128)])
def test_reads_of_a_straddling_block(vec, BM):
    BK = 16
    for m, nq in itertools.product({vec + 1, BM - 1, BM + 1, BM + vec - 1, 2 * BM - 1, 2 * BM + 3},
                                   (2, BK - 1, BK, BK + 1, 2 * BK, 2 * BK + 5)):
        if m % vec == 0 or m <= vec:
            continue
        j0 = (m - 1) // BM * BM  # the last row block
        if j0 + BM <= m:
            continue
        nwhole, nslices = (nq - 1) // BK, -(-nq // BK)
        assert nslices - nwhole == 1
        for s, v in itertools.product(range(nslices), range(BK * BM // vec)):
            l, j = s * BK + v // (BM // vec), j0 + v % (BM // vec) * vec
            at = (j if j < m else m - vec) + min(l, nq - 1) * m
            if s < nwhole:  # load_full
                assert l < nq and 0 <= at and at + vec <= m * nq
                kept = [at + x for x in range(vec)]
            else:  # load_ragged
                ac = min(at, nq * m - vec)
                assert 0 <= ac
                kept = _shift_mask([ac + x for x in range(vec)], at - ac, vec if l < nq else 0)
            for x in range(vec):
                if l >= nq:
                    assert kept[x] is None
                elif j + x < m:  # the others belong to rows past m, which are never stored
                    assert kept[x] == j + x + l * m
                else:
                    assert 0 <= kept[x] < m * nq


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,ms", [(np.float32, (5, 9, 17, 41, 63, 65, 95, 129, 258)), (np.float64, (3, 9, 17, 41, 63, 65, 95, 129))])
def test_straddling_blocks_vs_fp64(gpu, oracle, dtype, ms):
    import torch
    import ttm_amd
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    rng = np.random.default_rng(74)
    for m, nq, view in itertools.product(ms, (2, 16, 33, 96, 401, 1040), ("nn", "tn", "pad")):
        na, pia, q = {"tn": ([nq, 300], [1, 2], 1), "nn": ([260, nq], [1, 2], 2), "pad": ([521, nq], [1, 2], 2)}[view]
        wa = rc.dense_strides(na, pia)
        nc = list(na)
        nc[q - 1] = m
        wc = rc.dense_strides(nc, pia)
        a = rng.uniform(0.5, 1, int(np.prod(na))).astype(dtype)
        Bm = rng.uniform(-1, 1, (m, nq)).astype(dtype)
        Bm[0, :] = np.nan  # the next column's first rows
        Bm[1, nq - 1] = np.inf
        b = Bm.T.reshape(-1).copy()
        label = f"{np.dtype(dtype).name} {view} nq={nq} m={m}"
        print(label, flush=True)
        n = int(np.prod(nc))
        # B at the end of its allocation's used part, followed by values that must not be read
        Bd = torch.full((b.size + 64,), float("nan"), dtype=tdt, device=gpu)
        Bd[:b.size] = torch.from_numpy(b)
        C = torch.full((n + 4096,), 7.0, dtype=tdt, device=gpu)
        ttm_amd.force_kernel("gemm")
        ttm_amd.ttm_raw(q, 2, torch.from_numpy(a).to(gpu), na, wa, pia, Bd[:b.size], [m, nq], [1, 2], C[:n], nc, wc)
        torch.cuda.synchronize()
        assert ttm_amd.last_kernel()[0].startswith("k_gemm<"), label
        c = C.cpu().numpy()
        assert np.all(c[n:] == 7.0), label
        got = rc.as_nd(c[:n], nc, wc)
        rows = np.moveaxis(got, q - 1, 0)
        assert np.isnan(rows[0]).all() and np.isposinf(rows[1]).all(), label
        assert np.isfinite(rows[2:]).all(), label
        clean = Bm.copy()
        clean[:2] = 0
        bc = clean.T.reshape(-1).copy()
        ref = rc.as_nd(oracle.ttm_brute_f64(q, a, na, wa, bc, m, True, nc, wc), nc, wc)
        rows[:2] = 0
        err = rc.normwise_error(got.reshape(-1), ref.reshape(-1), a, bc)
        assert err <= 4 * nq * rc.eps(dtype), (label, ttm_amd.last_kernel(), err)
