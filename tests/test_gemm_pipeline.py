"""The pipelined loop of the gemm tiles (ttm_gemm.hip, PIPE).

On the CPU: the ragged last slice of an interior tile (load_ragged), whose
vectors are read at moved, in-range addresses and shifted and masked at the
store, takes exactly the elements of the slice and no read leaves its operand.
On the GPU: contractions around the lengths where the loop starts and where
its last slices change (whole and ragged), every view, both B orientations,
against the FP64 brute force, normwise <= 4 n_q eps.
"""
import itertools

import numpy as np
import pytest

import refcases as rc
from test_tile_bounds_cpu import Bounds, gemm_configs, gemm_problems, gemm_tile_accesses


def _shift_mask(v, d, nvalid, zero=None):
    return [(v[x + d] if x + d < len(v) else v[x]) if x < nvalid else zero for x in range(len(v))]


@pytest.mark.parametrize("cfg", [c for c in gemm_configs() if not c[7]], ids=lambda c: "-".join(map(str, c)))
def test_ragged_slice_takes_its_elements(cfg):
    t, vec, JT, NT, WM, BK, tn, bcol, _ = cfg
    BM, BN = WM * 16 * JT, (4 // WM) * 16 * NT
    for nq, m in itertools.product((BK + 1, BK + vec - 1, 2 * BK + 3, 3 * BK - 1), (BM, BM + vec)):
        w, outer = (1, BN) if tn else (BN, 1)
        l0 = nq // BK * BK
        j0 = 0 if m == BM else BM  # the second row block of m = BM + vec reads rows past m in place of none

        def along(row, l):  # (addresses, kept elements) of a vector along l
            lc = min(l, nq - vec)
            nvalid = 0 if l >= nq else min(vec, nq - l)
            return _shift_mask([row + lc + x for x in range(vec)], l - lc, nvalid), row + lc

        def across(col, l, step):
            start = col + min(l, nq - 1) * step
            return _shift_mask([start + x for x in range(vec)], 0, vec if l < nq else 0), start

        for v in range(BK * BN // vec):
            if tn:
                n, r = v // (BK // vec), v % (BK // vec) * vec
                kept, start = along(n * nq, l0 + r)
                want = [n * nq + l0 + r + x if l0 + r + x < nq else None for x in range(vec)]
            else:
                r, n = v // (BN // vec), v % (BN // vec) * vec
                kept, start = across(n, l0 + r, w)
                want = [n + x + (l0 + r) * w if l0 + r < nq else None for x in range(vec)]
            assert kept == want and 0 <= start and start + vec <= outer * nq * w
        for v in range(BK * BM // vec):
            if bcol:
                if (m - j0) % vec and j0 + BM > m:
                    continue
                r, j = v // (BM // vec), j0 + v % (BM // vec) * vec
                jc = j if j + vec <= m else m - vec
                kept, start = across(jc, l0 + r, m)
                want = [jc + x + (l0 + r) * m if l0 + r < nq else None for x in range(vec)]
            else:
                j, r = j0 + v // (BK // vec), v % (BK // vec) * vec
                jc = min(j, m - 1)
                kept, start = along(jc * nq, l0 + r)
                want = [jc * nq + l0 + r + x if l0 + r + x < nq else None for x in range(vec)]
            assert kept == want and 0 <= start and start + vec <= m * nq


@pytest.mark.parametrize("cfg", sorted({c[1:5] for c in gemm_configs() if c[6]}), ids=lambda c: "-".join(map(str, c)))
def test_tn_stores_cover_a_block_once(cfg):
    """The C[n][j] epilogue with swapped operands: every element of a BM x BN
    block is stored by exactly one lane, whole vectors inside their rows."""
    vec, JT, NT, WM = cfg
    BM, BN = WM * 16 * JT, (4 // WM) * 16 * NT
    for m, ncols in ((BM, BN), (BM - 1, BN - 3), (1, 1)):
        seen = np.zeros((BN, BM), dtype=int)
        for tid in range(256):
            lane, wave = tid & 63, tid >> 6
            lc, lr, wm, wn = lane & 15, lane >> 4, wave % WM, wave // WM
            jr = wm * 16 * JT + JT * lc
            for nt, r in itertools.product(range(NT), range(4)):
                k = wn * 16 * NT + NT * (4 * lr + r if vec == 4 else 4 * r + lr) + nt
                if k >= ncols:
                    continue
                n = JT if JT % vec == 0 and jr + JT <= m else max(0, min(JT, m - jr))
                seen[k, jr:jr + n] += 1
        assert np.all(seen[:ncols, :m] == 1) and seen.sum() == ncols * m


@pytest.mark.parametrize("vec,NT,WM", [(4, 4, 1), (4, 4, 2), (2, 2, 1), (2, 4, 2)])
@pytest.mark.parametrize("view", ["TN", "NN", "PAD"])
def test_48_and_96_row_tiles_in_bounds(vec, NT, WM, view):
    JT, BK = 3, 16
    tn, pad = view == "TN", view == "PAD"
    BM, BN = WM * 16 * JT, (4 // WM) * 16 * NT
    for outer, nq, w, m in gemm_problems(vec, tn, BM, BN, BK, pad):
        wp = 1 if tn else (w + vec - 1) // vec * vec
        ncols = outer if tn else outer * wp
        nj, nn = (m + BM - 1) // BM, (ncols + BN - 1) // BN
        a_vec = (nq % vec == 0) if tn else (w % vec == 0 and not pad)
        c_vec = (m % vec == 0) if tn else (w % vec == 0 and not pad)
        for bcol, (jb, nb) in itertools.product((True, False), {(0, 0), (nj - 1, nn - 1)}):
            chk = Bounds({"a": outer * nq * w, "b": m * nq, "c": outer * m * w})
            gemm_tile_accesses(chk, vec, JT, NT, WM, BK, "TN" if tn else "NN", bcol, pad, ncols=ncols, nq=nq, ld=nq,
                               w=w, wp=wp, m=m, j0=jb * BM, n0=nb * BN, flags=int(a_vec) | 2 * int(c_vec) | 8, a_off=0,
                               b_off=0, c_off=0, a_len=0 if tn else (ncols // wp) * nq * w)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,ms", [(np.float32, (33, 47, 48, 65, 95, 96, 190, 288)), (np.float64, (33, 48, 90, 480))])
def test_48_and_96_row_tiles_vs_fp64(gpu, oracle, dtype, ms):
    import torch
    import ttm_amd
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    rng = np.random.default_rng(72)
    for m, (na, pia, q) in itertools.product(ms, (([40, 300], [1, 2], 1), ([401, 260], [1, 2], 1), ([260, 41], [1, 2], 2),
                                                  ([131, 400, 2], [1, 2, 3], 2))):
        nq = na[q - 1]
        wa = rc.dense_strides(na, pia)
        nc = list(na)
        nc[q - 1] = m
        wc = rc.dense_strides(nc, pia)
        a = rng.uniform(-1, 1, int(np.prod(na))).astype(dtype)
        b = rng.uniform(-1, 1, m * nq).astype(dtype)
        label = f"{np.dtype(dtype).name} {na} q={q} m={m}"
        print(label, flush=True)
        n = int(np.prod(nc))
        C = torch.full((n + 4096,), float("nan"), dtype=tdt, device=gpu)
        ttm_amd.force_kernel("gemm")
        ttm_amd.ttm_raw(q, len(na), torch.from_numpy(a).to(gpu), na, wa, pia, torch.from_numpy(b).to(gpu), [m, nq], [2, 1],
                        C[:n], nc, wc)
        torch.cuda.synchronize()
        sym = ttm_amd.last_kernel()[0]
        assert ", 3, 4, " in sym or ", 3, 2, " in sym, (label, sym)
        c = C.cpu().numpy()
        assert np.all(np.isnan(c[n:])), label
        err = rc.normwise_error(c[:n], oracle.ttm_brute_f64(q, a, na, wa, b, m, False, nc, wc), a, b)
        assert err <= 4 * nq * rc.eps(dtype), (label, sym, err)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,nqs", [(np.float32, (95, 96, 97, 112, 127, 192, 193, 225)),
                                       (np.float64, (383, 384, 385, 399, 416, 433))])
def test_contractions_around_the_pipelined_loop(gpu, oracle, dtype, nqs):
    import torch
    import ttm_amd
    tdt = torch.float32 if dtype == np.float32 else torch.float64
    rng = np.random.default_rng(71)
    for nq, m, view in itertools.product(nqs, (10, 20, 40, 130), ("tn", "nn", "pad")):
        na, pia, q = {"tn": ([nq, 300], [1, 2], 1), "nn": ([260, nq], [1, 2], 2),
                      "pad": ([131, nq, 2], [1, 2, 3], 2)}[view]
        wa = rc.dense_strides(na, pia)
        nc = list(na)
        nc[q - 1] = m
        wc = rc.dense_strides(nc, pia)
        a = rng.uniform(-1, 1, int(np.prod(na))).astype(dtype)
        Bm = rng.uniform(-1, 1, (m, nq)).astype(dtype)
        A = torch.from_numpy(a).to(gpu)
        for colmajor in (False, True):
            b = (Bm.T if colmajor else Bm).reshape(-1).copy()
            label = f"{np.dtype(dtype).name} {view} nq={nq} m={m} col={colmajor}"
            print(label, flush=True)
            C = torch.full((int(np.prod(nc)),), float("nan"), dtype=tdt, device=gpu)
            ttm_amd.force_kernel("gemm")
            ttm_amd.ttm_raw(q, len(na), A, na, wa, pia, torch.from_numpy(b).to(gpu), [m, nq],
                            [1, 2] if colmajor else [2, 1], C, nc, wc)
            torch.cuda.synchronize()
            c64 = oracle.ttm_brute_f64(q, a, na, wa, b, m, colmajor, nc, wc)
            err = rc.normwise_error(C.cpu().numpy(), c64, a, b)
            assert err <= 4 * nq * rc.eps(dtype), (label, ttm_amd.last_kernel(), err)
