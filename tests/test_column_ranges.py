"""Reduced-precision products whose converted A is larger than one workspace
run in ranges of columns (ttm_columns.hpp): the ranges cover every column of a
fold once (tests/cpp/column_ranges.cpp, host code), and on the GPU each range's
results are the bits of a product over its columns alone, while the workspace
pool keeps its memory instead of mapping it on every call."""
import math
import pathlib
import shutil
import subprocess

import numpy as np
import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


def test_ranges_cover_every_column_once():
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    build = ROOT / "tests" / "_build"
    build.mkdir(exist_ok=True)
    exe = build / "column_ranges"
    cmd = [gxx, "-O1", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
           f"-I{ROOT / 'ttm_amd' / 'csrc'}", str(ROOT / "tests" / "cpp" / "column_ranges.cpp"), "-o", str(exe)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.startswith("0 violations"), run.stdout + run.stderr


@pytest.mark.parametrize("outer,w,i0,ncols", [(1, 1537, 0, 1537), (2, 1539, 1280, 259), (1, 1282, 1024, 258), (3, 5, 0, 15),
                                              (4, 259, 0, 1036), (2, 512, 256, 256), (1, 770, 512, 258)])
def test_nn_stores_of_a_range_cover_its_columns_once(outer, w, i0, ncols):
    """The C[j][n] epilogue of k_planes and k_fp8 on a range (i0: its first
    column within its slab, 0 for whole slabs): a lane's four columns go out as
    one vector only inside one slab and inside the range, so that no element
    of the next row or beyond C is written."""
    m, BN = 2, 128
    seen = np.zeros(outer * m * w, dtype=int)
    c0 = i0  # C's element of the range's first column (slab 0)
    for ncol0 in range(0, -(-ncols // BN) * BN, 4):
        if ncol0 >= ncols:
            continue
        k, i = divmod(ncol0, w)
        whole = i + 4 <= w and ncol0 + 4 <= ncols
        for j in range(m):
            base = c0 + k * m * w + i + j * w
            for nt in range(4):
                ii, kk = i + nt, 0
                while ii >= w:
                    ii, kk = ii - w, kk + 1
                if whole:
                    seen[base + nt] += 1
                elif ncol0 + nt < ncols:
                    seen[base + kk * m * w + ii - i] += 1
    want = np.zeros_like(seen).reshape(outer, m, w)
    if i0:
        want[0, :, i0:i0 + ncols] = 1
    else:
        want[: ncols // w, :, :] = 1
    assert np.array_equal(seen.reshape(outer, m, w), want)


# first-order extents, q: q fastest, slabs of 33, one slab, two slabs wider than a range
VIEWS = [([1023, 1500001], 1), ([33, 1023, 45001], 2), ([1500001, 1023], 2), ([750001, 1023, 2], 2)]


def _tensor(torch, buf, na):
    """A view of buf with extents na, first mode fastest."""
    strides, n = [], 1
    for x in na:
        strides.append(n)
        n *= x
    return torch.as_strided(buf, na, strides)


@pytest.mark.gpu
@pytest.mark.parametrize("prec,views,columns", [("bf16x3", VIEWS, 699050), ("fp16x2", VIEWS, 1048576),
                                                ("fp8", [([1023, 4200001], 1), ([4200001, 1023], 2)], 4067197)])
def test_ranges_match_products_of_their_columns(gpu, prec, views, columns):
    """`columns`: about the columns of a range (4 GiB over the bytes of one)."""
    import torch
    import ttm_amd
    from ttm_amd import _lib
    gen = torch.Generator(device=gpu)
    gen.manual_seed(6)
    numel = max(math.prod(na) for na, _ in views)
    buf = torch.empty(numel, device=gpu)
    for part in buf.split(1 << 30):
        part.uniform_(-1, 1, generator=gen)
    m = 70
    want = "k_fp8<" if prec == "fp8" else "k_planes<"
    for na, q in views:
        A = _tensor(torch, buf, na)
        B = torch.empty((m, na[q - 1]), device=gpu).uniform_(-1, 1, generator=gen)
        print(prec, na, q, flush=True)
        C = ttm_amd.ttm(q, A, B, precision=prec)
        assert ttm_amd.last_kernel()[0].startswith(want)
        torch.cuda.synchronize()
        assert 1 << 30 < _lib.workspace_bytes() <= 8 << 30  # kept, and bounded
        assert torch.isfinite(C).all()
        # around the first range's end and at both ends of the last mode of the columns
        mode = len(na) - 1 if na[-1] > 1000 and q != len(na) else 0
        per = 33 if na[0] == 33 else 1
        at = columns // per
        for lo in {0, min(na[mode] - 1023, max(0, at - 700)), na[mode] - 1023}:
            n = 1023 if per == 1 else 64  # odd, so that the parts take the same kernels
            Ap = A.narrow(mode, lo, n)
            strides = sorted(range(len(na)), key=lambda d: A.stride(d))
            Ap = Ap.permute(*reversed(strides)).contiguous().permute(*[list(reversed(strides)).index(d) for d in range(len(na))])
            Cp = ttm_amd.ttm(q, Ap, B, precision=prec)
            assert ttm_amd.last_kernel()[0].startswith(want)
            assert torch.equal(Cp, C.narrow(mode, lo, n)), (na, q, lo)
        del C
