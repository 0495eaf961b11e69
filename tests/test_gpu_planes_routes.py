"""Where reduced-precision products over pre-converted operands (ttm_lowp.hip,
planes) run and where they give way: captured in a graph (the same kernel and
the same bits as the eager call, on every replay), in a fixed scratch region
that holds their workspace and in one that does not; and what they make of
infinities, NaN and values beyond 16 bits, against the kernel that takes one
thread per element."""
import numpy as np
import pytest

import lowp_emul as le
import refcases as rc
from test_gpu_precision import PRECS, _say, case, check_vs_emulation, folded, run
from test_zz_no_alloc import _bind, _call

pytestmark = pytest.mark.gpu


def _kernel(prec):
    return "k_fp8<" if prec == "fp8" else "k_planes<"


@pytest.mark.parametrize("prec", PRECS)
def test_captured_products_are_the_eager_ones(gpu, prec):
    """Odd extents in both views, and an aligned product of few blocks."""
    import torch
    import ttm_amd
    gen = torch.Generator(device=gpu)
    gen.manual_seed(3)
    for na, q, m, want in (([61, 67, 19], 2, 70, _kernel(prec)), ([301, 203], 1, 90, _kernel(prec)),
                           ([256, 300, 4], 2, 70, {"fp8": "k_fp8<", "bf16x3": "k_lowp<"}.get(prec, "k_planes<"))):
        A = torch.rand(na[::-1], generator=gen, device=gpu).sub_(0.5).permute(*range(len(na) - 1, -1, -1))
        B = torch.rand((m, na[q - 1]), generator=gen, device=gpu).sub_(0.5)
        _say(prec, na, q, m)
        eager = ttm_amd.ttm(q, A, B, precision=prec)
        sym = ttm_amd.last_kernel()
        assert sym[0].startswith(want), (na, sym)
        C = torch.empty_strided(eager.shape, eager.stride(), device=gpu)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ttm_amd.ttm(q, A, B, precision=prec, out=C)
        assert ttm_amd.last_kernel() == sym, (na, ttm_amd.last_kernel(), sym)
        for _ in range(4):
            C.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(C, eager), na
            other = ttm_amd.ttm(q, A, B + 1, precision=prec)  # eager work between the replays
            assert ttm_amd.last_kernel() == sym and not torch.equal(other, eager)
        # new inputs in the same buffers
        A.mul_(-0.5)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, ttm_amd.ttm(q, A, B, precision=prec)), na


# (na, pia, q, m, precision, kernel of the pooled call, kernel in the fixed region)
FIXED = [
    ([61, 67, 19], [1, 2, 3], 2, 70, "bf16", "k_planes<", "k_planes<"),
    ([301, 203], [1, 2], 1, 90, "fp16x2", "k_planes<", "k_planes<"),
    ([61, 67, 19], [1, 2, 3], 2, 70, "fp8", "k_fp8<", "k_fp8<"),
    # 36 to 71 million padded elements: 72 to 212 MB of planes
    ([1001, 35, 555], [1, 2, 3], 2, 30, "bf16", "k_planes<", "k_lowp_generic"),
    ([1001, 35, 555], [1, 2, 3], 2, 30, "fp16x2", "k_planes<", "k_lowp_generic"),
    ([1001, 35, 555], [1, 2, 3], 2, 30, "fp8", "k_fp8<", "k_lowp_generic"),
    ([35, 1001 * 555], [1, 2], 1, 30, "bf16x3", "k_planes<", "k_lowp_generic"),
    # aligned, few blocks: the fused tiles instead
    ([8192, 128 * 40], [1, 2], 1, 70, "bf16", "k_planes<", "k_lowp<"),
]


@pytest.mark.parametrize("na,pia,q,m,prec,pooled,fixed", FIXED)
def test_fixed_scratch_region(gpu, na, pia, q, m, prec, pooled, fixed):
    import torch
    import ttm_amd
    from ttm_amd._lib import PRECISION_NAMES
    _, fn = _bind()
    gen = torch.Generator(device=gpu)
    gen.manual_seed(4)
    nq = na[q - 1]
    A = torch.rand(int(np.prod(na)), generator=gen, device=gpu).sub_(0.5)
    B = torch.rand(m * nq, generator=gen, device=gpu).sub_(0.5)
    nc = list(na)
    nc[q - 1] = m
    wa, wc = rc.dense_strides(na, pia), rc.dense_strides(nc, pia)
    C = torch.full((int(np.prod(nc)),), float("nan"), device=gpu)
    ref = torch.full_like(C, float("nan"))
    _say(prec, na, q, m)
    st = _call(fn, q, na, pia, A, B, [m, nq], [2, 1], C, int(PRECISION_NAMES[prec]), torch.cuda.current_stream().cuda_stream)
    assert st == 0, ttm_amd.lib().ttm_last_error().decode()
    ran = ttm_amd.last_kernel()[0]
    assert ran.startswith(fixed), ran

    def product(kernel):
        ttm_amd.force_kernel(kernel)
        ttm_amd.ttm_raw(q, len(na), A, na, wa, pia, B, [m, nq], [2, 1], ref, nc, wc, precision=prec)
        ttm_amd.force_kernel(None)
        return ttm_amd.last_kernel()[0]

    assert product(None).startswith(pooled)
    if fixed != pooled:  # the same bits where the same kernel runs, else those of the kernel that did
        near = torch.linalg.vector_norm((C - ref).double()) / torch.linalg.vector_norm(ref.double())
        assert near < 1e-5, float(near)
        if fixed == "k_lowp<":
            return
        assert product("lowp_generic") == ran
    assert torch.equal(C, ref)


@pytest.mark.parametrize("prec", PRECS)
def test_special_values_as_one_thread_per_element(gpu, prec):
    """Results that involve an infinity, a NaN or a value beyond the 16-bit
    range are the same special values in both kernels, all others match the
    emulation.  Zeros meet the infinities only in the padding."""
    import torch
    import ttm_amd
    rng = np.random.default_rng(23)
    for na, pia, q, m, colmajor in (([63, 77, 5], [1, 2, 3], 2, 70, False), ([77, 65], [1, 2], 1, 66, True),
                                    ([33, 301, 3], [1, 2, 3], 2, 65, True)):
        a, wa, Bm, b, nb, pib, nc, wc = case(rng, na, pia, q, m, colmajor, "uniform")
        A3 = folded(a, na, pia, q)  # a view of a
        K, L, W = A3.shape
        plants = [(0, 0, 0, np.inf), (K - 1, L - 1, W - 1, -np.inf), (K // 2, L // 2, W // 2, np.nan)]
        if prec in ("bf16", "fp16"):  # rounds to an infinity
            plants.append((1, 3, min(1, W - 1), 3.4e38 if prec == "bf16" else 1e6))
        for k, l, i, v in plants:
            A3[k, l, i] = v
        Bm[5, L - 1] = np.inf
        b = (Bm.T if colmajor else Bm).reshape(-1).copy()
        label = f"{prec} {na} q={q}"
        _say(label)
        c = folded(run(torch, gpu, q, a, na, wa, pia, b, nb, pib, nc, wc, prec), nc, pia, q)
        assert ttm_amd.last_kernel()[0].startswith(_kernel(prec)), label
        g = folded(run(torch, gpu, q, a, na, wa, pia, b, nb, pib, nc, wc, prec, "lowp_generic"), nc, pia, q)
        assert ttm_amd.last_kernel()[0] == "k_lowp_generic"
        touched = np.zeros(c.shape, dtype=bool)
        for k, l, i, _ in plants:
            touched[k, :, i] = True
        touched[:, 5, :] = True
        assert np.array_equal(np.isnan(c[touched]), np.isnan(g[touched])), label
        assert np.array_equal(np.isposinf(c[touched]), np.isposinf(g[touched])), label
        assert np.array_equal(np.isneginf(c[touched]), np.isneginf(g[touched])), label
        assert not np.isfinite(c[touched]).any() and np.isfinite(c[~touched]).all(), label
        # the rest: without the planted fibres and row, whose results are masked
        clean, Bc = np.where(np.isfinite(A3) & (np.abs(A3) <= 1), A3, 0).astype(np.float32), Bm.copy()
        Bc[5, L - 1] = 0
        if prec == "fp16x2":  # its scales come from all finite values, as in the emulation
            with np.errstate(invalid="ignore"):
                ref = le.emulate(prec, A3, Bm)
            bound = 4 * L * 2.0 ** -24 * np.einsum("jl,kli->kji", np.abs(Bc.astype(np.float64)), np.abs(clean)) * 1.001
            assert np.all(np.abs(c - ref)[~touched] <= bound[~touched] + 1e-30), label
        else:
            check = np.where(touched, 0, c)
            ref0 = le.emulate(prec, clean, Bc)
            check_vs_emulation(np.where(touched, ref0, check), clean.reshape(-1), [W, L, K], [1, 2, 3], 2, Bc, prec, label)
