"""fp32 GEMM vs fp64 NumPy matmul, through the C-ABI (haste_hip_gemm_f32)."""
import numpy as np
import pytest

from util import dev, host, relerr

pytestmark = pytest.mark.gpu

SHAPES = [
    # (trans_a, M, N, K)
    (False, 128, 128, 16), (False, 256, 384, 64), (False, 100, 200, 50), (False, 1, 1, 1),
    (False, 37, 53, 29), (True, 128, 128, 32), (True, 70, 130, 45), (True, 5, 20, 33),
    (False, 6400, 2048, 512),   # x*W of the metric config
    (False, 512, 2048, 6400),   # dW: split along K
    (True, 512, 2048, 6400),    # dR: split along K, A = h^T
    (False, 6400, 512, 2048),   # dx
    (False, 96, 96, 5000),      # split-K with ragged tiles
    # a step's products: up to 32 rows in the kernel that streams B into the MFMA operands, more in K pieces
    (False, 64, 1024, 4096), (False, 47, 6144, 1536), (False, 33, 772, 3000), (False, 128, 1024, 4096),
    (False, 100, 768, 3072),
    (False, 1, 2048, 512), (False, 16, 6144, 1536), (False, 5, 1300, 5200), (False, 32, 768, 3072),
    (False, 17, 4100, 332), (False, 3, 64, 1024), (False, 32, 16384, 1000),
    # whole tiles beside edge tiles, K pieces whose last stage is and is not whole
    (False, 300, 260, 250), (True, 384, 1000, 1600), (False, 640, 192, 2048), (True, 800, 512, 1000),
    (False, 1024, 1024, 17),
]


@pytest.mark.parametrize("trans_a,M,N,K", SHAPES)
@pytest.mark.parametrize("accumulate", [False, True])
def test_gemm_matches_numpy(trans_a, M, N, K, accumulate):
    from haste_amd import ops
    import torch
    r = np.random.default_rng(M * 7 + N * 3 + K)
    a = r.standard_normal((K, M) if trans_a else (M, K)).astype(np.float32)
    b = r.standard_normal((K, N)).astype(np.float32)
    c0 = r.standard_normal((M, N)).astype(np.float32)
    print("gemm", trans_a, M, N, K, accumulate, flush=True)
    out = dev(c0)
    ops.gemm(dev(a), dev(b), out=out, trans_a=trans_a, accumulate=accumulate)
    torch.cuda.synchronize()
    a64 = a.astype(np.float64)
    ref = (a64.T if trans_a else a64) @ b.astype(np.float64)
    if accumulate:
        ref = ref + c0
    assert relerr(host(out), ref) < 1e-5  # fp32 accumulation over K up to 6400


@pytest.mark.parametrize("trans_a,M,N,K,pad_a,pad_b", [(False, 256, 256, 128, 4, 4), (True, 384, 128, 96, 3, 1),
                                                        (False, 130, 100, 64, 3, 4), (True, 128, 256, 2048, 4, 0)])
def test_gemm_padded_leading_dimensions(trans_a, M, N, K, pad_a, pad_b):
    """Operands that are column ranges of wider arrays (lda > K, ldb > N), aligned and not."""
    import torch
    from haste_amd import lib as hlib
    g = torch.Generator().manual_seed(M + N + K)
    a_full = torch.randn((K, M + pad_a) if trans_a else (M, K + pad_a), generator=g).cuda()
    b_full = torch.randn(K, N + pad_b, generator=g).cuda()
    a = a_full[:, :M] if trans_a else a_full[:, :K]
    out = torch.zeros(M, N, device="cuda")
    print("gemm padded", trans_a, M, N, K, pad_a, pad_b, flush=True)
    hlib.call("haste_hip_gemm_f32", int(trans_a), M, N, K, a_full, a_full.stride(0), b_full, b_full.stride(0),
              out, out.stride(0), 0)
    torch.cuda.synchronize()
    ref = (a.double().t() if trans_a else a.double()) @ b_full[:, :N].double()
    assert relerr(host(out), host(ref)) < 1e-5


def test_gemm_split_k_is_run_to_run_identical():
    from haste_amd import ops
    import torch
    r = np.random.default_rng(5)
    a = dev(r.standard_normal((512, 6400)))
    b = dev(r.standard_normal((6400, 2048)))
    o1 = ops.gemm(a, b)
    o2 = ops.gemm(a, b)
    torch.cuda.synchronize()
    assert torch.equal(o1, o2)


@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (64, 64), (65, 63), (100, 7, 33), (6400, 512), (512, 2048)])
def test_transpose(shape):
    import torch
    from haste_amd import ops
    a = torch.randn(*shape, device="cuda")
    out = ops.transpose(a)
    ref = a.reshape(-1, shape[-1]).t().contiguous().reshape((shape[-1],) + tuple(shape[:-1]))
    assert out.shape == ref.shape and torch.equal(out, ref)


@pytest.mark.parametrize("shapes", [((1, 1), (3, 5), (65, 63)), ((100, 7, 33), (64, 64), (2, 130)),
                                    ((6400, 512), (512, 2048), (512, 2048))])
def test_three_transposes_in_one_launch(shapes):
    import torch
    from haste_amd import ops
    ms = [torch.randn(*s, device="cuda") for s in shapes]
    outs = ops.transpose3(*ms)
    for m, out in zip(ms, outs):
        assert torch.equal(out, ops.transpose(m))
    for dtype in (torch.float64, torch.float16):
        cast = [m.to(dtype) for m in ms]
        for m, out in zip(cast, ops.transpose3(*cast)):
            assert torch.equal(out, ops.transpose(m))


@pytest.mark.parametrize("trans_a", [True, False])
def test_gemm_operand_of_more_than_2_gib(trans_a):
    """B[K, N] of 2.1 GB (the dv of a backward pass with T*N*H = 2^27 and beyond: dW = x^T dv
    contracts over T*N): the contraction is cut into runs whose panels the kernel can address.
    Against the float64 product of the same float32 operands, on the GPU (NumPy would take
    minutes)."""
    import torch
    from haste_amd import ops
    M, N, K = 256, 2048, (1 << 18) + 48
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randn((K, M) if trans_a else (M, K), generator=g, device="cuda")
    b = torch.randn(K, N, generator=g, device="cuda")
    assert b.numel() * 4 > 1 << 31
    print("gemm over 2 GiB, trans_a =", trans_a, flush=True)
    c0 = torch.randn(M, N, generator=g, device="cuda")
    out = c0.clone()
    ops.gemm(a, b, out=out, trans_a=trans_a, accumulate=True)
    torch.cuda.synchronize()
    ref = c0.double()
    step = 1 << 15   # float64 copies of the operands, a slab of K at a time
    for k0 in range(0, K, step):
        a_slab = (a[k0:k0 + step].double().t() if trans_a else a[:, k0:k0 + step].double())
        ref += a_slab @ b[k0:k0 + step].double()
    err = float((out.double() - ref).abs().max() / ref.abs().max())
    assert err < 1e-5, err


def _bound(a64, b64, K):
    """What fp32 accumulation of exact products can be off by, element by element: one rounding
    (at most 2^-23: the matrix unit may truncate) per 16 k of the sum of the large partial
    products, 5 of the small ones, which are 2^-8 of them, and one each for adding the two sums
    and up to 64 K pieces; the partial products left out are 2^-24."""
    return (K / 16 * (1 + 5 / 256) + 66) * 2.0 ** -23 * (np.abs(a64) @ np.abs(b64))


@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("M,N,K", [
    (1, 1, 1), (63, 127, 31), (64, 128, 32), (65, 129, 33), (127, 2, 63), (128, 130, 64), (129, 255, 65),
    (66, 3, 7), (192, 257, 1029), (70, 70, 4099)])
@pytest.mark.parametrize("scale_a,scale_b", [(1.0, 1.0), (1e-37, 1.0), (1e-20, 1e-18), (1e30, 1e-30), (1e18, 1e18),
                                             (1e-37, 1e18), (1e-36, 1e10), (1e-41, 1e30), (1e30, 1e-43), (1e-22, 1e-22)])
def test_gemm_edges_and_range(trans_a, M, N, K, scale_a, scale_b):
    """Every edge of the 64 / 128 x 128 tiles and of the 32 k of a stage, operands from the smallest
    to the largest floats (what a float cannot represent of the result excepted)."""
    import torch
    from haste_amd import ops
    r = np.random.default_rng(M + 31 * N + 17 * K)
    a = (r.standard_normal((K, M) if trans_a else (M, K)) * scale_a).astype(np.float32)
    b = (r.standard_normal((K, N)) * scale_b).astype(np.float32)
    print("gemm edges", trans_a, M, N, K, scale_a, scale_b, flush=True)
    out = host(ops.gemm(dev(a), dev(b), trans_a=trans_a)).astype(np.float64)
    torch.cuda.synchronize()
    a64, b64 = (a.T if trans_a else a).astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(out - a64 @ b64) <= _bound(a64, b64, K) + K * 2.0 ** -149)


@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("M,N,K", [(150, 140, 512), (40, 130, 75), (512, 256, 2080)])
def test_gemm_operands_of_all_sizes_in_a_tile(trans_a, M, N, K):
    """Rows of A and columns of B from the smallest floats to large ones side by side: every result as
    accurate as its own operands allow, whatever lies beside it."""
    import torch
    from haste_amd import ops
    r = np.random.default_rng(M + N + K)
    rows, cols = 10.0 ** r.uniform(-44, 10, (M, 1)), 10.0 ** r.uniform(-44, 10, (1, N))
    rows[::5], cols[:, ::5] = 1.0, 1.0
    a = (r.standard_normal((M, K)) * rows).astype(np.float32)
    b = (r.standard_normal((K, N)) * cols).astype(np.float32)
    out = host(ops.gemm(dev(a.T if trans_a else a), dev(b), trans_a=trans_a)).astype(np.float64)
    torch.cuda.synchronize()
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(out - a64 @ b64) <= _bound(a64, b64, K) + K * 2.0 ** -149)


@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("M,N,K", [(130, 104, 512), (60, 200, 100)])
def test_gemm_memory_beside_the_matrices_does_not_matter(trans_a, M, N, K):
    """Operands that are columns of wider matrices: bit for bit the same product whatever the other columns hold."""
    import torch
    from haste_amd import lib
    gen = torch.Generator().manual_seed(M)
    wide = [torch.randn(K if trans_a else M, 260, generator=gen), torch.randn(K, 260, generator=gen)]
    wide = [m.cuda() for m in wide] if trans_a else [torch.randn(M, K, generator=gen).cuda(), wide[1].cuda()]
    outs = []
    for beside in (0.0, float("nan"), float("inf"), 3e38, 1e-40):
        if trans_a:
            wide[0][:, M:] = beside
        wide[1][:, N:] = beside
        out = torch.empty(M, N, device="cuda")
        lib.call("haste_hip_gemm_f32", int(trans_a), M, N, K, wide[0], wide[0].stride(0), wide[1], 260, out, N, 0)
        outs.append(out)
    assert all(torch.equal(out, outs[0]) for out in outs)
    a = wide[0][:, :M].t() if trans_a else wide[0]
    a64, b64 = a.cpu().double().numpy(), wide[1][:, :N].cpu().double().numpy()
    assert np.all(np.abs(host(outs[0]) - a64 @ b64) <= _bound(a64, b64, K))


@pytest.mark.parametrize("K", [1, 4, 6])
def test_gemm_few_rows_of_a_long_stride(K):
    """Rows 2^26 floats apart: the byte offset of rows that a stage of 32 k looks at beyond the last one
    wraps at 2^32, to the panel's first rows."""
    import torch
    from haste_amd import lib
    M, N, ld = 130, 70, 1 << 26
    r = np.random.default_rng(K)
    a, b = (r.standard_normal((K, n)).astype(np.float32) for n in (M, N))
    views = []
    for m in (a, b):
        t = torch.empty((K - 1) * ld + m.shape[1], device="cuda")
        views.append(t.as_strided(m.shape, (ld, 1)))
        views[-1].copy_(torch.from_numpy(m))
    out = torch.empty(M, N, device="cuda")
    print("gemm long stride", K, ld, flush=True)
    lib.call("haste_hip_gemm_f32", 1, M, N, K, views[0], ld, views[1], ld, out, N, 0)
    torch.cuda.synchronize()
    a64, b64 = a.T.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(host(out) - a64 @ b64) <= _bound(a64, b64, K))


@pytest.mark.parametrize("trans_a", [False, True])
def test_gemm_operands_that_are_not_finite(trans_a):
    """Infinities, NaNs and values beyond the largest bfloat16 give what float arithmetic gives, and
    leave the rest of their tile alone."""
    import torch
    from haste_amd import ops
    r = np.random.default_rng(3)
    M, N, K = 200, 150, 96
    a, b = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((K, N)).astype(np.float32)
    a[3, 5], a[100, 7], b[9, 20], a[150, 11] = np.inf, -np.inf, np.nan, 3.4e38
    b[11] = np.where(np.abs(b[11]) > 1, b[11] / 4, b[11])
    b[5, 30] = 0.0
    out = host(ops.gemm(dev(a.T if trans_a else a), dev(b), trans_a=trans_a))
    torch.cuda.synchronize()
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(out[inf], ref[inf].astype(np.float32))
    rows = [i for i in range(M) if i not in (3, 100, 150)]
    cols = [j for j in range(N) if j != 20]
    a64, b64 = a[rows].astype(np.float64), b[:, cols].astype(np.float64)
    assert np.all(np.abs(out[np.ix_(rows, cols)] - a64 @ b64) <= _bound(a64, b64, K))


@pytest.mark.parametrize("M,N,K", [(512, 512, 512), (256, 512, 6400), (128, 128, 40000)])
def test_gemm_is_at_least_as_accurate_as_float_products(M, N, K):
    """Against the float64 product: no further from it than a float32 product whose partial sums
    are rounded every two k, as the fp32 matrix instruction rounds them (on the CPU)."""
    import torch
    from haste_amd import ops
    g = torch.Generator().manual_seed(M + K)
    a, b = torch.randn(M, K, generator=g), torch.randn(K, N, generator=g)
    out = ops.gemm(a.cuda(), b.cuda()).cpu().double()
    rows = slice(0, 16)
    ref = a[rows].double() @ b.double()
    acc = torch.zeros(16, N)
    for k in range(0, K, 2):
        acc = (acc.double() + a[rows, k:k + 2].double() @ b[k:k + 2].double()).float()
    assert (out[rows] - ref).norm() <= (acc.double() - ref).norm()
