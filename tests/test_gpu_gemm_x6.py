"""GPU: the bf16-plane ("x6") fp32 products (mpq_gemm_x6, mpq_rankspace_pack) against fp64 and
against the fp32 MFMA kernel (mpq_gemm_f32), and the VAMP solver on the packed operator."""
import pytest
import torch

from mpq_amd import ops

pytestmark = pytest.mark.gpu


def _op(B, trans):
    return B.T if trans else B


def test_gemm_x6_known_answer_pins_the_plane_products(gpu):
    """a = 1 + 2^-9 + 2^-18 and b = 1 + 2^-10 + 2^-19 split into bf16 planes (1, 2^-9, 2^-18) and
    (1, 2^-10, 2^-19).  The six kept products sum to 1 + 2^-9 + 2^-10 + 2^-17 exactly (the dropped
    a1 b2, a2 b1, a2 b2 are below 2^-27, under half an fp32 ulp of the product), so with K = 32
    equal terms every entry is exactly 32 * that; dropping or mis-pairing any one plane product
    moves an entry by at least 32 * 2^-19 = 2^-14."""
    M, N, K = 160, 256, 32
    a = 1.0 + 2.0 ** -9 + 2.0 ** -18
    b = 1.0 + 2.0 ** -10 + 2.0 ** -19
    sign_r = torch.where(torch.arange(M) % 3 == 0, -1.0, 1.0)
    sign_c = torch.where(torch.arange(N) % 5 == 1, -1.0, 1.0)
    A = (sign_r.view(-1, 1) * a).expand(M, K).contiguous().float()
    B = (sign_c.view(1, -1) * b).expand(K, N).contiguous().float()
    assert float(A[1, 0]) == a and float(B[0, 0]) == b  # representable in fp32
    exact = 32.0 * (1.0 + 2.0 ** -9 + 2.0 ** -10 + 2.0 ** -17)
    for trans in (False, True):
        Bp = ops.gemm_x6_pack_b((B.T.contiguous() if trans else B).to(gpu), trans_b=trans)
        C = ops.gemm_x6(A.to(gpu), Bp, N).cpu().double()
        ref = exact * sign_r.view(-1, 1).double() * sign_c.view(1, -1).double()
        assert torch.equal(C, ref), float((C - ref).abs().max())


@pytest.mark.parametrize("M,N,K,trans", [(128, 512, 512, False), (128, 512, 512, True), (100, 256, 1024, False),
                                         (384, 1024, 2048, True), (1, 128, 32, False), (257, 384, 4096, False),
                                         (130, 256, 96, True)])
def test_gemm_x6_matches_fp64(gpu, M, N, K, trans):
    """Entry-wise error relative to sum_k |a_k b_k| against fp64: within twice the fp32 MFMA kernel's
    on the same operands, and below 2e-6.  K slices of a multiple of four 16-k slabs run the LDS-ring
    kernel, the others (K = 32, 96 here) the register-staged one (a dropped 2^-16-order plane product shows at K = 32 as
    ~3e-6 and above; the known-answer test pins the plane set exactly)."""
    g = torch.Generator().manual_seed(M * 13 + N + K)
    # columns of A and rows of op(B) with a spread of magnitudes (1e-3 .. 1e3)
    A = torch.randn(M, K, generator=g) * torch.exp(3.0 * torch.randn(1, K, generator=g))
    B = torch.randn(N, K, generator=g) if trans else torch.randn(K, N, generator=g)
    Bp = ops.gemm_x6_pack_b(B.to(gpu), trans_b=trans)
    C6 = ops.gemm_x6(A.to(gpu), Bp, N).cpu().double()
    Cf = ops.gemm(A.to(gpu), B.to(gpu), trans_b=trans).cpu().double()
    Bo = _op(B.double(), trans)
    ref = A.double() @ Bo
    mag = A.double().abs() @ Bo.abs()
    e6 = float(((C6 - ref).abs() / mag).max())
    ef = float(((Cf - ref).abs() / mag).max())
    print(f"x6 {e6:.3e} fp32 {ef:.3e}")
    assert e6 <= max(2.0 * ef, 2e-7) and e6 < 2e-6
    # deterministic (fixed split order)
    assert torch.equal(ops.gemm_x6(A.to(gpu), Bp, N).cpu().double(), C6)


def test_gemm_x6_pack_nn_equals_nt(gpu):
    g = torch.Generator().manual_seed(3)
    A = torch.randn(200, 768, generator=g)
    B = torch.randn(768, 640, generator=g)
    p1 = ops.gemm_x6_pack_b(B.to(gpu), trans_b=False)
    p2 = ops.gemm_x6_pack_b(B.T.contiguous().to(gpu), trans_b=True)
    assert torch.equal(p1.cpu(), p2.cpu())
    assert torch.equal(ops.gemm_x6(A.to(gpu), p1, 640).cpu(), ops.gemm_x6(A.to(gpu), p2, 640).cpu())


def test_gemm_x6_rejects_unsupported_shapes(gpu):
    A = torch.randn(8, 96, device=gpu)
    with pytest.raises(ValueError):
        ops.gemm_x6_pack_b(torch.randn(96, 100, device=gpu))   # N % 128 != 0
    with pytest.raises(ValueError):
        ops.gemm_x6_pack_b(torch.randn(48, 128, device=gpu))   # K % 32 != 0
    assert ops.rankspace_pack(torch.randn(200, 200, device=gpu), torch.randn(200, 200, device=gpu)) is None
    Bp = ops.gemm_x6_pack_b(torch.randn(96, 128, device=gpu))
    C = ops.gemm_x6(A, Bp, 128)
    assert C.shape == (8, 128)


def test_rankspace_pack_layout(gpu):
    """The packed operator is [V for r V | V for x V^T | Vs for x Vs]: each third gives the same
    product as mpq_gemm_x6 on the matching packing."""
    n = 256
    g = torch.Generator().manual_seed(9)
    V = torch.linalg.qr(torch.randn(n, n, generator=g, dtype=torch.float64))[0].float()
    S = torch.rand(n, generator=g) + 0.1
    Vs = V * S.view(1, -1)
    X = torch.randn(64, n, generator=g)
    pk = ops.rankspace_pack(V.to(gpu), Vs.to(gpu))
    assert pk is not None and pk.numel() == 3 * n * n
    Xg = X.to(gpu)
    for part, ref in ((0, X.double() @ V.double()), (1, X.double() @ V.double().T), (2, X.double() @ Vs.double())):
        C = ops.gemm_x6(Xg, pk[part * n * n:(part + 1) * n * n], n).cpu().double()
        assert float((C - ref).abs().max()) <= 2e-6 * float(ref.abs().max())


def test_gemm_x6_splitk_partials_sum_to_the_product(gpu):
    """mpq_gemm_x6_pack_a + mpq_gemm_x6_splitk (the VAMP solvers' launches): the partials added in
    split order are bit-identical to mpq_gemm_x6, and each partial is its K slice's product."""
    M, N, K = 128, 384, 2048
    g = torch.Generator().manual_seed(21)
    A = torch.randn(M, K, generator=g)
    B = torch.randn(K, N, generator=g)
    Bp = ops.gemm_x6_pack_b(B.to(gpu))
    Ap = ops.gemm_x6_pack_a(A.to(gpu))
    P, splits = ops.gemm_x6_splitk(Ap, Bp, M, N, K)
    assert splits > 1
    acc = P[0].clone()
    for s in range(1, splits):
        acc += P[s]
    assert torch.equal(acc.cpu(), ops.gemm_x6(A.to(gpu), Bp, N).cpu())
    ks = K // splits
    for s in (0, splits - 1):
        ref = A[:, s * ks:(s + 1) * ks].double() @ B[s * ks:(s + 1) * ks].double()
        assert float((P[s].cpu().double() - ref).abs().max()) <= 2e-6 * float(ref.abs().max())


def _plane_bound(A, B):
    """Entry-wise bound: each operand is held to 2^-24 relative whatever stands beside it, the dropped plane products
    are below 2^-22.4, and the roundings of the sums stay below what is left of 2^-20 for the sizes tested."""
    return 2.0 ** -20 * (A.abs() @ B.abs())


@pytest.mark.parametrize("M,N,K,splits", [
    (3, 128, 32, 1), (128, 128, 1024, 1), (129, 256, 1056, 1), (128, 128, 2112, 3), (100, 128, 96, 1),
    (128, 128, 17 * 1024, 1), (65, 128, 17 * 1024 + 32, 1),
    (128, 256, 3584, 1), (64, 128, 4096, 8)])
def test_plane_product_slices(gpu, M, N, K, splits):
    """Slab counts that are and are not multiples of the ring's four stages; splits of the caller's choice."""
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g).double().to(gpu)
    B = torch.randn(K, N, generator=g).double().to(gpu)
    Ap, Bp = ops.gemm_x6_pack_a(A.float()), ops.gemm_x6_pack_b(B.float())
    P, _ = ops.gemm_x6_splitk(Ap, Bp, M, N, K, splits=splits)
    assert bool(((P.double().sum(0) - A @ B).abs() <= _plane_bound(A, B)).all())


def test_plane_product_keeps_small_entries(gpu):
    """Rows of A and columns of B over 60 orders of magnitude: zero slabs first, columns that grow and
    shrink along K, values far below their row's or column's largest, zero rows and columns."""
    M, N, K = 128, 256, 4096
    g = torch.Generator().manual_seed(77)
    A = torch.randn(M, K, generator=g).double()
    B = torch.randn(K, N, generator=g).double()
    A[:32] *= 1e-30
    A[32:64, 1024:2048] *= 1e12
    A[64:96, 2048:] *= 1e-20
    A[96] = 0.0
    k = torch.arange(K, dtype=torch.float64).view(-1, 1)
    B[:, :32] *= torch.exp2(k / 64)          # grows by 2^64
    B[:, 32:64] *= torch.exp2(-k / 64)       # shrinks by 2^64
    B[:2000, 64:96] = 0.0                    # zero until a late slab
    B[:, 96:128] *= 1e20  # times 1e12 of A, still an fp32 number
    B[:, 128:160] *= 1e-7
    B[5, 128:160] = 1.0                      # one value 2^23 above the others, against a zero of A
    A[:16, 5] = 0.0
    B[:, 200] = 0.0
    A, B = A.float().double().to(gpu), B.float().double().to(gpu)
    C = ops.gemm_x6(A.float(), ops.gemm_x6_pack_b(B.float()), N).double()
    err, bound = (C - A @ B).abs(), _plane_bound(A, B)
    assert bool((err <= bound).all()), float((err / bound).nan_to_num(0).max())
    assert float(C[96].abs().max()) == 0.0 and float(C[:, 200].abs().max()) == 0.0


def test_plane_product_non_finite_stays_in_its_row_and_column(gpu):
    M, N, K = 40, 128, 2048
    g = torch.Generator().manual_seed(5)
    A, B = torch.randn(M, K, generator=g), torch.randn(K, N, generator=g)
    C0 = ops.gemm_x6(A.to(gpu), ops.gemm_x6_pack_b(B.to(gpu)), N).cpu()
    A[3, 1500], A[7, 2], B[900, 11] = float("inf"), float("nan"), float("-inf")
    C = ops.gemm_x6(A.to(gpu), ops.gemm_x6_pack_b(B.to(gpu)), N).cpu()
    bad = torch.zeros(M, N, dtype=torch.bool)
    bad[3], bad[7], bad[:, 11] = True, True, True
    assert not bool(torch.isfinite(C[bad]).any()) and torch.equal(C[~bad], C0[~bad])


@pytest.mark.parametrize("a,b", [(1e35, 1e-10), (1e-10, 1e35), (1e32, 1e-30), (-1e37, 1e-2)])
def test_plane_product_reaches_the_range_limits(gpu, a, b):
    """Operands near either end of fp32's range whose product is an ordinary number: no scaling may overflow or
    vanish on the way."""
    M, N, K = 40, 128, 1024
    A, B = torch.full((M, K), a, device=gpu), torch.full((K, N), b, device=gpu)
    ref = A.double() @ B.double()
    Bp = ops.gemm_x6_pack_b(B)
    P, _ = ops.gemm_x6_splitk(ops.gemm_x6_pack_a(A), Bp, M, N, K)
    for C in (ops.gemm_x6(A, Bp, N).double(), P.double().sum(0)):
        assert float(((C - ref) / ref).abs().max()) < 2.0 ** -18


@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (1, 128, 128), (100, 384, 384), (128, 1024, 1024), (256, 1152, 1152),
                                   (128, 2048, 2048), (256, 2048, 2048)])
def test_gemm_x6_small_products(gpu, M, N, K):
    """Entry-wise error relative to sum_k |a_k b_k| of products with few work-groups: one rounding per MFMA of a
    slice (6 per 16 k), one per partial summed and four for the split and the dropped plane products."""
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g) * torch.exp(2.0 * torch.randn(1, K, generator=g))
    B = torch.randn(K, N, generator=g)
    splits = ops._lib.load().mpq_gemm_x6_split_count(M, N, K)
    C = ops.gemm_x6(A.to(gpu), ops.gemm_x6_pack_b(B.to(gpu)), N).cpu().double()
    err = (C - A.double() @ B.double()).abs() / (A.double().abs() @ B.double().abs())
    assert float(err.max()) <= (6 * K / (16 * splits) + splits + 4) * 2.0**-24
