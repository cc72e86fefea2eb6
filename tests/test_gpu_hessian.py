"""GPU: Hessian accumulation (mpq_hessian_accumulate, bf16 MFMA SYRK) against fp64 products, and
the GPTQ / QUIP# accumulation conventions (mpq_amd/hessian.py) against fp64 restatements."""
import math

import pytest
import torch

from mpq_amd import hessian

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


@pytest.mark.parametrize("T,n", [(1000, 256), (37, 384), (4096, 1024), (0, 128)])
def test_syrk_matches_fp64(gpu, T, n):
    g = torch.Generator().manual_seed(T + n)
    X = torch.randn(T, n, generator=g) * torch.exp(torch.randn(n, generator=g))
    H0 = torch.randn(n, n, generator=g)
    H0 = H0 + H0.T
    H = H0.clone().to(gpu)
    hessian.accumulate(H, X.to(gpu), alpha=0.75, beta=0.5)
    H = H.cpu()
    ref = 0.5 * H0.double() + 0.75 * X.double().T @ X.double()
    assert _rel(H, ref) < 2e-6
    assert torch.equal(H, H.T)


def test_syrk_bf16_input_and_colsum(gpu):
    g = torch.Generator().manual_seed(3)
    X = torch.randn(3, 100, 512, generator=g).to(torch.bfloat16)
    H = torch.zeros(512, 512, device=gpu)
    cs = torch.zeros(512, device=gpu)
    hessian.accumulate(H, X.to(gpu), colsum=cs)
    Xd = X.reshape(-1, 512).double()
    assert _rel(H.cpu(), Xd.T @ Xd) < 2e-6
    assert torch.allclose(cs.cpu().double(), Xd.sum(0), rtol=1e-5, atol=1e-4)


def test_gptq_convention(gpu):
    g = torch.Generator().manual_seed(5)
    n = 256
    acc = hessian.GPTQHessian(n, gpu)
    Href = torch.zeros(n, n, dtype=torch.float64)
    ns = 0
    for b in (3, 1, 4):
        inp = torch.randn(b, 64, n, generator=g)
        acc.add_batch(inp.to(gpu))
        # classic GPTQ add_batch in fp64
        Href *= ns / (ns + b)
        ns += b
        x = math.sqrt(2 / ns) * inp.reshape(-1, n).double().T
        Href += x @ x.T
    assert acc.nsamples == ns
    assert _rel(acc.H.cpu(), Href) < 2e-6


def test_quip_convention(gpu):
    g = torch.Generator().manual_seed(6)
    n = 128
    acc = hessian.QuipHessian(n, gpu)
    xs = [torch.randn(200, n, generator=g) + 0.3 for _ in range(3)]
    for x in xs:
        acc.add_batch(x.to(gpu))
    H, mu, ct = acc.finalize()
    X = torch.cat(xs).double()
    mu_ref = X.mean(0)
    H_ref = X.T @ X / X.shape[0] - torch.outer(mu_ref, mu_ref)
    assert ct == X.shape[0]
    assert torch.allclose(mu.cpu().double(), mu_ref, atol=1e-5)
    assert _rel(H.cpu(), H_ref) < 1e-5


def test_rejects_bad_width(gpu):
    with pytest.raises(ValueError):
        hessian.accumulate(torch.zeros(100, 100, device=gpu), torch.zeros(10, 100, device=gpu))


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("T,n", [(1, 128), (31, 128), (33, 384), (127, 640), (129, 2432), (100, 2560),
                                 (256, 2560), (257, 2560), (271, 2560), (300, 2432)])
def test_syrk_slab_and_tile_edges(gpu, T, n, bf16):
    """Partial token slabs, the 64 x 64 tiles (up to 256 tokens, or below 200 tiles of 128 x 128: n <= 2432) and
    the 128 x 128 tiles, and the column sums.  Each entry sums T products exact to 2^-22 relative in fp32: its error is
    at most (2^-22 + (T + 2) 2^-24) sum |x_i x_j|."""
    g = torch.Generator().manual_seed(7 * T + n)
    X = torch.randn(T, n, generator=g) * torch.exp(torch.randn(n, generator=g))
    X = X.to(torch.bfloat16) if bf16 else X
    H = torch.zeros(n, n, device=gpu)
    cs = torch.ones(n, device=gpu)
    hessian.accumulate(H, X.to(gpu), colsum=cs)
    Xd = X.double().to(gpu)
    bound = (2.0 ** -22 + (T + 2) * 2.0 ** -24) * (Xd.abs().T @ Xd.abs())
    assert bool(((H.double() - Xd.T @ Xd).abs() <= bound).all())
    assert torch.equal(H, H.T)
    assert bool(((cs.double() - 1 - Xd.sum(0)).abs() <= (T + 2) * 2.0 ** -24 * (1 + Xd.abs().sum(0))).all())


@pytest.mark.parametrize("T,n", [(40, 256), (40, 2560), (259, 2560)])
def test_syrk_non_finite_activations(gpu, T, n):
    """Infinities, NaN and values that round to an infinity in bf16 act as in fp32 products."""
    g = torch.Generator().manual_seed(n)
    X = torch.randn(T, n, generator=g)
    X[5, 7], X[9, 100], X[3, 50] = float("inf"), float("nan"), 3.4e38
    X[3, 7] = 0.5  # 3.4e38 X[3, 7] must not overflow before the infinity of column 7 is added (fp32 would give NaN)
    H = torch.zeros(n, n, device=gpu)
    hessian.accumulate(H, X.to(gpu))
    H = H.cpu()
    ref = X.double().T @ X.double()
    ref = torch.where(ref.abs() > 3.4028235e38, ref.sign() * float("inf"), ref)
    assert torch.equal(torch.isnan(H), torch.isnan(ref))
    assert torch.equal(torch.isinf(H), torch.isinf(ref)) and torch.equal(H[torch.isinf(H)], ref[torch.isinf(ref)].float())
    ok = torch.isfinite(H)
    assert float((H[ok].double() - ref[ok]).abs().max() / 3.4e38) < 1e-6


def test_syrk_non_finite_activations_cost_one_more_product(gpu):
    """Infinities everywhere, or in one column, are summed again as one fp32 matrix product (measured: 5 times the
    finite call; a serial dot product per entry took 120 times), not entry by entry."""
    X = torch.randn(2048, 1024, generator=torch.Generator().manual_seed(3)).to(gpu)
    H = torch.zeros(1024, 1024, device=gpu)

    def best_ms(x):
        times = []
        for _ in range(6):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            hessian.accumulate(H, x)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times[1:])

    finite = best_ms(X)
    one = X.clone()
    one[7, 5] = float("inf")
    assert best_ms(one) < 20 * finite
    assert best_ms(torch.full_like(X, float("inf"))) < 20 * finite


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("T,n", [(3, 2560), (300, 256), (300, 2560)])
def test_syrk_adds_to_the_upper_triangle(gpu, T, n, bf16):
    """H = beta H + alpha X^T X of both tile sizes: the entries on and above the diagonal count, the others are
    written as their mirror image.  With H = 0, beta = 0 gives X^T X exactly as beta = 1 does."""
    g = torch.Generator().manual_seed(T + n)
    X = torch.randn(T, n, generator=g).to(torch.bfloat16 if bf16 else torch.float32).to(gpu)
    H0 = torch.randn(n, n, generator=g).to(gpu)
    H = hessian.accumulate(H0.clone(), X, alpha=0.75, beta=0.5)
    upper = torch.triu(H0.double())
    sym = upper + torch.triu(H0.double(), 1).T
    Xd = X.double()
    bound = 2.0 ** -23 * sym.abs() + (2.0 ** -22 + (T + 4) * 2.0 ** -24) * (Xd.abs().T @ Xd.abs())
    assert bool(((H.double() - 0.5 * sym - 0.75 * Xd.T @ Xd).abs() <= bound).all())
    assert torch.equal(H, H.T)
    P1 = hessian.accumulate(torch.zeros_like(H0), X)
    P0 = hessian.accumulate(torch.full_like(H0, float("nan")), X, beta=0.0)
    assert torch.equal(P0, P1)
