"""GPU: split-K partials lie 64-float aligned apart, also where rows x n is not a multiple of 64 floats;
the solvers' and polishes' targets W Vs are summed with that distance (errors against fp64)."""
import pytest
import torch

from mpq_amd import ops
from mpq_amd.codebook import E8P12_codebook
from mpq_amd.solver import E8P12VampConfig, UniformVampConfig

pytestmark = pytest.mark.gpu


def _problem(gpu, rows, n, seed):
    g = torch.Generator().manual_seed(seed)
    V = torch.linalg.qr(torch.randn(n, n, generator=g, dtype=torch.float64))[0].float()
    S = torch.exp(0.5 * torch.randn(n, generator=g))
    W = torch.randn(rows, n, generator=g)
    return W.to(gpu), V.contiguous().to(gpu), S.to(gpu), (V * S).contiguous().to(gpu)


def _start_error(W, x, Vs):
    return ((W.double() - x.double()) @ Vs.double()).square().sum(dim=1)


@pytest.mark.parametrize("rows,n", [(100, 1000), (7, 1025)])
def test_uniform_solver_and_polish(gpu, rows, n):
    W, V, S, Vs = _problem(gpu, rows, n, rows)
    assert (rows * n) % 64 and ops._lib.load().mpq_gemm_f32_split_count(rows, n, n) > 1
    scale, zero = ops.gptq_find_params(W, 128, 15)
    q, x = ops.uniform_rtn(W, scale, zero, 128, 15)
    ref = _start_error(W, x, Vs)
    _, _, _, rtn_err, _ = ops.uniform_vamp_solve(W, x, scale, zero, 128, 15, V, S, Vs, UniformVampConfig(iters=2))
    assert torch.allclose(rtn_err.double(), ref, rtol=1e-4)
    _, before, after, _, _ = ops.uniform_cd_polish(W, q, scale, zero, 128, 15, Vs, (Vs @ Vs.T).contiguous(),
                                                   block_rows=rows, sweeps=1)
    assert torch.allclose(before.double(), ref, rtol=1e-4) and bool((after <= before).all())


@pytest.mark.parametrize("rows,n", [(101, 1000), (7, 1032)])
def test_e8p12_solver_and_polish(gpu, rows, n):
    W, V, S, Vs = _problem(gpu, rows, n, n)
    assert (rows * n) % 64 and ops._lib.load().mpq_gemm_f32_split_count(rows, n, n) > 1
    x, idx = E8P12_codebook(gpu).quantize(W.reshape(-1, 8), return_idx=True)
    x, idx = x.reshape(rows, n).contiguous(), idx.reshape(rows, n // 8).long()
    ref = _start_error(W, x, Vs)
    _, _, before, after, _ = ops.e8p12_cd_polish(x, idx, Vs, ops.e8p12_cd_prepare(Vs), sweeps=1, block_rows=rows, W=W)
    assert torch.allclose(before.double(), ref, rtol=1e-4) and bool((after <= before * (1 + 1e-5)).all())
    # the solver's error is that of its own decision
    idx_v, hat, err, _, _, _ = ops.e8p12_vamp_solve(W, x, V, S, Vs, E8P12VampConfig(iters=2))
    assert torch.allclose(err.double(), _start_error(W, hat, Vs), rtol=1e-4)
