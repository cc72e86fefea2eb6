"""GPU: AWQ scale search (mpq_awq_w_mean, mpq_awq_search) against the CPU oracle (oracle/awq.py)."""
import pytest
import torch

from mpq_amd import awq, ops
from oracle import awq as oa
from tests.uniform_cases import make_layer

pytestmark = pytest.mark.gpu


def test_w_mean(gpu):
    g = torch.Generator().manual_seed(4)
    Ws = [torch.randn(64, 512, generator=g) * 0.02, torch.randn(32, 512, generator=g)]
    got = awq.compute_w_mean([w.to(gpu) for w in Ws], 128).cpu()
    ref = oa.compute_w_mean(Ws, 128)
    assert torch.allclose(got, ref, rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("rows,n,group", [(37, 960, 1), (37, 960, 2), (5, 960, 3), (37, 960, 5), (130, 960, 16),
                                          (7, 960, 60), (3, 960, 64), (37, 960, 96), (1, 960, 960)])
def test_w_mean_group_sizes(gpu, rows, n, group):
    """One to 64 lanes per group; groups that fill no power of two, rows whose groups fill no wave."""
    W = torch.randn(rows, n, generator=torch.Generator().manual_seed(group)) * 0.02
    assert torch.allclose(awq.compute_w_mean([W.to(gpu)], group).cpu(), oa.compute_w_mean([W], group), rtol=2e-6, atol=1e-7)


@pytest.mark.parametrize("bits,sym", [(4, False), (3, False), (4, True)])
def test_search_matches_oracle(gpu, bits, sym):
    W, H = make_layer(96, 256, tokens=1024, seed_key=f"awq:{bits}:{sym}")
    g = torch.Generator().manual_seed(9)
    X = torch.randn(1024, 256, generator=g) * torch.exp(torch.randn(256, generator=g))
    x_mean = X.abs().mean(0)
    w_mean = oa.compute_w_mean([W], 128)
    s_ref, e_ref, r_ref, l_ref = oa.search_linear(W, H, x_mean, w_mean, bits, 128, sym)
    s, e, r, losses = awq.search_best_scale_linear(W.to(gpu), H.to(gpu), x_mean.to(gpu), bits=bits, group_size=128,
                                                   sym=sym, w_mean=w_mean.to(gpu))
    losses = losses.cpu()
    assert torch.allclose(losses, torch.tensor(l_ref), rtol=2e-4)
    assert abs(r - r_ref) < 1e-6
    assert abs(e - e_ref) <= 2e-4 * e_ref
    assert torch.allclose(s.cpu(), s_ref, rtol=1e-5)


@pytest.mark.parametrize("rows,n", [(33, 1024), (130, 1152), (1025, 1024), (1023, 1024), (65, 4096)])
def test_search_on_packed_products_matches_fp64(gpu, rows, n):
    """From n = 1024 and rows n^2 = 2^30 the products D H run as x6 products on H packed once, below on the fp32
    kernel; rows that are no whole tiles, both sides of the rule.  The
    losses against fp64 on the same scales and deltas' formula: a weight that rounds the other way moves a
    loss by less than 1e-4 at these sizes (the fp32 path's own bar is 2e-4)."""
    g = torch.Generator().manual_seed(rows)
    W = 0.02 * torch.randn(rows, n, generator=g)
    X = torch.randn(2 * n, n, generator=g) * torch.exp(torch.randn(n, generator=g))
    H = X.T @ X / (2 * n)
    x_mean = X.abs().mean(0)
    w_mean = oa.compute_w_mean([W], 128)
    s_ref, e_ref, r_ref, l_ref = oa.search_linear(W, H, x_mean, w_mean, 4, 128, False)
    s, e, r, losses = awq.search_best_scale_linear(W.to(gpu), H.to(gpu), x_mean.to(gpu), bits=4, group_size=128)
    assert torch.allclose(losses.cpu(), torch.tensor(l_ref), rtol=2e-4)
    assert abs(r - r_ref) < 1e-6 and abs(e - e_ref) <= 2e-4 * e_ref and torch.allclose(s.cpu(), s_ref, rtol=1e-5)


@pytest.mark.parametrize("n,group", [(1024, 128), (384, 64)])
def test_search_takes_a_workspace_of_any_float_alignment(gpu, n, group):
    """The packed operands want 16-byte pieces; a workspace that begins 4 bytes off gives the same losses."""
    rows = 1100
    g = torch.Generator().manual_seed(n)
    W = (0.02 * torch.randn(rows, n, generator=g)).to(gpu)
    X = torch.randn(2 * n, n, generator=g).to(gpu)
    H, x_mean = (X.T @ X / (2 * n)).contiguous(), X.abs().mean(0)
    w_mean = awq.compute_w_mean([W], group)
    lib = ops._lib.load()
    need = int(lib.mpq_awq_workspace_size(rows, n))

    def losses(offset):
        ws = torch.empty(need + 4096, dtype=torch.uint8, device=gpu).fill_(0xFF)
        scales, out = torch.empty(n, device=gpu), torch.empty(20, device=gpu)
        ops._lib.call("mpq_awq_search", ops._lib.ptr(W), rows, n, ops._lib.ptr(H), ops._lib.ptr(x_mean),
                      ops._lib.ptr(w_mean), group, 4, 0, ops._lib.ptr(scales), ops._lib.ptr(out), 0, 0,
                      ops._lib.ptr(ws[256 + offset:]), need, ops._lib.stream_handle(gpu))
        assert bool((ws[:256 + offset] == 0xFF).all()) and bool((ws[256 + offset + need:] == 0xFF).all())
        return out

    assert torch.equal(losses(0), losses(4)) and torch.equal(losses(0), losses(252))
