"""GPU: the iteration at which each row block of a layer stops, against recorded ones.

A row block of the uniform VAMP ends at its first iterate that does not improve on the best one, and its
observation precision goes on to the next block (mpq/solver.py:678-699).  On layers like these the comparison
is close: rounding the decomposition or a product another way, however accurately, ends a block at another
iterate, and then some percent of its codes change, far more than the few per million that near-ties move
while the stops hold.  ``golden/layer_stops.json`` holds the stops and best iterates with every operand of the
products held to all 24 bits of its fp32 value and with fp32 slices of at least 256 (the uniform solver at
4096 columns and above runs on three exact bf16 planes, below on fp32 MFMA).

The inputs are exact on any machine: integer tokens, weights and channel scales, sums in float64.
"""
import json
import math
import os

import pytest
import torch

from mpq_amd.adapters.gptqmodel import GPTQAdapterConfig, run_mpq_quantization
from mpq_amd.solver import UniformVampConfig
from tests.uniform_cases import QCfg

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "layer_stops.json")
ROWS, BITS, GROUP, ITERS = 1024, 3, 128, 16


def exact_layer(n, seed, device):
    """(W, H): dyadic weights, and tokens with scaled channels, some of them outliers; damping a power of two."""
    g = torch.Generator().manual_seed(seed)
    T = 2 * n
    X = torch.randint(-3, 4, (T, n), generator=g)
    c = (8 + torch.randint(0, 8, (n,), generator=g)) * 2 ** torch.randint(0, 6, (n,), generator=g)
    c[torch.randperm(n, generator=g)[: n // 100]] *= 16
    W = torch.randint(-31, 32, (4, ROWS, n), generator=g).sum(0)
    X, c = X.to(device).double(), c.to(device).double()
    H = (X.T @ X) * c * c[:, None] / (T * 16)
    H += 2.0 ** round(math.log2(0.01 * float(torch.diagonal(H).mean()))) * torch.eye(n, device=device)
    return (W.float() / 2048).to(device), H.float()


def stops(n, seed, device):
    W, H = exact_layer(n, seed, device)
    st = run_mpq_quantization(W=W, H=H, quantizer=None, qcfg=QCfg(BITS, GROUP, "internal_hadamard"), module_name="m",
                              vamp_cfg=UniformVampConfig(iters=ITERS, polish_sweeps=0),
                              adapter_cfg=GPTQAdapterConfig(eigen_cache=False))[-1]
    return {"entered": st["vamp_iters_entered"], "best": st["vamp_iters"]}


# two-stage decomposition and fp32 products; at 4096 the packed products
@pytest.mark.parametrize("n,seed", [(2048, 73), (2048, 79), (1536, 10), (2048, 43), (2048, 75), (4096, 4), (4096, 17)])
def test_row_blocks_stop_where_they_did(gpu, n, seed):
    with open(GOLDEN) as f:
        want = json.load(f)[f"{n} {seed}"]
    assert stops(n, seed, gpu) == want
