"""What is timed: the work of a per-layer quantization run, through the framework's public entry points.

A run visits every linear of a model: it accumulates the Hessian of the linear's inputs, searches AWQ
scales, decomposes the Hessian, and solves for the codes (uniform grid or the E8P12 lattice codebook).
Sizes are those of the repository's own workloads: the Llama-3-8B- and Llama-3.2-1B-shaped linears of
bench.py and the small layers of the tests.  ``draw`` spreads over the same ranges, ragged sizes
among them.

Whole layers run without the polish and the polish runs from a given start, because the greedy polish
cascades: one code decided differently on a near-tie reorders the later decisions of its row block.
"""
from __future__ import annotations

import math

import torch

from mpq_amd import awq, hessian, ops
from mpq_amd.adapters.gptqmodel import GPTQAdapterConfig, run_mpq_quantization, vamp_hessian_eigen
from mpq_amd.adapters.quip_sharp import mpq_refine_codebook
from mpq_amd.codebook import E8P12_codebook
from mpq_amd.solver import UniformVampConfig, solve_uniform_rankspace_vamp

DEV = "cuda:0"


def listed():
    return [
        # nearest-codeword encoding of one small tensor: a single short launch
        {"name": "e8p12_quantize_small", "kind": "quantize", "vectors": 1000},
        # the same over a whole linear's 8-vectors (the E8P12 codebook benchmark's size)
        {"name": "e8p12_quantize_large", "kind": "quantize", "vectors": 1 << 24},
        # one calibration batch of bf16 activations into GPTQ's Hessian (q/k/v/o, gate/up inputs)
        {"name": "hessian_gptq_bf16", "kind": "hessian", "conv": "gptq", "n": 4096, "tokens": 8 * 2048, "bf16": True},
        # one fp32 batch of ragged length into QUIP#'s sums (Hessian and mean)
        {"name": "hessian_quip_f32", "kind": "hessian", "conv": "quip", "n": 2048, "tokens": 3001, "bf16": False},
        # AWQ scale search of one attention linear
        {"name": "awq_search", "kind": "awq", "rows": 4096, "n": 4096, "bits": 3, "group": 128},
        # decomposition of a linear's Hessian as the GPTQ adapter takes it, and the Gram matrix of its factor
        {"name": "eigh_f32", "kind": "eigh32", "n": 4096},
        # decomposition as the QUIP# adapter takes it (fp64)
        {"name": "eigh_f64", "kind": "eigh64", "n": 2048},
        # the smallest solve: one ragged 4-bit row block of a small layer
        {"name": "vamp_block_small", "kind": "block", "rows": 104, "n": 1000, "bits": 4, "group": 128},
        # the greedy polish of an attention linear, 3 sweeps
        {"name": "uniform_polish", "kind": "cd", "rows": 4096, "n": 4096, "bits": 3, "group": 128},
        # the E8P12 polish of the fused q/k/v linear, 3 sweeps
        {"name": "e8p12_polish", "kind": "e8cd", "rows": 3072, "n": 2048},
        # a whole down_proj: eigh, rotation, group parameters, 32 row blocks of VAMP
        {"name": "layer_down_proj", "kind": "layer", "rows": 4096, "n": 14336, "bits": 3, "group": 128,
         "rotation": "internal_hadamard", "desc_act": False},
        # a whole E8P12 down linear: fp64 eigh, 16 row blocks of VAMP
        {"name": "layer_e8p12_down", "kind": "refine", "rows": 2048, "n": 8192},
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["quantize", "hessian", "awq", "eigh32", "eigh64", "block", "cd", "e8cd", "layer", "refine"])
    if kind == "quantize":
        return {"kind": kind, "vectors": _log(rng, 256, 1 << 24)}
    if kind == "hessian":
        return {"kind": kind, "conv": rng.choice(["gptq", "quip"]), "n": _log(rng, 256, 4096, 128),
                "tokens": _log(rng, 100, 8 * 2048), "bf16": rng.random() < 0.5}
    if kind == "awq":
        return {"kind": kind, "rows": _log(rng, 64, 4096), "n": _log(rng, 256, 4096, 128),
                "bits": rng.choice([3, 4]), "group": 128}
    if kind == "eigh32":
        return {"kind": kind, "n": _log(rng, 100, 4096)}
    if kind == "eigh64":
        return {"kind": kind, "n": _log(rng, 100, 2048)}
    if kind == "block":
        return {"kind": kind, "rows": 8 * rng.randint(1, 16), "n": _log(rng, 104, 4096, rng.choice([8, 128])),
                "bits": rng.choice([4, 8]), "group": rng.choice([64, 128])}
    if kind == "cd":
        return {"kind": kind, "rows": _log(rng, 64, 4096, 8), "n": _log(rng, 256, 4096, rng.choice([8, 128])),
                "bits": rng.choice([2, 3, 4]), "group": rng.choice([64, 128])}
    if kind == "e8cd":
        return {"kind": kind, "rows": _log(rng, 64, 3072, 8), "n": _log(rng, 256, 2048, rng.choice([8, 128]))}
    if kind == "layer":
        aligned, rotation = rng.random() < 0.7, rng.choice(["none", "internal_hadamard"])
        return {"kind": kind, "rows": _log(rng, 64, 4096 if aligned else 1024),
                "n": _log(rng, 512, 14336, 1024) if aligned else _log(rng, 300, 6000),
                "bits": 4 if rotation == "none" else rng.choice([3, 4]), "group": rng.choice([64, 128]),
                "rotation": rotation, "desc_act": rng.random() < 0.25}
    return {"kind": kind, "rows": _log(rng, 64, 2048, 8), "n": _log(rng, 256, 8192, rng.choice([8, 128]))}


# ---- inputs ----------------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _weight(g, rows, n):
    return (0.02 * torch.randn(rows, n, device=DEV, generator=g)).to(torch.bfloat16).float()


def _channel_scales(g, n):
    """Lognormal channel scales with 1 % outlier channels, as LLM activations have."""
    c = torch.exp(torch.randn(n, device=DEV, generator=g))
    c[torch.randperm(n, device=DEV, generator=g)[: max(1, n // 100)]] *= 20.0
    return c


def _hessian(g, n, student=False):
    """Damped X^T X / T of synthetic tokens."""
    T = max(2048, min(2 * n, 16384))
    X = torch.randn(T, n, device=DEV, generator=g)
    if student:  # heavy-tailed tokens, 4 degrees of freedom
        X /= torch.sqrt(torch.randn(T, 4, device=DEV, generator=g).square().mean(dim=1, keepdim=True))
    else:
        X *= _channel_scales(g, n)
    H = (X.T @ X) / T
    H += 0.01 * torch.diagonal(H).mean() * torch.eye(n, device=DEV)
    return 0.5 * (H + H.T)


def _eigenbasis(g, n):
    """(V, S, Vs): an incoherent basis and the decaying spectrum of a rotated Hessian, in hand after its
    decomposition."""
    V = torch.linalg.qr(torch.randn(n, n, device=DEV, generator=g))[0].contiguous()
    lam = 4.0 * torch.exp(-6.0 * torch.arange(n, device=DEV) / n) + 0.02
    lam[: max(1, n // 100)] *= 50.0
    S = torch.sqrt(lam)
    return V, S, (V * S).contiguous()


class _QCfg:
    """The fields of GPTQModel's quantization config that the adapter reads."""

    def __init__(self, case):
        self.bits, self.group_size, self.desc_act = case["bits"], case["group"], case["desc_act"]
        self.mpq = type("Mpq", (), {"rotation_mode": case["rotation"], "solver": "vamp"})()


class _QuipArgs:
    """The QUIP# arguments of a VAMP pass without polish."""

    mpq_iters, mpq_damping, mpq_prior_tau = 16, 0.5, 0.2
    mpq_polish_sweeps, mpq_block_rows = 0, 128


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "quantize":
        return {"case": case, "cb": E8P12_codebook(DEV), "x": torch.randn(case["vectors"], 8, device=DEV, generator=g)}
    if kind == "hessian":
        X = torch.randn(case["tokens"], case["n"], device=DEV, generator=g) * _channel_scales(g, case["n"])
        return {"case": case, "x": X.to(torch.bfloat16) if case["bf16"] else X}
    if kind == "awq":
        H = _hessian(g, case["n"])
        return {"case": case, "W": _weight(g, case["rows"], case["n"]), "H": H,
                "x_mean": 0.8 * torch.sqrt(torch.diagonal(H)).contiguous()}
    if kind == "eigh32":
        return {"case": case, "H": _hessian(g, case["n"])}
    if kind == "eigh64":
        return {"case": case, "H": _hessian(g, case["n"], student=True).double()}
    if kind == "layer":
        return {"case": case, "W": _weight(g, case["rows"], case["n"]), "H": 2.0 * _hessian(g, case["n"]),
                "vamp": UniformVampConfig(iters=16, polish_sweeps=0), "adapter": GPTQAdapterConfig(eigen_cache=False)}
    if kind == "refine":
        Wr = torch.randn(case["rows"], case["n"], device=DEV, generator=g)
        zero = torch.zeros(case["rows"], case["n"] // 8, dtype=torch.int64, device=DEV)
        return {"case": case, "Wr": Wr, "H": _hessian(g, case["n"], student=True), "idx0": zero,
                "cb": E8P12_codebook(DEV)}
    V, S, Vs = _eigenbasis(g, case["n"])
    if kind == "e8cd":
        W = torch.randn(case["rows"], case["n"], device=DEV, generator=g)
        x, idx = E8P12_codebook(DEV).quantize(W.reshape(-1, 8), return_idx=True)
        return {"case": case, "W": W, "x": x.reshape(W.shape).contiguous(), "idx": idx.reshape(case["rows"], -1).long(),
                "Vs": Vs, "ctx": ops.e8p12_cd_prepare(Vs)}
    W = _weight(g, case["rows"], case["n"])
    maxq = 2 ** case["bits"] - 1
    scale, zero = ops.gptq_find_params(W, case["group"], maxq)
    q, x = ops.uniform_rtn(W, scale, zero, case["group"], maxq)
    s = {"case": case, "W": W, "scale": scale, "zero": zero, "maxq": maxq, "q": q, "x": x, "V": V, "S": S, "Vs": Vs}
    if kind == "cd":
        s["H"] = (Vs @ Vs.T).contiguous()
    else:
        s["Vh"] = V.T.contiguous()
        s["vamp"] = UniformVampConfig(iters=16, polish_sweeps=0)
    return s


# ---- one pass --------------------------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "quantize":
        vals, idx = s["cb"].quantize(s["x"], return_idx=True)
        return {"vals": vals, "idx": idx}
    if kind == "hessian":
        if case["conv"] == "gptq":
            acc = hessian.GPTQHessian(case["n"], DEV)
            acc.add_batch(s["x"])
            return {"H": acc.H}
        acc = hessian.QuipHessian(case["n"], DEV)
        acc.add_batch(s["x"])
        H, mu, ct = acc.finalize()
        return {"H": H, "mu": mu, "ct": ct}
    if kind == "awq":
        scales, err, ratio, losses = awq.search_best_scale_linear(s["W"], s["H"], s["x_mean"], bits=case["bits"],
                                                                  group_size=case["group"])
        return {"scales": scales, "err": err, "ratio": ratio, "losses": losses}
    if kind == "eigh32":
        # the eigenvectors themselves are fixed only up to signs and mixing within close eigenvalues: what a
        # solver builds from them is returned instead
        lam, _, V, Vs, floor = vamp_hessian_eigen(s["H"], use_cache=False)
        return {"lam": lam, "gram": ops.gemm(Vs, Vs, trans_b=True), "unit": ops.gemm(V, V, trans_b=True),
                "floor": floor}
    if kind == "eigh64":
        lam, V = ops.syevd(s["H"])
        return {"lam": lam, "gram": ops.gemm_f64(V * lam, V, trans_b=True), "unit": ops.gemm_f64(V, V, trans_b=True)}
    if kind == "block":
        q, x, err, rtn_err, _ = solve_uniform_rankspace_vamp(
            W=s["W"], x_rtn=s["x"], scale_full=s["scale"], zero_full=s["zero"], maxq=s["maxq"], V=s["V"], Vh=s["Vh"],
            S=s["S"], Vs=s["Vs"], cfg=s["vamp"], group_size=case["group"])
        return {"q": q, "x": x, "err": err, "rtn_err": rtn_err}
    if kind == "cd":
        q, before, after, improved, accepted = ops.uniform_cd_polish(
            s["W"], s["q"], s["scale"], s["zero"], case["group"], s["maxq"], s["Vs"], s["H"], block_rows=128, sweeps=3)
        return {"q": q, "before": before, "after": after, "improved": improved, "accepted": accepted}
    if kind == "e8cd":
        _, idx, before, after, accepted = ops.e8p12_cd_polish(s["x"], s["idx"], s["Vs"], s["ctx"], sweeps=3,
                                                              block_rows=128, W=s["W"])
        return {"idx": idx, "before": before, "after": after, "accepted": accepted}
    if kind == "layer":
        Q, q, scale, zero, g_idx, _, _ = run_mpq_quantization(
            W=s["W"], H=s["H"], quantizer=None, qcfg=_QCfg(case), module_name="model.layers.0.mlp.down_proj",
            vamp_cfg=s["vamp"], adapter_cfg=s["adapter"])
        return {"Q": Q, "q": q, "scale": scale, "zero": zero, "g_idx": g_idx}
    # the codes and the objective that they reach per row block; the decoded weights are the codes' codewords,
    # and a near-tie decided the other way is another codeword altogether, so the codes are what is compared
    _, idx, stats = mpq_refine_codebook(s["Wr"], s["H"], s["Wr"], s["idx0"], s["cb"], _QuipArgs(),
                                        module_name="model.layers.0.mlp.down")
    return {"idx": idx, "before": stats["exact_surrogate_before_chunk_means"],
            "after": stats["exact_surrogate_after_chunk_means"], "obs": stats["obs_precision_initial"]}


# ---- what a pass cannot do without -------------------------------------------------------------------

# one symmetric decomposition: reduction 4/3 n^3, tridiagonal eigenvectors 4/3 n^3, back-transformation 2 n^3
_EIGH = 4.0 / 3.0 + 4.0 / 3.0 + 2.0


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    rows = case.get("rows", 0)
    if kind == "quantize":  # 12334 floating-point operations per vector (factorized search), 8 floats in, 8 and an index out
        return {"bytes": 72.0 * case["vectors"], "flops": 12334.0 * case["vectors"]}
    if kind == "hessian":
        return {"bytes": (2.0 if case["bf16"] else 4.0) * case["tokens"] * n + 4.0 * n * n,
                "flops": float(case["tokens"]) * n * n}
    if kind == "awq":  # 20 ratios, each D H D^T with one product
        return {"bytes": 4.0 * (rows * n + n * n), "flops": 20 * 2.0 * rows * n * n}
    if kind == "eigh32":
        return {"bytes": 4.0 * 3 * n * n, "flops": (_EIGH + 2.0) * n ** 3}
    if kind == "eigh64":
        return {"bytes": 8.0 * 3 * n * n, "flops": (_EIGH + 2.0) * n ** 3}
    if kind == "block":  # W Vs, x_rtn Vs, then three products per iteration (at most 16)
        return {"bytes": 4.0 * (2 * n * n + 3 * rows * n), "flops": (4.0 + 6.0 * 4) * rows * n * n}
    if kind == "cd":  # two products in, one out, and one update of n entries per decision and sweep
        return {"bytes": 4.0 * (2 * n * n + rows * n), "flops": (6.0 + 2.0 * 3) * rows * n * n}
    if kind == "e8cd":  # products and updates as above, 65536 codewords x 8 coordinates per decision
        return {"bytes": 4.0 * (n * n + 2 * rows * n), "flops": (6.0 + 6.0) * rows * n * n + 3 * rows * (n / 8) * 65536 * 16.0}
    if kind == "layer":
        return {"bytes": 4.0 * (n * n + 2 * rows * n) + rows * n,
                "flops": _EIGH * n ** 3 + (4.0 + 6.0 * 16) * rows * n * n}
    return {"bytes": 4.0 * (n * n + 2 * rows * n), "flops": _EIGH * n ** 3 + (2.0 + 4.0 * 16) * rows * n * n}


# ---- tolerances and 64-bit values ----------------------------------------------------------------------


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"  # the search is exact and its results are codewords
    # "hessian", "awq", "eigh*": about four times the distance from 64 bits (the awq losses of small layers move
    # when a weight rounds the other way); the solvers: codes may differ on near-ties, about four times what
    # another order of the products' sums gives ("cd", "e8cd": a reordered near-tie moves later decisions too)
    return {
        "hessian": {"rel": 2e-5, "max": 6e-5},
        "awq": {"rel": 4e-5, "max": 2e-4},
        "eigh32": {"rel": 2.5e-4, "max": 8e-3},
        "eigh64": {"rel": 6e-14, "max": 4e-13},
        "block": {"rel": 5e-3, "max": 0.9, "differ": 1e-3},
        "cd": {"rel": 0.03, "max": 0.3, "differ": 0.01},
        "e8cd": {"rel": 0.03, "max": 0.3, "differ": 0.01},
        "layer": {"rel": 5e-3, "max": 0.9, "differ": 1e-3},
        "refine": {"rel": 5e-3, "max": 0.05, "differ": 1e-3},
    }[kind]


def _awq_exact(s):
    """The 20 losses sum(D H D^T) / rows, D = W - pseudo_quant(W s) / s, in float64."""
    case = s["case"]
    W, H, gs = s["W"].double(), s["H"].double(), case["group"]
    rows, n = W.shape
    a = W.abs().reshape(rows, n // gs, gs)
    w_mean = (a / (a.amax(dim=2, keepdim=True) + 1e-6)).reshape(rows, n).mean(dim=0)
    x_mean, maxq, losses = s["x_mean"].double(), 2 ** case["bits"] - 1, []
    for k in range(20):
        r = k / 20
        sc = (x_mean.pow(r) / (w_mean.pow(1 - r) + 1e-4)).clamp_min(1e-4)
        sc = sc / torch.sqrt(sc.max() * sc.min())
        Ws = (W * sc).reshape(rows, n // gs, gs)
        lo, hi = Ws.amin(dim=2, keepdim=True), Ws.amax(dim=2, keepdim=True)
        step = ((hi - lo).clamp_min(1e-5)) / maxq
        z = (-torch.round(lo / step)).clamp(0, maxq)
        D = W - ((torch.round(Ws / step) + z).clamp(0, maxq) - z).mul(step).reshape(rows, n) / sc
        losses.append(((D @ H) * D).sum() / rows)
    return torch.stack(losses)


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "quantize":
        if case["vectors"] > 16384:
            return None  # 65536 distances per vector
        grid, x = s["cb"].grid.double(), s["x"].double()
        idx = torch.cat([((p @ grid.T) - 0.5 * grid.square().sum(dim=1)).argmax(dim=1) for p in x.split(1024)])
        return {"vals": grid[idx], "idx": None}
    if kind == "hessian":
        X = s["x"].double()
        if case["conv"] == "gptq":
            return {"H": 2.0 * (X.T @ X)}
        mu = X.mean(dim=0)
        return {"H": X.T @ X / case["tokens"] - torch.outer(mu, mu), "mu": mu, "ct": None}
    if kind == "awq":
        return {"scales": None, "err": None, "ratio": None, "losses": _awq_exact(s)}
    if kind in ("eigh32", "eigh64"):
        # the damping keeps every eigenvalue above the adapter's floor, so the factor's Gram matrix is H
        H = s["H"].double()
        lam = torch.linalg.eigvalsh(H)
        out = {"lam": lam.flip(0) if kind == "eigh32" else lam, "gram": H, "unit": torch.eye(case["n"], device=DEV).double()}
        if kind == "eigh32":
            out["floor"] = None
        return out
    if kind in ("block", "cd", "e8cd"):
        # decisions of an iteration have no 64-bit value; the error of the given start has
        start = ((s["W"].double() - s["x"].double()) @ s["Vs"].double()).square().sum(dim=1)
        if kind == "block":
            return {"q": None, "x": None, "err": None, "rtn_err": start}
        if kind == "cd":
            return {"q": None, "before": start, "after": None, "improved": None, "accepted": None}
        return {"idx": None, "before": start, "after": None, "accepted": None}
    return None  # a chain of decisions: codes and what is decoded from them
