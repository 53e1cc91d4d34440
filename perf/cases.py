"""The work that is timed: calls of the public entry points at the sizes programs use them.

A case is a dict of plain values. Its "kind" names the entry point:

  ef      ef.ef_encode                one Linear: act order, factor, commits, sweeps, packing
  layers  ef.ef_encode_many           whole decoder layers (or a model) in one call
  hess    hessians.xtx_accumulate     the forward hook's H += X^T X, one activation batch
  hessn   hessians.xtx_accumulate_many   every input Hessian of some layers at once
  factor  ef.cholesky_inv_upper       the float64 inverse upper factor on its own
  codec   kquant.QUANTIZE / DEQUANTIZE   weighted or plain round-to-nearest, and the decode
  search  objective.tensor_err_many   the PERM search's objective under channel permutations
  tune    scale_tune.reconstruct      the distill stage's weight and its scale gradients
"""
import numpy as np
import torch

from perm_amd import ef, hessians, kquant, objective, scale_tune

BLOCK = {"Q8_0": (32, 34), "Q2_K": (256, 84), "Q3_K": (256, 110), "Q4_K": (256, 144),
         "Q5_K": (256, 176), "Q6_K": (256, 210)}
KQUANTS = ("Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K")
HAS_MIN = ("Q2_K", "Q4_K", "Q5_K")

# (name, rows, input width, input family) of one decoder layer
QWEN3_06B = (("attn_q", 2048, 1024, "qkv"), ("attn_k", 1024, 1024, "qkv"),
             ("attn_v", 1024, 1024, "qkv"), ("attn_output", 1024, 2048, "o"),
             ("ffn_gate", 3072, 1024, "gateup"), ("ffn_up", 3072, 1024, "gateup"),
             ("ffn_down", 1024, 3072, "down"))
LLAMA3_8B = (("attn_q", 4096, 4096, "qkv"), ("attn_k", 1024, 4096, "qkv"),
             ("attn_v", 1024, 4096, "qkv"), ("attn_output", 4096, 4096, "o"),
             ("ffn_gate", 14336, 4096, "gateup"), ("ffn_up", 14336, 4096, "gateup"),
             ("ffn_down", 4096, 14336, "down"))
MODELS = {"qwen3-0.6b": QWEN3_06B, "llama3-8b": LLAMA3_8B}
QWEN3_VOCAB = 151936


def listed():
    return [
        # encoding one Linear interactively: a 1024 x 1024 projection, imatrix weights and the
        # float64 Hessian a stored file expands to
        dict(name="ef-linear", kind="ef", ttype="Q2_K", rows=1024, n=1024, qw=True, h64=True),
        # one decoder layer of a small model at a mixed container (the tied-output recipe's
        # Q3_K attention and Q2_K MLP), its four Hessians as the hook leaves them
        dict(name="ef-layer-small", kind="layers", model="qwen3-0.6b", layers=1, mix="q3q2"),
        # the encode stage on a whole 28-layer model in one pass: the headline workload
        dict(name="ef-model", kind="layers", model="qwen3-0.6b", layers=28, mix="Q2_K"),
        # one wide decoder layer, the factor of a 14336-wide Hessian among it
        dict(name="ef-layer-wide", kind="layers", model="llama3-8b", layers=1, mix="Q4_K"),
        # the calibration hook on one 2048-token sequence, accumulating on the device
        dict(name="hess-hook", kind="hess", dtype="bf16", rows=2048, d=1024),
        # one layer's four input Hessians from a 65536-row calibration set
        dict(name="hess-layer", kind="hessn", dtype="bf16", model="qwen3-0.6b", layers=1, rows=65536),
        # float32 activations (a float32 or float16 model's hook) on an 8192-row set
        dict(name="hess-float32", kind="hess", dtype="f32", rows=8192, d=1024),
        # a caller's own factorization, at a width that is no multiple of any tile
        dict(name="factor-ragged", kind="factor", n=2000),
        # stock quantization of a projection with an imatrix, and the decode of its bytes
        dict(name="codec-q4k", kind="codec", ttype="Q4_K", rows=4096, n=4096, qw=True),
        # the tied output matrix: the largest tensor of a small model, plain Q6_K
        dict(name="codec-output", kind="codec", ttype="Q6_K", rows=QWEN3_VOCAB, n=1024, qw=False),
        # one candidate of the permutation search: four layers and the embedding's row sample
        dict(name="search-candidate", kind="search", layers=4, embed=True, sample=16384),
        # a distill step's forward and backward through one wide MLP matrix
        dict(name="tune-step", kind="tune", ttype="Q4_K", rows=14336, n=4096),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("ef", "layers", "hess", "hessn", "factor", "codec", "search", "tune"))
    if kind == "ef":
        return dict(kind=kind, ttype=rng.choice(KQUANTS), rows=_log(rng, 32, 8192),
                    n=256 * _log(rng, 1, 16), qw=rng.random() < 0.7, h64=rng.random() < 0.5)
    if kind == "layers":
        return dict(kind=kind, model="qwen3-0.6b", layers=_log(rng, 1, 28),
                    mix=rng.choice(KQUANTS + ("q3q2",)))
    if kind == "hess":
        if rng.random() < 0.5:
            return dict(kind=kind, dtype="bf16", rows=_log(rng, 64, 65536), d=8 * _log(rng, 32, 768))
        return dict(kind=kind, dtype="f32", rows=_log(rng, 64, 16384), d=_log(rng, 200, 4096))
    if kind == "hessn":
        return dict(kind=kind, dtype="bf16", model="qwen3-0.6b", layers=_log(rng, 1, 4),
                    rows=_log(rng, 512, 32768))
    if kind == "factor":
        return dict(kind=kind, n=_log(rng, 64, 4096))
    if kind == "codec":
        return dict(kind=kind, ttype=rng.choice(tuple(BLOCK)), rows=_log(rng, 1, 20000),
                    n=256 * _log(rng, 1, 24), qw=rng.random() < 0.5)
    if kind == "search":
        return dict(kind=kind, layers=_log(rng, 1, 8), embed=rng.random() < 0.5,
                    sample=_log(rng, 512, 16384))
    return dict(kind=kind, ttype=rng.choice(KQUANTS), rows=_log(rng, 16, 14336), n=256 * _log(rng, 1, 24))


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _activations(g, rows, d):
    """Student-t (nu = 4) rows times log-normal channel scales."""
    chi = sum(_randn(g, rows, 1) ** 2 for _ in range(4)) / 4
    return _randn(g, rows, d) / torch.sqrt(chi) * torch.exp(_randn(g, d))


def _hessian(g, d, rows):
    """X^T X of bf16 activations, symmetric float32."""
    x = _activations(g, rows, d).to(torch.bfloat16).float()
    h = x.T @ x
    return torch.tril(h) + torch.tril(h, -1).T


def _weights(g, rows, n):
    return _randn(g, rows, n) * 0.02


def _mixed(mix, name):
    if mix != "q3q2":
        return mix
    return "Q3_K" if name.startswith("attn") else "Q2_K"


def _families(model):
    out = {}
    for _name, _rows, n, fam in MODELS[model]:
        out[fam] = n
    return out


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "ef":
        n = case["n"]
        H = _hessian(g, n, 4 * n)
        qw = (H.diagonal() / (4 * n)).contiguous() if case["qw"] else None
        return dict(case, x=_weights(g, case["rows"], n), w=qw, H=H.double() if case["h64"] else H)
    if kind == "layers":
        tensors = []
        for l in range(case["layers"]):
            H = {}
            for fam, d in _families(case["model"]).items():
                rows = max(8192, d + d // 8)
                H[fam] = _hessian(g, d, rows)
            for name, rows, n, fam in MODELS[case["model"]]:
                tensors.append({"name": f"blk.{l}.{name}", "ttype": _mixed(case["mix"], name),
                                "x": _weights(g, rows, n), "H": H[fam],
                                "qw": (H[fam].diagonal() / 8192).contiguous()})
        return dict(case, tensors=tensors)
    if kind == "hess":
        X = _activations(g, case["rows"], case["d"])
        X = X.to(torch.bfloat16) if case["dtype"] == "bf16" else X
        return dict(case, X=X.unsqueeze(0), H=torch.zeros(case["d"], case["d"], device="cuda"))
    if kind == "hessn":
        ds = list(_families(case["model"]).values()) * case["layers"]
        return dict(case, X=[_activations(g, case["rows"], d).to(torch.bfloat16) for d in ds],
                    H=[torch.zeros(d, d, device="cuda") for d in ds])
    if kind == "factor":
        return dict(case, H=_hessian(g, case["n"], 4 * case["n"]).double())
    if kind == "codec":
        qw = _randn(g, case["n"]).abs() + 0.1 if case["qw"] else None
        return dict(case, x=_weights(g, case["rows"], case["n"]), w=qw)
    if kind == "search":
        return dict(case, items=_search_items(case, g))
    if kind == "tune":
        return dict(case, **_tune_inputs(case, g))
    raise KeyError(kind)


def _search_items(case, g):
    """The items one candidate is scored by: the residual permutation on every tensor that
    reads the residual stream, each layer's own permutation on its down and output inputs."""
    def perm(n):
        return torch.randperm(n, generator=g, device="cuda").to(torch.int32)

    res, items = perm(1024), []
    if case["embed"]:
        items.append(dict(x=_weights(g, QWEN3_VOCAB, 1024).half(), ttype="Q6_K", qw=None, perm=res,
                          rows_sample=case["sample"]))
    for _ in range(case["layers"]):
        for name, rows, n, fam in QWEN3_06B:
            items.append(dict(x=_weights(g, rows, n).half(), ttype=_mixed("q3q2", name),
                              qw=_randn(g, n).abs() + 0.1,
                              perm=res if fam in ("qkv", "gateup") else perm(n),
                              rows_sample=case["sample"]))
    return items


def _tune_inputs(case, g):
    """A tensor's linear form as build_torch_params holds it (random codes and scales in the
    container's ranges) and the gradient that arrives at its weight."""
    rows, n, tt = case["rows"], case["n"], case["ttype"]

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int16)

    sub = {"Q4_K": 32, "Q5_K": 32}.get(tt, 16)
    sc = {"Q2_K": (0, 16), "Q3_K": (-32, 32), "Q4_K": (0, 64), "Q5_K": (0, 64), "Q6_K": (-128, 128)}[tt]
    q = {"Q2_K": (0, 4), "Q3_K": (-4, 4), "Q4_K": (0, 16), "Q5_K": (0, 32), "Q6_K": (-32, 32)}[tt]
    A = (ints(*q, rows, n // sub, sub) * ints(*sc, rows, n // sub, 1)).reshape(rows, n)
    entry = {"d": _fp16_scales(g, rows, n), "dmin": None, "A": A, "B": None, "ttype": tt, "shape": (rows, n)}
    if tt in HAS_MIN:
        entry["dmin"] = _fp16_scales(g, rows, n)
        entry["B"] = ints(0, 16 if tt == "Q2_K" else 64, rows, n // sub, 1).expand(
            rows, n // sub, sub).reshape(rows, n).contiguous()
    for k in ("d", "dmin"):
        if entry[k] is not None:
            entry[k].requires_grad_(True)
    return dict(entry=entry, gW=_randn(g, rows, n))


def _fp16_scales(g, rows, n):
    return (torch.rand((rows, n // 256), generator=g, device="cuda") * 1e-3 + 1e-4).half().float()


# ---------------------------------------------------------------- the calls

def run(state):
    kind = state["kind"]
    if kind == "ef":
        return ef.ef_encode(state["x"], state["ttype"], state["w"], state["H"])
    if kind == "layers":
        got = ef.ef_encode_many(state["tensors"])
        if len(got) <= 28:
            return got
        # a whole model's bytes leave in one buffer, as the file driver copies them out
        by = {}
        for raw, rec in got.values():
            by.setdefault(rec.shape[1], []).append(rec)
        return {"raw": torch.cat([raw.reshape(-1) for raw, _ in got.values()]),
                "recon": [torch.cat(v) for v in by.values()]}
    if kind == "hess":
        return hessians.xtx_accumulate(state["X"], state["H"])
    if kind == "hessn":
        return hessians.xtx_accumulate_many(state["X"], state["H"])
    if kind == "factor":
        return ef.cholesky_inv_upper(state["H"])
    if kind == "codec":
        raw = kquant.QUANTIZE[state["ttype"]](state["x"], state["w"])
        return raw, kquant.DEQUANTIZE[state["ttype"]](raw, state["n"])
    if kind == "search":
        return objective.tensor_err_many(state["items"])
    e = state["entry"]
    W = scale_tune.reconstruct(e)
    wrt = [e["d"]] + ([e["dmin"]] if e["dmin"] is not None else [])
    return (W.detach(), *torch.autograd.grad(W, wrt, state["gW"]))


# ---------------------------------------------------------------- what a pass cannot do without

def _row_bytes(ttype, n):
    w, b = BLOCK[ttype]
    return n // w * b


def _ef_work(ttype, rows, n):
    """x read, the container and the reconstruction written; two sweeps of a product and a
    subtraction per (row, column pair)."""
    return rows * (8 * n + _row_bytes(ttype, n)), 2 * rows * n * (n - 1)


def work(case):
    kind = case["kind"]
    if kind == "ef":
        n = case["n"]
        b, f = _ef_work(case["ttype"], case["rows"], n)
        return {"bytes": b + n * n * (8 if case["h64"] else 4), "flops": f + 2 * n**3 // 3}
    if kind == "layers":
        b = f = 0
        for name, rows, n, _fam in MODELS[case["model"]]:
            tb, tf = _ef_work(_mixed(case["mix"], name), rows, n)
            b, f = b + tb, f + tf
        for d in _families(case["model"]).values():
            b, f = b + 4 * d * d, f + 2 * d**3 // 3
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    if kind in ("hess", "hessn"):
        ds = [case["d"]] if kind == "hess" else list(_families(case["model"]).values()) * case["layers"]
        e = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": sum(e * case["rows"] * d + 8 * d * d for d in ds),
                "flops": sum(case["rows"] * d * (d + 1) for d in ds)}
    if kind == "factor":
        return {"bytes": 16 * case["n"] ** 2, "flops": 2 * case["n"] ** 3 // 3}
    if kind == "codec":
        rows, n = case["rows"], case["n"]
        # encode: weights in, bytes out; decode: bytes in, weights out
        return {"bytes": rows * (8 * n + 2 * _row_bytes(case["ttype"], n)), "flops": 0}
    if kind == "search":
        w = case["layers"] * sum(min(rows, case["sample"]) * n for _k, rows, n, _f in QWEN3_06B)
        return {"bytes": 2 * (w + (case["sample"] * 1024 if case["embed"] else 0)), "flops": 0}
    # forward: A (and B) in, W out; backward: the gradient and A (and B) in
    ab = 4 if case["ttype"] in HAS_MIN else 2
    return {"bytes": case["rows"] * case["n"] * (2 * ab + 8), "flops": 4 * ab * case["rows"] * case["n"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("ef", "layers"):
        # The sweep is exact given its factor. A float64 factor formed in another order changes
        # single float32 entries of U; where a code then sits on a tie, the rest of its row
        # moves. Against torch's float64 Cholesky: nothing moved in tensors up to 3072 wide (one
        # moved row of about 1024 is then the least that can differ); at 14336 up to 1.8e-3 of
        # the bytes of a tensor, and its reconstruction by 9.6e-3 (single weights by 0.93).
        wide = (case["n"] if kind == "ef" else max(_families(case["model"]).values())) > 4096
        return {"rel": 0.03, "max": 0.99, "differ": 7e-3} if wide else \
            {"rel": 0.01, "max": 0.99, "differ": 1e-3}
    if kind in ("hess", "hessn"):
        return {"rel": 2e-6}  # up to 4.5e-7 from the float64 sums (the 3072-wide one)
    if kind == "factor":
        return {"rel": 1e-14}  # 8e-16 from torch's float64 Cholesky at 2000
    if kind == "tune":
        return {"rel": 4e-7}  # the weight is exact, the 256-term gradient sums 8e-8 off
    return "exact"  # the codec's bytes and the objective built on them


# ---------------------------------------------------------------- 64 bits, plain torch

def exact(case, seed):
    kind = case["kind"]
    if kind not in ("hess", "hessn", "factor", "tune"):
        return None  # bytes, and reconstructions that follow them
    s = prepare(case, seed)
    if kind == "hess":
        x = s["X"][0].double()
        return x.T @ x
    if kind == "hessn":
        out = []
        for X in s["X"]:
            h = 0
            for part in X.split(8192):
                h = h + part.double().T @ part.double()
            out.append(h)
        return out
    if kind == "factor":
        n = case["n"]
        H = s["H"]
        lam = 0.01 * float(np.mean(H.diagonal().cpu().numpy())) + 1e-8
        # U^T U = inv(H + lam I), U upper: with J the reversal, J (H + lam I) J = L L^T gives
        # U = J inv(L) J
        A = torch.flip(H + lam * torch.eye(n, device="cuda", dtype=torch.float64), (0, 1))
        L = torch.linalg.cholesky(A)
        eye = torch.eye(n, device="cuda", dtype=torch.float64)
        return torch.flip(torch.linalg.solve_triangular(L, eye, upper=False), (0, 1))
    e, g = s["entry"], s["gW"].double()
    rows, n = case["rows"], case["n"]

    def wide(v):
        return v.detach().double().repeat_interleave(256, dim=1)

    A = e["A"].double()
    W, gd = wide(e["d"]) * A, (g * A).reshape(rows, n // 256, 256).sum(-1)
    if e["dmin"] is None:
        return W, gd
    B = e["B"].double()
    return W - wide(e["dmin"]) * B, gd, -(g * B).reshape(rows, n // 256, 256).sum(-1)
