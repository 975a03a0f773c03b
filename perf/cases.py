"""Cases of the hybrid SpMM / SDDMM / sparse-attention path, as programs call it.

A case is a dict of plain values.  `prepare` makes what a program holds before
a call: the plan of its sparse operand (the tile search and the plan upload
are done once per sparsity pattern and kept, as a program keeps them) and
fresh dense operands, values and output buffers from the seed.  `run` is one
pass through the public entry points: `Plan.run_spmm`, `Plan.run_sddmm`,
`Plan.run_attention`, `BatchedSparseAttention.forward`, and forward +
backward through `SparseOperand` / `gcn_layer`.

Kinds:
  layer      C = A.B, A a block-pruned projection (10 % dense 16x16 blocks +
             1 % residual)
  batch      the block-pruned projections of an encoder, one launch
  uniform    C = A.B, A with uniformly drawn nonzeros, FP32
  graph      C = A.B over an R-MAT graph, FP32, rows summed in fixed order
  sddmm      sampled X.Y^T on an R-MAT graph's pattern
  gcn        one GCN layer, forward and backward (H, W and edge values)
  attention  fused sparse attention, head dimension 64, many uneven masks
  attend     sparse attention with another head dimension (SDDMM, row
             softmax, value refresh, SpMM)
  train      a pruned layer's forward and backward (weights and input)
"""
import functools
import math

import numpy as np
import torch

from stile_amd import _native, api, datasets
from stile_amd.attention import BatchedSparseAttention
from stile_amd.autograd import SparseOperand, gcn_layer

DEV = "cuda"


def listed():
    return [
        # token-by-token decode of 16 sequences through a pruned FFN-in
        # projection: the smallest call, launch and staging latency
        {"name": "layer_decode", "kind": "layer", "pattern": 0, "M": 3072, "K": 768, "N": 16,
         "blocks": "bfloat16", "b": "bfloat16", "pad": 0},
        # the same layer over a prefill of 4096 tokens: the benchmark's
        # headline configuration
        {"name": "layer_prefill", "kind": "layer", "pattern": 0, "M": 3072, "K": 768, "N": 4096,
         "blocks": "bfloat16", "b": "bfloat16", "pad": 0},
        # a projection of no convenient size in FP16, its activations a slice
        # of a wider buffer: ragged rows, columns and leading dimension
        {"name": "layer_odd_f16", "kind": "layer", "pattern": 1, "M": 1000, "K": 747, "N": 321,
         "blocks": "float16", "b": "float16", "pad": 30},
        # the FFN output projection of a BERT-large-shaped encoder (K = 4096)
        {"name": "layer_ffn_out", "kind": "layer", "pattern": 2, "M": 1024, "K": 4096, "N": 512,
         "blocks": "bfloat16", "b": "bfloat16", "pad": 0},
        # every other projection of that encoder, 24 layers, in one launch
        {"name": "encoder_batch", "kind": "batch", "pattern": 0, "layers": 24, "d": 1024, "ffn": 4096, "N": 128},
        # the small unstructured benchmark
        {"name": "uniform_n64", "kind": "uniform", "pattern": 0, "M": 4096, "K": 4096, "nnz": 167772, "N": 64},
        # aggregation over a large graph, run reproducibly: only sparse tiles
        {"name": "graph_sum", "kind": "graph", "pattern": 0, "scale": 17, "N": 128},
        # the SDDMM benchmark: edge scores of a graph
        {"name": "sddmm_rmat", "kind": "sddmm", "pattern": 0, "scale": 16, "K": 32},
        # one training step of a GCN layer
        {"name": "gcn_step", "kind": "gcn", "pattern": 0, "scale": 15, "F": 256},
        # four sequences of uneven length, 16 heads each, band + random mask
        {"name": "attention_band", "kind": "attention", "pattern": 0, "lens": "640,1501,2900,5120", "heads": 16},
        # the reference's LogSparse and strided masks at head dimension 128
        {"name": "attend_d128", "kind": "attend", "pattern": 0, "log": 2048, "strided": 1100, "d": 128},
        # fine-tuning step of a pruned layer: output, weight and input gradients
        {"name": "layer_train", "kind": "train", "pattern": 0, "M": 3072, "K": 768, "N": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "batch", "uniform", "graph", "sddmm", "gcn", "attention",
                       "attend", "train"])
    case = {"kind": kind, "pattern": rng.randrange(1, 1000)}
    if kind == "layer":
        case.update(M=_log(rng, 200, 4096), K=_log(rng, 200, 4096), N=_log(rng, 8, 4096))
        case.update(blocks=rng.choice(["bfloat16", "bfloat16", "float16", "float32"]))
        case.update(b=case["blocks"] if rng.random() < 0.7 else "float32", pad=rng.choice([0, 0, rng.randrange(1, 40)]))
        if rng.random() < 0.5:   # sizes of real layers are mostly multiples of 64
            case.update(M=64 * max(1, case["M"] // 64), K=64 * max(1, case["K"] // 64))
        if rng.random() < 0.5:
            case.update(N=8 * (case["N"] // 8))
        while case["M"] * case["K"] * case["N"] > 3072 * 768 * 4096:
            case["N"] = max(8, case["N"] // 2)
    elif kind == "batch":
        d = 64 * rng.randrange(2, 17)
        case.update(layers=rng.randrange(1, 25), d=d, ffn=d * rng.choice([2, 3, 4]), N=_log(rng, 8, 128))
    elif kind == "uniform":
        M, K = _log(rng, 300, 8192), _log(rng, 300, 8192)
        case.update(M=M, K=K, nnz=max(1, int(M * K * math.exp(rng.uniform(math.log(0.001), math.log(0.02))))),
                    N=_log(rng, 4, 512))
    elif kind == "graph":
        case.update(scale=rng.randrange(11, 17), N=_log(rng, 8, 256))
    elif kind == "sddmm":
        case.update(scale=rng.randrange(11, 16), K=_log(rng, 8, 256))
    elif kind == "gcn":
        case.update(scale=rng.randrange(11, 15), F=_log(rng, 16, 256))
    elif kind == "attention":
        lens = [_log(rng, 200, 3000) for _ in range(rng.randrange(1, 5))]
        case.update(lens=",".join(str(n) for n in lens), heads=rng.randrange(1, 17))
    elif kind == "attend":
        case.update(log=_log(rng, 200, 2048), strided=_log(rng, 200, 1100), d=rng.choice([32, 48, 80, 96, 128]))
    else:
        case.update(M=16 * _log(rng, 16, 192), K=16 * _log(rng, 16, 64), N=_log(rng, 16, 1024))
    return case


# ---------------------------------------------------------------------------
# Sparsity patterns and plans, kept per pattern.
# ---------------------------------------------------------------------------

_KEYS = {"layer": ("M", "K"), "batch": ("layers", "d", "ffn"), "uniform": ("M", "K", "nnz"), "graph": ("scale",),
         "sddmm": ("scale",), "gcn": ("scale",), "attention": ("lens", "heads"), "attend": ("log", "strided"),
         "train": ("M", "K")}
_PLAN_KEYS = {"layer": ("blocks",), "gcn": ("F",), "attend": ("d",)}


def _matrices(case):
    """The case's sparse matrices (a tuple of CSR matrices, one per instance)."""
    kind = case["kind"]
    return _matrices_of(kind, case["pattern"], tuple(case[k] for k in _KEYS[kind]))


@functools.lru_cache(maxsize=32)
def _matrices_of(kind, pattern, size):
    if kind in ("layer", "train"):
        M, K = size
        return (datasets.pruned_layer(seed=pattern, M=M, K=K, N=1)[0],)
    if kind == "batch":
        layers, d, ffn = size
        # one mask per projection, shared by the layers
        one = [datasets.pruned_layer(seed=pattern + 10 * j, M=m, K=d, N=1)[0]
               for j, m in enumerate((d, d, d, d, ffn))]
        return tuple(one * layers)
    if kind == "uniform":
        M, K, nnz = size
        return (datasets.uniform_spmm(seed=pattern, M=M, K=K, nnz=nnz, N=1)[0],)
    if kind in ("graph", "gcn"):
        return (datasets.gcn_graph(size[0], seed=pattern, feat=1)[0],)
    if kind == "sddmm":
        return (datasets.rmat_graph(size[0], seed=pattern),)
    if kind == "attention":
        lens, heads = size
        rng = np.random.default_rng(pattern)
        one = [datasets.attention_mask(int(n), rng=rng) for n in lens.split(",")]
        return tuple(m for m in one for _ in range(heads))
    return datasets.log_sparse_mask(size[0]), datasets.strided_mask(size[1])


def _plan(case):
    """What the program keeps for the case's sparse operand: a plan, a
    SparseOperand or a BatchedSparseAttention."""
    kind = case["kind"]
    return _plan_of(kind, case["pattern"], tuple(case[k] for k in _KEYS[kind]),
                    tuple(case[k] for k in _PLAN_KEYS.get(kind, ())))


def _packs(mats, blocks, **search):
    """One searched pack per matrix; a matrix that comes again is searched once."""
    found, opts = {}, api.options_for(blocks)
    for k, v in search.items():
        setattr(opts, k, v)
    for A in mats:
        if id(A) not in found:
            found[id(A)] = api.spmm_pack(A, opts)[0]
    return [found[id(A)] for A in mats]


@functools.lru_cache(maxsize=20)
def _plan_of(kind, pattern, size, opts):
    mats = _matrices_of(kind, pattern, size)
    if kind == "layer":
        return _native.Plan.spmm(_packs(mats, opts[0]), opts[0])
    if kind == "batch":
        return _native.Plan.spmm(_packs(mats, "bfloat16"), "bfloat16")
    if kind == "uniform":
        return _native.Plan.spmm(_packs(mats, "float32"), "float32")
    if kind == "graph":
        return _native.Plan.spmm(_packs(mats, "float32", only_ELL=True), "float32")
    if kind == "sddmm":
        return api.build_sddmm_plan(mats[0])
    if kind == "gcn":
        return SparseOperand(mats[0], blk_dtype="float32", device=DEV, N=opts[0], workers=1)
    if kind == "attention":
        return _native.Plan.attention(_packs(mats, "bfloat16"))
    if kind == "attend":
        return BatchedSparseAttention(list(mats), opts[0], device=DEV, workers=1, fused=False)
    return SparseOperand(mats[0], blk_dtype="bfloat16", device=DEV, N=1024, workers=1)


# ---------------------------------------------------------------------------
# Inputs, one pass, and what it cannot do without.
# ---------------------------------------------------------------------------

def _inputs(case, seed):
    """Dense operands and values, from the seed alone."""
    kind = case["kind"]
    mats = _matrices(case)
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))

    def randn(*shape):
        return torch.randn(*shape, device=DEV, generator=g)

    M = sum(A.shape[0] for A in mats)
    K = sum(A.shape[1] for A in mats)
    if kind in ("layer", "batch", "uniform", "graph"):
        dtype = getattr(torch, case.get("b", "bfloat16" if kind == "batch" else "float32"))
        N, pad = case["N"], case.get("pad", 0)
        return {"B": randn(K, N + pad).to(dtype)[:, :N]}
    if kind == "sddmm":
        return {"X": randn(M, case["K"]), "Y": randn(K, case["K"])}
    if kind == "gcn":
        F, A = case["F"], mats[0]
        near = torch.from_numpy(A.data).to(DEV)  # normalised edge weights, learned from there
        return {"H": randn(M, F), "W": randn(F, F) / math.sqrt(F), "values": near * (1 + 0.1 * randn(A.nnz)),
                "dY": randn(M, F) / math.sqrt(M)}
    if kind == "attention":
        return {n: randn(M, 64).to(torch.bfloat16) for n in "QKV"}
    if kind == "attend":
        return {n: randn(M, case["d"]) for n in "QKV"}
    near = torch.from_numpy(mats[0].data).to(DEV)
    return {"B": randn(K, case["N"]), "values": near + 0.002 * randn(mats[0].nnz), "dC": randn(M, case["N"])}


def prepare(case, seed):
    kind = case["kind"]
    plan = _plan(case)
    state = dict(_inputs(case, seed), kind=kind, plan=plan)
    if kind in ("layer", "batch", "uniform", "graph"):
        state["out"] = torch.empty(plan.M, case["N"], device=DEV)
    elif kind == "sddmm":
        state["out"] = torch.empty(plan.nnz, device=DEV)
    elif kind in ("attention", "attend"):
        state["out"] = torch.empty(state["Q"].shape[0], state["Q"].shape[1], device=DEV)
        state["scale"] = 1 / math.sqrt(state["Q"].shape[1])
    else:
        for name in ("H", "W", "values", "B"):
            if name in state:
                state[name].requires_grad_(True)
    return state


def run(state):
    s, kind, plan = state, state["kind"], state["plan"]
    if kind in ("layer", "batch", "uniform"):
        return plan.run_spmm(s["B"], s["out"])
    if kind == "graph":
        return plan.run_spmm(s["B"], s["out"], deterministic=True)
    if kind == "sddmm":
        return plan.run_sddmm(s["X"], s["Y"], s["out"])
    if kind == "attention":
        return plan.run_attention(s["Q"], s["K"], s["V"], s["scale"], s["out"])
    if kind == "attend":
        return plan.forward(s["Q"], s["K"], s["V"], out=s["out"])
    if kind == "gcn":
        y = gcn_layer(plan, s["H"], s["W"], s["values"])
        dH, dW, dvalues = torch.autograd.grad(y, (s["H"], s["W"], s["values"]), s["dY"])
        return {"y": y.detach(), "dH": dH, "dW": dW, "dvalues": dvalues}
    C = plan.spmm(s["B"], s["values"])
    dvalues, dB = torch.autograd.grad(C, (s["values"], s["B"]), s["dC"])
    return {"C": C.detach(), "dvalues": dvalues, "dB": dB}


def _operand_bytes(case, A):
    """Bytes of A: a full 16x16 block of a pruned matrix is its values and one
    index, any other nonzero a value and an index."""
    if case["kind"] not in ("layer", "batch", "train"):
        return 8 * A.nnz
    size = 4 if case.get("blocks") == "float32" else 2
    rows = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr)) // 16
    _, count = np.unique(rows.astype(np.int64) * (A.shape[1] // 16 + 1) + A.indices // 16, return_counts=True)
    full = int((count == 256).sum())
    return full * (256 * size + 4) + (A.nnz - 256 * full) * 8


def work(case):
    kind = case["kind"]
    mats = _matrices(case)
    nnz = sum(A.nnz for A in mats)
    M, K = sum(A.shape[0] for A in mats), sum(A.shape[1] for A in mats)
    sizes = {id(A): _operand_bytes(case, A) for A in mats}
    held = sum(sizes[id(A)] for A in mats) + 4 * (M + len(mats))
    if kind in ("layer", "batch", "uniform", "graph"):
        N = case["N"]
        b = {"float32": 4}.get(case.get("b", "bfloat16" if kind == "batch" else "float32"), 2)
        return {"bytes": held + K * N * b + M * N * 4, "flops": 2 * nnz * N}
    if kind == "sddmm":
        return {"bytes": held + (M + K) * case["K"] * 4, "flops": 2 * nnz * case["K"]}
    if kind == "gcn":
        F = case["F"]
        # forward H, W -> HW -> y; backward dY -> d(HW), dvalues, dH, dW
        return {"bytes": 3 * held + 4 * (M * F * 8 + 5 * F * F + nnz), "flops": 3 * 2 * nnz * F + 3 * 2 * M * F * F}
    if kind == "attention":
        return {"bytes": 4 * nnz + M * 64 * (3 * 2 + 4), "flops": 4 * nnz * 64}
    if kind == "attend":
        return {"bytes": 4 * nnz + M * case["d"] * 16, "flops": 4 * nnz * case["d"]}
    N = case["N"]
    return {"bytes": 3 * held + 4 * (3 * M * N + 3 * K * N + 2 * nnz), "flops": 3 * 2 * nnz * N}


# ---------------------------------------------------------------------------
# The same products in 64 bits.
# ---------------------------------------------------------------------------

def _coo(A):
    rows = np.repeat(np.arange(A.shape[0], dtype=np.int64), np.diff(A.indptr))
    return (torch.from_numpy(rows).to(DEV), torch.from_numpy(A.indices.astype(np.int64)).to(DEV),
            torch.from_numpy(A.data).to(DEV).double())


def _pieces(n, width):
    step = max(1, (1 << 26) // max(width, 1))
    return [slice(i, min(n, i + step)) for i in range(0, n, step)]


def _sum(rows, cols, vals, B, M):
    out = torch.zeros(M, B.shape[1], dtype=torch.float64, device=DEV)
    for p in _pieces(len(rows), B.shape[1]):
        out.index_add_(0, rows[p], vals[p, None] * B[cols[p]].double())
    return out


def _dots(rows, cols, X, Y):
    out = torch.empty(len(rows), dtype=torch.float64, device=DEV)
    for p in _pieces(len(rows), X.shape[1]):
        out[p] = (X[rows[p]].double() * Y[cols[p]].double()).sum(1)
    return out


def _attend(A, Q, K, V, scale):
    rows, cols, _ = _coo(A)
    s = _dots(rows, cols, Q, K) * scale
    top = torch.full((A.shape[0],), -math.inf, dtype=torch.float64, device=DEV)
    top.scatter_reduce_(0, rows, s, "amax")
    w = torch.exp(s - top[rows])
    total = torch.zeros(A.shape[0], dtype=torch.float64, device=DEV).index_add_(0, rows, w)
    return _sum(rows, cols, w / total[rows], V, A.shape[0])


def exact(case, seed):
    kind = case["kind"]
    mats = _matrices(case)
    v = {k: t.double() for k, t in _inputs(case, seed).items()}
    if kind in ("layer", "batch", "uniform", "graph"):
        parts, k0 = [], 0
        for A in mats:
            rows, cols, vals = _coo(A)
            B = v["B"][k0:k0 + A.shape[1]]
            if kind in ("layer", "batch"):
                dense = torch.zeros(A.shape, dtype=torch.float64, device=DEV)
                dense[rows, cols] = vals
                parts.append(dense @ B)
            else:
                parts.append(_sum(rows, cols, vals, B, A.shape[0]))
            k0 += A.shape[1]
        return torch.cat(parts)
    if kind in ("attention", "attend"):
        scale, parts, r0 = 1 / math.sqrt(v["Q"].shape[1]), [], 0
        for A in mats:
            r = slice(r0, r0 + A.shape[0])
            parts.append(_attend(A, v["Q"][r], v["K"][r], v["V"][r], scale))
            r0 += A.shape[0]
        return torch.cat(parts)
    rows, cols, _ = _coo(mats[0])
    if kind == "sddmm":
        return _dots(rows, cols, v["X"], v["Y"])
    M, K = mats[0].shape
    if kind == "gcn":
        HW = v["H"] @ v["W"]
        dHW = _sum(cols, rows, v["values"], v["dY"], K)
        return {"y": _sum(rows, cols, v["values"], HW, M), "dH": dHW @ v["W"].t(), "dW": v["H"].t() @ dHW,
                "dvalues": _dots(rows, cols, v["dY"], HW)}
    return {"C": _sum(rows, cols, v["values"], v["B"], M), "dvalues": _dots(rows, cols, v["dC"], v["B"]),
            "dB": _sum(cols, rows, v["values"], v["dC"], K)}
