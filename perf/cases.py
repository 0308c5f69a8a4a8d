"""The work the performance of this framework is measured on.

Five kinds of pass, all through the public entry points of `vectorsparse_amd.ops`:

    spmm       one SpMM with a pruned weight matrix (column-vector CSR) and a dense activation matrix
    sddmm      one SDDMM: a dense product sampled on a fixed mask
    train      forward and weight gradient of a pruned layer: Y = W X (SpMM), then dW = (dY X^T) on W's pattern (SDDMM)
    attention  one fixed-mask sparse attention layer, default route
    chain      the same layer as its three operators, which keeps the probabilities (what a training forward does)

Vector lengths are 1, 2, 4 and 8, operands fp16, outputs fp16 or fp32, sparsities 50 to 98 %.
"""
import math

import numpy as np
import torch

from vectorsparse_amd import colvec_csr as cv
from vectorsparse_amd import ops

SPARSITIES = (0.5, 0.7, 0.8, 0.9, 0.95, 0.98)


def listed():
    return [
        # the smallest call: the 256 x 256 x 128 problem at V = 4, through the operator as the benchmark calls it
        dict(name="spmm_small", op="spmm", entry="operator", V=4, m=256, n=256, k=128, sparsity=0.9, rows="uniform", kernel="wmma", out="f16"),
        # a 3x3 convolution of ResNet-50 (512 x 4608) at 90 %, mildly skewed rows: the headline shape
        dict(name="spmm_conv", op="spmm", entry="problem", V=8, m=512, n=4608, k=256, sparsity=0.9, rows="binomial", kernel="wmma", out="f16"),
        # unstructured pruning on the fine-grained path, one of the larger convolution shapes
        dict(name="spmm_fine_grained", op="spmm", entry="problem", V=1, m=2048, n=2304, k=256, sparsity=0.9, rows="binomial", kernel="cuda", out="f16"),
        # sizes that are multiples of nothing, fp32 result: a first layer (147 = 3 * 7 * 7 columns), odd dense width
        dict(name="spmm_ragged", op="spmm", entry="problem", V=2, m=1022, n=147, k=205, sparsity=0.7, rows="binomial", kernel="wmma", out="f32"),
        # rows of very different lengths (global pruning leaves some filters dense), schedule chosen by the library
        dict(name="spmm_skewed", op="spmm", entry="auto", V=8, m=8192, n=4608, k=256, sparsity=0.94, rows="pareto", kernel="wmma", out="f16"),
        # the largest call: a pruned 4096 x 4096 projection over the 2048 tokens of a prefill
        dict(name="spmm_tokens", op="spmm", entry="problem", V=4, m=4096, n=4096, k=2048, sparsity=0.8, rows="binomial", kernel="wmma", out="f16"),
        # SDDMM of 2048 x 2048 at 90 %, contraction length 64: the sparse-attention scores of one head
        dict(name="sddmm_mask", op="sddmm", V=8, m=2048, n=2048, k=64, sparsity=0.9, rows="binomial", kernel="wmma", out="f16"),
        # unstructured mask, moderate sparsity, long contraction: the large end of the SDDMM sweep
        dict(name="sddmm_fine_grained", op="sddmm", V=1, m=4096, n=4096, k=256, sparsity=0.8, rows="binomial", kernel="wmma", out="f16"),
        # a training step of a pruned layer over 512 samples: output and fp32 weight gradient
        dict(name="train_layer", op="train", V=4, m=2048, n=2304, k=512, sparsity=0.9, rows="binomial", out="f32"),
        # the sparse-transformer layer: 16 heads x 4096, local band of 256 and every 128th column
        dict(name="attention_band", op="attention", mask="band", V=8, heads=16, seq=4096, d=64, half_width=128, stride=128),
        # a band with global tokens: some rows attend to everything, everybody attends to some columns
        dict(name="attention_global", op="attention", mask="global", V=8, heads=8, seq=2048, d=64, half_width=64, stride=0, tokens=64),
        # a random mask with the probabilities kept for the backward pass: SDDMM, softmax and SpMM one after the other
        dict(name="attention_chain", op="chain", mask="random", V=4, heads=8, seq=2048, d=64, sparsity=0.95),
    ]


# What a drawn case may take: the gathered elements (nonzero vectors times dense width) of the largest listed one.
MOST_GATHER = 1024 * 4096 * 0.2 * 2048


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _some_width(rng, lo, hi):
    """A dense width: mostly a multiple of 8, now and then of 4, now and then of nothing."""
    w = _log(rng, lo, hi)
    step = rng.choice((8, 8, 8, 8, 4, 1))
    return max(step, w // step * step)


def draw(rng):
    op = rng.choice(("spmm", "spmm", "spmm", "sddmm", "sddmm", "train", "attention", "chain"))
    V = rng.choice((1, 2, 4, 8))
    sparsity = rng.choice(SPARSITIES) if rng.random() < 0.5 else round(rng.uniform(0.5, 0.98), 3)
    if op in ("attention", "chain"):
        heads, seq = rng.choice((1, 2, 4, 8, 12, 16)), _log(rng, 512 // V, 4096 // V) * V
        case = dict(op=op, mask=rng.choice(("band", "random", "global") if op == "attention" else ("band", "random")), V=V,
                    heads=heads, seq=seq, d=rng.choice((32, 64, 64, 128)))
        if case["mask"] == "random":
            case["sparsity"] = rng.choice((0.9, 0.95, 0.98))
            while case["heads"] * _nnz_vec(case) * 2 * case["d"] > MOST_GATHER:
                case["heads"] //= 2
        else:
            case.update(half_width=_log(rng, 16, 256), stride=rng.choice((0, 64, 128)))
            if case["mask"] == "global":
                case["tokens"] = rng.choice((16, 32, 64))
        return case
    m, n = max(1, _log(rng, 64, 4096) // V) * V, _log(rng, 64, 4608)
    case = dict(op=op, V=V, m=m, n=n, k=0, sparsity=sparsity, rows=rng.choice(("uniform", "binomial", "binomial")),
                kernel=rng.choice(("wmma", "wmma", "cuda")), out=rng.choice(("f16", "f16", "f32")))
    if op == "sddmm":
        case["k"] = rng.choice((32, 64, 64, 128, 256, _some_width(rng, 16, 512)))
    elif op == "train":
        case["k"] = _log(rng, 4, 64) * 8
        del case["kernel"]
    else:
        case["k"] = _some_width(rng, 32, 2048)
        case["entry"] = rng.choice(("operator", "problem", "problem", "auto"))
        if case["entry"] == "auto":
            case.update(rows=rng.choice(("binomial", "pareto")), kernel="wmma", out="f16")
    while _nnz_vec(case) * case["k"] * (2 if op == "train" else 1) > MOST_GATHER:
        case["k"] = max(8, case["k"] // 2)
    return case


# --------------------------------------------------------------------------- patterns

def _pattern(rng, n, lengths, V):
    """Distinct, sorted columns, uniform over the row."""
    offsets = np.zeros(len(lengths) + 1, dtype=np.int32)
    offsets[1:] = np.cumsum(lengths)
    cols = np.empty(int(offsets[-1]), dtype=np.int32)
    for i, length in enumerate(lengths):
        cols[offsets[i]:offsets[i + 1]] = np.sort(rng.choice(n, int(length), replace=False))
    return cv.ColVecCSR(len(lengths), n, V, offsets, cols)


def _pareto_lengths(rng, m_vec, n, sparsity):
    """Row lengths of a Pareto distribution with about the asked mean, the longest row dense."""
    lengths = (rng.pareto(1.5, m_vec) + 0.3) * n * (1.0 - sparsity) / 1.9
    lengths = np.minimum(lengths, n).astype(np.int64)
    lengths[int(rng.integers(m_vec))] = n
    return lengths


def _binomial_lengths(rng, m_vec, n, sparsity):
    """Binomial row lengths, the same total for every seed: a budget of nonzeros, spread at random."""
    lengths = rng.binomial(n, 1.0 - sparsity, size=m_vec)
    left = int(m_vec * n * (1.0 - sparsity)) - int(lengths.sum())
    while left:
        some = rng.choice(m_vec, min(abs(left), m_vec), replace=False)
        moved = np.clip(lengths[some] + (1 if left > 0 else -1), 0, n)
        left -= int((moved - lengths[some]).sum())
        lengths[some] = moved
    return lengths


def _band_columns(i, case):
    centre = i * case["V"] + case["V"] // 2
    lo, hi = max(0, centre - case["half_width"]), min(case["seq"] - 1, centre + case["half_width"])
    return lo, hi


def _attention_mask(case, seed):
    V, seq = case["V"], case["seq"]
    m_vec = seq // V
    rng = np.random.default_rng(seed)
    if case["mask"] == "random":
        return _pattern(rng, seq, _binomial_lengths(rng, m_vec, seq, case["sparsity"]), V)
    always = np.zeros(seq, dtype=bool)
    if case["stride"]:
        always[case["stride"] - 1::case["stride"]] = True
    tokens = case.get("tokens", 0)
    if tokens:  # tokens that attend to everything and that everybody attends to: whole vector rows, anywhere
        start = int(rng.integers(m_vec - tokens // V + 1)) * V
        always[start:start + tokens] = True
    rows = []
    for i in range(m_vec):
        keep = always.copy()
        if tokens and start <= i * V < start + tokens:
            keep[:] = True
        lo, hi = _band_columns(i, case)
        keep[lo:hi + 1] = True
        rows.append(np.flatnonzero(keep).astype(np.int32))
    offsets = np.zeros(m_vec + 1, dtype=np.int32)
    offsets[1:] = np.cumsum([len(r) for r in rows])
    return cv.ColVecCSR(m_vec, seq, V, offsets, np.concatenate(rows))


def _matrix_pattern(case, seed):
    m_vec, n, V = case["m"] // case["V"], case["n"], case["V"]
    if case["rows"] == "uniform":
        return cv.uniform_pattern(m_vec, n, case["sparsity"], seed, V)
    rng = np.random.default_rng(seed)
    lengths = _pareto_lengths if case["rows"] == "pareto" else _binomial_lengths
    return _pattern(rng, n, lengths(rng, m_vec, n, case["sparsity"]), V)


def _nnz_vec(case):
    """Nonzero vectors of a case's pattern, expected over seeds."""
    V = case["V"]
    if "seq" not in case:
        return int(case["m"] // V * case["n"] * (1.0 - case["sparsity"]))
    m_vec, seq = case["seq"] // V, case["seq"]
    if case["mask"] == "random":
        return int(m_vec * seq * (1.0 - case["sparsity"]))
    always = (seq // case["stride"] if case["stride"] else 0) + case.get("tokens", 0)
    band = sum(hi - lo + 1 for lo, hi in (_band_columns(i, case) for i in range(m_vec)))
    sparse_rows = m_vec - case.get("tokens", 0) // V
    return int(band * sparse_rows / m_vec + sparse_rows * always * (1 - band / (m_vec * seq)) + (m_vec - sparse_rows) * seq)


# --------------------------------------------------------------------------- one pass

def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(generator=gen)

    state = dict(case)
    dtype = torch.float32 if case.get("out") == "f32" else torch.float16
    if case["op"] in ("attention", "chain"):
        layer = ops.SparseAttention(_attention_mask(case, seed))
        shape = (case["heads"], case["seq"], case["d"])
        state.update(layer=layer, q=normal(*shape), key=normal(*shape), v=normal(*shape))
        if case["op"] == "attention":
            layer.plan(case["d"], case["d"], case["heads"])     # a fixed mask is analysed once
        return state
    pat = cv.random_values(_matrix_pattern(case, seed), seed)
    prob = ops.DeviceProblem(pat, sort=case["rows"] == "pareto")
    m, n, k = case["m"], case["n"], case["k"]
    state["prob"] = prob
    if case["op"] == "spmm":
        state.update(rhs=normal(n, k), c=torch.empty((m, k), dtype=dtype, device="cuda"))
    elif case["op"] == "sddmm":
        state.update(lhs=normal(m, k), rhs=normal(n, k), d=torch.empty((prob.nnz_vec, case["V"]), dtype=dtype, device="cuda"))
    else:
        state.update(x=normal(n, k), dy=normal(m, k) * 0.125, y=torch.empty((m, k), dtype=torch.float16, device="cuda"),
                     dw=torch.empty((prob.nnz_vec, case["V"]), dtype=dtype, device="cuda"))
    return state


def run(state):
    op = state["op"]
    if op == "attention":
        return state["layer"].forward(state["q"], state["key"], state["v"])
    if op == "chain":
        layer = state["layer"]
        probabilities = torch.empty((state["heads"], layer.prob.nnz_vec, layer.prob.vec_length), dtype=torch.float16, device="cuda")
        out = layer.forward(state["q"], state["key"], state["v"], fused=False, scores=probabilities)
        return out, probabilities
    prob = state["prob"]
    if op == "sddmm":
        return prob.sddmm(state["lhs"], state["rhs"], kernel=state["kernel"], out_dtype=state["d"].dtype, out=state["d"])
    if op == "train":
        y = prob.spmm(state["x"], out=state["y"])
        dw = prob.sddmm(state["dy"], state["x"], out_dtype=state["dw"].dtype, out=state["dw"])
        return y, dw
    if state["entry"] == "operator":
        call = ops.spmm.wmmaSpmm if state["kernel"] == "wmma" else ops.spmm.cudaSpmm
        return call(prob.m_vec, prob.vec_length, state["k"], prob.n, prob.row_indices, prob.row_offsets, prob.column_indices,
                    prob.values, state["rhs"], state["c"])
    return prob.spmm(state["rhs"], kernel=state["kernel"], out_dtype=state["c"].dtype, out=state["c"],
                     split_rows=None if state["entry"] == "auto" else False)


def work(case):
    """Each input read once, each output written once; two operations per nonzero and dense column."""
    V, nnz_vec = case["V"], _nnz_vec(case)
    if case["op"] in ("attention", "chain"):
        heads, seq, d = case["heads"], case["seq"], case["d"]
        pattern = 4 * nnz_vec + 8 * (seq // V)
        kept = 2 * heads * nnz_vec * V if case["op"] == "chain" else 0
        return {"bytes": pattern + 4 * 2 * heads * seq * d + kept, "flops": 4 * heads * nnz_vec * V * d}
    m, n, k = case["m"], case["n"], case["k"]
    pattern, out = 4 * nnz_vec + 8 * (m // V), 4 if case["out"] == "f32" else 2
    flops = 2 * nnz_vec * V * k
    if case["op"] == "spmm":
        return {"bytes": pattern + 2 * nnz_vec * V + 2 * n * k + out * m * k, "flops": flops}
    if case["op"] == "sddmm":
        return {"bytes": pattern + 2 * m * k + 2 * n * k + out * nnz_vec * V, "flops": flops}
    return {"bytes": pattern + 2 * nnz_vec * V + 2 * n * k + 4 * m * k + out * nnz_vec * V, "flops": 2 * flops}


def tolerance(case):
    # Measured against the same passes in 64 bits on the same inputs, times four: a result rounded to fp16 is off by
    # 2.1e-4 (largest 4.9e-4), an fp32 one by 5e-8 to 1.5e-7 (1.1e-6), an attention layer, which keeps scores or
    # probabilities in fp16 on the way, by 2.7e-4 to 5.4e-4 (6.9e-3).
    if case["op"] in ("attention", "chain"):
        return {"rel": 2.2e-3, "max": 2.8e-2}
    if case["op"] == "train" or case["out"] == "f16":
        return {"rel": 8.4e-4, "max": 2e-3}
    return {"rel": 6e-7, "max": 4.4e-6}
