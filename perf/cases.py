"""The work that programs have this framework do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" says which part of the framework it calls:

  spmm          one product with a Tiled-CSL weight (column-major, row-major or strided operands)
  split         one product with a weight split into 2:4 records and a residual (one launch, or two kernels)
  stack         one token step through chained decoder layers
  encode        a dense weight in device memory -> Tiled-CSL
  split_weight  a dense weight in device memory -> 2:4 records + residual lists
  host_encode   a dense weight in host memory -> Tiled-CSL, in host memory

Weights are N(0, 0.02) fp16 with random kept entries (uniform, or Beta(2, 8) densities per row),
activations N(0, 1) fp16: the distributions of the benchmark's configurations.
"""
import math

import torch

import graphneuralnetproj_amd as G
from graphneuralnetproj_amd import decoder_stack

TOKENS = (8, 16, 32, 64)  # what the kernels take


def listed():
    return [
        # The smallest product of the benchmark's configurations: a call is little more than its launch.
        dict(name="spmm_smallest", kind="spmm", M=1024, K=1024, N=8, sparsity=0.8, skewed=False, layout="column"),
        # A weight of odd size, eleven by ninety-one tiles, very sparse and with uneven rows, on row-major operands.
        dict(name="spmm_ragged_skewed", kind="spmm", M=1408, K=5824, N=32, sparsity=0.9, skewed=True, layout="row"),
        # Attention output projection (OPT-30B) while decoding: an ordinary product that fills the chip for a moment.
        dict(name="spmm_attention_out", kind="spmm", M=7168, K=7168, N=16, sparsity=0.8, skewed=False, layout="column"),
        # First feed-forward product (OPT-30B) at 16 tokens: the benchmark's headline.
        dict(name="spmm_ffn1", kind="spmm", M=28672, K=7168, N=16, sparsity=0.8, skewed=False, layout="column"),
        # Second feed-forward product: few rows, long sums, a denser weight and a batch of 32.
        dict(name="spmm_ffn2_batch32", kind="spmm", M=7168, K=28672, N=32, sparsity=0.7, skewed=False, layout="column"),
        # The largest: OPT-175B's first feed-forward product at the largest batch.
        dict(name="spmm_largest_batch64", kind="spmm", M=49152, K=12288, N=64, sparsity=0.8, skewed=False, layout="column"),
        # The same kind of product from 2:4 records and a residual, for a weight too dense for Tiled-CSL to pay.
        dict(name="split_ffn1", kind="split", M=28672, K=7168, N=16, sparsity=0.6, skewed=False, layout="column",
             form="one_launch"),
        # ... and at 64 tokens and 50 %, on this fork's row-major operands (OPT-66B attention projection).
        dict(name="split_qkv_batch64", kind="split", M=27648, K=9216, N=64, sparsity=0.5, skewed=False, layout="row",
             form="one_launch"),
        # Decoding one token step: eight chained products of two decoder layers, with strides and the fused clamp.
        dict(name="stack_decode", kind="stack", hidden=7168, layers=2, N=16, sparsity=0.8),
        # A model being loaded: a pruned weight that is on the GPU becomes Tiled-CSL ...
        dict(name="encode_ffn1", kind="encode", M=28672, K=7168, sparsity=0.8, skewed=False),
        # ... or records and residual lists;
        dict(name="split_weight_qkv", kind="split_weight", M=21504, K=7168, sparsity=0.6, skewed=False),
        # and a converter's program, which encodes in host memory.
        dict(name="host_encode", kind="host_encode", M=7168, K=7168, sparsity=0.8, skewed=False),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _shape(rng, most, step_k, most_rows=384, most_cols=49152):
    """M (a multiple of 128) and K (of step_k), each spread over its logarithm, with M * K <= most."""
    while True:
        M = 128 * max(1, round(_log_uniform(rng, 1, most_rows)))
        K = step_k * max(1, round(_log_uniform(rng, 256 / step_k, most_cols / step_k)))
        if M * K <= most:
            return M, K


def draw(rng):
    kind = rng.choices(("spmm", "split", "stack", "encode", "split_weight", "host_encode"), (10, 4, 1, 2, 2, 1))[0]
    skewed = rng.random() < 0.25
    if kind == "spmm":
        M, K = _shape(rng, 49152 * 12288, 64)
        return dict(kind=kind, M=M, K=K, N=rng.choice(TOKENS), sparsity=round(rng.uniform(0.6, 0.95), 3), skewed=skewed,
                    layout=rng.choice(("column", "column", "row", "strided")))
    if kind == "split":
        M, K = _shape(rng, 27648 * 9216, 128)
        form = rng.choice(("one_launch", "one_launch", "one_launch", "two_kernels"))
        return dict(kind=kind, M=M, K=K, N=rng.choice(TOKENS), sparsity=round(rng.uniform(0.5, 0.7), 3), skewed=False,
                    layout=rng.choice(("column", "row", "strided") if form == "one_launch" else ("column", "row")), form=form)
    if kind == "stack":
        return dict(kind=kind, hidden=128 * round(_log_uniform(rng, 4, 56)), layers=rng.choice((1, 2)), N=rng.choice(TOKENS[:3]),
                    sparsity=round(rng.uniform(0.7, 0.9), 3))
    M, K = _shape(rng, {"encode": 28672 * 7168, "split_weight": 21504 * 7168, "host_encode": 7168 * 7168}[kind],
                  128 if kind == "split_weight" else 64)
    sparsity = rng.uniform(0.5, 0.7) if kind == "split_weight" else rng.uniform(0.6, 0.95)
    return dict(kind=kind, M=M, K=K, sparsity=round(sparsity, 3), skewed=skewed and kind != "split_weight")


def _weight(M, K, sparsity, skewed, gen):
    """A pruned fp16 weight on the GPU.

    Values are drawn from `gen`. Which elements are kept is a random pattern of the shape with its tile rows, and
    the rows within them, permuted by `gen`: the packed size of a weight is the same for every seed.
    """
    dev = gen.device
    mask = torch.Generator(device=dev)
    mask.manual_seed(M * 65536 + K)
    keep = torch.full((M, 1), 1.0 - sparsity, device=dev)
    if skewed:  # Beta(2, 8) per row, from ten exponentials, scaled to the wanted mean
        e = -torch.log1p(-torch.rand((M, 10), generator=mask, device=dev))
        keep = ((e[:, :2].sum(1) / e.sum(1)) * ((1.0 - sparsity) / 0.2)).clamp_(max=1.0).unsqueeze(1)
    W = torch.empty((M, K), dtype=torch.float16, device=dev)
    step = max(128, (1 << 26) // K)
    for r in range(0, M, step):
        part = W[r:r + step]
        w = torch.randn(part.shape, generator=gen, device=dev).mul_(0.02)
        w = torch.where(w < 0, w - 1e-6, w + 1e-6)  # a kept value is never zero in fp16
        w.mul_(torch.rand(part.shape, generator=mask, device=dev) < keep[r:r + step])
        part.copy_(w)
    rows = torch.randperm(M // 128, generator=gen, device=dev)[:, None] * 128 + torch.randperm(128, generator=gen, device=dev)
    return W[rows.reshape(-1)]


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    kind = case["kind"]
    st = dict(case, stream=torch.cuda.current_stream())
    if kind == "stack":
        h, N = case["hidden"], case["N"]
        layers = [decoder_stack.build_layer_on_device(G, torch, dev, h, N, case["sparsity"], seed * 64 + i)[0]
                  for i in range(case["layers"])]
        st["stack"] = decoder_stack.Stack(G, torch, layers, h, N)
        st["x"] = torch.randn((N, h), generator=gen, device=dev).half()
        return st
    M, K = case["M"], case["K"]
    W = _weight(M, K, case["sparsity"], case["skewed"], gen)
    if kind == "host_encode":
        st["W"] = W.cpu().numpy()
        return st
    if kind in ("encode", "split_weight"):
        st["W"] = W
        return st
    N, layout = case["N"], case["layout"]
    slabs = 0
    if kind == "spmm":
        st["items"], st["offsets"] = G.encode_on_device(W)
        st["split"] = slabs = G.SpMM_SuggestSplitK_Bytes(M, N, K, st["items"].numel() // 4)
    else:
        st["records"], residual = G.split_pack_on_device(W)
        st["split"] = slabs = G.HeteroSparse_SuggestSplitK(M, N, K)
        if case["form"] == "one_launch":
            st["words"], st["lists"], st["longest"] = G.pack_residual_on_device(residual)
        else:
            st["items"], st["offsets"] = G.encode_on_device(residual)
            st["split2"] = G.SpMM_SuggestSplitK_Bytes(M, N, K, st["items"].numel() // 4)
            slabs += st["split2"]
    st["workspace"] = torch.empty(slabs * N * M, dtype=torch.float16, device=dev)
    if layout == "row":
        st["B"] = torch.randn((K, N), generator=gen, device=dev).half()
        st["C"] = torch.zeros((M, N), dtype=torch.float16, device=dev)
    else:  # strided: the first third of a fused buffer, as the attention output projection reads it
        st["ldb"] = 3 * K if layout == "strided" else K
        st["B"] = torch.randn((N, st["ldb"]), generator=gen, device=dev).half()
        st["C"] = torch.zeros((N, M), dtype=torch.float16, device=dev)
    return st


def run(st):
    kind = st["kind"]
    if kind == "stack":
        stack = st["stack"]
        stack.x[0].copy_(st["x"])
        return stack.step(st["stream"])
    if kind == "encode":
        return G.encode_on_device(st["W"])
    if kind == "split_weight":
        records, residual = G.split_pack_on_device(st["W"])
        return (records, residual) + G.pack_residual_on_device(residual)
    if kind == "host_encode":
        return G.InitSparseMatrixA_API(st["W"])
    M, N, K, B, C, ws, s, stream, layout = (st["M"], st["N"], st["K"], st["B"], st["C"], st["workspace"], st["split"],
                                            st["stream"], st["layout"])
    if kind == "spmm":
        if layout == "column":
            G.SpMM_SplitK_API(stream, None, st["items"], st["offsets"], B, C, M, N, K, ws, s)
        elif layout == "row":
            G.SpMM_SplitK_API_RowMajor(stream, None, st["items"], st["offsets"], B, C, M, N, K, ws, s)
        else:
            G.SpMM_SplitK_API_Strided(stream, st["items"], st["offsets"], B, st["ldb"], C, M, M, N, K, ws, s, G.SPMM_FLAG_RELU)
    elif st["form"] == "two_kernels":
        call = G.HeteroSparse_SpMM_API_RowMajor if layout == "row" else G.HeteroSparse_SpMM_API
        call(stream, st["records"], st["items"], st["offsets"], B, C, M, N, K, ws, s, st["split2"])
    elif layout == "column":
        G.HeteroSparse_Fused_SpMM_API(stream, st["records"], st["words"], st["lists"], st["longest"], B, C, M, N, K, ws, s)
    elif layout == "row":
        G.HeteroSparse_Fused_SpMM_API_RowMajor(stream, st["records"], st["words"], st["lists"], st["longest"], B, C, M, N, K, ws, s)
    else:
        G.HeteroSparse_Fused_SpMM_API_Strided(stream, st["records"], st["words"], st["lists"], st["longest"], B, st["ldb"], C, M,
                                              M, N, K, ws, s, G.SPMM_FLAG_RELU)
    return C


def exact(case, seed):
    """The product (or the chain of products) of the same inputs in 64 bits, by plain torch; None where whole values come out."""
    kind = case["kind"]
    if kind in ("encode", "split_weight", "host_encode"):
        return None
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    if kind == "stack":  # the layers' weights as decoder_stack draws them
        h, N = case["hidden"], case["N"]
        x = torch.randn((N, h), generator=gen, device=dev).half().double()
        for i in range(case["layers"]):
            g = torch.Generator(device=dev)
            g.manual_seed(seed * 64 + i)
            for M, K, clamp in ((3 * h, h, False), (h, h, False), (4 * h, h, True), (h, 4 * h, False)):
                W = torch.randn((M, K), generator=g, device=dev).mul_(0.02)
                W = W.mul_(torch.rand((M, K), generator=g, device=dev) >= case["sparsity"]).half().double()
                x = x[:, :K] @ W.t()
                if clamp:
                    x = x.relu()
        return x
    M, N, K, layout = case["M"], case["N"], case["K"], case["layout"]
    W = _weight(M, K, case["sparsity"], case["skewed"], gen).double()
    if layout == "row":
        return W @ torch.randn((K, N), generator=gen, device=dev).half().double()
    B = torch.randn((N, 3 * K if layout == "strided" else K), generator=gen, device=dev).half()[:, :K].double()
    C = B @ W.t()
    return C.relu() if layout == "strided" else C


def _csl_bytes(M, K, kept):
    tiles = (M // 128) * (K // 64)
    return 4.0 * M * K * kept + 6.0 * tiles + 4.0 * (tiles + 2)  # words, a tile's padding of 1.5 words, offsets


def _residual_share(kept):
    """Share of a weight's elements that a 2:4 part cannot hold: the third and fourth kept one of every four."""
    return (4 * kept ** 3 * (1 - kept) + 2 * kept ** 4) / 4


def work(case):
    kept = 1.0 - case["sparsity"]
    if case["kind"] == "stack":
        h, N = case["hidden"], case["N"]
        total = {"bytes": 0.0, "flops": 0.0}
        for M, K in decoder_stack.layer_shapes(h).values():
            total["bytes"] += case["layers"] * (_csl_bytes(M, K, kept) + 2.0 * N * (M + K))
            total["flops"] += case["layers"] * 2.0 * M * K * kept * N
        return total
    M, K = case["M"], case["K"]
    if case["kind"] in ("encode", "host_encode"):
        return {"bytes": 2.0 * M * K + _csl_bytes(M, K, kept), "flops": 0.0}
    split_bytes = 1.125 * M * K + 4.0 * M * K * _residual_share(kept) + 4.0 * (M // 16) * (K // 128)
    if case["kind"] == "split_weight":  # the dense residual is one of the outputs
        return {"bytes": 2.0 * M * K + 2.0 * M * K + split_bytes, "flops": 0.0}
    N = case["N"]
    weight = _csl_bytes(M, K, kept) if case["kind"] == "spmm" else split_bytes
    return {"bytes": weight + 2.0 * N * (M + K), "flops": 2.0 * M * K * kept * N}


def tolerance(case):
    if case["kind"] in ("encode", "split_weight", "host_encode"):
        return "exact"
    # Against the same product in 64 bits: rel 2.1e-4 (one rounding to fp16) to 3.1e-4 (slabs of partial sums in fp16
    # as well), max 5e-4 to 1.8e-3; a chain of eight 0.8e-3 to 1.4e-3, max 5.1e-3. Four times that.
    if case["kind"] == "stack":
        return {"rel": 5e-3, "max": 2e-2}
    return {"rel": 1.2e-3, "max": 7e-3}
