"""Cases of the streaming top-k encoder that its speed is measured on.

Every case is one call of a public op of `streamtopk_sae` on inputs that are
resident on the GPU: X (B, d) activations, W_enc (F, d) and b_enc (F,) of the
encoder, values and indices of each row's k largest scores out.

  exact   topk_sae_cuda_exact(X, W_enc, b_enc, k)
  approx  topk_sae_cuda_approx(X, W_enc, b_enc, k, c)
  cand    topk_sae_cuda_approx(..., candidate_buffer=): each 128-latent group's
          top c come back too
  merge   merge_topk_shards(values, indices, k): the last step of an encoder
          whose latents are split over `parts` GPUs

The inputs are those of streamtopk_sae.make_inputs (unit-norm encoder rows,
normal activations); the shards' results are sorted rows of normal scores.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "streamtopk-sae_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from streamtopk_sae import make_inputs, merge_topk_shards, topk_sae_cuda_approx, topk_sae_cuda_exact  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
_GROUP = 128

# The most one call may do: the largest listed case's multiply-adds (fp32 runs
# at a sixteenth of the 16-bit matrix rate) and encoder bytes.
_MAX_FLOPS = {"bf16": 2.2e12, "fp16": 2.2e12, "fp32": 1.375e11}
_MAX_W_BYTES = 4.3e9
_MAX_CAND = 3.4e7


def _case(name, op, dtype, B, d, F, k, c=0):
    return {"name": name, "op": op, "dtype": dtype, "B": B, "d": d, "F": F, "k": k, "c": c}


def listed():
    return [
        # one token of a served model, the smallest dictionary of the grids: launches and host work
        _case("token", "exact", "bf16", 1, 768, 16384, 32),
        # a few sequences' tokens on a wide model with a small dictionary
        _case("small_batch", "exact", "bf16", 32, 4096, 16384, 16),
        # an ordinary inference batch on a small model
        _case("batch_d768", "exact", "bf16", 128, 768, 65536, 32),
        # the headline: an inference batch on a large dictionary
        _case("headline", "exact", "bf16", 128, 2048, 262144, 64),
        # sizes that are no multiple of any tile, between an inference and a training batch
        _case("ragged_fp16", "exact", "fp16", 200, 1000, 100003, 64),
        # the headline's sizes with fp32 activations and weights
        _case("headline_fp32", "exact", "fp32", 128, 2048, 262144, 64),
        # feature extraction over a data set: a batch of 512 tokens
        _case("batch_512", "exact", "bf16", 512, 2048, 65536, 32),
        # an encoder's training batch in fp32
        _case("train_fp32", "exact", "fp32", 1024, 768, 65536, 32),
        # the largest batch on the widest model: compute-bound
        _case("train_wide", "exact", "bf16", 1024, 4096, 262144, 128),
        # per-group candidates of a small batch
        _case("candidates_small", "cand", "bf16", 32, 768, 65536, 16, 16),
        # per-group candidates of the largest dictionary
        _case("candidates", "cand", "bf16", 128, 2048, 1048576, 32, 32),
        # eight GPUs' shard results for a training batch
        {"name": "merge_shards", "op": "merge", "B": 1024, "k": 128, "parts": 8},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    op = rng.choice(["exact"] * 6 + ["approx", "cand", "cand", "merge"])
    if op == "merge":
        return {"op": op, "B": int(_log(rng, 1, 2048)), "k": rng.choice([8, 16, 32, 64, 128]),
                "parts": rng.randint(2, 8)}
    while True:
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        B = int(_log(rng, 1, 2049))
        d = 8 * int(_log(rng, 128, 4103) / 8)
        F = int(_log(rng, 4096, 1048577))
        k = rng.choice([16, 32, 32, 64, 64, 128])
        c = 0
        if op != "exact":
            c = rng.choice([x for x in (16, 32, 64, 128) if x >= k])
        if op == "cand":
            # a last group of at least c latents: no padding among the candidates
            F = -(-F // _GROUP) * _GROUP - rng.randint(0, _GROUP - c)
        if (2.0 * B * d * F <= _MAX_FLOPS[dtype] and F * d * _SIZE[dtype] <= _MAX_W_BYTES
                and (op != "cand" or B * -(-F // _GROUP) * c <= _MAX_CAND)):
            return {"op": op, "dtype": dtype, "B": B, "d": d, "F": F, "k": k, "c": c}


def _shard_parts(case, seed):
    """Each part's k largest scores of B rows, sorted, with global latent indices."""
    B, k, n = case["B"], case["k"], case["parts"]
    per = 32768   # latents of a shard
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    values, indices = [], []
    for p in range(n):
        # k of a shard's latents beat a threshold near the top of a normal sample
        v = 2.5 + 0.35 * torch.empty(B, k, device="cuda").exponential_(1.0, generator=g)
        values.append(torch.sort(v, dim=1, descending=True).values.contiguous())
        i = torch.argsort(torch.rand(B, 4 * k, device="cuda", generator=g), dim=1)[:, :k]
        indices.append((i * (per // (4 * k)) + p * per).to(torch.int32).contiguous())
    return values, indices


def prepare(case, seed):
    if case["op"] == "merge":
        values, indices = _shard_parts(case, seed)
        return {"case": case, "values": values, "indices": indices}
    X, W, b = make_inputs(case["B"], case["d"], case["F"], _DTYPES[case["dtype"]], seed=seed, device="cuda")
    state = {"case": case, "X": X, "W": W, "b": b}
    if case["op"] == "cand":
        state["candidates"] = torch.empty((case["B"], -(-case["F"] // _GROUP), case["c"]), dtype=torch.float32,
                                          device="cuda")
    return state


def run(state):
    case = state["case"]
    op, k = case["op"], case["k"]
    if op == "merge":
        return merge_topk_shards(state["values"], state["indices"], k)
    if op == "exact":
        return topk_sae_cuda_exact(state["X"], state["W"], state["b"], k)
    if op == "approx":
        return topk_sae_cuda_approx(state["X"], state["W"], state["b"], k, case["c"])
    V, I = topk_sae_cuda_approx(state["X"], state["W"], state["b"], k, case["c"],
                                candidate_buffer=state["candidates"])
    return V, I, state["candidates"]


def work(case):
    B, k = case["B"], case["k"]
    if case["op"] == "merge":
        n = case["parts"] * B * k
        return {"bytes": 8 * n + 8 * B * k, "flops": n}
    d, F, s = case["d"], case["F"], _SIZE[case["dtype"]]
    nbytes = B * d * s + F * d * s + 4 * F + 8 * B * k
    if case["op"] == "cand":
        nbytes += 4 * B * -(-F // _GROUP) * case["c"]
    return {"bytes": nbytes, "flops": 2 * B * d * F}


def tolerance(case):
    # scores are fp32 sums of exact (16-bit inputs) or rounded (fp32) products.
    # Measured against 64-bit sums over the listed cases: values 1.3e-7 .. 3.3e-7
    # (16-bit) and 3.9e-7 .. 6.4e-7 (fp32) off, single ones up to 2.8e-6; where
    # the k-th scores lie close (k = 128), 4e-4 of the indices change places.
    if case["op"] == "merge":
        return "exact"
    if case["dtype"] == "fp32":
        return {"rel": 2.5e-6, "max": 1.2e-5, "differ": 2e-3}
    return {"rel": 1.3e-6, "max": 1.2e-5, "differ": 2e-3}


def _exact_topk(v, i, k):
    top = torch.topk(v, k, dim=1)
    return top.values, torch.gather(i, 1, top.indices).to(torch.int32)


def exact(case, seed):
    state = prepare(case, seed)
    k = case["k"]
    if case["op"] == "merge":
        v = torch.cat(state["values"], dim=1).double()
        return _exact_topk(v, torch.cat(state["indices"], dim=1).long(), k)
    X, W, b = state["X"].double(), state["W"], state["b"].double()
    B, F, c = case["B"], case["F"], case["c"]
    cand = case["op"] == "cand"
    vals, idxs, groups = [], [], []
    step = 65536   # a whole number of groups
    for f0 in range(0, F, step):
        f1 = min(F, f0 + step)
        s = X @ W[f0:f1].double().T + b[f0:f1]
        top = torch.topk(s, min(k, f1 - f0), dim=1)
        vals.append(top.values)
        idxs.append(top.indices + f0)
        if cand:
            pad = -(f1 - f0) % _GROUP
            s = torch.nn.functional.pad(s, (0, pad), value=-math.inf).view(B, -1, _GROUP)
            groups.append(torch.topk(s, c, dim=2).values)
    V, I = _exact_topk(torch.cat(vals, dim=1), torch.cat(idxs, dim=1), k)
    return (V, I, torch.cat(groups, dim=1)) if cand else (V, I)
