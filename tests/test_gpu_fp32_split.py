"""fp32 inputs on the bf16 matrix cores (three bf16 parts per value, six of the
nine products): every score within the error bound of an fp32 sum of its terms
(parity.fp32_sum_bound), also where one product dominates the sum, and inputs
that the parts do not hold -- infinities, NaN, values next to the largest
float, values near the smallest -- give what an fp32 sum gives."""
import numpy as np
import pytest
import torch

import oracle
from parity import check_against_scores, term_magnitudes
from streamtopk_sae import make_inputs, topk_sae_cuda_approx, topk_sae_cuda_exact

pytestmark = pytest.mark.gpu


def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.parametrize("B,d,F,k", [
    (1, 32, 300, 1),          # one d-step
    (33, 1028, 9001, 64),     # partial last step, two row blocks
    (128, 4096, 8192, 128),   # the longest sum, four row blocks
    (600, 256, 20000, 64),    # a large batch
    (2100, 64, 6000, 16),     # past the batches of main_kernel: the fp32 matrix cores
])
def test_fp32_split_values(cuda_dev, B, d, F, k):
    print(f"case fp32 split B={B} d={d} F={F} k={k}", flush=True)
    X, W, b = make_inputs(B, d, F, torch.float32, seed=71, device=cuda_dev)
    X[:, 0] *= 1e4            # one product dominates: its low parts must be there
    W[:, 0] = W[:, 0].abs() + 1.0
    V, I = topk_sae_cuda_exact(X, W, b, k)
    torch.cuda.synchronize()
    S = oracle.scores_f64(_np(X), _np(W), _np(b))
    check_against_scores(V.cpu().numpy(), I.cpu().numpy(), S, k, 1e-5, "fp32 split", A=term_magnitudes(_np(X), _np(W), _np(b)),
                         d=d)


@pytest.mark.parametrize("case", ["inf", "nan", "largest", "tiny", "bias"])
@pytest.mark.parametrize("B,d,F", [(5, 96, 700), (70, 768, 9000)])   # without and with the split of d
def test_fp32_split_extremes(cuda_dev, case, B, d, F):
    print(f"case fp32 extremes {case} B={B} d={d} F={F}", flush=True)
    k = 16
    X, W, b = make_inputs(B, d, F, torch.float32, seed=72, device=cuda_dev)
    if case == "inf":
        W[::50, 3] = float("inf")
    elif case == "nan":
        W[::50, 3] = float("nan")
    elif case == "largest":
        W[::50, 3] = 3.4e38          # rounds past bf16's largest value
        X[:, 3] = X[:, 3].clamp(-1.0, 1.0) * 0.5
    elif case == "tiny":
        X *= 2.0 ** -118             # the lower parts are bf16 denormals
        b.zero_()
    elif case == "bias":
        b[::3] = -float("inf")
        b[1] = float("inf")
        X[0] = 0.0
    # the same sums in 64 bits, infinities and NaN as fp32 gives them (no sum
    # here leaves fp32's range but by an infinite term)
    S = X.double() @ W.double().T + b.double()
    V, I = topk_sae_cuda_exact(X, W, b, k)
    nt = (F + 127) // 128
    cb = torch.empty((B, nt, 16), dtype=torch.float32, device=cuda_dev)
    Vc, Ic = topk_sae_cuda_approx(X, W, b, k, 16, candidate_buffer=cb)
    torch.cuda.synchronize()
    order = torch.where(S.isnan(), torch.full_like(S, float("inf")), S)
    top = torch.topk(order, k, dim=1).values.cpu().numpy()
    A = (X.double().abs() @ W.double().abs().T).amax().item() if case == "tiny" else None
    for Vx, Ix in ((V, I), (Vc, Ic)):
        got = torch.gather(S, 1, Ix.long()).cpu().numpy()
        v = Vx.double().cpu().numpy()
        assert np.array_equal(np.isnan(v), np.isnan(got))
        assert np.array_equal(np.isinf(v), np.isinf(got))
        fin = np.isfinite(v)
        scale = A if A is not None else np.maximum(np.abs(got), 1.0)
        gk = np.where(np.isnan(got), np.inf, got)
        with np.errstate(invalid="ignore"):
            assert np.all((np.abs(v - got) / scale)[fin] <= 1e-5)
            assert np.all((gk == top) | (np.abs(gk - top) <= 2e-5 * (A if A is not None else np.maximum(np.abs(top), 1.0))))
