"""main_kernel's split of d over its waves (tiles of 128 or 64 latents, two or
four 128-byte sub-steps per step), its balanced ranges of latents and its
rotated columns, where they can go wrong: one step more or less than a whole
number of them, a partial last sub-step, a last tile of a few latents, several
row blocks, dictionaries with as few maxima as k, rows that are a multiple of
4 KiB, and rows that are no whole 128-byte lines.  Every value is held to the
error bound of an fp32 sum of its terms (parity.fp32_sum_bound)."""
import pytest
import torch

import oracle
from hooks import hooks
from parity import check_against_scores, term_magnitudes, tol_of
from streamtopk_sae import _lib, make_inputs, topk_sae_cuda_exact

pytestmark = pytest.mark.gpu

DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def _check(X, W, b, k, dtype_name, name):
    V, I = topk_sae_cuda_exact(X, W, b, k)
    torch.cuda.synchronize()
    Xn, Wn, bn = (t.float().cpu().numpy() for t in (X, W, b))
    check_against_scores(V.cpu().numpy(), I.cpu().numpy(), oracle.scores_f64(Xn, Wn, bn), k, tol_of(dtype_name), name,
                         A=term_magnitudes(Xn, Wn, bn), d=X.shape[1])
    return V, I


@pytest.mark.parametrize("B,d,F,k,dtype_name", [
    (1, 768, 16384, 32, "bf16"),      # four sub-steps, three whole steps
    (31, 776, 16384 + 5, 32, "fp16"),  # 13 sub-steps: the last step holds one, partial
    (32, 4096, 4096, 128, "bf16"),    # rotated columns; 128 maxima = k
    (33, 1000, 8197, 64, "bf16"),     # two row blocks or two sub-steps, a partial last one
    (64, 384, 20000, 64, "bf16"),     # six sub-steps: the fewest that split
    (64, 376, 20000, 64, "fp16"),     # five whole sub-steps and a partial one
    (65, 2048, 5000, 16, "bf16"),     # row blocks of which the last holds one row
    (128, 520, 8192, 128, "fp16"),
    (200, 2040, 4999, 64, "bf16"),    # every row of W starts elsewhere in its line
    (300, 2048, 70001, 32, "bf16"),   # whole 256-latent tiles, the last of a range partial
    (128, 1024, 256 * 256 + 16, 32, "fp16"),   # ranges of 256 and 272 latents
    (64, 404, 4100, 128, "fp32"),     # 13 sub-steps of fp32, the last partial
    (5, 1024, 9000, 8, "fp32"),       # rotated columns in fp32
    (2, 2048, 600, 16, "bf16"),       # fewer workgroups than an exchange needs
])
def test_split_shapes(cuda_dev, B, d, F, k, dtype_name):
    print(f"case split B={B} d={d} F={F} k={k} {dtype_name}", flush=True)
    X, W, b = make_inputs(B, d, F, DT[dtype_name], seed=61, device=cuda_dev)
    V, I = _check(X, W, b, k, dtype_name, "split")
    # without exchanged thresholds every score is a candidate: the same result
    # from the queues' spills and the segments' compactions
    with hooks(xch_wait=-1):
        V0, I0 = topk_sae_cuda_exact(X, W, b, k)
    assert torch.equal(V, V0) and torch.equal(I, I0)


@pytest.mark.parametrize("offset", [8, 64])
def test_split_unaligned_base(cuda_dev, offset):
    """W from a view that starts inside a 128-byte line (16-byte aligned)."""
    B, d, F, k = 40, 512, 9000, 32
    print(f"case split base offset {offset}", flush=True)
    X, W, b = make_inputs(B, d, F, torch.bfloat16, seed=62, device=cuda_dev)
    flat = torch.empty(F * d + offset, dtype=torch.bfloat16, device=cuda_dev)
    Wv = flat[offset:].view(F, d)
    Wv.copy_(W)
    V, I = _check(X, Wv, b, k, "bf16", "unaligned base")
    V1, I1 = topk_sae_cuda_exact(X, W, b, k)
    assert torch.equal(V, V1) and torch.equal(I, I1)


def test_split_ignores_values_past_its_rows(cuda_dev):
    """NaN and infinity in the latents after a partial last sub-step's row, in
    a neighbouring workgroup's range and in another row of X change no other
    score."""
    B, d, F, k = 8, 904, 8192, 16   # 14.1 sub-steps
    print("case split NaN neighbours", flush=True)
    X, W, b = make_inputs(B, d, F, torch.bfloat16, seed=63, device=cuda_dev)
    keep = torch.ones(F, dtype=torch.bool, device=cuda_dev)
    bad = torch.arange(3, F, 97, device=cuda_dev)
    keep[bad] = False
    W2, X2, b2 = W.clone(), X.clone(), b.clone()
    W2[bad] = float("nan")
    W2[bad[::2], 0] = float("inf")
    b2[bad] = -float("inf")
    X2[5] = float("inf")
    b2[keep] = b[keep]
    V, I = topk_sae_cuda_exact(X2, W2, b2, k)
    torch.cuda.synchronize()
    # rows other than 5: NaN scores rank first (as torch.topk ranks them)
    S = X2.double().nan_to_num(posinf=0.0).cpu() @ W.double().T.cpu() + b.double().cpu()
    rows = [r for r in range(B) if r != 5]
    assert torch.isnan(V[rows]).all()
    assert not keep[I[rows].long()].any()
    V1, I1 = topk_sae_cuda_exact(X2, W, b, k)   # row 5 alone is not finite
    for r in rows:
        want = torch.topk(S[r], k).indices
        assert set(I1[r].tolist()) == set(want.tolist())


@pytest.mark.parametrize("B,d,F,k,dtype_name", [
    (300, 256, 65536, 32, "bf16"),    # the large-batch kernel, within the static scratch
    (400, 64, 262144, 128, "bf16"),   # its workspace would not fit: the other kernel runs
    (257, 72, 33000, 16, "bf16"),     # 129 tiles
    (511, 4096, 33000, 64, "bf16"),   # rotated columns of the large-batch kernel
    (1886, 3656, 18787, 32, "fp32"),  # the streaming kernel's workspace would not fit: the large-batch one runs
])
def test_middle_batches(cuda_dev, B, d, F, k, dtype_name):
    """Batches of 257 rows and more, through the op and without allocation."""
    print(f"case middle {dtype_name} B={B} d={d} F={F} k={k}", flush=True)
    X, W, b = make_inputs(B, d, F, DT[dtype_name], seed=64, device=cuda_dev)
    V, I = topk_sae_cuda_exact(X, W, b, k)
    Vn, In = torch.empty_like(V), torch.empty_like(I)
    lib = _lib.load()
    code = {"bf16": _lib.STK_DTYPE_BF16, "fp32": _lib.STK_DTYPE_F32}[dtype_name]
    _lib.check(lib.stk_exact_forward_noalloc(X.data_ptr(), W.data_ptr(), b.data_ptr(), Vn.data_ptr(), In.data_ptr(),
                                             B, d, F, k, code, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    S = (X.double() @ W.double().T + b.double()).cpu().numpy()
    A = term_magnitudes(X, W, b)
    for v, i, name in ((V, I, "middle"), (Vn, In, "middle noalloc")):
        check_against_scores(v.cpu().numpy(), i.cpu().numpy(), S, k, tol_of(dtype_name), name, A=A, d=d)
