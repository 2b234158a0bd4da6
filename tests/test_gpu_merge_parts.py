"""merge_topk_shards of a list of parts, merged where they lie: against the
same parts stacked, and against a sort of all entries, for parts in
descending order and in any order, repeated and equal entries, NaN and
infinities, one part, and counts on either side of the in-place limits."""
import ctypes

import pytest
import torch

from streamtopk_sae import _lib, merge_topk_shards

pytestmark = pytest.mark.gpu


def _parts(B, k, n, dev, seed, ordered):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    v = torch.randn(n, B, k, device=dev, generator=g)
    v = (v * 8).round() / 8 + 0.0 if seed % 2 else v      # many equal values, no negative zero
    i = torch.argsort(torch.rand(B, n * k, device=dev, generator=g), dim=1).to(torch.int32)
    i = i.view(B, n, k).permute(1, 0, 2).contiguous()
    if ordered:   # value descending, then index ascending
        i, o = torch.sort(i, dim=2)
        v = torch.gather(v, 2, o)
        v, o = torch.sort(v, dim=2, descending=True, stable=True)
        i = torch.gather(i, 2, o)
    return v, i


def _want(v, i, k):
    n, B, _ = v.shape
    fv = v.permute(1, 0, 2).reshape(B, -1)
    fi = i.permute(1, 0, 2).reshape(B, -1)
    fi, o = torch.sort(fi, dim=1)
    fv = torch.gather(fv, 1, o)
    key = torch.where(fv.isnan(), torch.full_like(fv, float("inf")), fv).double() + fv.isnan().double() * 1e300
    o = torch.sort(key, dim=1, descending=True, stable=True).indices[:, :k]
    return torch.gather(fv, 1, o), torch.gather(fi, 1, o)


@pytest.mark.parametrize("ordered", [True, False])
@pytest.mark.parametrize("B,k,n", [(1, 1, 1), (3, 1, 16), (5, 2, 3), (40, 64, 4), (33, 128, 2), (7, 128, 8), (9, 128, 16),
                                   (2, 128, 32), (6, 128, 33), (1000, 16, 7)])
def test_parts(cuda_dev, B, k, n, ordered):
    for seed in (80, 81):
        print(f"case parts B={B} k={k} n={n} ordered={ordered} seed={seed}", flush=True)
        v, i = _parts(B, k, n, cuda_dev, seed, ordered)
        V, I = merge_topk_shards(list(v), list(i), k)     # (n > 16: stacked inside)
        Vs, Is = merge_topk_shards(v, i, k)
        Vw, Iw = _want(v, i, k)
        assert torch.equal(V, Vs) and torch.equal(I, Is)
        assert torch.equal(V, Vw) and torch.equal(I, Iw)


def test_parts_special_values(cuda_dev):
    print("case parts special values", flush=True)
    B, k, n = 4, 16, 3
    v, i = _parts(B, k, n, cuda_dev, 82, True)
    v[0, 1, 0] = float("inf")
    v[1, 2, :3] = float("nan")
    v[2, 3, :] = -float("inf")
    v[1, 0, 8:] = -3.4028234e38
    V, I = merge_topk_shards(list(v), list(i), k)
    Vw, Iw = _want(v, i, k)
    assert torch.equal(I, Iw) and torch.equal(V.nan_to_num(nan=7e37), Vw.nan_to_num(nan=7e37))
    # the same part twice: every entry comes out twice
    v, i = _parts(B, k, 1, cuda_dev, 84, True)
    V, I = merge_topk_shards([v[0], v[0]], [i[0], i[0]], k)
    assert torch.equal(V, v[0][:, :k // 2].repeat_interleave(2, dim=1))
    assert torch.equal(I, i[0][:, :k // 2].repeat_interleave(2, dim=1))


def test_parts_refusals(cuda_dev):
    v, i = _parts(4, 16, 3, cuda_dev, 86, True)
    with pytest.raises(RuntimeError):
        merge_topk_shards([v[0], v[1][:, :8]], [i[0], i[1][:, :8]], 16)
    with pytest.raises(RuntimeError):
        merge_topk_shards(list(v.double()), list(i), 16)
    with pytest.raises(RuntimeError):
        merge_topk_shards(list(v), list(i), 8)
    # parts that are no contiguous tensors are taken all the same
    V, I = merge_topk_shards([p.T.contiguous().T for p in v], list(i), 16)
    Vs, Is = merge_topk_shards(v, i, 16)
    assert torch.equal(V, Vs) and torch.equal(I, Is)
    lib = _lib.load()
    ptr = (ctypes.c_void_p * 17)(*[v.data_ptr()] * 17)
    assert lib.stk_topk_merge_parts(ptr, ptr, 17, 4, 16, v.data_ptr(), i.data_ptr(), None) == 1
    assert "at most 16 parts" in lib.stk_last_error().decode()
    assert lib.stk_topk_merge_parts(None, None, 2, 4, 16, v.data_ptr(), i.data_ptr(), None) == 1
