// stk_approx.hip -- kernels of the approximate (top-c per 128-latent group)
// variant that materialise the per-group candidates, for callers that ask for
// the candidate buffer (streamtopk_approx.cu:264-274 side effect).
//
//   group_kernel : TileStream (W streamed once, MFMA scores for 256 latents =
//                  two groups x up to 128 rows per tile); per 32-row block the
//                  scores go to LDS as order-preserving words, then each
//                  16-lane row of a wave sorts one (row, group)'s 128 keys in
//                  registers (bitonic network, one-direction form: 8 keys per
//                  lane, lane exchanges by DPP; 32-bit keys, with a 64-bit pass where truncated
//                  scores tie) and writes the group's top-c, descending, padded
//                  with (-FLT_MAX, -1) past the end of F
//                  (streamtopk_approx.cu:42-167).
//   cand_kernel  : per row, top-k over all group candidates -- the final
//                  torch.topk + gather of the reference (ops.py:80-81), on the
//                  device.  Only the groups whose head reaches a lower bound of
//                  the row's k-th largest candidate are read past their head.
#include "stk_group.h"

namespace stk {

size_t group_lds_bytes(int dt, int NB)
{
    const size_t xs = dt == DT_F32 ? kXSplitStride : kXRowStride;
    const size_t rings = 2 * (size_t)kGroupTile * kXRowStride + 2 * 32 * (size_t)NB * xs;
    return rings + 2 * kGroupTile * sizeof(float) + 32 * (size_t)NB * kHeadSlots * sizeof(uint64_t);
}

template <int DT, int NB, int C>
__global__ __launch_bounds__(kMainThreads, 1) void group_kernel(GroupArgs a)
{
    group_tiles<DT, NB, C, true>(a);
}

struct GroupKernel {
    template <int DT, int NB, int C>
    static auto kernel() { return group_kernel<DT, NB, C>; }
};

// Key of group g's head (its largest candidate), 0 for a padded group.
// Group g's head key from the compact heads (0 past the last group): one
// 8-byte word per group instead of a value and an index c entries apart.
__device__ __forceinline__ uint64_t head_key(const uint64_t* hd, int64_t g, int64_t G)
{
    const uint64_t h = hd[g < G ? g : G - 1];
    return g < G ? h : 0ull;
}

// Per row: top-k over the (value, index) candidates of every group.  Each
// group's candidates are in descending order, so the row's top k lie among
// the first k of every group, and a group whose head is below a key that k
// candidates reach holds none of them.  The heads' k-th largest maximum over
// the threads is such a key.
__global__ __launch_bounds__(kThreads) void cand_kernel(CandArgs a)
{
    __shared__ SelShared S;
    constexpr int U = 8;   // groups per thread whose heads are loaded together
    const int tid = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int k = a.k, c = a.c;
    const int64_t G = a.num_groups;
    const float* cv = a.cand_vals + row * G * c;
    const int32_t* ci = a.cand_idxs + row * G * c;
    const uint64_t* hd = a.heads + row * G;

    uint64_t m = 0;
    for (int64_t g0 = tid; g0 < G; g0 += U * kThreads) {
        uint64_t hk[U];
#pragma unroll
        for (int u = 0; u < U; ++u) hk[u] = head_key(hd, g0 + u * kThreads, G);
#pragma unroll
        for (int u = 0; u < U; ++u) m = hk[u] > m ? hk[u] : m;
    }
    const uint64_t T = kth_of_maxima(S, m, k, tid);   // >= 1; k candidates are >= T
    if (tid == 0) { S.cnt = 0; S.thr = T - 1; }
    __syncthreads();

    const int kk = k < c ? k : c;
    int64_t g0 = tid;
    int u0 = 0, e0 = 0;   // resume point after a full buffer
    uint32_t vpar = 0;    // block_any's call parity
    for (;;) {
        const uint64_t thr = S.thr;
        bool stalled = false;
        for (; g0 < G; g0 += U * kThreads, u0 = 0, e0 = 0) {
            uint64_t hk[U];
#pragma unroll
            for (int u = 0; u < U; ++u) hk[u] = head_key(hd, g0 + u * kThreads, G);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (stalled || u < u0 || hk[u] <= thr) continue;
                const int64_t base = (g0 + u * kThreads) * c;
                for (int e = (u == u0 ? e0 : 0); e < kk; ++e) {
                    const int32_t idx = ci[base + e];
                    if (idx < 0) break;
                    const uint64_t key = make_key(cv[base + e], idx);
                    if (key <= thr) break;
                    const int pos = atomicAdd(&S.cnt, 1);
                    if (pos >= kSelCap) {
                        stalled = true;
                        u0 = u;
                        e0 = e;
                        break;
                    }
                    S.buf[pos] = key;
                }
            }
            if (stalled) break;
        }
        __syncthreads();
        if (S.cnt >= kSelCap) select_compact(S, kSelCap, k, tid);
        if (!block_any<kThreads / 64>(stalled, S.vote, vpar, tid >> 6, tid & 63)) break;
    }
    const int n = S.cnt < kSelCap ? S.cnt : kSelCap;
    if (n > k) select_compact(S, n, k, tid);
    __syncthreads();
    const int mk = n < k ? n : k;
    if (tid < mk) {
        const uint64_t key = S.buf[tid];
        const int r = rank_desc<false>(S, mk, key, tid);
        a.V[row * k + r] = key_value(key);
        a.I[row * k + r] = key_index(key);
    }
}

hipError_t launch_group(int dt, int NB, const GroupArgs& a, dim3 grid, hipStream_t st)
{
    if (!nontemporal_w(a.W, a.d * (dt == DT_F32 ? 4 : 2), grid.y)) return launch_group_cached(dt, NB, a, grid, st);
    return launch_group_any<GroupKernel>(dt, NB, a, grid, st);
}

hipError_t launch_cand(const CandArgs& a, int64_t rows, hipStream_t st)
{
    launch(cand_kernel, dim3((unsigned)rows), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

}  // namespace stk
