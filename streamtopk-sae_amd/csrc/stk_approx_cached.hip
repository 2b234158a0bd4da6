// stk_approx_cached.hip -- group_kernel with cached loads of W, for several row
// blocks and for rows that are no whole 128-byte lines (nontemporal_w).
#include "stk_group.h"

namespace stk {

template <int DT, int NB, int C>
__global__ __launch_bounds__(kMainThreads, 1) void group_cached_kernel(GroupArgs a)
{
    group_tiles<DT, NB, C, false>(a);
}

struct GroupCachedKernel {
    template <int DT, int NB, int C>
    static auto kernel() { return group_cached_kernel<DT, NB, C>; }
};

hipError_t launch_group_cached(int dt, int NB, const GroupArgs& a, dim3 grid, hipStream_t st)
{
    return launch_group_any<GroupCachedKernel>(dt, NB, a, grid, st);
}

}  // namespace stk
