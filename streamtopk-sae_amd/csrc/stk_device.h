// stk_device.h -- device-side building blocks for the streaming top-k encoder
// on gfx950 (CDNA4): sort keys, the MFMA quad step, the score main loop
// (TileStream: W and X staged in LDS, 8 waves, used by main_kernel and
// group_kernel) and queue compaction helpers.
//
// Score layout.  Each wavefront owns blocks of 32 latents (W rows, the MFMA
// "A" operand) and NB blocks of 32 batch rows (X rows, the MFMA "B" operand),
// and accumulates the fp32 scores W_blk . X_blk^T with
// v_mfma_f32_32x32x{16 bf16|16 f16|2 f32}.
//
// Permuted reduction axis.  One "d-step" covers 128 bytes of every W row
// (64 bf16/fp16 or 32 fp32 elements).  Lane l holds row (l % 32) of its block
// and the contiguous half h = l / 32 of the d-step: 64 bytes, fetched as four
// 16-byte loads ("quads").  The MFMA's reduction index k is paired with the
// physical d index through the same (lane-half, quad, element) map for both
// operands, so every product W[f,d]*X[j,d] is formed exactly once; only the
// order of the fp32 sum differs from a plain left-to-right dot product.
//
// Accumulator layout of v_mfma_f32_32x32x*: register r of lane l holds row
// 8*(r/4) + 4*(l/32) + (r%4), column l % 32 (every GPU parity test depends on
// it: a wrong map scores the wrong latent).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace stk {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));

enum { DT_F32 = 0, DT_F16 = 1, DT_BF16 = 2 };

constexpr int kWaves = 4;            // wavefronts per workgroup
constexpr int kThreads = 64 * kWaves;
constexpr int kStepBytes = 128;      // bytes of one W/X row per d-step
constexpr int kXRowStride = 144;     // LDS bytes per staged X row (128 + 16 pad)
constexpr int kXSplitStride = 208;   // the same for fp32 X, as bf16 parts (3 * 64 + 16 pad)

template <int DT> struct Dt;
template <> struct Dt<DT_BF16> { static constexpr int esize = 2; static constexpr int DS = 64; };
template <> struct Dt<DT_F16>  { static constexpr int esize = 2; static constexpr int DS = 64; };
template <> struct Dt<DT_F32>  { static constexpr int esize = 4; static constexpr int DS = 32; };

// ---------------------------------------------------------------------------
// 64-bit sort keys.  High word: order-preserving image of the fp32 score
// (NaN canonicalised above +inf, as torch.topk ranks NaN first).  Low word:
// 0xFFFFFFFF - latent index, so among equal scores the lower index ranks
// higher.  Key 0 never occurs for a real entry.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t ordered_u32(float v)
{
    uint32_t u = __float_as_uint(v);
    uint32_t r = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return (v != v) ? 0xFFFFFFFFu : r;
}

__device__ __forceinline__ float key_value(uint64_t key)
{
    uint32_t r = (uint32_t)(key >> 32);
    uint32_t u = (r & 0x80000000u) ? (r & 0x7FFFFFFFu) : ~r;
    return __uint_as_float(u);
}

__device__ __forceinline__ int32_t key_index(uint64_t key)
{
    return (int32_t)(0xFFFFFFFFu - (uint32_t)key);
}

__device__ __forceinline__ uint64_t make_key(float v, int64_t idx)
{
    return ((uint64_t)ordered_u32(v) << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)idx);
}

// ---------------------------------------------------------------------------
// Threshold exchange helpers (main_kernel, mainl_kernel).  Every word the
// workgroups of one call share carries the call's tag (the workspace's epoch
// + 1, never 0) in its high half and its data in the low half, and is
// written and read whole with agent-scope atomic stores and loads (coherent
// across the XCDs' L2s word by word).  A reader polls the words it needs
// until enough carry the call's tag: no flag has to be ordered after the
// data, so no writer waits for its stores, and the last poll returns the
// data.  Words of earlier calls carry other tags; a workspace starts
// zero-filled, and tag 0 is never used.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void xch_put(uint64_t* p, uint32_t tag, uint32_t data)
{
    __hip_atomic_store(p, ((uint64_t)tag << 32) | data, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wave-level: polls n <= 64 * U words p[0..n) (U per lane) until at least
// `need` of them carry `tag`, for at most `wait` ticks of the 100 MHz
// real-time counter; v[u] receives the low half of word lane + 64 u if it
// carries the tag, else 0.  Returns how many of the n words carry the tag in
// the last poll (>= need unless the wait ran out; the same in every lane).
// wait == 0: one poll; wait < 0: none (every v[u] 0, returns 0).
template <int U>
__device__ __forceinline__ int xch_poll(const uint64_t* p, int n, int need, uint32_t tag, int64_t wait, int lane,
                                        uint32_t (&v)[U])
{
    if (wait < 0) {
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = 0u;
        return 0;
    }
    const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    for (;;) {
        int got = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = lane + 64 * u;
            bool tagged = false;
            v[u] = 0u;
            if (i < n) {
                const uint64_t w = __hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                tagged = (uint32_t)(w >> 32) == tag;
                v[u] = tagged ? (uint32_t)w : 0u;
            }
            got += __popcll(__ballot(tagged));
        }
        if (got >= need || (int64_t)(__builtin_amdgcn_s_memrealtime() - t0) >= wait) return got;
        __builtin_amdgcn_s_sleep(1);
    }
}

// Wave-level: a lower bound T of the k-th largest of the wave's non-zero
// values v (at least k of them), T <= T*, the exact k-th largest.  T* lies in
// [lo, hi], the smallest and largest non-zero values, so it shares their
// common leading bits; below those T is built bit by bit (the largest T with
// at least k values >= T) over 12 bits, the rest left 0: at most 2^-11 of a
// score image below T*.  The same in every lane.
template <int U>
__device__ __forceinline__ uint32_t xch_kth(const uint32_t (&v)[U], int k)
{
    uint32_t lo = ~0u, hi = 0u;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        lo = (v[u] != 0u && v[u] < lo) ? v[u] : lo;
        hi = v[u] > hi ? v[u] : hi;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t l2 = __shfl_xor(lo, off), h2 = __shfl_xor(hi, off);
        lo = l2 < lo ? l2 : lo;
        hi = h2 > hi ? h2 : hi;
    }
    const uint32_t diff = lo ^ hi;
    if (diff == 0u) return hi;
    const int top = 31 - __builtin_clz(diff);
    uint32_t T = hi & ~((2u << top) - 1u);   // the common leading bits (2u << 31 wraps to 0: none)
    const int stop = top >= 11 ? top - 11 : 0;
    for (int bit = top; bit >= stop; --bit) {
        const uint32_t c = T | (1u << bit);
        int cnt = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) cnt += __popcll(__ballot(v[u] >= c));
        T = cnt >= k ? c : T;
    }
    return T;
}

// Partial sums stored in a workspace keep no denormal (a positive one's bits
// could pass for an exchange tag in a word's high half): they are stored as
// zero, a change below any fp32 score's rounding once the bias is added.
__device__ __forceinline__ f32x4 flush_denorm4(f32x4 v)
{
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = __builtin_fabsf(v[e]) < 1.17549435e-38f ? 0.f : v[e];
    return v;
}

// The threshold key of score image T: the largest key below every key of
// that score (0, accept everything, for T = 0).
__device__ __forceinline__ uint64_t xch_key(uint32_t T)
{
    return T ? ((uint64_t)T << 32) - 1 : 0ull;
}

// Buffer resource (raw, gfx9 family): loads at byte offsets >= num_records
// return zeros, which bounds rows past B and latents past F, and a zero-length
// resource makes whole steps read as zeros.  The lane's
// offset is what the compiler documents as checked; gfx950 checks its sum with
// the scalar one, without wrapping (seen in both kinds of load, for scalar
// offsets below, at and past num_records).
// The streaming kernels build every resource uniform over the wave; its fields
// go through readfirstlane so that the compiler keeps it in scalar registers
// whatever its uniformity analysis concludes (a resource it takes for
// divergent costs a waterfall loop around every load).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, int64_t num_records)
{
    const uint64_t b = (uint64_t)base;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    const int n = __builtin_amdgcn_readfirstlane((int)num_records);
    return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), (short)0, n, 0x00020000);
}

// LDS loads (global -> LDS, no registers): lane i of one instruction writes
// the 16 bytes at ldsbase + 16*i.
__device__ __forceinline__ void lds_load16(__amdgpu_buffer_rsrc_t r, unsigned char* ldsbase, int voff, int soff)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)ldsbase, 16, voff, soff, 0, 0);
}

// ---------------------------------------------------------------------------
// Workgroup-wide OR of p.  Every thread of the workgroup calls it, the same
// number of times.  HIP's __syncthreads_or reads the workgroup size from the
// kernel's implicit arguments, and where registers are short the compiler
// reloads it at every call (a scalar memory load and its wait).  Here lane 0
// of each wave stores whether any lane of the wave has p into the wave's
// slot, one barrier, and every lane reads all slots.  The slots alternate
// between two sets from call to call (parity, a per-thread call counter), so a
// wave's store for the next call cannot meet a slower wave's read of this one:
// the next call's barrier lies between them.  vote: 2 * WAVES words of LDS,
// 16-byte aligned.
// ---------------------------------------------------------------------------
template <int WAVES>
__device__ __forceinline__ bool block_any(bool p, uint32_t* vote, uint32_t& parity, int wave, int lane)
{
    uint32_t* v = vote + (parity & 1u) * WAVES;
    ++parity;
    const bool wp = __ballot(p) != 0;
    if (lane == 0) v[wave] = wp ? 1u : 0u;
    __syncthreads();
    if constexpr (WAVES % 4 == 0) {
        u32x4 acc = *(const u32x4*)v;
#pragma unroll
        for (int w = 4; w < WAVES; w += 4) acc |= *(const u32x4*)(v + w);
        return (acc[0] | acc[1] | acc[2] | acc[3]) != 0u;
    } else {
        uint32_t acc = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) acc |= v[w];
        return acc != 0u;
    }
}

// Ring layout: row r's 16-byte chunk c sits in slot c ^ ((r >> 1) & 7) of the
// row's 128 bytes, so that the MFMA-layout reads (32 rows x one chunk per
// half-wave) hit 16 distinct 16-byte bank groups.
__device__ __forceinline__ int xswz(int r) { return (r >> 1) & 7; }

// ---------------------------------------------------------------------------
// One quad (16 bytes of W for this lane x 16 bytes of X) through the MFMA.
// ---------------------------------------------------------------------------
template <int DT>
__device__ __forceinline__ void mfma_quad(f32x16& acc, u32x4 a, u32x4 b);

template <>
__device__ __forceinline__ void mfma_quad<DT_BF16>(f32x16& acc, u32x4 a, u32x4 b)
{
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                  __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

template <>
__device__ __forceinline__ void mfma_quad<DT_F16>(f32x16& acc, u32x4 a, u32x4 b)
{
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                 __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
}

template <>
__device__ __forceinline__ void mfma_quad<DT_F32>(f32x16& acc, u32x4 a, u32x4 b)
{
#pragma unroll
    for (int e = 0; e < 4; ++e)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[e]), __uint_as_float(b[e]), acc, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// fp32 operands on the bf16 matrix cores.  A finite fp32 value is the sum of
// three bf16 values, v = v1 + v2 + v3: each is the rest so far rounded to
// nearest (8 significant bits, and the remainders are exact), so 24 bits are
// covered.  Of the nine products of two split values the six of weight 2^-16
// and more are formed (v1 w1, v1 w2, v2 w1, v1 w3, v2 w2, v3 w1), each exact
// in fp32 and accumulated in fp32; the three left out are below 2^-24 of
// v w each.  Six v_mfma_f32_32x32x16_bf16 take 192 cycles for what eight
// v_mfma_f32_32x32x2_f32 take 512.  The splits exist for normal, finite
// values: TileStream::fix_up recomputes scores that may have met others.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t pk_bf16(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// The three bf16 parts of a and b, packed (a in the low halves).
__device__ __forceinline__ void split3(float a, float b, uint32_t (&p)[3])
{
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        p[i] = pk_bf16(a, b);
        a -= __uint_as_float(p[i] << 16);
        b -= __uint_as_float(p[i] & 0xFFFF0000u);
    }
}

// ---------------------------------------------------------------------------
// Compacts the queue segments (in global memory) of this wave's rows that are
// full to their top-k: rows wave*R .. wave*R + R - 1 (R <= 64), segment of
// row r at qrow(r), cap keys; cnt and thr in LDS.  Segment keys are read
// through L2 (agent-scope atomic loads): other waves' plain stores are
// complete (fence + barrier before the call) but the reading CU's L1 may hold
// lines of an earlier compaction.  scr: cap keys of LDS for this wave.
// ---------------------------------------------------------------------------
template <int R, class RowSeg>
__device__ __forceinline__ void compact_full_rows(int* cnt, uint64_t* thr, uint64_t* scr, RowSeg qrow,
                                                  int cap, int k, int wave, int lane)
{
    const int myrow = wave * R + (lane < R ? lane : 0);
    uint64_t full = __ballot(lane < R && cnt[myrow] >= cap);
    while (full) {
        const int i = __builtin_ctzll(full);
        full &= full - 1;
        const int row = wave * R + i;
        auto* q = qrow(row);
        uint64_t e[3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const int idx = lane + 64 * m;
            e[m] = (idx < cap) ? __hip_atomic_load(q + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
            if (idx < cap) scr[idx] = e[m];
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        int rk[3] = {0, 0, 0};
        for (int ii = 0; ii < cap; ii += 2) {
            const u64x2 v = *(const u64x2*)(scr + ii);
#pragma unroll
            for (int m = 0; m < 3; ++m) rk[m] += (int)(v[0] > e[m]) + (int)(v[1] > e[m]);
        }
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            if (lane + 64 * m < cap && rk[m] < k) {
                q[rk[m]] = e[m];
                if (rk[m] == k - 1) thr[row] = e[m];
            }
        }
        if (lane == 0) cnt[row] = k;
        __builtin_amdgcn_wave_barrier();
    }
}

// Rank-compacts the n keys q[0..n) (k < n <= cap <= 192, distinct, written
// by this wave or read back through L2) to their k largest, in q[0..k), and
// returns the k-th largest.  One wave; scr is cap keys of LDS scratch.
__device__ __forceinline__ uint64_t compact_row(uint64_t* q, int n, uint64_t* scr, int cap, int k, int lane)
{
    uint64_t e[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const int idx = lane + 64 * m;
        e[m] = (idx < n) ? __hip_atomic_load(q + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        if (idx < cap) scr[idx] = e[m];
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    // ranks among the n keys (the zero padding up to n rounded to even ranks below every key)
    int rk[3] = {0, 0, 0};
    for (int ii = 0; ii < n; ii += 2) {
        const u64x2 v = *(const u64x2*)(scr + ii);
#pragma unroll
        for (int m = 0; m < 3; ++m) rk[m] += (int)(v[0] > e[m]) + (int)(v[1] > e[m]);
    }
    uint64_t kth = 0;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        if (lane + 64 * m < n && rk[m] < k) {
            q[rk[m]] = e[m];
            if (rk[m] == k - 1) kth = e[m];
        }
    }
    // exactly one lane holds the k-th key
    const uint64_t hit = __ballot(kth != 0);
    const int src = __builtin_ctzll(hit);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)kth, src);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(kth >> 32), src);
    __builtin_amdgcn_wave_barrier();
    return ((uint64_t)hi << 32) | lo;
}

// ---------------------------------------------------------------------------
// TileStream: the score main loop with both operands staged in LDS.  A tile
// is 32*WAVES/S latents x 32*NB rows; a step covers S 128-byte sub-steps of d.
// A tile takes nds2 steps: the nds real ones rounded up to even (a padding
// step reads zeros).
//   Split (S): the waves form S groups of WAVES / S; group q scores the tile's
//      latents over sub-step q of every step, and the groups' partial sums are
//      added in order before the epilogue (reduce).  Every step reads the same
//      32 KiB of W whatever S, so S divides the steps of a tile and multiplies
//      the tiles: a dictionary with fewer 256-latent tiles than CUs then
//      spreads over more of them.  bf16, B = 32, d = 4096, F = 16384 (64 tiles
//      of 64 steps, against 256 of 16): main_kernel 59.3 -> 31.3 us.
//   W: each step's kTileF rows x S*128 bytes are read with whole-line loads
//      (NT: nontemporal, see nontemporal_w), 8 S lanes per row, two steps
//      ahead in registers, and stored to a two-buffer LDS ring; each wave then
//      reads its 32 rows in the MFMA layout.  Loads straight into the MFMA
//      layout touch 32 rows per instruction, 32 bytes of each line, and stream
//      W at ~6 TB/s; whole-line nontemporal loads reach ~7 TB/s.
//   X: the row block's 32*NB rows of the step, the same way with ordinary
//      loads (every workgroup of the row block re-reads X from L2).
//   Rotation (rot): where a row is a multiple of 4 KiB, step s reads column
//      step (s + 7 x) % nds, x the workgroup's place along W.  All workgroups
//      start together, and at the same column their rows then fall on few
//      memory channels: bf16, B = 1, d = 2048, F = 65536 68.4 us unrotated,
//      47.7 us rotated (5.6 TB/s); F = 131072 124.6 and 85.9 us; at F = 2^18,
//      where the workgroups drift apart, 163 us either way.  At 2 KiB rows it
//      gained nothing.
// The tile's rows of W and the row block's of X are buffer resources, rebuilt
// per tile: rows past the range or past B, and the chunks past d of a partial
// last step (an offset past every resource), read as zeros without a branch
// or a mask, and a thread keeps one offset per operand.  bf16, B = 128,
// d = 1000, F = 65536 (partial last step, rows no whole lines): main_kernel
// 54.5 us with pointers, a branch for the last step and nontemporal loads,
// 42.5 us so.
// One barrier per step.  The loads of the next tile's first steps are in
// flight across the epilogue.
//
// run() calls epi(t, acc, bias) after the last d-step of tile t and then
// resets acc and waits for every outstanding memory operation: the epilogue
// may issue a data-dependent number of global stores, which the compiler
// cannot count, and the wait restores its exact counts for the d-step loop
// (the prefetched loads it includes have had the whole epilogue to land).
// The epilogue may use LDS other than ring buffer 0 (which holds the next
// tile's first step) and the bias buffers.  Ring buffer 1 (W and X) is idle
// during it: its last readers passed the tile's last barrier and its next
// writer runs after the epilogue, so an epilogue that uses it must end with a
// workgroup barrier.  The bias of tile t comes from LDS: wave 0 loads the next
// tile's bias inside the d-step loop and stores it within the same iteration.
// With kBiasInit the accumulators of each tile start at the bias of their
// latents (so acc holds the scores, bias included, when epi runs: the MFMAs
// add the products onto it); otherwise they start at zero and epi receives
// the bias to add.
// ---------------------------------------------------------------------------
template <int DT, int NB, int WAVES, int S, bool NT>
struct TileStream {
    static constexpr int DS = Dt<DT>::DS * S;                      // elements of d per step
    static constexpr int ES = Dt<DT>::esize;
    static constexpr int kThr = 64 * WAVES;
    static constexpr int kLatWaves = WAVES / S;                    // waves across a tile's latents
    static constexpr int kTileF = 32 * kLatWaves;                  // latents per tile
    static constexpr int kRowChunks = 8 * S;                       // 16-byte chunks of a row per step
    static constexpr int kWChunks = kTileF * kRowChunks / kThr;    // 16-byte W chunks per thread per step
    static constexpr int kXTotal = 32 * NB * kRowChunks;           // 16-byte X chunks per step
    static constexpr int kXChunks = (kXTotal + kThr - 1) / kThr;   // per thread
    static constexpr int kWBuf = S * kTileF * kXRowStride;         // bytes of one W ring buffer
    // LDS bytes of one row's sub-step of X: 128, or the three bf16 parts of 32
    // fp32 values, padded so that the MFMA-layout reads meet no bank conflict
    static constexpr bool kSplit = DT == DT_F32;
    static constexpr int kXStride = kSplit ? kXSplitStride : kXRowStride;
    static constexpr int kXBuf = S * 32 * NB * kXStride;           // bytes of one X ring buffer
    static constexpr int kRingBytes = 2 * kWBuf + 2 * kXBuf;
    static_assert(kXTotal % kThr == 0 || kXChunks == 1, "X chunk split");
    static_assert(kTileF * kRowChunks % kThr == 0, "W chunk split");
    static_assert(kThr % kRowChunks == 0, "a thread's chunks share their place in the row");
    static_assert(WAVES % S == 0 && S * NB <= 4, "ring size");
    // the split waves' partial sums (before each epilogue) fit W ring buffer 1
    static constexpr int kRedBytes = (WAVES - kLatWaves) * NB * 4096;
    static_assert(kRedBytes <= kWBuf, "partial sums fit the idle ring buffer");

    static constexpr int kQE = 16 / ES;                            // elements per 16-byte chunk

    const float* bias;
    int64_t F;                   // end of this workgroup's latents
    int64_t f_begin;             // its first latent (tile t starts at f_begin + t * kTileF)
    int ntiles, nds, nds2;
    int tail;                    // elements of d in the last step when it is partial, else 0
    int rot;                     // step s reads the columns of step (s + rot) % nds
    int tid, lane, wave, h, jl;
    const unsigned char* W;
    int64_t w_row_bytes;

    // load cursor (uniform): the tile's rows and the row block as buffer
    // resources (rows past the range or past B lie outside and read as zeros),
    // this thread's offset of its first chunk in each
    int lt, ls;
    __amdgpu_buffer_rsrc_t wres, xres;
    int woff, xoff;
    int toff;                    // added in the partial last step: out of range for a chunk past d

    // d, the row stride and the alignment of W decide the steps, the partial
    // last step, the load kind and the rotation; `x` is the workgroup's place
    // along W.
    __device__ __forceinline__ void init_steps(int64_t d, int x)
    {
        nds = (int)((d + DS - 1) / DS);
        tail = (int)(d % DS);
        nds2 = (nds + 1) / 2 * 2;
        w_row_bytes = d * ES;
        rot = (w_row_bytes & 4095) == 0 ? (int)(((unsigned)x * 7u) % (unsigned)nds) : 0;
    }

    __device__ __forceinline__ int col(int s) const   // column step of step s < nds
    {
        const int c = s + rot;
        return c >= nds ? c - nds : c;
    }

    static constexpr int kOut = 0x40000000;   // an offset beyond every resource (at most 256 rows of kMaxRowBytes)

    __device__ __forceinline__ void init_x(const unsigned char* X, int64_t B, int64_t b0)
    {
        const int64_t nrows = B - b0 < 32 * NB ? B - b0 : 32 * NB;
        xres = make_rsrc(X + b0 * w_row_bytes, nrows * w_row_bytes);
        const int off = tid / kRowChunks * (int)w_row_bytes + tid % kRowChunks * 16;
        woff = off;
        xoff = tid < kXTotal ? off : kOut;
        toff = (tid % kRowChunks) * kQE < tail ? 0 : kOut;
    }

    __device__ __forceinline__ void set_rows(int t)
    {
        const int64_t f0 = f_begin + (int64_t)t * kTileF;
        const int64_t n = F - f0 < kTileF ? F - f0 : kTileF;
        wres = make_rsrc(W + f0 * w_row_bytes, n * w_row_bytes);
    }

    // Loads of the cursor's step (past the last tile: any valid one), in
    // ascending address order; a thread's chunks lie kThr / kRowChunks rows
    // apart and share their place in the row.
    __device__ __forceinline__ void issue(u32x4 (&xr)[kXChunks], u32x4 (&wr)[kWChunks])
    {
        const bool real = lt < ntiles && ls < nds;   // else a padding step: zeros
        const int s = col(real ? ls : 0);
        const int so = __builtin_amdgcn_readfirstlane(s * (S * kStepBytes));
        const int to = !real ? kOut : (tail != 0 && s == nds - 1) ? toff : 0;
        // the chunks' rows go into the lane's offset, which the range check is
        // documented to cover; fp32, whose pipeline has no register left for
        // that (one spilled at 128 rows), into the scalar one, which gfx950
        // counts as well
        const int rows = kThr / kRowChunks * (int)w_row_bytes;
        const int vr = kSplit ? 0 : rows, sr = kSplit ? rows : 0;
#pragma unroll
        for (int p = 0; p < kXChunks; ++p)
            xr[p] = __builtin_amdgcn_raw_buffer_load_b128(xres, xoff + to + p * vr, so + p * sr, 0);
#pragma unroll
        for (int p = 0; p < kWChunks; ++p)
            wr[p] = __builtin_amdgcn_raw_buffer_load_b128(wres, woff + to + p * vr, so + p * sr, NT ? 2 : 0);
        if (lt < ntiles && ++ls == nds2) {
            ls = 0;
            ++lt;
            if (lt < ntiles) set_rows(lt);
        }
    }

    // LDS row of a thread's chunk p in a ring buffer of `rows` rows per
    // 128-byte sub-step
    __device__ __forceinline__ int ring_row(int p, int rows) const
    {
        const int c = tid + kThr * p;
        return ((c % kRowChunks) >> 3) * rows + c / kRowChunks;
    }

    __device__ __forceinline__ void store(const u32x4 (&xr)[kXChunks], const u32x4 (&wr)[kWChunks], unsigned char* xs,
                                          unsigned char* wsb) const
    {
#pragma unroll
        for (int p = 0; p < kWChunks; ++p)
            *(u32x4*)(wsb + ring_row(p, kTileF) * kXRowStride + (tid & 7) * 16) = wr[p];
#pragma unroll
        for (int p = 0; p < kXChunks; ++p) store_x(xr[p], p, xs);
    }

    // A thread's X chunk p to ring buffer xs; fp32 as its three bf16 parts
    // (X is split here, once for all waves).
    __device__ __forceinline__ void store_x(const u32x4& v, int p, unsigned char* xs) const
    {
        if (kXTotal % kThr != 0 && tid >= kXTotal) return;
        unsigned char* q = xs + ring_row(p, 32 * NB) * kXStride;
        if constexpr (kSplit) {
            uint32_t lo[3], hi[3];
            split3(__uint_as_float(v[0]), __uint_as_float(v[1]), lo);
            split3(__uint_as_float(v[2]), __uint_as_float(v[3]), hi);
#pragma unroll
            for (int i = 0; i < 3; ++i) *(u32x2*)(q + i * 64 + (tid & 7) * 8) = u32x2{lo[i], hi[i]};
        } else {
            *(u32x4*)(q + (tid & 7) * 16) = v;
        }
    }

    // compute() of the step in xs / wsb and store() of the loaded chunks to
    // the other buffers.
    __device__ __forceinline__ void compute_store(f32x16 (&acc)[NB], const unsigned char* xs, const unsigned char* wsb,
                                                  const u32x4 (&xr)[kXChunks], const u32x4 (&wr)[kWChunks],
                                                  unsigned char* xn, unsigned char* wn) const
    {
        if constexpr (kSplit) {
            split_step(acc, xs, wsb, xr, wr, xn, wn);
        } else {
            compute(acc, xs, wsb);
            store(xr, wr, xn, wn);
        }
    }

    __device__ __forceinline__ void compute(f32x16 (&acc)[NB], const unsigned char* xs, const unsigned char* wsb) const
    {
        // wave -> sub-step wave / kLatWaves, latents 32 (wave % kLatWaves) ..:
        // its W rows are ring rows 32 wave ..
        const unsigned char* xw = xs + (S > 1 ? wave / kLatWaves * (32 * NB) : 0) * kXStride;
        u32x4 w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = *(const u32x4*)(wsb + (wave * 32 + jl) * kXRowStride + h * 64 + q * 16);
        // two 32-row blocks at a time: two independent accumulation chains
        constexpr int NP = NB < 2 ? NB : 2;
#pragma unroll
        for (int n0 = 0; n0 < NB; n0 += NP) {
            u32x4 bx[NP][4];
#pragma unroll
            for (int n = 0; n < NP; ++n)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    bx[n][q] = *(const u32x4*)(xw + (32 * (n0 + n) + jl) * kXStride + h * 64 + q * 16);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int n = 0; n < NP; ++n) mfma_quad<DT>(acc[n0 + n], w[q], bx[n][q]);
        }
    }

    // fp32: compute() of the step in xs / wsb, and store() of the loaded chunks
    // xr / wr to xn / wn, in one pipeline: 2 NB groups (half g of a lane's
    // values, row block n) of six MFMAs on the three parts of W and of X, the
    // smallest products first.  Each group's X parts are read during the group
    // before, and the splits' VALU work goes between the MFMAs (six fit behind
    // a 32-cycle MFMA): W's second half during the first NB groups, the next
    // step's X during the others.  Left to the compiler, the splits ran in
    // clumps with the MFMAs idle: B = 128, d = 2048, F = 2^18 768 us, 692-729 so
    // (1044-1072 on the fp32 matrix cores).  What bounds it is the MFMAs at the
    // power limit's clock: with two of the six products (timing only) 416 us;
    // splitting by truncation, or one wave of each SIMD storing before its MFMAs
    // and the other after, changed nothing.
    __device__ __forceinline__ void split_step(f32x16 (&acc)[NB], const unsigned char* xs, const unsigned char* wsb,
                                               const u32x4 (&xr)[kXChunks], const u32x4 (&wr)[kWChunks],
                                               unsigned char* xn, unsigned char* wn) const
    {
        const unsigned char* xw = xs + (S > 1 ? wave / kLatWaves * (32 * NB) : 0) * kXStride + jl * kXStride + h * 32;
        const unsigned char* ww = wsb + (wave * 32 + jl) * kXRowStride + h * 64;
        u32x4 w[4], wp[2][3], bx[2][3];
#pragma unroll
        for (int q = 0; q < 4; ++q) w[q] = *(const u32x4*)(ww + q * 16);
        auto read_x = [&](int i) {   // parts of group i
#pragma unroll
            for (int k = 0; k < 3; ++k)
                bx[i & 1][k] = *(const u32x4*)(xw + 32 * (i % NB) * kXStride + k * 64 + (i / NB) * 16);
        };
        auto split_w = [&](int g, int e) {   // elements 2 e, 2 e + 1 of half g
            uint32_t pt[3];
            const u32x4 v = w[2 * g + e / 2];
            split3(__uint_as_float(v[2 * (e & 1)]), __uint_as_float(v[2 * (e & 1) + 1]), pt);
#pragma unroll
            for (int k = 0; k < 3; ++k) wp[g][k][e] = pt[k];
        };
        read_x(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) split_w(0, e);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int pw[6] = {2, 1, 0, 1, 0, 0}, px[6] = {0, 1, 2, 0, 1, 0};
#pragma unroll
        for (int i = 0; i < 2 * NB; ++i) {
            if (i + 1 < 2 * NB) read_x(i + 1);
            if (i < NB) {
#pragma unroll
                for (int e = i * 4 / NB; e < (i + 1) * 4 / NB; ++e) split_w(1, e);
            } else {
                const int j = i - NB;
#pragma unroll
                for (int p = j * kWChunks / NB; p < (j + 1) * kWChunks / NB; ++p)
                    *(u32x4*)(wn + ring_row(p, kTileF) * kXRowStride + (tid & 7) * 16) = wr[p];
#pragma unroll
                for (int p = j * kXChunks / NB; p < (j + 1) * kXChunks / NB; ++p) store_x(xr[p], p, xn);
            }
#pragma unroll
            for (int k = 0; k < 6; ++k) mfma_quad<DT_BF16>(acc[i % NB], wp[i / NB][pw[k]], bx[i & 1][px[k]]);
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // LDS reads
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);   // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    __device__ __forceinline__ void bias_load(float (&bn)[kTileF / 64], int t) const
    {
        const int64_t f0 = f_begin + (int64_t)t * kTileF;
        int64_t n = F - f0;
        n = n < 0 ? 0 : (n < kTileF ? n : kTileF);   // zeros past the range
        const __amdgpu_buffer_rsrc_t r = make_rsrc(bias + f0, n * 4);
#pragma unroll
        for (int e = 0; e < kTileF / 64; ++e)
            bn[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, lane * (kTileF / 64) * 4 + 4 * e, 0, 0));
    }

    __device__ __forceinline__ void bias_store(const float (&bn)[kTileF / 64], float* buf) const
    {
#pragma unroll
        for (int e = 0; e < kTileF / 64; ++e) buf[lane * (kTileF / 64) + e] = bn[e];
    }

    // Bias of this lane's latents: entry r is latent (within the tile)
    // wave*32 + 8*(r/4) + 4*h + r%4.
    __device__ __forceinline__ void bias_read(float (&bv)[16], const float* buf) const
    {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 v = *(const f32x4*)(buf + wave * 32 + g * 8 + h * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[4 * g + e] = v[e];
        }
    }

    __device__ __forceinline__ void acc_reset(f32x16 (&acc)[NB], const float* bias_buf, bool from_bias) const
    {
        if (from_bias && (S == 1 || wave < kLatWaves)) {
            float bv[16];
            bias_read(bv, bias_buf);
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][r] = bv[r];
        } else {
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
        }
    }

    // S > 1: the sub-step waves' partial sums, added in sub-step order to the
    // waves of sub-step 0 through W ring buffer 1 (idle; its next writer runs
    // after a barrier of the epilogue).
    __device__ __forceinline__ void reduce(f32x16 (&acc)[NB], unsigned char* red) const
    {
        if constexpr (S > 1) {
            f32x4* mine = (f32x4*)red + lane;
            if (wave >= kLatWaves) {
#pragma unroll
                for (int n = 0; n < NB; ++n)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        mine[(((wave - kLatWaves) * NB + n) * 4 + g) * 64] =
                            f32x4{acc[n][4 * g], acc[n][4 * g + 1], acc[n][4 * g + 2], acc[n][4 * g + 3]};
            }
            __syncthreads();
            if (wave < kLatWaves) {
#pragma unroll
                for (int q = 0; q < S - 1; ++q)
#pragma unroll
                    for (int n = 0; n < NB; ++n)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const f32x4 v = mine[(((q * kLatWaves + wave) * NB + n) * 4 + g) * 64];
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[n][4 * g + e] += v[e];
                        }
            }
        }
    }

    // fp32 (kSplit): whether score s of a latent with bias b may have met an
    // input that its three bf16 parts do not hold.  An infinite or NaN input,
    // or one that rounds past bf16's largest value, leaves no finite score
    // (one that equals an infinite bias, or whose bias is NaN, is right as it is);
    // inputs so small that their lower parts vanish matter only to a score as
    // small.  Scores of exactly zero are taken as they are.
    static constexpr uint32_t kTiny = 0x17800000u, kInf = 0x7F800000u;   // 2^-80, infinity
    __device__ __forceinline__ static bool suspect(float s, float b)
    {
        const uint32_t u = __float_as_uint(s) & 0x7FFFFFFFu, ub = __float_as_uint(b) & 0x7FFFFFFFu;
        return u != 0u && u - kTiny >= kInf - kTiny && !(u >= kInf && (ub > kInf || s == b));
    }

    // fp32: scores of tile t that are suspect are recomputed, with all others
    // of the wave, by the fp32 MFMA from operands read straight from memory:
    // slow, and reached only by inputs that are not finite, near the largest
    // float or tiny.
    __device__ __forceinline__ void fix_up(f32x16 (&acc)[NB], int t, const float* bias_buf) const
    {
        if constexpr (kSplit) {
            if (S > 1 && wave >= kLatWaves) return;
            uint32_t far = 0;   // a first look that also takes zeros
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t u = (__float_as_uint(acc[n][r]) & 0x7FFFFFFFu) - kTiny;
                    far = u > far ? u : far;
                }
            if (__ballot(far >= kInf - kTiny) == 0) return;
            float bv[16];
            bias_read(bv, bias_buf);
            bool bad = false;
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) bad |= suspect(acc[n][r], bv[r]);
            if (__ballot(bad) == 0) return;
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][r] = bv[r];
            const int64_t f0 = f_begin + (int64_t)t * kTileF;
            const int64_t nr = F - f0 < kTileF ? F - f0 : kTileF;
            const __amdgpu_buffer_rsrc_t wr = make_rsrc(W + f0 * w_row_bytes, nr * w_row_bytes);
            const int nq = (int)(w_row_bytes / 16);   // 16-byte chunks of a row
            // (the empty asm keeps the row offsets from being formed ahead of the
            // tile loop and held in registers through it)
            int jr = jl;
            asm volatile("" : "+v"(jr));
#pragma unroll 1
            for (int c0 = 0; c0 < nq; c0 += 8) {
#pragma unroll 1
                for (int q = 0; q < 4; ++q) {
                    const int c = c0 + 4 * h + q;
                    const int off = c < nq ? c * 16 : kOut;
                    const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(wr, off + (wave * 32 + jr) * (int)w_row_bytes, 0, 0);
#pragma unroll
                    for (int n = 0; n < NB; ++n) {
                        const u32x4 x =
                            __builtin_amdgcn_raw_buffer_load_b128(xres, off + (32 * n + jr) * (int)w_row_bytes, 0, 0);
                        mfma_quad<DT_F32>(acc[n], w, x);
                    }
                }
            }
        }
    }

    template <bool kBiasInit, class Epi>
    __device__ __forceinline__ void run(f32x16 (&acc)[NB], unsigned char* ring, float* bias_lds, Epi epi)
    {
        if (ntiles <= 0) return;
        unsigned char* ws0 = ring;
        unsigned char* ws1 = ring + kWBuf;
        unsigned char* xs0 = ring + 2 * kWBuf;
        unsigned char* xs1 = ring + 2 * kWBuf + kXBuf;
        lt = 0;
        ls = 0;
        set_rows(0);
        u32x4 w0[kWChunks], w1[kWChunks];
        u32x4 x0[kXChunks], x1[kXChunks];
        // the first two steps' loads go out first; wave 0's bias loads after
        // them, so that neither waits for the other's round trip
        issue(x0, w0);
        issue(x1, w1);
        float bn0[kTileF / 64];
        if (wave == 0) bias_load(bn0, 0);
        store(x0, w0, xs0, ws0);
        if (wave == 0) bias_store(bn0, bias_lds);
        issue(x0, w0);
        __syncthreads();
        acc_reset(acc, bias_lds, kBiasInit);
        for (int t = 0; t < ntiles; ++t) {
            float* bnext = bias_lds + ((t + 1) & 1) * kTileF;
            for (int s = 0; s < nds2; s += 2) {
                float bn[kTileF / 64];
                if (wave == 0) bias_load(bn, t + 1);   // past the last tile: clamped, unused
                compute_store(acc, xs0, ws0, x1, w1, xs1, ws1);
                issue(x1, w1);
                __syncthreads();
                compute_store(acc, xs1, ws1, x0, w0, xs0, ws0);
                issue(x0, w0);
                if (wave == 0) bias_store(bn, bnext);
                __syncthreads();
            }
            reduce(acc, ws1);
            if (kBiasInit) fix_up(acc, t, bias_lds + (t & 1) * kTileF);
            float bv[16];
            if (!kBiasInit) bias_read(bv, bias_lds + (t & 1) * kTileF);
            epi(t, acc, bv);
            acc_reset(acc, bias_lds + ((t + 1) & 1) * kTileF, kBiasInit);   // past the last tile: unused
            __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        }
    }
};

}  // namespace stk
