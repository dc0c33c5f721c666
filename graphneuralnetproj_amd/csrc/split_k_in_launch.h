// The split-K reduction inside a launch, shared by the Tiled-CSL kernel (spmm_kernels.hip) and the
// 2:4 kernel (a24_kernels.hip): the write-through stores and memory-served loads that carry slabs
// of partial sums between workgroups, and the tail in which the last workgroup to finish a group
// of rows adds that group's slabs up.  Stands in for csrc/Reduction_Kernel.cuh:24-47 where a launch
// can do the sum itself; same order of additions, hence the same bits.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace inlaunch {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));

// Stores and loads at system scope (write through every cache level / served from memory):
// how the slabs of partial sums travel between workgroups of one launch without cache
// maintenance.  A device-wide fence would write back and invalidate the whole L2 of the XCD,
// which the weight stream lives in.  Relaxed 64-bit atomics rather than inline assembly: the
// compiler then also keeps the store data registers untouched for as long as the hardware
// needs them (an assembly store's data was seen overwritten by the next VALU instruction).
__device__ __forceinline__ void store_through(_Float16* p, half4 v)
{
    __hip_atomic_store(reinterpret_cast<uint64_t*>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void store_through(_Float16* p, _Float16 v)
{
    __hip_atomic_store(reinterpret_cast<uint16_t*>(p), __builtin_bit_cast(uint16_t, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ half8 load_through(const _Float16* p)
{
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    u64x2 w;
    w[0] = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    w[1] = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return __builtin_bit_cast(half8, w);
}

// Fused split-K reduction, called by every thread of a workgroup that has just written its slab
// of partial sums (through to memory) for rows [row0, row0 + NROWS): the last of the Split_K
// workgroups that share those rows adds the slabs up, in slab order like the separate kernel
// (csrc/Reduction_Kernel.cuh:36-46), so both paths give the same bits.  `counter` is the rows'
// arrival count in device memory (zero between calls), `flag` one free LDS word, nthreads the
// number of threads of the workgroup that are still there (the first nthreads).
// Bits 8 and up of `relu` count further slabs that an earlier launch on the same stream left right
// behind this launch's own Split_K (the 2:4 part's partial sums); they are added after them.
// ROWMAJ: slabs and C are [M][N] (the rows' block is one contiguous run of NROWS * N values;
// ldc is not used) instead of one M vector per token.
// The sum moves eight rows at a time: NROWS, M and row0 must be multiples of 8, and M one of NROWS (the launchers check M).
// What bounds it is trips to memory (0.7 us each), then its own instructions, which nothing in the launch has run before:
// the number of rows and the layout are constants (no division for a run's place), and what is left behind the groups
// of four slabs takes one trip (one by one before), its code out of the way of those.  1024 x 1024 at 8 tokens in four
// batches 6.38 -> 6.26 us, 1024 x 2048 at 16 tokens in three 8.3 -> 7.9, in seven 7.93 -> 7.30.  (A last group of four
// that repeats its last slab and masks it: 2 to 4 % slower at five and eight slabs, each load goes to memory.)
template <int NROWS, bool ROWMAJ>
__device__ __forceinline__ void fused_reduction_tail(const _Float16* __restrict__ slabs, _Float16* __restrict__ C, int M,
                                                     int N, int ldc, int split_k, int relu, int row0,
                                                     unsigned int* counter, unsigned int* flag, int nthreads)
{
    // This workgroup's partial sums have reached memory before it is counted.  The hardware side
    // of that is the wait (the write-through stores are acknowledged at the coherence point); the
    // two workgroup-scope fences say the same to the compiler, which may then move neither the
    // slab stores below the counting nor the slab loads above it.  At workgroup scope a fence is
    // waits only: no cache is written back or invalidated (a wider fence would flush the L2 that
    // the weight stream lives in).
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), on top of what the compiler tracks itself
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    if (threadIdx.x == 0)
        *flag = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (*flag != static_cast<unsigned int>(split_k - 1))
        return;
    split_k += relu >> 8;
    relu &= 0xff;
    constexpr int kPerTok = NROWS / 8;
    const int total = kPerTok * N;  // runs of eight rows to sum
    const size_t slab = (size_t)M * N;
    // Every load is served from memory, and a thread can only add what has arrived.  A thread with
    // several runs of eight rows (64 tokens: four per thread) keeps four slabs of four runs in flight,
    // sixteen 16-byte loads, so that its trips to memory are ceil(split_k / 4) in all rather than per
    // run (9216 x 9216, 64 tokens, three batches: 28.9 -> 26.2 us).  Each element's slabs are still
    // added in slab order.  (Sixteen slabs of one run at a time, for the threads that have a single
    // run, measured 2 to 3 % slower than four even where there are only four.)
    auto sum_runs = [&](int c0, auto it_c) __attribute__((always_inline)) {
        constexpr int IT = decltype(it_c)::value, G = 4;
        int tok[IT], row[IT];
        uint32_t at[IT];  // (a slab is 4096 groups of rows and 64 tokens at most: 32 bits)
        float sum[IT][8];
#pragma unroll
        for (int i = 0; i < IT; i++) {
            const int c = IT == 1 || c0 + i * nthreads < total ? c0 + i * nthreads : c0;  // a run past the end repeats the first
            tok[i] = c / kPerTok, row[i] = c % kPerTok * 8;
            at[i] = ROWMAJ ? static_cast<uint32_t>(row0) * N + c * 8 : static_cast<uint32_t>(tok[i]) * M + row0 + row[i];
#pragma unroll
            for (int j = 0; j < 8; j++)
                sum[i][j] = 0.f;
        }
        const _Float16* from = slabs;
        int left = split_k;
        for (; left >= G; left -= G, from += G * slab) {
            half8 w[G][IT];
#pragma unroll
            for (int u = 0; u < G; u++)
#pragma unroll
                for (int i = 0; i < IT; i++)
                    w[u][i] = load_through(from + u * slab + at[i]);
#pragma unroll
            for (int u = 0; u < G; u++)
#pragma unroll
                for (int i = 0; i < IT; i++)
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        sum[i][j] += static_cast<float>(w[u][i][j]);
        }
        if (__builtin_expect(left > 0, 0)) {  // the rest
            half8 w[G - 1][IT];
#pragma unroll
            for (int u = 0; u < G - 1; u++)
                if (u == 0 || u < left)
#pragma unroll
                    for (int i = 0; i < IT; i++)
                        w[u][i] = load_through(from + u * slab + at[i]);
#pragma unroll
            for (int u = 0; u < G - 1; u++)
                if (u == 0 || u < left)
#pragma unroll
                    for (int i = 0; i < IT; i++)
#pragma unroll
                        for (int j = 0; j < 8; j++)
                            sum[i][j] += static_cast<float>(w[u][i][j]);
        }
#pragma unroll
        for (int i = 0; i < IT; i++) {
            if (IT > 1 && c0 + i * nthreads >= total)
                break;
            half8 o;
#pragma unroll
            for (int j = 0; j < 8; j++)
                o[j] = static_cast<_Float16>(relu ? fmaxf(sum[i][j], 0.f) : sum[i][j]);
            *reinterpret_cast<half8*>(C + (ROWMAJ ? (size_t)at[i] : (size_t)tok[i] * ldc + row0 + row[i])) = o;
        }
    };
    if (total <= nthreads) {
        if (static_cast<int>(threadIdx.x) < total)
            sum_runs(threadIdx.x, std::integral_constant<int, 1>{});
    } else {
        for (int c0 = threadIdx.x; c0 < total; c0 += nthreads * 4)
            sum_runs(c0, std::integral_constant<int, 4>{});
    }
    if (threadIdx.x == 0)
        *counter = 0;  // ready for the next call
}

}  // namespace inlaunch
