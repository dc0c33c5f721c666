// Running totals of per-tile or per-list counts in device memory, in place, by one workgroup, and two small functions on
// lanes and halves.  Shared by the Tiled-CSL encoder and the residual packer.
//
// Bound by the latency of its few trips to memory, not by bandwidth: 75264 counts are 0.3 MB.  A
// workgroup takes 16384 counts per step, 16 bytes per lane and load with whole lines per wave, the
// next step's loads in flight while this one adds; lane sums go through DPP, wave sums through LDS
// with one barrier per step.  (One chunk of consecutive counts per thread, read twice, had every
// load of a wave touch 64 lines: 133 us for 75264 counts, now 10;
// 38 us for 25088, now 7.)
#pragma once
#include <hip/hip_runtime.h>

namespace offscan {

constexpr int kThreads = 1024, kWaves = kThreads / 64, kRows = 4;
constexpr int kStep = kThreads * 4 * kRows;

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// min(x, 1) in both halves, in one instruction: the compiler takes a minimum with one apart into a comparison and a
// select per half.
__device__ __forceinline__ u16x2 at_most_one(u16x2 x)
{
    u16x2 r;
    asm("v_pk_min_u16 %0, %1, %2" : "=v"(r) : "v"(x), "s"(0x00010001));
    return r;
}

typedef int i32x4_u __attribute__((ext_vector_type(4), aligned(4)));  // any int boundary will do

// Inclusive sum over the lanes of a wave.
__device__ __forceinline__ int wave_inclusive_sum(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8: within 16 lanes
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // lane 15 of rows 0, 2 to rows 1, 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // lane 31 to rows 2, 3
    return x;
}

// counts[0 .. n-1] become inclusive running totals; returns the grand total (to every thread) and
// the largest count.  Totals beyond an int are cut off: the caller looks at the one returned.
// blockDim.x = kThreads.
__device__ __forceinline__ long long scan_in_place(int* counts, long n, int& largest)
{
    __shared__ int wave_sum[2][kWaves];
    __shared__ int wave_most[kWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto load = [&](long base, i32x4_u (&v)[kRows]) {
#pragma unroll
        for (int k = 0; k < kRows; k++) {
            const long e = base + wave * (kStep / kWaves) + k * 256 + lane * 4;
            v[k] = i32x4_u{0, 0, 0, 0};
            if (e + 4 <= n)
                v[k] = *reinterpret_cast<const i32x4_u*>(counts + e);
            else
                for (int i = 0; i < 4; i++)
                    if (e + i < n)
                        v[k][i] = counts[e + i];
        }
    };
    long long run = 0;
    int most = 0, side = 0;
    i32x4_u next[kRows];
    load(0, next);
    for (long base = 0; base < n; base += kStep, side ^= 1) {
        i32x4_u v[kRows];
#pragma unroll
        for (int k = 0; k < kRows; k++)
            v[k] = next[k];
        if (base + kStep < n)
            load(base + kStep, next);
        int before[kRows], sum = 0;  // total of the wave's elements before this lane's four of row k
#pragma unroll
        for (int k = 0; k < kRows; k++) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                most = v[k][i] > most ? v[k][i] : most;
            v[k][1] += v[k][0];
            v[k][2] += v[k][1];
            v[k][3] += v[k][2];
            const int incl = wave_inclusive_sum(v[k][3]);
            before[k] = sum + incl - v[k][3];
            sum += __builtin_amdgcn_readlane(incl, 63);
        }
        if (lane == 0)
            wave_sum[side][wave] = sum;
        __syncthreads();  // (the other half of wave_sum may be written for the next step meanwhile)
        int ahead = 0, all = 0;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const int s = wave_sum[side][w];
            ahead += w < wave ? s : 0;
            all += s;
        }
        const int start = static_cast<int>(run) + ahead;
#pragma unroll
        for (int k = 0; k < kRows; k++) {
            const long e = base + wave * (kStep / kWaves) + k * 256 + lane * 4;
            v[k] += start + before[k];
            if (e + 4 <= n)
                *reinterpret_cast<i32x4_u*>(counts + e) = v[k];
            else
                for (int i = 0; i < 4; i++)
                    if (e + i < n)
                        counts[e + i] = v[k][i];
        }
        run += all;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const int other = __shfl_xor(most, o);
        most = other > most ? other : most;
    }
    if (lane == 0)
        wave_most[wave] = most;
    __syncthreads();
    largest = 0;
    for (int w = 0; w < kWaves; w++)
        largest = wave_most[w] > largest ? wave_most[w] : largest;
    return run;
}

// Every count becomes zero: what stands in for totals that no int holds.
__device__ __forceinline__ void clear_counts(int* counts, long n)
{
    for (long e = threadIdx.x; e < n; e += kThreads)
        counts[e] = 0;
}

}  // namespace offscan
