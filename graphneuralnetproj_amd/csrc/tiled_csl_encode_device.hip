// Tiled-CSL encoder on the GPU, bit-identical to the reference's host encoder
// InitSparseMatrixA_API (csrc/SpMM_API.cu:241-438) and to tiled_csl_encode.cpp.
//
// The reference simulates 32 per-bank stacks with repeated arg-max pops.  Two facts make
// the same output computable in parallel, one workgroup per 128x64 tile:
//   * row m contributes exactly one pair of adjacent columns to every bank: swizzled column
//     c ^ ((m & 7) << 3) has bank (swizzled >> 1), so bank b of row m holds swizzled
//     positions 2b and 2b+1 (csrc/SpMM_API.cu:330-334).  A bank's list is therefore the kept
//     elements among 256 candidates in a fixed order, and an element's place in it is a
//     prefix count;
//   * the pop order is "level = tallest stack down to 1, banks in id order, every bank at
//     least that tall" (the largest stack with the lowest id wins each arg-max,
//     csrc/SpMM_API.cu:223-234), and the emission order (:379-424) is index arithmetic on it.
// So every element computes its own place in the pop order.  Three kernels: count per tile, scan,
// emit.  No counterpart in the reference, which encodes on one host thread.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "offset_scan.h"

namespace {

constexpr int kTileRows = 128, kTileCols = 64, kBanks = 32, kThreads = 256, kWaves = kThreads / 64;
constexpr int kRowGroups = kThreads / kBanks, kRowsPerThread = kTileRows / kRowGroups;  // 8, 16
constexpr int kMaxLevel = 2 * kTileRows + 4;  // 256 per bank + up to 3 pads stay below

using offscan::u16x2;
// The matrix and the words may lie at any element: callers' views begin anywhere (the loads and stores are as wide all the same).
typedef uint32_t pair_any __attribute__((aligned(2)));
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4_word __attribute__((ext_vector_type(4), aligned(4)));

// 1 in each half that holds a kept value (csrc/SpMM_API.cu:262: fabs(float(v)) > 0, i.e. not +-0 and
// not NaN), else 0.
__device__ __forceinline__ u16x2 kept_halves(uint32_t pair)
{
    const u16x2 mag = __builtin_bit_cast(u16x2, pair & 0x7fff7fffu);
    const u16x2 number = __builtin_elementwise_sub_sat(u16x2{0x7c01, 0x7c01}, mag);  // zero for NaN
    return offscan::at_most_one(__builtin_elementwise_min(mag, number));
}

// Vectors per tile into offsets[tile + 1].  Bound by HBM (the matrix is read once): a wave reads 32
// rows of up to eight consecutive tiles, a contiguous KiB per load, all in flight.  (Four bytes per
// lane, one tile per workgroup: 86 us for 411 MB, now 74, and 63 where the emit kernel before it stored past
// the cache.)  Workgroups go from the matrix's
// start to its end, the emit kernel's from end to start: it begins with what is left in the
// last-level cache.
constexpr int kCountTiles = 8;
__global__ __launch_bounds__(kThreads) void tcsl_count_tiles(const uint16_t* __restrict__ A, int K, int tiles_k,
                                                            int* __restrict__ offsets)
{
    __shared__ int part[kWaves][kCountTiles];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int spans = (tiles_k + kCountTiles - 1) / kCountTiles;
    const int row_tile = blockIdx.x / spans, first = (blockIdx.x % spans) * kCountTiles;
    int n = 0;
    if (first + (lane >> 3) < tiles_k) {
        constexpr int kRows = kTileRows / kWaves;
        const uint16_t* src = A + ((size_t)row_tile * kTileRows + wave * kRows) * K + (size_t)first * kTileCols + lane * 8;
        u32x4_any v[kRows];
#pragma unroll
        for (int r = 0; r < kRows; r++)
            v[r] = *reinterpret_cast<const u32x4_any*>(src + (size_t)r * K);
        u16x2 c = {0, 0};
#pragma unroll
        for (int r = 0; r < kRows; r++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                c += kept_halves(v[r][i]);
        n = c[0] + c[1];
    }
    for (int o = 4; o > 0; o >>= 1)
        n += __shfl_xor(n, o);
    if ((lane & 7) == 0)
        part[wave][lane >> 3] = n;
    __syncthreads();
    if (threadIdx.x < kCountTiles && first + (int)threadIdx.x < tiles_k) {
        int nz = 0;
        for (int w = 0; w < kWaves; w++)
            nz += part[w][threadIdx.x];
        offsets[(size_t)row_tile * tiles_k + first + threadIdx.x + 1] = (nz + 3) / 4;  // vectors of four words, zero padded (:289)
    }
}

// offsets[1..tiles] hold per-tile vector counts; turn them into the running total
// (offsets[0] = 0, offsets[tiles + 1] = total, :426-435).  One workgroup.  If the total does
// not fit an int, offsets[tiles + 1] is set to -1.
__global__ __launch_bounds__(offscan::kThreads) void tcsl_scan_offsets(int* __restrict__ offsets, long tiles)
{
    int most;
    const long long total = offscan::scan_in_place(offsets + 1, tiles, most);
    const bool fits = total <= 0x7fffffffLL;
    if (!fits)
        offscan::clear_counts(offsets + 1, tiles);
    if (threadIdx.x == 0) {
        offsets[0] = 0;
        offsets[tiles + 1] = fits ? static_cast<int>(total) : -1;
    }
}

// Smallest and largest value of lanes 0 .. 31, whose copies lanes 32 .. 63 hold.
template<typename Op>
__device__ __forceinline__ int half_wave_reduce(int x, int neutral, Op op)
{
    x = op(x, __builtin_amdgcn_update_dpp(neutral, x, 0x111, 0xf, 0xf, false));  // row_shr 1, 2, 4, 8: within 16 lanes
    x = op(x, __builtin_amdgcn_update_dpp(neutral, x, 0x112, 0xf, 0xf, false));
    x = op(x, __builtin_amdgcn_update_dpp(neutral, x, 0x114, 0xf, 0xf, false));
    x = op(x, __builtin_amdgcn_update_dpp(neutral, x, 0x118, 0xf, 0xf, false));
    x = op(x, __builtin_amdgcn_update_dpp(neutral, x, 0x142, 0xa, 0xf, false));  // lane 15 to lanes 16 .. 31
    return __builtin_amdgcn_readlane(x, 31);
}

// The packed words of one tile, by one workgroup; thread (rg, b) owns the sixteen column pairs that
// rows 16 rg .. +15 give to bank b, and keeps them in registers.  Bound by instruction issue (32
// candidates per thread, a fifth of them kept at 80 % sparsity) beside the read of the matrix and
// the write of the words.
//   * An element's place in its bank's list is a prefix count; its place in the pop order is the
//     number of pops before its level plus the number of lower banks as tall, both from one LDS
//     read of the level's entry (mask of banks, pops before).  The four waves fill that table two levels at a
//     time from ballots on the banks' sizes (the upper lanes hold the banks as well), each its quarter of the levels.
//     A candidate that is not kept reads an entry whose pops lie behind the sequence: eight instructions a candidate, kept or not.
//   * Words go into LDS in pop order and leave it in the order of emission (:379-424), which is plain
//     arithmetic on the output position: four conflict-free reads and one 16-byte store per vector.
//   * 4096 words of LDS for the sequence, so that seven workgroups share a compute unit; a tile beyond
//     that (50 % dense) takes another pass over the registers for every 3968 words.
//   * The words are stored past the caches (nt): whole lines that nothing here reads again (21504 x 7168 at 60 %: 111 us,
//     now 97; the count kernel of the next weight 72 us, now 63).
// (Bank lists staged in LDS, level sums by one thread over 260 levels, words stored one by one:
// 303 us for a 28672 x 7168 weight at 80 %; 766 instructions per wave and tile: 124; now 99 to 107 by the run.  Alone, 21504 x 7168
// at 50 / 80 / 95 %: 157 / 97 / 88 us, now 132 / 77 / 70; 1024 x 1024 at 80 %: 5.3, now 4.9.)
constexpr int kSeqWords = 4096, kPassWords = kSeqWords - 128;  // the first pass takes the tail's up to 124 pops as well

// Offset: of a lane's rows in bytes, the upper row group's being 32 K.  64 bits from K = 2^27 on; below, 32, which the loads
// take beside a uniform address (two instructions fewer for each of a lane's sixteen).
template<typename Offset>
__global__ __launch_bounds__(kThreads, 7) void tcsl_emit_tiles(const uint16_t* __restrict__ A, int K, int tiles_k,
                                                              const int* __restrict__ offsets, uint32_t* __restrict__ items)
{
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    __shared__ uint32_t seq[kSeqWords + 64];   // pops first .. first + kSeqWords - 1; then where words of other passes go
    // entry kMaxLevel - l: banks at least l tall, pops made before the level starts; entry 0: where words that are not go
    __shared__ u32x2 levels[kMaxLevel + 1];
    __shared__ int grp_count[kRowGroups][kBanks];
    __shared__ int grp_zero[kRowGroups][kBanks];

    const int t = gridDim.x - 1 - blockIdx.x;
    const int words = (offsets[t + 1] - offsets[t]) * 4;
    if (words == 0)
        return;  // an all-zero tile emits nothing (uniform for the workgroup)
    const uint16_t* tile = A + (size_t)(t / tiles_k) * kTileRows * K + (size_t)(t % tiles_k) * kTileCols;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b = threadIdx.x & 31, rg = threadIdx.x >> 5;

    // 1. this thread's 16 rows of bank b: mark the kept elements, note the first other position.
    //    Row m gives bank b the pair of adjacent columns whose swizzled positions are 2 b, 2 b + 1.
    // (a row's address is uniform but for this lane's part, of which there are eight)
    const uint8_t* const rows = reinterpret_cast<const uint8_t*>(tile) + (size_t)(wave * 2 * kRowsPerThread) * K * 2;
    const Offset own_row = (rg & 1) * static_cast<Offset>(kRowsPerThread * 2) * K;
    uint32_t pairs[kRowsPerThread];
#pragma unroll
    for (int i = 0; i < kRowsPerThread; i++)
        pairs[i] = *reinterpret_cast<const pair_any*>(rows + (size_t)i * K * 2 + (own_row + ((b << 2) ^ ((i & 7) << 4))));
    uint32_t halves[2] = {0, 0};  // rows 0 .. 7, 8 .. 15: bit 2 (i % 8) + 16 h for element h of row i
#pragma unroll
    for (int i = 0; i < kRowsPerThread; i++)
        halves[i >> 3] |= __builtin_bit_cast(uint32_t, kept_halves(pairs[i])) << (2 * (i & 7));
    const uint32_t kept = ((halves[0] | halves[0] >> 15) & 0xffffu) | (halves[1] | halves[1] >> 15) << 16;  // bit 2 i + h
    const int own = __popc(kept);
    const int z = __ffs(static_cast<int>(~kept)) - 1;  // the first position in row order
    const int corner = rg * kRowsPerThread * kTileCols + 2 * b;  // position = row * 64 + swizzled column (:330-339)
    grp_count[rg][b] = own;
    grp_zero[rg][b] = z < 0 ? -1 : corner + (z >> 1) * kTileCols + (z & 1);
    __syncthreads();

    // 2. the bank's size, and this thread's first place in its list
    int size = 0, rank = 0;
#pragma unroll
    for (int g = 0; g < kRowGroups; g++) {
        const int c = grp_count[g][b];
        rank += g < rg ? c : 0;
        size += c;
    }
    // 3. zero padding to a multiple of four, each pad on the currently smallest bank (lowest id on
    //    ties), pointing at that bank's first zero position (:352-365).  Every wave works it out.
    const int real = size;  // of the bank, without pads
    const int count = __builtin_amdgcn_readlane(offscan::wave_inclusive_sum(lane < kBanks ? size : 0), 63);
    if ((count + 3) / 4 * 4 != words)
        return;  // these are not this tile's offsets (every wave sees the same count)
    for (int pad = (4 - count % 4) % 4; pad > 0; pad--) {
        const int low = half_wave_reduce(size << 5 | b, 0x7fffffff, [](int x, int y) { return x < y ? x : y; });
        size += (low & 31) == b ? 1 : 0;
    }
    // 4. pop order: level = tallest down to 1, banks by id
    const int top = half_wave_reduce(size, 0, [](int x, int y) { return x > y ? x : y; });
    const int share = (top + kWaves - 1) / kWaves;
    const int lo = 1 + wave * share, hi = lo + share - 1 < top ? lo + share - 1 : top;
    if (lo <= hi) {
        const int above = size - hi;
        int pops = __builtin_amdgcn_readlane(offscan::wave_inclusive_sum(lane < kBanks && above > 0 ? above : 0), 63);
        const int upper = lane >> 5;  // the upper lanes' copies of the banks look at the level below
        for (int l = hi; l >= lo; l -= 2) {  // (level lo - 1 may be written as well: the next wave's, with the same entry)
            const uint64_t both = __ballot(size >= l - upper);
            const uint32_t mask = static_cast<uint32_t>(both), mask_below = static_cast<uint32_t>(both >> 32);
            const int pops_below = pops + __popc(mask);
            if (b == 0)
                levels[kMaxLevel - l + upper] = u32x2{upper ? mask_below : mask, static_cast<uint32_t>(upper ? pops_below : pops)};
            pops = pops_below + __popc(mask_below);
        }
    }
    if (threadIdx.x == 0)
        levels[0] = u32x2{~0u, words <= kPassWords ? static_cast<uint32_t>(kSeqWords) : 1u << 30};
    __syncthreads();

    // 5. emission (:379-424): V vectors = R groups of 32 lanes + rem lanes.  The first 4 * rem pops
    //    fill the tail (lane = pop % rem, slot 3 - pop / rem), the rest the main part (lane =
    //    pop' % 32, arrival kk = pop' / 32 written at reverse position 4 R - 1 - kk).
    const uint32_t below = (1u << b) - 1u;
    const int vecs = words / 4, R = vecs / 32, rem = vecs % 32;
    u32x4_word* const out = reinterpret_cast<u32x4_word*>(items) + offsets[t];
    const int dump = kSeqWords + lane;
    // The words of pops first .. last - 1 into the sequence.  Level entries are read sixteen at a time,
    // ahead of the writes that depend on them: one by one, every element pays a trip to LDS.
    auto place_words = [&](int first, int last, auto all) __attribute__((always_inline)) {
        auto place = [&](u32x2 e, uint32_t word) __attribute__((always_inline)) {
            int pop = static_cast<int>(e[1]) + __popc(e[0] & below);
            if constexpr (!decltype(all)::value)  // else the tile's words fit one pass
                pop = pop >= first && pop < last ? pop - first : dump;
            seq[pop] = word;
        };
        const uint8_t* const entries = reinterpret_cast<const uint8_t*>(levels);
        int entry = (kMaxLevel - rank) * 8;  // the byte of the level below the next kept element's
        uint32_t at = static_cast<uint32_t>(corner) << 16, live = kept;
        // (opaque: or the compiler prepares all 32 words and places ahead of both ways, and spills)
        asm volatile("" : "+v"(entry), "+v"(at), "+v"(live));
#pragma unroll
        for (int i0 = 0; i0 < kRowsPerThread; i0 += 8) {
            u32x2 e[16];
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const int used = static_cast<int>(live << (31 - 2 * i0 - j)) >> 31;  // 0 or -1
                entry += used << 3;
                asm("" : "+v"(entry));  // (or the compiler sums `used` up on the side)
                e[j] = *reinterpret_cast<const u32x2*>(entries + (entry & used));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const uint32_t pair = pairs[i0 + j / 2], position = at + (((i0 + j / 2) * kTileCols + (j & 1)) << 16);
                place(e[j], (j & 1 ? pair >> 16 : pair & 0xffffu) | position);
            }
        }
        if (rg == 0 && size > real) {  // the pads, behind the bank's last element
            int p = -1;
            for (int g = 0; g < kRowGroups && p < 0; g++)
                p = grp_zero[g][b];
            for (int l = real + 1; l <= size; l++)
                place(levels[kMaxLevel - l], static_cast<uint32_t>(p) << 16);
        }
    };
    // groups of 32 vectors out of the sequence, whose word `from` is the first of their 128 pops
    auto write_groups = [&](int from, int done, int groups) __attribute__((always_inline)) {
        for (int i = threadIdx.x; i < groups * 32; i += kThreads) {
            const int g = i >> 5, at = from + g * 128 + (i & 31);  // pops 128 g + 32 (3 - s) + lane
            u32x4_word v;
#pragma unroll
            for (int s = 0; s < 4; s++)
                v[s] = seq[at + (3 - s) * 32];
            __builtin_nontemporal_store(v, out + ((R - 1 - done - g) * 32 + (i & 31)));
        }
    };
    auto write_tail = [&]() __attribute__((always_inline)) {
        if ((int)threadIdx.x < rem) {
            u32x4_word v;
#pragma unroll
            for (int s = 0; s < 4; s++)
                v[s] = seq[(3 - s) * rem + threadIdx.x];
            out[R * 32 + threadIdx.x] = v;
        }
    };
    if (words <= kPassWords) {
        place_words(0, words, std::true_type{});
        __syncthreads();
        write_tail();
        write_groups(4 * rem, 0, R);
        return;
    }
    for (int first = 0, last = 4 * rem + kPassWords; first < words; first = last, last += kPassWords) {
        place_words(first, last, std::false_type{});
        __syncthreads();
        const int from = first == 0 ? 4 * rem : 0;
        const int done = (first + from - 4 * rem) / 128;  // groups of earlier passes
        if (first == 0)
            write_tail();
        write_groups(from, done, R - done < kPassWords / 128 ? R - done : kPassWords / 128);
        __syncthreads();  // the sequence is written afresh
    }
}

}  // namespace

// TileOffsets (tiles + 2 ints, device memory) of the dense row-major fp16 matrix A (device memory).
extern "C" int tcsl_launch_encode_offsets(void* stream, const void* A, int M, int K, int* offsets)
{
    const long tiles_k = K / kTileCols, tiles = (long)(M / kTileRows) * tiles_k;
    if (tiles < 1 || tiles > 0x7fffffffL)
        return static_cast<int>(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const long spans = (tiles_k + kCountTiles - 1) / kCountTiles * (M / kTileRows);
    hipLaunchKernelGGL(tcsl_count_tiles, dim3((unsigned)spans), dim3(kThreads), 0, s, static_cast<const uint16_t*>(A), K,
                       (int)tiles_k, offsets);
    hipLaunchKernelGGL(tcsl_scan_offsets, dim3(1), dim3(offscan::kThreads), 0, s, offsets, tiles);
    return static_cast<int>(hipGetLastError());
}

// The packed words, 4 * offsets[tiles + 1] of them, given the offsets computed above.
extern "C" int tcsl_launch_encode_items(void* stream, const void* A, int M, int K, const int* offsets, void* items)
{
    const long tiles_k = K / kTileCols, tiles = (long)(M / kTileRows) * tiles_k;
    if (tiles < 1 || tiles > 0x7fffffffL)
        return static_cast<int>(hipErrorInvalidValue);
    auto* const emit = K < 1 << 27 ? tcsl_emit_tiles<uint32_t> : tcsl_emit_tiles<uint64_t>;
    hipLaunchKernelGGL(emit, dim3((unsigned)tiles), dim3(kThreads), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(A), K, (int)tiles_k, offsets, static_cast<uint32_t*>(items));
    return static_cast<int>(hipGetLastError());
}
