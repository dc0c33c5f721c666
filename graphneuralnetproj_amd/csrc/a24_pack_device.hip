// A weight that is in device memory becomes 2:4 records, a dense residual and the residual's lists
// of words (layouts: a24_format.h), with the same bits as the host functions in a24_pack.cpp.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "offset_scan.h"

namespace {
constexpr int kRecordBytes = 2304;
constexpr int kGroupBlocks = 8;  // records of eight row blocks are stored together, unit by unit
}  // namespace

// Split and pack on the GPU: the same bits as the host's decompose + pack (a24_pack.cpp), for
// weights that are already in device memory: the first two kept values of every group of four
// (kernel_benchmark/spmm_decompose.h:12-51) go to the record, the others to the dense residual (when
// asked for one), zero elsewhere.
//
// Bound by HBM.  A workgroup takes 16 rows of four consecutive units, a wave four of the rows: every
// load, and every store to the residual, is one contiguous KiB, and the four records leave through LDS in
// whole lines.  What becomes of a group of four is a function of which of its elements are kept,
// looked up in a table of sixteen entries.  (A thread per lane of a record, which reads its own four
// granules, half a line to sixteen rows per load, and works the positions out by comparing: 217 us on a
// 21504 x 7168 weight, half of them vector instructions; now 114.  1024 x 1024: 5.5 us, now 3.3.)
namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
using offscan::u16x2;
typedef u32x4 u32x4_any __attribute__((aligned(2)));   // the matrices' granules may lie at any element,
typedef u32x4 u32x4_byte __attribute__((aligned(1)));  // the records at any byte
typedef unsigned u32_byte __attribute__((aligned(1)));

// 1 in each half that is kept: unequal to zero as a float (NaN counts, -0 does not)
__device__ __forceinline__ unsigned kept_halves(unsigned pair)
{
    return __builtin_bit_cast(unsigned, offscan::at_most_one(__builtin_bit_cast(u16x2, pair & 0x7fff7fffu)));
}

constexpr int kSplitUnits = 4;  // units per workgroup
// A record in LDS: its eight 256-byte blocks of values (block = step / 2 * 4 + column group) 272 bytes apart, then the
// positions; records 2432 apart.  The 64 eight-byte writes of a row (a unit's 16 granules, four units) fall
// two to a bank, which is as few as there can be.
constexpr int kBlockStride = 272, kRecordStride = 8 * kBlockStride + 256;

struct SplitEntry {
    unsigned values;     // v_perm selector: the record's two values of the group (0xc: a zero byte)
    unsigned rest;       // ... and the residual's elements 2 and 3 (elements 0 and 1 are among the first two)
    unsigned positions;  // 2 bits each
    unsigned unused;
};
// Entry for the kept elements `mask` of a group; a group with fewer than two is filled at free positions.
constexpr SplitEntry split_entry(unsigned mask)
{
    unsigned pos[2] = {0, 1}, rest = 0x0c0c0c0cu;
    int n = 0;
    for (unsigned e = 0; e < 4; e++)
        if (mask >> e & 1) {
            if (n < 2)
                pos[n] = e;
            else
                rest = e == 2 ? (rest & 0xffff0000u) | 0x0504u : (rest & 0xffffu) | 0x07060000u;
            n++;
        }
    bool have0 = n >= 1, have1 = n >= 2;
    if (n == 1 && pos[0] == 3) {  // the free slot goes before it
        have0 = false;
        have1 = true;
        pos[0] = 2;
        pos[1] = 3;
    } else if (n == 1) {
        pos[1] = 3;
    }
    const unsigned v0 = have0 ? 0x0100u + 0x0202u * pos[0] : 0x0c0cu, v1 = have1 ? 0x0100u + 0x0202u * pos[1] : 0x0c0cu;
    return SplitEntry{v0 | v1 << 16, rest, pos[0] | pos[1] << 2, 0u};
}
struct SplitTable {
    SplitEntry e[16];
};
constexpr SplitTable make_split_table()
{
    SplitTable t{};
    for (unsigned m = 0; m < 16; m++)
        t.e[m] = split_entry(m);
    return t;
}
__constant__ const SplitTable split_table = make_split_table();

}  // namespace

template<bool RESIDUAL>
__global__ __launch_bounds__(256) void a24_split_pack_kernel(const uint16_t* __restrict__ A, uint8_t* __restrict__ packed,
                                                             uint16_t* __restrict__ residual, int K, int units)
{
    __shared__ __attribute__((aligned(16))) uint8_t records[kSplitUnits * kRecordStride];
    __shared__ u32x4 table[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int spans = (units + kSplitUnits - 1) / kSplitUnits;
    const unsigned rb = blockIdx.x / spans;
    const int u0 = static_cast<int>(blockIdx.x % spans) * kSplitUnits;
    const int u = u0 + (lane >> 4), g = lane & 15;
    const bool live = u < units;
    const size_t at = ((size_t)rb * 16 + wave * 4) * K + (size_t)u * 128 + g * 8;
    u32x4 in[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        in[j] = u32x4{0u, 0u, 0u, 0u};
        if (live)
            in[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(A + at + (size_t)j * K));
    }
    if (threadIdx.x < 16)
        table[threadIdx.x] = reinterpret_cast<const u32x4*>(split_table.e)[threadIdx.x];
    __syncthreads();
    // lane (column group g % 4, row) of a record keeps step g / 4's values of this granule
    uint8_t* const rec = records + (lane >> 4) * kRecordStride;
    uint8_t* const value = rec + ((g >> 3) * 4 + (g & 3)) * kBlockStride + wave * 64 + ((g >> 2) & 1) * 8;
    uint8_t* const place = rec + 8 * kBlockStride + (g & 3) * 64 + wave * 16;
    const uint8_t* const entries = reinterpret_cast<const uint8_t*>(table);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        unsigned flags = 0;  // element 2 i + h kept: bit 2 i + 16 h
#pragma unroll
        for (int i = 0; i < 4; i++)
            flags |= kept_halves(in[j][i]) << (2 * i);
        const unsigned mask = flags | flags >> 15;
        const u32x4 lo = *reinterpret_cast<const u32x4*>(entries + ((mask << 4) & 0xf0u));
        const u32x4 hi = *reinterpret_cast<const u32x4*>(entries + (mask & 0xf0u));
        *reinterpret_cast<u32x2*>(value + j * 16) = u32x2{__builtin_amdgcn_perm(in[j][1], in[j][0], lo[0]),
                                                          __builtin_amdgcn_perm(in[j][3], in[j][2], hi[0])};
        if (RESIDUAL && live)
            *reinterpret_cast<u32x4_any*>(residual + at + (size_t)j * K) =
                u32x4{0u, __builtin_amdgcn_perm(in[j][1], in[j][0], lo[1]), 0u, __builtin_amdgcn_perm(in[j][3], in[j][2], hi[1])};
        // the four steps' positions of (column group, row) are four lanes apart
        int word = static_cast<int>((lo[2] | hi[2] << 4) << (8 * (g >> 2)));
        word |= __builtin_amdgcn_update_dpp(0, word, 0x124, 0xf, 0xf, false);  // row_ror 4, 8
        word |= __builtin_amdgcn_update_dpp(0, word, 0x128, 0xf, 0xf, false);
        if (g < 4)
            *reinterpret_cast<int*>(place + j * 4) = word;
    }
    __syncthreads();
    // records are numbered ((rb / 8) * units + u) * 8 + rb % 8
    uint8_t* const out = packed + ((size_t)(rb / kGroupBlocks * units + u0) * kGroupBlocks + rb % kGroupBlocks) * kRecordBytes;
#pragma unroll
    for (int j = 0; j < kSplitUnits * 128 / 256; j++) {
        const int id = threadIdx.x + j * 256, r = id >> 7, granule = id & 127;
        if (u0 + r < units)
            __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(records + r * kRecordStride + (granule >> 4) * kBlockStride + (granule & 15) * 16),
                                        reinterpret_cast<u32x4_byte*>(out + (size_t)r * kGroupBlocks * kRecordBytes + granule * 16));
    }
    if (u0 + wave < units)
        *reinterpret_cast<u32_byte*>(out + (size_t)wave * kGroupBlocks * kRecordBytes + 2048 + lane * 4) =
            *reinterpret_cast<const unsigned*>(records + wave * kRecordStride + 8 * kBlockStride + lane * 4);
}

// A: row-major M x K fp16 in device memory (M % 16 == 0, K % 128 == 0, checked by the caller);
// residual may be null.
extern "C" int a24_launch_split_pack(void* stream, const void* A, void* packed, void* residual, int M, int K)
{
    const int units = K / 128;
    const long blocks = static_cast<long>(M / 16) * ((units + kSplitUnits - 1) / kSplitUnits);
    if (blocks < 1 || blocks > 0x7fffffffL)
        return static_cast<int>(hipErrorInvalidValue);
    auto* const kernel = residual ? a24_split_pack_kernel<true> : a24_split_pack_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t*>(A), static_cast<uint8_t*>(packed), static_cast<uint16_t*>(residual), K, units);
    return static_cast<int>(hipGetLastError());
}

// The residual lists on the GPU, from the dense residual that the split above leaves in device
// memory: the same words in the same order as the host's pack_residual (a24_pack.cpp).  Three
// kernels: count per list, scan, emit.
namespace {

constexpr int kMaxListWords = 16 * 128 / 2;  // a residual holds at most two of every four

// x + the lanes of the mask below this one
__device__ __forceinline__ int lower_lanes(uint64_t mask, int x)
{
    return static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(mask >> 32),
                                                      __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), static_cast<unsigned>(x))));
}
__device__ __forceinline__ bool residual_kept(unsigned v)
{
    return (v & 0x7fffu) != 0;
}

// Words per list into offsets[list + 1].  Bound by HBM (the residual is read once).  A wave takes the
// 16 rows of up to four consecutive units: sixteen loads of one contiguous KiB each, all in flight
// together.  (One list per wave, 64 bytes per lane: a load instruction touched 32 half lines and a
// 21504 x 7168 residual of 308 MB took 105 us; now 73.)  Workgroups run from the matrix's end to its
// start, and the emit kernel from start to end: each begins with what the kernel before it left in
// the last-level cache.
__global__ __launch_bounds__(256) void a24_residual_count_kernel(const uint16_t* __restrict__ A2, int K, int units,
                                                                 unsigned tasks, int* __restrict__ offsets)
{
    const unsigned task = (gridDim.x - 1 - blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (task >= tasks)
        return;
    const int L = threadIdx.x & 63;
    const unsigned spans = (units + 3) / 4;
    const unsigned rb = task / spans;
    const int u = static_cast<int>(task % spans) * 4 + (L >> 4);
    int n = 0;
    if (u < units) {
        const uint16_t* src = A2 + (size_t)rb * 16 * K + (size_t)u * 128 + (L & 15) * 8;
        u32x4 v[16];
#pragma unroll
        for (int r = 0; r < 16; r++)
            v[r] = *reinterpret_cast<const u32x4*>(src + (size_t)r * K);
        u16x2 c = {0, 0};
#pragma unroll
        for (int r = 0; r < 16; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                c += __builtin_bit_cast(u16x2, kept_halves(v[r][i]));
            }
        n = c[0] + c[1];
    }
    for (int o = 8; o > 0; o >>= 1)
        n += __shfl_xor(n, o);
    if ((L & 15) == 0 && u < units)
        offsets[((size_t)(rb / kGroupBlocks) * units + u) * kGroupBlocks + rb % kGroupBlocks + 1] = n;
}

// offsets[1..lists] hold the lists' lengths; turn them into running totals (offsets[0] = 0) and
// report the longest.  One workgroup.  A total beyond what an int holds gives offsets[lists] = -1.
__global__ __launch_bounds__(offscan::kThreads) void a24_residual_scan_kernel(int* __restrict__ offsets, long lists,
                                                                              int* __restrict__ longest)
{
    int most;
    const long long total = offscan::scan_in_place(offsets + 1, lists, most);
    const bool fits = total <= 0x7fffffffLL - 64;
    if (!fits) {
        __syncthreads();
        offscan::clear_counts(offsets + 1, lists);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (!fits)
            offsets[lists] = -1;
        offsets[0] = 0;
        *longest = most;
    }
}

// The words.  Bound by instruction issue beside the read of the residual (21504 x 7168: 51 us at 95 % sparsity, where
// nothing is dealt, 99 at 60 %).
//
// In a list's order (a24_pack.cpp: order_by_bank) the words of one LDS bank are neighbours: banks by
// (count descending, number ascending), a bank's words as collected.  A bank's words come from 16
// known column pairs, one per row (row r: pair bank ^ (r << 2)), so lane b of a list's wave reads
// bank b's 32 candidates itself, a whole 256-byte row per load, and knows its count, its place
// among the banks (a ballot per count there is) and its words without any exchange.  Where a word goes is then
// the result of dealing the banks' words to the rounds, bank after bank, each depending on the one
// before; it depends on the counts alone, so one LANE deals for one list: the lists of a workgroup
// side by side (one lane of one wave dealing for the wave's only list took 1150 us on the
// 21504 x 7168 residual of a 60 % sparse weight; 32 lists side by side, word by word, 137; a lap of a bank at a time, every
// lane at its own bank, 110; with 16 lists 99).  A list of at most 64 words stays in row-major order, as the host leaves it.
//
// The residual is read a second time for the writing (from the last-level cache) instead of kept in
// registers: more workgroups per compute unit, whose dealing waves hide each other.  Seven of 16 lists: 64 vector registers and
// 96 scalar ones are the most a wave may have (with 97, six: 7168 x 7168, 70 words a list, 34 us -> 43).
constexpr int kEmitWaves = 4;
// Lists per workgroup: the lists of a wave follow one another and the others wait while one wave deals, so few lists
// are better spread over more waves, and many are better dealt 16 at a time (whole calls at 50 / 60 / 95 %:
// 2048 x 4096 = 4096 lists: eight to a workgroup 22 / 17 / 7 us, 16 25 / 19 / 10; 5120 x 5248 = 13120: 35 / 26 / 15 and
// 36 / 29 / 16; 4096 x 8192 = 16384: 40 / 30 / 16 and 37 / 30 / 16; 7168 x 7168 = 25088: 56 / 42 / 22 and 52 / 41 / 23).
constexpr int kManyLists = 16, kFewLists = 8;
constexpr long kManyFrom = 16384;

// A word of the bank-sorted sequence goes to the round that has the fewest words of its bank, then
// the most room, then the lowest number.  So a bank's words go round by round in laps: once around the
// rounds that have room, those with the most room first, then around again.
//
// For a list of at most four rounds a word's place in code is one byte, (room - 1) * 4 + (3 - round); for longer
// lists the place is written as two bytes.  (Three more bytes: what a lap writes beyond its own words.)
__device__ __forceinline__ constexpr int place_bytes(int n)
{
    return n <= 256 ? n + 3 : 2 * n;
}
// The last places of a list's four rounds, a byte each, the last round's first (n <= 256).
__device__ __forceinline__ unsigned round_ends(int n)
{
    unsigned ends = 0;
#pragma unroll
    for (int k = 0; k < 4; k++)
        ends |= static_cast<unsigned>((256 - 64 * k < n ? 256 - 64 * k : n) - 1) << (8 * k);
    return ends;
}
// n > 256: `ends` is not looked at
__device__ __forceinline__ int place_of(const uint8_t* places, int p, int n, unsigned ends)
{
    if (n > 256)
        return places[p] | places[p + n] << 8;
    const unsigned code = places[p];
    return static_cast<int>(__builtin_amdgcn_perm(0, ends, (code & 3u) | 0x0c0c0c00u) - (code >> 2));
}

// Deals one list of n words, 64 < n <= 64 * R and n <= 256, whose banks hold counts[0] >= counts[1] >= ... words
// (a byte after the last one may be read).  A step of the loop is one lap of this lane's current bank, whatever bank the
// other lanes are at.  The rounds' codes are kept in order, largest first; a round without room has a negative one.
template<int R>
__device__ __forceinline__ void deal_laps(const uint8_t* counts, int n, uint8_t* places)
{
    static_assert(R >= 2 && R <= 4, "two bits for the round");
    int key[R];
    const int rounds = (n + 63) >> 6;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int room = r < rounds - 1 ? 64 : (r == rounds - 1 ? n - 64 * (rounds - 1) : 0);
        key[r] = (room - 1) * 4 + (3 - r);
    }
    auto order = [&](int a, int b) __attribute__((always_inline)) {
        const int x = key[a], y = key[b];
        key[a] = x > y ? x : y;
        key[b] = x > y ? y : x;
    };
    const uint8_t* const end = places + n;
    int c = counts[0], following = counts[1];
    while (places < end) {
#pragma unroll
        for (int j = 0; j < R; j++)  // what is not taken is written over by the next lap
            places[j] = static_cast<uint8_t>(key[j]);
        int taken = 1;
        key[0] -= 4;
#pragma unroll
        for (int j = 1; j < R; j++) {
            const bool takes = c > j && key[j] >= 0;
            key[j] -= takes ? 4 : 0;
            taken += takes ? 1 : 0;
        }
        places += taken;
        c -= taken;
        order(0, 1);
        if constexpr (R == 3) {
            order(1, 2);
            order(0, 1);
        } else if constexpr (R == 4) {
            order(2, 3);
            order(0, 2);
            order(1, 3);
            order(1, 2);
        }
        counts += c == 0 ? 1 : 0;
        c = c == 0 ? following : c;
        following = counts[1];
    }
}

// ... of 256 < n <= 1024 words, word by word: the largest of keys (63 - words of the bank, room - 1, last - round), zero
// for a full round.
__device__ __forceinline__ void deal_long(const unsigned* counts, int n, uint8_t* places)
{
    constexpr int R = 16, kRoundBits = 4, kLast = (1 << kRoundBits) - 1;
    constexpr unsigned kRoom = 1u << kRoundBits, kOne = 64u << kRoundBits;  // units of the two upper fields
    unsigned key[R];
    const int rounds = (n + 63) >> 6;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int room = r < rounds - 1 ? 64 : (r == rounds - 1 ? n - 64 * (rounds - 1) : 0);
        key[r] = room > 0 ? 63 * kOne + (room - 1) * kRoom + (kLast - r) : 0u;
    }
    unsigned four = counts[0];
    for (int k = 0; k < 16 && four != 0; k++) {
        const unsigned next = k < 15 ? counts[k + 1] : 0u;
        for (; four != 0; four >>= 8) {  // (largest first: once a byte is zero all that follow are)
#pragma unroll
            for (int r = 0; r < R; r++)
                key[r] = key[r] ? (key[r] & (kOne - 1)) | 63 * kOne : 0u;
            for (int c = four & 0xffu; c > 0; c--, places++) {
                unsigned best = key[0];
#pragma unroll
                for (int r = 1; r < R; r++)
                    best = key[r] > best ? key[r] : best;
                const unsigned room = best & (kOne - kRoom);  // minus one
                const int end = 1024 - 64 * static_cast<int>(best & kLast);
                const int place = (end < n ? end : n) - 1 - static_cast<int>(room / kRoom);
                places[0] = static_cast<uint8_t>(place);
                places[n] = static_cast<uint8_t>(place >> 8);
                const unsigned then = room == 0 ? 0u : best - kOne - kRoom;
#pragma unroll
                for (int r = 0; r < R; r++)
                    key[r] = key[r] == best ? then : key[r];
            }
        }
        four = next;
    }
}

template<int kEmitLists>
__global__ __launch_bounds__(kEmitWaves * 64, 8) void a24_residual_emit_kernel(const uint16_t* __restrict__ A2, int K, int units,
                                                                               long lists, const int* __restrict__ offsets,
                                                                               uint32_t* __restrict__ words)
{
    constexpr int kListsPerWave = kEmitLists / kEmitWaves;
    constexpr int kPlaces = kEmitLists * place_bytes(256);  // bytes: lists of 256 words (an ordinary residual has up to 200) are dealt in one pass
    constexpr int kImages = kEmitWaves * 16 * 64 * 4;  // bytes, per wave: a list's block, [row][bank] column pairs
    static_assert(kPlaces >= place_bytes(kMaxListWords), "the longest list has to fit");
    __shared__ __attribute__((aligned(16))) uint8_t room[kImages + kPlaces];  // the places, then the images
    __shared__ unsigned sorted[kEmitLists][17];      // counts of a list's banks, one byte each, largest first
    __shared__ int length[kEmitLists];
    const int L = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int total = offsets[lists];
    if (total < 0)  // the word count did not fit an int: no offset of this table means anything, nothing is written
        return;
    if (blockIdx.x == 0 && w == 0)  // the padding behind the last list
        words[(size_t)total + L] = 0;
    uint8_t* const places = room;
    unsigned* const image = reinterpret_cast<unsigned*>(room + kPlaces) + w * (16 * 64);

    // wave w takes the workgroup's lists w, w + 4, ...
    auto list_of = [&](int i) { return (long)blockIdx.x * kEmitLists + i * kEmitWaves + w; };
    auto block_of = [&](long list) {
        const unsigned unit_row = static_cast<unsigned>(list / kGroupBlocks);  // (128-row group, unit)
        const unsigned group = unit_row / units, u = unit_row % units;
        return A2 + (((size_t)group * kGroupBlocks + list % kGroupBlocks) * 16 * K + (size_t)u * 128);
    };
    // (in the global address space by name: the compiler does not see that through the asm below)
    auto load_list = [&](long list, unsigned (&pairs)[16]) {
        auto* src = (const __attribute__((address_space(1))) uint16_t*)block_of(list);
        int lane = L;
        // (opaque: else the compiler issues the loads of all lists ahead of the first one's use, 300 registers)
        asm volatile("" : "+s"(src), "+v"(lane)::"memory");
#pragma unroll
        for (int r = 0; r < 16; r++)
            pairs[r] = *(const __attribute__((address_space(1))) unsigned*)(src + (size_t)r * K + 2 * (lane ^ (r << 2)));
    };
    unsigned kept[kListsPerWave];  // bit 2 r + h: element h of row r's pair
    int start[kListsPerWave];      // where the bank's words begin in the bank-sorted sequence

    // 1. counts of the banks, their order; lists of one round are written at once
#pragma unroll
    for (int i = 0; i < kListsPerWave; i++) {
        const long list = list_of(i);
        const int li = i * kEmitWaves + w;
        kept[i] = 0;
        start[i] = 0;
        if (list >= lists) {
            if (L == 0)
                length[li] = 0;
            continue;
        }
        unsigned pairs[16];
        load_list(list, pairs);
        unsigned halves[2] = {0, 0};  // rows 0 .. 7, 8 .. 15: bit 2 (r % 8) + 16 h
#pragma unroll
        for (int r = 0; r < 16; r++)
            halves[r >> 3] |= kept_halves(pairs[r]) << (2 * (r & 7));
        const unsigned mask = ((halves[0] | halves[0] >> 15) & 0xffffu) | (halves[1] | halves[1] >> 15) << 16;
        kept[i] = mask;
        const int count = __popc(mask);
        // the banks' places from the last one on: by count upwards (a few counts only), equal ones by number
        int n = 0, banks = 64, before = 0, place = 0;  // words and banks of the counts so far; this bank's
        uint64_t left = ~0ull;
        for (int c = 0; left != 0; c++) {
            const uint64_t same = __ballot(count == c);
            const int number = __popcll(same);
            const int lower = lower_lanes(same, 0);
            n += c * number;
            banks -= number;
            before = count == c ? c * lower - n : before;
            place = count == c ? banks + lower : place;
            left &= ~same;
        }
        start[i] = n + before;
        reinterpret_cast<uint8_t*>(sorted[li])[place] = static_cast<uint8_t>(count);
        // (a block with more kept values than a residual can hold is not this format's input: nothing is written,
        // nor where the offsets are not those of this matrix: the words would land in other lists' room or behind all)
        int at = offsets[list];
        const bool fits = n <= kMaxListWords && n == offsets[list + 1] - at;
        if (L == 0)
            length[li] = fits && n > 64 ? n : 0;
        if (fits && n > 0 && n <= 64) {  // in row-major order
#pragma unroll
            for (int half = 0; half < 2; half++) {
#pragma unroll
                for (int r = 0; r < 8; r++)
                    image[r * 64 + L] = pairs[half * 8 + r];
                asm volatile("" ::: "memory");  // other lanes' words are read below
                unsigned natural[8];  // columns 2 L and 2 L + 1
#pragma unroll
                for (int r8 = 0; r8 < 8; r8++)
                    natural[r8] = image[r8 * 64 + (L ^ ((half * 8 + r8) << 2))];
#pragma unroll
                for (int r8 = 0; r8 < 8; r8++) {
                    const int r = half * 8 + r8;
                    const unsigned pair = natural[r8];
                    const bool lo = residual_kept(pair), hi = residual_kept(pair >> 16);
                    const uint64_t los = __ballot(lo), his = __ballot(hi);
                    const int place = lower_lanes(his, lower_lanes(los, at));
                    const unsigned address = r * 256 + (((L >> 2) ^ r) << 4) + (L & 3) * 4;
                    if (lo)
                        words[(size_t)place] = (pair & 0xffffu) | address << 16;
                    if (hi)
                        words[(size_t)place + (lo ? 1 : 0)] = pair >> 16 | (address + 2) << 16;
                    at += static_cast<int>(__popcll(los) + __popcll(his));
                }
                asm volatile("" ::: "memory");
            }
        }
    }
    __syncthreads();

    // 2. deal as many of the lists as there is room for (all of them, but for very dense ones), 3. write them.  With a list of
    // more than 256 words among them the images' room is the places' as well (ten lists of 1024 words), and values come from
    // memory one by one: a pass costs as much as its longest list, so what counts is how few there are (21504 x 7168, 300 / 700
    // words a list: 921 / 4834 us with the places' own room, 357 / 1265 with both; with 32 lists to a workgroup 660 / 3030).
    const int mine = L < kEmitLists ? length[L] : 0;
    const int through = offscan::wave_inclusive_sum(mine > 0 ? place_bytes(mine) : 0);  // room for lists 0 .. L
    const int more = __any(mine > 256) ? kImages : 0;  // bytes of the images' room that are the places'
    for (int first = 0, dealt = 0; first < kEmitLists;) {
        const uint64_t fit = __ballot(L < kEmitLists && through - dealt <= kPlaces + more);  // 0 .. last - 1: totals only grow
        const int last = __popcll(fit);
        const int at = through - place_bytes(mine) - dealt;
        if (w == 0 && L >= first && L < last && mine > 0) {
            const uint8_t* const counts = reinterpret_cast<const uint8_t*>(sorted[L]);
            if (mine > 256)  // (lane by lane: the form of a list's places goes by its own length)
                deal_long(sorted[L], mine, places + at);
            else if (__any(mine > 192))
                deal_laps<4>(counts, mine, places + at);
            else if (__any(mine > 128))
                deal_laps<3>(counts, mine, places + at);
            else
                deal_laps<2>(counts, mine, places + at);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kListsPerWave; i++) {
            const int li = i * kEmitWaves + w;
            const int n = __builtin_amdgcn_readlane(mine, li);
            if (li < first || li >= last || n == 0)
                continue;
            const uint8_t* const list_places = places + __builtin_amdgcn_readlane(at, li);
            uint32_t* const out = words + (size_t)offsets[list_of(i)];
            const unsigned ends = round_ends(n);
            int p = start[i];
            if (more) {
                const uint16_t* const src = block_of(list_of(i));
                unsigned lane = L;
                asm volatile("" : "+v"(lane));  // (or what is made of it is kept in registers from list to list)
                for (unsigned mask = kept[i]; mask; mask &= mask - 1, p++) {
                    const unsigned e = __builtin_ctz(mask), r = e / 2;
                    const unsigned value = src[(size_t)r * K + 2 * (lane ^ (r << 2)) + e % 2];
                    out[static_cast<unsigned>(place_of(list_places, p, n, ends))] = value | (e * 130u & 0xf02u) << 16 | lane << 18;
                }
                continue;
            }
            unsigned pairs[16];
            load_list(list_of(i), pairs);
#pragma unroll
            for (int r = 0; r < 16; r++)
                image[r * 64 + L] = pairs[r];
            asm volatile("" ::: "memory");
            for (unsigned mask = kept[i]; mask; mask &= mask - 1, p++) {
                const unsigned e = __builtin_ctz(mask);
                const unsigned address = (e * 130u & 0xf02u) | L * 4;  // (e / 2) * 256 + (e % 2) * 2: here as in the product's own image
                const unsigned value = *reinterpret_cast<const unsigned short*>(reinterpret_cast<const uint8_t*>(image) + address);
                out[static_cast<unsigned>(place_of(list_places, p, n, ends))] = value | address << 16;
            }
            asm volatile("" ::: "memory");
        }
        first = last;
        if (first < kEmitLists) {
            dealt = __builtin_amdgcn_readlane(through, first - 1);
            __syncthreads();  // the places are dealt afresh
        }
    }
}

}  // namespace

// A2: row-major M x K fp16 in device memory (M % 128 == 0, K % 128 == 0, checked by the caller).
// offsets: (M / 16) * (K / 128) + 1 ints; *longest: the longest list's length.
extern "C" int a24_launch_residual_offsets(void* stream, const void* A2, int M, int K, int* offsets, int* longest)
{
    const int units = K / 128;
    const long lists = static_cast<long>(M / 16) * units;
    if (lists < 1 || lists > 0x7ffffff0L)
        return static_cast<int>(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const long tasks = static_cast<long>(M / 16) * ((units + 3) / 4);
    hipLaunchKernelGGL(a24_residual_count_kernel, dim3((unsigned)((tasks + 3) / 4)), dim3(256), 0, s,
                       static_cast<const uint16_t*>(A2), K, units, (unsigned)tasks, offsets);
    hipLaunchKernelGGL(a24_residual_scan_kernel, dim3(1), dim3(offscan::kThreads), 0, s, offsets, lists, longest);
    return static_cast<int>(hipGetLastError());
}

// words: offsets[last] + 64 of them (the last 64 are zeroed).
extern "C" int a24_launch_residual_words(void* stream, const void* A2, int M, int K, const int* offsets, void* words)
{
    const int units = K / 128;
    const long lists = static_cast<long>(M / 16) * units;
    if (lists < 1 || lists > 0x7ffffff0L)
        return static_cast<int>(hipErrorInvalidValue);
    auto launch = [&](auto* kernel, int per_group) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((lists + per_group - 1) / per_group)), dim3(kEmitWaves * 64), 0,
                           static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(A2), K, units, lists, offsets,
                           static_cast<uint32_t*>(words));
    };
    if (lists >= kManyFrom)
        launch(a24_residual_emit_kernel<kManyLists>, kManyLists);
    else
        launch(a24_residual_emit_kernel<kFewLists>, kFewLists);
    return static_cast<int>(hipGetLastError());
}
