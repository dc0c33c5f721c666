// Host-side Tiled-CSL encoder: dense row-major fp16 weight -> packed
// (value,index) words + TileOffsets, bit-exact with the reference's
// InitSparseMatrixA_API (csrc/SpMM_API.cu:241-438) but organised differently:
//
//   * The reference simulates 32 stacks and runs a 32-way arg-max for every
//     word it emits.  Its pop order has a closed form: with bank sizes s[b],
//     the sequence of pops is "for level = max(s) down to 1, for bank b = 0..31
//     in order, if s[b] >= level take element level-1 of bank b" (the largest
//     stack with the lowest id always wins, so equal-height stacks are drained
//     in id order, one layer at a time).  The emission order (tail drawn first,
//     main part after, both written last-in first-out) is then pure index
//     arithmetic on that sequence; see emit_tile().
//   * Tiles are independent once their output offsets are known, so the work is
//     two passes (count -> prefix sum -> encode) spread over a small thread pool
//     by tile row.  The reference is single threaded.
//
// Plain C++ and SSE2 (part of every x86-64, the only hosts this card has): no HIP here.
#include <emmintrin.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "tiled_csl_format.h"

namespace tcsl {

namespace {

// The reference keeps an element when fabs(float(v)) > 0 (csrc/SpMM_API.cu:262):
// +-0 and NaN are dropped, subnormals and infinities are kept.
inline bool kept(uint16_t h)
{
    const uint16_t mag = h & 0x7fffu;
    return mag != 0 && mag <= 0x7c00u;
}

int pool_size(long work_items)
{
    int n = 0;
    if (const char* e = std::getenv("SPMM_ENCODE_THREADS"))
        n = std::atoi(e);
    if (n <= 0) {
        n = static_cast<int>(std::thread::hardware_concurrency());
        if (n <= 0)
            n = 1;
        if (n > 16)
            n = 16;
    }
    if (n > work_items)
        n = static_cast<int>(work_items);
    return n < 1 ? 1 : n;
}

// One bit per element of a tile's row: kept or not.
inline uint64_t kept_mask(const uint16_t* row)
{
    const __m128i magnitude = _mm_set1_epi16(0x7fff), past_inf = _mm_set1_epi16(0x7c01), zero = _mm_setzero_si128();
    uint64_t mask = 0;
    for (int i = 0; i < kTileCols; i += 16) {
        const __m128i a = _mm_and_si128(_mm_loadu_si128(reinterpret_cast<const __m128i*>(row + i)), magnitude);
        const __m128i b = _mm_and_si128(_mm_loadu_si128(reinterpret_cast<const __m128i*>(row + i + 8)), magnitude);
        const __m128i ka = _mm_and_si128(_mm_cmpgt_epi16(a, zero), _mm_cmpgt_epi16(past_inf, a));
        const __m128i kb = _mm_and_si128(_mm_cmpgt_epi16(b, zero), _mm_cmpgt_epi16(past_inf, b));
        mask |= static_cast<uint64_t>(static_cast<uint32_t>(_mm_movemask_epi8(_mm_packs_epi16(ka, kb)))) << i;
    }
    return mask;
}

int count_tile(const uint16_t* tile, int ld)
{
    int nz = 0;
    for (int m = 0; m < kTileRows; m++)
        nz += __builtin_popcountll(kept_mask(tile + static_cast<size_t>(m) * ld));
    return nz;
}

constexpr int kChunkTiles = 16;  // tiles of a tile row that one thread encodes at a time

// Room for the words of a caller that takes it as it comes, to be given back with free(); *user, a void*, is
// the room.  Large rooms are aligned to huge pages and the system is asked for them: the first touch of
// 41 MB in 4 KiB pages costs 10000 faults.
void* allocate_words(void* user, size_t bytes)
{
    constexpr size_t kHuge = size_t(2) << 20;
    void** const room = static_cast<void**>(user);
    if (bytes < 2 * kHuge) {
        *room = std::malloc(bytes ? bytes : 1);
    } else if (posix_memalign(room, kHuge, bytes) == 0) {
        (void)madvise(*room, bytes / kHuge * kHuge, MADV_HUGEPAGE);  // a hint: refused, nothing is lost
    } else {
        *room = nullptr;
    }
    return *room;
}

constexpr int kLevels = kTileRows * kTileCols / kBanks + kVec;  // 256 positions per bank + pads
struct TileScratch {
    uint32_t words[kLevels * kBanks];  // a bank's element number l in row kLevels - 1 - l: levels upwards run backwards
    uint32_t next[kBanks];             // where each bank's next element goes
    int16_t size[kBanks];
    uint64_t row[kTileRows];           // kept_mask of every row
};

// First position of bank b that is not kept, in row order; -1: none.
int first_zero_of(const TileScratch& ws, int b)
{
    for (int m = 0; m < kTileRows; m++) {
        const int n = (2 * b) ^ ((m & 7) << 3);  // columns n, n + 1 are the bank's pair
        const unsigned gone = ~static_cast<unsigned>(ws.row[m] >> n) & 3u;
        if (gone)
            return m * kTileCols + 2 * b + ((gone & 1u) ? 0 : 1);
    }
    return -1;
}

// Encodes one tile into dst; returns the number of words written (a multiple of 4).
//
// Bound by the instructions per kept element, so rows are tested 16 elements at a time and only set bits are
// visited; the banks' elements lie level by level, the first level last, so that the levels that all banks
// reach are the pop sequence as they lie (37 of some 66 levels at 80 %, most of the words) and only those above
// them are moved together; and the emission order's groups of 32 x 4 words are transposed 4 x 4 words at a time.
// (7168 x 7168 on 16 threads, the whole call from Python with no copy of the words: 2.4 ms at 80 %, 3.1 at 60 %; with a
// list per bank, every word moved into the pop sequence: 2.9 and 4.2; element by element, in two sets of
// threads, with the copy: 15.1 at 80 %.)
int emit_tile(const uint16_t* tile, int ld, uint32_t* dst, TileScratch& ws)
{
    for (int b = 0; b < kBanks; b++)
        ws.next[b] = (kLevels - 1) * kBanks + b;
    int count = 0;
    for (int m = 0; m < kTileRows; m++) {
        const uint16_t* row = tile + static_cast<size_t>(m) * ld;
        __builtin_prefetch(row + kTileCols);  // the next tile's part of the row: two lines
        __builtin_prefetch(row + kTileCols + 32);
        const int flip = (m & 7) << 3;
        const uint64_t mask = kept_mask(row);
        ws.row[m] = mask;
        count += __builtin_popcountll(mask);
        for (uint64_t rest = mask; rest; rest &= rest - 1) {
            const int n = __builtin_ctzll(rest);
            const int swz = n ^ flip;  // swizzled column (csrc/SpMM_API.cu:332-333)
            const int b = swz >> 1;    // 4-byte LDS bank of that position (:334)
            const uint32_t at = ws.next[b];
            ws.next[b] = at - kBanks;
            ws.words[at] = pack_item(row[n], m * kTileCols + swz);
        }
    }
    if (count == 0)
        return 0;
    for (int b = 0; b < kBanks; b++)
        ws.size[b] = static_cast<int16_t>(kLevels - 1 - static_cast<int>(ws.next[b] / kBanks));
    // zero padding to a multiple of 4, each pad on the currently smallest bank (:352-365)
    const int pad = (kVec - count % kVec) % kVec;
    for (int p = 0; p < pad; p++) {
        int b = 0;
        for (int i = 1; i < kBanks; i++)
            if (ws.size[i] < ws.size[b])
                b = i;
        // the smallest bank of a tile that needs padding always has a zero position
        ws.words[ws.next[b]] = pack_item(0, first_zero_of(ws, b));
        ws.next[b] -= kBanks;
        ws.size[b]++;
        count++;
    }
    // pop sequence, closed form: levels from the tallest down, banks in order.  The levels above the smallest bank's
    // are moved up against those below, from the lowest one on: a word never moves over one that is still to move.
    int top = 0, full = kLevels;
    for (int b = 0; b < kBanks; b++) {
        top = std::max<int>(top, ws.size[b]);
        full = std::min<int>(full, ws.size[b]);
    }
    uint32_t* seq = ws.words + (kLevels - full) * kBanks;
    const __m128i* const sizes = reinterpret_cast<const __m128i*>(ws.size);
    for (int level = full + 1; level <= top; level++) {
        const __m128i under = _mm_set1_epi16(static_cast<short>(level - 1));
        auto taller = [&](int i) { return _mm_cmpgt_epi16(_mm_loadu_si128(sizes + i), under); };
        uint32_t banks = static_cast<uint32_t>(_mm_movemask_epi8(_mm_packs_epi16(taller(0), taller(1))))
                         | static_cast<uint32_t>(_mm_movemask_epi8(_mm_packs_epi16(taller(2), taller(3)))) << 16;
        const uint32_t* const from = ws.words + (kLevels - level) * kBanks;
        while (banks) {  // from the last bank on
            const int b = 31 - __builtin_clz(banks);
            *--seq = from[b];
            banks ^= 1u << b;
        }
    }
    // emission (:379-424).  V vectors = R full groups of 32 lanes + `rem` lanes.
    // The first 4*rem pops fill the tail, lane b receiving pops v*rem + b; the
    // rest fill the main part, lane b receiving pops 4*rem + k*32 + b, k = 0..4R-1.
    // Both are written out in reverse arrival order, main part first.
    const int vecs = count / kVec;
    const int R = vecs / kGroup, rem = vecs % kGroup;
    const uint32_t* mainq = seq + kVec * rem;
    for (int r = 0; r < R; r++) {
        const uint32_t* const group = mainq + (kVec * (R - r) - kVec) * kGroup;  // arrivals k = 4(R-r)-4 .. +3
        for (int b = 0; b < kGroup; b += 4) {
            auto arrival = [&](int k) { return _mm_loadu_si128(reinterpret_cast<const __m128i*>(group + k * kGroup + b)); };
            const __m128i v0 = arrival(3), v1 = arrival(2), v2 = arrival(1), v3 = arrival(0);
            const __m128i lo01 = _mm_unpacklo_epi32(v0, v1), hi01 = _mm_unpackhi_epi32(v0, v1);
            const __m128i lo23 = _mm_unpacklo_epi32(v2, v3), hi23 = _mm_unpackhi_epi32(v2, v3);
            __m128i* const to = reinterpret_cast<__m128i*>(dst + (r * kGroup + b) * kVec);
            _mm_storeu_si128(to, _mm_unpacklo_epi64(lo01, lo23));
            _mm_storeu_si128(to + 1, _mm_unpackhi_epi64(lo01, lo23));
            _mm_storeu_si128(to + 2, _mm_unpacklo_epi64(hi01, hi23));
            _mm_storeu_si128(to + 3, _mm_unpackhi_epi64(hi01, hi23));
        }
    }
    uint32_t* tail = dst + R * kGroup * kVec;
    for (int b = 0; b < rem; b++)
        for (int v = 0; v < kVec; v++)
            tail[b * kVec + v] = seq[(kVec - 1 - v) * rem + b];
    return count;
}

// One tile without reordering (csrc/SpMM_API.cu:514-551): kept elements in scan order, and the
// first `pads` elements of the scan that are not kept, with whatever bits they hold.
int emit_tile_noreorder(const uint16_t* tile, int ld, uint32_t* dst, int pads)
{
    int w = 0;
    for (int m = 0; m < kTileRows; m++) {
        const uint16_t* row = tile + static_cast<size_t>(m) * ld;
        const int flip = (m & 7) << 3;
        for (int n = 0; n < kTileCols; n++) {
            const uint16_t v = row[n];
            if (kept(v)) {
                dst[w++] = pack_item(v, m * kTileCols + (n ^ flip));
            } else if (pads > 0) {
                pads--;
                dst[w++] = pack_item(v, m * kTileCols + (n ^ flip));
            }
        }
    }
    return w;
}

bool bad_shape(int M, int K)
{
    return M <= 0 || K <= 0 || M % kTileRows != 0 || K % kTileCols != 0;
}

int encode_impl(const uint16_t* A, int M, int K, uint32_t** items_out, int** offsets_out, bool reorder)
{
    if (!A || !items_out || !offsets_out)
        return kErrNullPointer;
    if (bad_shape(M, K))
        return kErrBadShape;
    const size_t entries = static_cast<size_t>(M / kTileRows) * (K / kTileCols) + kOffsetPadding;
    int* const offs = static_cast<int*>(std::malloc(entries * sizeof(int)));
    if (!offs)
        return kErrNoMemory;
    void* items = nullptr;
    const int rc = encode_into(A, M, K, reorder, allocate_words, &items, offs);
    if (rc < 0) {
        std::free(items);
        std::free(offs);
        return rc;
    }
    *items_out = static_cast<uint32_t*>(items);
    *offsets_out = offs;
    return rc;
}

}  // namespace

int encode(const uint16_t* A, int M, int K, uint32_t** items_out, int** offsets_out)
{
    return encode_impl(A, M, K, items_out, offsets_out, true);
}

int encode_noreorder(const uint16_t* A, int M, int K, uint32_t** items_out, int** offsets_out)
{
    return encode_impl(A, M, K, items_out, offsets_out, false);
}

int encode_into(const uint16_t* A, int M, int K, bool reorder, void* (*allocate)(void* user, size_t bytes), void* user, int* offs)
{
    if (!A || !allocate || !offs)
        return kErrNullPointer;
    if (bad_shape(M, K))
        return kErrBadShape;
    const int tr = M / kTileRows, tc = K / kTileCols;
    const long ntiles = static_cast<long>(tr) * tc;

    // One set of threads for both passes (making threads costs about as much as counting a few tile
    // rows): counts, a meeting at which the caller's thread adds them up and asks for the room, words.
    uint32_t* items = nullptr;
    int rc = 0;
    std::atomic<bool> ok{true};
    std::atomic<long> next_row{0}, next_chunk{0};
    std::mutex mu;
    std::condition_variable all_in, met;
    const long chunks_per_row = (tc + kChunkTiles - 1) / kChunkTiles, chunks = tr * chunks_per_row;
    const int threads = pool_size(chunks);
    int started = threads, arrived = 0;
    bool ready = false;
    auto add_up = [&]() {  // under mu: exclusive, and every count is in
        ready = true;
        offs[0] = 0;
        long total_vecs = 0;
        for (long t = 0; t < ntiles; t++) {
            total_vecs += offs[t + 1];
            if (total_vecs > INT32_MAX) {
                rc = kErrTooLarge;
                return;
            }
            offs[t + 1] = static_cast<int>(total_vecs);
        }
        offs[ntiles + 1] = static_cast<int>(total_vecs);  // trailing empty tile (:433-435)
        items = static_cast<uint32_t*>(allocate(user, static_cast<size_t>(total_vecs) * kVec * sizeof(uint32_t)));
        if (!items)
            rc = kErrNoMemory;
    };
    auto work = [&](bool caller) {
        // pass 1: padded word count of every tile, stored in offs[t + 1]; whole rows, in memory order
        for (long i; (i = next_row.fetch_add(1)) < tr;) {
            int* const counts = offs + i * tc + 1;
            std::fill(counts, counts + tc, 0);
            for (int m = 0; m < kTileRows; m++) {
                const uint16_t* row = A + (static_cast<size_t>(i) * kTileRows + m) * K;
                for (int j = 0; j < tc; j++)
                    counts[j] += __builtin_popcountll(kept_mask(row + static_cast<size_t>(j) * kTileCols));
            }
            for (int j = 0; j < tc; j++)
                counts[j] = (counts[j] + kVec - 1) / kVec;
        }
        {
            std::unique_lock<std::mutex> lock(mu);
            arrived++;
            if (caller) {
                all_in.wait(lock, [&] { return arrived == started; });
                add_up();
                met.notify_all();
            } else {
                if (arrived == started)
                    all_in.notify_one();
                met.wait(lock, [&] { return ready; });
            }
            if (rc != 0)
                return;
        }
        // pass 2: every tile into its slot
        TileScratch* ws = new (std::nothrow) TileScratch;
        if (!ws) {
            ok = false;
            return;
        }
        // The chunks that are encoded at the same time are a share apart: threads next to each other would all fault on
        // the same huge page of new memory, and each clear one for it (words of 7168 x 7168 at 80 %: 2.2 ms, now 1.8).
        const long share = (chunks + threads - 1) / threads;
        for (long taken; (taken = next_chunk.fetch_add(1)) < share * threads;) {
            const long c = taken % threads * share + taken / threads;
            if (c >= chunks)
                continue;
            const long i = c / chunks_per_row;
            const int j0 = static_cast<int>(c % chunks_per_row) * kChunkTiles, j1 = std::min(j0 + kChunkTiles, tc);
            for (int j = j0; j < j1; j++) {
                const long t = i * tc + j;
                const uint16_t* tile = A + static_cast<size_t>(i) * kTileRows * K + static_cast<size_t>(j) * kTileCols;
                uint32_t* dst = items + static_cast<size_t>(offs[t]) * kVec;
                int n;
                if (reorder) {
                    n = emit_tile(tile, K, dst, *ws);
                } else {
                    const int nz = count_tile(tile, K);
                    n = emit_tile_noreorder(tile, K, dst, (kVec - nz % kVec) % kVec);
                }
                if (n != (offs[t + 1] - offs[t]) * kVec)
                    ok = false;
            }
        }
        delete ws;
    };
    std::vector<std::thread> pool;
    try {
        pool.reserve(threads - 1);
        for (int t = 1; t < threads; t++)
            pool.emplace_back(work, false);
    } catch (...) {  // fewer threads than wanted: go on with those that there are
        std::lock_guard<std::mutex> lock(mu);
        started = static_cast<int>(pool.size()) + 1;
    }
    work(true);
    for (auto& th : pool)
        th.join();
    if (rc == 0 && !ok)
        rc = kErrNoMemory;
    return rc != 0 ? rc : static_cast<int>(ntiles + kOffsetPadding);
}

int encode_file(const char* dense, int M, int K, const char* nz_path, const char* off_path, const char* sizes_path)
{
    if (!dense || !nz_path || !off_path || !sizes_path)
        return kErrNullPointer;
    if (bad_shape(M, K))
        return kErrBadShape;
    const size_t bytes = static_cast<size_t>(M) * K * sizeof(uint16_t);
    std::vector<uint16_t> host(static_cast<size_t>(M) * K);
    std::ifstream in(dense, std::ios::in | std::ios::binary);
    if (!in.is_open()) {
        std::fprintf(stderr, "file %s cannot be opened, loadDataArrayFromBin fails. \n", dense);
        return kErrFile;
    }
    in.read(reinterpret_cast<char*>(host.data()), static_cast<std::streamsize>(bytes));
    const size_t got = static_cast<size_t>(in.gcount());
    if (got != bytes) {
        std::fprintf(stderr, "file %s only has %zu, but request %zu, loading DenseMatrix fails! \n", dense, got, bytes);
        return kErrFile;
    }
    in.close();

    uint32_t* items = nullptr;
    int* offs = nullptr;
    const int num_offsets = encode(host.data(), M, K, &items, &offs);
    if (num_offsets < 0)
        return num_offsets;
    const int nnz = offs[num_offsets - 1] * kVec;

    std::ofstream out_sizes(sizes_path, std::ios::out | std::ios::binary);
    std::ofstream out_nz(nz_path, std::ios::out | std::ios::binary);
    std::ofstream out_off(off_path, std::ios::out | std::ios::binary);
    int rc = 0;
    if (!out_sizes.is_open() || !out_nz.is_open() || !out_off.is_open()) {
        std::fprintf(stderr, "GenSparseMatrixBinFile() ERROR: file %s, %s, or %s cannot be opened or created. \n",
                     sizes_path, nz_path, off_path);
        rc = kErrFile;
    } else {
        // int32 NNZ then int32 NumOffsets (csrc/SpMM_API.cu:1613-1615)
        out_sizes.write(reinterpret_cast<const char*>(&nnz), sizeof(int));
        out_sizes.write(reinterpret_cast<const char*>(&num_offsets), sizeof(int));
        out_nz.write(reinterpret_cast<const char*>(items), static_cast<std::streamsize>(sizeof(uint32_t)) * nnz);
        out_off.write(reinterpret_cast<const char*>(offs), static_cast<std::streamsize>(sizeof(int)) * num_offsets);
        // a short write may only show when the buffers are flushed: close first, then look
        out_sizes.close();
        out_nz.close();
        out_off.close();
        if (out_sizes.fail() || out_nz.fail() || out_off.fail())
            rc = kErrFile;
    }
    std::free(items);
    std::free(offs);
    return rc;
}

}  // namespace tcsl
