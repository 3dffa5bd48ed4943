// CSR -> mBSR conversion (counterpart of CSR2BSR_GPU, csr_matvec_device.c:1201-1267).
//
// Design: a block row's entries (the up-to-4 CSR rows 4br..4br+3) are sorted by
// the 32-bit key (block column << 4 | r*4 + c).  Sorted order IS the compressed
// value order of the mBSR layout (blocks ascending, bits ascending), so values
// land at val[I[4br] + rank] directly, block columns come from the key heads
// and bitmaps from OR-ing the low nibble of keys that share a head.  Sorting
// makes the conversion independent of the CSR column order (HYPRE rows start
// with the diagonal), unlike the reference's windowed bitmask that assumes
// sorted columns once ncols > 32768 (csr_matvec_device.c:701-722).
//
// A workgroup converts a tile of consecutive block rows (cut by a pass over the
// row pointers so that a tile starts about every 768 entries and holds at most
// kTileCap): rank sort of each row's keys in LDS, coalesced loads and stores,
// the tile's blocks packed.  Then one workgroup scans the tiles' block counts
// and the packed blocks are copied to their places.  Tiles over the capacity (a
// block row of more than 256 entries) are left to a second pass: the rows before
// the last as a tile, the last by itself (as a tile up to kTileCap entries, a
// workgroup of 1024 threads up to 8192).
// Larger block rows return AMGT_ERR_UNSUPPORTED.
#include "internal.hpp"
#include "rowpass.hpp"

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

namespace amgt {

namespace {

constexpr uint32_t kPadKey = 0xFFFFFFFFu;

enum : int { kErrDup = 1, kErrCol = 2, kErrBig = 4, kErrPtr = 8 };

constexpr int kTileThreads = 256;
constexpr int kTileCap = 1024;   // entries of a tile
constexpr int kTileRows = 128;   // block rows of a tile, at most
constexpr int kRowCap = 8192;    // entries of a block row, at most
// entries between the starts of two tiles: the tile's last block row must fit
// behind them (257 or 513 entries); 768 for block rows of at most 128 on average
constexpr int kTileStart = 768, kTileStartLong = 512, kTileLongRow = 128;
// Block rows over this many entries: places by binary search of their CSR rows
// where those ascend, instead of counting all keys (few rows of 700 beside 7-pt
// ones: the tile took 75 us, the latency of one workgroup's counting).
constexpr int kLongRank = 192;
// CSR rows over this many entries per lane are numbered by the whole workgroup
constexpr int kFillTurns = 32, kFillList = kTileCap / kFillTurns;

// row pointer i, kept inside [0, nnz]: the pointers are verified only with the
// readback after the sorts, so no load may follow a wrong one out of the arrays
__device__ __forceinline__ int entry_at(const int32_t *__restrict__ I, int i, int nnz) {
    const int v = I[i];
    return v < 0 ? 0 : (v > nnz ? nnz : v);
}

// Key of CSR entry p in block row starting at row r0.
__device__ __forceinline__ uint32_t entry_key(int p, int r0, int nrows, int ncols,
                                              const int32_t *__restrict__ I,
                                              const int32_t *__restrict__ J, int *err) {
    int c = J[p];
    if (c < 0 || c >= ncols) {
        *err |= kErrCol;
        c = 0;
    }
    int r = (p >= I[min(r0 + 1, nrows)]) + (p >= I[min(r0 + 2, nrows)]) +
            (p >= I[min(r0 + 3, nrows)]);
    return (uint32_t(c >> 2) << 4) | uint32_t(r << 2) | uint32_t(c & 3);
}

// First block row of every tile: block row br belongs to tile I[4 br] / start +
// br / rows (start entries, rows block rows: a new tile begins where either
// count passes a multiple).  A tile thus holds at most `rows` block rows and
// start - 1 entries before its last one, whatever the row lengths: with a fixed
// number of block rows per tile the regular runs of long rows of an
// interpolation operator (24 entries per block row where the average is 13.5)
// passed the capacity.  Every tile gets a value even for row pointers that do
// not ascend, which are reported.
__global__ __launch_bounds__(kTileThreads) void k_conv_cut(int32_t nrows, int32_t brow,
                                                           int32_t nnz, int32_t start,
                                                           int32_t rows, int32_t ntiles,
                                                           const int32_t *__restrict__ I,
                                                           int32_t *__restrict__ tile_lo,
                                                           int32_t *__restrict__ err) {
    const int br = blockIdx.x * kTileThreads + threadIdx.x;
    int bad = 0;
    for (int r = 4 * br; br < brow && r < min(4 * br + 4, nrows); ++r) bad |= I[r + 1] < I[r];
    bad = __syncthreads_or(bad);
    // err[0] collects the errors of the listed tiles, err[1 + k] those seen here
    if (threadIdx.x == 0) err[1 + blockIdx.x] = bad ? kErrPtr : 0;
    if (br == 0) err[0] = 0;
    if (br > brow) return;
    const int before = br > 0 ? entry_at(I, 4 * (br - 1), nnz) / start + (br - 1) / rows : -1;
    const int key = br < brow ? entry_at(I, 4 * br, nnz) / start + br / rows : ntiles;
    for (int t = before + 1; t <= key; ++t) tile_lo[t] = br;
}

// What a tile leaves behind: its block count, the largest block count of its
// rows and their squares' sum, error bits, whether it exceeds the capacity.
struct TilePart {
    int32_t blocks;
    uint32_t mx_flags;  // largest block count << 8 | over << 4 | error bits
    unsigned long long sumsq;
    static constexpr uint32_t kOver = 16u;
};
struct ConvTotals {
    int32_t nblk, max_blocks, err, over;
    unsigned long long sumsq;
};

// A tile (kList: a tile over the capacity, in two parts: workgroup 2 k takes the
// rows of tile tiles[k] before its last, at most start - 1 entries, workgroup
// 2 k + 1 the last one alone, if it fits, written to its own slot with its block
// count in rel).  Every entry's place in its block row is the number of smaller
// keys there, counted over an LDS copy of the row's keys (four per read; rows
// padded to a multiple of four with keys above all others).  The blocks of the
// tile go to tmp_col / tmp_map from the tile's first entry on, packed; rel = a
// block row's first block within the tile.
// The entries of a tile are contiguous in the CSR and in the output, so loads
// and stores are coalesced and all lanes work; a wave per block row (28 entries
// of 64 lanes on 7-pt 128^3, a pass over per-row slots to pack the blocks) took
// 241 + 126 us there against the copy rate's 67.
template <bool kList>
__global__ __launch_bounds__(kTileThreads) void k_conv_tile(
    int32_t nrows, int32_t ncols, int32_t nnz, const int32_t *__restrict__ I,
    const int32_t *__restrict__ J, const double *__restrict__ A,
    const int32_t *__restrict__ tile_lo, const int32_t *__restrict__ tiles,
    double *__restrict__ val, int32_t *__restrict__ tmp_col,
    uint16_t *__restrict__ tmp_map, int32_t *__restrict__ rel,
    TilePart *__restrict__ parts, int values_only) {
    constexpr int NW = kTileThreads / 64, EPT = kTileCap / kTileThreads;
    constexpr int kPad = kTileCap + 3 * kTileRows;
    __shared__ __align__(16) uint32_t s_key[kPad];     // padded rows; then the block bitmaps
    __shared__ __align__(16) uint32_t s_sorted[kTileCap];
    __shared__ uint16_t s_rid[kTileCap];               // CSR row within the tile
    __shared__ int s_I[4 * kTileRows + 1];             // row starts within the tile
    __shared__ int s_ps[kTileRows + 1];                // padded block row starts
    __shared__ int s_first[kTileRows + 1];
    __shared__ int s_wt[NW], s_err, s_longest, s_descends;
    __shared__ int s_list[kFillList], s_nlist;         // CSR rows filled by all threads
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int t0, rows, part;  // first block row, block rows, index in parts
    if constexpr (kList) {
        part = tiles[blockIdx.x >> 1];
        t0 = tile_lo[part];
        rows = tile_lo[part + 1] - t0 - 1;
        if (blockIdx.x & 1) {
            t0 += rows;
            rows = 1;
        }
        if (rows <= 0 || rows > kTileRows) return;
    } else {
        part = blockIdx.x;
        t0 = tile_lo[part];
        rows = tile_lo[part + 1] - t0;
        if (rows <= 0 || rows > kTileRows) {  // (over kTileRows: bad row pointers)
            if (tid == 0) parts[part] = TilePart{0, 0u, 0ull};
            return;
        }
    }
    const int nr = min(4 * rows, nrows - 4 * t0);  // CSR rows
    const int base = entry_at(I, 4 * t0, nnz);
    const int n = entry_at(I, 4 * t0 + nr, nnz) - base;
    if (n < 0 || n > kTileCap) {  // uniform
        if (!kList && tid == 0) {
            const int last = base + n - entry_at(I, 4 * (t0 + rows - 1), nnz);
            parts[part] =
                TilePart{0, TilePart::kOver | (last > kRowCap ? uint32_t(kErrBig) : 0u), 0ull};
        }
        return;  // (kList: k_sort_block's row)
    }
    int cj[EPT];
    double ca[EPT];
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        const int e = tid + k * kTileThreads;
        cj[k] = e < n ? J[base + e] : 0;
        ca[k] = (A && e < n) ? A[base + e] : 0.0;
    }
    for (int t = tid; t <= nr; t += kTileThreads) {
        const int v = entry_at(I, 4 * t0 + t, nnz) - base;
        s_I[t] = v < 0 ? 0 : (v > n ? n : v);
    }
    for (int t = tid; t < kPad; t += kTileThreads) s_key[t] = kPadKey;
    for (int t = tid; t < kTileCap; t += kTileThreads) {
        s_sorted[t] = kPadKey;
        s_rid[t] = 0;
    }
    if (tid == 0) s_err = s_descends = s_nlist = 0;
    __syncthreads();
    if (w == 0) {  // padded starts of the block rows, two per lane
        int len[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int r = 2 * lane + u;
            len[u] = 0;
            if (r < rows) len[u] = (max(s_I[min(4 * r + 4, nr)] - s_I[4 * r], 0) + 3) & ~3;
        }
        const int incl = wave_incl_sum(len[0] + len[1]);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int at = incl - len[1] - (u == 0 ? len[0] : 0);
            if (2 * lane + u <= rows) s_ps[2 * lane + u] = at;
        }
        const int longest = wave_incl_max(max(len[0], len[1]));
        if (lane == 63 && rows == kTileRows) s_ps[rows] = incl;
        if (lane == 63) s_longest = longest;
    }
    {  // the entries' rows: a power of two of lanes per row
        int lpr = kTileThreads;
        while (lpr > 1 && nr * lpr > kTileThreads) lpr >>= 1;
        for (int row = tid / lpr; row < nr; row += kTileThreads / lpr) {
            if (s_I[row + 1] - s_I[row] > kFillTurns * lpr) {
                if (tid % lpr == 0) {
                    const int at = atomicAdd(&s_nlist, 1);
                    if (at < kFillList) s_list[at] = row;  // (always, for ascending pointers)
                }
                continue;
            }
            for (int e = s_I[row] + tid % lpr; e < s_I[row + 1]; e += lpr) s_rid[e] = uint16_t(row);
        }
    }
    __syncthreads();
    if (s_nlist > 0) {  // uniform
        for (int k = 0; k < min(s_nlist, kFillList); ++k) {
            const int row = s_list[k];
            for (int e = s_I[row] + tid; e < s_I[row + 1]; e += kTileThreads) s_rid[e] = uint16_t(row);
        }
        __syncthreads();
    }
    uint32_t key[EPT];
    int rid[EPT];
    int err = 0;
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        const int e = tid + k * kTileThreads;
        key[k] = kPadKey;
        rid[k] = 0;
        if (e < n) {
            int c = cj[k];
            if (c < 0 || c >= ncols) {
                err |= kErrCol;
                c = 0;
            }
            rid[k] = s_rid[e];
            const int br = rid[k] >> 2;
            key[k] = (uint32_t(c >> 2) << 4) | uint32_t((rid[k] & 3) << 2) | uint32_t(c & 3);
            const int at = s_ps[br] + (e - s_I[4 * br]);
            if (at >= 0 && at < kPad) s_key[at] = key[k];  // (always, for ascending pointers)
        }
    }
    __syncthreads();
    // long block rows: whether their CSR rows ascend from the second entry on
    // (ascending columns, or the diagonal first)
    if (s_longest > kLongRank) {  // uniform
#pragma unroll
        for (int k = 0; k < EPT; ++k) {
            const int e = tid + k * kTileThreads;
            if (e >= n || e - 1 <= s_I[rid[k]]) continue;
            const int br = rid[k] >> 2, at = s_ps[br] + (e - s_I[4 * br]);
            if (s_ps[br + 1] - s_ps[br] > kLongRank && at > 0 && at < kPad && s_key[at - 1] >= key[k])
                s_descends = 1;
        }
        __syncthreads();
    }
    const bool search = s_longest > kLongRank && s_descends == 0;
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        const int e = tid + k * kTileThreads;
        if (e >= n) continue;
        const int br = rid[k] >> 2;
        int rank = 0;
        int j1 = min(s_ps[br + 1], kPad);
        if (search && j1 - s_ps[br] > kLongRank) {
            // the four CSR rows' smaller keys: the first, and a binary search of the rest
            const int off = s_ps[br] - s_I[4 * br];
            int lo[4], len[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b = s_I[min(4 * br + q, nr)];
                len[q] = s_I[min(4 * br + q + 1, nr)] - b - 1;
                lo[q] = b + 1 + off;
                if (len[q] >= 0) rank += s_key[min(unsigned(b + off), unsigned(kPad - 1))] < key[k];
                rank -= lo[q];
            }
            while (max(max(len[0], len[1]), max(len[2], len[3])) > 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (len[q] <= 0) continue;
                    const int half = len[q] >> 1;
                    const bool up = s_key[min(unsigned(lo[q] + half), unsigned(kPad - 1))] < key[k];
                    lo[q] = up ? lo[q] + half + 1 : lo[q];
                    len[q] = up ? len[q] - half - 1 : half;
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) rank += lo[q];
            j1 = 0;  // (no counting below)
        }
        auto below = [&](const uint4 &kk) {
            return (kk.x < key[k] ? 1 : 0) + (kk.y < key[k] ? 1 : 0) + (kk.z < key[k] ? 1 : 0) +
                   (kk.w < key[k] ? 1 : 0);
        };
        int j = s_ps[br];
        for (; j + 32 <= j1; j += 32) {  // long rows: the reads' latency once per eight
            uint4 kk[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) kk[u] = *reinterpret_cast<const uint4 *>(&s_key[j + 4 * u]);
#pragma unroll
            for (int u = 0; u < 8; ++u) rank += below(kk[u]);
        }
        for (; j < j1; j += 4) rank += below(*reinterpret_cast<const uint4 *>(&s_key[j]));
        const int to = min(s_I[4 * br] + rank, n - 1);
        s_sorted[to] = key[k];
        // places within the entry's own block row: a wave's stores stay within a
        // few cache lines
        if (A) val[base + to] = ca[k];
    }
    __syncthreads();
    // four consecutive sorted entries per thread; equal keys (duplicate
    // entries) share a place and leave a hole
    const int p0 = EPT * tid;
    uint32_t sk[EPT];
    int sb[EPT], head[EPT], nh = 0;
    uint32_t pk = (p0 > 0 && p0 < n) ? s_sorted[p0 - 1] : kPadKey;
    int pb = (p0 > 0 && p0 < n) ? s_rid[p0 - 1] >> 2 : -1;
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        const bool in = p0 + k < n;
        sk[k] = in ? s_sorted[p0 + k] : kPadKey;
        sb[k] = in ? s_rid[p0 + k] >> 2 : -1;
        if (in && sk[k] == kPadKey) err |= kErrDup;
        head[k] = in && (sb[k] != pb || (sk[k] >> 4) != (pk >> 4)) ? 1 : 0;
        nh += head[k];
        pk = sk[k];
        pb = sb[k];
    }
    if (err) atomicOr(&s_err, err);
    if (values_only) {
        __syncthreads();
        if (tid == 0) {
            if constexpr (kList) {
                if (s_err) atomicOr(&parts[part].mx_flags, uint32_t(s_err));
            } else {
                parts[part] = TilePart{0, uint32_t(s_err), 0ull};
            }
        }
        return;
    }
    const int incl = wave_incl_sum(nh);
    if (lane == 63) s_wt[w] = incl;
    for (int t = tid; t < kTileCap; t += kTileThreads) s_key[t] = 0u;  // the bitmaps
    __syncthreads();
    int slot = incl - nh - 1, total = 0;  // the block of the entry before this thread's
#pragma unroll
    for (int q = 0; q < NW; ++q) {
        if (q < w) slot += s_wt[q];
        total += s_wt[q];
    }
    uint32_t map = 0;
    int prevb = (p0 > 0 && p0 < n) ? s_rid[p0 - 1] >> 2 : -1;
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
        if (p0 + k >= n) break;
        if (head[k]) {
            if (map) atomicOr(&s_key[slot], map);
            map = 0;
            ++slot;
            tmp_col[base + slot] = int32_t(sk[k] >> 4);
            if (sb[k] != prevb) s_first[sb[k]] = slot;
        }
        map |= 1u << (sk[k] & 15u);
        prevb = sb[k];
    }
    if (map) atomicOr(&s_key[slot], map);
    __syncthreads();
    for (int t = tid; t < total; t += kTileThreads) tmp_map[base + t] = uint16_t(s_key[t]);
    if (w == 0) {
        // a row's first block; an empty row's is the next entry's
        auto first_of = [&](int br) {
            if (br >= rows) return total;
            const int lo = s_I[4 * br];
            return lo < n ? s_first[s_rid[lo] >> 2] : total;
        };
        if (kList && (blockIdx.x & 1)) {
            if (lane == 0) {
                rel[t0] = total;
                if (s_err) atomicOr(&parts[part].mx_flags, uint32_t(s_err));
            }
        } else {
            unsigned long long sq = 0ull;
            int mx = 0;
            const int f0 = first_of(2 * lane), f1 = first_of(2 * lane + 1),
                      f2 = first_of(2 * lane + 2);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int c = max(u == 0 ? f1 - f0 : f2 - f1, 0);
                if (2 * lane + u >= rows) continue;
                rel[t0 + 2 * lane + u] = u == 0 ? f0 : f1;
                sq += static_cast<unsigned long long>(c) * unsigned(c);
                mx = max(mx, c);
            }
            for (int d = 32; d > 0; d >>= 1) sq += __shfl_xor(sq, d);
            mx = wave_incl_max(mx);
            if (lane == 63) {
                const uint32_t flags = uint32_t(mx) << 8 | uint32_t(s_err);
                if constexpr (kList) {  // (the last row's workgroup adds its errors)
                    parts[part].blocks = total;
                    parts[part].sumsq = sq;
                    atomicOr(&parts[part].mx_flags, flags);
                } else {
                    parts[part] = TilePart{total, flags, sq};
                }
            }
        }
    }
}

// ---- block rows of kTileCap + 1 to CAP entries: the last row of a listed tile
// (no other row of a tile can be that long), a workgroup each.  Where the CSR rows
// ascend, as they mostly do, they are four sorted runs, and an entry's place is
// its place in its run plus the smaller keys of the other three, by binary search;
// otherwise a bitonic sort.  Bound by the latency of the steps in one workgroup
// (bitonic: 78 barriers for 4096 keys).  1024 threads for every length: a second
// launch of 256 threads for up to 2048 entries follows instead of overlapping
// (few rows of 1000 to 8000 entries, whole conversion: 525 against 441 us with the
// bitonic sort, 327 with ranks; 1250 block rows of 1200 entries 318 -> 190, 225
// of 3600 216 -> 160).  One workgroup per listed tile, not per row of it: those
// rows took 5500 us when most workgroups were empty.
template <int THREADS, int CAP>
__global__ __launch_bounds__(THREADS) void k_sort_block(
    int32_t nrows, int32_t ncols, int32_t nnz, const int32_t *__restrict__ I,
    const int32_t *__restrict__ J, const double *__restrict__ A,
    const int32_t *__restrict__ tile_lo, const int32_t *__restrict__ tiles,
    double *__restrict__ val, int32_t *__restrict__ tmp_col,
    uint16_t *__restrict__ tmp_map, int32_t *__restrict__ blk_cnt, int32_t *__restrict__ err_out,
    int values_only) {
    __shared__ uint32_t s_key[CAP];
    __shared__ int32_t s_aux[CAP];  // source index, then block rank
    __shared__ int32_t s_wave_tot[THREADS / 64];
    __shared__ int s_err, s_descends;
    constexpr int EPT = CAP / THREADS;
    const int t = threadIdx.x;
    const int br = tile_lo[tiles[blockIdx.x] + 1] - 1;
    if (br < 0) return;
    const int r0 = 4 * br;
    const int s = entry_at(I, r0, nnz);
    const int n = entry_at(I, min(r0 + 4, nrows), nnz) - s;
    if (n <= kTileCap || n > CAP) return;  // k_conv_tile's row (or refused before)
    int np = 64;
    while (np < n) np <<= 1;
    if (t == 0) s_err = s_descends = 0;
    int err = 0;
    for (int i = t; i < np; i += THREADS) {
        if (i < n) {
            s_key[i] = entry_key(s + i, r0, nrows, ncols, I, J, &err);
            s_aux[i] = s + i;
        } else {
            s_key[i] = kPadKey;
            s_aux[i] = 0;
        }
    }
    __syncthreads();
    // ascending: every key above the one before it in its CSR row (also no duplicates)
    for (int i = t; i < n; i += THREADS) {
        if (i == 0) continue;
        const uint32_t a = s_key[i - 1], b = s_key[i];
        if (((a ^ b) & 12u) == 0u && a >= b) s_descends = 1;
    }
    __syncthreads();
    if (!s_descends) {
        int run[5];
#pragma unroll
        for (int q = 0; q < 5; ++q)
            run[q] = min(max(entry_at(I, min(r0 + q, nrows), nnz) - s, 0), n);
        uint32_t key[EPT];
        int rank[EPT];
#pragma unroll
        for (int u = 0; u < EPT; ++u) {
            const int i = t + u * THREADS;
            key[u] = i < n ? s_key[i] : 0u;
            rank[u] = i;
            const int own = int(key[u] >> 2) & 3;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // i counts the runs before its own in full: take back their keys
                // above, and add the smaller keys of the runs after it
                if (i >= n || q == own) continue;
                int lo = run[q], hi = run[q + 1];
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (s_key[mid] < key[u]) lo = mid + 1;
                    else hi = mid;
                }
                rank[u] += q < own ? lo - run[q + 1] : lo - run[q];
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < EPT; ++u) {
            const int i = t + u * THREADS;
            if (i < n) {
                s_key[rank[u]] = key[u];
                s_aux[rank[u]] = s + i;
            }
        }
        __syncthreads();
    }
    for (int k = 2; s_descends && k <= np; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = t; i < np; i += THREADS) {
                int p = i ^ j;
                if (p > i) {
                    bool up = (i & k) == 0;
                    uint32_t a = s_key[i], b = s_key[p];
                    if ((a > b) == up) {
                        s_key[i] = b;
                        s_key[p] = a;
                        int x = s_aux[i];
                        s_aux[i] = s_aux[p];
                        s_aux[p] = x;
                    }
                }
            }
            __syncthreads();
        }
    }
    for (int i = t; i < n; i += THREADS) {
        if (A) val[s + i] = A[s_aux[i]];
        if (i > 0 && s_key[i] == s_key[i - 1]) err |= kErrDup;
    }
    if (err) atomicOr(&s_err, err);
    __syncthreads();
    if (!values_only) {
        // block ranks: inclusive scan of head flags over the sorted keys,
        // processed in chunks of THREADS with a running carry
        int carry = 0;
        const int lane = t & 63, wv = t >> 6;
        for (int base = 0; base < n; base += THREADS) {
            int i = base + t;
            int head = 0;
            if (i < n) head = (i == 0) || ((s_key[i] >> 4) != (s_key[i - 1] >> 4));
            uint64_t bal = __ballot(head);
            uint64_t le = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
            int incl = __popcll(bal & le);
            if (lane == 63) s_wave_tot[wv] = __popcll(bal);
            __syncthreads();
            int before = 0, total = 0;
            for (int q = 0; q < THREADS / 64; ++q) {
                int v = s_wave_tot[q];
                if (q < wv) before += v;
                total += v;
            }
            if (i < n) s_aux[i] = carry + before + incl - 1;  // block rank
            carry += total;
            __syncthreads();
        }
        // heads write block column and bitmap (<= 16 entries per block)
        for (int i = t; i < n; i += THREADS) {
            uint32_t key = s_key[i];
            bool head = (i == 0) || ((s_key[i - 1] >> 4) != (key >> 4));
            if (head) {
                uint32_t map = 0;
                for (int d = 0; d < 16 && i + d < n; ++d) {
                    uint32_t kk = s_key[i + d];
                    if ((kk >> 4) != (key >> 4)) break;
                    map |= 1u << (kk & 15u);
                }
                int rank = s_aux[i];
                tmp_col[s + rank] = int32_t(key >> 4);
                tmp_map[s + rank] = uint16_t(map);
            }
        }
        if (t == 0) blk_cnt[br] = carry;
    }
    if (t == 0 && s_err) atomicOr(err_out, s_err);
}

// Adds the last row of every listed tile (its block count in rel) to the tile's
// part; rel then holds the row's first block within the tile.
__global__ __launch_bounds__(kTileThreads) void k_conv_list_sum(
    int32_t ntiles, const int32_t *__restrict__ tile_lo, const int32_t *__restrict__ tiles,
    int32_t *__restrict__ rel, TilePart *__restrict__ parts) {
    const int k = blockIdx.x * kTileThreads + threadIdx.x;
    if (k >= ntiles) return;
    const int t = tiles[k], br = tile_lo[t + 1] - 1;
    TilePart p = parts[t];
    const uint32_t c = uint32_t(rel[br]);
    rel[br] = p.blocks;
    p.blocks += int32_t(c);
    p.sumsq += static_cast<unsigned long long>(c) * c;
    p.mx_flags = max(p.mx_flags >> 8, c) << 8 | (p.mx_flags & 0xffu);
    parts[t] = p;
}

// One workgroup: the tiles' first blocks, the totals and the list of the tiles
// over the capacity (in no order); four consecutive tiles per thread and step.
constexpr int kFinThreads = 1024;
__global__ __launch_bounds__(kFinThreads) void k_conv_finish(int32_t ntiles, int32_t nerr,
                                                             const TilePart *__restrict__ parts,
                                                             const int32_t *__restrict__ err_in,
                                                             int32_t *__restrict__ first,
                                                             int32_t *__restrict__ tiles,
                                                             ConvTotals *__restrict__ tot) {
    constexpr int NW = kFinThreads / 64;
    __shared__ int s_w[NW], s_mx[NW], s_err[NW], s_over;
    __shared__ unsigned long long s_sq[NW];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int run = 0, mx = 0, err = 0;
    unsigned long long sq = 0ull;
    if (threadIdx.x == 0) s_over = 0;
    for (int k = threadIdx.x; k < nerr; k += kFinThreads) err |= err_in[k];
    __syncthreads();
    for (int g = 0; g < ntiles; g += 4 * kFinThreads) {
        const int t = g + 4 * int(threadIdx.x);
        TilePart p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) p[u] = t + u < ntiles ? parts[t + u] : TilePart{};
        int sum = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            sum += p[u].blocks;
            mx = max(mx, int(p[u].mx_flags >> 8));
            err |= int(p[u].mx_flags & 15u);
            if (p[u].mx_flags & TilePart::kOver) tiles[atomicAdd(&s_over, 1)] = t + u;
            sq += p[u].sumsq;
        }
        const int incl = wave_incl_sum(sum);
        __syncthreads();  // the previous step's totals are read
        if (lane == 63) s_w[w] = incl;
        __syncthreads();
        int at = run + incl - sum, all = 0;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            if (q < w) at += s_w[q];
            all += s_w[q];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (t + u < ntiles) first[t + u] = at;
            at += p[u].blocks;
        }
        run += all;
    }
    for (int d = 32; d > 0; d >>= 1) {
        mx = max(mx, __shfl_xor(mx, d));
        err |= __shfl_xor(err, d);
        sq += __shfl_xor(sq, d);
    }
    if (lane == 0) {
        s_mx[w] = mx;
        s_err[w] = err;
        s_sq[w] = sq;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        ConvTotals r{run, 0, 0, s_over, 0ull};
        for (int q = 0; q < NW; ++q) {
            r.max_blocks = max(r.max_blocks, s_mx[q]);
            r.err |= s_err[q];
            r.sumsq += s_sq[q];
        }
        *tot = r;
    }
}

// row pointers of a matrix without rows
__global__ void k_empty_ptrs(int32_t *blk_ptr, int32_t *val_ptr) {
    if (threadIdx.x == 0) blk_ptr[0] = val_ptr[0] = 0;
}

// The tiles' blocks to their places, block and value row pointers.
__global__ __launch_bounds__(kTileThreads) void k_conv_pack(
    int32_t nrows, int32_t brow, int32_t nblk, const int32_t *__restrict__ I,
    const int32_t *__restrict__ tile_lo, const TilePart *__restrict__ parts, const int32_t *__restrict__ first,
    const int32_t *__restrict__ rel, const int32_t *__restrict__ tmp_col,
    const uint16_t *__restrict__ tmp_map, int32_t *__restrict__ blk_ptr,
    int32_t *__restrict__ blk_col, uint16_t *__restrict__ blk_map,
    int32_t *__restrict__ val_ptr) {
    const int t = blockIdx.x, t0 = tile_lo[t], rows = tile_lo[t + 1] - t0;
    if (rows <= 0) return;
    const int to = first[t];
    if (threadIdx.x < unsigned(rows)) {  // rows <= kTileRows < kTileThreads
        blk_ptr[t0 + threadIdx.x] = to + rel[t0 + threadIdx.x];
        val_ptr[t0 + threadIdx.x] = I[4 * (t0 + threadIdx.x)];
    }
    if (t0 + rows == brow && threadIdx.x == 0) {
        blk_ptr[brow] = nblk;
        val_ptr[brow] = I[nrows];
    }
    const int blocks = parts[t].blocks;
    // a listed tile's last row has its blocks in its own slot
    const bool over = (parts[t].mx_flags & TilePart::kOver) != 0u;
    const int body = over ? rel[t0 + rows - 1] : blocks;
    const int from = I[4 * t0], from_last = I[4 * (t0 + rows - 1)] - body;
    for (int k = threadIdx.x; k < blocks; k += kTileThreads) {
        const int at = (k < body ? from : from_last) + k;
        blk_col[to + k] = tmp_col[at];
        blk_map[to + k] = tmp_map[at];
    }
}

}  // namespace

int row_stats_launch(const int32_t *blk_ptr, int32_t brow, RowStats *d_stats, hipStream_t s) {
    rowpass::Part *parts = nullptr;
    AMGT_TRY(tmp_alloc_t(&parts, size_t(rowpass::groups(brow)) + 1, s));
    const int st = rowpass::count(brow, rowpass::BlockDiff{blk_ptr}, INT64_MAX, INT64_MAX, parts,
                                  d_stats, s);
    tmp_free(parts, s);
    return st;
}

double stand_from(const RowStats &h, int64_t nblk, int32_t brow) {
    // sqrt(sum (c - avg)^2 / brow) with sum (c - avg)^2 = (brow*sum c^2 - nblk^2) / brow,
    // the numerator exact in 128-bit integers (the reference sums doubles with
    // atomics and takes sqrtf, csr_matvec_device.c:1245-1249)
    if (brow <= 0) return 0.0;
    const __int128 num = static_cast<__int128>(h.sumsq) * brow - static_cast<__int128>(nblk) * nblk;
    const double var = double(num) / (double(brow) * double(brow));
    return var > 0.0 ? std::sqrt(var) : 0.0;
}

namespace {

// Device scratch of one conversion: one block (each block of the pool costs a
// lookup and, when it is given back, an event).
struct ConvWork {
    int32_t ntiles = 0, nerr = 0;
    TilePart *parts = nullptr;
    ConvTotals *tot = nullptr;
    int32_t *first = nullptr, *rel = nullptr, *tmp_col = nullptr, *tiles = nullptr;
    int32_t *tile_lo = nullptr, *err = nullptr;
    uint16_t *tmp_map = nullptr;
    char *block = nullptr;
    hipStream_t s = nullptr;
    ~ConvWork() { tmp_free(block, s); }
    int alloc(size_t brow, size_t nnz, bool blocks) {
        size_t bytes = 0;
        auto place = [&](auto *&p, size_t n) {
            if (block) p = reinterpret_cast<std::decay_t<decltype(p)>>(block + bytes);
            bytes += (n * sizeof(*p) + 255) & ~size_t(255);
        };
        auto all = [&] {
            bytes = 0;
            place(parts, size_t(ntiles));
            place(tot, 1);
            place(first, size_t(ntiles));
            place(tiles, size_t(ntiles));
            place(tile_lo, size_t(ntiles) + 1);
            place(err, size_t(nerr));
            if (blocks) {
                place(rel, brow);
                place(tmp_col, nnz);
                place(tmp_map, nnz);
            }
        };
        all();
        AMGT_TRY(tmp_alloc_t(&block, bytes, s));
        all();
        return AMGT_OK;
    }
};

// Sorts every tile (values, and unless values_only the packed blocks) and reads
// the totals back with rowptr[0] and rowptr[nrows], which are verified: one
// synchronisation unless a tile exceeds the capacity.
int sort_tiles(int32_t nrows, int32_t ncols, int64_t nnz, const int32_t *I, const int32_t *J,
               const double *A, int32_t brow, double *val, int values_only, ConvWork &w,
               ConvTotals *ht, hipStream_t s) {
    w.s = s;
    // smaller tiles where there would be too few to fill the chip
    const int32_t nz = int32_t(nnz);
    const int32_t full = nnz <= int64_t(kTileLongRow) * brow ? kTileStart : kTileStartLong;
    const int32_t start = std::max(64, std::min(full, nz / 2048));
    const int32_t rows = std::max(4, std::min(kTileRows, brow / 1024));
    w.ntiles = brow > 0 ? nz / start + brow / rows + 1 : 0;
    const unsigned cuts = unsigned(brow / kTileThreads + 1);
    w.nerr = w.ntiles > 0 ? int32_t(cuts) + 1 : 0;
    AMGT_TRY(w.alloc(size_t(brow), size_t(nnz), !values_only));
    if (w.ntiles > 0) {
        hipLaunchKernelGGL(k_conv_cut, dim3(cuts), dim3(kTileThreads), 0, s, nrows, brow, nz, start, rows, w.ntiles, I, w.tile_lo, w.err);
        hipLaunchKernelGGL((k_conv_tile<false>), dim3(unsigned(w.ntiles)), dim3(kTileThreads), 0,
                           s, nrows, ncols, nz, I, J, A, w.tile_lo,
                           static_cast<const int32_t *>(nullptr), val, w.tmp_col, w.tmp_map, w.rel,
                           w.parts, values_only);
    }
    auto totals = [&](int32_t *ends) -> int {
        hipLaunchKernelGGL(k_conv_finish, dim3(1), dim3(kFinThreads), 0, s, w.ntiles, w.nerr, w.parts,
                           w.err, w.first, w.tiles, w.tot);
        AMGT_HIP(hipGetLastError());
        const Readback rb[3] = {{ht, w.tot, sizeof(ConvTotals)},
                                {&ends[0], I, sizeof(int32_t)},
                                {&ends[1], I + nrows, sizeof(int32_t)}};
        return readback(rb, 3, s);
    };
    int32_t ends[2] = {0, 0};
    AMGT_TRY(totals(ends));
    if (ends[0] != 0 || int64_t(ends[1]) != nnz) {
        set_error("CSR->mBSR: rowptr[0] must be 0 and rowptr[nrows] must equal nnz");
        return AMGT_ERR_INPUT;
    }
    if (ht->err & kErrPtr) {
        set_error("CSR->mBSR: row pointers must ascend");
        return AMGT_ERR_INPUT;
    }
    if (ht->err & kErrBig) {
        set_error("CSR->mBSR: a block row has more than 8192 entries (4 rows with > 2048 "
                  "nonzeros on average); this build does not convert such rows");
        return AMGT_ERR_UNSUPPORTED;
    }
    if (ht->over > 0) {  // the tiles over the capacity, their last rows by themselves
        const unsigned nt = unsigned(ht->over);
        hipLaunchKernelGGL((k_conv_tile<true>), dim3(2 * nt), dim3(kTileThreads), 0, s, nrows,
                           ncols, nz, I, J, A, w.tile_lo, w.tiles, val, w.tmp_col, w.tmp_map,
                           w.rel, w.parts, values_only);
        hipLaunchKernelGGL((k_sort_block<1024, kRowCap>), dim3(nt), dim3(1024), 0, s, nrows, ncols,
                           nz, I, J, A, w.tile_lo, w.tiles, val, w.tmp_col, w.tmp_map, w.rel,
                           w.err, values_only);
        if (values_only) {  // (nothing to read back; the caller's arrays are read until here)
            AMGT_HIP(hipGetLastError());
            AMGT_HIP(hipStreamSynchronize(s));
            return AMGT_OK;
        }
        hipLaunchKernelGGL(k_conv_list_sum, dim3((nt + kTileThreads - 1) / kTileThreads),
                           dim3(kTileThreads), 0, s, ht->over, w.tile_lo, w.tiles, w.rel, w.parts);
        AMGT_HIP(hipGetLastError());
        AMGT_TRY(totals(ends));
    }
    return AMGT_OK;
}

}  // namespace

// (its last kernel may be pending on return)
static int convert(int32_t nrows, int32_t ncols, int64_t nnz, const int32_t *rowptr,
                   const int32_t *colidx, const double *A, hipStream_t s, Mbsr *out) {
    Mbsr &m = *out;
    m = Mbsr();
    m.nrows = nrows;
    m.ncols = ncols;
    m.brow = (nrows + 3) / 4;
    m.bcol = (ncols + 3) / 4;
    m.nnz = nnz;
    // a matrix without nonzeros has (empty) values even when no value pointer is given
    m.pattern_only = (A == nullptr && nnz > 0);
    if (nnz >= (int64_t(1) << 31)) {
        set_error("CSR->mBSR: nnz exceeds int32 indexing");
        return AMGT_ERR_UNSUPPORTED;
    }
    if (ncols > (1 << 30) - 8) {
        // block column << 4 must stay below the padding key 0xFFFFFFFF
        set_error("CSR->mBSR: ncols > 2^30 - 8 does not fit the 32-bit sort key");
        return AMGT_ERR_UNSUPPORTED;
    }
    m.blk_ptr = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * (size_t(m.brow) + 1), s));
    m.val_ptr = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * (size_t(m.brow) + 1), s));
    if (!m.blk_ptr || !m.val_ptr) {
        set_error("CSR->mBSR: allocation failed");
        return AMGT_ERR_ALLOC;
    }
    if (!m.pattern_only) {
        m.val = static_cast<double *>(dev_alloc(sizeof(double) * size_t(nnz ? nnz : 1), s));
        if (!m.val) {
            set_error("CSR->mBSR: value allocation failed");
            return AMGT_ERR_ALLOC;
        }
    }
    ConvWork w;
    ConvTotals ht{};
    AMGT_TRY(sort_tiles(nrows, ncols, nnz, rowptr, colidx, A, m.brow, m.val, 0, w, &ht, s));
    if (ht.err & kErrCol) {
        set_error("CSR->mBSR: column index out of range");
        return AMGT_ERR_INPUT;
    }
    if (ht.err & kErrDup) {
        set_error("CSR->mBSR: duplicate (row, col) entry");
        return AMGT_ERR_INPUT;
    }
    const int32_t nblk = ht.nblk;
    m.nblk = nblk;
    m.blk_col = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * size_t(nblk ? nblk : 1), s));
    m.blk_map = static_cast<uint16_t *>(dev_alloc(sizeof(uint16_t) * size_t(nblk ? nblk : 1), s));
    if (!m.blk_col || !m.blk_map) {
        set_error("CSR->mBSR: block allocation failed");
        return AMGT_ERR_ALLOC;
    }
    if (w.ntiles > 0)
        hipLaunchKernelGGL(k_conv_pack, dim3(unsigned(w.ntiles)), dim3(kTileThreads), 0, s, nrows,
                           m.brow, nblk, rowptr, w.tile_lo, w.parts, w.first, w.rel, w.tmp_col,
                           w.tmp_map, m.blk_ptr, m.blk_col, m.blk_map, m.val_ptr);
    else
        hipLaunchKernelGGL(k_empty_ptrs, dim3(1), dim3(64), 0, s, m.blk_ptr, m.val_ptr);
    AMGT_HIP(hipGetLastError());
    m.stand = stand_from(RowStats{{0, 0, 0}, ht.max_blocks, ht.sumsq}, nblk, m.brow);
    m.avg_nnz = nblk ? double(nnz) / double(nblk) : 0.0;
    m.max_row_blocks = ht.max_blocks;
    m.spmv_kernel = default_spmv_kernel(m);
    return AMGT_OK;
}

int csr_to_mbsr(int32_t nrows, int32_t ncols, int64_t nnz, const int32_t *rowptr,
                const int32_t *colidx, const double *A, hipStream_t s, Mbsr *out) {
    AMGT_TRY(convert(nrows, ncols, nnz, rowptr, colidx, A, s, out));
    // k_conv_pack reads the caller's row pointers and writes the handle's arrays:
    // wait, so that the caller may free or change its arrays and use the handle on
    // any stream (no stream of another user would know of this one's work)
    AMGT_HIP(hipStreamSynchronize(s));
    return AMGT_OK;
}

int mbsr_refresh_values(Mbsr *Ap, const int32_t *rowptr, const int32_t *colidx,
                        const double *A, hipStream_t s) {
    Mbsr &m = *Ap;
    if (m.pattern_only || !m.val) {
        m.val = static_cast<double *>(dev_alloc(sizeof(double) * size_t(m.nnz ? m.nnz : 1), s));
        if (!m.val) {
            set_error("value allocation failed");
            return AMGT_ERR_ALLOC;
        }
        m.pattern_only = false;
    }
    ConvWork w;
    ConvTotals ht{};
    const int st = sort_tiles(m.nrows, m.ncols, m.nnz, rowptr, colidx, A, m.brow, m.val, 1, w, &ht, s);
    // low-precision copies and the transpose are stale now
    dev_free(m.val32, s);
    m.val32 = nullptr;
    dev_free(m.val16, s);
    m.val16 = nullptr;
    m.half_fits = -1;
    if (m.trans) {
        mbsr_release(m.trans, s);
        delete m.trans;
        m.trans = nullptr;
    }
    return st;
}

}  // namespace amgt
