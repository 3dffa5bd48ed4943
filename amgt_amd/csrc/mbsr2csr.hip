// mBSR -> CSR export (counterpart of BSR2CSR_step1-3 with bsr2csr_get_ptr and
// bsr2csr_get_idx_val, csr_spgemm_device.c:1344-1440, 1501-1525).
//
// Columns come out ascending within a row: blocks are stored by ascending block
// column and the bits of a row nibble by ascending column.  The entries of a
// block row are the same range of both value arrays, so row pointers need no
// scan over the matrix: the first row starts at the block row's value pointer.
// A workgroup takes a tile of consecutive block rows (cut about every 768
// entries): a scan over its blocks of the four row counts of each bitmap
// (four 16-bit fields) gives every block its place in each row, the entries
// move through LDS into row order and leave coalesced.
#include "internal.hpp"

#include <algorithm>

namespace amgt {

namespace {

constexpr int kThreads = 256;
constexpr int kCap = 1024;       // entries (and blocks) of a tile held in LDS
constexpr int kMaxRows = 128;    // block rows of a tile, at most
// entries between the starts of two tiles, and for longer block rows
constexpr int kStart = 768, kStartLong = 512, kLongRow = 128;
constexpr int kPartBlocks = 768;  // blocks of a row exported in parts, more than

// first block row of every tile: block row br belongs to tile
// val_ptr[br] / start + br / rows
__global__ __launch_bounds__(kThreads) void k_export_cut(int32_t brow, int32_t start, int32_t rows,
                                                         int32_t ntiles,
                                                         const int32_t *__restrict__ val_ptr,
                                                         int32_t *__restrict__ tile_lo) {
    const int br = blockIdx.x * kThreads + threadIdx.x;
    if (br > brow) return;
    const int before = br > 0 ? val_ptr[br - 1] / start + (br - 1) / rows : -1;
    const int key = br < brow ? val_ptr[br] / start + br / rows : ntiles;
    for (int t = before + 1; t <= key; ++t) tile_lo[t] = br;
}

// row counts of a bitmap in four 16-bit fields
__device__ __forceinline__ uint32_t counts01(uint32_t m) {
    return uint32_t(__popc(m & 0xFu)) | uint32_t(__popc(m & 0xF0u)) << 16;
}
__device__ __forceinline__ uint32_t counts23(uint32_t m) {
    return uint32_t(__popc(m & 0xF00u)) | uint32_t(__popc(m & 0xF000u)) << 16;
}
__device__ __forceinline__ int field_sum(uint32_t a, uint32_t b) {
    return int((a & 0xFFFFu) + (a >> 16) + (b & 0xFFFFu) + (b >> 16));
}

// One wave exports part `part` of `parts` of block row br's blocks: 16 block slots x
// 4 rows per step, each lane's place from scans over the slots.  For the tiles the
// LDS form does not hold.
__device__ void export_row(int br, int part, int parts, int32_t nrows, const int32_t *__restrict__ blk_ptr,
                           const int32_t *__restrict__ blk_col,
                           const uint16_t *__restrict__ blk_map,
                           const int32_t *__restrict__ val_ptr, const double *__restrict__ val,
                           int32_t *__restrict__ I, int32_t *__restrict__ J,
                           double *__restrict__ A) {
    const int lane = threadIdx.x & 63;
    const int r = lane & 3, s = lane >> 2;
    const int p0 = blk_ptr[br], p1 = blk_ptr[br + 1];
    const int per = (p1 - p0 + 16 * parts - 1) / (16 * parts) * 16;
    const int j0 = min(p0 + part * per, p1), j1 = min(j0 + per, p1);
    int rowlen = 0, before = 0;  // entries of row r, of them before the part
#pragma unroll 4
    for (int j = p0 + s; j < p1; j += 16) {
        const int c = __popc((blk_map[j] >> (4 * r)) & 0xFu);
        rowlen += c;
        before += j < j0 ? c : 0;
    }
    for (int d = 4; d < 64; d <<= 1) {  // lane r: row r
        rowlen += __shfl_xor(rowlen, d);
        before += __shfl_xor(before, d);
    }
    int voff = val_ptr[br];
    int woff = voff;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int len = __shfl(rowlen, q);
        if (q < r) woff += len;
    }
    const int row = 4 * br + r;
    if (part == 0 && s == 0 && row < nrows) I[row] = woff;
    woff += before;
#pragma unroll
    for (int q = 0; q < 4; ++q) voff += __shfl(before, q);
    const uint32_t low = (1u << (4 * r)) - 1u;
    for (int jb = j0; jb < j1; jb += 16) {
        const int j = jb + s;
        uint32_t m = 0;
        int col = 0;
        if (j < j1) {
            m = blk_map[j];
            col = blk_col[j];
        }
        const uint32_t nib = (m >> (4 * r)) & 0xFu;
        const int cb = __popc(m);
        const int cn = __popc(nib);
        int ib = cb, in = cn;
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) {
            int tb = __shfl_up(ib, 4 * d);
            int tn = __shfl_up(in, 4 * d);
            if (s >= d) {
                ib += tb;
                in += tn;
            }
        }
        const int totb = __shfl(ib, 60 + r);
        const int totn = __shfl(in, 60 + r);
        int o = voff + (ib - cb) + __popc(m & low);
        int w = woff + (in - cn);
        if (row < nrows) {
            uint32_t t = nib;
            while (t) {
                const int c = __builtin_ctz(t);
                t &= t - 1u;
                J[w] = 4 * col + c;
                if (A) A[w] = val[o];
                ++w;
                ++o;
            }
        }
        voff += totb;
        woff += totn;
    }
}

__global__ __launch_bounds__(kThreads) void k_export_tile(
    int32_t nrows, int32_t brow, const int32_t *__restrict__ tile_lo,
    const int32_t *__restrict__ blk_ptr, const int32_t *__restrict__ blk_col,
    const uint16_t *__restrict__ blk_map, const int32_t *__restrict__ val_ptr,
    const double *__restrict__ val, int32_t *__restrict__ I, int32_t *__restrict__ J,
    double *__restrict__ A) {
    constexpr int NW = kThreads / 64, BPT = kCap / kThreads;
    __shared__ uint2 s_pre[kCap + 1];    // fields before block b; then the values in row order
    __shared__ int32_t s_bc[kCap];       // block columns
    __shared__ uint16_t s_map[kCap];
    __shared__ int32_t s_col[kCap];      // columns in row order
    __shared__ uint16_t s_to[kCap];      // place of the tile's p-th value
    __shared__ uint8_t s_rid[kCap];      // block row of a block
    __shared__ int s_bp[kMaxRows + 1];   // first blocks of the block rows
    __shared__ uint32_t s_w01[NW], s_w23[NW];
    double *const s_val = reinterpret_cast<double *>(s_pre);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int t0 = tile_lo[blockIdx.x], rows = tile_lo[blockIdx.x + 1] - t0;
    if (t0 + rows == brow && rows > 0 && tid == 0) I[nrows] = val_ptr[brow];
    if (rows <= 0) return;
    const int b0 = blk_ptr[t0], nb = blk_ptr[t0 + rows] - b0;
    const int base = val_ptr[t0], n = val_ptr[t0 + rows] - base;
    if (n > kCap || nb > kCap) {  // uniform
        // the last row, the only one that can be long, in a part per wave if it is (40000
        // rows of 100 entries, every eighth of 1100: 456 us by one wave, 220; each part
        // counts all bitmaps, which does not pay for rows of 600)
        const int parts = blk_ptr[t0 + rows] - blk_ptr[t0 + rows - 1] > kPartBlocks ? NW : 1;
        for (int k = w; k < rows - 1 + parts; k += NW) {
            const int r = min(k, rows - 1);
            export_row(t0 + r, k - r, r < rows - 1 ? 1 : parts, nrows, blk_ptr, blk_col, blk_map,
                       val_ptr, val, I, J, A);
        }
        return;
    }
    double v[BPT];  // the tile's values, wanted at the end
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
        const int p = tid + k * kThreads;
        v[k] = (A && p < n) ? val[base + p] : 0.0;
    }
    for (int b = tid; b < nb; b += kThreads) {
        s_map[b] = blk_map[b0 + b];
        s_bc[b] = blk_col[b0 + b];
    }
    for (int t = tid; t <= rows; t += kThreads) s_bp[t] = blk_ptr[t0 + t] - b0;
    __syncthreads();
    {  // the blocks' rows: a power of two of lanes per block row
        int lpr = kThreads;
        while (rows * lpr > kThreads) lpr >>= 1;  // rows <= kThreads / 2
        const int r = tid / lpr;
        if (r < rows)
            for (int b = s_bp[r] + tid % lpr; b < s_bp[r + 1]; b += lpr) s_rid[b] = uint8_t(r);
    }
    uint32_t m[BPT], a01 = 0, a23 = 0;
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
        m[k] = BPT * tid + k < nb ? uint32_t(s_map[BPT * tid + k]) : 0u;
        a01 += counts01(m[k]);
        a23 += counts23(m[k]);
    }
    const uint32_t i01 = uint32_t(wave_incl_sum(int(a01)));
    const uint32_t i23 = uint32_t(wave_incl_sum(int(a23)));
    if (lane == 63) {
        s_w01[w] = i01;
        s_w23[w] = i23;
    }
    __syncthreads();
    uint32_t e01 = i01 - a01, e23 = i23 - a23;
    for (int q = 0; q < w; ++q) {
        e01 += s_w01[q];
        e23 += s_w23[q];
    }
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
        s_pre[BPT * tid + k] = make_uint2(e01, e23);
        e01 += counts01(m[k]);
        e23 += counts23(m[k]);
    }
    if (tid == kThreads - 1) s_pre[kCap] = make_uint2(e01, e23);
    __syncthreads();
    // start of row r of the block row with blocks [f, l), within the tile
    auto row_start = [&](int f, int l, int r) {
        const uint2 pf = s_pre[f], pl = s_pre[l];
        const uint32_t d01 = pl.x - pf.x, d23 = pl.y - pf.y;
        return field_sum(pf.x, pf.y) + (r > 0 ? int(d01 & 0xFFFFu) : 0) +
               (r > 1 ? int(d01 >> 16) : 0) + (r > 2 ? int(d23 & 0xFFFFu) : 0);
    };
    for (int t = tid; t < 4 * rows; t += kThreads)
        if (4 * t0 + t < nrows)
            I[4 * t0 + t] = base + row_start(s_bp[t >> 2], s_bp[(t >> 2) + 1], t & 3);
    // four lanes per block, a row each
    for (int t = tid; t < 4 * nb; t += kThreads) {
        const int b = t >> 2, r = t & 3, br = s_rid[b], f = s_bp[br];
        const uint32_t mb = s_map[b], nib = (mb >> (4 * r)) & 0xFu;
        const uint2 pb = s_pre[b], pf = s_pre[f];
        const uint32_t q = (r & 2) ? pb.y - pf.y : pb.x - pf.x;
        int to = row_start(f, s_bp[br + 1], r) + int((r & 1) ? q >> 16 : q & 0xFFFFu);
        int src = field_sum(pb.x, pb.y) + __popc(mb & ((1u << (4 * r)) - 1u));
        const int c0 = 4 * s_bc[b];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (!((nib >> c) & 1u)) continue;
            s_to[src++] = uint16_t(to);
            s_col[to++] = c0 + c;
        }
    }
    __syncthreads();  // (the prefixes are read)
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
        const int p = tid + k * kThreads;
        if (p < n) s_val[s_to[p]] = v[k];
    }
    __syncthreads();
    for (int p = tid; p < n; p += kThreads) {
        J[base + p] = s_col[p];
        if (A) A[base + p] = s_val[p];
    }
}

__global__ void k_zero_one(int32_t *p) {
    if (threadIdx.x == 0) *p = 0;
}

}  // namespace

int mbsr_to_csr(const Mbsr &M, hipStream_t s, int64_t *nnz, int32_t **rowptr, int32_t **colidx,
                double **val) {
    *nnz = 0;
    *rowptr = nullptr;
    *colidx = nullptr;
    *val = nullptr;
    int32_t *I = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * (size_t(M.nrows) + 1), s));
    if (!I) {
        set_error("CSR export: row pointer allocation failed");
        return AMGT_ERR_ALLOC;
    }
    // nnz of the export equals the handle's nnz (sum of popcounts)
    const int64_t n = M.nnz;
    int32_t *J = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * size_t(n ? n : 1), s));
    double *A = nullptr;
    if (!M.pattern_only) A = static_cast<double *>(dev_alloc(sizeof(double) * size_t(n ? n : 1), s));
    int32_t *tile_lo = nullptr;
    // smaller tiles where there would be too few to fill the chip
    const int32_t full = n <= int64_t(kLongRow) * M.brow ? kStart : kStartLong;
    const int32_t start = std::max(64, std::min(full, int32_t(n / 2048)));
    const int32_t rows = std::max(4, std::min(kMaxRows, M.brow / 1024));
    const int32_t ntiles = M.brow > 0 ? int32_t(n / start) + M.brow / rows + 1 : 0;
    int st = (!J || (!M.pattern_only && !A)) ? AMGT_ERR_ALLOC : AMGT_OK;
    if (st != AMGT_OK) set_error("CSR export: allocation failed");
    if (st == AMGT_OK) st = tmp_alloc_t(&tile_lo, size_t(ntiles) + 1, s);
    if (st == AMGT_OK) {
        if (ntiles > 0) {
            hipLaunchKernelGGL(k_export_cut, dim3(unsigned(M.brow / kThreads + 1)), dim3(kThreads),
                               0, s, M.brow, start, rows, ntiles, M.val_ptr, tile_lo);
            hipLaunchKernelGGL(k_export_tile, dim3(unsigned(ntiles)), dim3(kThreads), 0, s, M.nrows,
                               M.brow, tile_lo, M.blk_ptr, M.blk_col, M.blk_map, M.val_ptr, M.val,
                               I, J, A);
        } else {
            hipLaunchKernelGGL(k_zero_one, dim3(1), dim3(64), 0, s, I);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            set_error(std::string("CSR export: ") + hipGetErrorString(e));
            st = AMGT_ERR_HIP;
        }
    }
    tmp_free(tile_lo, s);
    if (st != AMGT_OK) {
        dev_free(I, s);
        dev_free(J, s);
        dev_free(A, s);
        return st;
    }
    *nnz = n;
    *rowptr = I;
    *colidx = J;
    *val = A;
    return AMGT_OK;
}

}  // namespace amgt
