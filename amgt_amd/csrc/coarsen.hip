// BoomerAMG setup on the device, one process: strength of connection, PMIS
// coarsening and extended+i interpolation (with max-elements truncation) on
// CSR operators.
//
// Counterparts: hypre_BoomerAMGCreateSDevice (par_strength_device.c:34),
// hypre_BoomerAMGCoarsenPMISDevice (par_coarsen_device.c:30),
// hypre_BoomerAMGBuildExtPIInterpDevice (par_lr_interp_device.c:991) and
// hypre_BoomerAMGInterpTruncationDevice (par_interp_trunc_device.c:731).  The
// results follow HYPRE's host algorithms on one process (par_strength.c:75,
// par_coarsen.c:2101, par_lr_interp.c:1025, par_csr_matrix.c:2866 with
// qsort.c:395), which the reference's own regression outputs pin, so the
// device hierarchy equals the CPU one entry for entry:
//  * S: strong columns in row order, no diagonal;
//  * PMIS measures |S^T row| + hypre_Rand() from seed 2747 (the Park-Miller
//    stream jumped to each row's draw), the independent set of each pass taken
//    exactly as the host loop leaves it;
//  * P rows in the host's discovery order, weights accumulated in the host's
//    order with contraction off (no fused multiply-add), truncated rows
//    ordered by the host's quicksort.
// The diagonal of a row is found by column (HYPRE keeps it first; exports of
// the mBSR handles have ascending columns).
#include "internal.hpp"
#include "rowpass.hpp"

#include <algorithm>
#include <vector>

namespace amgt {

namespace {

constexpr int kThreads = 256;
// extended+i rows of 257 to 512 entries take the wave kernel on levels of at most
// kWaveMaxRows rows: at 74 KB of LDS two waves fit a CU, worth it only when the
// thread kernel would leave the chip idle behind a few long serial rows (300000
// rows of 400: 639 ms against 420 by threads).  Shorter ones take it on any level
// (thread / wave kernel, ms: 300000 rows of 80 23.0 / 11.2, of 120 47 / 18, of 200 119 /
// 89; 2.2 M of 70 111 / 68).
constexpr int kWaveMaxRows = 1 << 18;

inline unsigned grid_of(int64_t n) { return unsigned((n + kThreads - 1) / kThreads); }

// position of a_ii in row i, or -1: the first entry (HYPRE's diagonal-first
// rows), else a binary search (rows with ascending columns, the exports of
// mBSR handles), else a scan.  A search can only return an entry of column i,
// and a CSR row holds at most one, so any row order gives the same answer.
__device__ __forceinline__ int64_t diag_pos(const int32_t *__restrict__ I,
                                            const int32_t *__restrict__ J, int i) {
    const int64_t b = I[i], e = I[i + 1];
    if (b == e) return -1;
    if (J[b] == i) return b;
    int64_t lo = b, hi = e - 1;
    while (lo <= hi) {
        const int64_t mid = (lo + hi) >> 1;
        const int c = J[mid];
        if (c == i) return mid;
        if (c < i) lo = mid + 1; else hi = mid - 1;
    }
    for (int64_t p = b; p < e; ++p)
        if (J[p] == i) return p;
    return -1;
}

// ---- strength (par_strength.c:75-528, one function) ---------------------------
// A thread per row; the entries of the workgroup's `per` rows are staged in LDS
// with coalesced loads, as many rows at a time as fit (7-pt: all 256, 1792 of
// kStageEntries), and the strong columns leave through LDS; a row that does not
// fit by itself is walked in memory.  (Threads walking their rows in memory: 81 us
// to count and 188 us to fill on 7-pt 128^3, 176 MB read by each; whole calls
// 360 -> 196 us, 27-pt 64^3 547 -> 154.)  A workgroup's parts follow each other, so
// small levels give it fewer rows (125-pt 30^3: 248 us walked, 961 with 256 rows a
// workgroup, 142 with 16).
constexpr int kStageEntries = 2048;

#pragma clang fp contract(off)
// row entries [b, e) of j / a; strong columns to out (kFill), their number
// returned; d: the diagonal's position or -1
template <bool kFill, typename P>
__device__ __forceinline__ int strong_entries(const int32_t *j, const double *a, P b, P e, P d,
                                              double theta, double max_row_sum, int32_t *out) {
    const double diag = d >= 0 ? a[d] : 0.0;
    double row_scale = 0.0, row_sum = diag;
    // eight entries' loads at a time, ahead of the chains of sums and of the stores
    // (which could alias them)
    constexpr int U = 8;
    for (P p0 = b; p0 < e; p0 += U) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = a[p0 + u < e ? p0 + u : p0];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool on = p0 + u < e && p0 + u != d;
            const bool beyond = diag < 0 ? v[u] > row_scale : v[u] < row_scale;
            row_scale = on && beyond ? v[u] : row_scale;
            row_sum = on ? row_sum + v[u] : row_sum;
        }
    }
    int c = 0;
    // a row too dominant by the row-sum test keeps only weak dependencies
    if (!(fabs(row_sum) > fabs(diag) * max_row_sum && max_row_sum < 1.0)) {
        const double thr = theta * row_scale;
        for (P p0 = b; p0 < e; p0 += U) {
            double v[U];
            int32_t k[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const P p = p0 + u < e ? p0 + u : p0;
                v[u] = a[p];
                k[u] = kFill ? j[p] : 0;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool weak = diag < 0 ? (v[u] <= thr) : (v[u] >= thr);
                if (p0 + u < e && p0 + u != d && !weak) {
                    if (kFill) out[c] = k[u];
                    ++c;
                }
            }
        }
    }
    return c;
}

template <bool kFill>
__global__ __launch_bounds__(kThreads) void k_strength(int32_t n, int32_t per,
                                                      const int32_t *__restrict__ I,
                                                      const int32_t *__restrict__ J,
                                                      const double *__restrict__ A, double theta,
                                                      double max_row_sum, int32_t *__restrict__ cnt,
                                                      const int32_t *__restrict__ SI,
                                                      int32_t *__restrict__ SJ) {
    __shared__ double s_a[kStageEntries];
    __shared__ int32_t s_j[kStageEntries];
    __shared__ int32_t s_out[kFill ? kStageEntries : 1];
    __shared__ int32_t s_I[kThreads + 1];
    __shared__ int32_t s_d[kThreads];  // the diagonals' places
    const int r0 = blockIdx.x * per, m = min(per, n - r0), tid = threadIdx.x;  // per <= kThreads
    for (int t = tid; t <= m; t += kThreads) s_I[t] = I[r0 + t];
    s_d[tid] = INT_MAX;
    __syncthreads();
    for (int ra = 0; ra < m;) {  // rows ra .. rb - 1 of the workgroup's (uniform)
        const int e0 = s_I[ra];
        int rb = s_I[m] - e0 <= kStageEntries ? m : ra;
        for (int hi = m; rb < hi;) {
            const int mid = (rb + hi + 1) >> 1;
            if (s_I[mid] - e0 <= kStageEntries) rb = mid;
            else hi = mid - 1;
        }
        const bool staged = rb > ra;
        rb = max(rb, ra + 1);
        const bool mine = tid >= ra && tid < rb;
        const int i = r0 + tid, ne = s_I[rb] - e0;
        if (staged) {
            for (int t = tid; t < ne; t += kThreads) {
                const int j = J[e0 + t], q = j - r0;
                s_j[t] = j;
                s_a[t] = A[e0 + t];
                if (q >= ra && q < rb && e0 + t >= s_I[q] && e0 + t < s_I[q + 1])
                    atomicMin(&s_d[q], t);
            }
            __syncthreads();
            const int o0 = kFill ? SI[r0 + ra] : 0;
            if (mine) {
                const int d = s_d[tid];
                const int c = strong_entries<kFill>(s_j, s_a, s_I[tid] - e0, s_I[tid + 1] - e0,
                                                    d == INT_MAX ? -1 : d, theta, max_row_sum,
                                                    kFill ? s_out + (SI[i] - o0) : nullptr);
                if (!kFill) cnt[i] = c;
            }
            if constexpr (kFill) {
                __syncthreads();
                const int no = SI[r0 + rb] - o0;
                for (int t = tid; t < no; t += kThreads) SJ[o0 + t] = s_out[t];
            }
            if (rb < m) __syncthreads();  // (uniform; the next part takes the place)
        } else if (mine) {
            const int c = strong_entries<kFill, int64_t>(J, A, I[i], I[i + 1], diag_pos(I, J, i),
                                                         theta, max_row_sum,
                                                         kFill ? SJ + SI[i] : nullptr);
            if (!kFill) cnt[i] = c;
        }
        ra = rb;
    }
}

// ---- PMIS (par_coarsen.c:2101-2813 on one process) ------------------------------
__global__ __launch_bounds__(kThreads) void k_col_count(int32_t n, const int32_t *__restrict__ SI,
                                                       const int32_t *__restrict__ SJ,
                                                       int32_t *__restrict__ cnt) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    for (int p = SI[i]; p < SI[i + 1]; ++p) atomicAdd(&cnt[SJ[p]], 1);
}

// x_{k} = a^k x_0 mod m of the Park-Miller generator (random.c:43-101); all
// products stay below 2^62.  m = 2^31 - 1, so 2^31 = 1 (mod m) and a product is
// reduced by adding its upper and lower 31 bits (twice), without a division.
__device__ __forceinline__ uint64_t pm_mod(uint64_t v) {
    constexpr uint64_t kM = 2147483647u;
    v = (v & kM) + (v >> 31);
    v = (v & kM) + (v >> 31);
    return v >= kM ? v - kM : v;
}
__device__ __forceinline__ uint64_t pm_jump(uint64_t x0, uint64_t k) {
    uint64_t r = 1u, b = 16807u;
    while (k) {
        if (k & 1u) r = pm_mod(r * b);
        b = pm_mod(b * b);
        k >>= 1;
    }
    return pm_mod(r * x0);
}

// measures and the initial graph (par_coarsen.c:2230-2400, IndepSetInit with
// seed 2747); a row with no strong dependence is marked -3 and left out
__global__ __launch_bounds__(kThreads) void k_pmis_init(int32_t n, const int32_t *__restrict__ SI,
                                                       const int32_t *__restrict__ cnt,
                                                       double *__restrict__ measure,
                                                       int32_t *__restrict__ cf,
                                                       int32_t *__restrict__ any) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const double r = double(pm_jump(2747u, uint64_t(i) + 1u)) / 2147483647.0;
    const double m = double(cnt[i]) + r;
    if (SI[i + 1] == SI[i]) {
        cf[i] = -3;
        measure[i] = 0.0;
    } else {
        cf[i] = 0;
        measure[i] = m;
        *any = 1;
    }
}

// CF_init 1 (HMIS, par_coarsen.c:2353-2386): cf holds the markers of the Ruge
// first pass.  C points stay C and join the graph; F points are undecided
// again; a Z point (it influences nobody) joins the graph as undecided if its
// measure reaches 1 or it depends on some point, else it is F; points without
// strong dependence stay out.  Graph membership is a positive measure, so the
// points left out get measure 0 (the host leaves a Z point's measure below 1,
// which no comparison with > 1 can see).
__global__ __launch_bounds__(kThreads) void k_pmis_init_hmis(int32_t n,
                                                            const int32_t *__restrict__ SI,
                                                            const int32_t *__restrict__ cnt,
                                                            double *__restrict__ measure,
                                                            int32_t *__restrict__ cf,
                                                            int32_t *__restrict__ any) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const double r = double(pm_jump(2747u, uint64_t(i) + 1u)) / 2147483647.0;
    const double m = double(cnt[i]) + r;
    int c = cf[i];
    if (c == -3) {
        measure[i] = 0.0;
        return;
    }
    if (c == -1) c = 0;
    if (c == -2) {
        if (!(m >= 1.0) && SI[i + 1] == SI[i]) {
            cf[i] = -1;
            measure[i] = 0.0;
            return;
        }
        c = 0;
    }
    cf[i] = c;
    measure[i] = m;
    *any = 1;
}

// independent set, first half (par_coarsen.c:2510-2556): a node of the graph
// with measure > 1 loses against any S neighbour (either direction) with a
// larger measure > 1; the host's clearing stores are idempotent, so plain
// stores of 1 reproduce them
__global__ __launch_bounds__(kThreads) void k_pmis_clear(int32_t n, const int32_t *__restrict__ SI,
                                                        const int32_t *__restrict__ SJ,
                                                        const double *__restrict__ measure,
                                                        int32_t *__restrict__ lost) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const double mi = measure[i];
    if (!(mi > 1)) return;
    for (int p = SI[i]; p < SI[i + 1]; ++p) {
        const int j = SJ[p];
        const double mj = measure[j];
        if (mj > 1) {
            if (mi > mj) lost[j] = 1;
            else if (mj > mi) lost[i] = 1;
        }
    }
}

// graph nodes are the ones with a positive measure (decided and isolated nodes
// have measure 0; a random draw is > 0)
__global__ __launch_bounds__(kThreads) void k_pmis_set(int32_t n, const double *__restrict__ measure,
                                                      const int32_t *__restrict__ lost,
                                                      int32_t *__restrict__ cf) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    if (measure[i] > 1 && !lost[i]) cf[i] = 1;
}

// C and F points (par_coarsen.c:2583-2666): a graph node of measure < 1 is F;
// a node outside the set that depends on a C point is F.  Then the subgraph
// update (:2690-2760): decided nodes leave, *any = 1 if one stays.  (A row's
// measure is read and written by its own thread only.)  Clears `lost` for the
// next pass.
__global__ __launch_bounds__(kThreads) void k_pmis_cf(int32_t n, const int32_t *__restrict__ SI,
                                                     const int32_t *__restrict__ SJ,
                                                     double *__restrict__ measure,
                                                     int32_t *__restrict__ cf,
                                                     int32_t *__restrict__ lost,
                                                     int32_t *__restrict__ any) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const double mi = measure[i];
    if (!(mi > 0)) return;
    lost[i] = 0;
    int c = cf[i];
    if (mi < 1) cf[i] = c = -1;
    if (c <= 0) {
        for (int p = SI[i]; p < SI[i + 1]; ++p)
            if (cf[SJ[p]] > 0) {
                cf[i] = c = -1;
                break;
            }
    }
    if (c != 0) measure[i] = 0.0;
    else *any = 1;
}

struct NotCoarse {
    const int32_t *cf;
    __device__ int64_t operator()(int i) const { return cf[i] >= 0 ? 0 : 1; }
};

// ---- extended+i interpolation (par_lr_interp.c:1025-1928, one process) -----------
// upper bound of a row's entries: 1 for C, 0 for isolated, else the strong C
// neighbours plus the strong dependencies of the strong F neighbours
__global__ __launch_bounds__(kThreads) void k_extpi_ub(int32_t n, const int32_t *__restrict__ SI,
                                                      const int32_t *__restrict__ SJ,
                                                      const int32_t *__restrict__ cf,
                                                      int64_t *__restrict__ ub) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    int64_t u = 0;
    if (cf[i] >= 0) {
        u = 1;
    } else if (cf[i] != -3) {
        for (int p = SI[i]; p < SI[i + 1]; ++p) {
            const int i1 = SJ[p];
            if (cf[i1] >= 0) u += 1;
            else if (cf[i1] != -3) u += SI[i1 + 1] - SI[i1];
        }
    }
    ub[i] = u;
}

// Per-row open-addressing table (linear probing, power-of-two size, at least
// twice the entries it can receive): fine column -> position in the row (>= 0)
// or kStrongF for a strong F neighbour; keys start at -1.  It stands for the
// host's P_marker array, so every membership test is O(1).
constexpr int32_t kStrongF = -2;

__device__ __forceinline__ uint32_t h_slot(int k, uint32_t mask) {
    return (uint32_t(k) * 2654435761u) & mask;
}

// slots are (key, value) pairs: one 8-byte load per probe
__device__ __forceinline__ int h_find(const int2 *__restrict__ kv, uint32_t mask, int k) {
    for (uint32_t h = h_slot(k, mask);; h = (h + 1) & mask) {
        const int2 e = kv[h];
        if (e.x == k) return e.y;
        if (e.x == -1) return -1;
    }
}

__device__ __forceinline__ void h_put(int2 *__restrict__ kv, uint32_t mask, int k, int v) {
    for (uint32_t h = h_slot(k, mask);; h = (h + 1) & mask) {
        const int32_t kk = kv[h].x;
        if (kk == -1 || kk == k) {
            kv[h] = make_int2(k, v);
            return;
        }
    }
}

// qsort.c:395-417 (descending |w|) with an explicit stack in place of the
// recursion.  Each partition step is the host's; the two subranges it leaves
// are disjoint and sorted independently, so the order in which they are
// sorted does not change the result: the smaller one goes first, which keeps
// the stack within log2(length) entries.
__device__ void qsort2_abs(int32_t *v, double *w, int left, int right) {
    int stack[2 * 40];
    int top = 0;
    stack[top++] = left;
    stack[top++] = right;
    while (top > 0) {
        const int r = stack[--top];
        const int l = stack[--top];
        if (l >= r) continue;
        const int mid = (l + r) / 2;
        {
            const int32_t tv = v[l];
            v[l] = v[mid];
            v[mid] = tv;
            const double tw = w[l];
            w[l] = w[mid];
            w[mid] = tw;
        }
        int last = l;
        for (int i = l + 1; i <= r; ++i) {
            if (fabs(w[i]) > fabs(w[l])) {
                ++last;
                const int32_t tv = v[last];
                v[last] = v[i];
                v[i] = tv;
                const double tw = w[last];
                w[last] = w[i];
                w[i] = tw;
            }
        }
        {
            const int32_t tv = v[l];
            v[l] = v[last];
            v[last] = tv;
            const double tw = w[l];
            w[l] = w[last];
            w[last] = tw;
        }
        // larger subrange pushed first, smaller one popped next
        if (last - 1 - l > r - (last + 1)) {
            stack[top++] = l;
            stack[top++] = last - 1;
            stack[top++] = last + 1;
            stack[top++] = r;
        } else {
            stack[top++] = last + 1;
            stack[top++] = r;
            stack[top++] = l;
            stack[top++] = last - 1;
        }
    }
}

// Where a row's finished entries go: a fixed slot of `stride` entries per row
// when rows are truncated to at most that many, else at off[i].
struct RowSlots {
    const int64_t *off;
    int32_t stride;
    int32_t *sj;
    double *sw;
    int32_t *cnt;
    __device__ __forceinline__ int64_t at(int i) const {
        return stride > 0 ? int64_t(i) * stride : off[i];
    }
};

// One thread per listed row: the row's columns (fine indices) and weights in
// the host's discovery order into work arrays at woff[t] (the weights at woff[t] -
// wfirst: only this kernel's rows have them), truncated there, then copied to the
// row's slot.
__global__ __launch_bounds__(kThreads) void k_extpi_row(
    int32_t count, const int32_t *__restrict__ rows, const int32_t *__restrict__ I,
    const int32_t *__restrict__ J, const double *__restrict__ A, const int32_t *__restrict__ SI,
    const int32_t *__restrict__ SJ, const int32_t *__restrict__ cf, int max_elmts,
    const int64_t *__restrict__ woff, int64_t wfirst, int32_t *__restrict__ wcol,
    double *__restrict__ wval, const int64_t *__restrict__ hoff, int2 *__restrict__ hkv, RowSlots out,
    int32_t *__restrict__ use) {
    const int t = blockIdx.x * kThreads + threadIdx.x;
    if (t >= count) return;
    const int i = rows[t];
    int32_t *cols = wcol + woff[t];
    double *w = wval + (woff[t] - wfirst);
    int2 *kv = hkv + hoff[t];
    const uint32_t mask = uint32_t(hoff[t + 1] - hoff[t]) - 1u;
    // structure (:1501-1560)
    int c = 0;
    for (int p = SI[i]; p < SI[i + 1]; ++p) {
        const int i1 = SJ[p];
        if (cf[i1] >= 0) {
            if (h_find(kv, mask, i1) < 0) {
                h_put(kv, mask, i1, c);
                cols[c++] = i1;
            }
        } else if (cf[i1] != -3) {
            h_put(kv, mask, i1, kStrongF);
            const int q1 = SI[i1 + 1];
            for (int q0 = SI[i1]; q0 < q1; q0 += 8) {  // eight strong neighbours at a time
                int k8[8], f8[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) k8[u] = q0 + u < q1 ? SJ[q0 + u] : -1;
#pragma unroll
                for (int u = 0; u < 8; ++u) f8[u] = k8[u] >= 0 ? cf[k8[u]] : -1;
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int k1 = k8[u];
                    if (f8[u] >= 0 && h_find(kv, mask, k1) < 0) {
                        h_put(kv, mask, k1, c);
                        cols[c++] = k1;
                    }
                }
            }
        }
    }
    for (int q = 0; q < c; ++q) w[q] = 0.0;
    // weights (:1630-1708)
    const int64_t di = diag_pos(I, J, i);
    double diagonal = di >= 0 ? A[di] : 0.0;
    for (int64_t jj = I[i]; jj < I[i + 1]; ++jj) {
        if (jj == di) continue;
        const int i1 = J[jj];
        const int pos = h_find(kv, mask, i1);
        if (pos >= 0) {
            w[pos] += A[jj];
            continue;
        }
        if (pos == kStrongF) {
            const int64_t d1 = diag_pos(I, J, i1);
            const int sgn = (d1 >= 0 && A[d1] < 0) ? -1 : 1;
            // both passes over row i1 in the host's order, its entries loaded
            // eight at a time so that the loads overlap
            const int64_t b1 = I[i1], e1 = I[i1 + 1];
            double sum = 0.0;
            for (int64_t q0 = b1; q0 < e1; q0 += 8) {
                int j8[8];
                double a8[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    j8[u] = q0 + u < e1 ? J[q0 + u] : -1;
                    a8[u] = q0 + u < e1 ? A[q0 + u] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    if (q0 + u >= e1 || q0 + u == d1) continue;
                    const int i2 = j8[u];
                    if ((i2 == i || h_find(kv, mask, i2) >= 0) && (sgn * a8[u]) < 0)
                        sum += a8[u];
                }
            }
            if (sum != 0) {
                const double distribute = A[jj] / sum;
                for (int64_t q0 = b1; q0 < e1; q0 += 8) {
                    int j8[8];
                    double a8[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        j8[u] = q0 + u < e1 ? J[q0 + u] : -1;
                        a8[u] = q0 + u < e1 ? A[q0 + u] : 0.0;
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        if (q0 + u >= e1 || q0 + u == d1) continue;
                        const int i2 = j8[u];
                        if ((sgn * a8[u]) < 0) {
                            const int p2 = h_find(kv, mask, i2);
                            if (p2 >= 0) w[p2] += distribute * a8[u];
                            if (i2 == i) diagonal += distribute * a8[u];
                        }
                    }
                }
            } else {
                diagonal += A[jj];
            }
        } else if (cf[i1] != -3) {
            diagonal += A[jj];
        }
    }
    if (diagonal != 0)
        for (int q = 0; q < c; ++q) w[q] /= -diagonal;
    // truncation (par_csr_matrix.c:3130-3215: tol 0, rescale)
    if (max_elmts > 0 && c > max_elmts) {
        double row_sum = 0.0;
        for (int q = 0; q < c; ++q) row_sum += w[q];
        qsort2_abs(cols, w, 0, c - 1);
        double scale = 0.0;
        for (int q = 0; q < max_elmts; ++q) scale += w[q];
        if (scale != 0. && scale != row_sum) {
            scale = row_sum / scale;
            for (int q = 0; q < max_elmts; ++q) w[q] *= scale;
        }
        c = max_elmts;
    }
    const int64_t o = out.at(i);
    for (int q = 0; q < c; ++q) {
        out.sj[o + q] = cols[q];
        out.sw[o + q] = w[q];
    }
    out.cnt[i] = c;
    use[i] = 0;
}

// ---- extended+i, one wave per row (long rows of coarse levels) ------------------
// The same results as k_extpi_row: the host's order of discovery and of
// accumulation is kept, the independent parts run across the lanes.
//  * discovery: the candidate columns in the host's order (lane per strong
//    dependency, offsets by a scan), first occurrences found with an LDS
//    table (atomicMin of the candidate index), positions by a prefix count;
//  * per entry jj of row i (lane per entry): its kind, and for a strong F
//    neighbour i1 the sum over row i1 in row order, the distribution factor
//    and its term for the diagonal;
//  * the weights, entry by entry jj in row order: a C neighbour's a_ij to its
//    column (one lane), a strong F neighbour's distribution over the entries
//    of row i1 that are P columns (a lane per entry of row i1, its column
//    looked up in the LDS table), so every weight receives its terms in the
//    host's order;
//  * the diagonal and the row sums in order, the truncation by ranks.
// capacities: WA entries of row i (A and S), WT distinct P columns kept in
// LDS, WH table slots: at most WT + 64 candidate columns (the insertions stop
// once WT is passed) plus WA strong F neighbours ever enter the table, which
// stays at most about half full (8.5 to 74 KB of LDS, below).
template <int WA, int WT, int WH>
struct WaveRow {
    static_assert(2 * (WT + 64 + WA) <= WH + 128 && (WH & (WH - 1)) == 0, "table size");
    int32_t acol[WA];
    double aval[WA];
    int32_t scol[WA];
    int32_t hkey[WH];
    int32_t hval[WH];
    int32_t pcol[WT];
    double pw[WT];
    double jdist[WA];
    double jdiag[WA];
    int32_t jinfo[WA];  // >= 0: P position; -1 none; -2 strong F (distribute); at the
                         // end, with jdist, the kept columns and weights
    int32_t jsgn[WA];
    int32_t jb1[WA];    // strong F neighbour: its row's range in J / A
    int32_t je1[WA];
    int32_t sc[3];
};

template <int WH>
__device__ __forceinline__ int lds_find(const int32_t *hkey, const int32_t *hval, int k) {
    for (uint32_t h = h_slot(k, WH - 1);; h = (h + 1) & (WH - 1)) {
        const int32_t kk = hkey[h];
        if (kk == k) return hval[h];
        if (kk == -1) return -1;
    }
}

// slot of key k (inserted if absent) in the wave's table
template <int WH>
__device__ __forceinline__ uint32_t lds_slot(int32_t *hkey, int k) {
    for (uint32_t h = h_slot(k, WH - 1);; h = (h + 1) & (WH - 1)) {
        const int32_t prev = atomicCAS(&hkey[h], -1, k);
        if (prev == -1 || prev == k) return h;
    }
}

// exclusive prefix sum over the wave's 64 lanes; *tot = total
__device__ __forceinline__ int wave_excl(int v, int *tot) {
    const int lane = threadIdx.x & 63;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(incl, d);
        if (lane >= d) incl += t;
    }
    *tot = __shfl(incl, 63);
    return incl - v;
}

template <int WA, int WT, int WH>
__global__ __launch_bounds__(64) void k_extpi_wave(
    int32_t count, const int32_t *__restrict__ rows, const int32_t *__restrict__ I,
    const int32_t *__restrict__ J, const double *__restrict__ A, const int32_t *__restrict__ SI,
    const int32_t *__restrict__ SJ, const int32_t *__restrict__ cf,
    const int8_t *__restrict__ dneg, const int64_t *__restrict__ woff,
    int32_t *__restrict__ wcol, int max_elmts, RowSlots out, int32_t *__restrict__ use,
    int overflow_code, int32_t *__restrict__ ovf) {
    __shared__ WaveRow<WA, WT, WH> s;
    if (blockIdx.x >= unsigned(count)) return;
    const int lane = threadIdx.x;
    const int i = rows[blockIdx.x];
    int32_t *cand = wcol + woff[blockIdx.x];  // the row's candidates
    const int a0 = I[i], la = I[i + 1] - a0;
    const int s0 = SI[i], ls = SI[i + 1] - s0;
    for (int t = lane; t < la; t += 64) {
        s.acol[t] = J[a0 + t];
        s.aval[t] = A[a0 + t];
    }
    for (int t = lane; t < ls; t += 64) s.scol[t] = SJ[s0 + t];
    for (int t = lane; t < WH; t += 64) {
        s.hkey[t] = -1;
        s.hval[t] = INT_MAX;
    }
    if (lane == 0) {
        s.sc[0] = -1;  // the diagonal's place
        s.sc[2] = 0;   // distinct candidate columns
    }
    __syncthreads();
    // candidates in the host's order (par_lr_interp.c:1501-1560)
    int T = 0;
    for (int b0 = 0; b0 < ls; b0 += 64) {
        const int p = b0 + lane;
        int i1 = 0, k = 0;
        int cf1 = 0, q0 = 0, q1 = 0;
        if (p < ls) {
            i1 = s.scol[p];
            cf1 = cf[i1];
            if (cf1 >= 0) {
                k = 1;
            } else if (cf1 != -3) {
                q0 = SI[i1];
                q1 = SI[i1 + 1];
                // the strong neighbours of i1 and their markers, eight at a
                // time so that the loads overlap
                for (int q = q0; q < q1; q += 8) {
                    int c8[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) c8[u] = q + u < q1 ? SJ[q + u] : -1;
#pragma unroll
                    for (int u = 0; u < 8; ++u) k += (c8[u] >= 0 && cf[c8[u]] >= 0) ? 1 : 0;
                }
            }
        }
        int tot;
        int o = T + wave_excl(k, &tot);
        if (p < ls && k > 0) {
            if (cf1 >= 0) {
                cand[o] = i1;
            } else {
                for (int q = q0; q < q1; q += 8) {  // in order, as counted
                    int c8[8], f8[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) c8[u] = q + u < q1 ? SJ[q + u] : -1;
#pragma unroll
                    for (int u = 0; u < 8; ++u) f8[u] = c8[u] >= 0 ? cf[c8[u]] : -1;
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (f8[u] >= 0) cand[o++] = c8[u];
                }
            }
        }
        T += tot;
    }
    __threadfence_block();
    __syncthreads();
    // first occurrences; a row with more distinct columns than WT is left to
    // the thread kernel (the insertions stop early enough that the table never
    // fills: at most WT + 64 keys before every lane sees the count)
    for (int t = lane; t < T; t += 64) {
        if (s.sc[2] > WT) break;
        const int col = cand[t];
        uint32_t h = h_slot(col, WH - 1);
        for (;; h = (h + 1) & (WH - 1)) {
            const int32_t prev = atomicCAS(&s.hkey[h], -1, col);
            if (prev == -1) {
                atomicAdd(&s.sc[2], 1);
                break;
            }
            if (prev == col) break;
        }
        atomicMin(&s.hval[h], t);
    }
    __syncthreads();
    if (s.sc[2] > WT) {  // to the next capacity or the thread kernel
        if (lane == 0) {
            use[i] = overflow_code;
            atomicAdd(ovf, 1);
        }
        return;
    }
    int c = 0;
    for (int b0 = 0; b0 < T; b0 += 64) {
        const int t = b0 + lane;
        bool first = false;
        int col = 0;
        if (t < T) {
            col = cand[t];
            first = lds_find<WH>(s.hkey, s.hval, col) == t;
        }
        int tot;
        const int pos = c + wave_excl(first ? 1 : 0, &tot);
        if (first) s.pcol[pos] = col;
        c += tot;
    }
    __syncthreads();
    // table: column -> position, strong F neighbours -> kStrongF
    for (int p = lane; p < c; p += 64) s.hval[lds_slot<WH>(s.hkey, s.pcol[p])] = p;
    for (int p = lane; p < ls; p += 64) {
        const int i1 = s.scol[p];
        if (cf[i1] < 0 && cf[i1] != -3) s.hval[lds_slot<WH>(s.hkey, i1)] = kStrongF;
    }
    __syncthreads();
    // per entry of row i
    for (int jj = lane; jj < la; jj += 64) {
        const int i1 = s.acol[jj];
        int info = -1, sgn = 1;
        double dist = 0.0, dterm = 0.0;
        if (i1 != i) {
            const int v = lds_find<WH>(s.hkey, s.hval, i1);
            if (v >= 0) {
                info = v;
            } else if (v == kStrongF) {
                const int64_t b1 = I[i1], e1 = I[i1 + 1];
                s.jb1[jj] = int32_t(b1);
                s.je1[jj] = int32_t(e1);
                sgn = dneg[i1] ? -1 : 1;
                // the host's sum in the host's order; the row's entries are
                // loaded eight at a time so that their loads overlap, and the
                // entry of column i is noted on the way (the row's columns are
                // distinct, so there is at most one)
                double sum = 0.0, aqi = 0.0;
                int64_t q = b1, qi = -1;
                for (; q + 8 <= e1; q += 8) {
                    int jq[8];
                    double aq[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        jq[u] = J[q + u];
                        aq[u] = A[q + u];
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int i2 = jq[u];
                        if (i2 == i1) continue;
                        if (i2 == i) {
                            qi = q + u;
                            aqi = aq[u];
                        }
                        if ((i2 == i || lds_find<WH>(s.hkey, s.hval, i2) >= 0) &&
                            (sgn * aq[u]) < 0)
                            sum += aq[u];
                    }
                }
                for (; q < e1; ++q) {
                    const int i2 = J[q];
                    if (i2 == i1) continue;
                    const double aq1 = A[q];
                    if (i2 == i) {
                        qi = q;
                        aqi = aq1;
                    }
                    if ((i2 == i || lds_find<WH>(s.hkey, s.hval, i2) >= 0) && (sgn * aq1) < 0)
                        sum += aq1;
                }
                if (sum != 0) {
                    info = -2;
                    dist = s.aval[jj] / sum;
                    if (qi >= 0 && (sgn * aqi) < 0) dterm = dist * aqi;
                } else {
                    dterm = s.aval[jj];
                }
            } else if (cf[i1] != -3) {
                dterm = s.aval[jj];
            }
        }
        s.jinfo[jj] = info;
        s.jsgn[jj] = sgn;
        s.jdist[jj] = dist;
        s.jdiag[jj] = dterm;
    }
    __syncthreads();
    // weights, entry by entry in row order (the host's order of accumulation
    // for every column): a C neighbour adds a_ij to its column's weight; a
    // strong F neighbour i1 distributes over the entries of row i1 that are P
    // columns, a lane per entry (a row's columns are distinct, so no two lanes
    // add to one weight)
    for (int p = lane; p < c; p += 64) s.pw[p] = 0.0;
    __syncthreads();
    for (int jj = 0; jj < la; ++jj) {
        const int info = s.jinfo[jj];  // wave-uniform
        if (info >= 0) {
            if (lane == 0) s.pw[info] += s.aval[jj];
        } else if (info == -2) {
            const double dj = s.jdist[jj];
            const int sg = s.jsgn[jj];
            for (int q = s.jb1[jj] + lane; q < s.je1[jj]; q += 64) {
                const double aq = A[q];
                const int pos = lds_find<WH>(s.hkey, s.hval, J[q]);  // -1 / kStrongF: no P column
                if (pos >= 0 && (sg * aq) < 0) s.pw[pos] += dj * aq;
            }
        }
        __syncthreads();  // the next entry's terms may go to the same weights
    }
    // the diagonal in row order (every lane the same sum; 0.0 for the entries
    // that add nothing)
    double diagonal = 0.0;
    for (int t = lane; t < la; t += 64)
        if (s.acol[t] == i) s.sc[0] = t;
    __syncthreads();
    if (s.sc[0] >= 0) diagonal = s.aval[s.sc[0]];
    for (int jj = 0; jj < la; ++jj) diagonal += s.jdiag[jj];
    if (diagonal != 0)
        for (int q = lane; q < c; q += 64) s.pw[q] /= -diagonal;
    __syncthreads();
    // truncation (par_csr_matrix.c:3130-3215): where the kept weights are
    // distinct in magnitude, sorted order is the order of the ranks, which the
    // lanes count (the host's quicksort on one lane took most of a long row's
    // time); else the quicksort
    const bool trunc = max_elmts > 0 && c > max_elmts;
    const int cc = trunc ? max_elmts : c;
    int32_t *kcol = s.pcol;
    double *kw = s.pw;
    if (trunc) {  // uniform
        double row_sum = 0.0;
        for (int q = 0; q < c; ++q) row_sum += s.pw[q];
        bool tie = max_elmts > WA;  // the kept entries' LDS
        if (!tie)
            for (int q = lane; q < c; q += 64) {
                const double a = fabs(s.pw[q]);
                int above = 0, same = 0;
                for (int t = 0; t < c; ++t) {
                    const double b = fabs(s.pw[t]);
                    above += b > a ? 1 : 0;
                    same += b == a ? 1 : 0;
                }
                if (above < max_elmts) {
                    if (same != 1) {
                        tie = true;
                    } else {
                        s.jinfo[above] = s.pcol[q];
                        s.jdist[above] = s.pw[q];
                    }
                }
            }
        if (__ballot(tie) == 0ull) {
            kcol = s.jinfo;
            kw = s.jdist;
        } else if (lane == 0) {
            qsort2_abs(s.pcol, s.pw, 0, c - 1);
        }
        __syncthreads();
        double scale = 0.0;
        for (int q = 0; q < max_elmts; ++q) scale += kw[q];
        if (scale != 0. && scale != row_sum) {
            scale = row_sum / scale;
            __syncthreads();
            for (int q = lane; q < max_elmts; q += 64) kw[q] *= scale;
        }
    }
    __syncthreads();
    if (lane == 0) {
        out.cnt[i] = cc;
        use[i] = 0;
    }
    const int64_t o = out.at(i);
    for (int q = lane; q < cc; q += 64) {
        out.sj[o + q] = kcol[q];
        out.sw[o + q] = kw[q];
    }
}

// ---- extended+i, G lanes per row (G = 8, 16, 32: rows of up to G entries in A and S) ----
// The same results as k_extpi_row.  64 / G rows share a wave, a row's state is
// 4 G columns and a table of 8 G slots in LDS (152 G bytes: 1.2 KB for G = 8, 39 KB
// per workgroup whatever G, four workgroups per CU), a lane holds one entry of A and one of S.  The
// thread kernel is bound by its per-row tables in global memory (scattered
// probes, a few lanes of a cache line used); here only the neighbours' rows
// are read from memory, all of a row's neighbours at once, and every probe
// and accumulation is in LDS.
//  * discovery: each lane counts the columns its strong neighbour contributes,
//    a prefix over the lanes places them in one list in the host's order, the
//    lanes insert the list's columns into the table with their place
//    (atomicMin keeps the first) and a ballot counts the firsts before each;
//  * lane jj: kind of entry jj; for a strong F neighbour the sum over its row
//    in row order, the entries' columns looked up on the way and the terms of
//    P columns (few of a row's entries) kept in LDS;
//  * the weights entry by entry in row order, a lane per term (the columns of
//    one entry are distinct);
//  * truncation: if the largest weights are distinct in magnitude the sorted
//    order is the order of their ranks, which the lanes count; otherwise lane 0
//    of the group runs the host's quicksort.
// Issue-bound by the probe loops, which diverge: the first form, which walked
// each lane's own columns three times (37 loops), took 1140 us on 7-pt 128^3
// (1.5 M F rows), this one 906, the thread kernel 4845 us.
constexpr int kTerms = 4;  // terms of one neighbour kept in LDS
template <int G>
struct GroupRow {
    double pw[4 * G];          // first the list of candidate columns (8 G), then weights
    double ta[kTerms * G];     // terms of entry jj at kTerms * jj; kept columns at the end
    int2 kv[8 * G];            // (column, place then position); kept weights at the end
    uint64_t tp[G];            // positions of the terms, 16 bits each (0xffff: none)
    int32_t pcol[4 * G];
};
static_assert(sizeof(GroupRow<8>) == 152 * 8 && sizeof(GroupRow<32>) == 152 * 32, "LDS per row");

template <int WH>
__device__ __forceinline__ int kv_find(const int2 *kv, int k) {
    for (uint32_t h = h_slot(k, WH - 1);; h = (h + 1) & (WH - 1)) {
        const int2 e = kv[h];
        if (e.x == k) return e.y;
        if (e.x == -1) return -1;
    }
}

// the host's quicksort (qsort2_abs) for at most 128 entries: the pending
// subranges, at most one per halving, stay in two registers (8 bits per bound)
__device__ void qsort2_abs_128(int32_t *v, double *w, int right) {
    uint64_t lo = uint64_t(right), hi = 0;  // (left << 8 | right), newest lowest
    int top = right > 0 ? 1 : 0;
    while (top > 0) {
        const int l = int((lo >> 8) & 0xffu), r = int(lo & 0xffu);
        lo = (lo >> 16) | (hi << 48);
        hi >>= 16;
        --top;
        const int mid = (l + r) / 2;
        {
            const int32_t tv = v[l];
            v[l] = v[mid];
            v[mid] = tv;
            const double tw = w[l];
            w[l] = w[mid];
            w[mid] = tw;
        }
        const double piv = fabs(w[l]);
        int last = l;
        for (int i = l + 1; i <= r; ++i) {
            if (fabs(w[i]) > piv) {
                ++last;
                const int32_t tv = v[last];
                v[last] = v[i];
                v[i] = tv;
                const double tw = w[last];
                w[last] = w[i];
                w[i] = tw;
            }
        }
        {
            const int32_t tv = v[l];
            v[l] = v[last];
            v[last] = tv;
            const double tw = w[l];
            w[l] = w[last];
            w[last] = tw;
        }
        const bool left_big = last - l > r - last;
        for (int half = 0; half < 2; ++half) {  // the larger subrange first
            const bool left = (half == 0) == left_big;
            const int nl = left ? l : last + 1, nr = left ? last - 1 : r;
            if (nl >= nr) continue;
            hi = (hi << 16) | (lo >> 48);
            lo = (lo << 16) | uint64_t(nl << 8 | nr);
            ++top;
        }
    }
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int G>
__global__ __launch_bounds__(kThreads) void k_extpi_group(
    int32_t n, const int32_t *__restrict__ I, const int32_t *__restrict__ J,
    const double *__restrict__ A, const int32_t *__restrict__ SI, const int32_t *__restrict__ SJ,
    const int32_t *__restrict__ cf, const int8_t *__restrict__ dneg, int max_elmts, RowSlots out,
    int32_t *__restrict__ use, int per, int code, int overflow_code, int32_t *__restrict__ ovf) {
    constexpr int NG = kThreads / G, WH = 8 * G, WT = 4 * G;
    __shared__ GroupRow<G> s_row[NG];
    __shared__ int32_t s_list[kThreads];
    __shared__ int s_wc[kThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    // this kernel's rows among the workgroup's `per`, packed
    const int row = blockIdx.x * per + tid;
    const bool mine = tid < per && row < n && use[row] == code;
    const uint64_t bal = __ballot(mine);
    if (lane == 0) s_wc[tid >> 6] = __popcll(bal);
    __syncthreads();
    int at = 0, total = 0;
#pragma unroll
    for (int q = 0; q < kThreads / 64; ++q) {
        if (q < (tid >> 6)) at += s_wc[q];
        total += s_wc[q];
    }
    if (mine) s_list[at + __popcll(bal & ((1ull << lane) - 1ull))] = row;
    __syncthreads();
    GroupRow<G> &s = s_row[tid / G];
    int32_t *const cand = reinterpret_cast<int32_t *>(s.pw);  // 8 G candidates
    double *const tw = reinterpret_cast<double *>(s.kv);      // 4 G kept weights
    int32_t *const keep = reinterpret_cast<int32_t *>(s.ta);  // and their columns
    const int gl = tid % G;
    const int sh = lane - gl;  // first lane of the group
    const uint64_t gones = (1ull << G) - 1ull, gmask = gones << sh;
    constexpr int TL = 6 * G;  // candidates: with G strong F neighbours 7 G of 8 G slots
    for (int k0 = 0; k0 < total; k0 += NG) {  // uniform: every lane stays for the wave steps
        const bool on = k0 + tid / G < total;
        const int i = on ? s_list[k0 + tid / G] : 0;
        int a0 = 0, la = 0, s0 = 0, ls = 0;
        if (on) {
            a0 = I[i];
            la = I[i + 1] - a0;
            s0 = SI[i];
            ls = SI[i + 1] - s0;
        }
        int ac = -1, sc = -1;
        double av = 0.0;
        if (gl < la) {
            ac = J[a0 + gl];
            av = A[a0 + gl];
        }
        if (gl < ls) sc = SJ[s0 + gl];
        for (int t = gl; t < WH; t += G) s.kv[t] = make_int2(-1, INT_MAX);
        const int cfa = ac >= 0 ? cf[ac] : -3;
        const int cfs = sc >= 0 ? cf[sc] : -3;
        const bool strongF = cfs < 0 && cfs != -3;
        int q0 = 0, q1 = 0;
        if (strongF) {
            q0 = SI[sc];
            q1 = SI[sc + 1];
        }
        int c8[8], f8[8];  // the first eight strong neighbours of sc and their markers
#pragma unroll
        for (int u = 0; u < 8; ++u) c8[u] = q0 + u < q1 ? SJ[q0 + u] : -1;
#pragma unroll
        for (int u = 0; u < 8; ++u) f8[u] = c8[u] >= 0 ? cf[c8[u]] : -1;
        int nk = cfs >= 0 ? 1 : 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) nk += f8[u] >= 0 ? 1 : 0;
        for (int q = q0 + 8; q < q1; ++q) nk += cf[SJ[q]] >= 0 ? 1 : 0;
        int o = nk;
#pragma unroll
        for (int d = 1; d < G; d <<= 1) {
            const int t = __shfl_up(o, d, G);
            if (gl >= d) o += t;
        }
        const int T = __shfl(o, G - 1, G);
        o -= nk;
        const bool fits = T <= TL;
        if (fits && nk > 0) {
            if (cfs >= 0) cand[o++] = sc;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (f8[u] >= 0) cand[o++] = c8[u];
            for (int q = q0 + 8; q < q1; ++q) {
                const int col = SJ[q];
                if (cf[col] >= 0) cand[o++] = col;
            }
        }
        wave_lds_sync();
        // candidate t: its slot; the smallest place of a column stays with it
        int ct[6], slot[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) {
            const int t = gl + m * G;
            const bool in = fits && t < T;
            ct[m] = 0;
            slot[m] = 0;
            if (!__ballot(in)) continue;
            if (in) {
                ct[m] = cand[t];
                uint32_t h = h_slot(ct[m], WH - 1);
                for (;; h = (h + 1) & (WH - 1)) {
                    const int32_t prev = atomicCAS(&s.kv[h].x, -1, ct[m]);
                    if (prev == -1 || prev == ct[m]) break;
                }
                atomicMin(&s.kv[h].y, t);
                slot[m] = int(h);
            }
        }
        wave_lds_sync();
        int c = 0;
#pragma unroll
        for (int m = 0; m < 6; ++m) {
            const int t = gl + m * G;
            const bool in = fits && t < T;
            if (!__ballot(in)) continue;
            const bool first = in && s.kv[slot[m]].y == t;
            const uint64_t f = (__ballot(first) >> sh) & gones;
            const int pos = c + __popcll(f & ((1ull << gl) - 1ull));
            if (first && pos < WT) {
                s.pcol[pos] = ct[m];
                s.kv[slot[m]].y = pos;  // at most the column's place: equals no later one
            }
            c += __popcll(f);
        }
        const bool over = !fits || c > WT;
        const bool go = on && !over;
        if (!go) c = 0;
        if (on && over && gl == 0) {
            use[i] = overflow_code;
            atomicAdd(ovf, 1);
        }
        if (go && strongF) {
            uint32_t h = h_slot(sc, WH - 1);
            for (;; h = (h + 1) & (WH - 1)) {
                const int32_t prev = atomicCAS(&s.kv[h].x, -1, sc);
                if (prev == -1 || prev == sc) break;
            }
            s.kv[h].y = kStrongF;
        }
        wave_lds_sync();
        for (int q = gl; q < c; q += G) s.pw[q] = 0.0;  // (the candidates are done)
        // this lane's entry of row i
        int b1 = 0, e1 = 0, neg = 0, nt = 0;
        bool spread = false;
        uint64_t tp = ~0ull;
        double dist = 0.0, dterm = 0.0;
        double *const ta = s.ta + kTerms * gl;
        if (go && ac >= 0 && ac != i) {
            const int v = kv_find<WH>(s.kv, ac);
            if (v >= 0) {
                ta[0] = av;
                tp = ~0xffffull | uint64_t(v);
            } else if (v == kStrongF) {
                b1 = I[ac];
                e1 = I[ac + 1];
                neg = dneg[ac];
                double sum = 0.0, aqi = 0.0;
                bool back = false;  // row ac holds column i with the right sign
                for (int q = b1; q < e1; q += 8) {
                    int j8[8];
                    double a8[8];
                    int2 e8[8];
                    uint32_t h8[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        j8[u] = q + u < e1 ? J[q + u] : ac;
                        a8[u] = q + u < e1 ? A[q + u] : 0.0;
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        h8[u] = h_slot(j8[u], WH - 1);
                        e8[u] = s.kv[h8[u]];
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        if (j8[u] == ac || !(neg ? a8[u] > 0.0 : a8[u] < 0.0)) continue;
                        if (j8[u] == i) {
                            back = true;
                            aqi = a8[u];
                            sum += a8[u];
                            continue;
                        }
                        while (e8[u].x != j8[u] && e8[u].x != -1) {
                            h8[u] = (h8[u] + 1) & (WH - 1);
                            e8[u] = s.kv[h8[u]];
                        }
                        if (e8[u].x == -1 || e8[u].y < 0) continue;
                        sum += a8[u];
                        if (nt < kTerms) {
                            ta[nt] = a8[u];
                            tp ^= uint64_t(0xffffu ^ e8[u].y) << (16 * nt);
                        }
                        ++nt;
                    }
                }
                if (sum != 0) {
                    dist = av / sum;
                    if (back) dterm = dist * aqi;
                    spread = nt > kTerms;
                    if (spread) tp = ~0ull;
                    else
                        for (int t = 0; t < nt; ++t) ta[t] = dist * ta[t];
                } else {
                    tp = ~0ull;
                    dterm = av;
                }
            } else if (cfa != -3) {
                dterm = av;
            }
        }
        s.tp[gl] = tp;
        wave_lds_sync();
        const int maxla = __builtin_amdgcn_readlane(wave_incl_max(la), 63);
        const double aii = (go && ac == i) ? av : 0.0;
        const uint64_t has_d = __ballot(go && ac == i) & gmask;
        double diagonal = __shfl(aii, has_d ? __ffsll((unsigned long long)has_d) - 1 : lane);
        for (int jj = 0; jj < maxla; ++jj) {
            // 0.0 for the entries that add nothing (adding it changes no sum
            // that is compared or divided by)
            diagonal += __shfl(dterm, jj, G);
            if (gl < kTerms) {
                const int p = reinterpret_cast<const uint16_t *>(&s.tp[jj])[gl];
                if (p < WT) s.pw[p] += s.ta[kTerms * jj + gl];
            }
            if (__ballot(gl == jj && spread)) {
                // a neighbour with more terms: its row again, a lane per entry
                const double dj = __shfl(dist, jj, G);
                const int ng = __shfl(neg, jj, G), bj = __shfl(b1, jj, G);
                const int ej = __shfl(int(spread), jj, G) ? __shfl(e1, jj, G) : bj;
                for (int q = bj + gl; q < ej; q += G) {
                    const double aq = A[q];
                    if (!(ng ? aq > 0.0 : aq < 0.0)) continue;
                    const int p = kv_find<WH>(s.kv, J[q]);
                    if (p >= 0) s.pw[p] += dj * aq;
                }
            }
            wave_lds_sync();
        }
        if (diagonal != 0)
            for (int q = gl; q < c; q += G) s.pw[q] /= -diagonal;
        wave_lds_sync();
        // truncation (par_csr_matrix.c:3130-3215: tol 0, rescale)
        const bool trunc = max_elmts > 0 && c > max_elmts;
        const int cc = trunc ? max_elmts : c;
        double factor = 1.0;
        if (__ballot(trunc)) {
            double row_sum = 0.0;
            int rk[4];
            bool tie = false;
            if (trunc) {
                for (int q = 0; q < c; ++q) row_sum += s.pw[q];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const int q = gl + m * G;
                    rk[m] = INT_MAX;
                    if (q >= c) continue;
                    const double a = fabs(s.pw[q]);
                    int above = 0, same = 0;
                    for (int r = 0; r < c; ++r) {
                        const double b = fabs(s.pw[r]);
                        above += b > a ? 1 : 0;
                        same += b == a ? 1 : 0;
                    }
                    rk[m] = above;
                    // (a weight that is no number equals nothing, not even itself)
                    if (above < max_elmts && same != 1) tie = true;
                }
            }
            const bool sorted = (__ballot(tie) & gmask) != 0ull;
            if (trunc && sorted && gl == 0) qsort2_abs_128(s.pcol, s.pw, c - 1);
            wave_lds_sync();
            if (trunc) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const int q = gl + m * G;
                    const int to = sorted ? q : rk[m];
                    if (q < c && to < max_elmts) {
                        keep[to] = s.pcol[q];
                        tw[to] = s.pw[q];
                    }
                }
            }
            wave_lds_sync();
            if (trunc) {
                double scale = 0.0;
                for (int q = 0; q < max_elmts; ++q) scale += tw[q];
                if (scale != 0. && scale != row_sum) factor = row_sum / scale;
            }
        }
        if (go) {
            const int64_t o = out.at(i);
            for (int q = gl; q < cc; q += G) {
                out.sj[o + q] = trunc ? keep[q] : s.pcol[q];
                out.sw[o + q] = trunc ? tw[q] * factor : s.pw[q];
            }
            if (gl == 0) {
                out.cnt[i] = cc;
                use[i] = 0;
            }
        }
        wave_lds_sync();  // the next row reuses the state
    }
}
#pragma clang fp contract(fast)

// Which kernel a row of extended+i takes (0: none, C points, isolated rows and
// finished ones).  Codes 1..8 are listed rows: the wave kernels by row length
// (each with a small table of P columns, then, for a row with more distinct
// columns, the large one), then the thread kernel.  Codes 9..11: the lane-group
// kernels, which find their rows themselves; their overflow goes to kTier64.
constexpr int kTier64 = 1, kTier64Big = 2, kTier128 = 3, kTier128Big = 4, kTier256 = 5,
              kTier256Big = 6, kTier512 = 7, kThreadRow = 8, kGroup8 = 9, kGroup16 = 10,
              kGroup32 = 11;
constexpr int kListed = 8, kCodes = 11;

// per row: C flag, kernel code, sign of the diagonal; C rows (the identity,
// par_lr_interp.c:1488-1495) and isolated rows are finished here
__global__ __launch_bounds__(kThreads) void k_extpi_class(
    int32_t n, const int32_t *__restrict__ I, const int32_t *__restrict__ J,
    const double *__restrict__ A, const int32_t *__restrict__ SI, const int32_t *__restrict__ cf,
    int longest, int32_t *__restrict__ flag, int32_t *__restrict__ use,
    int8_t *__restrict__ dneg, RowSlots out) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const int f = cf[i];
    const int len = max(I[i + 1] - I[i], SI[i + 1] - SI[i]);
    int u = 0;
    if (f >= 0) {
        const int64_t o = out.at(i);
        out.sj[o] = i;
        out.sw[o] = 1.0;
        out.cnt[i] = 1;
    } else if (f == -3) {
        out.cnt[i] = 0;
    } else {
        u = len <= 8 ? kGroup8 : (len <= 16 ? kGroup16 : (len <= 32 ? kGroup32 : kThreadRow));
        if (len > 32 && len <= 64) u = kTier64;
        if (len > 64 && len <= longest)  // of the wave kernels
            u = len <= 128 ? kTier128 : (len <= 256 ? kTier256 : kTier512);
    }
    flag[i] = f >= 0 ? 1 : 0;
    use[i] = u;
    const int64_t d = diag_pos(I, J, i);
    dneg[i] = (d >= 0 && A[d] < 0) ? 1 : 0;
}

// rows per code: one partial per workgroup, one workgroup scans the listed
// codes' partials into list offsets (the lists follow each other in the order
// of the codes), then the lists are written, rows ascending
struct CodeTotals {
    int32_t c[kCodes];
};
// parts[q * ng + workgroup]: rows of code q + 1
__global__ __launch_bounds__(kThreads) void k_code_part(int32_t n, const int32_t *__restrict__ use,
                                                       int32_t ng, int32_t *__restrict__ parts) {
    __shared__ int s_c[kThreads / 64][kCodes];
    const int i = blockIdx.x * kThreads + threadIdx.x;
    const int u = i < n ? use[i] : 0;
#pragma unroll
    for (int q = 0; q < kCodes; ++q) {
        const uint64_t m = __ballot(u == q + 1);
        if ((threadIdx.x & 63) == 0) s_c[threadIdx.x >> 6][q] = __popcll(m);
    }
    __syncthreads();
    if (threadIdx.x < kCodes) {
        int c = 0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w) c += s_c[w][threadIdx.x];
        parts[int64_t(threadIdx.x) * ng + blockIdx.x] = c;
    }
}
// one workgroup, a wave per code; eight loads in flight per lane
__global__ __launch_bounds__(64 * kCodes) void k_code_finish(int32_t ng,
                                                            int32_t *__restrict__ parts,
                                                            CodeTotals *__restrict__ tot) {
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    int32_t *p = parts + int64_t(q) * ng;
    int run = 0;
    for (int base = 0; base < ng; base += 512) {
        int v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int k = base + 64 * u + lane;
            v[u] = k < ng ? p[k] : 0;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int k = base + 64 * u + lane;
            const int incl = wave_incl_sum(v[u]);
            if (k < ng) p[k] = run + incl - v[u];
            run += __builtin_amdgcn_readlane(incl, 63);
        }
    }
    if (lane == 0) tot->c[q] = run;
}
__global__ __launch_bounds__(kThreads) void k_code_list(int32_t n, const int32_t *__restrict__ use,
                                                       const int32_t *__restrict__ parts,
                                                       const CodeTotals *__restrict__ tot,
                                                       int32_t *__restrict__ list) {
    __shared__ int s_c[kThreads / 64][kListed];
    const int i = blockIdx.x * kThreads + threadIdx.x;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int u = i < n ? use[i] : 0;
    uint64_t m = 0ull;
#pragma unroll
    for (int q = 0; q < kListed; ++q) {
        const uint64_t b = __ballot(u == q + 1);
        if (u == q + 1) m = b;
        if (lane == 0) s_c[w][q] = __popcll(b);
    }
    __syncthreads();
    if (u < 1 || u > kListed) return;
    int pos = parts[int64_t(u - 1) * gridDim.x + blockIdx.x] + __popcll(m & ((1ull << lane) - 1ull));
    for (int q = 0; q < u - 1; ++q) pos += tot->c[q];
    for (int q = 0; q < w; ++q) pos += s_c[q][u - 1];
    list[pos] = i;
}

// upper bound of each listed row's candidates (k_extpi_ub) and, for the rows
// of the thread kernel (from t_thread on), its table: the power of two at or
// above twice its candidates and strong dependencies
__global__ __launch_bounds__(kThreads) void k_listed_sizes(
    int32_t count, const int32_t *__restrict__ list, int32_t t_thread,
    const int32_t *__restrict__ SI, const int32_t *__restrict__ SJ, const int32_t *__restrict__ cf,
    int64_t *__restrict__ ub, int64_t *__restrict__ hs) {
    const int t = blockIdx.x * kThreads + threadIdx.x;
    if (t >= count) return;
    const int i = list[t];
    int64_t u = 0;
    for (int p = SI[i]; p < SI[i + 1]; ++p) {
        const int i1 = SJ[p];
        if (cf[i1] >= 0) u += 1;
        else if (cf[i1] != -3) u += SI[i1 + 1] - SI[i1];
    }
    ub[t] = u;
    int64_t z = 0;
    if (t >= t_thread) {
        const int64_t need = 2 * (u + (SI[i + 1] - SI[i]));
        z = 1;
        while (z < need) z <<= 1;
    }
    hs[t] = z;
}

__global__ __launch_bounds__(kThreads) void k_extpi_out(
    int32_t n, const int32_t *__restrict__ PI, RowSlots rows, const int32_t *__restrict__ f2c,
    int32_t *__restrict__ PJ, double *__restrict__ PA) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const int64_t s = rows.at(i);
    const int len = PI[i + 1] - PI[i];
    for (int q = 0; q < len; ++q) {
        PJ[PI[i] + q] = f2c[rows.sj[s + q]];
        PA[PI[i] + q] = rows.sw[s + q];
    }
}

// the same with a thread per slot (a power of two of slots per row)
__global__ __launch_bounds__(kThreads) void k_extpi_out_slots(
    int64_t slots, int shift, const int32_t *__restrict__ PI, RowSlots rows,
    const int32_t *__restrict__ f2c, int32_t *__restrict__ PJ, double *__restrict__ PA) {
    const int64_t t = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (t >= slots) return;
    const int i = int(t >> shift), q = int(t) & ((1 << shift) - 1);
    const int p = PI[i];
    if (q >= PI[i + 1] - p) return;
    PJ[p + q] = f2c[rows.sj[t]];
    PA[p + q] = rows.sw[t];
}

struct Tmp {
    hipStream_t s;
    std::vector<void *> ptrs;
    explicit Tmp(hipStream_t st) : s(st) {}
    ~Tmp() {
        for (void *p : ptrs) tmp_free(p, s);
    }
    template <typename T>
    int get(T **p, size_t n) {
        const int st = tmp_alloc_t(p, n, s);
        if (st == AMGT_OK) ptrs.push_back(*p);
        return st;
    }
};

}  // namespace

}  // namespace amgt

using namespace amgt;

extern "C" {

int amgt_amg_strength(int32_t n, const int32_t *A_i, const int32_t *A_j, const double *A_data,
                      double theta, double max_row_sum, int64_t *nnzS, int32_t **S_i,
                      int32_t **S_j, void *stream) {
    AMGT_CHECK_ARG(nnzS && S_i && S_j, "NULL output argument");
    AMGT_CHECK_ARG(n >= 0, "negative size");
    // column and value arrays may be NULL when the matrix has no entries
    AMGT_CHECK_ARG(n == 0 || A_i, "NULL row pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    *nnzS = 0;
    *S_i = nullptr;
    *S_j = nullptr;
    Tmp tmp(s);
    int32_t *cnt = nullptr;
    AMGT_TRY(tmp.get(&cnt, size_t(n) + 1));
    int32_t *si = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * (size_t(n) + 1), s));
    if (!si) {
        set_error("allocation of S row pointer failed");
        return AMGT_ERR_ALLOC;
    }
    // rows per workgroup: 1024 workgroups if there are rows for them (eight each)
    int32_t per = 8;
    while (per < kThreads && int64_t(n) >= int64_t(2 * per) * 1024) per *= 2;
    const dim3 wgs(unsigned((int64_t(n) + per - 1) / per));
    if (n > 0) {
        hipLaunchKernelGGL((k_strength<false>), wgs, dim3(kThreads), 0, s, n, per, A_i, A_j,
                           A_data, theta, max_row_sum, cnt, nullptr, nullptr);
        AMGT_HIP(hipGetLastError());
    }
    int st = exclusive_scan_i32(cnt, si, n, s);
    if (st != AMGT_OK) {
        dev_free(si, s);
        return st;
    }
    int32_t total = 0;
    {
        const Readback rb[1] = {{&total, si + n, sizeof(int32_t)}};
        AMGT_TRY(readback(rb, 1, s));
    }
    int32_t *sjj = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * (size_t(total) + 1), s));
    if (!sjj) {
        dev_free(si, s);
        set_error("allocation of S columns failed");
        return AMGT_ERR_ALLOC;
    }
    if (n > 0) {
        hipLaunchKernelGGL((k_strength<true>), wgs, dim3(kThreads), 0, s, n, per, A_i, A_j, A_data, theta, max_row_sum, nullptr, si, sjj);
        AMGT_HIP(hipGetLastError());
    }
    *nnzS = total;
    *S_i = si;
    *S_j = sjj;
    return AMGT_OK;
}

int amgt_amg_pmis(int32_t n, const int32_t *S_i, const int32_t *S_j, int cf_init,
                  int32_t *cf_marker, int32_t *n_coarse, void *stream) {
    AMGT_CHECK_ARG(n_coarse, "NULL output argument");
    AMGT_CHECK_ARG(n >= 0, "negative size");
    AMGT_CHECK_ARG(n == 0 || (S_i && cf_marker), "NULL row pointer or marker array");
    if (cf_init != 0 && cf_init != 1 && cf_init != 2) {
        set_error("PMIS: only CF_init 0, 1 (HMIS) and 2 (coarsen types 8, 10 and 9) are supported");
        return AMGT_ERR_UNSUPPORTED;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    *n_coarse = 0;
    if (n == 0) return AMGT_OK;
    Tmp tmp(s);
    // one flag per pass: whether a node stayed undecided
    constexpr int kFlags = 64;
    int32_t *cnt = nullptr, *lost = nullptr, *any = nullptr;
    double *measure = nullptr;
    AMGT_TRY(tmp.get(&cnt, size_t(n) * 2));  // cnt and lost, cleared together
    lost = cnt + n;
    AMGT_TRY(tmp.get(&any, kFlags));
    AMGT_TRY(tmp.get(&measure, n));
    AMGT_HIP(hipMemsetAsync(cnt, 0, sizeof(int32_t) * 2 * size_t(n), s));
    AMGT_HIP(hipMemsetAsync(any, 0, sizeof(int32_t) * kFlags, s));
    const dim3 g(grid_of(n)), b(kThreads);
    hipLaunchKernelGGL(k_col_count, g, b, 0, s, n, S_i, S_j, cnt);
    if (cf_init == 1)
        hipLaunchKernelGGL(k_pmis_init_hmis, g, b, 0, s, n, S_i, cnt, measure, cf_marker, any);
    else
        hipLaunchKernelGGL(k_pmis_init, g, b, 0, s, n, S_i, cnt, measure, cf_marker, any);
    AMGT_HIP(hipGetLastError());
    // Every pass decides at least the nodes of largest measure, so the loop
    // ends within n passes.  A pass after the last one changes nothing, so on
    // small levels, where waiting for the flag costs more than a pass, every
    // second flag is read (and none after the start: an empty graph is as good
    // as any).
    const int per_check = n <= 65536 ? 2 : 1;
    int32_t h_any = 1;
    if (per_check == 1) {
        const Readback rb[1] = {{&h_any, any, sizeof(int32_t)}};
        AMGT_TRY(readback(rb, 1, s));
    }
    int flag = 0;  // the last pass's flag
    for (int64_t iter = 0; h_any && iter <= int64_t(n) + 1; ++iter) {
        if (!cf_init || iter) {
            hipLaunchKernelGGL(k_pmis_clear, g, b, 0, s, n, S_i, S_j, measure, lost);
            hipLaunchKernelGGL(k_pmis_set, g, b, 0, s, n, measure, lost, cf_marker);
        }
        if (++flag == kFlags) {
            AMGT_HIP(hipMemsetAsync(any, 0, sizeof(int32_t) * kFlags, s));
            flag = 0;
        }
        hipLaunchKernelGGL(k_pmis_cf, g, b, 0, s, n, S_i, S_j, measure, cf_marker, lost,
                           any + flag);
        AMGT_HIP(hipGetLastError());
        if (iter % per_check == per_check - 1) {
            const Readback rb[1] = {{&h_any, any + flag, sizeof(int32_t)}};
            AMGT_TRY(readback(rb, 1, s));
        }
    }
    if (h_any) {
        set_error("PMIS did not converge");
        return AMGT_ERR_INPUT;
    }
    rowpass::Part *parts = nullptr;
    RowStats *tot = nullptr;
    RowStats ht{};
    AMGT_TRY(tmp.get(&parts, size_t(rowpass::groups(n))));
    AMGT_TRY(tmp.get(&tot, 1));
    AMGT_TRY(rowpass::count(n, NotCoarse{cf_marker}, 0, 0, parts, tot, s));
    const Readback rb[1] = {{&ht, tot, sizeof(RowStats)}};
    AMGT_TRY(readback(rb, 1, s));
    *n_coarse = ht.cnt[0];
    return AMGT_OK;
}

int amgt_amg_extpi_interp(int32_t n, const int32_t *A_i, const int32_t *A_j,
                          const double *A_data, const int32_t *S_i, const int32_t *S_j,
                          const int32_t *cf_marker, int max_elmts, int32_t *n_coarse,
                          int64_t *nnzP, int32_t **P_i, int32_t **P_j, double **P_data,
                          void *stream) {
    AMGT_CHECK_ARG(n_coarse && nnzP && P_i && P_j && P_data, "NULL output argument");
    AMGT_CHECK_ARG(n >= 0 && max_elmts >= 0, "negative size");
    AMGT_CHECK_ARG(n == 0 || (A_i && S_i && cf_marker), "NULL row pointer or marker array");
    hipStream_t s = static_cast<hipStream_t>(stream);
    *n_coarse = 0;
    *nnzP = 0;
    *P_i = nullptr;
    *P_j = nullptr;
    *P_data = nullptr;
    Tmp tmp(s);
    const dim3 g(grid_of(n)), b(kThreads);
    // Rows truncated to a few entries get a fixed slot each (a power of two,
    // so that the output kernel takes a thread per slot); otherwise the slots
    // are sized by the rows' upper bounds.
    constexpr int kMaxSlot = 16;
    int shift = 0;  // of the fixed slots
    RowSlots slots{};
    int32_t *flag = nullptr, *f2c = nullptr, *cnt = nullptr, *use = nullptr, *ovf = nullptr;
    int8_t *dneg = nullptr;
    int32_t *parts = nullptr;
    CodeTotals *tot = nullptr;
    AMGT_TRY(tmp.get(&flag, size_t(n) + 1));
    AMGT_TRY(tmp.get(&f2c, size_t(n) + 1));
    AMGT_TRY(tmp.get(&cnt, size_t(n) + 1));
    AMGT_TRY(tmp.get(&use, size_t(n) + 1));
    AMGT_TRY(tmp.get(&dneg, size_t(n) + 1));
    AMGT_TRY(tmp.get(&ovf, 1));
    AMGT_TRY(tmp.get(&parts, size_t(g.x) * kCodes + 1));
    AMGT_TRY(tmp.get(&tot, 1));
    int64_t total_slots = 0;
    if (max_elmts > 0 && max_elmts <= kMaxSlot) {
        while ((1 << shift) < max_elmts) ++shift;
        slots.stride = 1 << shift;
        total_slots = int64_t(n) << shift;
    } else {
        int64_t *ub = nullptr, *off = nullptr;
        AMGT_TRY(tmp.get(&ub, size_t(n) + 1));
        AMGT_TRY(tmp.get(&off, size_t(n) + 1));
        if (n > 0)
            hipLaunchKernelGGL(k_extpi_ub, g, b, 0, s, n, S_i, S_j, cf_marker, ub);
        AMGT_HIP(hipGetLastError());
        AMGT_TRY(exclusive_scan_i64(ub, off, n, s));
        const Readback rb[1] = {{&total_slots, off + n, sizeof(int64_t)}};
        AMGT_TRY(readback(rb, 1, s));
        slots.off = off;
    }
    AMGT_TRY(tmp.get(&slots.sj, size_t(total_slots)));
    AMGT_TRY(tmp.get(&slots.sw, size_t(total_slots)));
    slots.cnt = cnt;

    // rows per kernel
    CodeTotals h{};
    int32_t nc = 0, nnz = 0, h_ovf = 0;
    auto count_codes = [&]() -> int {
        hipLaunchKernelGGL(k_code_part, g, b, 0, s, n, use, int32_t(g.x), parts);
        hipLaunchKernelGGL(k_code_finish, dim3(1), dim3(64 * kCodes), 0, s, int32_t(g.x), parts,
                           tot);
        AMGT_HIP(hipGetLastError());
        return AMGT_OK;
    };
    if (n > 0) {
        hipLaunchKernelGGL(k_extpi_class, g, b, 0, s, n, A_i, A_j, A_data, S_i, cf_marker,
                           n <= kWaveMaxRows ? 512 : 256, flag, use, dneg, slots);
        AMGT_TRY(count_codes());
    }
    AMGT_TRY(exclusive_scan_i32(flag, f2c, n, s));
    if (n > 0) {
        const Readback rb[2] = {{&nc, f2c + n, sizeof(int32_t)}, {&h, tot, sizeof(CodeTotals)}};
        AMGT_TRY(readback(rb, 2, s));
    }
    AMGT_HIP(hipMemsetAsync(ovf, 0, sizeof(int32_t), s));
    int32_t *pi = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * (size_t(n) + 1), s));
    if (!pi) {
        set_error("allocation of P row pointer failed");
        return AMGT_ERR_ALLOC;
    }
    auto fail = [&](int st) {
        dev_free(pi, s);
        return st;
    };
    // the listed rows, then those that overflowed a table (at most kTier64,
    // its large table, the thread kernel: each round moves a row on)
    auto listed_rows = [&]() -> int {
        int32_t np = 0;
        for (int q = 0; q < kListed; ++q) np += h.c[q];
        if (np == 0) return AMGT_OK;
        int32_t *list = nullptr, *wcol = nullptr;
        int64_t *ub = nullptr, *woff = nullptr, *hs = nullptr, *hoff = nullptr;
        double *wval = nullptr;
        int2 *hkv = nullptr;
        const int32_t nthread = h.c[kThreadRow - 1];
        AMGT_TRY(tmp.get(&list, size_t(np)));
        AMGT_TRY(tmp.get(&ub, size_t(np) + 1));
        AMGT_TRY(tmp.get(&woff, size_t(np) + 1));
        AMGT_TRY(tmp.get(&hs, size_t(np) + 1));
        hipLaunchKernelGGL(k_code_list, g, b, 0, s, n, use, parts, tot, list);
        hipLaunchKernelGGL(k_listed_sizes, dim3(grid_of(np)), b, 0, s, np, list, np - nthread, S_i,
                           S_j, cf_marker, ub, hs);
        AMGT_HIP(hipGetLastError());
        AMGT_TRY(exclusive_scan_i64(ub, woff, np, s));
        int64_t total_w = 0, total_h = 0, wfirst = 0;
        if (nthread > 0) {  // (the thread kernel's rows are the last ones)
            AMGT_TRY(tmp.get(&hoff, size_t(np) + 1));
            AMGT_TRY(exclusive_scan_i64(hs, hoff, np, s));
            const Readback rb[3] = {{&total_w, woff + np, sizeof(int64_t)},
                                    {&total_h, hoff + np, sizeof(int64_t)},
                                    {&wfirst, woff + (np - nthread), sizeof(int64_t)}};
            AMGT_TRY(readback(rb, 3, s));
            AMGT_TRY(tmp.get(&wval, size_t(total_w - wfirst)));
            AMGT_TRY(tmp.get(&hkv, size_t(total_h)));
            AMGT_HIP(hipMemsetAsync(hkv, 0xff, sizeof(int2) * size_t(total_h), s));
        } else {
            const Readback rb[1] = {{&total_w, woff + np, sizeof(int64_t)}};
            AMGT_TRY(readback(rb, 1, s));
        }
        AMGT_TRY(tmp.get(&wcol, size_t(total_w)));
        int32_t t0 = 0;
        for (int code = 1; code <= kListed; ++code) {
            const int32_t cw = h.c[code - 1];
            if (cw == 0) continue;
            const int32_t *rows = list + t0;
            const int64_t *wo = woff + t0;
#define AMGT_EXTPI_WAVE(WA_, WT_, WH_, NEXT_)                                                  \
    hipLaunchKernelGGL((k_extpi_wave<WA_, WT_, WH_>), dim3(unsigned(cw)), dim3(64), 0, s, cw,  \
                       rows, A_i, A_j, A_data, S_i, S_j, cf_marker, dneg, wo, wcol, max_elmts, \
                       slots, use, NEXT_, ovf)
            switch (code) {
                case kTier64: AMGT_EXTPI_WAVE(64, 128, 512, kTier64Big); break;      // 8.5 KB
                case kTier64Big: AMGT_EXTPI_WAVE(64, 384, 1024, kThreadRow); break;  // 15.5 KB
                case kTier128: AMGT_EXTPI_WAVE(128, 256, 1024, kTier128Big); break;  // 17 KB
                case kTier256: AMGT_EXTPI_WAVE(256, 768, 2048, kTier256Big); break;  // 37 KB
                case kTier128Big: AMGT_EXTPI_WAVE(256, 768, 2048, kThreadRow); break;
                case kTier256Big: AMGT_EXTPI_WAVE(256, 1536, 4096, kThreadRow); break;  // 62 KB
                case kTier512: AMGT_EXTPI_WAVE(512, 1536, 4096, kThreadRow); break;  // 74 KB
                default:
                    hipLaunchKernelGGL(k_extpi_row, dim3(grid_of(cw)), b, 0, s, cw, rows, A_i, A_j,
                                       A_data, S_i, S_j, cf_marker, max_elmts, wo, wfirst, wcol, wval,
                                       hoff + t0, hkv, slots, use);
            }
#undef AMGT_EXTPI_WAVE
            t0 += cw;
        }
        AMGT_HIP(hipGetLastError());
        return AMGT_OK;
    };
    // (after the lists of round 0 are written: an overflow changes the row's code)
    auto group_rows = [&]() -> int {
        // rows per workgroup: up to 256 (its groups then take rows of this kernel
        // only, one after the other), fewer on small levels, where the time is that
        // of one group's rows (512^2 5-pt, level 3, 3481 rows of 27: 797 us with
        // 256, the wave kernel 327)
#define AMGT_EXTPI_GROUP(G_, CODE_)                                                            \
    if (h.c[CODE_ - 1] > 0) {                                                                  \
        const int per = std::max(kThreads / G_, std::min(kThreads, (n + 2047) / 2048));        \
        hipLaunchKernelGGL((k_extpi_group<G_>), dim3(unsigned((n + per - 1) / per)), b, 0, s,  \
                           n, A_i, A_j, A_data, S_i, S_j, cf_marker, dneg, max_elmts, slots,   \
                           use, per, CODE_, kTier64, ovf);                                     \
    }
        AMGT_EXTPI_GROUP(8, kGroup8);
        AMGT_EXTPI_GROUP(16, kGroup16);
        AMGT_EXTPI_GROUP(32, kGroup32);
#undef AMGT_EXTPI_GROUP
        AMGT_HIP(hipGetLastError());
        return AMGT_OK;
    };
    for (int round = 0; n > 0 && round < 4; ++round) {
        int st = listed_rows();
        if (st == AMGT_OK && round == 0) st = group_rows();
        if (st == AMGT_OK) st = exclusive_scan_i32(cnt, pi, n, s);
        if (st == AMGT_OK) {
            const Readback rb[2] = {{&nnz, pi + n, sizeof(int32_t)}, {&h_ovf, ovf, sizeof(int32_t)}};
            st = readback(rb, 2, s);
        }
        if (st == AMGT_OK && h_ovf == 0) break;
        if (st == AMGT_OK) st = count_codes();
        if (st == AMGT_OK) {
            const Readback rb[1] = {{&h, tot, sizeof(CodeTotals)}};
            st = readback(rb, 1, s);
        }
        if (st == AMGT_OK && hipMemsetAsync(ovf, 0, sizeof(int32_t), s) != hipSuccess)
            st = AMGT_ERR_HIP;
        if (st != AMGT_OK) return fail(st);
    }
    if (n == 0) AMGT_TRY(exclusive_scan_i32(cnt, pi, 0, s));
    int32_t *pj = static_cast<int32_t *>(dev_alloc(sizeof(int32_t) * (size_t(nnz) + 1), s));
    double *pa = static_cast<double *>(dev_alloc(sizeof(double) * (size_t(nnz) + 1), s));
    if (!pj || !pa) {
        set_error("allocation of P failed");
        if (pj) dev_free(pj, s);
        if (pa) dev_free(pa, s);
        return fail(AMGT_ERR_ALLOC);
    }
    if (n > 0) {
        if (slots.stride > 0)
            hipLaunchKernelGGL(k_extpi_out_slots, dim3(grid_of(total_slots)), b, 0, s, total_slots,
                               shift, pi, slots, f2c, pj, pa);
        else
            hipLaunchKernelGGL(k_extpi_out, g, b, 0, s, n, pi, slots, f2c, pj, pa);
        if (hipGetLastError() != hipSuccess) {
            set_error("extended+i interpolation: kernel launch failed");
            dev_free(pj, s);
            dev_free(pa, s);
            return fail(AMGT_ERR_HIP);
        }
    }
    *n_coarse = nc;
    *nnzP = nnz;
    *P_i = pi;
    *P_j = pj;
    *P_data = pa;
    return AMGT_OK;
}

}  // extern "C"
