/*
 * FP64 column kernel for wide columns (adaptive builds, and static ones past the
 * given-pattern kernels): one column of M per workgroup of eight waves,
 * |J| <= 40, |I| <= 384.
 *
 * What bounds it: few columns reach these sizes (954 of the 262,144-column
 * random band), so the launch takes as long as its slowest column: six steps
 * of up to 33 columns by 364 rows and 3,500 candidates there.  One wave per
 * column spent 1.8 to 2.1 ms in a chain of LDS passes.  Eight waves split the
 * columns of A(I,J) (column j on wave j % 8) and keep them in registers, six
 * rows to a lane; a reflector costs one barrier (its column through LDS,
 * double buffered) and at most six dot products per wave.  The index sets need
 * no sort of I: distinct rows come from an LDS hash, a row's position is the
 * number of smaller rows.  Candidates come out of a bitmap over their range
 * (bitonic sort past 294,912 indices); their scores add the entries of I's
 * rows, which are a tenth of what the candidates' columns hold: one bucket of
 * entries per candidate instead of a pass over its column (3.7 against 55 us
 * per step of that slowest column) or over the rows one by one.  The launch
 * takes 0.50 ms on the 50,021-column band and 0.56 ms on the 262,144-column
 * one, FP64, against 1.79 and 2.09 ms; most of it is the QR (40 us per solve),
 * bound by VALU issue: two waves to a SIMD and the norm formed by each.
 *
 * Every rounding is that of the fixed 64-lane order (row r on lane r % 64, a
 * lane's rows in order, then the butterfly) and of the sequential sums: the
 * same bits as the one-wave kernels, whose saved states it resumes and which
 * resume its own.
 */
#include "device_common.h"
#include "spai_host.h"

namespace mspai {

namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kJ = kWideJ, kI = kWideI, kU = kWideU, kRaw = kWideRaw;
constexpr int kRowsLane = kI / kWave;                     // rows per lane
constexpr int kCols = (kJ + 1 + kWaves - 1) / kWaves;     // columns per wave, the right-hand side among them
constexpr int kSlots = (kCols + 3) / 4 * 4;               // sums formed four at a time
constexpr int kHash = 1024;                               // slots of the row hash
constexpr int kPer = kU / kThreads;                       // scores per thread
static_assert(kI % kWave == 0 && kI + 1 <= kThreads && kHash >= 2 * kI, "sizes");

struct WideLds {
    union {
        double A[kJ * kI];  // A(I,J), column-major: from the gather to the residual
        struct {            // the augmentation
            int raw[kRaw];
            int cand[kU];
            union {
                unsigned bits[(kJ * kI * 2) - kRaw - kU];  // the bitmap and its words' ranks
                struct {                                   // then the raw entries by candidate, and the scores
                    int bucket[kRaw];
                    int first[kU + 1];
                };
                double score[kU];
            };
        };
    };
    double R[kJ * (kJ + 1) / 2];  // columns packed
    double qb[kJ];
    double v[2][kI];
    double rhs[kI];
    double r[kI];
    double x[kJ];
    double wsum[kNumWork];
    double red[kWaves];
    int ired[kWaves];
    int J[kJ];
    int rows[kI];  // distinct rows in order of arrival
    int key[kHash];
    unsigned short rank[kHash];  // position in sorted I of the row in a slot
    unsigned short slot_of[kI];
    int segs[kJ];
    int segoff[kJ + 1];
    int rowbase[kI];  // row of I by position: its place in the row pattern, less its place in the raw list
    int sel[kJ];
    int count;
};
constexpr int kWords = sizeof(WideLds::bits) / sizeof(unsigned) / 2;  // bitmap words
static_assert(kRaw == 1 << 13 && kI < 1 << 18, "a bucket's entry packs the row above its place in the raw list");

__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave); }

/* Reduction over the workgroup with an operation that any order serves. */
template <class T, class Op>
__device__ __forceinline__ T block_reduce(T v, T* red, Op op)
{
    v = Group<kWave>::allreduce(v, op);
    if (lane_id() == 0) red[wave_index()] = v;
    __syncthreads();
    T t = red[0];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) t = op(t, red[k]);
    __syncthreads();
    return t;
}
__device__ __forceinline__ int block_sum(WideLds& w, int v)
{
    return block_reduce(v, w.ired, [](int a, int b) { return a + b; });
}
__device__ __forceinline__ double block_sum(WideLds& w, double v)
{
    return block_reduce(v, w.red, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double block_min(WideLds& w, double v)
{
    return block_reduce(v, w.red, [](double a, double b) { return fmin(a, b); });
}
__device__ __forceinline__ int block_min(WideLds& w, int v)
{
    return block_reduce(v, w.ired, [](int a, int b) { return a < b ? a : b; });
}
__device__ __forceinline__ int block_max(WideLds& w, int v)
{
    return block_reduce(v, w.ired, [](int a, int b) { return a > b ? a : b; });
}
__device__ __forceinline__ bool block_any(WideLds& w, bool p) { return block_sum(w, (int)p) != 0; }

/* Exclusive prefix sum over the threads; *total: the sum. */
__device__ __forceinline__ int block_scan(WideLds& w, int v, int* total)
{
    const int incl = Group<kWave>::scan_incl(v);
    if (lane_id() == kWave - 1) w.ired[wave_index()] = incl;
    __syncthreads();
    int off = 0, sum = 0;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
        off += k < wave_index() ? w.ired[k] : 0;
        sum += w.ired[k];
    }
    __syncthreads();
    *total = sum;
    return off + incl - v;
}

__device__ __forceinline__ unsigned row_slot(int row) { return ((unsigned)row * 0x9e3779b1u) >> 22; }
static_assert(kHash == 1 << 10, "row_slot");

/* More distinct rows have arrived than the working set holds. */
__device__ __forceinline__ bool rows_full(const WideLds& w)
{
    return __hip_atomic_load(&w.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > kI;
}

/* Slot of `row`, added when new.  -1: more rows than the working set holds,
 * looked at every eighth probe (in a full table every insertion would
 * otherwise walk all of it). */
__device__ __forceinline__ int row_insert(WideLds& w, int row)
{
    unsigned slot = row_slot(row);
    for (int probe = 0; probe < kHash; ++probe) {
        if ((probe & 7) == 7 && rows_full(w)) break;
        const int old = atomicCAS(&w.key[slot], -1, row);
        if (old == -1) {
            const int k = atomicAdd(&w.count, 1);
            if (k < kI) {
                w.rows[k] = row;
                w.slot_of[k] = (unsigned short)slot;
            }
            return (int)slot;
        }
        if (old == row) return (int)slot;
        slot = (slot + 1) & (kHash - 1);
    }
    return -1;
}

/* Position of `row` in sorted I, or -1. */
__device__ __forceinline__ int row_position(const WideLds& w, int row)
{
    unsigned slot = row_slot(row);
    for (int probe = 0; probe < kHash; ++probe) {
        const int k = w.key[slot];
        if (k == row) return w.rank[slot];
        if (k == -1) return -1;
        slot = (slot + 1) & (kHash - 1);
    }
    return -1;
}

/* Column of J that holds flat entry e of its columns. */
__device__ __forceinline__ int entry_column(const WideLds& w, int n, int e)
{
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (w.segoff[mid] <= e) lo = mid;
        else hi = mid;
    }
    return lo;
}

/* The distinct rows of J's columns (Get_I_Set, src/Spai_Sub.imp:65-122) with
 * their positions; |I|, or -1 when they are more than kI. */
__device__ __forceinline__ int index_set(const BuildArgs& a, WideLds& w, int n)
{
    const int tid = threadIdx.x;
    for (int t = tid; t < kHash; t += kThreads) w.key[t] = -1;
    if (tid < kI) w.rows[tid] = 0x7fffffff;
    if (tid == 0) w.count = 0;
    int start = 0, cnt = 0, total;
    if (tid < n) {
        start = a.A.colptr[w.J[tid]];
        cnt = a.A.colptr[w.J[tid] + 1] - start;
    }
    const int off = block_scan(w, cnt, &total);
    if (tid < n) {
        w.segs[tid] = start;
        w.segoff[tid] = off;
    }
    if (tid == 0) w.segoff[n] = total;
    __syncthreads();
    /* n columns with at most kI distinct rows each: a longer list cannot fit
     * (inserting one of 10,000 entries took 1.9 ms) */
    if (total > n * kI) return -1;
    for (int e = tid; e < total && !rows_full(w); e += kThreads) {
        const int t = entry_column(w, n, e);
        row_insert(w, a.A.rowind[w.segs[t] + e - w.segoff[t]]);
    }
    __syncthreads();
    const int m = w.count;
    if (m > kI) return -1;
    if (tid < m) {
        const int mine = w.rows[tid];
        int rk = 0;
        for (int u = 0; u < m; u += 4) {
            const int4 o = *reinterpret_cast<const int4*>(&w.rows[u]);
            rk += (o.x < mine) + (o.y < mine) + (o.z < mine) + (o.w < mine);
        }
        w.rank[w.slot_of[tid]] = (unsigned short)rk;
    }
    __syncthreads();
    return m;
}

/* A(I,J) and the right-hand side (Create_submatrix, Create_ek_Hat /
 * Create_bk_Hat); the status bit of a target outside I. */
__device__ __forceinline__ int gather(const BuildArgs& a, WideLds& w, int m, int n, int col)
{
    const int tid = threadIdx.x;
    for (int j = wave_index(); j < n; j += kWaves)
        for (int r = lane_id(); r < kI; r += kWave)
            if (r < m) w.A[j * kI + r] = 0.0;
    if (tid < kI) w.rhs[tid] = 0.0;
    __syncthreads();
    const int total = w.segoff[n];
    for (int e = tid; e < total; e += kThreads) {
        const int t = entry_column(w, n, e);
        const int src = w.segs[t] + e - w.segoff[t];
        const double val = a.A.val[src];
        w.A[t * kI + row_position(w, a.A.rowind[src])] = val;  // every row of J's columns is in I
    }
    bool hit = false;
    if (!a.B.colptr) {
        const int pos = row_position(w, col);
        hit = pos >= 0;
        if (hit && tid == 0) w.rhs[pos] = 1.0;
    } else {
        const int e1 = a.B.colptr[col + 1];
        for (int e = a.B.colptr[col] + tid; e < e1; e += kThreads) {
            const int pos = row_position(w, a.B.rowind[e]);
            if (pos >= 0) {
                hit = true;
                w.rhs[pos] = a.B.val[e];
            }
        }
        hit = block_any(w, hit);
    }
    __syncthreads();
    return hit ? 0 : COL_K_NOT_IN_I;
}

/* Approximative_Solution (src/Spai_Unrestrained.imp:135-195): Householder QR
 * with Q^T b carried along, back substitution; x in w.x.  Status bits. */
__device__ __forceinline__ int solve(WideLds& w, int m, int n)
{
    const int lane = lane_id(), wave = wave_index();
    double x[kCols][kRowsLane];
#pragma unroll
    for (int s = 0; s < kCols; ++s) {
        const int j = wave + kWaves * s;
#pragma unroll
        for (int q = 0; q < kRowsLane; ++q) {
            const int r = lane + kWave * q;
            x[s][q] = 0.0;
            if (r < m && j < n) x[s][q] = w.A[j * kI + r];
            if (r < m && j == n) x[s][q] = w.rhs[r];
        }
    }
    const int k = m < n ? m : n;
    bool singular = false;
#pragma unroll
    for (int si = 0; si < kCols; ++si) {
        if (kWaves * si >= k) break;
#pragma unroll 1
        for (int c = 0; c < kWaves; ++c) {
            const int i = kWaves * si + c;
            if (i >= k) break;
            double* const vb = w.v[c & 1];
            if (wave == c) {
#pragma unroll
                for (int q = 0; q < kRowsLane; ++q)
                    if (kWave * q < m) vb[lane + kWave * q] = x[si][q];
            }
            /* the other buffer's readers passed the barrier of the step before */
            __syncthreads();
            double v[kRowsLane];
#pragma unroll
            for (int q = 0; q < kRowsLane; ++q) v[q] = kWave * q < m ? vb[lane + kWave * q] : 0.0;
            const double alpha = vb[i];
            double p = 0.0;
#pragma unroll
            for (int q = 0; q < kRowsLane; ++q) {
                const int r = lane + kWave * q;
                if (r > i && r < m) p = __fma_rn(v[q], v[q], p);
            }
            const double xn2 = Group<kWave>::sum_fixed(p);
            double rii = alpha;
            if (i + 1 < m && xn2 != 0.0) {
                const double nrm = sqrt(__fma_rn(alpha, alpha, xn2));
                const double beta = -copysign(nrm, alpha);
                const double tau = (beta - alpha) / beta;
                const double scal = 1.0 / (alpha - beta);
                const double mt = -tau;
                rii = beta;
#pragma unroll
                for (int q = 0; q < kRowsLane; ++q) v[q] = v[q] * scal;
                v[0] = lane == i ? 1.0 : v[0];
                /* the wave's columns after i, from the first slot that may hold one */
                const int s0 = wave > c ? si : si + 1;
                double d[kSlots];
#pragma unroll
                for (int s = 0; s < kSlots; ++s) d[s] = 0.0;
#pragma unroll
                for (int q = 0; q < kRowsLane; ++q) {
                    const int r = lane + kWave * q;
                    if (r >= i && r < m) {
#pragma unroll
                        for (int s = si; s < kCols; ++s) d[s] = __fma_rn(v[q], x[s][q], d[s]);
                    }
                }
#pragma unroll
                for (int s = 0; s < kSlots; s += 4) {
                    if (s + 4 > si && wave + kWaves * s <= n) {
                        double t[4] = {d[s], d[s + 1], d[s + 2], d[s + 3]};
                        Group<kWave>::sum4_bcast(t);
#pragma unroll
                        for (int u = 0; u < 4; ++u) d[s + u] = mt * t[u];
                    }
                }
#pragma unroll
                for (int q = 0; q < kRowsLane; ++q) {
                    const int r = lane + kWave * q;
                    if (r >= i && r < m) {
#pragma unroll
                        for (int s = si; s < kCols; ++s)
                            if (s >= s0) x[s][q] = __fma_rn(v[q], d[s], x[s][q]);
                    }
                }
                if (wave == c) x[si][0] = lane == i ? beta : x[si][0];
            }
            singular |= rii == 0.0;
        }
    }
    /* R and Q^T b: rows below |J| sit in the first of a lane's rows */
#pragma unroll
    for (int s = 0; s < kCols; ++s) {
        const int j = wave + kWaves * s;
        if (j < n && lane <= j) w.R[j * (j + 1) / 2 + lane] = x[s][0];
        if (j == n && lane < n) w.qb[lane] = x[s][0];
    }
    __syncthreads();
    int st = 0;
    double b = lane < n ? w.qb[lane] : 0.0;
    if (m < n) {
        st = COL_UNDERDET;
        b = 0.0;
    } else if (singular) {
        st = COL_SINGULAR;
    } else if (wave == 0) {  // dtrsm order; a singular R leaves Q^T b
        for (int K = n - 1; K >= 0; --K) {
            double xk = Group<kWave>::lane_value(b, K);
            if (xk != 0.0) {
                xk = xk / w.R[K * (K + 1) / 2 + K];
                if (lane == K) b = xk;
                else if (lane < K) b = __fma_rn(-xk, w.R[K * (K + 1) / 2 + lane], b);
            }
        }
    }
    if (wave == 0 && lane < n) w.x[lane] = b;
    __syncthreads();
    return st;
}

/* Residual_Norm (src/Spai_Sub.imp:915-941): r = A(I,J) x - b in dgemv's
 * column order, the norm from the sequential sum of squares. */
__device__ __forceinline__ double residual(WideLds& w, int m, int n)
{
    const int tid = threadIdx.x;
    double* const sq = w.v[0];
    if (tid < m) {
        double r = -w.rhs[tid];
#pragma unroll 4
        for (int j = 0; j < n; ++j) {
            const double xj = w.x[j];
            const double t = __fma_rn(xj, w.A[j * kI + tid], r);
            r = xj != 0.0 ? t : r;
        }
        w.r[tid] = r;
        sq[tid] = __dmul_rn(r, r);
    } else if (tid < kI) {
        sq[tid] = 0.0;
    }
    __syncthreads();
    double sum = 0.0;  // formed by every thread; a row past |I| adds +0
    for (int r = 0; r < m; r += 8) {
        double2 d[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = *reinterpret_cast<const double2*>(sq + r + 2 * q);
#pragma unroll
        for (int q = 0; q < 4; ++q) sum = __dadd_rn(__dadd_rn(sum, d[q].x), d[q].y);
    }
    return sqrt(sum);
}
static_assert(kI % 8 == 0, "the sum of squares reads eight rows at a time");

/* One step of refinement by the normal equations with the FP64 factor, as the
 * given-pattern kernels take it: x -= (R^T R)^-1 A^T r, r = A x - b of the last
 * residual, unless the step is larger than 1e-10 max|x| (or NaN).  Bins of a
 * mixed chain only, whose other kernels refine an FP32 solution: the unrefined
 * QR is further from the exact solution (random band, columns of 112 to 329
 * rows: 1.8e-16 against 0.5e-16 of max|x| on average). */
__device__ __forceinline__ void refine(WideLds& w, int m, int n)
{
    const int lane = lane_id();
    for (int j = wave_index(); j < n; j += kWaves) {
        double p = 0.0;
#pragma unroll
        for (int q = 0; q < kRowsLane; ++q) {
            const int r = lane + kWave * q;
            if (r < m) p = __fma_rn(w.A[j * kI + r], w.r[r], p);
        }
        p = Group<kWave>::sum_fixed(p);
        if (lane == 0) w.qb[j] = p;
    }
    __syncthreads();
    if (wave_index() == 0) {
        const double x = lane < n ? w.x[lane] : 0.0;
        const double dinv = lane < n ? 1.0 / w.R[lane * (lane + 1) / 2 + lane] : 0.0;
        double d = lane < n ? w.qb[lane] : 0.0;
        for (int K = 0; K < n; ++K) {  // R^T y = A^T r
            const double yk = Group<kWave>::lane_value(d * dinv, K);
            if (lane == K) d = yk;
            else if (lane > K && lane < n) d = __fma_rn(-yk, w.R[lane * (lane + 1) / 2 + K], d);
        }
        for (int K = n - 1; K >= 0; --K) {  // R d = y
            const double dk = Group<kWave>::lane_value(d * dinv, K);
            if (lane == K) d = dk;
            else if (lane < K) d = __fma_rn(-dk, w.R[K * (K + 1) / 2 + lane], d);
        }
        const double xm = Group<kWave>::max(fabs(x));
        if (__ballot(lane < n && !(fabs(d) <= 1e-10 * xm)) == 0ull && lane < n) w.x[lane] = x - d;
    }
    __syncthreads();
}

/* Ascending bitonic sort of w.raw[0..count). */
__device__ __forceinline__ void sort_raw(WideLds& w, int count)
{
    const int tid = threadIdx.x;
    int N = 1;
    while (N < count) N <<= 1;
    for (int i = count + tid; i < N; i += kThreads) w.raw[i] = 0x7fffffff;
    __syncthreads();
    for (int size = 2; size <= N; size <<= 1)
        for (int j = size >> 1; j > 0; j >>= 1) {
            for (int i = tid; i < N; i += kThreads) {
                const int p = i ^ j;
                if (p > i) {
                    const int x = w.raw[i], y = w.raw[p];
                    if ((x > y) == ((i & size) == 0)) {
                        w.raw[i] = y;
                        w.raw[p] = x;
                    }
                }
            }
            __syncthreads();
        }
}

/* The candidates U \ J in increasing order into w.cand, U the distinct values
 * of w.raw[0..total), all in [lo, hi]; their number, or -1 when they are more
 * than kU.  With `slots` (the sort is not done then, which loses the order of
 * the raw list) w.raw[e] becomes the entry's place in w.cand, or -1 for an
 * entry of J. */
__device__ __forceinline__ int candidates(WideLds& w, int total, int lo, int hi, int n, bool* slots)
{
    const int tid = threadIdx.x;
    if (total == 0) return 0;
    int count = 0;
    *slots = ((hi - lo) >> 5) < kWords;
    if (*slots) {
        const int words = ((hi - lo) >> 5) + 1;
        for (int t = tid; t < words; t += kThreads) w.bits[t] = 0u;
        __syncthreads();
        for (int e = tid; e < total; e += kThreads) {
            const int d = w.raw[e] - lo;
            atomicOr(&w.bits[d >> 5], 1u << (d & 31));
        }
        __syncthreads();
        if (tid < n && w.J[tid] >= lo && w.J[tid] <= hi) {
            const int d = w.J[tid] - lo;
            atomicAnd(&w.bits[d >> 5], ~(1u << (d & 31)));
        }
        __syncthreads();
        /* an odd run of words per thread: neighbours' reads spread over the banks */
        const int per = ((words + kThreads - 1) / kThreads) | 1;
        const int t0 = tid * per, t1 = min(t0 + per, words);
        int mine = 0;
        for (int t = t0; t < t1; ++t) mine += __popc(w.bits[t]);
        int o = block_scan(w, mine, &count);
        if (count > kU) return -1;
        for (int t = t0; t < t1; ++t) {
            unsigned b = w.bits[t];
            w.bits[kWords + t] = (unsigned)o;
            while (b) {
                const int k = __ffs(b) - 1;
                b &= b - 1u;
                w.cand[o++] = lo + (t << 5) + k;
            }
        }
        __syncthreads();
        for (int e = tid; e < total; e += kThreads) {
            const int d = w.raw[e] - lo;
            const unsigned b = w.bits[d >> 5], bit = 1u << (d & 31);
            w.raw[e] = (b & bit) ? (int)w.bits[kWords + (d >> 5)] + __popc(b & (bit - 1u)) : -1;
        }
        __syncthreads();
        return count;
    }
    sort_raw(w, total);
    for (int base = 0; base < total; base += kThreads) {
        const int e = base + tid;
        bool keep = e < total && (e == 0 || w.raw[e - 1] != w.raw[e]);
        if (keep) {
            const int p = lower_bound_i(w.J, n, w.raw[e]);
            keep = !(p < n && w.J[p] == w.raw[e]);
        }
        int chunk;
        const int o = count + block_scan(w, (int)keep, &chunk);
        if (count + chunk > kU) return -1;
        if (keep) w.cand[o] = w.raw[e];
        count += chunk;
    }
    __syncthreads();
    return count;
}

constexpr int kMoves = -2;

/* Augment_Sparsity (src/Spai_Sub.imp:1010-1116): the new |J|, -1 when there is
 * no candidate, or kMoves when a list outgrows the working set or a tie of
 * scores straddles the cut (the generic kernel orders those). */
__device__ __forceinline__ int augment(const BuildArgs& a, WideLds& w, int col, int m, int n, double rn, int* st,
                                       double* wk, int* near)
{
    const int tid = threadIdx.x;
    const bool col_in = row_position(w, col) >= 0;
    const int nl = col_in ? m : m + 1;
    /* the row patterns of L = I u {col} */
    int len = 0, e0 = 0, total;
    if (tid < nl) {
        const int l = tid < m ? w.rows[tid] : col;
        e0 = a.rp_ptr[l];
        len = a.rp_ptr[l + 1] - e0;
    }
    const int off = block_scan(w, len, &total);
    if (total > kRaw) return kMoves;
    int lo = 0x7fffffff, hi = -1;
    constexpr int kD = 12;  // loads in flight
    for (int e = 0; e < len; e += kD) {
        int v[kD];
#pragma unroll
        for (int q = 0; q < kD; ++q) v[q] = e + q < len ? a.rp_ind[e0 + e + q] : 0;
#pragma unroll
        for (int q = 0; q < kD; ++q)
            if (e + q < len) {
                w.raw[off + e + q] = v[q];
                lo = min(lo, v[q]);
                hi = max(hi, v[q]);
            }
    }
    lo = block_min(w, lo);
    hi = block_max(w, hi);
    bool slots = false;
    const int c = candidates(w, total, lo, hi, n, &slots);
    if (c < 0) return kMoves;
    if (wk && tid == 0) wk[3] += 8.0 * nl + 4.0 * total;
    if (c == 0) return -1;
    /* rho_j = sqrt(||r||^2 - (r^T a_j)^2 / ||a_j||^2), numerator over I only,
     * in the order of the rows.  The raw list holds exactly the entries of I's
     * rows: they are put into one bucket per candidate (a tenth of what the
     * candidates' columns hold), each bucket summed by one thread in order of
     * the rows; a candidate with a long bucket is summed over its column. */
    const double rn2 = __dmul_rn(rn, rn);
    constexpr int kBucket = 16;
    const bool by_rows = slots && a.rp_val != nullptr;
    int rp0 = -1;  // position of this thread's row of I
    if (tid < m) {
        rp0 = w.rank[w.slot_of[tid]];
        w.rowbase[rp0] = e0 - off;
    }
    if (by_rows) {
        for (int t = tid; t <= c; t += kThreads) w.first[t] = 0;
        __syncthreads();
        if (tid < m)  // the entries of col, when not in I, are candidates only
            for (int e = off; e < off + len; ++e)
                if (w.raw[e] >= 0) atomicAdd(&w.first[w.raw[e] + 1], 1);
        __syncthreads();
        /* counts to first places: the counts sit one slot up, so that placing
         * an entry leaves first[t] at the end of bucket t */
        int cnt[kPer], mine = 0;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int t = tid * kPer + k;
            cnt[k] = t < c ? w.first[t + 1] : 0;
            mine += cnt[k];
        }
        int all;
        int o = block_scan(w, mine, &all);
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int t = tid * kPer + k;
            if (t < c) w.first[t + 1] = o;
            o += cnt[k];
        }
        __syncthreads();
        if (tid < m)
            for (int e = off; e < off + len; ++e)
                if (w.raw[e] >= 0) w.bucket[atomicAdd(&w.first[w.raw[e] + 1], 1)] = rp0 << 13 | e;
        __syncthreads();
    }
    double rho[kPer], part = 0.0;
    int entries = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        rho[k] = INFINITY;
        if (tid + k * kThreads < c) {
            const int t = tid + k * kThreads;
            const int j = w.cand[t];
            const double ajn = a.ajn[j];
            int b0 = 0, b1 = kBucket + 1;
            if (by_rows) {
                b0 = w.first[t];  // bucket t ends at first[t + 1], where bucket t + 1 starts
                b1 = w.first[t + 1];
            }
            double num = 0.0;
            if (b1 - b0 <= kBucket) {
                int last = -1;
                for (int b = b0; b < b1; ++b) {
                    int next = 0x7fffffff;  // the first entry after the last one taken
                    for (int u = b0; u < b1; ++u) {
                        const int x = w.bucket[u];
                        next = x > last ? min(next, x) : next;
                    }
                    last = next;
                    const int row = next >> 13;
                    num = __dadd_rn(num, __dmul_rn(w.r[row], a.rp_val[w.rowbase[row] + (next & (kRaw - 1))]));
                }
            } else {
                const int e1 = a.A.colptr[j + 1];
                for (int e = a.A.colptr[j]; e < e1; ++e) {
                    const int pos = row_position(w, a.A.rowind[e]);
                    if (pos >= 0) num = __dadd_rn(num, __dmul_rn(w.r[pos], a.A.val[e]));
                }
            }
            const double n2 = __dmul_rn(num, num);
            rho[k] = sqrt(__dsub_rn(rn2, __ddiv_rn(n2, __dmul_rn(ajn, ajn))));
            part += rho[k];
            if (wk) entries += a.A.colptr[j + 1] - a.A.colptr[j];
        }
    }
    if (wk) {
        entries = block_sum(w, entries);
        if (tid == 0) {
            wk[4] += 16.0 * c + 12.0 * entries;
            wk[5] += (double)c;
        }
    }
    /* the mean threshold: the sequential sum where the order of the sum could
     * decide a score (any order is within 4 (c + 1) u of it), as in the
     * one-wave kernels */
    auto live = [&](int k) { return tid + k * kThreads < c; };
    double mean = block_sum(w, part);
    if (a.use_mean) mean = __ddiv_rn(mean, (double)c);
    bool exact = wk != nullptr || !isfinite(mean);
    if (!exact) {
        const double band = 4.0 * (double)(c + 1) * 0x1p-53 * mean;
        bool inside = false;
#pragma unroll
        for (int k = 0; k < kPer; ++k) inside |= live(k) && fabs(rho[k] - mean) <= band;
        exact = block_any(w, inside);
    }
    if (exact) {
        /* the buckets are read out (the block's sum came after them) */
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            if (live(k)) w.score[tid + k * kThreads] = rho[k];
        __syncthreads();
        double seq = 0.0;  // formed by every thread
        for (int t = 0; t < c; ++t) seq = __dadd_rn(seq, w.score[t]);
        mean = a.use_mean ? __ddiv_rn(seq, (double)c) : seq;
    }
    if (isnan(mean)) {
        *st |= COL_NAN_RHO;
        return n;
    }
    if (near) {
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < kPer; ++k) cnt += live(k) && fabs(rho[k] - mean) <= kNearMargin * fabs(mean);
        near[0] += block_sum(w, cnt);
    }
    int q = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) q += live(k) && rho[k] <= mean;
    q = block_sum(w, q);
    const int sneed = a.maxnew < q ? a.maxnew : q;
    if (sneed <= 0) return n;
    if (n + sneed > kJ) return kMoves;
    /* the sneed-th smallest score and the number of scores below it */
    double prev = -1.0, vstar = 0.0;
    int below = 0, ties = 0;
    for (int it = 0; it < c; ++it) {
        double v = INFINITY;
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            if (live(k) && rho[k] > prev) v = fmin(v, rho[k]);
        v = block_min(w, v);
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < kPer; ++k) cnt += live(k) && rho[k] == v;
        cnt = block_sum(w, cnt);
        if (below + cnt >= sneed || cnt == 0) {
            vstar = v;
            ties = cnt;
            break;
        }
        below += cnt;
        prev = v;
    }
    const int take_ties = sneed - below;
    if (near && q > sneed) {
        double vnext = INFINITY;
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            if (live(k) && rho[k] > vstar) vnext = fmin(vnext, rho[k]);
        vnext = block_min(w, vnext);
        near[1] += (take_ties != ties || vnext - vstar <= kNearMargin * vstar) ? 1 : 0;
    }
    if (take_ties != ties) return kMoves;
    /* J <- sort(J u selected) */
    if (tid == 0) w.count = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k)
        if (live(k) && rho[k] <= vstar) w.sel[atomicAdd(&w.count, 1)] = w.cand[tid + k * kThreads];
    __syncthreads();
    if (tid == 0)
        for (int t = 0; t < sneed; ++t) {
            int i = n + t - 1;
            for (; i >= 0 && w.J[i] > w.sel[t]; --i) w.J[i + 1] = w.J[i];
            w.J[i + 1] = w.sel[t];
        }
    __syncthreads();
    return n + sneed;
}

/* One column from its start pattern or the state an earlier launch left;
 * true when it moves on (its state is then left for the next launch, as the
 * one-wave kernels leave theirs: the step in nsolve, J and the counters).
 * fresh: not routed, no launch has seen the column. */
__device__ __forceinline__ bool wide_column(const BuildArgs& a, WideLds& w, int col, bool fresh)
{
    const int tid = threadIdx.x;
    double* const wk = a.work ? w.wsum : nullptr;
    int st = 0, step0 = -1, n;
    int near[3] = {0, 0, 0};
    const size_t o = a.direct ? (size_t)a.p_ptr[col] : (size_t)col * a.cap;
    const int mark = fresh ? 0 : a.nsolve[col];
    const int* jsrc;
    if (mark < 0) {
        step0 = -mark - 2;
        n = a.m_len[col];
        st = a.status[col];
        jsrc = a.m_idx + o;
    } else {
        const int p0 = a.p_ptr[col];
        n = a.p_ptr[col + 1] - p0;
        jsrc = a.p_ind + p0;
    }
    if (n > kJ) {
        __syncthreads();  // every thread has read the mark
        if (mark < 0 && !a.save_state && tid == 0) a.nsolve[col] = 0;
        return true;
    }
    if (wk) {
        if (tid < kNumWork) wk[tid] = mark < 0 ? a.work[(size_t)col * kNumWork + tid] : 0.0;
        if (mark < 0) {
            const double pk = a.res[col];
            near[2] = (int)(pk * 0x1p-40);
            near[1] = (int)((pk - near[2] * 0x1p40) * 0x1p-20);
            near[0] = (int)(pk - near[2] * 0x1p40 - near[1] * 0x1p20);
        }
    }
    if (tid < n) w.J[tid] = jsrc[tid];
    __syncthreads();
    int solves = step0 + 1, moved = -2, st0 = st, near0[3], m = 0, st1 = 0;
    bool whole = true;  // A(I,J) is in LDS
    double rn = 1.0e50, wk0 = 0.0;
    for (int step = step0; step < a.ns; ++step) {
        st0 = st;
        for (int q = 0; q < 3; ++q) near0[q] = near[q];
        if (wk && tid < kNumWork) wk0 = wk[tid];
        m = index_set(a, w, n);
        if (m < 0) {
            moved = step;
            break;
        }
        st |= gather(a, w, m, n, col);
        st1 = solve(w, m, n);
        st |= st1;
        ++solves;
        if (wk && tid == 0) {
            const double dm = (double)m, dn = (double)n, kk = dm < dn ? dm : dn;
            wk[0] = __dadd_rn(wk[0], __dsub_rn(2.0 * dm * dn * dn, (2.0 / 3.0) * kk * kk * kk));
            wk[1] = __dadd_rn(wk[1], (4.0 * dm * dn - 2.0 * dn * dn) + dn * dn + 2.0 * dm * dn);
            wk[2] += 8.0 * dn + 12.0 * (double)w.segoff[n];
            wk[6] += dm;
            wk[7] += dn;
        }
        rn = residual(w, m, n);
        if (wk) near[2] += fabs(rn - a.epsilon) <= kNearMargin * a.epsilon;
        if (rn <= a.epsilon || step == a.ns - 1) break;
        const int nn = augment(a, w, col, m, n, rn, &st, wk, wk ? near : nullptr);
        if (nn == kMoves) {
            moved = step;
            break;
        }
        if (nn < 0) {
            whole = false;  // the augmentation's lists took its place
            break;
        }
        n = nn;
    }
    __syncthreads();
    if (moved > -2) {
        if (!a.save_state) {
            if (tid == 0) a.nsolve[col] = 0;
            return true;
        }
        if (tid < n) a.m_idx[o + tid] = w.J[tid];
        if (wk && tid < kNumWork) a.work[(size_t)col * kNumWork + tid] = wk0;
        if (tid == 0) {
            a.m_len[col] = n;
            a.status[col] = st0;
            a.nsolve[col] = -(moved + 2);
            if (wk) a.res[col] = near0[0] + near0[1] * 0x1p20 + near0[2] * 0x1p40;
        }
        return true;
    }
    if (a.refine && solves > 0 && !(st1 & (COL_UNDERDET | COL_SINGULAR))) {
        if (!whole) gather(a, w, m, n, col);
        refine(w, m, n);
    }
    if (tid < n) {
        a.m_idx[o + tid] = w.J[tid];
        a.m_val[o + tid] = w.x[tid];
    }
    if (tid == 0) {
        a.m_len[col] = n;
        a.res[col] = rn;
        a.nsolve[col] = solves;
        a.status[col] = st | a.status_or;
    }
    if (wk && tid < kNumWork) a.work[(size_t)col * kNumWork + tid] = wk[tid];
    if (a.lwork) {
        if (tid < kNumWork) atomicAdd(&a.lwork[tid], w.wsum[tid]);
        if (tid == 0) {
            atomicAdd(&a.lwork[kNumWork], 1.0);
            atomicAdd(&a.lwork[kNumWork + 4], (double)n);
            for (int q = 0; q < 3; ++q)
                if (near[q]) atomicAdd(&a.lwork[kNumWork + 1 + q], (double)near[q]);
        }
    }
    return false;
}

/* Columns queue[0..*nqueue) (all columns 0..a.nqueue without a queue), one
 * per workgroup: the first by block index, further ones by the atomic. */
__global__ __launch_bounds__(kThreads, 2) void wide_column_kernel(BuildArgs a, const int* queue, const int* nqueue,
                                                                 int* head)
{
    extern __shared__ __align__(16) char smem[];
    WideLds& w = *reinterpret_cast<WideLds*>(smem);
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.stamp = wall_clock64();
    const int nq = queue ? *nqueue : a.nqueue;
    for (int q = blockIdx.x; q < nq;) {
        const int col = queue ? queue[q] : q;
        if (wide_column(a, w, col, !queue) && threadIdx.x == 0) a.overflow[atomicAdd(a.n_overflow, 1)] = col;
        __syncthreads();
        if (threadIdx.x == 0) w.count = (int)gridDim.x + atomicAdd(head, 1);
        __syncthreads();
        q = w.count;
        __syncthreads();
    }
}

}  // namespace

size_t wide_lds_bytes() { return sizeof(WideLds); }

void launch_wide(const BuildArgs& a, const int* queue, const int* nqueue, int* head, int blocks, hipStream_t stream)
{
    hipLaunchKernelGGL(wide_column_kernel, dim3(blocks), dim3(kThreads), sizeof(WideLds), stream, a, queue, nqueue,
                       head);
}

}  // namespace mspai
