/*
 * Column kernels for a given pattern: static builds (no augmentation) and
 * the adjoint, one column of M per group of lanes.
 *
 * Lane (g, h) of a group, h = lane % 4, holds rows 4k + h (k < KR) of the
 * columns g + CG s (s < S) of [A(I,J) | b] in registers, the right-hand side
 * being column |J|.  A column's dot product in the 64-lane order is then an
 * in-lane tree over k (the butterfly's steps 32, 16, 8, 4 pair rows whose k
 * differ in one bit) followed by two quad permutes (steps 2 and 1), so KR
 * terms cost KR multiplies and KR - 1 adds with no lane move, and one quad
 * reduction serves CG columns per wave slot.  The Householder vector goes
 * through LDS once per reflector: its column's four lanes write it, every
 * lane reads the KR rows it owns (used for S columns each).  Every rounding
 * is that of the fixed order: the same bits as the column kernels of the
 * adaptive builds and their oracle.
 *
 * What bounds it: VALU issue in FP64 (at 4 cycles per wave instruction).
 * Rows and slots that a step no longer touches are skipped at compile time
 * (rows) or by a uniform branch (slots).  On P(A^2) of the 3D
 * variable-coefficient operator (|J| <= 25, |I| <= 63, n = 2,097,152) an FP64
 * build takes 27.5 ms, 5.0 K VALU instructions per column; with four rows per
 * lane and four lane moves per dot product (the adaptive builds' register QR)
 * it took 64.1 ms and 13.3 K.  Values and gradient of the 48^3 operator: 8.2
 * -> 3.4 ms; of MSPAI probing on the 64^3 Laplacian at precision 1: 3.3 ->
 * 1.3 ms.
 *
 * Precision 1 runs the same FP64 factorization and one step of refinement:
 * FP32 is no faster here (non-packed FP32 issues at the FP64 rate) and its
 * factor needs two or three steps; the refined solution is as close to the
 * exact one as those gave (1.6e-16 against 1.7e-16 on the 101^3 operator, 16.6
 * against 38.4 ms), which the unrefined FP64 QR is not (3.7e-16).
 *
 * The index sets need no sorted I: the distinct rows of J's columns go into
 * a hash table in LDS, a row's position is the number of smaller rows.
 */
#include <algorithm>

#include "device_common.h"
#include "spai_host.h"

namespace mspai {

namespace {

/* double of the lane xor 1 or xor 2 (quad permutes) */
template <int S>
__device__ __forceinline__ double quad_sum_step(double p)
{
    return p + Group<16>::xor_lane<S>(p);
}

/* Working set of one column in LDS. */
template <int CG, int S, int KR>
struct __align__(16) StaticLds {
    static constexpr int G = 4 * CG;       // lanes
    static constexpr int kRows = 4 * KR;   // |I|
    static constexpr int kCols = S * CG;   // |J| and the right-hand side
    static constexpr int kSlots = 2 * kRows;
    /* doubles per lane of a staged column slot: KR rows and 16 bytes that
     * spread the lanes' b128 accesses over the banks */
    static constexpr int kChunk = KR + 2;
    double stage[G * kChunk];  // a slot of A(I,J); after the QR: R (packed columns), then Q^T b
    double v[4 * kChunk];      // the reflector's column
    double r[kRows];           // b, then the residual (adjoint: b - C m)
    double x[kCols];           // the solution (adjoint: lambda)
    double y[kCols];           // adjoint: m
    int rows[kRows];           // distinct rows in order of arrival
    int key[kSlots];
    unsigned char rank[kSlots];   // position in sorted I of the row in a slot
    unsigned char slot_of[kRows];
    int count;
    static_assert(G * kChunk >= kCols * (kCols - 1) / 2 + kCols, "R and Q^T b fit the staging region");
};

template <int SLOTS>
__device__ __forceinline__ unsigned row_slot(int row)
{
    return ((unsigned)row * 0x9e3779b1u) >> (33 - __builtin_ctz(2 * SLOTS));
}

/* More distinct rows have arrived than the working set holds: the column
 * moves on, and no further row needs a place (every insertion into a full
 * table walks all of it: patterns on three columns of 10,000 entries took 15
 * and 27 ms in the first two kinds, 0.03 ms now). */
template <class W>
__device__ __forceinline__ bool rows_full(const W& w)
{
    return __hip_atomic_load(&w.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > W::kRows;
}

/* Slot of `row`, added when new (-1: the table is full, which takes more
 * rows than the working set holds). */
template <class W>
__device__ __forceinline__ int hash_insert(W& w, int row)
{
    unsigned slot = row_slot<W::kSlots>(row);
    for (int probe = 0; probe < W::kSlots; ++probe) {
        const int old = atomicCAS(&w.key[slot], -1, row);
        if (old == -1) {
            const int k = atomicAdd(&w.count, 1);
            if (k < W::kRows) {
                w.rows[k] = row;
                w.slot_of[k] = (unsigned char)slot;
            }
            return (int)slot;
        }
        if (old == row) return (int)slot;
        slot = (slot + 1) & (W::kSlots - 1);
    }
    return -1;
}

/* Position of `row` in I, or -1. */
template <class W>
__device__ __forceinline__ int hash_position(const W& w, int row)
{
    unsigned slot = row_slot<W::kSlots>(row);
    for (int probe = 0; probe < W::kSlots; ++probe) {
        const int k = w.key[slot];
        if (k == row) return w.rank[slot];
        if (k == -1) return -1;
        slot = (slot + 1) & (W::kSlots - 1);
    }
    return -1;
}

/* Value of group lane K in every lane of its group (K uniform in the wave). */
template <int G>
__device__ __forceinline__ double group_value(double v, int K)
{
    if constexpr (G >= 32) return Group<G>::lane_value(v, K);
    return __shfl(v, K, G);
}

constexpr int kMovesOn = 1;

/* b <- (R^T R)^-1 b, b_l on group lane l, R in packed columns; the pivots'
 * reciprocals are formed once (refinement only: its corrections need no last
 * bit). */
template <int G, int kCols>
__device__ __forceinline__ double refine_solve(const double* R, double b, int l, int n)
{
    const double dinv = l < n ? 1.0 / R[l * (l + 1) / 2 + l] : 0.0;
    for (int K = 0; K < kCols - 1; ++K) {
        if (!__any(K < n)) break;
        const double yk = group_value<G>(b * dinv, K);
        if (l == K) b = yk;
        else if (l > K && l < n) b = __fma_rn(-yk, R[l * (l + 1) / 2 + K], b);
    }
    for (int K = kCols - 2; K >= 0; --K) {
        if (!__any(K < n)) continue;
        const double dk = group_value<G>(b * dinv, K);
        if (K < n) {
            if (l == K) b = dk;
            else if (l < K) b = __fma_rn(-dk, R[K * (K + 1) / 2 + l], b);
        }
    }
    return b;
}

/* Whether a refinement step d of x (one entry per lane) is small enough to
 * be trusted, max|d| <= 1e-10 max|x| over the group: a factor too ill
 * conditioned for the normal equations gives a larger one (or NaN), and the
 * column keeps its QR solution. */
template <int G>
__device__ __forceinline__ bool step_trusted(double d, double x)
{
    double xm = fabs(x);
#pragma unroll
    for (int off = G / 2; off >= 1; off /= 2) xm = fmax(xm, __shfl_xor(xm, off, kWave));
    const unsigned long long out = __ballot(!(fabs(d) <= 1e-10 * xm));
    const int base = (int)threadIdx.x & ~(G - 1);
    return ((out >> base) & ((1ull << G) - 1ull)) == 0ull;
}

/* Work counters of a column (as the adaptive kernels count one solve; a
 * refinement step is not counted) and its share of the launch's totals. */
template <int S, int G>
__device__ __forceinline__ void count_column(const BuildArgs& a, int col, int m, int n, double rn, bool moves, int l,
                                             int h, const int (&cnt)[S], bool near)
{
    static_assert(G >= kNumWork, "a lane per counter");
    int entries = 0;
#pragma unroll
    for (int s = 0; s < S; ++s) entries += h == 0 ? cnt[s] : 0;
#pragma unroll
    for (int off = G / 2; off >= 1; off /= 2) entries += __shfl_xor(entries, off, kWave);
    if (col < 0 || moves || l >= kNumWork) return;
    const double dm = (double)m, dn = (double)n, kk = dm < dn ? dm : dn;
    const double v = l == 0   ? __dsub_rn(2.0 * dm * dn * dn, (2.0 / 3.0) * kk * kk * kk)
                     : l == 1 ? (4.0 * dm * dn - 2.0 * dn * dn) + dn * dn + 2.0 * dm * dn
                     : l == 2 ? 8.0 * dn + 12.0 * (double)entries
                     : l == 6 ? dm
                     : l == 7 ? dn
                              : 0.0;
    a.work[(size_t)col * kNumWork + l] = v;
    atomicAdd(&a.lwork[l], v);
    if (l == 0) {
        atomicAdd(&a.lwork[kNumWork], 1.0);
        if (near && fabs(rn - a.epsilon) <= kNearMargin * a.epsilon) atomicAdd(&a.lwork[kNumWork + 3], 1.0);
        atomicAdd(&a.lwork[kNumWork + 4], dn);
    }
}

/* One column per group: the build (kBack false) or the adjoint of a column
 * of M.  kRefine (builds and adjoints at precision 1) adds one step of
 * refinement by the normal equations with the FP64 factor: x += (R^T R)^-1
 * A^T (b - A x), lambda += (R^T R)^-1 (g - A^T A lambda).  col < 0: none.
 * Whole-wave call; returns kMovesOn (uniform in the group) when the column
 * does not fit. */
template <int CG, int S, int KR, bool kBack, bool kRefine, bool kCount>
__device__ __forceinline__ int static_column(const BuildArgs& a, StaticLds<CG, S, KR>& w, int col)
{
    using W = StaticLds<CG, S, KR>;
    constexpr int G = W::G, CH = W::kChunk, kRows = W::kRows;
    constexpr int kOwn = kRows / G;  // rows per lane in row order: l, l + G, ...
    const int l = threadIdx.x & (G - 1), h = l & 3, g = l >> 2;
    int p0 = 0, n = 0;
    bool moves = false;
    if (col >= 0) {
        p0 = a.p_ptr[col];
        n = a.p_ptr[col + 1] - p0;
        if (n > W::kCols - 1) moves = true;
    }
    if (moves) n = 0;
    int start[S], cnt[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int j = g + CG * s;
        start[s] = cnt[s] = 0;
        if (j < n) {
            const int J = a.p_ind[p0 + j];
            start[s] = a.A.colptr[J];
            cnt[s] = a.A.colptr[J + 1] - start[s];
        }
    }
    for (int t = l; t < W::kSlots; t += G) w.key[t] = -1;
    for (int t = l; t < kRows; t += G) {
        w.rows[t] = 0x7fffffff;
        w.r[t] = 0.0;
    }
    if (l == 0) w.count = 0;
    __syncthreads();
    /* Get_I_Set: the four lanes of a column take its entries in turn; the
     * loads of the first two entries of every slot are in flight together */
    int rw[S][2];
    unsigned ps[S];  // hash slots of those two entries, one byte each
    bool full = false;  // seen where so many entries may have gone in: past the
                        // first eight of a column, and past a table's worth
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int q = 0; q < 2; ++q) rw[s][q] = h + 4 * q < cnt[s] ? a.A.rowind[start[s] + h + 4 * q] : -1;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        ps[s] = 0u;
        if (2 * G * s >= W::kSlots) full = full || rows_full(w);
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (rw[s][q] >= 0 && !full) ps[s] |= (unsigned)(hash_insert(w, rw[s][q]) & 0xff) << (8 * q);
        for (int e = h + 8; e < cnt[s] && !full; e += 4) {
            hash_insert(w, a.A.rowind[start[s] + e]);
            full = rows_full(w);
        }
    }
    __syncthreads();
    int m = w.count;
    if (m > kRows) {
        moves = true;
        n = m = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) cnt[s] = 0;
    }
    {
        int mine[kOwn], rk[kOwn];
#pragma unroll
        for (int q = 0; q < kOwn; ++q) {
            mine[q] = w.rows[l + G * q];
            rk[q] = 0;
        }
        for (int u = 0; u < m; u += 4) {
            const int4 o = *reinterpret_cast<const int4*>(&w.rows[u]);
#pragma unroll
            for (int q = 0; q < kOwn; ++q)
                rk[q] += (o.x < mine[q]) + (o.y < mine[q]) + (o.z < mine[q]) + (o.w < mine[q]);
        }
#pragma unroll
        for (int q = 0; q < kOwn; ++q)
            if (l + G * q < m) w.rank[w.slot_of[l + G * q]] = (unsigned char)rk[q];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < S; ++s) {
        /* positions instead of slots */
        if (rw[s][0] >= 0 && m > 0) {
            unsigned p = w.rank[ps[s] & 0xff];
            if (rw[s][1] >= 0) p |= (unsigned)w.rank[(ps[s] >> 8) & 0xff] << 8;
            ps[s] = p;
        }
    }
    /* the right-hand side (Create_ek_Hat / Create_bk_Hat) in w.r */
    bool hit = false;
    if (col >= 0 && m > 0) {
        if (!a.B.colptr) {
            const int pos = hash_position(w, col);
            hit = pos >= 0;
            if (hit && l == 0) w.r[pos] = 1.0;
        } else {
            const int e1 = a.B.colptr[col + 1];
            for (int e = a.B.colptr[col]; e < e1; ++e) {
                const int pos = hash_position(w, a.B.rowind[e]);
                if (pos >= 0) {
                    hit = true;
                    if (l == 0) w.r[pos] = a.B.val[e];
                }
            }
        }
    }
    if constexpr (kBack) {
        for (int j = l; j < n; j += G) {
            w.y[j] = a.m_in[p0 + j];
            w.x[j] = a.gM[p0 + j];
        }
    }
    __syncthreads();
    double res[kOwn];  // rows l, l + G, ..: b_i, less the columns seen so far
    if constexpr (kBack) {
#pragma unroll
        for (int q = 0; q < kOwn; ++q) res[q] = w.r[l + G * q];
    }

    /* the columns of slot s, staged in LDS: chunk (column, h) holds rows 4k + h */
    double* const mine = w.stage + l * CH;
    auto stage_slot = [&](int s, int st, int ct, unsigned pk) {
        double2* const z = reinterpret_cast<double2*>(mine);
#pragma unroll
        for (int k = 0; k < KR / 2; ++k) z[k] = make_double2(0.0, 0.0);
        __syncthreads();
        double* const cols = w.stage + 4 * g * CH;
        double v[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) v[q] = h + 4 * q < ct ? a.A.val[st + h + 4 * q] : 0.0;
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (h + 4 * q < ct) {
                const int pos = (int)((pk >> (8 * q)) & 0xff);
                cols[(pos & 3) * CH + (pos >> 2)] = v[q];
            }
        for (int e = h + 8; e < ct; e += 4) {
            const int pos = hash_position(w, a.A.rowind[st + e]);
            cols[(pos & 3) * CH + (pos >> 2)] = a.A.val[st + e];
        }
        __syncthreads();
    };
    double x[S][KR];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (__any(CG * s < n || (!kBack && CG * s == n))) {
            stage_slot(s, start[s], cnt[s], ps[s]);
#pragma unroll
            for (int k = 0; k < KR; k += 2) {
                const double2 d = *reinterpret_cast<const double2*>(mine + k);
                x[s][k] = d.x;
                x[s][k + 1] = d.y;
            }
            if (!kBack && g + CG * s == n) {
#pragma unroll
                for (int k = 0; k < KR; ++k) x[s][k] = w.r[4 * k + h];
            }
            if constexpr (kBack) {
#pragma unroll
                for (int c = 0; c < CG; ++c) {
                    const int j = CG * s + c;
                    const double yj = j < n ? w.y[j] : 0.0;
#pragma unroll
                    for (int q = 0; q < kOwn; ++q) {
                        const int r = l + G * q;
                        res[q] = __fma_rn(-yj, w.stage[(4 * c + (r & 3)) * CH + (r >> 2)], res[q]);
                    }
                }
            }
            __syncthreads();
        } else {
#pragma unroll
            for (int k = 0; k < KR; ++k) x[s][k] = 0.0;
        }
    }

    /* Householder QR; column |J| takes Q^T b (build only) */
    const int kk = m < n ? m : n;
    const int last = kBack ? n - 1 : n;  // last live column
    bool singular = false;
#pragma unroll
    for (int sp = 0; sp < S; ++sp) {
        constexpr int kBound = CG < 4 ? 1 : CG / 4;  // values of k that hold rows i of this slot
        const int k0 = sp * CG / 4;                  // the first of them (constant once unrolled)
        if (!__any(sp * CG < kk)) break;
#pragma unroll 1
        for (int c = 0; c < CG; ++c) {
            const int i = sp * CG + c;
            if (!__any(i < kk)) break;
            if (i < kk && g == c) {
#pragma unroll
                for (int k = 0; k < KR; k += 2)
                    if (k + 1 >= k0)
                        *reinterpret_cast<double2*>(w.v + h * CH + k) = make_double2(x[sp][k], x[sp][k + 1]);
            }
            __syncthreads();
            double v[KR], p[KR];
#pragma unroll
            for (int k = 0; k < KR; k += 2)
                if (k + 1 >= k0) {
                    const double2 d = *reinterpret_cast<const double2*>(w.v + h * CH + k);
                    v[k] = d.x;
                    v[k + 1] = d.y;
                }
            const double alpha = w.v[(i & 3) * CH + (i >> 2)];
            __syncthreads();
            /* the 64-lane order over a row set that starts at k0: terms of
             * rows below 4 k0 are +0, which leaves a sum unchanged */
            auto tree = [&](double (&t)[KR]) {
#pragma unroll
                for (int half = KR / 2; half >= 1; half /= 2)
#pragma unroll
                    for (int k = 0; k < KR / 2; ++k)
                        if (k < half) t[k] = (half == KR / 2 && k < k0) ? t[k + half] : t[k] + t[k + half];
                double s0 = quad_sum_step<2>(t[0]);
                return quad_sum_step<1>(s0);
            };
#pragma unroll
            for (int k = 0; k < KR; ++k)
                if (k >= k0) {
                    p[k] = __fma_rn(v[k], v[k], 0.0);
                    if (k < k0 + kBound) p[k] = 4 * k + h > i ? p[k] : 0.0;
                }
            const double xn2 = tree(p);
            const bool taken = i < kk && i + 1 < m && xn2 != 0.0;
            double rii = alpha;
            if (taken) {
                const double nrm = sqrt(__fma_rn(alpha, alpha, xn2));
                const double beta = -copysign(nrm, alpha);
                const double tau = (beta - alpha) / beta;
                const double scal = 1.0 / (alpha - beta);
                const double mt = -tau;
                rii = beta;
#pragma unroll
                for (int k = 0; k < KR; ++k)
                    if (k >= k0) {
                        v[k] = v[k] * scal;
                        if (k < k0 + kBound) v[k] = 4 * k + h == i ? 1.0 : v[k];
                    }
#pragma unroll
                for (int s = sp; s < S; ++s) {
                    if (__any(CG * s <= last)) {
#pragma unroll
                        for (int k = 0; k < KR; ++k)
                            if (k >= k0) {
                                p[k] = __fma_rn(v[k], x[s][k], 0.0);
                                if (k < k0 + kBound) p[k] = 4 * k + h >= i ? p[k] : 0.0;
                            }
                        const double t = mt * tree(p);
#pragma unroll
                        for (int k = 0; k < KR; ++k)
                            if (k >= k0) {
                                const double u = __fma_rn(v[k], t, x[s][k]);
                                /* columns up to i take junk below their R: never read */
                                x[s][k] = (k >= k0 + kBound || 4 * k + h >= i) ? u : x[s][k];
                            }
                    }
                }
#pragma unroll
                for (int k = 0; k < KR; ++k)
                    if (k >= k0 && k < k0 + kBound) x[sp][k] = (g == c && 4 * k + h == i) ? beta : x[sp][k];
            }
            singular |= i < kk && rii == 0.0;
        }
    }

    /* R (columns packed) and Q^T b to LDS, then one row per lane */
    double* const R = w.stage;
    double* const qb = w.stage + W::kCols * (W::kCols - 1) / 2;
    auto store_factor = [&]() {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int j = g + CG * s;
#pragma unroll
            for (int k = 0; k < KR; ++k) {
                const int r = 4 * k + h;
                if (4 * k < CG * (s + 1) && r <= j && j < n) R[j * (j + 1) / 2 + r] = x[s][k];
                if (4 * k < W::kCols && !kBack && j == n && r < n) qb[r] = x[s][k];
            }
        }
        __syncthreads();
    };
    /* out_j = sum over column j's entries of C_ij w_i, w over I in w.v */
    auto transposed = [&](double* out) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int j = g + CG * s;
            double t = 0.0;
            for (int e = h; e < cnt[s]; e += 4) {
                const int pos = e < 8 ? (int)((ps[s] >> (2 * (e & ~3))) & 0xff)
                                      : hash_position(w, a.A.rowind[start[s] + e]);
                t = __fma_rn(a.A.val[start[s] + e], w.v[pos], t);
            }
            t = quad_sum_step<1>(quad_sum_step<2>(t));
            if (h == 0 && j < n) out[j] = t;
        }
        __syncthreads();
    };
    static_assert(4 * CH >= kRows, "w.v holds a vector over I");
    /* the staged columns times the vector y over J, added to acc (rows l, l + G, ..) */
    auto times = [&](const double* y, double (&acc)[kOwn]) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (__any(CG * s < n)) {
                stage_slot(s, start[s], cnt[s], ps[s]);
#pragma unroll
                for (int c = 0; c < CG; ++c) {
                    const int j = CG * s + c;
                    const double yj = j < n ? y[j] : 0.0;
#pragma unroll
                    for (int q = 0; q < kOwn; ++q) {
                        const int r = l + G * q;
                        const double t = __fma_rn(yj, w.stage[(4 * c + (r & 3)) * CH + (r >> 2)], acc[q]);
                        acc[q] = yj != 0.0 ? t : acc[q];
                    }
                }
                __syncthreads();
            }
        }
    };
    store_factor();
    int st = hit ? 0 : COL_K_NOT_IN_I;
    bool solve = n > 0;
    if (m < n) {
        st |= COL_UNDERDET;
        solve = false;
    } else if (singular) {
        st |= COL_SINGULAR;
        solve = false;
    }
    if constexpr (kBack) {
        /* degenerate columns have no gradient */
        double b = l < n ? w.x[l] : 0.0;
        const int top = W::kCols - 1;
        for (int K = 0; K < top; ++K) {  // R^T y = dL/dm
            if (!__any(K < n)) break;
            const double yk = group_value<G>(b, K) / (K < n ? R[K * (K + 1) / 2 + K] : 1.0);
            if (l == K) b = yk;
            else if (l > K && l < n) b = __fma_rn(-yk, R[l * (l + 1) / 2 + K], b);
        }
        for (int K = top - 1; K >= 0; --K) {  // R lambda = y
            if (!__any(K < n)) continue;
            const double dk = group_value<G>(b, K) / (K < n ? R[K * (K + 1) / 2 + K] : 1.0);
            if (K < n) {
                if (l == K) b = dk;
                else if (l < K) b = __fma_rn(-dk, R[K * (K + 1) / 2 + l], b);
            }
        }
        if (!solve) {
#pragma unroll
            for (int s = 0; s < S; ++s) cnt[s] = 0;
        }
        __syncthreads();
        if (l < n) w.x[l] = b;
        __syncthreads();
        /* s = C lambda beside r = b - C m */
        double sv[kOwn];
#pragma unroll
        for (int q = 0; q < kOwn; ++q) sv[q] = 0.0;
        times(w.x, sv);
        if constexpr (kRefine) {
#pragma unroll
            for (int q = 0; q < kOwn; ++q) w.v[l + G * q] = sv[q];
            __syncthreads();
            transposed(w.x);
            store_factor();
            const double gm = l < n ? a.gM[p0 + l] - w.x[l] : 0.0;
            const double d = refine_solve<G, W::kCols>(R, gm, l, n);
            if (step_trusted<G>(d, b)) b += d;
            __syncthreads();
            if (l < n) w.x[l] = b;
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kOwn; ++q) sv[q] = 0.0;
            times(w.x, sv);
        }
        double* const sb = w.stage;
#pragma unroll
        for (int q = 0; q < kOwn; ++q) {
            w.r[l + G * q] = res[q];
            sb[l + G * q] = sv[q];
        }
        __syncthreads();
        /* dL/dC_ij += r_i lambda_j - s_i m_j over the stored entries of J */
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int j = g + CG * s;
            const double lam = j < n ? w.x[j] : 0.0, mj = j < n ? w.y[j] : 0.0;
            for (int e = h; e < cnt[s]; e += 4) {
                const int pos = e < 8 ? (int)((ps[s] >> (2 * (e & ~3))) & 0xff)
                                      : hash_position(w, a.A.rowind[start[s] + e]);
                atomicAdd(&a.gC[start[s] + e], __fma_rn(w.r[pos], lam, -sb[pos] * mj));
            }
        }
        if (a.gB && a.B.colptr && solve) {
            const int e0 = a.B.colptr[col], e1 = a.B.colptr[col + 1];
            for (int e = e0 + l; e < e1; e += G) {
                const int pos = hash_position(w, a.B.rowind[e]);
                a.gB[e] = pos >= 0 ? sb[pos] : 0.0;
            }
        }
        __syncthreads();
        return moves ? kMovesOn : 0;
    }
    double b = (l < n && !(st & COL_UNDERDET)) ? qb[l] : 0.0;
    /* dtrsm order; a singular R leaves Q^T b */
    for (int K = W::kCols - 2; K >= 0; --K) {
        if (!__any(solve && K < n)) continue;
        double xk = group_value<G>(b, K);
        if (solve && K < n && xk != 0.0) {
            xk = xk / R[K * (K + 1) / 2 + K];
            if (l == K) b = xk;
            else if (l < K) b = __fma_rn(-xk, R[K * (K + 1) / 2 + l], b);
        }
    }
    __syncthreads();
    if (l < n) w.x[l] = b;
    /* r = A(I,J) x - b in dgemv's column order, then the sequential sum of
     * squares */
#pragma unroll
    for (int q = 0; q < kOwn; ++q) res[q] = -w.r[l + G * q];
    __syncthreads();
    times(w.x, res);
    if constexpr (kRefine) {
#pragma unroll
        for (int q = 0; q < kOwn; ++q) w.v[l + G * q] = res[q];
        __syncthreads();
        transposed(w.y);
        store_factor();
        const double d = refine_solve<G, W::kCols>(R, l < n ? w.y[l] : 0.0, l, n);
        if (step_trusted<G>(d, b) && solve) b -= d;
        __syncthreads();
        if (l < n) w.x[l] = b;
#pragma unroll
        for (int q = 0; q < kOwn; ++q) res[q] = -w.r[l + G * q];
        __syncthreads();
        times(w.x, res);
    }
    if (l < n) a.m_val[p0 + l] = b;
#pragma unroll
    for (int q = 0; q < kOwn; ++q) w.r[l + G * q] = l + G * q < m ? __dmul_rn(res[q], res[q]) : 0.0;
    __syncthreads();
    double sum = 0.0;
    for (int r = 0; r < m; r += 2) {
        const double2 d = *reinterpret_cast<const double2*>(w.r + r);
        sum = __dadd_rn(__dadd_rn(sum, d.x), d.y);  // a row past |I| adds +0
    }
    __syncthreads();
    if (l == 0 && col >= 0) {
        if (moves) {
            a.nsolve[col] = 0;  // the next launch starts the column afresh
        } else {
            a.m_len[col] = n;
            a.res[col] = sqrt(sum);
            a.nsolve[col] = 1;
            a.status[col] = st;
        }
    }
    if constexpr (kCount) count_column<S, G>(a, col, m, n, sqrt(sum), moves, l, h, cnt, !kRefine);
    return moves ? kMovesOn : 0;
}

/* Columns queue[0..*nqueue), or 0..nall without a queue; the groups of block
 * b take neighbouring columns, blocks stride over the queue.  Columns that do
 * not fit go to a.overflow. */
template <int CG, int S, int KR, bool kBack, bool kRefine, bool kCount, int kWaves>
__global__ __launch_bounds__(64, kWaves) void static_column_kernel(BuildArgs a, const int* queue, const int* nqueue,
                                                                  int nall)
{
    using W = StaticLds<CG, S, KR>;
    constexpr int NG = kWave / W::G;
    __shared__ W work[NG];
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.stamp = wall_clock64();
    const int nq = queue ? *nqueue : nall;
    const int g = (int)threadIdx.x / W::G;
    /* workgroups go round-robin to the 8 XCDs: XCD x takes the x-th
     * contiguous eighth, so that neighbouring columns meet in one L2 */
    constexpr unsigned kXcd = 8;
    const unsigned per = gridDim.x / kXcd, b = blockIdx.x;
    const unsigned slot = b < per * kXcd ? (b % kXcd) * per + b / kXcd : b;
    for (long long q0 = (long long)slot * NG; q0 < nq; q0 += (long long)gridDim.x * NG) {
        const long long q = q0 + g;
        const int col = q < nq ? (queue ? queue[q] : (int)q) : -1;
        const int outcome = static_column<CG, S, KR, kBack, kRefine, kCount>(a, work[g], col);
        if (outcome == kMovesOn && (threadIdx.x & (W::G - 1)) == 0) a.overflow[atomicAdd(a.n_overflow, 1)] = col;
        __syncthreads();
    }
}

/* M of a static build has the start pattern: its column pointers, indices
 * and number of entries. */
__global__ __launch_bounds__(256) void copy_pattern_kernel(int ncols, int nnz, const int* p_ptr, const int* p_ind,
                                                          int* colptr, int* rowind, int* count, unsigned long long* stamp)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();
    const int stride = (int)(gridDim.x * blockDim.x);
    const int t0 = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    for (int t = t0; t <= ncols; t += stride) colptr[t] = p_ptr[t];
    for (long long t = t0; t < nnz; t += stride) rowind[t] = p_ind[t];
    if (t0 == 0) *count = nnz;
}

template <int CG, int S, int KR, int kWaves>
void launch_kind(const BuildArgs& a, bool back, bool refine, const int* queue, const int* nqueue, int nall,
                 int num_cu, hipStream_t stream)
{
    constexpr int NG = kWave / (4 * CG);
    const long long all = ((long long)nall + NG - 1) / NG;
    /* a queue's length is known on the device only: a grid that fills the
     * chip strides over it */
    const unsigned grid = (unsigned)(queue ? std::min<long long>(all, (long long)num_cu * 4 * kWaves) : all);
    if (grid == 0) return;
    /* builds with work counters have kernels of their own: with the counting
     * in the others the 101^3 operator's build at precision 1, which keeps no
     * counters, took 16.67 instead of 16.55 ms */
    const auto k = back     ? (refine ? &static_column_kernel<CG, S, KR, true, true, false, kWaves>
                                      : &static_column_kernel<CG, S, KR, true, false, false, kWaves>)
                   : a.work ? (refine ? &static_column_kernel<CG, S, KR, false, true, true, kWaves>
                                      : &static_column_kernel<CG, S, KR, false, false, true, kWaves>)
                            : (refine ? &static_column_kernel<CG, S, KR, false, true, false, kWaves>
                                      : &static_column_kernel<CG, S, KR, false, false, false, kWaves>);
    hipLaunchKernelGGL(k, dim3(grid), dim3(kWave), 0, stream, a, queue, nqueue, nall);
}

}  // namespace

void launch_static_columns(int kind, const BuildArgs& a, bool back, bool refine, const int* queue, const int* nqueue,
                           int nall, int num_cu, hipStream_t stream)
{
    switch (kind) {
    case 0: launch_kind<2, 4, 8, 3>(a, back, refine, queue, nqueue, nall, num_cu, stream); break;
    case 1: launch_kind<4, 4, 16, 2>(a, back, refine, queue, nqueue, nall, num_cu, stream); break;
    default: launch_kind<8, 4, 16, 2>(a, back, refine, queue, nqueue, nall, num_cu, stream); break;
    }
}

void launch_copy_pattern(int ncols, int nnz, const int* p_ptr, const int* p_ind, int* colptr, int* rowind,
                         int* count, unsigned long long* stamp, hipStream_t stream)
{
    const long long t = std::max<long long>(nnz, ncols + 1);
    const unsigned grid = (unsigned)std::min<long long>((t + 255) / 256, 4096);
    hipLaunchKernelGGL(copy_pattern_kernel, dim3(grid), dim3(256), 0, stream, ncols, nnz, p_ptr, p_ind, colptr,
                       rowind, count, stamp);
}

}  // namespace mspai
