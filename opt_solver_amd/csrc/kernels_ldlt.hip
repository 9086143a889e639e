// HIP kernels of the indefinite (LDL^T, threshold 1x1 / 2x2 pivoting)
// numeric phase. Compiled with -ffp-contract=off: every multiply and add
// below rounds separately, as the reference's ldlt_kernel.cpp
// (solver/CMakeLists.txt:632-642), so the unblocked front kernel
// reproduces ldlt_factor_front's pivot sequence and values bit for bit.
#include "smfgpu_ldlt.hpp"
#include "mfma_tile.hpp"

#include <cfloat>
#include <type_traits>

namespace smfgpu {

constexpr int kLT = 256;            // threads per workgroup
constexpr double kWeakPivotRatio = 1e-6;  // ldlt_kernel.hpp:100

// ---------------------------------------------------------------------------
// Workgroup reductions (exact: max and first argmax).
template <int NT>
struct RedScratchT {
    double v[NT];
    int i[NT];
};
using RedScratch = RedScratchT<kLT>;

// (max, first index of the max) over the thread's candidates, reduced
// across the workgroup: ties keep the smaller index, as a sequential scan
// with a strict '>' does.
// One wavefront (every lane active): within each row of 16 lanes the
// partners of four DPP steps (quad swaps of 1 and 2, half-row mirror, row
// mirror) bring every lane the row's result; the four rows' results are
// then read from lanes 0, 16, 32, 48. Max and first-argmax do not depend on
// the order of combination.
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = dpp_i<CTRL>(static_cast<int>(b));
    const int hi = dpp_i<CTRL>(static_cast<int>(b >> 32));
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}
__device__ __forceinline__ double lane_d(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), l);
    const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), l);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;
__device__ __forceinline__ bool better_first(double b, int ib, double a, int ia) {
    return b > a || (b == a && ib >= 0 && (ia < 0 || ib < ia));
}
template <int CTRL>
__device__ __forceinline__ void maxfirst_step(double &v, int &idx) {
    const double b = dpp_d<CTRL>(v);
    const int ib = dpp_i<CTRL>(idx);
    if (better_first(b, ib, v, idx)) {
        v = b;
        idx = ib;
    }
}
template <int CTRL>
__device__ __forceinline__ void max_step(double &v) {
    const double b = dpp_d<CTRL>(v);
    if (b > v) v = b;
}

// What __syncthreads gives a workgroup, for NT threads; one wavefront's LDS
// accesses happen in its own order.
template <int NT>
__device__ __forceinline__ void wg_sync() {
    if constexpr (NT == 64) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

template <int NT>
__device__ __forceinline__ void red_maxfirst(RedScratchT<NT> &rs, double v, int idx, double &outv, int &outi) {
    if constexpr (NT == 64) {
        maxfirst_step<kDppXor1>(v, idx);
        maxfirst_step<kDppXor2>(v, idx);
        maxfirst_step<kDppHalfMirror>(v, idx);
        maxfirst_step<kDppMirror>(v, idx);
        double bv = lane_d(v, 0);
        int bi = __builtin_amdgcn_readlane(idx, 0);
        for (int r = 16; r < 64; r += 16) {
            const double c = lane_d(v, r);
            const int ic = __builtin_amdgcn_readlane(idx, r);
            if (better_first(c, ic, bv, bi)) {
                bv = c;
                bi = ic;
            }
        }
        outv = bv;
        outi = bi;
        return;
    }
    const int tid = threadIdx.x;
    rs.v[tid] = v;
    rs.i[tid] = idx;
    __syncthreads();
    for (int w = NT / 2; w > 0; w >>= 1) {
        if (tid < w) {
            const double a = rs.v[tid], b = rs.v[tid + w];
            const int ia = rs.i[tid], ib = rs.i[tid + w];
            if (b > a || (b == a && ib >= 0 && (ia < 0 || ib < ia))) {
                rs.v[tid] = b;
                rs.i[tid] = ib;
            }
        }
        __syncthreads();
    }
    outv = rs.v[0];
    outi = rs.i[0];
    __syncthreads();
}

template <int NT>
__device__ __forceinline__ double red_max(RedScratchT<NT> &rs, double v) {
    if constexpr (NT == 64) {
        max_step<kDppXor1>(v);
        max_step<kDppXor2>(v);
        max_step<kDppHalfMirror>(v);
        max_step<kDppMirror>(v);
        double m = lane_d(v, 0);
        for (int r = 16; r < 64; r += 16) {
            const double c = lane_d(v, r);
            if (c > m) m = c;
        }
        return m;
    }
    const int tid = threadIdx.x;
    rs.v[tid] = v;
    __syncthreads();
    for (int w = NT / 2; w > 0; w >>= 1) {
        if (tid < w && rs.v[tid + w] > rs.v[tid]) rs.v[tid] = rs.v[tid + w];
        __syncthreads();
    }
    const double out = rs.v[0];
    __syncthreads();
    return out;
}

// View of one front: element (i, j), i >= j, at F[j * ld + i].
struct FV {
    double *F;
    int ld, f;
    __device__ __forceinline__ double &at(int i, int j) const { return F[static_cast<int64_t>(j) * ld + i]; }
    __device__ __forceinline__ double sym(int i, int j) const { return i >= j ? at(i, j) : at(j, i); }
};

// Column sweeps keep kU independent loads in flight per thread: the loads
// of a group are issued from clamped (in-range) addresses before any use,
// and only the in-range elements are used or stored. Updates read and
// write different columns, which the compiler cannot tell apart, so
// without the explicit grouping every element waits out a full memory
// latency.
constexpr int kU = 4;
// A one-wavefront workgroup's front has at most 48 rows, in LDS: one load
// covers a sweep.
template <int ST>
constexpr int sweep_loads = ST == 64 ? 1 : kU;

// f(i, v) for v = ld(i), i = lo, lo + ST, ... < hi, in increasing i per
// thread
template <int ST, class Ld, class Fn>
__device__ __forceinline__ void sweep(int lo, int hi, Ld &&ld, Fn &&fn) {
    constexpr int U = sweep_loads<ST>;
    for (int i0 = lo; i0 < hi; i0 += U * ST) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = ld(min(i0 + u * ST, hi - 1));
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u * ST < hi) fn(i0 + u * ST, v[u]);
    }
}

// c[i] = c[i] - a[i] * l (multiply, then subtract), i = lo, lo + st, ... < hi;
// c and a are different columns
__device__ __forceinline__ void col_axpy(double *c, const double *a, double l, int lo, int hi, int st) {
    for (int i0 = lo; i0 < hi; i0 += kU * st) {
        double cv[kU], av[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int i = min(i0 + u * st, hi - 1);
            cv[u] = c[i];
            av[u] = a[i];
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (i0 + u * st < hi) c[i0 + u * st] = __dsub_rn(cv[u], __dmul_rn(av[u], l));
    }
}

// c[i] = c[i] - (a0[i] * l0 + a1[i] * l1)
__device__ __forceinline__ void col_axpy2(double *c, const double *a0, const double *a1, double l0, double l1, int lo,
                                          int hi, int st) {
    for (int i0 = lo; i0 < hi; i0 += kU * st) {
        double cv[kU], x0[kU], x1[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int i = min(i0 + u * st, hi - 1);
            cv[u] = c[i];
            x0[u] = a0[i];
            x1[u] = a1[i];
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (i0 + u * st < hi)
                c[i0 + u * st] = __dsub_rn(cv[u], __dadd_rn(__dmul_rn(x0[u], l0), __dmul_rn(x1[u], l1)));
    }
}

// dst[i] = src[i] (different arrays)
__device__ __forceinline__ void col_copy(double *dst, const double *src, int lo, int hi, int st) {
    for (int i0 = lo; i0 < hi; i0 += kU * st) {
        double v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) v[u] = src[min(i0 + u * st, hi - 1)];
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (i0 + u * st < hi) dst[i0 + u * st] = v[u];
    }
}

// exchange a[i] and b[i] (different columns, or a row and a column that
// share no element over the range)
template <int ST, class PA, class PB>
__device__ __forceinline__ void swap_range(PA &&pa, PB &&pb, int lo, int hi) {
    constexpr int U = sweep_loads<ST>;
    for (int i0 = lo; i0 < hi; i0 += U * ST) {
        double x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = min(i0 + u * ST, hi - 1);
            x[u] = *pa(i);
            y[u] = *pb(i);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u * ST < hi) {
                *pa(i0 + u * ST) = y[u];
                *pb(i0 + u * ST) = x[u];
            }
    }
}

// min_abs: the front's in-order static pivot (static_pivot_in_order, 0 off);
// S: static pivoting of the launch (fronts pick theirs with
// front_static_value)
struct Prm {
    double u, eff_small, small_pivot;
    double min_abs;
    StaticPrm S;
};

// The pivoting parameters of front F: its static value (0: none) and, in
// the in-order mode, min_abs (ldlt_kernel.cpp:1131-1132 and
// multifrontal_serial.cpp:624-629: a fallback front keeps in-order only when
// static pivoting is on overall).
__device__ __forceinline__ double front_prm(const Prm &prm, const FrontLd &F, Prm &fp) {
    fp = prm;
    const double sp = front_static_value(prm.S, F.root, F.nd, F.psym);
    fp.min_abs = (prm.S.sp > 0.0 && (prm.S.flags & kStaticInOrder)) ? sp : 0.0;
    return sp;
}

// static_counts_as_zero (ldlt_kernel.cpp:325-328): a fallback front keeps a
// pivot raised from an exact zero as a zero (static_zero_stays_zero set).
__device__ __forceinline__ bool static_as_zero(int raised, const Prm &prm, const FrontLd &F) {
    if (raised == 0) return false;
    const bool fallback = prm.S.fallback > 0.0 && (F.root != 0 || F.nd > F.psym);
    const bool stays = fallback || (prm.S.flags & kStaticZeroStaysZero);
    return (prm.S.flags & kStaticAsZero) || (raised == 2 && stays);
}

// two_by_two_ok (ldlt_kernel.cpp:97-122): the block of columns c0 and c1,
// off0 and off1 their largest entries outside it.
__device__ __forceinline__ bool two_by_two_ok(const FV &A, int c0, int c1, double off0, double off1, const Prm &prm,
                                              double &growth) {
    growth = 0.0;
    const double d00 = A.at(c0, c0);
    const double d10 = A.sym(c1, c0);
    const double d11 = A.at(c1, c1);
    double s2 = fabs(d00);
    if (s2 < fabs(d10)) s2 = fabs(d10);
    if (s2 < fabs(d11)) s2 = fabs(d11);
    if (!(s2 >= prm.eff_small && isfinite(s2))) return false;
    const double a = d00 / s2, b = d10 / s2, c = d11 / s2;
    const double det_s = __dsub_rn(__dmul_rn(a, c), __dmul_rn(b, b));
    if (!(fabs(det_s) > prm.small_pivot)) return false;
    if (off0 > 0.0 || off1 > 0.0) {
        const double bound0 = __dadd_rn(__dmul_rn(fabs(c), off0), __dmul_rn(fabs(b), off1)) / s2;
        const double bound1 = __dadd_rn(__dmul_rn(fabs(b), off0), __dmul_rn(fabs(a), off1)) / s2;
        const double bm = bound0 > bound1 ? bound0 : bound1;
        if (prm.u * bm > fabs(det_s)) return false;
        growth = bm / fabs(det_s);
    }
    return true;
}

// select_pivot (ldlt_kernel.cpp:127-275) with workgroup reductions. Every
// thread returns the same choice.
template <int NT>
__device__ void select_pivot_wg(const FV &A, int k, int ne, int limit, const Prm &prm, RedScratchT<NT> &rs, int &kind,
                                int &pa, int &pb) {
    const int tid = threadIdx.x;
    const int f = A.f;
    kind = 0;
    pa = pb = -1;
    if (prm.min_abs > 0.0) {
        // in order, no search: column k or nothing (then the static path)
        const double d0 = A.at(k, k);
        if (isfinite(d0) && fabs(d0) >= prm.min_abs) {
            kind = 1;
            pa = k;
        }
        return;
    }
    if (k < limit) {
        const double a0 = fabs(A.at(k, k));
        if (a0 >= prm.eff_small) {
            const double *ck = &A.at(0, k);
            double m = 0.0;
            sweep<NT>(k + 1 + tid, f, [&](int i) { return ck[i]; }, [&](int, double v) { m = fmax(m, fabs(v)); });
            const double colmax = red_max(rs, m);
            if (!(prm.u * colmax > a0) && !(a0 < kWeakPivotRatio * colmax)) {
                kind = 1;
                pa = k;
                return;
            }
        }
    }
    for (int cand = k; cand < limit; ++cand) {
        const double a_cand = fabs(A.at(cand, cand));
        // largest entry over the eligible rows [k, ne) other than cand (first
        // index on ties), then the largest of the rest
        // One sweep of the column: each thread keeps its largest entry (first
        // index), the largest of its other entries, and the maximum over
        // rows [ne, f). The thread holding the overall first argmax then
        // contributes its second value to m2, every other thread its first.
        const int ext0 = max(ne, cand + 1);
        double bv = -1.0, b2 = 0.0, mel = 0.0;
        int bi = -1;
        const auto top2 = [&](int i, double x) {
            const double v = fabs(x);
            if (v > bv) {
                b2 = fmax(b2, bv);
                bv = v;
                bi = i;
            } else {
                b2 = fmax(b2, v);
            }
        };
        // rows [k, cand) of the candidate's row, then rows (cand, ne) and
        // [ext0, f) of its column: each thread still meets its indices in
        // increasing order
        const double *cc = &A.at(0, cand);
        const int k1 = k + tid;
        sweep<NT>(k1, min(cand, ne), [&](int i) { return A.at(cand, i); }, top2);
        {
            // first index of this thread's sequence past cand
            const int c1 = cand + 1 + (((k1 - (cand + 1)) % NT) + NT) % NT;
            sweep<NT>(c1, ne, [&](int i) { return cc[i]; }, top2);
            const int e1 = ext0 + (((k1 - ext0) % NT) + NT) % NT;
            sweep<NT>(e1, f, [&](int i) { return cc[i]; }, [&](int, double x) { mel = fmax(mel, fabs(x)); });
        }
        double m1;
        int r_best;
        red_maxfirst(rs, bv, bi, m1, r_best);
        if (!(m1 > 0.0)) {
            m1 = 0.0;
            r_best = -1;
        }
        const double m2 = red_max(rs, (r_best >= 0 && bi == r_best) ? b2 : fmax(bv, 0.0));
        const double m_ext = red_max(rs, mel);
        bool weak = false;
        double weak_growth = 0.0;
        if (a_cand >= prm.eff_small && !(prm.u * m1 > a_cand)) {
            if (!(prm.u * m_ext > a_cand)) {
                const double colmax = fmax(m1, m_ext);
                if (!(a_cand < kWeakPivotRatio * colmax)) {
                    kind = 1;
                    pa = cand;
                    return;
                }
                weak = true;
                weak_growth = colmax / a_cand;
            }
        }
        if (r_best < k || r_best >= limit || m1 <= 0.0) {
            if (weak) {
                kind = 1;
                pa = cand;
                return;
            }
            continue;
        }
        // partner column: max excluding r_best, and excluding cand too
        double o2 = 0.0, o1 = 0.0;
        const auto part = [&](int i, double x) {
            const double v = fabs(x);
            o2 = fmax(o2, v);
            if (i != cand) o1 = fmax(o1, v);
        };
        const double *cr = &A.at(0, r_best);
        sweep<NT>(k + tid, r_best, [&](int i) { return A.at(r_best, i); }, part);
        sweep<NT>(r_best + 1 + (((k + tid - (r_best + 1)) % NT) + NT) % NT, f, [&](int i) { return cr[i]; }, part);
        const double om2 = red_max(rs, o2);
        const double off1 = red_max(rs, o1);
        double growth2;
        const bool ok2 = k + 1 < limit && two_by_two_ok(A, cand, r_best, fmax(m2, m_ext), off1, prm, growth2);
        if (ok2 && (!weak || growth2 < weak_growth)) {
            kind = 2;
            pa = cand;
            pb = r_best;
            return;
        }
        if (weak) {
            kind = 1;
            pa = cand;
            return;
        }
        const double a_r = fabs(A.at(r_best, r_best));
        if (a_r >= prm.eff_small && (om2 == 0.0 || a_r >= prm.u * om2)) {
            kind = 1;
            pa = r_best;
            return;
        }
    }
}

// Partner rows of a stalled first-pass panel (ldlt_kernel.cpp:1052-1075):
// for each failed column pos of [k, pl) in order, the first row of [pl, ne)
// holding the column's largest entry, kept when that entry exceeds the
// column's largest entry inside the panel and the row is no earlier
// column's partner. (column, partner) row ids go to order (at most 64
// pairs, nb / 2 when smaller); returns the number of ids written. Every
// thread returns the same count.
template <int NT>
__device__ int partner_pairs_wg(const FV &A, int k, int pl, int ne, int nb, const int32_t *rows, int32_t *order,
                                RedScratchT<NT> &rs) {
    const int tid = threadIdx.x;
    int np = 0;
    const int max_pairs = min(nb / 2, 64);
    for (int pos = k; pos < pl && np / 2 < max_pairs; ++pos) {
        double inl = 0.0;
        for (int i = k + tid; i < pl; i += NT)
            if (i != pos) inl = fmax(inl, fabs(A.sym(i, pos)));
        const double in_max = red_max(rs, inl);
        double bv = 0.0;
        int bi = -1;
        const double *cp = &A.at(0, pos);
        sweep<NT>(pl + tid, ne, [&](int i) { return cp[i]; }, [&](int i, double x) {
            const double v = fabs(x);
            if (v > bv) {
                bv = v;
                bi = i;
            }
        });
        double out_max;
        int r;
        red_maxfirst(rs, bv, bi, out_max, r);
        if (r < 0 || !(out_max > in_max)) continue;
        bool taken = false;
        for (int t = 1; t < np; t += 2) taken = taken || order[t] == rows[r];
        if (taken) continue;
        if (tid == 0) {
            order[np] = rows[pos];
            order[np + 1] = rows[r];
        }
        np += 2;
        __syncthreads();
    }
    return np;
}

// Lanes per column when the workgroup sweeps the lower part of several
// columns of up to `len` rows: log2 of a power of two covering len (at most
// the workgroup), so NT >> lg columns are in flight at a time.
template <int NT = kLT>
__device__ __forceinline__ int lg_rows(int len) {
    int lg = 0;
    while ((1 << lg) < len && (1 << lg) < NT) ++lg;
    return lg;
}

// sym_swap (ldlt_kernel.cpp:333-345): positions p < q. Columns [c_lo, p)
// swap rows p and q (c_lo = 0: all earlier columns).
template <int NT = kLT>
__device__ void sym_swap_wg(const FV &A, int p, int q, int32_t *rows, double *W, int wld, int w_cols, int c_lo) {
    if (p == q) return;
    if (p > q) {
        const int t = p;
        p = q;
        q = t;
    }
    const int tid = threadIdx.x;
    const int f = A.f;
    wg_sync<NT>();
    if (tid == 0) {
        const double t = A.at(p, p);
        A.at(p, p) = A.at(q, q);
        A.at(q, q) = t;
        const int32_t tr = rows[p];
        rows[p] = rows[q];
        rows[q] = tr;
    }
    // rows p and q of the columns before p; column p and row q between
    // them; columns p and q below q
    swap_range<NT>([&](int m) { return &A.at(p, m); }, [&](int m) { return &A.at(q, m); }, c_lo + tid, p);
    swap_range<NT>([&](int m) { return &A.at(m, p); }, [&](int m) { return &A.at(q, m); }, p + 1 + tid, q);
    swap_range<NT>([&](int m) { return &A.at(m, p); }, [&](int m) { return &A.at(m, q); }, q + 1 + tid, f);
    swap_range<NT>([&](int idx) { return &W[static_cast<int64_t>(idx) * wld + p]; },
               [&](int idx) { return &W[static_cast<int64_t>(idx) * wld + q]; }, tid, w_cols);
    wg_sync<NT>();
}

// Brings the rows order[0..np) to positions k, k + 1, ... in turn with
// sym_swap (ldlt_kernel.cpp:1076-1082): each row id is unique and, when
// its turn comes, lies in [k + t, ne); the workgroup finds it in one
// parallel sweep instead of a sequential scan.
template <int NT>
__device__ void place_rows_wg(const FV &A, int k, int ne, int np, const int32_t *order, int32_t *rows,
                              RedScratchT<NT> &rs) {
    const int tid = threadIdx.x;
    for (int t = 0; t < np; ++t) {
        const int32_t want = order[t];
        int mine = -1;
        for (int i0 = k + t + tid; i0 < ne; i0 += kU * NT) {
            int32_t v[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) v[u] = rows[min(i0 + u * NT, ne - 1)];
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (i0 + u * NT < ne && v[u] == want) mine = i0 + u * NT;
        }
        double hit;
        int q;
        red_maxfirst(rs, mine >= 0 ? 1.0 : 0.0, mine, hit, q);
        if (q >= k + t) sym_swap_wg<NT>(A, k + t, q, rows, nullptr, 0, 0, 0);
    }
}

// eliminate_1x1 (ldlt_kernel.cpp:350-432): columns (k, ucol_end) get the
// rank-1 update c_j[i] -= c_k[i] * (c_k[j] / d) (multiply, then subtract),
// the unscaled column is saved in W column w_col, then c_k is scaled.
template <int NT = kLT>
__device__ void elim1_wg(const FV &A, int k, int ucol_end, double *W, int wld, int w_col) {
    const int tid = threadIdx.x;
    const int f = A.f;
    const double inv_d = 1.0 / A.at(k, k);
    double *ck = &A.at(0, k);
    if (W) col_copy(W + static_cast<int64_t>(w_col) * wld, ck, k + 1 + tid, f, NT);
    if (ucol_end > k + 1) {
        const int lg = lg_rows<NT>(f - (k + 1));
        for (int jb = k + 1; jb < ucol_end; jb += NT >> lg) {
            const int j = jb + (tid >> lg);
            if (j >= ucol_end) continue;
            const double lj = __dmul_rn(A.at(j, k), inv_d);
            if (lj == 0.0) continue;
            col_axpy(&A.at(0, j), ck, lj, j + (tid & ((1 << lg) - 1)), f, 1 << lg);
        }
    }
    __syncthreads();
    for (int i = k + 1 + tid; i < f; i += NT) ck[i] = __dmul_rn(ck[i], inv_d);
    __syncthreads();
}

// eliminate_2x2 (ldlt_kernel.cpp:436-545)
template <int NT = kLT>
__device__ void elim2_wg(const FV &A, int k, int ucol_end, double *W, int wld, int w_col) {
    const int tid = threadIdx.x;
    const int f = A.f;
    const double d00 = A.at(k, k), d10 = A.at(k + 1, k), d11 = A.at(k + 1, k + 1);
    double s = fabs(d00);
    if (s < fabs(d10)) s = fabs(d10);
    if (s < fabs(d11)) s = fabs(d11);
    const double a = d00 / s, b = d10 / s, c = d11 / s;
    const double inv = 1.0 / __dmul_rn(__dsub_rn(__dmul_rn(a, c), __dmul_rn(b, b)), s);
    const double i00 = __dmul_rn(c, inv), i10 = __dmul_rn(-b, inv), i11 = __dmul_rn(a, inv);
    double *ck0 = &A.at(0, k), *ck1 = &A.at(0, k + 1);
    if (W) {
        col_copy(W + static_cast<int64_t>(w_col) * wld, ck0, k + 2 + tid, f, NT);
        col_copy(W + static_cast<int64_t>(w_col + 1) * wld, ck1, k + 2 + tid, f, NT);
    }
    if (ucol_end > k + 2) {
        const int lg = lg_rows<NT>(f - (k + 2));
        for (int jb = k + 2; jb < ucol_end; jb += NT >> lg) {
            const int j = jb + (tid >> lg);
            if (j >= ucol_end) continue;
            const double a0 = A.at(j, k), a1 = A.at(j, k + 1);
            const double l0 = __dadd_rn(__dmul_rn(i00, a0), __dmul_rn(i10, a1));
            const double l1 = __dadd_rn(__dmul_rn(i10, a0), __dmul_rn(i11, a1));
            if (l0 == 0.0 && l1 == 0.0) continue;
            col_axpy2(&A.at(0, j), ck0, ck1, l0, l1, j + (tid & ((1 << lg) - 1)), f, 1 << lg);
        }
    }
    __syncthreads();
    for (int i = k + 2 + tid; i < f; i += NT) {
        const double a0 = A.at(i, k), a1 = A.at(i, k + 1);
        A.at(i, k) = __dadd_rn(__dmul_rn(i00, a0), __dmul_rn(i10, a1));
        A.at(i, k + 1) = __dadd_rn(__dmul_rn(i10, a0), __dmul_rn(i11, a1));
    }
    __syncthreads();
}

__device__ __forceinline__ void inertia_1x1(double d, double small, int *cnt) {
    if (!isfinite(d) || fabs(d) < small) ++cnt[2];
    else if (d > 0.0) ++cnt[0];
    else ++cnt[1];
}

// add_inertia_2x2 (dense_indef.cpp:52-88) with scaled_det_2x2 (pivoting.cpp:18-28)
__device__ void inertia_2x2(double d00, double d10, double d11, double small, int *cnt) {
    if (d10 == 0.0) {
        inertia_1x1(d00, small, cnt);
        inertia_1x1(d11, small, cnt);
        return;
    }
    double s = fabs(d00);
    if (s < fabs(d10)) s = fabs(d10);
    if (s < fabs(d11)) s = fabs(d11);
    double det_s = 0.0;
    if (isfinite(s) && s != 0.0) {
        const double a = d00 / s, b = d10 / s, c = d11 / s;
        det_s = __dsub_rn(__dmul_rn(a, c), __dmul_rn(b, b));
    }
    if (s == 0.0 || !isfinite(det_s)) {
        cnt[2] += 2;
        return;
    }
    if (det_s < -small) {
        ++cnt[0];
        ++cnt[1];
        return;
    }
    const double tr_s = __dadd_rn(d00 / s, d11 / s);
    if (fabs(det_s) <= small) {
        ++cnt[2];
        if (tr_s > small) ++cnt[0];
        else if (tr_s < -small) ++cnt[1];
        else ++cnt[2];
    } else {
        if (tr_s > 0.0) cnt[0] += 2;
        else if (tr_s < 0.0) cnt[1] += 2;
        else cnt[2] += 2;
    }
}

// force_static_pivot (ldlt_kernel.cpp:285-320): the column of [k, ne)
// whose diagonal is largest relative to its column (first on ties; column k
// in the in-order mode), |d| raised to sp keeping its sign when smaller.
// raised: 0 as it is, 1 from a nonzero |d|, 2 from an exact zero (below
// eff_small or not finite). Every thread returns the same column.
template <int NT>
__device__ int force_static_wg(const FV &A, int k, int ne, double sp, const Prm &prm, RedScratchT<NT> &rs,
                               int &raised, int &nstatic, double &growth) {
    const int tid = threadIdx.x;
    const int f = A.f;
    int best = k;
    double best_ratio = -1.0, best_colmax = 0.0;
    const int search_end = prm.min_abs > 0.0 ? k : ne;
    for (int cand = k; cand < search_end; ++cand) {
        double m = 0.0;
        const double *cc = &A.at(0, cand);
        sweep<NT>(k + tid, cand, [&](int i) { return A.at(cand, i); }, [&](int, double v) { m = fmax(m, fabs(v)); });
        sweep<NT>(cand + 1 + tid, f, [&](int i) { return cc[i]; }, [&](int, double v) { m = fmax(m, fabs(v)); });
        const double colmax = red_max(rs, m);
        const double a = fabs(A.at(cand, cand));
        const double ratio = colmax > 0.0 ? a / colmax : a;
        if (ratio > best_ratio) {
            best_ratio = ratio;
            best = cand;
            best_colmax = colmax;
        }
    }
    wg_sync<NT>();
    double dv = A.at(best, best);
    raised = 0;
    if (!(fabs(dv) >= sp)) {
        raised = (isfinite(dv) && fabs(dv) >= prm.eff_small) ? 1 : 2;
        dv = dv < 0.0 ? -sp : sp;
        ++nstatic;
        wg_sync<NT>();
        if (tid == 0) A.at(best, best) = dv;
    }
    if (best_colmax > 0.0 && fabs(dv) > 0.0) growth = fmax(growth, best_colmax / fabs(dv));
    wg_sync<NT>();
    return best;
}

// apply_pivot (ldlt_kernel.cpp:665-698). Thread 0 keeps the counters.
template <int NT = kLT>
__device__ void apply_pivot_wg(const FV &A, int kind, int pa, int pb, int &k, int32_t *rows, int8_t *tags, double *W,
                               int wld, int w_cols, int ucol_end, const Prm &prm, int *cnt, double &flops, int c_lo,
                               bool as_zero = false) {
    const int f = A.f;
    if (kind == 1) {
        sym_swap_wg<NT>(A, k, pa, rows, W, wld, w_cols, c_lo);
        if (threadIdx.x == 0) {
            if (as_zero) ++cnt[2];
            else inertia_1x1(A.at(k, k), prm.eff_small, cnt);
            tags[k] = 1;
        }
        elim1_wg<NT>(A, k, ucol_end, W, wld, w_cols);
        const double rem = static_cast<double>(f - (k + 1));
        flops += rem + rem * (rem + 1.0);
        k += 1;
        return;
    }
    int partner = pb;
    if (pa != k) {
        sym_swap_wg<NT>(A, k, pa, rows, W, wld, w_cols, c_lo);
        if (partner == k) partner = pa;
    }
    if (partner != k + 1) sym_swap_wg<NT>(A, k + 1, partner, rows, W, wld, w_cols, c_lo);
    if (threadIdx.x == 0) {
        inertia_2x2(A.at(k, k), A.at(k + 1, k), A.at(k + 1, k + 1), prm.small_pivot, cnt);
        tags[k] = 2;
        tags[k + 1] = -1;
    }
    wg_sync<NT>();
    elim2_wg<NT>(A, k, ucol_end, W, wld, w_cols);
    const double rem = static_cast<double>(f - (k + 2));
    flops += 6.0 * rem + 2.0 * rem * (rem + 1.0);
    k += 2;
}

// ---------------------------------------------------------------------------
// Unblocked fronts (f < blocked_min_front): the whole front in LDS, one
// workgroup, ldlt_factor_front's unblocked loop (ldlt_kernel.cpp:977-993).
constexpr int kSmallMax = 95;

__global__ __launch_bounds__(kLT) void k_ldlt_small(LdltDev d, const int32_t *__restrict__ flist, Prm prm) {
    __shared__ double Fs[kSmallMax * kSmallMax];
    __shared__ RedScratch rs;
    __shared__ int cnt[3];
    const int s = flist[blockIdx.x];
    FrontLd &Fd = d.fronts[s];
    const int f = Fd.f, ne = Fd.ne;
    double *G = d.arena + Fd.fofs;
    int32_t *rows = d.rows + Fd.rofs;
    int8_t *tags = d.tags + Fd.rofs;
    const int tid = threadIdx.x;
    for (int idx = tid; idx < f * f; idx += kLT) Fs[idx] = G[idx];
    if (tid < 3) cnt[tid] = 0;
    __syncthreads();
    FV A{Fs, f, f};
    int k = 0;
    double flops = 0.0;
    Prm fp;
    const double sp = front_prm(prm, Fd, fp);
    int nstatic = 0;
    double growth = 0.0;
    while (k < ne) {
        int kind, pa, pb;
        select_pivot_wg(A, k, ne, ne, fp, rs, kind, pa, pb);
        bool az = false;
        if (kind == 0) {
            if (!(sp > 0.0)) break;
            int raised;
            pa = force_static_wg(A, k, ne, sp, fp, rs, raised, nstatic, growth);
            kind = 1;
            az = static_as_zero(raised, fp, Fd);
        }
        apply_pivot_wg(A, kind, pa, pb, k, rows, tags, nullptr, 0, 0, f, fp, cnt, flops, 0, az);
    }
    __syncthreads();
    for (int idx = tid; idx < f * f; idx += kLT) G[idx] = Fs[idx];
    if (tid == 0) {
        Fd.p = k;
        Fd.npos = cnt[0];
        Fd.nneg = cnt[1];
        Fd.nzero = cnt[2];
        Fd.flops = flops;
        Fd.nstatic = nstatic;
        Fd.growth = growth;
        Fd.stalls = Fd.pulls = Fd.rotated = Fd.searches = 0;  // unblocked: no panels
    }
}

void launch_ldlt_small(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, double u, double eff_small,
                       double small_pivot, const StaticPrm &S) {
    if (nf <= 0) return;
    Prm prm{u, eff_small, small_pivot, 0.0, S};
    for (int64_t o = 0; o < nf; o += kMaxLaunchGroups)
        k_ldlt_small<<<dim3(static_cast<unsigned>(std::min<int64_t>(kMaxLaunchGroups, nf - o))), kLT, 0, st>>>(
            d, flist + o, prm);
}

// ---------------------------------------------------------------------------
// Blocked fronts (f >= blocked_min_front), one workgroup per front in global
// memory: ldlt_factor_front's blocked path (ldlt_kernel.cpp:1028-1139):
// first pass over nb-wide panels with partner pulls and rotation of failed
// columns, second pass with a full search on a stall, deferred panel
// updates, final Schur update. W (f x nb) in the front's workspace.
__device__ void deferred_update_wg(const FV &A, int p0, int p1, int c0, int e, const double *W, int wld) {
    const int jb = p1 - p0;
    const int m = e - c0;
    if (jb <= 0 || m <= 0) return;
    const int f = A.f;
    const int tid = threadIdx.x;
    const int lg = lg_rows(f - c0);
    const int st = 1 << lg;
    for (int cb = c0; cb < e; cb += kLT >> lg) {
        const int j = cb + (tid >> lg);
        if (j >= e) continue;
        double *cj = &A.at(0, j);
        // kU rows at a time, each summed over t in order
        for (int i0 = j + (tid & (st - 1)); i0 < f; i0 += kU * st) {
            double sacc[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) sacc[u] = 0.0;
            for (int t = 0; t < jb; ++t) {
                const double w = W[static_cast<int64_t>(t) * wld + j];
                const double *ct = &A.at(0, p0 + t);
                double v[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) v[u] = ct[min(i0 + u * st, f - 1)];
#pragma unroll
                for (int u = 0; u < kU; ++u) sacc[u] += v[u] * w;
            }
#pragma unroll
            for (int u = 0; u < kU; ++u)
                if (i0 + u * st < f) cj[i0 + u * st] -= sacc[u];
        }
    }
    __syncthreads();
}

__device__ void schur_update_wg(const FV &A, int p, int e, const int8_t *tags) {
    const int f = A.f;
    const int q = f - e;
    if (p <= 0 || q <= 0) return;
    const int64_t tot = static_cast<int64_t>(q) * q;
    for (int64_t idx = threadIdx.x; idx < tot; idx += kLT) {
        const int jj = static_cast<int>(idx / q), ii = static_cast<int>(idx % q);
        if (ii < jj) continue;
        const int i = e + ii, j = e + jj;
        double sacc = 0.0;
        for (int c = 0; c < p; ++c) {
            const int8_t tg = tags[c];
            double ld;
            if (tg == 1) ld = A.at(j, c) * A.at(c, c);
            else if (tg == 2) ld = A.at(j, c) * A.at(c, c) + A.at(j, c + 1) * A.at(c + 1, c);
            else if (tg == -1) ld = A.at(j, c - 1) * A.at(c, c - 1) + A.at(j, c) * A.at(c, c);
            else ld = 0.0;
            sacc += A.at(i, c) * ld;
        }
        A.at(i, j) -= sacc;
    }
    __syncthreads();
}

__global__ __launch_bounds__(kLT) void k_ldlt_blocked(LdltDev d, const int32_t *__restrict__ flist, Prm prm,
                                                     int32_t nb) {
    __shared__ RedScratch rs;
    __shared__ int cnt[3];
    __shared__ int32_t order[128];
    const int s = flist[blockIdx.x];
    FrontLd &Fd = d.fronts[s];
    const int f = Fd.f, ne = Fd.ne;
    int32_t *rows = d.rows + Fd.rofs;
    int8_t *tags = d.tags + Fd.rofs;
    double *W = d.work + Fd.wofs;
    const int wld = f;
    const int tid = threadIdx.x;
    FV A{d.arena + Fd.fofs, f, f};
    if (tid < 3) cnt[tid] = 0;
    __syncthreads();
    int k = 0;
    double flops = 0.0;
    Prm fp;
    const double sp = front_prm(prm, Fd, fp);
    const Prm &prm_f = fp;
    int nstatic = 0;
    double growth = 0.0;
    int n_stall = 0, n_pull = 0, n_rot = 0, n_search = 0;
    // the first pass with stall handling is for threshold pivoting only
    // (ldlt_kernel.cpp:1028); static fronts go straight to the second
    if (!(sp > 0.0) && !(fp.min_abs > 0.0)) {
        int live = ne, k_paired = -1;
        while (k < live) {
            const int ps = k;
            const int pl = min(live, ps + nb);
            bool stalled = false;
            while (k < pl) {
                int kind, pa, pb;
                select_pivot_wg(A, k, ne, pl, prm_f, rs, kind, pa, pb);
                if (kind == 0) {
                    stalled = true;
                    break;
                }
                apply_pivot_wg(A, kind, pa, pb, k, rows, tags, W, wld, k - ps, pl, prm_f, cnt, flops, 0);
            }
            deferred_update_wg(A, ps, k, pl, ne, W, wld);
            n_stall += stalled ? 1 : 0;
            if (stalled && k != k_paired) {
                // (failed column, partner) row-id pairs, distinct partners
                const int np = partner_pairs_wg(A, k, pl, ne, nb, rows, order, rs);
                if (np > 0) {
                    n_pull += np / 2;
                    place_rows_wg(A, k, ne, np, order, rows, rs);
                    live = max(live, k + np);
                    k_paired = k;
                    continue;
                }
            }
            if (stalled) {
                const int m = pl - k;
                const int mv = min(m, live - pl);
                for (int t = 0; t < mv; ++t) sym_swap_wg(A, k + t, live - mv + t, rows, nullptr, 0, 0, 0);
                live -= m;
                n_rot += m;
            }
        }
    }
    while (k < ne) {
        const int ps = k;
        const int pl = min(ne, ps + nb);
        bool stalled = false;
        while (k < pl) {
            int kind, pa, pb;
            select_pivot_wg(A, k, ne, pl, prm_f, rs, kind, pa, pb);
            if (kind == 0) {
                stalled = true;
                break;
            }
            apply_pivot_wg(A, kind, pa, pb, k, rows, tags, W, wld, k - ps, pl, prm_f, cnt, flops, 0);
        }
        deferred_update_wg(A, ps, k, pl, ne, W, wld);
        if (stalled && k < ne) {
            ++n_search;
            const int ss = k;
            int kind, pa, pb;
            select_pivot_wg(A, k, ne, ne, prm_f, rs, kind, pa, pb);
            bool az = false;
            if (kind == 0) {
                if (!(sp > 0.0)) break;
                int raised;
                pa = force_static_wg(A, k, ne, sp, prm_f, rs, raised, nstatic, growth);
                kind = 1;
                az = static_as_zero(raised, prm_f, Fd);
            }
            apply_pivot_wg(A, kind, pa, pb, k, rows, tags, W, wld, 0, ss, prm_f, cnt, flops, 0, az);
            deferred_update_wg(A, ss, k, k, ne, W, wld);
        }
    }
    schur_update_wg(A, k, ne, tags);
    if (tid == 0) {
        Fd.p = k;
        Fd.npos = cnt[0];
        Fd.nneg = cnt[1];
        Fd.nzero = cnt[2];
        Fd.flops = flops;
        Fd.nstatic = nstatic;
        Fd.growth = growth;
        Fd.stalls = n_stall;
        Fd.pulls = n_pull;
        Fd.rotated = n_rot;
        Fd.searches = n_search;
    }
}

void launch_ldlt_blocked(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, double u,
                         double eff_small, double small_pivot, int32_t nb, const StaticPrm &S) {
    if (nf <= 0) return;
    Prm prm{u, eff_small, small_pivot, 0.0, S};
    for (int64_t o = 0; o < nf; o += kMaxLaunchGroups)
        k_ldlt_blocked<<<dim3(static_cast<unsigned>(std::min<int64_t>(kMaxLaunchGroups, nf - o))), kLT, 0, st>>>(
            d, flist + o, prm, nb);
}

// ---------------------------------------------------------------------------
// Large fronts: ldlt_factor_front's blocked path (ldlt_kernel.cpp:1028-1139)
// split over kernels. The panel kernel runs the pivot logic of one panel
// (select_pivot / apply_pivot on the panel's columns, the unscaled columns
// kept in W); the update kernel applies the deferred updates on MFMA; the
// stall kernel does the partner pulls or the rotation of a stalled panel.
// The deferred update of a panel (columns [pl, ne), rows [pl, f),
// ldlt_kernel.cpp:705-761) is applied at once to the outer block's columns
// and held back for the columns past it until a flush; sums differ from the
// reference's only in order.

// Tile `tile` of the lower part (row block >= column block) of nrb x ncb
// tile blocks, in 8 x 8 super-blocks: super-columns left to right, each
// from its diagonal super-block down, tiles column-major inside a
// super-block. Consecutive tiles (one XCD's run) then share 8 row and 8
// column operand panels, which stay in its L2.
__device__ __forceinline__ void super_block_tile(int nrb, int ncb, int tile, int &ib, int &jb) {
    int sj = 0, rem = tile;
    for (;; ++sj) {
        const int w = min(8, ncb - 8 * sj), h = min(8, nrb - 8 * sj);
        // diagonal super-block: column jj holds rows jj .. h-1
        const int diag = w * h - w * (w - 1) / 2;
        const int total = diag + w * (nrb - 8 * sj - h);
        if (rem < total || 8 * (sj + 1) >= ncb) {
            if (rem < diag) {
                int jj = 0;
                while (rem >= h - jj) {
                    rem -= h - jj;
                    ++jj;
                }
                ib = 8 * sj + jj + rem;
                jb = 8 * sj + jj;
                return;
            }
            rem -= diag;
            const int below = nrb - 8 * sj - h;  // rows under the diagonal super-block
            const int nf = below / 8, lr = below % 8;
            const int base = 8 * sj + h;
            if (rem < nf * 8 * w) {
                const int b = rem / (8 * w), q = rem % (8 * w);
                ib = base + 8 * b + q % 8;
                jb = 8 * sj + q / 8;
            } else {
                const int q = rem - nf * 8 * w;
                ib = base + 8 * nf + q % lr;
                jb = 8 * sj + q / lr;
            }
            return;
        }
        rem -= total;
    }
}

// MFMA tile of C[i][j] -= sum_t A[i][t] * B[j][t - boff] over the lower
// part of rows [c0, f) x columns [c0, c1) of front F (c1 - c0 <= f - c0);
// tile `tile` of the region in super-block order. MODE 0: FP64 MFMA;
// 1: FP32 MFMA on the FP64 operands (rounded as they enter LDS); 2: BF16
// MFMA (operands rounded to bf16); 3: split BF16 (hi / lo operands, four
// MFMAs). Modes 1-3 accumulate in FP32 over the panel and subtract the
// result from the FP64 entries.
constexpr int kBigKcBf = 32;  // panel columns per LDS stage of the BF16 tiles (FP64 operands in registers)
template <int MODE, int TILE = kT>
__host__ __device__ constexpr int big_lds_bytes() {
    return MODE <= 1 ? 4 * 16 * TILE * static_cast<int>(sizeof(double)) : bf_lds_bytes<MODE == 3, kBigKcBf, TILE>();
}
template <int MODE, int TILE = kT>
__device__ __forceinline__ void big_tile(const LdltDev &d, const FrontLd &F, const double *Bm, int boff, int c0, int c1, int t0,
                         int t1, int tile, unsigned char *smem) {
    typedef typename std::conditional<MODE == 0, double, float>::type E;
    typedef SyrkMfma<E> M;
    const int f = F.f;
    int ib, jb;
    super_block_tile((f - c0 + TILE - 1) / TILE, (c1 - c0 + TILE - 1) / TILE, tile, ib, jb);
    constexpr int kNB = TILE / 32, kW = TILE / 2;  // MFMA blocks of a wave each way, its rows
    const int i0 = c0 + ib * TILE, j0 = c0 + jb * TILE;
    double *G = d.arena + F.fofs;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wr = w >> 1, wc = w & 1;
    const bool active = (i0 + wr * kW + kW - 1) >= (j0 + wc * kW);
    typename M::acc_t acc[kNB][kNB];
#pragma unroll
    for (int a = 0; a < kNB; ++a)
#pragma unroll
        for (int b = 0; b < kNB; ++b) acc[a][b] = M::zero();
    if constexpr (MODE <= 1) {
        if (active) tile_loop<E, true, 16, 2, double, TILE>(G, Bm, f, boff, i0, j0, f, c1, t0, t1, smem, acc);
        else tile_loop<E, false, 16, 2, double, TILE>(G, Bm, f, boff, i0, j0, f, c1, t0, t1, smem, acc);
    } else {
        if (active) tile_loop_bf16<MODE == 3, true, kBigKcBf, double, TILE>(G, Bm, f, boff, i0, j0, f, c1, t0, t1, smem, acc);
        else tile_loop_bf16<MODE == 3, false, kBigKcBf, double, TILE>(G, Bm, f, boff, i0, j0, f, c1, t0, t1, smem, acc);
    }
    if (!active) return;
    double *junk = d.junk + threadIdx.x;
#pragma unroll
    for (int m = 0; m < kNB; ++m) {
        double *dst[kNB][4];
        double old[kNB][4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = j0 + wc * kW + m * 16 + M::row(v, lane);
            double *col = G + static_cast<int64_t>(min(j, c1 - 1)) * f;
#pragma unroll
            for (int nn = 0; nn < kNB; ++nn) {
                const int i = i0 + wr * kW + nn * 16 + (lane & 15);
                dst[nn][v] = (i < f && j < c1 && i >= j) ? col + i : junk;
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int nn = 0; nn < kNB; ++nn) old[nn][v] = *dst[nn][v];
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int nn = 0; nn < kNB; ++nn) *dst[nn][v] = old[nn][v] - acc[m][nn][v];
    }
}

// Tiles [lo, hi) of a launch's range of nt for this workgroup's XCD, which
// its workgroups stride over: workgroups are dispatched to the 8 XCDs round
// robin by linear index, so with a multiple of 8 per front, part % 8
// is the XCD. Each XCD then works through a contiguous run of tiles (one
// column block's operand panel stays in its L2) instead of every eighth.
struct XcdRange {
    int lo, hi, step;
};
__device__ __forceinline__ XcdRange xcd_range(const BigPart &g, int nt) {
    const int x = g.part & 7, per = g.parts >> 3;
    const int lo = static_cast<int>(static_cast<int64_t>(nt) * x / 8);
    const int hi = static_cast<int>(static_cast<int64_t>(nt) * (x + 1) / 8);
    return XcdRange{lo + (g.part >> 3), hi, per};
}

template <int TILE = kT>
__device__ __forceinline__ int big_tiles(int f, int c0, int c1) {
    if (c1 <= c0) return 0;
    const int nr = (f - c0 + TILE - 1) / TILE, nc = (c1 - c0 + TILE - 1) / TILE;
    return nc * nr - nc * (nc - 1) / 2;
}

// ---------------------------------------------------------------------------
// Speculative panel groups (first pass of the large-front path). When every
// pivot of a panel passes select_pivot's first test (the diagonal against u
// times the largest entry of its column, ldlt_kernel.cpp:145-178), the
// panel's pivots are 1x1, in order, without swaps, and each row of the front
// goes through a fixed sequence of row-local operations: eliminate_1x1's
// rank-1 updates within the panel (ldlt_kernel.cpp:350-432) and the deferred
// update of the later columns (705-761). A group of up to four panels of 16
// is evaluated under that assumption, a round of four launches: the region
// launch (one workgroup per front; it first moves the rows of a panel that
// stalled in the round before) factors the group's 64 x 64 diagonal region;
// the rows launch carries the rows below it through the same pivots and
// records per pivot the largest entry of its column; the panel launch applies
// the first test to each pivot in order, accepts the leading panels that pass
// and writes their columns; the update launch applies the deferred updates. A
// panel that fails is factored by the panel launch's full search. A row's
// operations are those of the one-panel path with each multiply and subtract
// fused.
// Guarded loads are unconditional loads from clamped (in-front) addresses
// times a 0 / 1 mask, so the compiler keeps every load of a row in flight
// (inputs are finite: the factorization rejects non-finite values).
__device__ __forceinline__ double masked(double v, bool keep) { return v * (keep ? 1.0 : 0.0); }

// Columns of the group the one-panel path would factor next if no panel
// stalled: panels of nb from k, each ending at min(live, start + nb), the
// group ending after the panel whose end triggers the outer block's flush.
// Every panel but the last has 16 columns.
__device__ __forceinline__ int group_cols(const BigLd &B, int nb) {
    if (B.pass != 0 || !B.spec || nb != 16 || B.k >= B.live) return 0;
    int pos = B.k;
    for (int m = 0; m < 4 && pos < B.live; ++m) {
        const int pl = min(B.live, pos + nb);
        if (pl > B.oe) break;
        pos = pl;
        if (pl + nb > B.oe || pl >= B.live) break;
    }
    return pos - B.k;
}

// Group buffer per front (doubles).
constexpr int64_t kGMax = 0;                    // 64: per pivot the bits of the largest |entry| below it in its column
constexpr int64_t kGdPiv = 64;                  // 64: pivots
constexpr int64_t kGdInv = 128;                 // 64: 1 / pivot
constexpr int64_t kGdWd = 192;                  // 64 x 64: [t][r] row r of the region at pivot t, unscaled
constexpr int64_t kGdFin = kGdWd + 64 * 64;     // 64 x 64: [c][r] the region's final entries (r > c: row r's multiplier)
static_assert(kGdFin + 64 * 64 == kGroupBuf, "group buffer layout");

// 1 / d: the hardware estimate (better than 2^-20), a third-order step in
// the residual e = 1 - d y, and one Newton step for the last bit
__device__ __forceinline__ double pivot_rcp(double d) {
    double y = __builtin_amdgcn_rcp(d);
    double e = fma(-d, y, 1.0);
    y = fma(y, fma(e, e, e), y);
    e = fma(-d, y, 1.0);
    return fma(y, e, y);
}
// v of lane C of the lane's row of 16 lanes
template <int C>
__device__ __forceinline__ double row_bcast(double v) {
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + C, 0xf, 0xf, true);
}

// Pivot J of a 16-column panel of the region: a the diagonal block's row,
// x the lane's own row, inv 1 / pivot. l receives the scaled column (rows
// past the pivot), a and x keep theirs unscaled. The next pivot's column
// goes first.
template <int J, int C>
__device__ __forceinline__ void region_cols(double (&a)[16], double (&x)[16], double la) {
    if constexpr (C < 16) {
        const double m = row_bcast<C>(la);
        a[C] = fma(-a[J], m, a[C]);
        x[C] = fma(-x[J], m, x[C]);
        region_cols<J, C + 1>(a, x, la);
    }
}
template <int J>
__device__ __forceinline__ void region_pivots(double (&a)[16], double (&x)[16], double (&l)[16], double (&dv)[16],
                                              double (&iv)[16], double dj, double inv) {
    if constexpr (J < 16) {
        dv[J] = dj;
        iv[J] = inv;
        const double la = a[J] * inv;
        l[J] = x[J] * inv;
        double dn = 0.0, in = 0.0;
        if constexpr (J + 1 < 16) {
            const double m = row_bcast<J + 1>(la);
            a[J + 1] = fma(-a[J], m, a[J + 1]);
            dn = row_bcast<J + 1>(a[J + 1]);
            in = pivot_rcp(dn);
            x[J + 1] = fma(-x[J], m, x[J + 1]);
        }
        region_cols<J, J + 2>(a, x, la);
        region_pivots<J + 1>(a, x, l, dv, iv, dn, in);
    }
}

constexpr int kRLd = 81;  // column stride of the region's LDS squares (odd: a column scan by 64 lanes spreads over the banks)

// Block (i, c) of the region -= W block (i, p) times L block (c, p)^T
__device__ __forceinline__ void region_update(double *S, const double *Ls, int p, int i, int c) {
    const int lr = threadIdx.x & 15, lk = (threadIdx.x & 63) >> 4;
    v4d_t acc;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = S[(16 * c + 4 * v + lk) * kRLd + 16 * i + lr];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(Ls[(16 * p + 4 * kk + lk) * kRLd + 16 * c + lr],
                                                   -S[(16 * p + 4 * kk + lk) * kRLd + 16 * i + lr], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) S[(16 * c + 4 * v + lk) * kRLd + 16 * i + lr] = acc[v];
}

// Partner pulls or rotation of a stalled first-pass panel
// (ldlt_kernel.cpp:1052-1097); every column is current (flushed).
__device__ void big_stall_wg(const LdltDev &d, BigLd &B, int32_t nb, RedScratch &rs, int32_t *order) {
    FrontLd &Fd = d.fronts[B.s];
    const int f = Fd.f, ne = Fd.ne;
    int32_t *rows = d.rows + Fd.rofs;
    FV A{d.arena + Fd.fofs, f, f};
    const int tid = threadIdx.x;
    const int k = B.k, pl = B.pl;
    const int live = B.live, k_paired = B.k_paired;
    __syncthreads();  // every thread has read the state before thread 0 changes it
    if (k != k_paired) {
        const int np = partner_pairs_wg(A, k, pl, ne, nb, rows, order, rs);
        if (np > 0) {
            place_rows_wg(A, k, ne, np, order, rows, rs);
            if (tid == 0) {
                B.live = max(live, k + np);
                B.k_paired = k;
                B.stalled = 0;
                B.stalls += 1;
                B.pulls += np / 2;
            }
            return;
        }
    }
    const int m = pl - k;
    const int mv = min(m, live - pl);
    for (int t = 0; t < mv; ++t) sym_swap_wg(A, k + t, live - mv + t, rows, nullptr, 0, 0, 0);
    if (tid == 0) {
        B.live = live - m;
        B.stalled = 0;
        B.stalls += 1;
        B.rotated += m;
    }
}

// One workgroup per front: the pulls or rotation of a panel that stalled in
// the round before, then the next group's diagonal region [ps, ps + ncols)
// (padded to 64 with the identity) in 16-column panels: wavefront 0 runs a
// panel's pivots in registers, one row of the region per lane and beside it
// the diagonal block's row (multipliers broadcast inside each row of 16
// lanes by DPP), then the columns right of it are updated on FP64 MFMA, the
// next panel's by every wavefront, the rest by wavefronts 1 to 3 beside the
// next panel's pivots. Bound by wavefront 0's chain of 64 pivots: 42 us with
// one wavefront and every multiplier through readlane, 12.8 us now.
__global__ __launch_bounds__(kLT) void k_big_region(LdltDev d, BigLd *__restrict__ states, double *__restrict__ gpart,
                                                    int32_t nb) {
    __shared__ double S[64 * kRLd];   // the region, columns unscaled once factored
    __shared__ double Ls[64 * kRLd];  // final entries: multipliers below the pivots, pivots on the diagonal
    __shared__ double dd[64], invd[64];
    __shared__ RedScratch rs;
    __shared__ int32_t order[128];
    // (every wavefront has read it when big_stall_wg changes it)
    if (states[blockIdx.x].pass == 0 && states[blockIdx.x].stalled) {
        big_stall_wg(d, states[blockIdx.x], nb, rs, order);
        __syncthreads();
    }
    if (gpart == nullptr) return;
    const BigLd B = states[blockIdx.x];
    const int ps = B.k, ncols = group_cols(B, nb);
    if (ncols <= 0) return;
    const FrontLd F = d.fronts[B.s];
    const int f = F.f;
    const double *G = d.arena + F.fofs;
    double *gp = gpart + blockIdx.x * kGroupBuf;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    {
        double v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            v[i] = G[static_cast<int64_t>(ps + min(w + 4 * i, ncols - 1)) * f + ps + min(lane, ncols - 1)];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int c = w + 4 * i;
            S[c * kRLd + lane] = (lane < ncols && c <= lane) ? v[i] : (lane == c ? 1.0 : 0.0);
        }
    }
    const int nblk = (ncols + 15) / 16;
    __syncthreads();
    for (int p = 0; p < nblk; ++p) {
        if (w == 0) {
            double a[16], x[16], l[16], dv[16], iv[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                a[c] = S[(16 * p + c) * kRLd + 16 * p + lr];
                x[c] = S[(16 * p + c) * kRLd + lane];
            }
            const double d0 = row_bcast<0>(a[0]);
            region_pivots<0>(a, x, l, dv, iv, d0, pivot_rcp(d0));
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                const int col = 16 * p + c;
                S[col * kRLd + lane] = x[c];
                Ls[col * kRLd + lane] = lane > col ? l[c] : x[c];
                dd[col] = dv[c];
                invd[col] = iv[c];
            }
        } else if (p > 0) {
            // the rest of panel p - 1's update: columns from p + 1 on
            int t = 0;
            for (int c = p + 1; c < nblk; ++c)
                for (int i = c; i < nblk; ++i)
                    if (t++ % 3 == w - 1) region_update(S, Ls, p - 1, i, c);
        }
        __syncthreads();
        if (p + 1 < nblk) {
            if (w + p + 1 < nblk) region_update(S, Ls, p, w + p + 1, p + 1);
            __syncthreads();
        }
    }
    // the largest entry below each pivot, one quarter of the rows per wave
    {
        double mx = 0.0;
        if (lane < ncols)
            for (int r = max(16 * w, lane + 1); r < min(16 * w + 16, ncols); ++r) mx = fmax(mx, fabs(S[lane * kRLd + r]));
        rs.v[tid] = mx;
    }
    __syncthreads();
    if (tid < 64) {
        reinterpret_cast<unsigned long long *>(gp + kGMax)[tid] = static_cast<unsigned long long>(
            __double_as_longlong(fmax(fmax(rs.v[tid], rs.v[tid + 64]), fmax(rs.v[tid + 128], rs.v[tid + 192]))));
        if (tid < ncols) {
            gp[kGdPiv + tid] = dd[tid];
            gp[kGdInv + tid] = invd[tid];
        }
    }
    for (int e = tid; e < 64 * 64; e += kLT) {
        const int c = e >> 6, r = e & 63;
        if (c < 16 * nblk) {
            gp[kGdWd + e] = S[c * kRLd + r];
            gp[kGdFin + e] = Ls[c * kRLd + r];
        }
    }
}

// Largest of 8 values per lane over the wavefront, value e in the lanes
// whose top three bits are e: three halving exchanges (halves of the
// wavefront, rows of 16 lanes, rotation by 8), then the 8 lanes that share e.
__device__ __forceinline__ double wave_max8(double (&v)[8]) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const auto pick = [](u2 lo, u2 hi) {
        return fmax(__hiloint2double(hi[0], lo[0]), __hiloint2double(hi[1], lo[1]));
    };
#pragma unroll
    for (int k = 0; k < 4; ++k)
        v[k] = pick(__builtin_amdgcn_permlane32_swap(__double2loint(v[k]), __double2loint(v[k + 4]), false, false),
                    __builtin_amdgcn_permlane32_swap(__double2hiint(v[k]), __double2hiint(v[k + 4]), false, false));
#pragma unroll
    for (int k = 0; k < 2; ++k)
        v[k] = pick(__builtin_amdgcn_permlane16_swap(__double2loint(v[k]), __double2loint(v[k + 2]), false, false),
                    __builtin_amdgcn_permlane16_swap(__double2hiint(v[k]), __double2hiint(v[k + 2]), false, false));
    const bool up = (threadIdx.x & 8) != 0;
    double t = fmax(up ? v[1] : v[0], dpp_d<0x128>(up ? v[0] : v[1]));
    t = fmax(t, dpp_d<kDppXor1>(t));
    t = fmax(t, dpp_d<kDppXor2>(t));
    return fmax(t, dpp_d<kDppHalfMirror>(t));
}

// Rows of a group below its diagonal region, [ps + ncols, f), kGroupRows
// (one wavefront, a row per lane) per workgroup: column maxima per pivot to
// the group buffer (atomic maxima of the bits of |entry|), each row's
// unscaled column entries to W (the columns the panel kernel's pivots will
// have: W column ps - pend0 + t, pend0 being the W base the panel kernel
// starts from) and its final group entries to W's speculation columns
// [big_spec, big_spec + 64). Nothing of the front square changes: a rejected
// panel finds its columns as they were. W columns of rejected pivots are
// rewritten (rows below the pivot) when those positions get their pivots.
// A row's 64 columns stay in its lane's registers. Panel by panel: the
// earlier panels' update on FP64 MFMA (operands and result through LDS, which
// turns the tile's layout into rows per lane), then the panel's 16 pivots,
// their multipliers broadcast inside each row of 16 lanes by DPP. Bound by
// latency: the columns' loads, then one wavefront's work in turn (96 MFMAs of
// 64 cycles' issue, 480 FMAs with a broadcast each, and the panels' trips
// through LDS between them). 58 us with separate
// multiplies and subtracts, multipliers from LDS and 256 rows a workgroup;
// 32 us with all 2016 FMAs of a row on the vector unit; 16.8 us now.
constexpr int kGLd = 80;  // LDS column stride: the two lane rows of a half wavefront fall on different banks

template <int P, int T, int J>
__device__ __forceinline__ void group_cols_fma(double (&a)[kGroupCols], double na, double l) {
    if constexpr (J < 16) {
        a[16 * P + J] = fma(na, row_bcast<J>(l), a[16 * P + J]);
        group_cols_fma<P, T, J + 1>(a, na, l);
    }
}
template <int P, int T>
__device__ __forceinline__ void group_pivots(double (&a)[kGroupCols], const double (&l)[16]) {
    if constexpr (T < 15) {
        group_cols_fma<P, T, T + 1>(a, -a[16 * P + T], l[T]);
        group_pivots<P, T + 1>(a, l);
    }
}
// Panel P of the rows' columns; Lc[t][j]: multiplier of column j by pivot t;
// X: the earlier panels' columns (slot per panel), D in a slot not needed any
// more.
template <int P>
__device__ __forceinline__ void group_panel(double (&a)[kGroupCols], const double (*Lc)[kGLd], double (*X)[16][kGLd]) {
    const int lane = threadIdx.x, lr = lane & 15, lk = lane >> 4;
    if constexpr (P > 0) {
        v4d_t acc[4];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) acc[rt] = v4d_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < P; ++i)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const double l = Lc[16 * i + 4 * kk + lk][16 * P + lr];
#pragma unroll
                for (int rt = 0; rt < 4; ++rt)
                    acc[rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(l, X[i][4 * kk + lk][16 * rt + lr], acc[rt], 0, 0, 0);
            }
        double (*D)[kGLd] = X[P < 2 ? P : 2];
        __syncthreads();
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int v = 0; v < 4; ++v) D[4 * v + lk][16 * rt + lr] = acc[rt][v];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 16; ++c) a[16 * P + c] -= D[c][lane];
    }
    double l[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) l[t] = Lc[16 * P + t][16 * P + lr];
    group_pivots<P, 0>(a, l);
    if constexpr (P < 3) {
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 16; ++c) X[P][c][lane] = a[16 * P + c];
        __syncthreads();
    }
}

__global__ __launch_bounds__(kGroupRows) void k_big_group(LdltDev d, const BigLd *__restrict__ states,
                                                          const BigPart *__restrict__ grid,
                                                          double *__restrict__ gpart) {
    static_assert(kGroupRows == 64, "one wavefront, a row per lane");
    __shared__ double Lc[kGroupCols][kGLd];
    __shared__ double X[3][16][kGLd];
    __shared__ double invs[kGroupCols];
    const BigPart g = grid[blockIdx.x];
    const BigLd B = states[g.front];
    const int ps = B.k, ncols = group_cols(B, 16);
    if (ncols <= 0) return;
    const FrontLd F = d.fronts[B.s];
    const int f = F.f;
    const int lane = threadIdx.x;
    const int i = ps + ncols + g.part * kGroupRows + lane;
    if (ps + ncols + g.part * kGroupRows >= f) return;
    const bool rowok = i < f;
    const double *Gi = d.arena + F.fofs + static_cast<int64_t>(ps) * f + min(i, f - 1);
    const double *__restrict__ gp = gpart + g.front * kGroupBuf;
    double a[kGroupCols];
#pragma unroll
    for (int c = 0; c < kGroupCols; ++c) a[c] = Gi[static_cast<int64_t>(min(c, ncols - 1)) * f];
    invs[lane] = gp[kGdInv + min(lane, ncols - 1)];
    // the multipliers (columns past the region's panels are not read)
#pragma unroll
    for (int t0 = 0; t0 < kGroupCols; t0 += 16) {
        if (t0 < ncols) {
            double v[16];
#pragma unroll
            for (int t = 0; t < 16; ++t) v[t] = gp[kGdFin + (t0 + t) * 64 + lane];
#pragma unroll
            for (int t = 0; t < 16; ++t) Lc[t0 + t][lane] = v[t];
        }
    }
#pragma unroll
    for (int c = 0; c < kGroupCols; ++c) a[c] = masked(a[c], rowok && c < ncols);
    __syncthreads();
    group_panel<0>(a, Lc, X);
    if (ncols > 16) group_panel<1>(a, Lc, X);
    if (ncols > 32) group_panel<2>(a, Lc, X);
    if (ncols > 48) group_panel<3>(a, Lc, X);
    double *W = d.work + F.wofs;
    double *Wu = W + static_cast<int64_t>(ps - B.pend0) * f + i;    // from the W column of the group's first pivot
    double *Wf = W + static_cast<int64_t>(big_spec(F.ne)) * f + i;
    auto *gmax = reinterpret_cast<unsigned long long *>(gpart + g.front * kGroupBuf + kGMax);
#pragma unroll
    for (int c0 = 0; c0 < kGroupCols; c0 += 8) {
        if (c0 >= ncols) break;
        double m[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int c = c0 + u;
            m[u] = fabs(a[c]);
            if (rowok && c < ncols) {
                Wu[static_cast<int64_t>(c) * f] = a[c];
                Wf[static_cast<int64_t>(c) * f] = a[c] * invs[c];
            }
        }
        const double mx = wave_max8(m);
        const int c = c0 + (lane >> 3);
        if ((lane & 7) == 0 && c < ncols)
            atomicMax(gmax + c, static_cast<unsigned long long>(__double_as_longlong(mx)));
    }
}

// Leading panels of a group that pass the first test: the number of accepted
// columns, from the pivots and column maxima the region and rows launches
// left (lane c of every wavefront tests column c). A NaN pivot fails; a NaN
// below it (only an overflow makes one, the input is finite) is passed over by
// the maxima, as by select_pivot's.
__device__ __forceinline__ int group_accepted(const double *gp, int gcols, const Prm &prm, double &piv) {
    const int c = threadIdx.x & 63;
    bool ok = true;
    piv = 0.0;
    if (c < gcols) {
        piv = gp[kGdPiv + c];
        const double a0 = fabs(piv), cm = gp[kGMax + c];
        ok = a0 >= prm.eff_small && prm.u * cm <= a0 && !(a0 < kWeakPivotRatio * cm);
    }
    const unsigned long long bad = __ballot(!ok);
    if (bad == 0) return gcols;
    return (__ffsll(bad) - 1) / 16 * 16;
}

// The panel launch, a workgroup per kGroupRows rows of a front: every
// workgroup judges the group and copies the accepted panels' columns of its
// rows from W's speculation columns to the front; the first one also writes
// the region's own entries and does the pivot logic: what to update and
// flush, or, without an accepted group, one panel with the full pivot
// search. It reads the round's states and writes the next ones (other
// workgroups still read the old).
__global__ __launch_bounds__(kLT) void k_big_panel(LdltDev d, const BigLd *__restrict__ states,
                                                  BigLd *__restrict__ next, const BigPart *__restrict__ grid,
                                                  Prm prm, int32_t nb, const double *__restrict__ gpart) {
    __shared__ RedScratch rs;
    __shared__ int cnt[3];
    const BigPart g = grid[blockIdx.x];
    BigLd B = states[g.front];
    const int pass = B.pass;
    const int gcols = gpart ? group_cols(B, nb) : 0;
    const int tid = threadIdx.x;
    if (pass == 2) {
        // done: nothing for this round's update launch
        if (g.part == 0 && tid == 0) {
            B.u_p1 = B.u_p0;
            B.x_p1 = B.x_p0;
            B.stalled = 0;
            next[g.front] = B;
        }
        return;
    }
    if (gcols <= 0 && g.part > 0) return;
    FrontLd &Fd = d.fronts[B.s];
    const int f = Fd.f, ne = Fd.ne;
    int32_t *rows = d.rows + Fd.rofs;
    int8_t *tags = d.tags + Fd.rofs;
    double *W = d.work + Fd.wofs;
    FV A{d.arena + Fd.fofs, f, f};
    int k = B.k, oe = B.oe, pend0 = B.pend0, full = B.full;
    const int live = B.live;
    double flops = B.flops;
    int u_c0 = 0, u_c1 = 0, u_p0 = 0, u_p1 = 0, x_c0 = ne, x_p0 = 0, x_p1 = 0, w_base = pend0;
    int stalled = 0, npass = pass, ps = k, pl = k;
    int spec = B.spec, searched = 0;
    bool group_done = false;
    int nacc = 0, npos = 0, nzero = 0;
    if (gcols > 0) {
        const double *gp = gpart + g.front * kGroupBuf;
        double piv;
        nacc = group_accepted(gp, gcols, prm, piv);
        if (nacc > 0) {
            // rows below the region: eight columns' loads in flight
            const int i = k + gcols + g.part * kGroupRows + (tid & 63);
            if (i < f) {
                const double *src = W + static_cast<int64_t>(big_spec(ne)) * f + i;
                double *dst = A.F + static_cast<int64_t>(k) * f + i;
                for (int c0 = 16 * (tid >> 6); c0 < min(nacc, 16 * (tid >> 6) + 16); c0 += 8) {
                    double v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = src[static_cast<int64_t>(min(c0 + u, nacc - 1)) * f];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (c0 + u < nacc) dst[static_cast<int64_t>(c0 + u) * f] = v[u];
                }
            }
        }
        if (g.part > 0) return;
        if (nacc > 0) {
            // the region's entries; a row of it at or past nacc went through
            // the same operations on the accepted columns as a row below it
            const int64_t wcol0 = k - pend0;
            for (int e = tid; e < kGroupCols * kGroupCols; e += kLT) {
                const int c = e >> 6, rw = e & 63;
                if (c < nacc && rw < gcols && c <= rw) {
                    A.at(k + rw, k + c) = gp[kGdFin + e];
                    if (c < rw) W[(wcol0 + c) * f + k + rw] = gp[kGdWd + e];
                }
            }
            // inertia of the accepted pivots, as inertia_1x1; flops in exact
            // integers
            const bool in = (tid & 63) < nacc;
            const bool zero = in && (!isfinite(piv) || fabs(piv) < prm.eff_small);
            const bool pos = in && !zero && piv > 0.0;
            nzero = __popcll(__ballot(zero));
            npos = __popcll(__ballot(pos));
            for (int kk = 0; kk < nacc; ++kk) {
                const double rem = static_cast<double>(f - (k + kk + 1));
                flops += rem + rem * (rem + 1.0);
            }
            for (int c = tid; c < nacc; c += kLT) tags[k + c] = 1;
            const int kn = k + nacc;
            if (kn < oe) {
                u_c0 = kn;
                u_c1 = oe;
                u_p0 = k;
                u_p1 = kn;
            }
            if (kn + nb > oe || kn >= live) {
                if (kn > pend0 && oe < ne) {
                    x_c0 = oe;
                    x_p0 = pend0;
                    x_p1 = kn;
                }
                pend0 = kn;
                oe = min(ne, kn + B.outer);
            }
            spec = nacc == gcols ? 1 : 0;  // a panel failed inside: the next panel goes the one-panel way
            ps = k + ((nacc - 1) / 16) * 16;
            pl = kn;
            k = kn;
            group_done = true;
        }
    }
    if (tid < 3) cnt[tid] = states[g.front].cnt[tid] + (tid == 0 ? npos : (tid == 1 ? nacc - npos - nzero : nzero));
    __syncthreads();
    if (group_done) {
    } else if (pass == 0) {
        spec = 1;
        if (k >= live) {
            // the first pass is over: what is held back goes out, then the
            // second pass (single-level updates)
            if (k > pend0 && oe < ne) {
                x_c0 = oe;
                x_p0 = pend0;
                x_p1 = k;
            }
            pend0 = k;
            oe = ne;
            npass = 1;
        } else {
            ps = k;
            pl = min(live, ps + nb);
            while (k < pl) {
                int kind, pa, pb;
                select_pivot_wg(A, k, ne, pl, prm, rs, kind, pa, pb);
                if (kind == 0) {
                    stalled = 1;
                    break;
                }
                apply_pivot_wg(A, kind, pa, pb, k, rows, tags, W + static_cast<int64_t>(ps - pend0) * f, f, k - ps, pl,
                               prm, cnt, flops, 0);
            }
            if (k > ps && pl < oe) {
                u_c0 = pl;
                u_c1 = oe;
                u_p0 = ps;
                u_p1 = k;
            }
            // flush before pulls / rotation (they move columns past the
            // outer block), at the end of the outer block and of the pass
            if (stalled || k + nb > oe || k >= live) {
                if (k > pend0 && oe < ne) {
                    x_c0 = oe;
                    x_p0 = pend0;
                    x_p1 = k;
                }
                pend0 = k;
                oe = min(ne, k + B.outer);
            }
        }
    } else {
        oe = ne;
        if (full) {
            // a stalled second-pass panel: one pivot from a search over all
            // the remaining columns (ldlt_kernel.cpp:1119-1131)
            searched = 1;
            const int ss = k;
            int kind, pa, pb;
            select_pivot_wg(A, k, ne, ne, prm, rs, kind, pa, pb);
            if (kind == 0) {
                npass = 2;
            } else {
                apply_pivot_wg(A, kind, pa, pb, k, rows, tags, W, f, 0, ss, prm, cnt, flops, 0);
                u_c0 = k;
                u_c1 = ne;
                u_p0 = ss;
                u_p1 = k;
                w_base = ss;
                pend0 = k;
            }
            full = 0;
        } else if (k >= ne) {
            npass = 2;
        } else {
            ps = k;
            pl = min(ne, ps + nb);
            while (k < pl) {
                int kind, pa, pb;
                select_pivot_wg(A, k, ne, pl, prm, rs, kind, pa, pb);
                if (kind == 0) {
                    stalled = 1;
                    break;
                }
                apply_pivot_wg(A, kind, pa, pb, k, rows, tags, W, f, k - ps, pl, prm, cnt, flops, 0);
            }
            w_base = ps;
            if (k > ps && pl < ne) {
                u_c0 = pl;
                u_c1 = ne;
                u_p0 = ps;
                u_p1 = k;
            }
            if (stalled) full = 1;
            pend0 = k;
        }
    }
    // every eligible column is a pivot: no second pass, and this iteration's
    // updates are the last
    if (pass == 0 && k >= ne) npass = 2;
    __syncthreads();
    if (tid == 0) {
        B.k = k;
        B.pass = npass;
        B.full = full;
        B.stalled = stalled;
        B.ps = ps;
        B.pl = pl;
        B.oe = oe;
        B.pend0 = pend0;
        B.u_c0 = u_c0;
        B.u_c1 = u_c1;
        B.u_p0 = u_p0;
        B.u_p1 = u_p1;
        B.x_c0 = x_c0;
        B.x_p0 = x_p0;
        B.x_p1 = x_p1;
        B.w_base = w_base;
        B.cnt[0] = cnt[0];
        B.cnt[1] = cnt[1];
        B.cnt[2] = cnt[2];
        B.flops = flops;
        B.searches += searched;
        B.spec = spec;
        next[g.front] = B;
    }
}

// The requested update and flush of every front, its tiles by stride over
// its workgroups. The update (a group's 64 columns applied to the rest of
// their outer block) has few tiles and little depth: 64 x 64 tiles while that
// is at most two of them a workgroup (the chip's share of the front: more
// read their operands too often): 15.9 us an update and flush against 22.4
// with 128 x 128 tiles (fronts of up to 1700 rows), 36.7 against 42.5 (8216
// rows). SMALL: the updates of fronts whose flush is
// k_big_wide's, all in 64 x 64 tiles (LDS of three workgroups a CU, not
// one): 22.1 against 23.8 us (23348 rows; 19 us its traffic).
template <int MODE, bool SMALL>
__global__ __launch_bounds__(kLT, 2) void k_big_update(LdltDev d, const BigLd *__restrict__ states,
                                                       const BigPart *__restrict__ grid) {
    constexpr int kS = 64;
    __shared__ __attribute__((aligned(16))) unsigned char smem[SMALL ? big_lds_bytes<MODE, kS>() : big_lds_bytes<MODE>()];
    const BigPart g = grid[blockIdx.x];
    const BigLd B = states[g.front];
    if (B.prec != MODE) return;  // another precision's launch
    const FrontLd F = d.fronts[B.s];
    const double *W = d.work + F.wofs;
    const bool u = B.u_p1 > B.u_p0;
    int t1 = u ? big_tiles<kS>(F.f, B.u_c0, B.u_c1) : 0;
    const bool small = SMALL || (MODE <= 1 && t1 <= 2 * g.parts);
    if (!small) t1 = big_tiles(F.f, B.u_c0, B.u_c1);
    const int t2 = (!SMALL && B.x_p1 > B.x_p0) ? big_tiles(F.f, B.x_c0, F.ne) : 0;
    const XcdRange xr = xcd_range(g, t1 + t2);
    for (int tile = xr.lo; tile < xr.hi; tile += xr.step) {
        if ((SMALL || MODE <= 1) && small && tile < t1) {
            big_tile<MODE, kS>(d, F, W, B.w_base, B.u_c0, B.u_c1, B.u_p0, B.u_p1, tile, smem);
        } else if constexpr (!SMALL) {
            const bool up = tile < t1;
            big_tile<MODE>(d, F, W, B.w_base, up ? B.u_c0 : B.x_c0, up ? B.u_c1 : F.ne, up ? B.u_p0 : B.x_p0,
                           up ? B.u_p1 : B.x_p1, up ? tile : tile - t1, smem);
        }
        __syncthreads();
    }
}

// L*D columns [c0, c1) of every done front, rows [ne, f), into W (the
// column order of schur_update's fill_ld_column, ldlt_kernel.cpp:764-816)
__global__ __launch_bounds__(kLT) void k_big_ld(LdltDev d, const BigLd *__restrict__ states,
                                               const BigPart *__restrict__ grid, int32_t c0, int32_t width,
                                               int32_t wide) {
    const BigPart g = grid[blockIdx.x];
    const BigLd B = states[g.front];
    if ((B.prec >= 2 && d.xpl != nullptr) != (wide != 0)) return;  // the other chunk width's fronts
    const FrontLd F = d.fronts[B.s];
    const int f = F.f, ne = F.ne, p = B.k;
    const int c1 = min(p, c0 + width);
    if (c1 <= c0 || ne >= f) return;
    const double *G = d.arena + F.fofs;
    const int8_t *tags = d.tags + F.rofs;
    double *W = d.work + F.wofs;
    const int q = f - ne;
    const int64_t tot = static_cast<int64_t>(c1 - c0) * q;
    for (int64_t idx = static_cast<int64_t>(g.part) * kLT + threadIdx.x; idx < tot;
         idx += static_cast<int64_t>(g.parts) * kLT) {
        const int c = c0 + static_cast<int>(idx / q);
        const int j = ne + static_cast<int>(idx % q);
        const int8_t tg = tags[c];
        double v = 0.0;
        if (tg == 1) {
            v = G[static_cast<int64_t>(c) * f + j] * G[static_cast<int64_t>(c) * f + c];
        } else if (tg == 2) {
            v = __dadd_rn(G[static_cast<int64_t>(c) * f + j] * G[static_cast<int64_t>(c) * f + c],
                          G[static_cast<int64_t>(c + 1) * f + j] * G[static_cast<int64_t>(c) * f + c + 1]);
        } else if (tg == -1) {
            v = __dadd_rn(G[static_cast<int64_t>(c - 1) * f + j] * G[static_cast<int64_t>(c - 1) * f + c],
                          G[static_cast<int64_t>(c) * f + j] * G[static_cast<int64_t>(c) * f + c]);
        }
        W[static_cast<int64_t>(c - c0) * f + j] = v;
    }
}

template <int MODE>
__global__ __launch_bounds__(kLT, 2) void k_big_cbupdate(LdltDev d, const BigLd *__restrict__ states,
                                                         const BigPart *__restrict__ grid, int32_t c0,
                                                         int32_t width) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[big_lds_bytes<MODE>()];
    const BigPart g = grid[blockIdx.x];
    const BigLd B = states[g.front];
    if (B.prec != MODE) return;
    const FrontLd F = d.fronts[B.s];
    const int c1 = min(B.k, c0 + width);
    if (c1 <= c0 || F.ne >= F.f) return;
    const double *W = d.work + F.wofs;
    const XcdRange xr = xcd_range(g, big_tiles(F.f, F.ne, F.f));
    for (int tile = xr.lo; tile < xr.hi; tile += xr.step) {
        big_tile<MODE>(d, F, W, c0, F.ne, F.f, c0, c1, tile, smem);
        __syncthreads();
    }
}

// 256 x 256 tile of the outer-block updates on the bf16 planes (modes 2,
// 3): C[i][j] -= sum_c A[i][c] B[j][c] over plane columns [0, np), lower
// part of rows [c0, f) x columns [c0, c1) of front F, tile `tile` in
// super-block order.
template <int MODE>
__device__ __forceinline__ void big_tile_w(const LdltDev &d, const FrontLd &F, const uint16_t *pl, int c0, int c1,
                                           int np, int tile, unsigned char *smem) {
    const int f = F.f;
    int ib, jb;
    super_block_tile((f - c0 + kTW - 1) / kTW, (c1 - c0 + kTW - 1) / kTW, tile, ib, jb);
    const int i0 = c0 + ib * kTW, j0 = c0 + jb * kTW;
    double *G = d.arena + F.fofs;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wr = w & 3, wc = w >> 2;
    const bool active = (i0 + wr * 64 + 63) >= (j0 + wc * 128);
    v4f_t acc[8][4];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = v4f_t{0.f, 0.f, 0.f, 0.f};
    const int64_t ps = static_cast<int64_t>(big_work(F.ne)) * f;
    tile_loop_bf16p_w<MODE == 3, kBigKcBf>(pl, pl + ps, pl + 2 * ps, pl + 3 * ps, f, i0, j0, f, c1, 0, np, active, smem,
                                           acc);
    if (!active) return;
    const int ib0 = i0 + wr * 64, jb0 = j0 + wc * 128;
    if (ib0 + 63 < f && jb0 + 127 < c1 && ib0 >= jb0 + 127) {
        // the wave's 64 x 128 block lies inside the front's lower triangle:
        // no masks, and two column blocks (32 entries per lane) at a time,
        // their loads in flight together before their stores
        double *base = G + static_cast<int64_t>(jb0 + 4 * (lane >> 4)) * f + ib0 + (lane & 15);
#pragma unroll
        for (int m0 = 0; m0 < 8; m0 += 2) {
            double old[2][4][4];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const double *col = base + static_cast<int64_t>((m0 + h) * 16 + v) * f;
#pragma unroll
                    for (int nn = 0; nn < 4; ++nn) old[h][nn][v] = col[nn * 16];
                }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    double *col = base + static_cast<int64_t>((m0 + h) * 16 + v) * f;
#pragma unroll
                    for (int nn = 0; nn < 4; ++nn) col[nn * 16] = old[h][nn][v] - acc[m0 + h][nn][v];
                }
        }
        return;
    }
    double *junk = d.junk + threadIdx.x;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        double *dst[4][4];
        double old[4][4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = jb0 + m * 16 + 4 * (lane >> 4) + v;
            double *col = G + static_cast<int64_t>(min(j, c1 - 1)) * f;
#pragma unroll
            for (int nn = 0; nn < 4; ++nn) {
                const int i = ib0 + nn * 16 + (lane & 15);
                dst[nn][v] = (i < f && j < c1 && i >= j) ? col + i : junk;
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int nn = 0; nn < 4; ++nn) old[nn][v] = *dst[nn][v];
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int nn = 0; nn < 4; ++nn) *dst[nn][v] = old[nn][v] - acc[m][nn][v];
    }
}

__device__ __forceinline__ int big_tiles_w(int f, int c0, int c1) {
    if (c1 <= c0) return 0;
    const int nr = (f - c0 + kTW - 1) / kTW, nc = (c1 - c0 + kTW - 1) / kTW;
    return nc * nr - nc * (nc - 1) / 2;
}

// The outer-block updates of BF16 / split-BF16 fronts on their planes, in
// 256 x 256 tiles: CB, the contribution block's chunk at c0 (after
// k_big_ld and k_big_pack<true>); else the flush request (after
// k_big_pack<false>).
template <int MODE, bool CB>
__global__ __launch_bounds__(kWideThreads) void k_big_wide(LdltDev d, const BigLd *__restrict__ states,
                                                           const BigPart *__restrict__ grid, int32_t c0,
                                                           int32_t width) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[bfw_lds_bytes<MODE == 3, kBigKcBf>()];
    const BigPart g = grid[blockIdx.x];
    const BigLd B = states[g.front];
    if (B.prec != MODE) return;
    const FrontLd F = d.fronts[B.s];
    int r0, rc, np;
    if (CB) {
        const int c1 = min(B.k, c0 + width);
        if (c1 <= c0 || F.ne >= F.f) return;
        r0 = F.ne;
        rc = F.f;
        np = c1 - c0;
    } else {
        if (B.x_p1 <= B.x_p0) return;
        r0 = B.x_c0;
        rc = F.ne;
        np = B.x_p1 - B.x_p0;
    }
    const uint16_t *pl = d.xpl + 4 * F.wofs;
    const XcdRange xr = xcd_range(g, big_tiles_w(F.f, r0, rc));
    for (int tile = xr.lo; tile < xr.hi; tile += xr.step) {
        big_tile_w<MODE>(d, F, pl, r0, rc, np, tile, smem);
        __syncthreads();
    }
}

// bf16 planes of an outer-block update's operands in the packed layout of
// tile_loop_bf16p (row i, plane column c at (c / 8) f 8 + 8 i + c % 8), for
// the fronts of BF16 (high part) or split-BF16 (both parts) precision:
// A = front columns [p0, p0 + np), rows [r0, f); B = W columns from p0 - w0,
// rows [r0, rb); plane columns [np, np rounded up to 8) zero. CB: the
// contribution-block chunk at c0 (W from k_big_ld), else the flush request.
template <bool CB>
__global__ __launch_bounds__(kLT) void k_big_pack(LdltDev d, const BigLd *__restrict__ states,
                                                  const BigPart *__restrict__ grid, int32_t c0, int32_t width) {
    const BigPart gr = grid[blockIdx.x];
    const BigLd B = states[gr.front];
    if (B.prec < 2) return;
    const FrontLd F = d.fronts[B.s];
    const int f = F.f;
    int p0, np, w0, r0, rb;
    if (CB) {
        const int c1 = min(B.k, c0 + width);
        if (c1 <= c0 || F.ne >= f) return;
        p0 = c0;
        np = c1 - c0;
        w0 = c0;
        r0 = F.ne;
        rb = f;
    } else {
        if (B.x_p1 <= B.x_p0) return;
        p0 = B.x_p0;
        np = B.x_p1 - B.x_p0;
        w0 = B.w_base;
        r0 = B.x_c0;
        rb = F.ne;
    }
    const bool split = B.prec == 3;
    const double *G = d.arena + F.fofs;
    const double *W = d.work + F.wofs;
    uint16_t *pl = d.xpl + 4 * F.wofs;
    const int64_t ps = static_cast<int64_t>(big_work(F.ne)) * f;
    const int ng = (np + 7) / 8;
    const int nr = f - r0;
    const int64_t tot = 2 * static_cast<int64_t>(ng) * nr;
    for (int64_t idx = static_cast<int64_t>(gr.part) * kLT + threadIdx.x; idx < tot;
         idx += static_cast<int64_t>(gr.parts) * kLT) {
        const int i = r0 + static_cast<int>(idx % nr);
        const int64_t q = idx / nr;
        const int g = static_cast<int>(q % ng);
        const int op = static_cast<int>(q / ng);  // 0: A, 1: B
        if (op == 1 && i >= rb) continue;
        const double *src = op == 0 ? G + static_cast<int64_t>(p0) * f : W + static_cast<int64_t>(p0 - w0) * f;
        v8bf_t hi, lo;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int c = 8 * g + u;
            const float x = c < np ? static_cast<float>(src[static_cast<int64_t>(c) * f + i]) : 0.f;
            hi[u] = static_cast<__bf16>(x);
            lo[u] = static_cast<__bf16>(x - static_cast<float>(hi[u]));
        }
        const int64_t o = static_cast<int64_t>(op) * 2 * ps + static_cast<int64_t>(g) * f * 8 + static_cast<int64_t>(i) * 8;
        *reinterpret_cast<v8bf_t *>(pl + o) = hi;
        if (split) *reinterpret_cast<v8bf_t *>(pl + o + ps) = lo;
    }
}

__global__ void k_big_finish(LdltDev d, const BigLd *__restrict__ states, int32_t nbig) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbig) return;
    const BigLd B = states[b];
    FrontLd &F = d.fronts[B.s];
    F.p = B.k;
    F.npos = B.cnt[0];
    F.nneg = B.cnt[1];
    F.nzero = B.cnt[2];
    F.flops = B.flops;
    F.stalls = B.stalls;
    F.pulls = B.pulls;
    F.rotated = B.rotated;
    F.searches = B.searches;
}

void launch_big_update(hipStream_t st, const LdltDev &d, const BigLd *states, const BigGrid &g,
                       const int32_t *nmode) {
    const dim3 nt(g.ntiles);
    if (d.xpl != nullptr && nmode[2] + nmode[3] > 0) k_big_pack<false><<<nt, kLT, 0, st>>>(d, states, g.tiles, 0, 0);
    if (nmode[0] > 0) k_big_update<0, false><<<nt, kLT, 0, st>>>(d, states, g.tiles);
    if (nmode[1] > 0) k_big_update<1, false><<<nt, kLT, 0, st>>>(d, states, g.tiles);
    // BF16 modes on planes: the flush is k_big_wide's
    if (d.xpl != nullptr) {
        if (nmode[2] > 0) k_big_update<2, true><<<nt, kLT, 0, st>>>(d, states, g.tiles);
        if (nmode[3] > 0) k_big_update<3, true><<<nt, kLT, 0, st>>>(d, states, g.tiles);
    } else {
        if (nmode[2] > 0) k_big_update<2, false><<<nt, kLT, 0, st>>>(d, states, g.tiles);
        if (nmode[3] > 0) k_big_update<3, false><<<nt, kLT, 0, st>>>(d, states, g.tiles);
    }
    if (d.xpl != nullptr) {
        if (nmode[2] > 0) k_big_wide<2, false><<<dim3(g.nwide), kWideThreads, 0, st>>>(d, states, g.wide, 0, 0);
        if (nmode[3] > 0) k_big_wide<3, false><<<dim3(g.nwide), kWideThreads, 0, st>>>(d, states, g.wide, 0, 0);
    }
}

void launch_big_round(hipStream_t st, const LdltDev &d, BigLd *states, BigLd *next, int32_t nbig, const BigGrid &g,
                      double u, double eff_small, double small_pivot, int32_t nb, double *gpart,
                      const int32_t *nmode) {
    const Prm prm{u, eff_small, small_pivot};
    k_big_region<<<dim3(nbig), kLT, 0, st>>>(d, states, gpart, nb);
    if (gpart != nullptr) k_big_group<<<dim3(g.nrows), kGroupRows, 0, st>>>(d, states, g.rows, gpart);
    k_big_panel<<<dim3(g.nrows), kLT, 0, st>>>(d, states, next, g.rows, prm, nb, gpart);
    launch_big_update(st, d, next, g, nmode);
}

void launch_big_cb(hipStream_t st, const LdltDev &d, const BigLd *states, const BigGrid &g, int32_t c0, int32_t width,
                   const int32_t *nmode, bool wide) {
    const dim3 nt(g.ntiles);
    k_big_ld<<<nt, kLT, 0, st>>>(d, states, g.tiles, c0, width, wide ? 1 : 0);
    if (wide) {
        // the BF16 modes' fronts on planes
        k_big_pack<true><<<nt, kLT, 0, st>>>(d, states, g.tiles, c0, width);
        if (nmode[2] > 0) k_big_wide<2, true><<<dim3(g.nwide), kWideThreads, 0, st>>>(d, states, g.wide, c0, width);
        if (nmode[3] > 0) k_big_wide<3, true><<<dim3(g.nwide), kWideThreads, 0, st>>>(d, states, g.wide, c0, width);
        return;
    }
    if (nmode[0] > 0) k_big_cbupdate<0><<<nt, kLT, 0, st>>>(d, states, g.tiles, c0, width);
    if (nmode[1] > 0) k_big_cbupdate<1><<<nt, kLT, 0, st>>>(d, states, g.tiles, c0, width);
    if (d.xpl == nullptr) {
        if (nmode[2] > 0) k_big_cbupdate<2><<<nt, kLT, 0, st>>>(d, states, g.tiles, c0, width);
        if (nmode[3] > 0) k_big_cbupdate<3><<<nt, kLT, 0, st>>>(d, states, g.tiles, c0, width);
    }
}

void launch_big_finish(hipStream_t st, const LdltDev &d, const BigLd *states, int32_t nbig) {
    if (nbig <= 0) return;
    k_big_finish<<<dim3((nbig + 63) / 64), 64, 0, st>>>(d, states, nbig);
}

// ---------------------------------------------------------------------------
// Rows of a level laid out on the host: the fronts' records, their row ids
// (children's delayed rows in child order, then the symbolic rows) and
// cleared tags; a workgroup per front.
__global__ __launch_bounds__(kLT) void k_ldlt_rows(LdltDev d, LdltAsm A, const FrontLd *__restrict__ patch,
                                                  const int32_t *__restrict__ ids) {
    const int s = ids[blockIdx.x];
    const FrontLd F = patch[blockIdx.x];
    const int tid = threadIdx.x;
    if (tid == 0) d.fronts[s] = F;
    int32_t *rows = d.rows + F.rofs;
    int dp = 0;
    for (int c = A.child_ptr[s]; c < A.child_ptr[s + 1]; ++c) {
        const FrontLd &K = d.fronts[A.child_idx[c]];
        const int del = K.delayed;
        const int32_t *crow = d.rows + K.rofs + K.p;
        for (int t = tid; t < del; t += kLT) rows[dp + t] = crow[t];
        dp += del;
    }
    const int32_t *sr = A.sym_rows + A.sym[s].rofs;
    for (int t = tid; t < F.f - F.nd; t += kLT) rows[F.nd + t] = sr[t];
    for (int t = tid; t < F.f; t += kLT) d.tags[F.rofs + t] = 0;
}

void launch_ldlt_rows(hipStream_t st, const LdltDev &d, const LdltAsm &A, const FrontLd *patch, const int32_t *ids,
                      int32_t nf) {
    for (int64_t o = 0; o < nf; o += kMaxLaunchGroups)
        k_ldlt_rows<<<dim3(static_cast<unsigned>(std::min<int64_t>(kMaxLaunchGroups, nf - o))), kLT, 0, st>>>(
            d, A, patch + o, ids + o);
}

// Assembly of the level's fronts (f x f squares in the arena, lower
// triangle), column by column, rows from the diagonal down: zero, original
// entries of the front's own pivot columns, then each child's CB column in
// child order; the CB of a child is the trailing (f_c - p_c) square of its
// own front, its first rows and columns the delayed ones. Which child columns
// meet in a column is known from the symbolic fronts (A.col_ptr), and where
// their rows go too: delayed ones to the child's place among the front's
// first nd rows, symbolic ones by their map, nd further. Fronts of up to
// kAsmWaveRows rows take a wavefront per column (its LDS accesses happen in
// its own order, no barriers), larger ones a workgroup per column in chunks
// of kAsmChunkL rows. Bound by memory, and by the chain of loads to a
// column's first entry: a column's loads go out four per thread at a time. 5.7 ms
// for 23348 columns of a root and sixteen fronts of 8900 (20 GB; 6.4 ms with
// per-column task lists made and uploaded by the host, 5 ms of host time).
constexpr int kAsmChunkL = 2048;

template <int NT>
__device__ void assemble_column(const LdltDev &d, const LdltAsm &A, int s, const FrontLd &F, int64_t srow, int c,
                                double *buf) {
    constexpr int kChunk = NT == 64 ? kAsmWaveRows : kAsmChunkL;
    constexpr int kCur = 16;  // children whose place in the column is kept
    __shared__ int cur[kCur];
    const int tid = NT == 64 ? threadIdx.x & 63 : threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int f = F.f, nd = F.nd;
    double *colp = d.arena + F.fofs + static_cast<int64_t>(c) * f;
    // the strict upper triangle is never read: left as it is
    const int oc = c - nd;  // symbolic column (own pivot column when in [0, psym))
    for (int r0 = c; r0 < f; r0 += kChunk) {
        const int r1 = min(f, r0 + kChunk);
        for (int r = r0 + tid; r < r1; r += NT) buf[r - r0] = 0.0;
        wg_sync<NT>();
        if (oc >= 0 && oc < F.psym) {
            const int j = F.col0 + oc;
            const int k0 = d.pcol_ptr[j], k1 = d.pcol_ptr[j + 1];
            for (int k = k0 + tid; k < k1; k += NT) {
                const int lr = nd + d.amap[k];
                if (lr >= r0 && lr < r1) buf[lr - r0] += d.av[k];
            }
            wg_sync<NT>();
        }
        // column jj of child ch, its delayed rows at dp; e: its number here
        const auto add = [&](int e, int ch, int jj, int dp) {
            const FrontLd &C = d.fronts[ch];
            const int cp = C.p, cf = C.f, q = cf - cp, del = C.delayed;
            // (without a branch: some valid address where no map is read)
            const int32_t *sm = q > del ? A.sym_cmap + A.sym_cmofs[ch] : A.sym_rows;
            const double *cbcol = d.arena + C.fofs + static_cast<int64_t>(cp + jj) * cf + cp;
            const auto place = [&](int ii) {
                const int m = sm[max(ii - del, 0)];
                return ii < del ? dp + ii : nd + m;
            };
            // first row at or past key: 64 places at a time
            const auto lbound = [&](int lo, int hi, int key) {
                while (lo < hi) {
                    const int step = (hi - lo + 63) >> 6;
                    const int i = min(lo + lane * step, hi - 1);
                    const int below = __popcll(__ballot(lo + lane * step < hi && place(i) < key));
                    if (below == 0) return lo;
                    hi = min(hi, lo + below * step);
                    lo += (below - 1) * step + 1;
                }
                return lo;
            };
            // the rows of the chunk: they follow the chunk before's, no more
            // than the chunk has places
            const int lo = r0 == c ? jj : (e < kCur ? cur[e] : lbound(jj, q, r0));
            const int hi = r1 == f ? q : lbound(lo, min(q, lo + r1 - r0), r1);
            for (int i0 = lo + tid; i0 < hi; i0 += 4 * NT) {
                int x[4];
                double v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int ii = min(i0 + u * NT, hi - 1);
                    x[u] = place(ii);
                    v[u] = cbcol[ii];
                }
                // (a column's places differ: read all, then write)
                double b[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) b[u] = buf[x[u] - r0];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (i0 + u * NT < hi) buf[x[u] - r0] = b[u] + v[u];
            }
            wg_sync<NT>();
            if (NT > 64 && e < kCur && tid == 0) cur[e] = hi;
        };
        if (oc >= 0) {
            const int e0 = A.col_ptr[srow + oc], e1 = A.col_ptr[srow + oc + 1];
            for (int e = e0; e < e1; ++e) {
                const ChildCol k = A.cc[e];
                add(e - e0, k.ch, k.jj + d.fronts[k.ch].delayed, 0);
            }
        } else {
            // a delayed column: one child's
            int dp = 0;
            for (int e = A.child_ptr[s]; e < A.child_ptr[s + 1]; ++e) {
                const int ch = A.child_idx[e];
                const int del = d.fronts[ch].delayed;
                if (c < dp + del) {
                    add(0, ch, c - dp, dp);
                    break;
                }
                dp += del;
            }
        }
        for (int r = r0 + tid; r < r1; r += NT) colp[r] = buf[r - r0];
        wg_sync<NT>();
    }
}

template <int NT>
__global__ __launch_bounds__(kLT) void k_ldlt_assemble(LdltDev d, LdltAsm A, const AsmPart *__restrict__ parts) {
    __shared__ double buf[NT == 64 ? kAsmWaveRows * (kLT / 64) : kAsmChunkL];
    constexpr int kW = kLT / NT, kPer = kAsmCols / kW;  // columns of a workgroup, workgroups of a part
    const AsmPart t = parts[blockIdx.x / kPer];
    const FrontLd F = d.fronts[t.s];
    const int w = threadIdx.x / NT;
    const int c = t.c + kW * (blockIdx.x % kPer) + w;
    if (c < F.f) assemble_column<NT>(d, A, t.s, F, A.sym[t.s].rofs, c, buf + w * kAsmWaveRows);
}

void launch_ldlt_assemble(hipStream_t st, const LdltDev &d, const LdltAsm &A, const AsmPart *parts, int64_t nwave,
                          int64_t nwg) {
    constexpr int64_t kMax = kMaxLaunchGroups / kAsmCols;
    const auto grid = [=](int64_t n, int64_t per) { return dim3(static_cast<unsigned>(std::min<int64_t>(kMax, n) * per)); };
    for (int64_t o = 0; o < nwave; o += kMax)
        k_ldlt_assemble<64><<<grid(nwave - o, kAsmCols / (kLT / 64)), kLT, 0, st>>>(d, A, parts + o);
    for (int64_t o = 0; o < nwg; o += kMax)
        k_ldlt_assemble<kLT><<<grid(nwg - o, kAsmCols), kLT, 0, st>>>(d, A, parts + nwave + o);
}

// ---------------------------------------------------------------------------
// Front epilogue (multifrontal_serial.cpp:892-945): a root's unaccepted
// eligible columns become zero pivots (tag 0); D^-1 per pivot as
// build_inline_dinv (solve_diag.cpp:49-123): kinds 1 / 2 / 0. The stored
// factor columns keep D on the diagonal, a 2x2 block's off-diagonal moved
// to the strict upper slot (c, c+1), zeros elsewhere above the diagonal
// and in a zero pivot's column; the square itself is left as it is (its
// trailing part is the contribution block).
__device__ __forceinline__ double stored_entry(const double *G, int ld, int c, int i, int8_t tg) {
    const bool up = i < c;
    const bool zero = up ? !(tg == -1 && i == c - 1) : (tg == 0 || (tg == 2 && i == c + 1));
    const double v = G[up ? static_cast<int64_t>(c > 0 ? c - 1 : 0) * ld + c : static_cast<int64_t>(c) * ld + i];
    return zero ? 0.0 : v;
}

// The epilogue of one front whose square (leading dimension ld) and pivot tags
// are at G and tags, in global memory or LDS; store: also write its stored
// factor columns, a column per wavefront at a time.
// LANES: at most 64 rows.
template <int NT = kLT, bool LANES = false>
__device__ void finish_front_wg(const LdltDev &d, FrontLd &F, const double *G, int ld, int8_t *tags, bool store) {
    __shared__ int n2;
    const int f = F.f;
    int p = F.p;
    const int tid = threadIdx.x;
    const bool root = F.root != 0;
    int ps = p;
    if (root && p < F.ne) {
        for (int c = p + tid; c < F.ne; c += NT) tags[c] = 0;
        ps = F.ne;
    }
    wg_sync<NT>();
    if (tid == 0) {
        F.pstore = ps;
        if (root && p < F.ne) F.nzero += F.ne - p;
        F.delayed = root ? 0 : F.ne - p;
        n2 = 0;
    }
    wg_sync<NT>();
    if constexpr (LANES) {
        const int c2 = __popcll(__ballot(tid < ps && tags[min(tid, f - 1)] == 2));
        if (tid == 0) F.n2x2 = c2;
    } else {
        int mine = 0;
        for (int c = tid; c < ps; c += NT) mine += tags[c] == 2;
        if (mine) atomicAdd(&n2, mine);
        wg_sync<NT>();
        if (tid == 0) F.n2x2 = n2;
    }
    for (int c = tid; c < ps; c += NT) {
        const double *Lc = G + static_cast<int64_t>(c) * ld;
        const int8_t tg = tags[c];
        const double d00 = Lc[c];
        double *dv = d.dinv + 3 * (F.dofs + c);
        int8_t *dk = d.dkind + F.dofs + c;
        if (tg == 2) {
            const double d10 = Lc[c + 1];
            const double d11 = G[static_cast<int64_t>(c + 1) * ld + c + 1];
            double sc = fabs(d00);
            if (sc < fabs(d10)) sc = fabs(d10);
            if (sc < fabs(d11)) sc = fabs(d11);
            double det_s = 0.0;
            if (isfinite(sc) && sc != 0.0) det_s = __dsub_rn(__dmul_rn(d00 / sc, d11 / sc), __dmul_rn(d10 / sc, d10 / sc));
            if (sc == 0.0 || !isfinite(det_s) || det_s == 0.0) {
                dv[0] = dv[1] = dv[2] = 0.0;
            } else {
                dv[0] = (d11 / sc) / det_s / sc;
                dv[1] = -(d10 / sc) / det_s / sc;
                dv[2] = (d00 / sc) / det_s / sc;
            }
            *dk = 2;
        } else if (tg == -1) {
            dv[0] = dv[1] = dv[2] = 0.0;
            *dk = 0;
        } else if (tg == 1) {
            dv[0] = (d00 == 0.0 || !isfinite(d00)) ? 0.0 : 1.0 / d00;
            dv[1] = dv[2] = 0.0;
            *dk = 1;
        } else {
            dv[0] = dv[1] = dv[2] = 0.0;
            *dk = 1;
        }
    }
    if (!store) return;
    double *O = d.fac + F.lofs;
    if constexpr (LANES) {
        // a row per lane, 8 columns' reads in flight
        const int lane = tid & 63, i = min(lane, f - 1);
        for (int c0 = 8 * (tid >> 6); c0 < ps; c0 += NT / 8) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = stored_entry(G, ld, min(c0 + u, ps - 1), i, tags[min(c0 + u, ps - 1)]);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c0 + u < ps && lane < f) O[static_cast<int64_t>(c0 + u) * f + lane] = v[u];
        }
        return;
    }
    for (int c = tid >> 6; c < ps; c += NT / 64) {
        const int8_t tg = tags[c];
        for (int i = tid & 63; i < f; i += 64) O[static_cast<int64_t>(c) * f + i] = stored_entry(G, ld, c, i, tg);
    }
}

__global__ __launch_bounds__(kLT) void k_ldlt_epilogue(LdltDev d, const int32_t *__restrict__ flist,
                                                       int32_t n_inline) {
    FrontLd &F = d.fronts[flist[blockIdx.x]];
    finish_front_wg(d, F, d.arena + F.fofs, F.f, d.tags + F.rofs, static_cast<int>(blockIdx.x) < n_inline);
}

// ---------------------------------------------------------------------------
// A front of at most 64 rows in LDS by NW wavefronts, the unblocked steps
// with a row per lane: columns of a fixed odd length kLd (a row's entries lie
// in different banks), kCU spare columns behind the last. What bounds a front
// is the number of instructions that its wavefronts go through one after the
// other. So
// - a wavefront takes kCU columns at a time, every lane and every column of
//   the group, without a test: what that leaves above the diagonal and in
//   the spare columns is read by nothing, a lane past the last row repeats
//   that row (tested lanes and columns were three times the instructions);
// - each wavefront scales the pivot columns for itself (lcol); the columns
//   are scaled in place after the step's barrier, by the first wavefront,
//   which also swaps rows: no other reads a finished column;
// - the pivot test is a ballot, the search looks at all candidates at once.
constexpr int kCU = 8;
constexpr int kLaneRows = 64;  // rows at most

struct LanePick {
    int cand, take, partner;
};
template <int NW>
struct LaneLds {
    double lcol[NW][2][kLaneRows + kCU];
    LanePick pick[NW];
};

// select_pivot's search over the candidates [k, limit): 2^lg lanes per
// candidate, each meeting its rows in increasing order, so the lanes of a
// candidate find what a sequential scan finds; the first candidate that a
// test accepts is the choice. (One candidate after the other by one
// wavefront took about 2500 cycles each, and badly pivoted fronts look at
// many.)
template <int NW>
__device__ __forceinline__ void lane_search(const FV &A, int k, int ne, const Prm &prm, LaneLds<NW> &S, int &kind,
                                            int &pa, int &pb) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int f = A.f, ld = A.ld;
    const int nc = ne - k;
    if (nc <= 0) return;
    // lanes per candidate: all candidates in one go, at most 8 lanes each
    int lg = 0;
    while (lg < 3 && nc << (lg + 1) <= 64 * NW) ++lg;
    const int g = 1 << lg, slice = lane & (g - 1);
    const int cl = w * (64 >> lg) + (lane >> lg);
    const bool live = cl < nc;
    const int cand = k + min(cl, nc - 1);
    // fn(row, |entry|) for the lane's rows of [lo, hi) in column c of the
    // symmetric matrix; NaN entries, row c and rows out of range as -1
    constexpr int kR = NW == 1 ? 8 : 4;
    const auto rows = [&](int c, int lo, int hi, auto &&fn) {
        for (int i0 = lo + slice; i0 - slice < hi; i0 += g * kR) {
            double v[kR];
#pragma unroll
            for (int u = 0; u < kR; ++u) {
                const int i = min(i0 + g * u, f - 1);
                v[u] = A.F[i < c ? i * ld + c : c * ld + i];
            }
#pragma unroll
            for (int u = 0; u < kR; ++u) {
                const int i = i0 + g * u;
                fn(i, i < hi && i != c ? fmax(fabs(v[u]), -1.0) : -1.0);
            }
        }
    };
    const double a_cand = fabs(A.at(cand, cand));
    // largest entry over the eligible rows [k, ne) other than cand (first
    // index on ties), the largest of the rest, the largest of rows [ne, f)
    double m1 = -1.0, m2 = 0.0, m_ext = 0.0;
    int r_best = -1;
    rows(cand, k, ne, [&](int i, double v) {
        m2 = fmax(m2, fmin(v, m1));
        if (v > m1) {
            m1 = v;
            r_best = i;
        }
    });
    rows(cand, ne, f, [&](int, double v) { m_ext = fmax(m_ext, v); });
    const auto join = [&](auto ctrl) {
        constexpr int C = decltype(ctrl)::value;
        const double n1 = dpp_d<C>(m1), n2 = dpp_d<C>(m2);
        const int rb = dpp_i<C>(r_best);
        m_ext = fmax(m_ext, dpp_d<C>(m_ext));
        m2 = fmax(fmax(m2, n2), fmin(m1, n1));
        if (better_first(n1, rb, m1, r_best)) {
            m1 = n1;
            r_best = rb;
        }
    };
    if (lg > 0) join(std::integral_constant<int, kDppXor1>{});
    if (lg > 1) join(std::integral_constant<int, kDppXor2>{});
    if (lg > 2) join(std::integral_constant<int, kDppHalfMirror>{});
    if (!(m1 > 0.0)) {
        m1 = 0.0;
        r_best = -1;
    }
    // 0: refused, 1: alone, 2: with its partner, 3: its partner alone
    int take = 0;
    bool weak = false;
    double weak_growth = 0.0;
    if (live && a_cand >= prm.eff_small && !(prm.u * m1 > a_cand) && !(prm.u * m_ext > a_cand)) {
        const double colmax = fmax(m1, m_ext);
        if (!(a_cand < kWeakPivotRatio * colmax)) {
            take = 1;
        } else {
            weak = true;
            weak_growth = colmax / a_cand;
        }
    }
    const bool pair = live && take == 0 && r_best >= k;
    if (weak && !pair) take = 1;
    const unsigned long long sure = __ballot(take != 0);
    // candidates before the first one taken already may still pair up
    if (__ballot(pair && (sure == 0 || lane < __builtin_ctzll(sure))) != 0) {
        // partner column: max excluding r_best, and excluding cand too
        const int r = pair ? r_best : cand;
        double om2 = 0.0, off1 = 0.0;
        rows(r, k, f, [&](int i, double v) {
            om2 = fmax(om2, v);
            off1 = fmax(off1, i != cand ? v : 0.0);
        });
        const auto join2 = [&](auto ctrl) {
            constexpr int C = decltype(ctrl)::value;
            om2 = fmax(om2, dpp_d<C>(om2));
            off1 = fmax(off1, dpp_d<C>(off1));
        };
        if (lg > 0) join2(std::integral_constant<int, kDppXor1>{});
        if (lg > 1) join2(std::integral_constant<int, kDppXor2>{});
        if (lg > 2) join2(std::integral_constant<int, kDppHalfMirror>{});
        if (pair) {
            double growth2;
            const bool ok2 = k + 1 < ne && two_by_two_ok(A, cand, r, fmax(m2, m_ext), off1, prm, growth2);
            const double a_r = fabs(A.at(r, r));
            if (ok2 && (!weak || growth2 < weak_growth)) take = 2;
            else if (weak) take = 1;
            else if (a_r >= prm.eff_small && (om2 == 0.0 || a_r >= prm.u * om2)) take = 3;
        }
    }
    const unsigned long long taken = __ballot(take != 0);
    LanePick P{-1, 0, -1};
    if (taken != 0) {
        const int l = __builtin_ctzll(taken);
        P.cand = __builtin_amdgcn_readlane(cand, l);
        P.take = __builtin_amdgcn_readlane(take, l);
        P.partner = __builtin_amdgcn_readlane(r_best, l);
    }
    if constexpr (NW > 1) {
        // the wavefronts' candidates follow each other
        if (lane == 0) S.pick[w] = P;
        __syncthreads();
        for (int v = NW - 1; v >= 0; --v)
            if (S.pick[v].take != 0) P = S.pick[v];
    }
    if (P.take == 0) return;
    kind = P.take == 2 ? 2 : 1;
    pa = P.take == 3 ? P.partner : P.cand;
    if (P.take == 2) pb = P.partner;
}

// select_pivot: the same choice as select_pivot_wg with limit = ne.
template <int NW>
__device__ __forceinline__ void lane_select(const FV &A, int k, int ne, const Prm &prm, LaneLds<NW> &S, int &kind,
                                            int &pa, int &pb) {
    const int lane = threadIdx.x & 63;
    const int f = A.f;
    kind = 0;
    pa = pb = -1;
    const double d0 = A.at(k, k), a0 = fabs(d0);
    if (prm.min_abs > 0.0) {
        // in order, no search: column k or nothing (then the static path)
        if (isfinite(d0) && a0 >= prm.min_abs) {
            kind = 1;
            pa = k;
        }
        return;
    }
    if (a0 >= prm.eff_small) {
        // u * colmax and kWeakPivotRatio * colmax are the largest of the
        // rows' products (rounding is monotone)
        const double v = fabs(A.at(min(lane, f - 1), k));
        if (__ballot(lane > k && lane < f && (prm.u * v > a0 || a0 < kWeakPivotRatio * v)) == 0) {
            kind = 1;
            pa = k;
            return;
        }
    }
    lane_search<NW>(A, k, ne, prm, S, kind, pa, pb);
}

// sym_swap by the first wavefront, a row per lane: the lane's pair of
// entries, itself twice where nothing moves
template <int NW>
__device__ __forceinline__ void lane_swap(const FV &A, int p, int q, int32_t *rows) {
    if (p == q) return;
    if (p > q) {
        const int t = p;
        p = q;
        q = t;
    }
    wg_sync<64 * NW>();
    if (threadIdx.x < 64) {
        const int m = min(static_cast<int>(threadIdx.x), A.f - 1), ld = A.ld;
        const int ia = m < p ? m * ld + p : p * ld + m;
        int ib = m == p ? q * ld + q : (m < q ? m * ld + q : q * ld + m);
        if (m == q) ib = ia;
        const double x = A.F[ia], y = A.F[ib];
        const int32_t rp = rows[p], rq = rows[q];
        wg_sync<64>();
        A.F[ia] = y;
        A.F[ib] = x;
        rows[p] = rq;
        rows[q] = rp;
    }
    wg_sync<64 * NW>();
}

// columns (k + np - 1, f) minus the pivot columns' products: lane i's
// unscaled entries u0 (u1), the scaled columns in l0 (l1)
template <int NW, int NP>
__device__ __forceinline__ void lane_update(const FV &A, int j1, int i, double u0, double u1, const double *l0,
                                            const double *l1) {
    for (int j0 = j1 + kCU * (threadIdx.x >> 6); j0 < A.f; j0 += kCU * NW) {
        double a[kCU], b[kCU], c[kCU];
#pragma unroll
        for (int e = 0; e < kCU; ++e) {
            a[e] = l0[j0 + e];
            if (NP == 2) b[e] = l1[j0 + e];
            c[e] = A.at(i, j0 + e);
        }
#pragma unroll
        for (int e = 0; e < kCU; ++e) {
            // eliminate_1x1 and eliminate_2x2 skip columns of zero factors
            const double v = NP == 2 ? __dsub_rn(c[e], __dadd_rn(__dmul_rn(u0, a[e]), __dmul_rn(u1, b[e])))
                                     : __dsub_rn(c[e], __dmul_rn(u0, a[e]));
            const bool skip = NP == 2 ? a[e] == 0.0 && b[e] == 0.0 : a[e] == 0.0;
            A.at(i, j0 + e) = skip ? c[e] : v;
        }
    }
}

// apply_pivot (ldlt_kernel.cpp:665-698); every thread keeps the counters
template <int NW>
__device__ __forceinline__ void lane_apply(const FV &A, int kind, int pa, int pb, int &k, int32_t *rows, int8_t *tags,
                                           const Prm &prm, LaneLds<NW> &S, int (&cnt)[3], double &flops,
                                           bool as_zero) {
    const int f = A.f;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = min(lane, f - 1);
    double *l0 = S.lcol[w][0], *l1 = S.lcol[w][1];
    if (kind == 1) {
        lane_swap<NW>(A, k, pa, rows);
        const double dk = A.at(k, k), u = A.at(i, k);
        if (as_zero) ++cnt[2];
        else inertia_1x1(dk, prm.eff_small, cnt);
        const double s = __dmul_rn(u, 1.0 / dk);
        l0[lane] = s;
        wg_sync<64>();
        lane_update<NW, 1>(A, k + 1, i, u, 0.0, l0, l1);
        wg_sync<64 * NW>();
        if (w == 0) {
            tags[k] = 1;
            A.at(i, k) = i > k ? s : u;
            wg_sync<64>();
        }
        const double rem = static_cast<double>(f - (k + 1));
        flops += rem + rem * (rem + 1.0);
        k += 1;
        return;
    }
    int partner = pb;
    if (pa != k) {
        lane_swap<NW>(A, k, pa, rows);
        if (partner == k) partner = pa;
    }
    if (partner != k + 1) lane_swap<NW>(A, k + 1, partner, rows);
    const double d00 = A.at(k, k), d10 = A.at(k + 1, k), d11 = A.at(k + 1, k + 1);
    const double u0 = A.at(i, k), u1 = A.at(i, k + 1);
    inertia_2x2(d00, d10, d11, prm.small_pivot, cnt);
    double s = fabs(d00);
    if (s < fabs(d10)) s = fabs(d10);
    if (s < fabs(d11)) s = fabs(d11);
    const double a = d00 / s, b = d10 / s, c = d11 / s;
    const double inv = 1.0 / __dmul_rn(__dsub_rn(__dmul_rn(a, c), __dmul_rn(b, b)), s);
    const double i00 = __dmul_rn(c, inv), i10 = __dmul_rn(-b, inv), i11 = __dmul_rn(a, inv);
    const double s0 = __dadd_rn(__dmul_rn(i00, u0), __dmul_rn(i10, u1));
    const double s1 = __dadd_rn(__dmul_rn(i10, u0), __dmul_rn(i11, u1));
    l0[lane] = s0;
    l1[lane] = s1;
    wg_sync<64>();
    lane_update<NW, 2>(A, k + 2, i, u0, u1, l0, l1);
    wg_sync<64 * NW>();
    if (w == 0) {
        tags[k] = 2;
        tags[k + 1] = -1;
        A.at(i, k) = i > k + 1 ? s0 : u0;
        A.at(i, k + 1) = i > k + 1 ? s1 : u1;
        wg_sync<64>();
    }
    const double rem = static_cast<double>(f - (k + 2));
    flops += 6.0 * rem + 2.0 * rem * (rem + 1.0);
    k += 2;
}

// ---------------------------------------------------------------------------
// Levels of small fronts laid out on the device.
//
// One wavefront's fronts have at most kDevWaveMax rows (their squares of 21 KB,
// 24 KB with the rest, let six workgroups share a CU), several wavefronts'
// kLaneRows.
constexpr int kDevWaveMax = 48;
template <int ROWS>
constexpr int lane_square = (ROWS + 1) * (ROWS + kCU);
constexpr int kDevKids = 8;   // children whose records are kept in LDS

struct DevChild {
    int64_t cb, rows, cmap;  // contribution block, its row ids, its symbolic rows' positions in the parent
    int32_t f, q, del;       // leading dimension, size, delayed columns
};

template <int FMAX>
struct DevLds {
    double Fs[FMAX == kDevWaveMax ? lane_square<kDevWaveMax> : FMAX * FMAX];
    int32_t rows[FMAX], cpos[FMAX], cptr[FMAX + 1];
    int8_t tags[FMAX];
    int cnt[3];
    LaneLds<FMAX == kDevWaveMax ? 1 : kLT / 64> lane;
    FrontLd F;
    DevChild kid[kDevKids];
    bool ok;
};

__device__ __forceinline__ DevChild dev_child(const LdltDev &d, const DevLevel &L, int ch) {
    const FrontLd &C = d.fronts[ch];
    DevChild K;
    K.cb = C.fofs + static_cast<int64_t>(C.p) * C.f + C.p;
    K.rows = C.rofs + C.p;
    K.cmap = L.sym_cmofs[ch];
    K.f = C.f;
    K.q = C.f - C.p;
    K.del = C.delayed;
    return K;
}

// Layout: a front's size follows from its children's results (nd = their
// delayed columns, f = nd + symbolic rows, ne = nd + symbolic pivots, as the
// host layout); its four offsets are bumps of the counters. A front larger
// than L.fmax, or a bump past the room, refuses the level (atomicMin of the
// level index); the level is then laid out again whole, from its children,
// which nothing of it has changed. By the first wavefront of the front's
// workgroup: a child per lane, the front's record and the first children's
// to LDS. laid: the record is there already, only the children are read
// (the second launch of a level, for its fronts above kDevWaveMax rows).
template <int FMAX>
__device__ void dev_layout(const DevLevel &L, const LdltDev &d, int s, int32_t lv, bool laid, DevLds<FMAX> &S) {
    const int lane = threadIdx.x & 63;
    // a refused level is left whole to the host (a front of it may be
    // refusing it right now: one reading decides for the workgroup)
    const unsigned long long refused = __atomic_load_n(&L.ctr[kDcLevel], __ATOMIC_RELAXED);
    const FrontDev Sy = L.sym[s];
    const int32_t parent = L.parent[s];
    const int c0 = L.child_ptr[s], nc = L.child_ptr[s + 1] - c0;
    int nd = 0;
    for (int o = 0; o < nc; o += 64) {
        int del = 0;
        if (o + lane < nc) {
            const DevChild K = dev_child(d, L, L.child_idx[c0 + o + lane]);
            if (o + lane < kDevKids) S.kid[o + lane] = K;
            del = K.del;
        }
        del += dpp_i<kDppXor1>(del);
        del += dpp_i<kDppXor2>(del);
        del += dpp_i<kDppHalfMirror>(del);
        del += dpp_i<kDppMirror>(del);
        for (int r = 0; r < 64; r += 16) nd += __builtin_amdgcn_readlane(del, r);
    }
    if (__ballot(refused <= static_cast<unsigned long long>(lv)) != 0) {
        if (lane == 0) S.ok = false;
        return;
    }
    if (laid) {
        if (lane == 0) {
            S.F = d.fronts[s];
            S.ok = S.F.f > kDevWaveMax;  // the others are done
        }
        return;
    }
    const long long f = nd + Sy.f, ne = nd + Sy.p;
    bool over = f > L.fmax;
    unsigned long long why = kDevWhySize;
    long long at = 0;
    if (!over) {
        // lane k bumps counter k
        static_assert(kDcSq == 0 && kDcFac == 1 && kDcRows == 2 && kDcDinv == 3, "counter order");
        const long long sz = lane == 0 ? (f * f + 63) / 64 * 64 : (lane == 1 ? f * ne : (lane == 2 ? f : ne));
        if (lane < 4) at = static_cast<long long>(atomicAdd(&L.ctr[lane], static_cast<unsigned long long>(sz)));
        over = __ballot(lane < 4 && at + sz > L.cap[lane & 3]) != 0;
        why = kDevWhyRoom;
    }
    const long long o1 = __shfl(at, 1, 64), o2 = __shfl(at, 2, 64), o3 = __shfl(at, 3, 64);
    if (lane == 0) {
        S.ok = !over;
        if (over) {
            atomicMin(&L.ctr[kDcLevel], static_cast<unsigned long long>(lv));
            atomicOr(&L.ctr[kDcWhy], why);
        }
        FrontLd F{};
        F.nd = nd;
        F.psym = Sy.p;
        F.col0 = Sy.col0;
        F.f = static_cast<int32_t>(f);
        F.ne = static_cast<int32_t>(ne);
        F.root = parent < 0 ? 1 : 0;
        F.dev = 1;
        F.fofs = at;
        F.lofs = o1;
        F.rofs = o2;
        F.dofs = o3;
        S.F = F;
    }
}

// One front by NT threads, the square in LDS: row list (children's delayed
// columns in child order, then the symbolic rows), assembly (zero, the
// front's original entries, each child's contribution block in child
// order: per entry the host layout's order of sums), the unblocked
// factorization, the epilogue, and the contribution block written back to
// the front's square for the parent. Row ids and tags stay in LDS until the
// end: a store to memory in a pivot step is waited for at its next barrier
// (about 2000 cycles a pivot).
// A chain is one workgroup's instructions and memory latencies in turn: a
// front of 24-31 rows (121-level stage chain) takes 21.1 us by four
// wavefronts, 28 by one (44 with row ids and tags in memory, a layout launch
// before and tested eliminations). 192 such chains of up to 401 levels: 8.9
// ms by four wavefronts, 11.6 by one.
// ROWS: the unblocked steps with a row per lane, a front of at most ROWS
// rows; 0: by workgroup reductions.
template <int NT, int ROWS, int FMAX>
__device__ void dev_front(const LdltDev &d, const DevLevel &L, int s, const Prm &prm, DevLds<FMAX> &S,
                          RedScratchT<NT> &rs) {
    double *Fs = S.Fs;
    const FrontDev Sy = L.sym[s];
    const FrontLd F = S.F;
    const int f = F.f, ne = F.ne, nd = F.nd;
    constexpr bool kLanes = ROWS > 0;
    static_assert(!kLanes || (ROWS <= kLaneRows && lane_square<ROWS> <= sizeof(S.Fs) / sizeof(double)), "fits");
    const int ld = kLanes ? ROWS + 1 : f;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    // original entries of the own pivot columns (one per row and column):
    // the columns' entries are contiguous; their pointers go to LDS once and
    // each lane finds the column of its entries there
    for (int t = tid; t <= F.psym; t += NT) S.cptr[t] = d.pcol_ptr[F.col0 + t];
    for (int t = tid; t < Sy.f; t += NT) S.rows[nd + t] = L.sym_rows[Sy.rofs + t];
    for (int idx = tid; idx < f * ld; idx += NT) Fs[idx] = 0.0;
    for (int t = tid; t < f; t += NT) S.tags[t] = 0;
    if (tid < 3) S.cnt[tid] = 0;
    wg_sync<NT>();
    {
        const int e0 = S.cptr[0], e1 = S.cptr[F.psym];
        constexpr int kE = 4;
        for (int e = e0 + tid; e < e1; e += kE * NT) {
            int r[kE], lo[kE], hi[kE];
            double a[kE];
#pragma unroll
            for (int u = 0; u < kE; ++u) {
                const int eu = min(e + u * NT, e1 - 1);
                r[u] = d.amap[eu];
                a[u] = d.av[eu];
                lo[u] = 0;
                hi[u] = F.psym;
            }
            // the column oc with cptr[oc] <= e < cptr[oc + 1]
            for (int w2 = F.psym; w2 > 1; w2 = (w2 + 1) >> 1)
#pragma unroll
                for (int u = 0; u < kE; ++u) {
                    const int mid = (lo[u] + hi[u]) >> 1;
                    if (S.cptr[mid] <= min(e + u * NT, e1 - 1)) lo[u] = mid;
                    else hi[u] = mid;
                }
#pragma unroll
            for (int u = 0; u < kE; ++u)
                if (e + u * NT < e1) Fs[(nd + lo[u]) * ld + nd + r[u]] += a[u];
        }
    }
    wg_sync<NT>();
    int dp = 0;
    const int c0 = L.child_ptr[s], nc = L.child_ptr[s + 1] - c0;
    for (int c = 0; c < nc; ++c) {
        const DevChild C = c < kDevKids ? S.kid[c] : dev_child(d, L, L.child_idx[c0 + c]);
        const int q = C.q, del = C.del;
        for (int ii = tid; ii < q; ii += NT) S.cpos[ii] = ii < del ? dp + ii : nd + L.sym_cmap[C.cmap + ii - del];
        for (int t = tid; t < del; t += NT) S.rows[dp + t] = d.rows[C.rows + t];
        wg_sync<NT>();
        // lane = row of the child's block; each wavefront's columns kG at
        // a time, their loads in flight together
        const double *cb = d.arena + C.cb;
        constexpr int kG = NT == 64 ? 16 : 8, kW = NT / 64;
        for (int i0 = 0; i0 < q; i0 += 64) {
            const int ii = i0 + lane, ic = min(ii, q - 1);
            const int pi = S.cpos[ic];
            for (int j0 = w; j0 < min(q, i0 + 64); j0 += kG * kW) {
                double v[kG], x[kG];
                int at[kG];
#pragma unroll
                for (int u = 0; u < kG; ++u) {
                    const int jj = min(j0 + kW * u, q - 1);
                    v[u] = cb[static_cast<int64_t>(jj) * C.f + max(ic, jj)];
                    at[u] = S.cpos[jj] * ld + pi;
                }
#pragma unroll
                for (int u = 0; u < kG; ++u) x[u] = Fs[at[u]];
#pragma unroll
                for (int u = 0; u < kG; ++u)
                    if (j0 + kW * u <= ii && ii < q) Fs[at[u]] = x[u] + v[u];
            }
        }
        wg_sync<NT>();
        dp += del;
    }
    FV A{Fs, ld, f};
    int k = 0;
    int own[3] = {0, 0, 0};
    int *cnt = kLanes ? own : S.cnt;
    double flops = 0.0;
    Prm fp;
    const double sp = front_prm(prm, F, fp);
    int nstatic = 0;
    double growth = 0.0;
    while (k < ne) {
        int kind, pa, pb;
        if constexpr (kLanes) lane_select<NT / 64>(A, k, ne, fp, S.lane, kind, pa, pb);
        else select_pivot_wg(A, k, ne, ne, fp, rs, kind, pa, pb);
        bool az = false;
        if (kind == 0) {
            if (!(sp > 0.0)) break;
            int raised;
            pa = force_static_wg(A, k, ne, sp, fp, rs, raised, nstatic, growth);
            kind = 1;
            az = static_as_zero(raised, fp, F);
        }
        if constexpr (kLanes) lane_apply<NT / 64>(A, kind, pa, pb, k, S.rows, S.tags, fp, S.lane, own, flops, az);
        else apply_pivot_wg<NT>(A, kind, pa, pb, k, S.rows, S.tags, nullptr, 0, 0, f, fp, cnt, flops, 0, az);
    }
    wg_sync<NT>();
    if (tid == 0) {
        S.F.p = k;
        S.F.npos = cnt[0];
        S.F.nneg = cnt[1];
        S.F.nzero = cnt[2];
        S.F.flops = flops;
        S.F.nstatic = nstatic;
        S.F.growth = growth;  // stalls to searches stay 0: unblocked, no panels
    }
    // contribution block (lower part of columns [k, f)) for the parent
    if (!F.root) {
        double *G = d.arena + F.fofs;
        if constexpr (kLanes) {
            const int i = min(lane, f - 1);
            for (int j0 = k + 8 * w; j0 < f; j0 += NT / 8) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = Fs[min(j0 + u, f - 1) * ld + i];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (lane >= j0 + u && lane < f) G[static_cast<int64_t>(j0 + u) * f + lane] = v[u];
            }
        } else {
            for (int j = k + w; j < f; j += NT / 64)
                for (int i = j + lane; i < f; i += 64) G[static_cast<int64_t>(j) * f + i] = Fs[j * ld + i];
        }
    }
    wg_sync<NT>();
    finish_front_wg<NT, kLanes>(d, S.F, Fs, ld, S.tags, true);
    wg_sync<NT>();
    if (tid == 0) d.fronts[s] = S.F;
    for (int t = tid; t < f; t += NT) {
        d.rows[F.rofs + t] = S.rows[t];
        d.tags[F.rofs + t] = S.tags[t];
    }
}

// A level's fronts, one workgroup each.
// CLASS 0 (64 threads): layout, then the fronts of at most 48 rows (one
// wavefront and 25 KB of LDS: many fronts per CU); a larger one keeps its
// layout for the CLASS 1 launch (256 threads). CLASS 2 (256 threads): layout
// and any front, four wavefronts each: where a level has few fronts
// (kDevOneLaunch), and for a whole band of levels, each workgroup going up its
// chain of fronts. CLASS 3: layout and workgroup reductions whatever the size.
template <int CLASS>
__global__ __launch_bounds__(CLASS == 0 ? 64 : kLT) void k_dev_fronts(LdltDev d, DevLevel L,
                                                                     const int32_t *__restrict__ flist, int32_t lv,
                                                                     Prm prm) {
    __shared__ DevLds<CLASS == 0 ? kDevWaveMax : kDevFrontMax> S;
    __shared__ RedScratchT<CLASS == 0 ? 64 : kLT> rs;
    for (int s = flist[blockIdx.x];;) {
        if (threadIdx.x < 64) dev_layout(L, d, s, lv, CLASS == 1, S);
        __syncthreads();
        if (!S.ok) return;
        if constexpr (CLASS == 0) {
            if (S.F.f <= kDevWaveMax) dev_front<64, kDevWaveMax>(d, L, s, prm, S, rs);
            else if (threadIdx.x == 0) d.fronts[s] = S.F;
        } else if (CLASS != 3 && S.F.f <= kLaneRows) {
            dev_front<kLT, kLaneRows>(d, L, s, prm, S, rs);
        } else {
            dev_front<kLT, 0>(d, L, s, prm, S, rs);
        }
        if constexpr (CLASS != 2) return;
        // on to the parent: this front is its only child in the band
        s = L.parent[s];
        if (s < 0) return;
        lv = L.lev[s];
        if (lv >= L.end) return;
        __syncthreads();
    }
}

void launch_dev_fronts(hipStream_t st, const LdltDev &d, const DevLevel &L, const int32_t *flist, int32_t nf,
                       int32_t lv, double u, double eff_small, double small_pivot, const StaticPrm &S, bool wave) {
    if (nf <= 0) return;
    Prm prm{u, eff_small, small_pivot, 0.0, S};
    for (int64_t o = 0; o < nf; o += kMaxLaunchGroups) {
        const dim3 grid(static_cast<unsigned>(std::min<int64_t>(kMaxLaunchGroups, nf - o)));
        if (!wave) {
            // every front on kLT threads (tuning)
            k_dev_fronts<3><<<grid, kLT, 0, st>>>(d, L, flist + o, lv, prm);
        } else if (nf <= kDevOneLaunch) {
            k_dev_fronts<2><<<grid, kLT, 0, st>>>(d, L, flist + o, lv, prm);
        } else {
            k_dev_fronts<0><<<grid, 64, 0, st>>>(d, L, flist + o, lv, prm);
            k_dev_fronts<1><<<grid, kLT, 0, st>>>(d, L, flist + o, lv, prm);
        }
    }
}

// Stored columns of large fronts: grid (column stride, fronts).
__global__ __launch_bounds__(kLT) void k_ldlt_store(LdltDev d, const int32_t *__restrict__ flist) {
    const FrontLd F = d.fronts[flist[blockIdx.y]];
    const int f = F.f;
    const int8_t *tags = d.tags + F.rofs;
    const double *G = d.arena + F.fofs;
    double *O = d.fac + F.lofs;
    for (int c = blockIdx.x; c < F.pstore; c += gridDim.x) {
        const int8_t tg = tags[c];
        for (int i = threadIdx.x; i < f; i += kLT) O[static_cast<int64_t>(c) * f + i] = stored_entry(G, f, c, i, tg);
    }
}

__global__ void k_front_gather(const FrontLd *fronts, FrontLd *out, const int32_t *ids, int32_t np) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np) out[i] = fronts[ids[i]];
}

void launch_front_gather(hipStream_t st, const FrontLd *fronts, FrontLd *out, const int32_t *ids, int32_t np) {
    if (np <= 0) return;
    k_front_gather<<<dim3((np + 127) / 128), 128, 0, st>>>(fronts, out, ids, np);
}

void launch_ldlt_epilogue(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, int32_t n_inline) {
    if (nf <= 0) return;
    for (int64_t o = 0; o < nf; o += kMaxLaunchGroups) {
        const int64_t m = std::min<int64_t>(kMaxLaunchGroups, nf - o);
        const int32_t inl = static_cast<int32_t>(std::max<int64_t>(0, std::min<int64_t>(m, n_inline - o)));
        k_ldlt_epilogue<<<dim3(static_cast<unsigned>(m)), kLT, 0, st>>>(d, flist + o, inl);
    }
}

void launch_ldlt_store(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, int32_t max_cols) {
    if (nf <= 0 || max_cols <= 0) return;
    for (int32_t o = 0; o < nf; o += kStoreFronts) {
        const StoreGrid g = store_grid(nf - o, max_cols);
        k_ldlt_store<<<dim3(g.per, g.fronts), kLT, 0, st>>>(d, flist + o);
    }
}

// ---------------------------------------------------------------------------
// D^-1 step of the LDL^T solve (apply_dinv, solve_backward.cpp:156-173): per pivot,
// kind 1 scales, kind 2 applies the 2x2 inverse, kind 0 (second column of a
// 2x2) is skipped. The L sweeps are in kernels_solve.hip. gridDim.y
// workgroups share a front's pivots (a front of 14,000 pivots is 200 us of
// scattered reads for one).
__global__ void k_ldlt_diag(LdltDev d, const int32_t *__restrict__ flist, int32_t nf, double *__restrict__ y,
                            int32_t n, int32_t nrhs) {
    const int fi = blockIdx.x;
    if (fi >= nf) return;
    const FrontLd F = d.fronts[flist[fi]];
    const int32_t *rows = d.rows + F.rofs;
    for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < F.pstore; c += gridDim.y * blockDim.x) {
        const int8_t kd = d.dkind[F.dofs + c];
        const double *dv = d.dinv + 3 * (F.dofs + c);
        for (int r = 0; r < nrhs; ++r) {
            double *yr = y + static_cast<int64_t>(r) * n;
            if (kd == 1) {
                yr[rows[c]] *= dv[0];
            } else if (kd == 2) {
                const double r0 = yr[rows[c]], r1 = yr[rows[c + 1]];
                yr[rows[c]] = dv[0] * r0 + dv[1] * r1;
                yr[rows[c + 1]] = dv[1] * r0 + dv[2] * r1;
            }
        }
    }
}

// The diagonal-only solve job (solve_diag, solve_diag.cpp:236-261, over
// the entries process_front pushes, multifrontal_serial.cpp:921-942): D
// read from the stored columns (d on the diagonal, a 2x2 block's
// off-diagonal in slot (c, c+1)); a 1x1 pivot divides (a zero or
// non-finite d, and a root's zero pivot, give 0), a 2x2 block takes
// solve_2x2_scaled (pivoting.cpp:30-62).
__global__ void k_ldlt_diag_div(LdltDev d, const int32_t *__restrict__ flist, int32_t nf, double *__restrict__ y,
                                int32_t n, int32_t nrhs) {
    const int fi = blockIdx.x;
    if (fi >= nf) return;
    const FrontLd F = d.fronts[flist[fi]];
    const int32_t *rows = d.rows + F.rofs;
    const int8_t *tags = d.tags + F.rofs;
    const double *L = d.fac + F.lofs;
    const int64_t f = F.f;
    for (int c = threadIdx.x; c < F.pstore; c += blockDim.x) {
        const int8_t tg = tags[c];
        if (tg == -1) continue;
        const double d00 = L[c * f + c];
        for (int r = 0; r < nrhs; ++r) {
            double *yr = y + static_cast<int64_t>(r) * n;
            if (tg != 2) {
                yr[rows[c]] = (d00 == 0.0 || !isfinite(d00)) ? 0.0 : yr[rows[c]] / d00;
                continue;
            }
            const double d10 = L[(c + 1) * f + c], d11 = L[(c + 1) * f + c + 1];
            const double x0 = yr[rows[c]], x1 = yr[rows[c + 1]];
            double s = fabs(d00);
            if (s < fabs(d10)) s = fabs(d10);
            if (s < fabs(d11)) s = fabs(d11);
            double y0 = 0.0, y1 = 0.0;
            if (isfinite(s) && s != 0.0) {
                const double a = d00 / s, b = d10 / s, cc = d11 / s;
                const double det_s = a * cc - b * b;
                if (isfinite(det_s) && det_s != 0.0) {
                    if (!isfinite(x0) || !isfinite(x1)) {
                        y0 = x0;
                        y1 = x1;
                    } else {
                        const double rs = fmax(fabs(x0), fabs(x1));
                        if (rs != 0.0) {
                            const double r0 = x0 / rs, r1 = x1 / rs;
                            const double u0 = (cc * r0 - b * r1) / det_s;
                            const double u1 = (-b * r0 + a * r1) / det_s;
                            const double ratio = rs / s;
                            y0 = u0 * ratio;
                            y1 = u1 * ratio;
                        }
                    }
                }
            }
            yr[rows[c]] = y0;
            yr[rows[c + 1]] = y1;
        }
    }
}

void launch_ldlt_diag_div(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, double *y, int32_t n,
                          int32_t nrhs) {
    if (nf <= 0) return;
    for (int64_t o = 0; o < nf; o += kMaxLaunchGroups) {
        const int32_t m = static_cast<int32_t>(std::min<int64_t>(kMaxLaunchGroups, nf - o));
        k_ldlt_diag_div<<<dim3(static_cast<unsigned>(m)), 64, 0, st>>>(d, flist + o, m, y, n, nrhs);
    }
}

void launch_ldlt_diag(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, int32_t max_p, double *y,
                      int32_t n, int32_t nrhs) {
    if (nf <= 0) return;
    const int32_t threads = max_p > 64 ? kLT : 64;
    const int32_t parts = std::max(1, std::min(16, (max_p + threads - 1) / threads));
    for (int64_t o = 0; o < nf; o += kMaxLaunchGroups) {
        const int32_t m = static_cast<int32_t>(std::min<int64_t>(kMaxLaunchGroups, nf - o));
        k_ldlt_diag<<<dim3(static_cast<unsigned>(m), parts), threads, 0, st>>>(d, flist + o, m, y, n, nrhs);
    }
}

}  // namespace smfgpu
