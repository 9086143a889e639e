// A15: forward and backward sweeps of the SPD factor, level by level.
//
// A front's pivot columns are solved in blocks of kSB = 128 (two 64-pivot
// diagonal blocks whose inverses the Cholesky kernel stored in their strict
// upper triangles). One launch per step covers every front of a level:
// in step j one workgroup per front (the "triangle" item) applies block
// j-1's update to block j's rows and solves block j, while the other items
// apply block j-1's update to the rest of the front (forward: 64-row chunks;
// backward: 64-column chunks). Kernel boundaries order the steps, no
// workgroup waits for another. Reference: solve.cpp:858-1075 (the sweeps),
// solve_forward.cpp / solve_backward.cpp (per-front dense steps).
//
// y is the permuted right-hand side block, n x nrhs (ld n). Rows of a front
// below its pivots belong to ancestors that sibling fronts of the same level
// also update: those forward updates are atomic adds.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "smfgpu_internal.hpp"
#include "smfgpu_ldlt.hpp"

namespace smfgpu {
namespace {

constexpr int kSB = 128;        // pivot columns per step
constexpr int kSD = 64;         // diagonal block (stored inverse)
constexpr int kSThreads = 512;  // eight waves

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2du __attribute__((ext_vector_type(2), aligned(8)));  // two rows of a column (8-byte aligned)

// a of the lane's half plus b of the other's: lanes of the first half (ROW 32:
// of the wavefront, 16: of each pair of rows of 16 lanes) get a + a of their
// partner lane, the others b + b of theirs
template <int ROW>
__device__ __forceinline__ double swap_add(double a, double b) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    const unsigned al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b), bh = __double2hiint(b);
    u2 l, h;
    if constexpr (ROW == 32) {
        l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
        h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    } else {
        l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
        h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    }
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}

// Products of 16 rows or columns of L (lane lr = lane % 16) with the
// right-hand sides, the sum's index split over the four rows of lanes lk =
// lane / 16. More than four right-hand sides: FP64 MFMA 16x16x4, the
// right-hand sides as the 16 rows of the result (A operand: lane lr holds
// right-hand side lr, lanes past NR zeros); one takes 64 entries of L for up
// to 16 of them in 64 cycles, 19 TB/s over the chip, so a sweep stays bound by
// reading L, once for all 16. Up to four: FMAs (an item's 512 MFMAs are 3.4
// us of its CU, the FMAs of one right-hand side 0.3) and a sum over lk.
template <int NR>
struct Acc {
    double a[NR];
    __device__ __forceinline__ Acc() {
#pragma unroll
        for (int r = 0; r < NR; ++r) a[r] = 0.0;
    }
    __device__ __forceinline__ void add(const double (*v)[NR], int t, double l) {
#pragma unroll
        for (int r = 0; r < NR; ++r) a[r] += v[t][r] * l;
    }
    __device__ __forceinline__ void put(double (*part)[NR], int col) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const double s = swap_add<32>(a[r], a[r]);
            const double q = swap_add<16>(s, s);
            if ((threadIdx.x & 48) == 0) part[col][r] = q;
        }
    }
    __device__ __forceinline__ bool finite() const {
        bool f = true;
#pragma unroll
        for (int r = 0; r < NR; ++r) f = f && isfinite(a[r]);
        return f;
    }
};
template <>
struct Acc<16> {
    v4d a = {0.0, 0.0, 0.0, 0.0};
    __device__ __forceinline__ void add(const double (*v)[16], int t, double l) {
        a = __builtin_amdgcn_mfma_f64_16x16x4f64(v[t][threadIdx.x & 15], l, a, 0, 0, 0);
    }
    // accumulator: right-hand side 4 v + lk, column lr
    __device__ __forceinline__ void put(double (*part)[16], int col) {
        const int lk = (threadIdx.x & 63) >> 4;
#pragma unroll
        for (int v = 0; v < 4; ++v) part[col][4 * v + lk] = a[v];
    }
    __device__ __forceinline__ bool finite() const {
        return isfinite(a[0]) && isfinite(a[1]) && isfinite(a[2]) && isfinite(a[3]);
    }
};

// The triangle's three 64 x 64 blocks, element (t = rl, c = g + 8 e): BLK 0:
// upper part of the first diagonal block (t <= c: inverse rows and the
// diagonal), 1: rows 64.. of the block below it, 2: second diagonal block.
// The first one needed is read before the item's update, the others after it
// (their 32 registers would leave one workgroup per CU).
// Guarded loads are unconditional loads from clamped (in-front) addresses
// times a 0 / 1 mask: a select around a load lets the compiler move the
// load into a branch that waits for every load in flight.
__device__ __forceinline__ double masked(double v, bool keep) { return v * (keep ? 1.0 : 0.0); }

template <int BLK>
__device__ __forceinline__ void tri_load(double (&R)[8], const double *Lb, int f, int tk, int tkb, int rl, int g) {
    const int na = min(kSD, tkb), nb = tkb - kSD;
    const int nr = BLK == 0 ? na : max(nb, 1), nc = BLK == 2 ? max(nb, 1) : na;
    const int row = tk + min((BLK > 0 && nb > 0 ? kSD : 0) + min(rl, nr - 1), tkb - 1);
    const int col = tk + (BLK == 2 && nb > 0 ? kSD : 0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int c = g + 8 * e;
        R[e] = masked(Lb[static_cast<int64_t>(col + min(c, nc - 1)) * f + row],
                      BLK == 1 ? rl < nb && c < na : rl <= c && c < (BLK == 0 ? na : nb));
    }
}

__device__ __forceinline__ void put_block(double (*Dg)[kSD + 1], const double (&v)[8], int rl, int g) {
#pragma unroll
    for (int e = 0; e < 8; ++e) Dg[rl][g + 8 * e] = v[e];
}

// 1 / d: the hardware estimate (better than 2^-20), a third-order step and
// one Newton step for the last bit
__device__ __forceinline__ double recip(double d) {
    double y = __builtin_amdgcn_rcp(d);
    double e = fma(-d, y, 1.0);
    y = fma(y, fma(e, e, e), y);
    e = fma(-d, y, 1.0);
    return fma(y, e, y);
}

// a diagonal block: the inverse's transpose, its diagonal 1 / L_cc (columns
// past n zero)
__device__ __forceinline__ void put_diag(double (*Dg)[kSD + 1], const double (&v)[8], int rl, int g, int n) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int c = g + 8 * e;
        Dg[rl][c] = (rl == c && c < n) ? recip(v[e]) : v[e];
    }
}

// part[h][i][r] = sum over half h of k of D(i, k) v[k][r], D(i, k) =
// TR ? Dg[k][i] : Dg[i][k], 64 x 64; wave w: 16 of i (w % 4), half w / 4.
// TRI: a diagonal block, D zero for k > i (TR) or k < i. Its zeros times a
// value that is not finite would be NaN in entries that do not depend on it:
// a wavefront that meets one takes those sums again over the triangle only.
template <int NR, bool TR, bool TRI>
__device__ __forceinline__ void block_times(const double (*Dg)[kSD + 1], const double (*v)[NR],
                                            double (*part)[kSD][NR]) {
    const int lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4, w = threadIdx.x >> 6;
    const int i = 16 * (w & 3) + lr, h = w >> 2;
    Acc<NR> acc;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
        const int k = 32 * h + 4 * kk + lk;
        acc.add(v, k, TR ? Dg[k][i] : Dg[i][k]);
    }
    acc.put(part[h], i);
    if (TRI && __ballot(!acc.finite()) != 0) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        for (int r = lk; r < NR; r += 4) {
            if (isfinite(part[h][i][r])) continue;
            double s = 0.0;
            for (int k = 32 * h; k < 32 * h + 32; ++k)
                if (TR ? k <= i : k >= i) s += (TR ? Dg[k][i] : Dg[i][k]) * v[k][r];
            part[h][i][r] = s;
        }
    }
}

// Forward update of rows [lo, hi): y[row] -= sum_{t < kb} L[row][k + t] zs[t]
// (zs zero past kb). Rows in the triangle [tk, tk + tkb) go to yb (LDS),
// other own pivot rows in place, ancestor rows by atomic add. ROWS rows at a
// time: a lane takes two rows (16-byte loads), the waves 32 rows each and
// shares of the kSB columns.
template <int NR, int ROWS>
__device__ void fwd_update(const double *Lb, const int32_t *frows, int f, int p, int col0, int k, int kb, int lo,
                           int hi, const double (*zs)[NR], double (*part)[kSD][NR], double (*yb)[NR], int tk, int tkb,
                           double *y, int n, int nrhs) {
    constexpr int kTiles = ROWS / 32, kSplit = 8 / kTiles, kCols = kSB / kSplit;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4, w = tid >> 6;
    const int pt = w % kTiles, c0 = w / kTiles * kCols;
    double (*pp)[NR] = reinterpret_cast<double (*)[NR]>(part);  // kSplit x ROWS
    for (int r0 = lo; r0 < hi; r0 += ROWS) {
        const int row = r0 + 32 * pt + 2 * lr;
        const double *Lr = Lb + static_cast<int64_t>(k) * f + min(row, f - 2);
        Acc<NR> acc0, acc1;
        v2du l[kCols / 4];
#pragma unroll
        for (int kk = 0; kk < kCols / 4; ++kk) {
            if (c0 + 4 * kk >= kb) break;
            l[kk] = *reinterpret_cast<const v2du *>(Lr + static_cast<int64_t>(min(c0 + 4 * kk + lk, kb - 1)) * f);
        }
#pragma unroll
        for (int kk = 0; kk < kCols / 4; ++kk) {
            if (c0 + 4 * kk >= kb) break;
            const double l0 = row > f - 2 ? l[kk][1] : l[kk][0];  // the front's last row alone
            acc0.add(zs, c0 + 4 * kk + lk, l0);
            acc1.add(zs, c0 + 4 * kk + lk, l[kk][1]);
        }
        double (*q)[NR] = pp + w / kTiles * ROWS + 32 * pt;
        acc0.put(q, 2 * lr);
        acc1.put(q, 2 * lr + 1);
        __syncthreads();
        for (int e = tid; e < ROWS * NR; e += kSThreads) {
            const int rr = e % ROWS, r = e / ROWS;
            const int i = r0 + rr;
            if (i < hi && r < nrhs) {
                double sum = 0.0;
#pragma unroll
                for (int g = 0; g < kSplit; ++g) sum += pp[g * ROWS + rr][r];
                if (i >= tk && i < tk + tkb) {
                    yb[i - tk][r] = y[col0 + i + static_cast<int64_t>(r) * n] - sum;
                } else if (i < p) {
                    y[col0 + i + static_cast<int64_t>(r) * n] -= sum;
                } else {
                    unsafeAtomicAdd(&y[static_cast<int64_t>(frows[i]) + static_cast<int64_t>(r) * n], -sum);
                }
            }
        }
        __syncthreads();
    }
}

template <int NR>
struct FwdLds {
    double Dg[kSD][kSD + 1];
    double zs[kSB][NR];
    double yb[kSB][NR];
    double part[4][kSD][NR];  // partial sums: 4 x 64 or 2 x 128 rows, 2 x 64 in the triangles
};

// out[i][r] = base[i][r] - (or without base: =) part[0] + part[1], i < n
template <int NR, bool SUB>
__device__ __forceinline__ void add_halves(double (*out)[NR], const double (*part)[kSD][NR], int n) {
    for (int e = threadIdx.x; e < kSD * NR; e += kSThreads) {
        const int i = e / NR, r = e % NR;
        const double v = part[0][i][r] + part[1][i][r];
        if (SUB) {
            if (i < n) out[i][r] -= v;
        } else {
            out[i][r] = i < n ? v : 0.0;
        }
    }
}

template <int NR>
__device__ void fwd_item(const DevPtrs &d, const SolveItem &it, double *__restrict__ y, int32_t n, int32_t nrhs,
                         FwdLds<NR> &S) {
    auto &Dg = S.Dg;
    auto &zs = S.zs;
    auto &yb = S.yb;
    auto &part = S.part;
    const FrontDev F = d.fronts[it.s];
    const int f = F.f, p = F.p;
    const double *Lb = d.L + F.lofs;
    const int32_t *frows = d.rows + F.rofs;
    const int tid = threadIdx.x, rl = tid & 63, g = tid >> 6;
    double Ra[8], Rb[8], Rc[8];
    if (it.tkb > 0) tri_load<0>(Ra, Lb, f, it.tk, it.tkb, rl, g);
    for (int idx = tid; idx < kSB * NR; idx += kSThreads) {
        const int t = idx % kSB, r = idx / kSB;
        zs[t][r] = (t < it.kb && r < nrhs) ? y[F.col0 + it.k + t + static_cast<int64_t>(r) * n] : 0.0;
        if (it.tkb > 0) yb[t][r] = (it.kb == 0 && t < it.tkb && r < nrhs) ? y[F.col0 + it.tk + t + static_cast<int64_t>(r) * n] : 0.0;
    }
    __syncthreads();
    if (it.kb > 0)
        fwd_update<NR, 64>(Lb, frows, f, p, F.col0, it.k, it.kb, it.a0, it.a1, zs, part, yb, it.tk, it.tkb, y, n, nrhs);
    if (it.tkb <= 0) return;
    // the triangle: z_a = inv(L_a) y_a; y_b -= L_ba z_a; z_b = inv(L_b) y_b
    const int na = min(kSD, it.tkb), nb = it.tkb - kSD;
    if (nb > 0) {
        tri_load<1>(Rb, Lb, f, it.tk, it.tkb, rl, g);
        tri_load<2>(Rc, Lb, f, it.tk, it.tkb, rl, g);
    }
    put_diag(Dg, Ra, rl, g, na);
    __syncthreads();
    block_times<NR, true, true>(Dg, yb, part);
    __syncthreads();
    add_halves<NR, false>(zs, part, na);
    if (nb > 0) put_block(Dg, Rb, rl, g);
    __syncthreads();
    if (nb > 0) {
        block_times<NR, false, false>(Dg, zs, part);
        __syncthreads();
        add_halves<NR, true>(yb + kSD, part, nb);
        put_diag(Dg, Rc, rl, g, nb);
        __syncthreads();
        block_times<NR, true, true>(Dg, yb + kSD, part);
        __syncthreads();
        add_halves<NR, false>(zs + kSD, part, nb);
        __syncthreads();
    } else if (it.kb > 0) {
        // zs past the block still holds the block before
        for (int e = tid; e < kSD * NR; e += kSThreads) zs[kSD + e / NR][e % NR] = 0.0;
        __syncthreads();
    }
    // zs now holds z of the whole block, zeros past tkb
    for (int idx = tid; idx < it.tkb * nrhs; idx += kSThreads) {
        const int t = idx % it.tkb, r = idx / it.tkb;
        y[F.col0 + it.tk + t + static_cast<int64_t>(r) * n] = zs[t][r];
    }
    if (it.flags & 2)  // the rows below the last block, by this workgroup
        fwd_update<NR, 128>(Lb, frows, f, p, F.col0, it.tk, it.tkb, it.tk + it.tkb, f, zs, part, yb, -1, 0, y, n, nrhs);
}

template <int NR>
__global__ __launch_bounds__(kSThreads, NR == 1 ? 4 : 1) void k_fwd_step(DevPtrs d, const SolveItem *__restrict__ items,
                                                       double *__restrict__ y, int32_t n, int32_t nrhs) {
    __shared__ FwdLds<NR> S;
    fwd_item<NR>(d, items[blockIdx.x], y, n, nrhs, S);
}

template <int NR>
constexpr int kXs = NR > 4 ? 256 : kSolveSeg;  // rows of x a backward update stages at a time

// Backward update of columns [c0, c1): y[col0 + c] -= sum_{i in [r0, r1)}
// L[i][c] x_i, x_i = y[col0 + i] for own pivot rows, y[rows[i]] else. 64
// columns at a time: wave w takes 16 of them (w % 4) and half of the rows; a
// lane takes 4 consecutive rows of its column (two 16-byte loads, whole cache
// lines across the lanes), 64 rows of loads in flight and the next 64 behind
// them. Columns of the triangle go to v (LDS).
template <int NR>
__device__ void bwd_update(const double *Lb, const int32_t *frows, int f, int p, int col0, int r0, int r1, int c0,
                           int c1, bool atomic, double (*xs)[NR], double (*part)[kSD][NR], double (*v)[NR], int tk,
                           int tkb, double *y, int n, int nrhs) {
    constexpr int kX = kXs<NR>, kU = 4;
    const int tid = threadIdx.x;
    const int lane = tid & 63, lr = lane & 15, lk = lane >> 4, w = tid >> 6, h = w >> 2;
    const int nr = r1 - r0;
    for (int cb = c0; cb < c1; cb += 64) {
        const int c = min(cb + 16 * (w & 3) + lr, c1 - 1);
        const double *Lc = Lb + static_cast<int64_t>(c) * f + r0;
        Acc<NR> acc;
        for (int s0 = 0; s0 < nr; s0 += kX) {
            const int ns = min(kX, nr - s0);
            const int half = (ns + 31) / 32 * 16;  // rows of a wave, a multiple of 16
            const int g0 = s0 + h * half, ge = min(s0 + ns, g0 + half);
            v2du l[2][kU][2];
            const auto load = [&](v2du (&q)[kU][2], int g) {
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const int i = g + 16 * u + 4 * lk;
                    if (g + 16 * u >= ge) break;
                    if (g + 16 * u + 16 <= nr) {
                        q[u][0] = *reinterpret_cast<const v2du *>(Lc + i);
                        q[u][1] = *reinterpret_cast<const v2du *>(Lc + i + 2);
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j) q[u][j >> 1][j & 1] = Lc[min(i + j, nr - 1)];
                    }
                }
            };
            const auto mul = [&](const v2du (&q)[kU][2], int g) {
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    if (g + 16 * u >= ge) break;
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc.add(xs, g - s0 + 16 * u + 4 * lk + j, q[u][j >> 1][j & 1]);
                }
            };
            load(l[0], g0);
            if (cb > c0 || s0 > 0) __syncthreads();
            if (cb == c0 || nr > kX) {
                for (int idx = tid; idx < kX * NR; idx += kSThreads) {
                    const int i = idx % kX, r = idx / kX;
                    double xv = 0.0;
                    if (i < ns && r < nrhs) {
                        const int row = r0 + s0 + i;
                        const int64_t gi = row < p ? static_cast<int64_t>(col0 + row) : static_cast<int64_t>(frows[row]);
                        xv = y[gi + static_cast<int64_t>(r) * n];
                    }
                    xs[i][r] = xv;
                }
            }
            __syncthreads();
            for (int g = g0; g < ge; g += 32 * kU) {
                load(l[1], g + 16 * kU);
                mul(l[0], g);
                if (g + 16 * kU >= ge) break;
                load(l[0], g + 32 * kU);
                mul(l[1], g + 16 * kU);
            }
        }
        acc.put(part[h], 16 * (w & 3) + lr);
        __syncthreads();
        for (int e = tid; e < kSD * NR; e += kSThreads) {
            const int cc = cb + e % kSD, r = e / kSD;
            if (cc < c1 && r < nrhs) {
                const double s = part[0][e % kSD][r] + part[1][e % kSD][r];
                double *dst = &y[col0 + cc + static_cast<int64_t>(r) * n];
                if (cc >= tk && cc < tk + tkb) v[cc - tk][r] = *dst - s;
                else if (atomic) unsafeAtomicAdd(dst, -s);
                else *dst -= s;
            }
        }
    }
    __syncthreads();
}

template <int NR>
struct BwdLds {
    double Dg[kSD][kSD + 1];
    double xs[kXs<NR>][NR];
    double v[kSB][NR];
    double xo[kSB][NR];
    double part[2][kSD][NR];
};

template <int NR>
__device__ void bwd_item(const DevPtrs &d, const SolveItem &it, double *__restrict__ y, int32_t n, int32_t nrhs,
                         BwdLds<NR> &S) {
    auto &Dg = S.Dg;
    auto &xs = S.xs;
    auto &v = S.v;
    auto &xo = S.xo;
    auto &part = S.part;
    const FrontDev F = d.fronts[it.s];
    const int f = F.f, p = F.p;
    const double *Lb = d.L + F.lofs;
    const int32_t *frows = d.rows + F.rofs;
    const int tid = threadIdx.x, rl = tid & 63, g = tid >> 6;
    double Ra[8], Rb[8], Rc[8];
    const int na = min(kSD, it.tkb), nb = it.tkb - kSD;
    if (it.tkb > 0) {
        if (nb > 0) tri_load<2>(Rc, Lb, f, it.tk, it.tkb, rl, g);
        else tri_load<0>(Ra, Lb, f, it.tk, it.tkb, rl, g);
        for (int idx = tid; idx < kSB * NR; idx += kSThreads) {
            const int t = idx % kSB, r = idx / kSB;
            v[t][r] = (it.kb == 0 && t < it.tkb && r < nrhs) ? y[F.col0 + it.tk + t + static_cast<int64_t>(r) * n] : 0.0;
        }
        __syncthreads();
    }
    if (it.kb > 0)
        bwd_update<NR>(Lb, frows, f, p, F.col0, it.k, it.k + it.kb, it.a0, it.a1, (it.flags & 1) != 0, xs, part, v,
                       it.tk, it.tkb, y, n, nrhs);
    if (it.tkb <= 0) return;
    // the triangle, second diagonal block first:
    // x_b = inv(L_b)^T v_b; v_a -= L_ba^T x_b; x_a = inv(L_a)^T v_a
    if (nb > 0) {
        tri_load<1>(Rb, Lb, f, it.tk, it.tkb, rl, g);
        tri_load<0>(Ra, Lb, f, it.tk, it.tkb, rl, g);
        put_diag(Dg, Rc, rl, g, nb);
        __syncthreads();
        block_times<NR, false, true>(Dg, v + kSD, part);
        __syncthreads();
        add_halves<NR, false>(xo + kSD, part, nb);
        put_block(Dg, Rb, rl, g);  // Dg[t][c] = L_ba[t][c]
        __syncthreads();
        block_times<NR, true, false>(Dg, xo + kSD, part);
        __syncthreads();
        add_halves<NR, true>(v, part, na);
    }
    put_diag(Dg, Ra, rl, g, na);
    __syncthreads();
    block_times<NR, false, true>(Dg, v, part);
    __syncthreads();
    add_halves<NR, false>(xo, part, na);
    __syncthreads();
    for (int idx = tid; idx < it.tkb * nrhs; idx += kSThreads) {
        const int t = idx % it.tkb, r = idx / it.tkb;
        y[F.col0 + it.tk + t + static_cast<int64_t>(r) * n] = xo[t][r];
    }
}

template <int NR>
__global__ __launch_bounds__(kSThreads, NR == 1 ? 4 : 1) void k_bwd_step(DevPtrs d, const SolveItem *__restrict__ items,
                                                       double *__restrict__ y, int32_t n, int32_t nrhs) {
    __shared__ BwdLds<NR> S;
    bwd_item<NR>(d, items[blockIdx.x], y, n, nrhs, S);
}

// ---------------------------------------------------------------------------
// One launch per sweep: a workgroup per item, each taking a ticket (its
// item, in sweep order) when it starts; before an item of step t runs,
// every item of step t - 1 has finished (its counter reached the step's
// item count): the ordering the per-step launches get from kernel
// boundaries, without the launches. Tickets go out in increasing order to
// running workgroups and an item waits only on items with smaller tickets,
// so the waits end however the workgroups are dispatched. There is no loop
// around the item: every wave meets the same barriers in the same order.
// Writes to y are released with a device-scope fence before the counter
// moves and acquired after the wait. A wait that runs out (never expected)
// sets err and lets every later wait through, so the launch always ends.
constexpr int64_t kSweepSpin = int64_t{1} << 18;

__device__ __forceinline__ void sweep_wait(int32_t *cnt, int32_t target, int32_t *err) {
    for (int64_t spin = 0; __hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target; ++spin) {
        if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
        if (spin > kSweepSpin) {
            atomicExch(err, 1);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    __threadfence();
}

template <int NR, bool FWD>
__global__ __launch_bounds__(kSThreads) void k_sweep(DevPtrs d, const SolveItem *__restrict__ items,
                                                    const int32_t *__restrict__ step_of,
                                                    const int32_t *__restrict__ step_cnt, int32_t *ctr, int32_t *err,
                                                    double *__restrict__ y, int32_t n, int32_t nrhs) {
    __shared__ typename std::conditional<FWD, FwdLds<NR>, BwdLds<NR>>::type S;
    __shared__ int32_t s_item;
    if (threadIdx.x == 0) {
        const int32_t i = atomicAdd(&ctr[0], 1);  // < the grid size, the item count
        const int32_t t = step_of[i];
        if (t > 0) sweep_wait(&ctr[t], step_cnt[t - 1], err);  // counter of step t - 1
        s_item = i;
    }
    __syncthreads();
    const int32_t i = __builtin_amdgcn_readfirstlane(s_item);
    const SolveItem it = items[i];
    if constexpr (FWD) fwd_item<NR>(d, it, y, n, nrhs, S);
    else bwd_item<NR>(d, it, y, n, nrhs, S);
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        atomicAdd(&ctr[1 + step_of[i]], 1);
    }
}

__global__ void k_zero_i32(int32_t *p, int32_t n) {
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}


// ---------------------------------------------------------------------------
// Sweeps of an LDL^T factor (unit L with D on the stored diagonal; the D^-1
// step runs between them): steps of kLS pivots (a large front's dense
// triangle costs two launches per kLS pivots), each solved by its triangle
// item as up to four 64-pivot sub-blocks. Items: forward triangle {tk, tkb:
// this block; kItemFused: then the rows [a0, a1) below it}, forward chunk
// {rows [a0, a1), update by the block [k, k+kb)}, backward chunk {columns
// [a0, a1), contributions of rows [k, k+kb); kItemAtomic}, backward
// triangle {tk, tkb; k, kb: rows below the pivots whose contributions it
// takes itself}. Triangles of more than kLB pivots (kItemWide) have kernels
// of their own. Every item takes NR right-hand sides at a time, so L is read
// once for all of them.
constexpr int kLB = 64;    // sub-block: a unit triangle in LDS, substituted by one wave
constexpr int kLS = 256;   // pivots per step
constexpr int kLThreads = 256;
constexpr int kLWide = 512;   // threads of a wide triangle item
constexpr int kLSeg = 512;    // rows of a backward tail item

__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Sum over the wavefront of M (8 or 16) values per lane. Each halving step
// exchanges half of the values with a partner lane, so the M sums end up in
// different lanes: value e(lane) = the lane's top log2(M) bits. 32: the two
// halves of the wavefront (v_permlane32_swap: {a.lo, b.lo}, {a.hi, b.hi}),
// 16: rows of 16 lanes, 8 and 4: inside a row (rotation by 8, mirror of 8
// lanes); the lanes that share e are then added.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, false),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, false));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppRor8 = 0x128;
template <int M>
__device__ __forceinline__ double wave_sums(double (&v)[M]) {
    static_assert(M == 8 || M == 16, "values per lane");
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < M / 2; ++k) v[k] = swap_add<32>(v[k], v[k + M / 2]);
#pragma unroll
    for (int k = 0; k < M / 4; ++k) v[k] = swap_add<16>(v[k], v[k + M / 4]);
#pragma unroll
    for (int k = 0; k < M / 8; ++k) {
        const double keep = lane & 8 ? v[k + M / 8] : v[k], give = lane & 8 ? v[k] : v[k + M / 8];
        v[k] = keep + dpp_move<kDppRor8>(give);
    }
    double t = v[0];
    if constexpr (M == 16) {
        const double keep = lane & 4 ? v[1] : v[0], give = lane & 4 ? v[0] : v[1];
        t = keep + dpp_move<kDppHalfMirror>(give);
    }
    t += dpp_move<kDppXor1>(t);
    t += dpp_move<kDppXor2>(t);
    if constexpr (M == 8) t += dpp_move<kDppHalfMirror>(t);
    return t;
}
template <int M>
__device__ __forceinline__ int wave_sums_index() {
    return (threadIdx.x & 63) >> (M == 16 ? 2 : 3);
}

// sum_{c < kb} L(i, k + c) xs[r][c] (kb <= kLS) for row i = r0 + (tid & 63)
// (< r1), wave w taking the columns [w q, (w + 1) q), q = ceil(kb / 4),
// in order; the total ((w0 + w1) + (w2 + w3)) lands in part[r][0][row]. The
// loads go out 16 columns at a time (clamped addresses, masked values), so
// a workgroup waits on a column group's latency, not each column's.
template <int NR, int XS>
__device__ __forceinline__ void rows_times_block(const double *L, int f, int k, int kb, int r0, int r1,
                                                 const double (*xs)[XS], double (*part)[4][kLB]) {
    constexpr int kG = 16;
    const int row = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = min(r0 + row, r1 - 1);
    const int q = (kb + 3) >> 2;
    const int cb = w * q, ce = min(kb, cb + q);
    double acc[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = 0.0;
    if (ce > cb) {
        const double *Lc = L + static_cast<int64_t>(k) * f + i;
        for (int c = cb; c < ce; c += kG) {
            double lv[kG];
#pragma unroll
            for (int j = 0; j < kG; ++j) lv[j] = Lc[static_cast<int64_t>(min(c + j, ce - 1)) * f];
#pragma unroll
            for (int j = 0; j < kG; ++j)
                if (c + j < ce) {
#pragma unroll
                    for (int r = 0; r < NR; ++r) acc[r] += lv[j] * xs[r][c + j];
                }
        }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) part[r][w][row] = acc[r];
    __syncthreads();
    if (w < NR) {
        double(*p)[kLB] = part[w];
        p[0][row] = (p[0][row] + p[1][row]) + (p[2][row] + p[3][row]);
    }
    __syncthreads();
}

// the unit triangle of sub-block [c0, c0 + nc): T[c][l] = L(c0 + l, c0 + c), l > c
__device__ __forceinline__ void load_unit_triangle(const double *L, int f, int c0, int nc, double (*T)[kLB + 1]) {
    for (int e = threadIdx.x; e < kLB * kLB; e += kLThreads) {
        const int c = e >> 6, l = e & 63;
        T[c][l] = (c < nc && l < nc && l > c) ? L[static_cast<int64_t>(c0 + c) * f + c0 + l] : 0.0;
    }
}

// One wavefront's substitution with the unit triangle T (zero on and above
// the diagonal and past the block): lane l holds y_l (0 past the block). Bound
// by the 64 dependent steps; T's values are read 16 steps ahead of the chain,
// the solved value is broadcast through scalar registers (through LDS a step
// took about 150 cycles, here about 30). T's zeros times a value that is not
// finite would be NaN in the lanes solved before it: such a block is solved
// again with a test on the lane.
__device__ __forceinline__ double unit_forward(const double (*T)[kLB + 1], double y0, int nc) {
    const int l = threadIdx.x & 63;
    double yv = y0;
#pragma unroll
    for (int c0 = 0; c0 < kLB; c0 += 16) {
        if (c0 >= nc) break;
        double t[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = T[c0 + u][l];
#pragma unroll
        for (int u = 0; u < 16; ++u) yv -= t[u] * lane_value(yv, c0 + u);
    }
    if (__ballot(!isfinite(yv)) != 0) {
        yv = y0;
        for (int c = 0; c < min(nc, kLB); ++c) {
            const double v = lane_value(yv, c);
            if (l > c && l < nc) yv -= T[c][l] * v;
        }
    }
    return yv;
}
__device__ __forceinline__ double unit_backward(const double (*T)[kLB + 1], double y0, int nc) {
    const int l = threadIdx.x & 63;
    double yv = y0;
#pragma unroll
    for (int c0 = kLB - 16; c0 >= 0; c0 -= 16) {
        if (c0 >= nc) continue;
        double t[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = T[l][c0 + u];
#pragma unroll
        for (int u = 15; u >= 0; --u) yv -= t[u] * lane_value(yv, c0 + u);
    }
    if (__ballot(!isfinite(yv)) != 0) {
        yv = y0;
        for (int c = min(nc, kLB) - 1; c > 0; --c) {
            const double v = lane_value(yv, c);
            if (l < c) yv -= T[l][c] * v;
        }
    }
    return yv;
}

template <int NR>
__global__ __launch_bounds__(kLThreads) void k_ldlt_fwd_step(LdltDev d, const SolveItem *__restrict__ items,
                                                            double *__restrict__ y, int32_t n, int32_t nrhs) {
    static_assert(NR <= kLThreads / 64, "one wave per right-hand side in the triangles");
    __shared__ double xs[NR][kLS];  // the block solved (in the step before, or here)
    __shared__ double part[NR][4][kLB];
    __shared__ double T[kLB][kLB + 1];
    const SolveItem it = items[blockIdx.x];
    const FrontLd F = d.fronts[it.s];
    const int f = F.f, p = F.pstore;
    const double *L = d.fac + F.lofs;
    const int32_t *rows = d.rows + F.rofs;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const bool tri = (it.flags & kItemTri) != 0;
    if (tri) load_unit_triangle(L, f, it.tk, it.tkb, T);
    for (int r0 = 0; r0 < nrhs; r0 += NR) {
        const int nr = min(NR, nrhs - r0);
        double *yr = y + static_cast<int64_t>(r0) * n;
        if (tri) {
            __syncthreads();  // the triangle in LDS
            if (w < nr) {
                double *yw = yr + static_cast<int64_t>(w) * n;
                const bool in = lane < it.tkb;
                const int32_t g = rows[it.tk + min(lane, it.tkb - 1)];
                const double yv = unit_forward(T, in ? yw[g] : 0.0, it.tkb);
                if (in) yw[g] = yv;
                xs[w][lane] = in ? yv : 0.0;
            } else if (w < NR) {
                xs[w][lane] = 0.0;
            }
            __syncthreads();
            if (it.flags & kItemFused) {
                // the rows below, with the block just solved
                for (int rb = it.a0; rb < it.a1; rb += kLB) {
                    const int re = min(rb + kLB, it.a1);
                    rows_times_block<NR>(L, f, it.tk, it.tkb, rb, re, xs, part);
                    if (w < nr && rb + lane < re)
                        unsafeAtomicAdd(&yr[static_cast<int64_t>(w) * n + rows[rb + lane]], -part[w][0][lane]);
                    __syncthreads();
                }
            }
        } else {
            for (int e = tid; e < NR * kLS; e += kLThreads) {
                const int r = e / kLS, t = e % kLS;
                xs[r][t] = (r < nr && t < it.kb) ? yr[static_cast<int64_t>(r) * n + rows[it.k + t]] : 0.0;
            }
            __syncthreads();
            rows_times_block<NR>(L, f, it.k, it.kb, it.a0, it.a1, xs, part);
            const int i = it.a0 + lane;
            if (w < nr && i < it.a1) {
                double *dst = &yr[static_cast<int64_t>(w) * n + rows[i]];
                if (i >= p) unsafeAtomicAdd(dst, -part[w][0][lane]);
                else *dst -= part[w][0][lane];
            }
            __syncthreads();
        }
    }
}

// Wide triangles (kLB < tkb <= kLS), one workgroup of 512: the whole
// triangle is read into registers up front (its ten 64 x 64 blocks, eight
// columns of each per wave, lane = row: one memory latency instead of one
// per sub-block), then per sub-block one wave per right-hand side
// substitutes with the block's unit triangle from LDS and every wave applies
// its columns to the rows below. Bound by the substitution chains and the
// read of the triangle by one CU. One step of a 43,245-row KKT's sweeps took
// 54 us forward and 67 us backward with the blocks read in turn and the
// right-hand sides one after the other.
constexpr int kTriBlocks = 10;
__host__ __device__ constexpr int tri_block(int i, int j) { return i * (i + 1) / 2 + j; }

__device__ __forceinline__ void load_wide_triangle(const double *L, int f, int tk, int tkb,
                                                   double (&R)[kTriBlocks][8]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (64 * i >= tkb) break;
        const int row = tk + min(64 * i + lane, tkb - 1);
#pragma unroll
        for (int j = 0; j <= i; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                R[tri_block(i, j)][e] = L[static_cast<int64_t>(tk + min(64 * j + 8 * w + e, tkb - 1)) * f + row];
    }
}
// sub-block j's unit triangle to LDS
__device__ __forceinline__ void put_unit_triangle(const double (&v)[8], int nc, double (*T)[kLB + 1]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int e = 0; e < 8; ++e) T[8 * w + e][lane] = (lane > 8 * w + e && lane < nc) ? v[e] : 0.0;
}

template <int NR>
__global__ __launch_bounds__(kLWide) void k_ldlt_fwd_tri(LdltDev d, const SolveItem *__restrict__ items,
                                                         double *__restrict__ y, int32_t n, int32_t nrhs) {
    __shared__ double T[kLB][kLB + 1];
    __shared__ double Y[NR][kLS];
    __shared__ double part[NR][8][kLS - kLB];
    const SolveItem it = items[blockIdx.x];
    const FrontLd F = d.fronts[it.s];
    const int f = F.f, tk = it.tk, tkb = it.tkb;
    const int32_t *rows = d.rows + F.rofs + tk;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    double R[kTriBlocks][8];
    load_wide_triangle(d.fac + F.lofs, f, tk, tkb, R);
    for (int r0 = 0; r0 < nrhs; r0 += NR) {
        const int nr = min(NR, nrhs - r0);
        double *yr = y + static_cast<int64_t>(r0) * n;
        for (int e = tid; e < NR * kLS; e += kLWide) {
            const int r = e / kLS, t = e % kLS;
            Y[r][t] = (r < nr && t < tkb) ? yr[static_cast<int64_t>(r) * n + rows[t]] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (64 * j >= tkb) break;
            put_unit_triangle(R[tri_block(j, j)], tkb - 64 * j, T);
            __syncthreads();
            if (w < nr) {
                const double yv = unit_forward(T, Y[w][64 * j + lane], tkb - 64 * j);
                Y[w][64 * j + lane] = yv;
                if (64 * j + lane < tkb) yr[static_cast<int64_t>(w) * n + rows[64 * j + lane]] = yv;
            }
            __syncthreads();
            if (j == 3 || 64 * (j + 1) >= tkb) break;
            const int nbelow = tkb - 64 * (j + 1);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                double x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = Y[r][64 * j + 8 * w + e];
#pragma unroll
                for (int i = j + 1; i < 4; ++i) {
                    if (64 * i >= tkb) break;
                    double acc = 0.0;
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc += R[tri_block(i, j)][e] * x[e];
                    part[r][w][64 * (i - j - 1) + lane] = acc;
                }
            }
            __syncthreads();
            for (int e = tid; e < NR * (kLS - kLB); e += kLWide) {
                const int r = e / (kLS - kLB), t = e % (kLS - kLB);
                if (t < nbelow) {
                    double acc = 0.0;
#pragma unroll
                    for (int g = 0; g < 8; ++g) acc += part[r][g][t];
                    Y[r][64 * (j + 1) + t] -= acc;
                }
            }
        }
        __syncthreads();
    }
}

template <int NR>
__global__ __launch_bounds__(kLWide) void k_ldlt_bwd_tri(LdltDev d, const SolveItem *__restrict__ items,
                                                         double *__restrict__ y, int32_t n, int32_t nrhs) {
    __shared__ double T[kLB][kLB + 1];
    __shared__ double X[NR][kLS];
    __shared__ double U[NR][kLB];
    const SolveItem it = items[blockIdx.x];
    const FrontLd F = d.fronts[it.s];
    const int f = F.f, tk = it.tk, tkb = it.tkb;
    const int32_t *rows = d.rows + F.rofs + tk;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    double R[kTriBlocks][8];
    load_wide_triangle(d.fac + F.lofs, f, tk, tkb, R);
    for (int r0 = 0; r0 < nrhs; r0 += NR) {
        const int nr = min(NR, nrhs - r0);
        double *yr = y + static_cast<int64_t>(r0) * n;
        for (int e = tid; e < NR * kLS; e += kLWide) {
            const int r = e / kLS, t = e % kLS;
            X[r][t] = (r < nr && t < tkb) ? yr[static_cast<int64_t>(r) * n + rows[t]] : 0.0;
        }
#pragma unroll
        for (int j = 3; j >= 0; --j) {
            if (64 * j >= tkb) continue;
            __syncthreads();  // the sub-block solved before (or X) in LDS, its triangle read
            const bool below = j < 3 && 64 * (j + 1) < tkb;
            put_unit_triangle(R[tri_block(j, j)], tkb - 64 * j, T);
            if (below) {
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    double acc[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[e] = 0.0;
#pragma unroll
                    for (int i = j + 1; i < 4; ++i) {
                        if (64 * i >= tkb) break;
                        const double x = X[r][64 * i + lane];
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc[e] += R[tri_block(i, j)][e] * x;
                    }
                    const double v = wave_sums<8>(acc);
                    if ((lane & 7) == 0) U[r][8 * w + wave_sums_index<8>()] = v;
                }
            }
            __syncthreads();
            if (w < nr) {
                double yv = X[w][64 * j + lane];
                if (below) yv -= U[w][lane];
                yv = unit_backward(T, yv, tkb - 64 * j);
                X[w][64 * j + lane] = yv;
                if (64 * j + lane < tkb) yr[static_cast<int64_t>(w) * n + rows[64 * j + lane]] = yv;
            }
        }
        __syncthreads();
    }
}

// Backward contributions of rows [k, k + kb) (values xs) to the columns
// [c0, c1): each wave takes 16 columns at a time, its lanes the rows t =
// lane + 64 m in order, the 16 columns' loads of one m in flight together;
// out(r, c, sum) once per column and right-hand side.
template <int NR, class Out>
__device__ __forceinline__ void cols_times_rows(const double *L, int f, int k, int kb, int c0, int c1,
                                                const double (*xs)[kLSeg], Out &&out) {
    constexpr int kG = 16;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int cb = c0 + w * kG; cb < c1; cb += 4 * kG) {
        double acc[NR][kG];
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int j = 0; j < kG; ++j) acc[r][j] = 0.0;
        for (int t0 = 0; t0 < kb; t0 += 64) {
            const int t = min(t0 + lane, kb - 1);
            double lv[kG];
#pragma unroll
            for (int j = 0; j < kG; ++j) lv[j] = L[static_cast<int64_t>(min(cb + j, c1 - 1)) * f + k + t];
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const double xv = t0 + lane < kb ? xs[r][t] : 0.0;
#pragma unroll
                for (int j = 0; j < kG; ++j) acc[r][j] += lv[j] * xv;
            }
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const double v = wave_sums<kG>(acc[r]);
            const int c = cb + wave_sums_index<kG>();
            if ((lane & 3) == 0 && c < c1) out(r, c, v);
        }
    }
}

template <int NR>
__global__ __launch_bounds__(kLThreads) void k_ldlt_bwd_step(LdltDev d, const SolveItem *__restrict__ items,
                                                            double *__restrict__ y, int32_t n, int32_t nrhs) {
    static_assert(NR <= kLThreads / 64, "one wave per right-hand side in the triangles");
    __shared__ double xs[NR][kLSeg];
    __shared__ double upd[NR][kLB];
    __shared__ double T[kLB][kLB + 1];
    const SolveItem it = items[blockIdx.x];
    const FrontLd F = d.fronts[it.s];
    const int f = F.f;
    const double *L = d.fac + F.lofs;
    const int32_t *rows = d.rows + F.rofs;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const bool tri = (it.flags & kItemTri) != 0;
    if (tri) load_unit_triangle(L, f, it.tk, it.tkb, T);
    for (int r0 = 0; r0 < nrhs; r0 += NR) {
        const int nr = min(NR, nrhs - r0);
        double *yr = y + static_cast<int64_t>(r0) * n;
        for (int e = tid; e < NR * kLSeg; e += kLThreads) {
            const int r = e / kLSeg, t = e % kLSeg;
            if (t < it.kb) xs[r][t] = r < nr ? yr[static_cast<int64_t>(r) * n + rows[it.k + t]] : 0.0;
        }
        __syncthreads();
        if (!tri) {
            cols_times_rows<NR>(L, f, it.k, it.kb, it.a0, it.a1, xs, [&](int r, int c, double acc) {
                if (r >= nr) return;
                double *dst = &yr[static_cast<int64_t>(r) * n + rows[c]];
                if (it.flags & kItemAtomic) unsafeAtomicAdd(dst, -acc);
                else *dst -= acc;
            });
            __syncthreads();
            continue;
        }
        // the block's columns: contributions of the rows below the pivots
        // (when the item carries them)
        if (it.kb > 0) {
            cols_times_rows<NR>(L, f, it.k, it.kb, it.tk, it.tk + it.tkb, xs,
                                [&](int r, int c, double acc) { upd[r][c - it.tk] = acc; });
            __syncthreads();
        }
        if (w < nr) {
            double *yw = yr + static_cast<int64_t>(w) * n;
            const bool in = lane < it.tkb;
            const int32_t g = rows[it.tk + min(lane, it.tkb - 1)];
            double yv = in ? yw[g] : 0.0;
            if (it.kb > 0 && in) yv -= upd[w][lane];
            yv = unit_backward(T, yv, it.tkb);
            if (in) yw[g] = yv;
        }
        __syncthreads();
    }
}

// Chains of fronts of at most 64 rows: one wavefront goes along its chain,
// lane i at row i of a front. Forward: the pivots' right-hand sides and, for
// the rows below, zero; each pivot's column (lane = row) subtracts its solved
// value from the lanes below it, and the rows below add theirs to y. What
// bounds it is the chain: an addition to y, the next front's read of it and
// its pivots' steps one after the other. So the next front's row ids and
// first kChainCols columns are loaded during the front before, and accesses
// of one wavefront to the same y need no wait between them. 121 fronts of
// 24-31 rows: 114 us forward, 227 us backward (a launch a level: 640 and 590
// us).
constexpr int kChainCols = 32;

// y is read from where the additions happen
__device__ __forceinline__ double y_load(const double *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct ChainCols {
    double t[kChainCols];
    int32_t g;
    __device__ __forceinline__ void load(const LdltDev &d, const ChainFront &c) {
        const int i = min(static_cast<int>(threadIdx.x), c.f - 1);
        g = d.rows[c.rofs + i];
        const double *L = d.fac + c.lofs + i;
#pragma unroll
        for (int u = 0; u < kChainCols; ++u) t[u] = L[static_cast<int64_t>(min(u, c.p - 1)) * c.f];
    }
};

template <int NR>
__global__ __launch_bounds__(64) void k_ldlt_fwd_chain(LdltDev d, const int32_t *__restrict__ ptr,
                                                      const ChainFront *__restrict__ fronts, double *y, int32_t n,
                                                      int32_t nrhs) {
    const int lane = threadIdx.x;
    const int r0 = blockIdx.y * NR, nr = min(NR, nrhs - r0);
    double *yr = y + static_cast<int64_t>(r0) * n;
    const int j0 = ptr[blockIdx.x], j1 = ptr[blockIdx.x + 1];
    if (j0 >= j1) return;
    ChainFront c = fronts[j0], cn = fronts[min(j0 + 1, j1 - 1)];
    // front j, its columns in x, while the next one's are loaded to xn
    const auto front = [&](int j, const ChainCols &x, ChainCols &xn) {
        double yv[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const double v = y_load(yr + static_cast<int64_t>(min(r, nr - 1)) * n + x.g);
            yv[r] = lane < c.p ? v : 0.0;
        }
        double acc[4][NR] = {};  // the rows below: four sums, as they round less than one
        const ChainFront cnn = fronts[min(j + 2, j1 - 1)];
        xn.load(d, cn);
        const double *L = d.fac + c.lofs + min(lane, c.f - 1);
#pragma unroll
        for (int c0 = 0; c0 < kChainRows; c0 += 16) {
            if (c0 >= c.p) break;
            double t[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                if (c0 < kChainCols) t[u] = x.t[c0 + u];
                else t[u] = L[static_cast<int64_t>(min(c0 + u, c.p - 1)) * c.f];
                if (lane <= c0 + u || c0 + u >= c.p) t[u] = 0.0;
            }
#pragma unroll
            for (int u = 0; u < 16; ++u)
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const double v = lane_value(yv[r], c0 + u);
                    yv[r] -= t[u] * v;
                    acc[u & 3][r] -= t[u] * v;
                }
        }
        bool finite = true;
#pragma unroll
        for (int r = 0; r < NR; ++r) finite = finite && isfinite(yv[r]);
        if (__ballot(!finite) != 0) {
            // as in unit_forward: again, with a test on the lane
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const double v = y_load(yr + static_cast<int64_t>(min(r, nr - 1)) * n + x.g);
                yv[r] = lane < c.p ? v : 0.0;
                for (int k = 0; k < 4; ++k) acc[k][r] = 0.0;
            }
            for (int c0 = 0; c0 < c.p; c0 += 4)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (c0 + u >= c.p) break;
                    const double t = L[static_cast<int64_t>(c0 + u) * c.f];
#pragma unroll
                    for (int r = 0; r < NR; ++r) {
                        const double v = lane_value(yv[r], c0 + u);
                        if (lane > c0 + u) {
                            yv[r] -= t * v;
                            acc[u][r] -= t * v;
                        }
                    }
                }
        }
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (r < nr) {
                double *dst = yr + static_cast<int64_t>(r) * n + x.g;
                if (lane < c.p) *dst = yv[r];
                else if (lane < c.f) unsafeAtomicAdd(dst, (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]));
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        c = cn;
        cn = cnn;
    };
    ChainCols a, b;
    a.load(d, c);
    for (int j = j0; j < j1; j += 2) {
        front(j, a, b);
        if (j + 1 < j1) front(j + 1, b, a);
    }
}

// Backward: from the top of the chain; the columns go through LDS, lane c
// then takes column c's entries against the rows' solved values, last row
// first.
template <int NR>
__global__ __launch_bounds__(64) void k_ldlt_bwd_chain(LdltDev d, const int32_t *__restrict__ ptr,
                                                      const ChainFront *__restrict__ fronts, double *y, int32_t n,
                                                      int32_t nrhs) {
    __shared__ double T[kChainRows][kChainRows + 1];
    const int lane = threadIdx.x;
    const int r0 = blockIdx.y * NR, nr = min(NR, nrhs - r0);
    double *yr = y + static_cast<int64_t>(r0) * n;
    const int j0 = ptr[blockIdx.x], j1 = ptr[blockIdx.x + 1];
    if (j0 >= j1) return;
    ChainFront c = fronts[j1 - 1], cn = fronts[max(j1 - 2, j0)];
    const auto front = [&](int j, const ChainCols &x, ChainCols &xn) {
        double yv[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) yv[r] = y_load(yr + static_cast<int64_t>(min(r, nr - 1)) * n + x.g);
        const ChainFront cnn = fronts[max(j - 2, j0)];
        xn.load(d, cn);
        const double *L = d.fac + c.lofs + min(lane, c.f - 1);
#pragma unroll
        for (int c0 = 0; c0 < kChainRows; c0 += 16) {
            if (c0 >= c.p) break;
            double t[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                if (c0 < kChainCols) t[u] = x.t[c0 + u];
                else t[u] = L[static_cast<int64_t>(min(c0 + u, c.p - 1)) * c.f];
            }
#pragma unroll
            for (int u = 0; u < 16; ++u) T[c0 + u][lane] = (lane > c0 + u && lane < c.f) ? t[u] : 0.0;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // the rows below the pivots: four sums of their own, then taken off
        // (off the right-hand side one by one, each would round at its size)
        double acc[4][NR] = {};
#pragma unroll
        for (int i0 = kChainRows - 16; i0 >= 0; i0 -= 16) {
            if (i0 >= c.f || i0 + 16 <= c.p) continue;
            double t[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                t[u] = T[lane][i0 + u];
                if (lane >= c.p || i0 + u < c.p) t[u] = 0.0;
            }
#pragma unroll
            for (int u = 15; u >= 0; --u)
#pragma unroll
                for (int r = 0; r < NR; ++r) acc[u & 3][r] += t[u] * lane_value(yv[r], i0 + u);
        }
#pragma unroll
        for (int r = 0; r < NR; ++r) yv[r] -= (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
#pragma unroll
        for (int i0 = kChainRows - 16; i0 >= 0; i0 -= 16) {
            if (i0 >= c.p) continue;
            double t[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                t[u] = T[lane][i0 + u];
                if (lane >= c.p || i0 + u >= c.p) t[u] = 0.0;
            }
#pragma unroll
            for (int u = 15; u >= 0; --u)
#pragma unroll
                for (int r = 0; r < NR; ++r) yv[r] -= t[u] * lane_value(yv[r], i0 + u);
        }
        bool finite = true;
#pragma unroll
        for (int r = 0; r < NR; ++r) finite = finite && (isfinite(yv[r]) || lane >= c.p);
        if (__ballot(!finite) != 0) {
            // as in unit_backward: again, with a test on the lane
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                yv[r] = y_load(yr + static_cast<int64_t>(min(r, nr - 1)) * n + x.g);
                for (int k = 0; k < 4; ++k) acc[k][r] = 0.0;
            }
            const int lc = min(lane, c.p - 1);
            for (int i0 = (c.f - 1) / 4 * 4; i0 + 4 > c.p; i0 -= 4)
#pragma unroll
                for (int u = 3; u >= 0; --u) {
                    if (i0 + u >= c.f || i0 + u < c.p) continue;
#pragma unroll
                    for (int r = 0; r < NR; ++r) acc[u][r] += T[lc][i0 + u] * lane_value(yv[r], i0 + u);
                }
#pragma unroll
            for (int r = 0; r < NR; ++r) yv[r] -= (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
            for (int i = c.p - 1; i > 0; --i)
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const double v = lane_value(yv[r], i);
                    if (lane < i) yv[r] -= T[lane][i] * v;
                }
        }
#pragma unroll
        for (int r = 0; r < NR; ++r)
            if (r < nr && lane < c.p) yr[static_cast<int64_t>(r) * n + x.g] = yv[r];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        c = cn;
        cn = cnn;
    };
    ChainCols a, b;
    a.load(d, c);
    for (int j = j1 - 1; j >= j0; j -= 2) {
        front(j, a, b);
        if (j - 1 >= j0) front(j - 1, b, a);
    }
}

}  // namespace

// right-hand sides per pass of an item: the smallest of 1, 2, 4 that covers
// them, 4 when there are more (a triangle's waves; accumulators in registers)
template <class Go>
static void by_rhs(int32_t nrhs, Go &&go) {
    if (nrhs == 1) go(std::integral_constant<int, 1>{});
    else if (nrhs == 2) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 4>{});
}

void launch_ldlt_fwd_step(hipStream_t st, const LdltDev &d, const SolveItem *items, int64_t count, bool wide,
                          double *y, int32_t n, int32_t nrhs) {
    for (int64_t o = 0; o < count; o += kMaxLaunchGroups) {
        const dim3 grid(static_cast<unsigned>(std::min(kMaxLaunchGroups, count - o)));
        by_rhs(nrhs, [&](auto nr) {
            if (wide) k_ldlt_fwd_tri<decltype(nr)::value><<<grid, kLWide, 0, st>>>(d, items + o, y, n, nrhs);
            else k_ldlt_fwd_step<decltype(nr)::value><<<grid, kLThreads, 0, st>>>(d, items + o, y, n, nrhs);
        });
    }
}

void launch_ldlt_chains(hipStream_t st, const LdltDev &d, bool fwd, const int32_t *ptr, const ChainFront *fronts,
                        int64_t count, double *y, int32_t n, int32_t nrhs) {
    for (int64_t o = 0; o < count; o += kMaxLaunchGroups) {
        const unsigned g = static_cast<unsigned>(std::min(kMaxLaunchGroups, count - o));
        by_rhs(nrhs, [&](auto nr) {
            constexpr int NR = decltype(nr)::value;
            const dim3 grid(g, static_cast<unsigned>((nrhs + NR - 1) / NR));
            if (fwd) k_ldlt_fwd_chain<NR><<<grid, 64, 0, st>>>(d, ptr + o, fronts, y, n, nrhs);
            else k_ldlt_bwd_chain<NR><<<grid, 64, 0, st>>>(d, ptr + o, fronts, y, n, nrhs);
        });
    }
}

void launch_ldlt_bwd_step(hipStream_t st, const LdltDev &d, const SolveItem *items, int64_t count, bool wide,
                          double *y, int32_t n, int32_t nrhs) {
    for (int64_t o = 0; o < count; o += kMaxLaunchGroups) {
        const dim3 grid(static_cast<unsigned>(std::min(kMaxLaunchGroups, count - o)));
        by_rhs(nrhs, [&](auto nr) {
            if (wide) k_ldlt_bwd_tri<decltype(nr)::value><<<grid, kLWide, 0, st>>>(d, items + o, y, n, nrhs);
            else k_ldlt_bwd_step<decltype(nr)::value><<<grid, kLThreads, 0, st>>>(d, items + o, y, n, nrhs);
        });
    }
}

void launch_sweep(hipStream_t st, const DevPtrs &d, bool forward, const SolveItem *items, const int32_t *step_of,
                  const int32_t *step_cnt, int32_t nitems, int32_t nsteps, int32_t *ctr, int32_t *err, double *y,
                  int32_t n, int32_t nrhs) {
    if (nitems <= 0) return;
    k_zero_i32<<<dim3(std::max(1, std::min(64, (nsteps + 1 + 255) / 256))), 256, 0, st>>>(ctr, nsteps + 1);
    const dim3 grid(static_cast<unsigned>(nitems));  // one workgroup per item
    if (forward) {
        if (nrhs == 1) k_sweep<1, true><<<grid, kSThreads, 0, st>>>(d, items, step_of, step_cnt, ctr, err, y, n, nrhs);
        else if (nrhs <= 4) k_sweep<4, true><<<grid, kSThreads, 0, st>>>(d, items, step_of, step_cnt, ctr, err, y, n, nrhs);
        else k_sweep<16, true><<<grid, kSThreads, 0, st>>>(d, items, step_of, step_cnt, ctr, err, y, n, nrhs);
    } else {
        if (nrhs == 1) k_sweep<1, false><<<grid, kSThreads, 0, st>>>(d, items, step_of, step_cnt, ctr, err, y, n, nrhs);
        else if (nrhs <= 4) k_sweep<4, false><<<grid, kSThreads, 0, st>>>(d, items, step_of, step_cnt, ctr, err, y, n, nrhs);
        else k_sweep<16, false><<<grid, kSThreads, 0, st>>>(d, items, step_of, step_cnt, ctr, err, y, n, nrhs);
    }
}

void launch_fwd_step(hipStream_t st, const DevPtrs &d, const SolveItem *items, int64_t count, double *y, int32_t n,
                     int32_t nrhs) {
    for (int64_t o = 0; o < count; o += kMaxLaunchGroups) {
        const dim3 grid(static_cast<unsigned>(std::min(kMaxLaunchGroups, count - o)));
        if (nrhs == 1) k_fwd_step<1><<<grid, kSThreads, 0, st>>>(d, items + o, y, n, nrhs);
        else if (nrhs <= 4) k_fwd_step<4><<<grid, kSThreads, 0, st>>>(d, items + o, y, n, nrhs);
        else k_fwd_step<16><<<grid, kSThreads, 0, st>>>(d, items + o, y, n, nrhs);
    }
}

void launch_bwd_step(hipStream_t st, const DevPtrs &d, const SolveItem *items, int64_t count, double *y, int32_t n,
                     int32_t nrhs) {
    for (int64_t o = 0; o < count; o += kMaxLaunchGroups) {
        const dim3 grid(static_cast<unsigned>(std::min(kMaxLaunchGroups, count - o)));
        if (nrhs == 1) k_bwd_step<1><<<grid, kSThreads, 0, st>>>(d, items + o, y, n, nrhs);
        else if (nrhs <= 4) k_bwd_step<4><<<grid, kSThreads, 0, st>>>(d, items + o, y, n, nrhs);
        else k_bwd_step<16><<<grid, kSThreads, 0, st>>>(d, items + o, y, n, nrhs);
    }
}

}  // namespace smfgpu
