// Device data of the indefinite (LDL^T) numeric phase. Front sizes grow with
// the delayed pivots children pass up, so they are known only when a
// level starts: the host lays the level out (offsets into the arenas
// below) after reading back its children's results.
#pragma once

#include "smfgpu_internal.hpp"

#include <vector>

namespace smfgpu {

// Front s of the current factorization. Its f x f square (column-major,
// leading dimension f, lower triangle) lives in the arena at fofs from its
// assembly until its parent has assembled the trailing (f - p) square, the
// contribution block (delayed rows first). Columns [0, pstore) are copied
// to the factor store at lofs (leading dimension f) in the FactorKeep
// layout: unit L, D on the diagonal, a 2x2 block's off-diagonal in slot
// (c, c+1), zeros elsewhere above the diagonal.
struct FrontLd {
    int32_t f, ne, nd, psym;  // rows, eligible columns, delayed columns received, own pivots
    int32_t col0;             // first own pivot column (permuted numbering)
    int32_t root;             // 1: no parent (unaccepted columns become zero pivots)
    int32_t p, pstore;        // accepted pivots; stored pivot columns
    int32_t npos, nneg, nzero, n2x2;
    int32_t delayed;
    int32_t dev;              // 1: laid out on the device (its square is not in the host's pool)
    int32_t nstatic;          // pivots whose |d| static pivoting raised
    // blocked fronts: first-pass panels that stalled, partner pairs pulled,
    // failed columns rotated to the end, second-pass full searches
    int32_t stalls, pulls, rotated, searches;
    double growth;            // largest column max / |d| over its static pivots
    double flops;
    int64_t fofs;             // arena offset of the square
    int64_t lofs;             // factor-store offset of the stored columns
    int64_t rofs;             // offset of the row ids / tags
    int64_t wofs;             // offset of the panel workspace W (blocked fronts)
    int64_t dofs;             // offset of the pivots' D^-1 entries
};

struct LdltDev {
    FrontLd *fronts;          // per supernode
    double *arena;            // front squares
    double *fac;              // stored factor columns
    int32_t *rows;            // per front: f row ids (permuted numbering), pivoted order
    int8_t *tags;             // per front: pivot tags (1, 2, -1, 0), same offsets as rows
    double *work;
    double *dinv;             // 3 per pivot
    int8_t *dkind;            // 1, 2, 0 per pivot
    const int32_t *pcol_ptr;
    const int32_t *amap;      // per permuted entry: position among its front's symbolic rows
    const double *av;
    double *junk;             // target of masked-out stores of the MFMA updates (contents meaningless)
    uint16_t *xpl;            // bf16 operand planes of the large fronts' outer-block updates (BF16 / split BF16):
                              // per front at 4 wofs, planes A hi, A lo, B hi, B lo of big_work(ne) f entries each
};

// Large fronts (multi-workgroup blocked LDL^T): one state per front,
// advanced in rounds by a region kernel (one workgroup per front: a stalled
// panel's partner pulls / rotation, a speculative group's diagonal region),
// the group's rows kernel, a panel kernel (the blocked algorithm's pivot
// logic on the group or on a panel of nb columns) and an update kernel (many
// workgroups, MFMA), launched in turn by the host until every front is done. The per-panel deferred
// updates go to the columns of a kBigOuter-wide outer block; the pivots'
// updates of the columns beyond it are held back (their unscaled columns
// kept in W) and applied in one flush when the outer block ends, before a
// stall's pulls or rotation, and before the second pass.
// BF16 and split-BF16 fronts on bf16 planes take wider outer blocks (and
// contribution-block chunks), 1024 by default: their 256 x 256 tiles then
// read and write the FP64 entries once per rank-1024 update instead of
// once per rank-512 one, which bounds them (the FP32 accumulators sum
// twice as many products).
constexpr int32_t kBigOuter = 512;
constexpr int32_t kBigOuterMax = 1024;
// W columns of a front with ne eligible columns: an outer block's pivots
// (L*D chunks of the final update), then a speculative group's final
// entries, from column big_spec on. A multiple of 8 columns: an operand
// plane of as many bf16 columns then keeps its reader's 16-byte alignment.
__host__ __device__ constexpr int32_t big_spec(int32_t ne) {
    return ne < kBigOuterMax ? (ne + 7) / 8 * 8 : kBigOuterMax;
}
__host__ __device__ constexpr int32_t big_work(int32_t ne) { return big_spec(ne) + 64; }
// Workspace entries of a front of f rows and `cols` W columns: a multiple of
// 8, so that the next front's planes, at 4 bf16 entries per entry, start on 16
// bytes too.
__host__ __device__ constexpr int64_t work_room(int32_t f, int32_t cols) {
    return (static_cast<int64_t>(f) * cols + 7) / 8 * 8;
}
static_assert(kBigOuterMax >= kBigOuter, "W holds the pivots of an outer block");
struct BigLd {
    int32_t s;                  // supernode
    int32_t k, live, k_paired;  // next pivot position, end of the live eligible columns, pulls' guard
    int32_t pass;               // 0 first pass, 1 second pass, 2 done
    int32_t full;               // second pass: next step is a full-search pivot
    int32_t stalled;            // first pass: the last panel stalled
    int32_t ps, pl;             // the last panel
    int32_t oe;                 // outer block end
    int32_t outer;              // outer block width (kBigOuter, or the plan's ldlt_outer_wide on planes)
    int32_t pend0;              // pivots [pend0, k) held back for the columns >= oe; W column 0
    int32_t u_c0, u_c1, u_p0, u_p1;  // update request: columns [u_c0, u_c1), rows [u_c0, f), pivots [u_p0, u_p1)
    int32_t x_c0, x_p0, x_p1;        // flush request: columns [x_c0, ne), rows [x_c0, f), pivots [x_p0, x_p1)
    int32_t w_base;             // pivot of W column 0 for both requests
    int32_t cnt[3];
    int32_t stalls, pulls, rotated, searches;  // as FrontLd's
    int32_t spec;               // 1: the next first-pass iteration tries a speculative group
    int32_t prec;               // precision code of the MFMA updates: 0 FP64, 1 FP32, 2 BF16, 3 split BF16
    double flops;
};
// Workgroup `part` of the `parts` a launch gives front `front` of the level's
// large fronts. A level's launches share one list per kind of work, sized by
// each front: a list entry per workgroup instead of the largest front's
// number for every front (a level mixes fronts of 96 rows with fronts of
// thousands, and an empty workgroup still costs its dispatch).
struct BigPart {
    int32_t front, part, parts;
};
struct BigGrid {
    const BigPart *rows;    // kGroupRows-row chunks (group and panel kernels)
    const BigPart *tiles;   // 128 x 128 update tiles, a multiple of 8 per front (one run of tiles per XCD)
    const BigPart *wide;    // 256 x 256 update tiles, likewise
    int32_t nrows, ntiles, nwide;
};
// The list of row chunks, chunks[b] of front b: every front's first chunk, then
// every front's second one, and so on. A front's first workgroup does its
// pivot logic; workgroups go to the 8 XCDs in turn, so lists front by front
// put the pivot logic of equal fronts of 2, 4 or 8 chunks on 4, 2 or one
// of them.
inline void row_parts(const std::vector<int32_t> &chunks, std::vector<BigPart> &out) {
    bool more = true;
    for (int32_t i = 0; more; ++i) {
        more = false;
        for (size_t b = 0; b < chunks.size(); ++b)
            if (i < chunks[b]) {
                out.push_back(BigPart{static_cast<int32_t>(b), i, chunks[b]});
                more = true;
            }
    }
}
constexpr int32_t kGroupCols = 64;   // columns of a speculative group (four panels of 16)
constexpr int32_t kGroupRows = 64;   // rows per workgroup below a group's diagonal region
static_assert(big_work(1) - big_spec(1) == kGroupCols, "W holds a group's speculative columns");
constexpr int64_t kGroupBuf = 192 + 2 * 64 * 64;  // group buffer per front (doubles)

// Static pivoting (control.hpp:333-364): sp = static_pivot_tol * max|A|
// (0: off), fallback = fallback_static_pivot_tol * max|A| for roots and
// fronts that receive more delayed columns than their width; flags as
// SMFGPU_STATIC_*.
struct StaticPrm {
    double sp, fallback;
    int32_t flags;
};
constexpr int32_t kStaticAsZero = 1, kStaticZeroStaysZero = 2, kStaticInOrder = 4;
// whether front F pivots statically, and with which value
__host__ __device__ inline double front_static_value(const StaticPrm &S, int32_t root, int32_t nd, int32_t psym) {
    return (S.fallback > 0.0 && (root != 0 || nd > psym)) ? S.fallback : S.sp;
}

// Levels of small fronts laid out on the device: one workgroup per front (of
// the lowest level of a band: levels whose fronts all have one child in the
// band, so each workgroup goes up its own chain of fronts) that
// lays it out (its size from its children's delays, offsets by a bump of the
// counters below), builds the row list, assembles, factors (the unblocked
// kernel's steps) and stores the front with the square in LDS. A level whose
// fronts do not all fit is refused: the counters record the first refused
// level and the reason, the launches of later levels return at once, and the
// refused level is laid out again whole (the fronts of it that ran changed
// nothing of their children).
constexpr int32_t kDevFrontMax = 95;   // largest realized front of a device level (blocked_min_front - 1)
constexpr int32_t kDevSymMax = 64;     // largest symbolic front of a level laid out on the device
enum : int32_t { kDcSq = 0, kDcFac = 1, kDcRows = 2, kDcDinv = 3, kDcLevel = 4, kDcWhy = 5, kDcN = 6 };
constexpr unsigned long long kDevWhySize = 1, kDevWhyRoom = 2;  // refusal: a front too large / a buffer full
struct DevLevel {
    const FrontDev *sym;        // symbolic fronts (f, p, col0, rofs)
    const int32_t *sym_rows;    // symbolic row ids
    const int32_t *sym_cmap;    // per child: its symbolic CB rows' positions among the parent's symbolic rows
    const int64_t *sym_cmofs;
    const int32_t *child_ptr, *child_idx, *parent;
    unsigned long long *ctr;    // kDcN counters: next free square / factor / row / D^-1 offsets, refused level, reason
    int64_t cap[4];             // ends of the room for the four offsets
    int32_t fmax;               // largest realized front taken
    const int32_t *lev;         // level per front
    int32_t end;                // a workgroup goes on from a front to its parent while that lies below this level
};
void launch_dev_fronts(hipStream_t st, const LdltDev &d, const DevLevel &L, const int32_t *flist, int32_t nf,
                       int32_t lv, double u, double eff_small, double small_pivot, const StaticPrm &S, bool wave);
// Fronts of a level up to which one launch takes both sizes, and a band: the
// four-wavefront workgroups (80 KB of LDS) that the card holds at a time. More
// of them wait for a place, and a launch a level with a wavefront a front is
// the faster one: 1536 trajectory systems of horizons up to 200 31.1 ms in
// one launch and 26.1 in a launch a level, 1024 22.2 and 20.9, 640 15.5 and
// 14.4; 520 still 11.8 and 12.1.
constexpr int32_t kDevOneLaunch = 512;

void launch_ldlt_small(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, double u, double eff_small,
                       double small_pivot, const StaticPrm &S);
void launch_ldlt_blocked(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, double u,
                         double eff_small, double small_pivot, int32_t nb, const StaticPrm &S);
// Assembly of a level laid out on the host: its plan-time tables, and groups
// of kAsmCols columns from c of front s, those of fronts of up to
// kAsmWaveRows rows (a wavefront per column) before those of larger ones (a
// workgroup per column).
struct LdltAsm {
    const FrontDev *sym;        // symbolic fronts
    const int32_t *sym_rows;    // symbolic row ids
    const int32_t *sym_cmap;    // as DevLevel
    const int64_t *sym_cmofs;
    const int32_t *child_ptr, *child_idx;
    const int32_t *col_ptr;     // per symbolic row of every front: its children's symbolic columns there,
    const ChildCol *cc;         // in child order
};
struct AsmPart {
    int32_t s, c;
};
constexpr int32_t kAsmCols = 8, kAsmWaveRows = 1024;
// records, row ids and cleared tags of the level's fronts (patch[i]: front ids[i])
void launch_ldlt_rows(hipStream_t st, const LdltDev &d, const LdltAsm &A, const FrontLd *patch, const int32_t *ids,
                      int32_t nf);
void launch_ldlt_assemble(hipStream_t st, const LdltDev &d, const LdltAsm &A, const AsmPart *parts, int64_t nwave,
                          int64_t nwg);
// epilogue (pivot counts, D^-1) of the fronts in flist; it also stores the
// factor columns of the first n_inline fronts, launch_ldlt_store those of
// the rest (many workgroups per front)
void launch_ldlt_epilogue(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, int32_t n_inline);
void launch_ldlt_store(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, int32_t max_cols);
// A store launch: `per` workgroups for each of the next `fronts` fronts, which
// are the grid's rows (65536 at most): about 8192 workgroups, at least 16 a
// front.
constexpr int32_t kStoreFronts = 32768;
struct StoreGrid {
    int32_t per, fronts;
};
inline StoreGrid store_grid(int32_t nf, int32_t max_cols) {
    const int32_t m = nf < kStoreFronts ? nf : kStoreFronts;
    const int32_t per = 8192 / m > 16 ? 8192 / m : 16;
    return StoreGrid{per < max_cols ? per : max_cols, m};
}
void launch_ldlt_diag(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, int32_t max_p, double *y,
                      int32_t n, int32_t nrhs);
// the diagonal-only solve job: D from the stored columns, by division
void launch_ldlt_diag_div(hipStream_t st, const LdltDev &d, const int32_t *flist, int32_t nf, double *y, int32_t n,
                          int32_t nrhs);
// flags of the LDL^T sweeps' items
constexpr int32_t kItemAtomic = 1;  // backward chunk: several items add to its columns
constexpr int32_t kItemTri = 2;     // a block's triangle, else a chunk
constexpr int32_t kItemFused = 4;   // forward: the triangle, then the rows [a0, a1) below it in the same workgroup
constexpr int32_t kItemWide = 8;    // a triangle of more than 64 pivots
// kinds of a sweep's steps: wide triangles, a band of chains, or (0) the other
// items
constexpr uint8_t kStepWide = 1, kStepChains = 2;
// a front of a chain: at most kChainRows rows
constexpr int32_t kChainRows = 64;
struct ChainFront {
    int64_t lofs, rofs;
    int32_t f, p;
};
// a band of levels in one launch: chain c is the fronts [ptr[c], ptr[c + 1])
// from the lowest level up
void launch_ldlt_chains(hipStream_t st, const LdltDev &d, bool fwd, const int32_t *ptr, const ChainFront *fronts,
                        int64_t count, double *y, int32_t n, int32_t nrhs);
// one step of the blocked forward / backward sweep (items of all fronts of
// a level); wide: the step's triangles of more than 64 pivots, else its
// other items (the two are independent)
void launch_ldlt_fwd_step(hipStream_t st, const LdltDev &d, const SolveItem *items, int64_t count, bool wide,
                          double *y, int32_t n, int32_t nrhs);
void launch_ldlt_bwd_step(hipStream_t st, const LdltDev &d, const SolveItem *items, int64_t count, bool wide,
                          double *y, int32_t n, int32_t nrhs);
// one round of the level's large fronts: the states of the round and,
// written by the panel launch, the next ones; gpart: the group buffers (null:
// one panel per round); nmode[m]: fronts whose updates run in precision code m
// (0 FP64, 1 FP32, 2 BF16, 3 split BF16), a launch per code in use
void launch_big_round(hipStream_t st, const LdltDev &d, BigLd *states, BigLd *next, int32_t nbig, const BigGrid &g,
                      double u, double eff_small, double small_pivot, int32_t nb, double *gpart,
                      const int32_t *nmode);
// final contribution-block update with pivots [c0, c0 + width) of every
// front (L*D of the chunk into W first); wide: the fronts on bf16 planes, else
// the others
void launch_big_cb(hipStream_t st, const LdltDev &d, const BigLd *states, const BigGrid &g, int32_t c0, int32_t width,
                   const int32_t *nmode, bool wide);
// the finished fronts' results, from their states to their records
void launch_big_finish(hipStream_t st, const LdltDev &d, const BigLd *states, int32_t nbig);

}  // namespace smfgpu
