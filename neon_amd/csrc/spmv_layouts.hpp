// The matrix layouts of the Krylov solvers, the symmetric sliced layout's row sums and the CG scalars,
// shared by the launch-per-phase kernels (krylov_kernels.hpp) and the resident grids
// (grid_kernels.hpp).
#pragma once

#include "common.hpp"
#include "neon_hip.h"

#include <cfloat>
#include <type_traits>

namespace neon_amd
{
// Scalars of one Krylov iteration, ping-ponged between two device slots so that the
// kernel that computes iteration k+1's scalars never overwrites what others still read.
struct krylov_state
{
    double rz;        // r . z  (Eigen's absNew, CUDA's "residual")
    double rr;        // r . r
    double rhs2;      // b . b
    double threshold; // Eigen: max(tol^2 ||b||^2, DBL_MIN)
    double alpha, beta, omega, rho; // BiCGSTAB scalars (alpha reused by CG for reports)
    double aux0, aux1;               // reliable-update bookkeeping (mixed precision)
    int32_t it;   // iterations as the reference counts them
    int32_t done; // 0 running, 1 converged, 2 iteration limit, 3 non-finite, 4 breakdown
    int32_t restarts;
    int32_t refine; // mixed precision: a reliable update is due this iteration
};

enum : int32_t
{
    KRYLOV_RUNNING = 0,
    KRYLOV_CONVERGED = 1,
    KRYLOV_LIMIT = 2,
    KRYLOV_NONFINITE = 3,
    KRYLOV_BREAKDOWN = 4,
    KRYLOV_REFINE = 5, // mixed precision: a reliable update is due
    KRYLOV_ABORTED = 6, // a resident grid gave up waiting (the host solves by launches instead)
};

// ----------------------------------------------------------------- SpMV layouts
// Node-block CSR: the tangent of a 3-dof-per-node mesh keeps its values in ordinary
// row-major CSR order (sorted columns), but every dof row of node n has the same column set
// {3m+j : m in adj(n), j < 3}, so the kernels read one int32 block column per 9 values:
//   row 3n+i, block s (node m = bcol[bptr[n]+s]), column 3m+j
//   -> val[9 bptr[n] + i (3 deg n) + 3 s + j].
struct nb_matrix
{
    int32_t nodes;
    const int32_t* bptr;
    const int32_t* bcol;
};

struct csr_matrix
{
    int32_t rows;
    const int32_t* rp;
    const int32_t* ci;
};

// Entries that a workgroup of the resident CSR grid takes at a time.  Its workgroups own equal runs of
// rows, so the one with the most entries sets the pace: 4 to 7 us for each chunk that it has more than
// the mean, against what the launches lose on the exchanges and passes (10 us, 2 us per mean chunk) and
// on the longest row, which they give `lanes` lanes (some 0.25 us per step).  Per iteration, grid /
// launches before this rule: 100,000 rows of 7 entries and 400 more rows of 20, 60, 160, 500 entries side by side
// 19 / 29, 32 / 35, 77 / 47, 223 / 82 us; 64 of 2,000 133 / 126; 4 of 5,000 31 / 129; one of 16,457 29 / 352.
constexpr int kCsrChunk = 4096;
__host__ __device__ inline bool csr_grid_pays(int64_t largest_block, double mean_block, int64_t longest_row, int lanes)
{
    return 5.0 * (double(largest_block) - mean_block) / kCsrChunk
           <= 10.0 + 2.0 * mean_block / kCsrChunk + 0.25 * double(longest_row) / lanes;
}

// Sliced node-block layout: a copy of the node-block values in which every wavefront load
// reads one contiguous span.  Slice s holds the 64 consecutive nodes 64 s ... 64 s + 63 (lane l:
// node snode[64 s + l]; an empty lane past the last node, snode -1 - m, gathers like node m and
// holds zero values) and sptr[s+1] - sptr[s] steps, the largest block count among them; step kk
// of a node is its kk-th block (ascending column node, as in bcol), and steps past a node's
// block count hold zero values.  The 9 values of a step form one record of 9 x 64 values:
// value t = 3 i + j of lane l sits at
//   sval[576 (sptr[s] + kk) + sell_pos<VT>(t, l)]:
// the first 8 in groups of W = 16 / sizeof(VT) per lane (one 16-byte load per lane and group;
// group g spans 64 W values), the ninth after them (one value per lane).
// A step's column offsets (column node - lane node): scode[step] < 0 encodes one offset shared
// by the slice's lanes (shared_offset()) except at most two exception lanes, named by
// slane[s] (8 bits each, 0xff for none), whose 16-bit offsets are in sexc[step]; scode[step]
// >= 0 indexes 64 per-lane offsets at soff16 / soff32 [scode * 64 + lane].  A slice's steps
// are all of one kind (the product tests the first code of each chunk of 64 steps).
template <typename VT>
__host__ __device__ constexpr int sell_pos(int t, int lane)
{
    constexpr int W = 16 / int(sizeof(VT));
    return t < 8 ? (t / W) * 64 * W + lane * W + t % W : 512 + lane;
}

struct sell_matrix
{
    int32_t nodes;
    int32_t slices;
    const int32_t* sptr;   // [slices + 1] first step of each slice
    const int32_t* snode;  // [slices * 64] node of each lane (-1 - m: empty lane gathering like node m)
    const int32_t* slane;  // [slices] exception lanes of a slice's shared steps (8 bits each, 0xff: none)
    const int32_t* scode;  // [steps] shared_code(offset) or the step's index into the per-lane offsets
    const int32_t* sexc;   // [steps] 16-bit offsets of the exception lanes (shared steps)
    const int16_t* soff16; // per-lane offsets when every one fits 16 bits (else null)
    const int32_t* soff32; // per-lane offsets in 32 bits (used when soff16 is null)
};
constexpr int64_t kSharedBias = int64_t(1) << 30;
__host__ __device__ inline int32_t shared_code(int64_t offset)
{
    return int32_t(int64_t(INT32_MIN) + kSharedBias + offset);
}
__host__ __device__ inline int64_t shared_offset(int32_t code) { return int64_t(code) - INT32_MIN - kSharedBias; }

// ------------------------------------------------ symmetric sliced layout
// For a symmetric tangent the copy keeps the diagonal block and the upper blocks (column node -
// row node = o > 0) only.  Slice s holds nodes 64 s .. 64 s + 63 (one per lane); its records of
// 9 x 64 values (sell_pos layout) are the diagonal block (record rdiag[s]) and one record per
// offset o in the slice's direct list (the upper offsets of its lanes' nodes): lane l's block
// (i, i + o), zero where node i has no such neighbour.  The product adds, for every lane node i,
// K(i, i + o) x(i + o) for the direct offsets and the transpose of K(i - o, i) x(i - o) for the
// slice's lower offsets (those of its lanes' lower neighbours): that block is lane (i - o) % 64
// of the record for o of slice (i - o) / 64, which is one of the two slices floor((64 s - o) /
// 64) and the next one, whose record indices the entry carries.  Every off-diagonal value is
// read twice, and the schedule makes the second read follow the first closely enough to be
// served by the L2.  A slice's entries merge the two lists by offset, each {o, direct record or
// -1, record in slice floor((64 s - o) / 64) or -1, record in the next slice or -1}, so that the
// direct and the transposed read of one offset are issued together.
// Schedule: wave slot q (workgroup q / 4, on XCD (q / 4) % 8) takes slice sched[q] (-1: none).
// The host orders the slices in tiles (a band of the in-plane index, then plane by plane) and
// gives each XCD one contiguous eighth of that order, so a slice's neighbours one plane down
// were read on the same XCD a few workgroups earlier.
constexpr int kMaxSymEntries = 40; // <= 64: a slice's entries fit one wavefront's lanes
typedef int int4v __attribute__((ext_vector_type(4)));
struct sym_matrix
{
    int32_t nodes;
    int32_t slices;
    int32_t slots;          // wave slots of the schedule (a multiple of 32)
    int64_t records;        // records of the copy
    const int32_t* sched;   // [slots] slice of each wave slot, -1 for none
    const int32_t* rdiag;   // [slices] record of each slice's diagonal block
    const int32_t* eptr;    // [slices + 1] entry range of each slice
    const int4v* ent;       // entries, by slice and ascending offset
    const int32_t* rslice;  // [records] slice of each record (packing)
    const int32_t* roff;    // [records] offset of each record, 0 for the diagonal (packing)
};

// What a wavefront needs of slice s before it can read its records: the diagonal record and the
// slice's entries (at most kMaxSymEntries <= 64), lane k holding entry k (one coalesced load, then
// each entry read from its lane: no scalar-load wait in the loop).
struct sym_head
{
    int32_t s, ne;
    int32_t rdiag;
    int4v mine;
};
__device__ __forceinline__ sym_head sym_load_head(sym_matrix const& A, int32_t s, int lane)
{
    sym_head h;
    h.s = s;
    h.rdiag = A.rdiag[s];
    int32_t const e0 = A.eptr[s];
    h.ne = A.eptr[s + 1] - e0;
    h.mine = lane < h.ne ? A.ent[e0 + lane] : int4v{0, 0, -1, -1};
    return h;
}

// One slice's rows of the product: lane l's three row sums (node 64 s + l) over the diagonal record
// (when first is 0) and the entries first, first + STEP, first + 2 STEP, ...  FP32
// accumulation rotates over four accumulator sets as in spmv_sell_kernel; FP64 uses one.  back: the
// entries in descending order.  xo: x at the lane's own node; x (a pointer, or anything indexed like one) is read at the column nodes.
template <int STEP, typename VT, typename XT, typename AT, typename XV>
__device__ __forceinline__ void sym_slice_rows(sym_matrix const& A, const VT* __restrict__ val, XV x, sym_head const& h,
                                               int lane, int32_t first, bool back, XT xo0, XT xo1, XT xo2, AT& r0, AT& r1,
                                               AT& r2)
{
    int32_t const s = h.s;
    int64_t const nodes = A.nodes;
    int64_t const i = int64_t(s) * 64 + lane;
    int64_t const ic = i < nodes ? i : nodes - 1;
    int64_t const rdiag = h.rdiag;
    constexpr int W = 16 / int(sizeof(VT));
    typedef VT vec_t __attribute__((ext_vector_type(W)));
    // the 9 values of lane l of the record at rec (NT: nontemporal, for a record read once)
    auto load_rec = [&](const VT* rec, int l, VT(&v)[9], auto nt) {
#pragma unroll
        for (int g = 0; g < 8 / W; ++g)
        {
            const vec_t* src = reinterpret_cast<const vec_t*>(rec + g * 64 * W) + l;
            vec_t q;
            if constexpr (decltype(nt)::value)
                q = __builtin_nontemporal_load(src);
            else
                q = *src;
#pragma unroll
            for (int j = 0; j < W; ++j) v[g * W + j] = q[j];
        }
        if constexpr (decltype(nt)::value)
            v[8] = __builtin_nontemporal_load(rec + 512 + l);
        else
            v[8] = rec[512 + l];
    };
    AT a0 = AT(0), a1 = AT(0), a2 = AT(0), b0 = AT(0), b1 = AT(0), b2 = AT(0);
    AT c0 = AT(0), c1 = AT(0), c2 = AT(0), d0 = AT(0), d1 = AT(0), d2 = AT(0);
    // one block's product (transposed: K^T x) into the next accumulator set
    auto accumulate = [&](VT const(&v)[9], XT x0_, XT x1_, XT x2_, bool tr) {
        AT const x0 = AT(x0_), x1 = AT(x1_), x2 = AT(x2_);
        AT n0, n1, n2;
        if (tr)
        {
            n0 = a0 + (AT(v[0]) * x0 + AT(v[3]) * x1 + AT(v[6]) * x2);
            n1 = a1 + (AT(v[1]) * x0 + AT(v[4]) * x1 + AT(v[7]) * x2);
            n2 = a2 + (AT(v[2]) * x0 + AT(v[5]) * x1 + AT(v[8]) * x2);
        }
        else
        {
            n0 = a0 + (AT(v[0]) * x0 + AT(v[1]) * x1 + AT(v[2]) * x2);
            n1 = a1 + (AT(v[3]) * x0 + AT(v[4]) * x1 + AT(v[5]) * x2);
            n2 = a2 + (AT(v[6]) * x0 + AT(v[7]) * x1 + AT(v[8]) * x2);
        }
        if constexpr (sizeof(AT) == 4)
        {
            a0 = b0, a1 = b1, a2 = b2;
            b0 = c0, b1 = c1, b2 = c2;
            c0 = d0, c1 = d1, c2 = d2;
            d0 = n0, d1 = n1, d2 = n2;
        }
        else
        {
            a0 = n0, a1 = n1, a2 = n2;
        }
    };
    if (STEP == 1 || first == 0)
    {
        VT v[9];
        load_rec(val + rdiag * 576, lane, v, std::true_type{});
        accumulate(v, xo0, xo1, xo2, false);
    }
    // one entry's operands: the stored block K(i, i + o) and x(i + o) (zero where the slice
    // has no direct record for o), and the transpose of K(i - o, i) and x(i - o) (x counts
    // as zero where node i - o does not exist or holds no block for o: its values are then
    // read from the slice's own diagonal record, in bounds)
    int32_t const ne = h.ne;
    int4v const mine = h.mine;
    struct pair_t
    {
        VT v[9], w[9];
        XT x0, x1, x2, z0, z1, z2;
        bool dv, jv;
    };
    auto fetch = [&](int32_t m0) {
        int32_t const m = back ? ne - 1 - m0 : m0;
        pair_t o;
        int4v const e{__builtin_amdgcn_readlane(mine.x, m), __builtin_amdgcn_readlane(mine.y, m),
                      __builtin_amdgcn_readlane(mine.z, m), __builtin_amdgcn_readlane(mine.w, m)};
        int64_t const off = e.x;
        int64_t const rd = e.y;
        o.dv = rd >= 0;
        int64_t const mi = i + off < nodes ? i + off : nodes - 1;
        load_rec(val + (o.dv ? rd : rdiag) * 576, lane, o.v, std::false_type{});
        o.x0 = x[3 * mi], o.x1 = x[3 * mi + 1], o.x2 = x[3 * mi + 2];
        int64_t const j0 = i - off;
        int64_t const sa = (int64_t(s) * 64 - off) >> 6; // floor division by 64
        int64_t const rt = (j0 >> 6) == sa ? int64_t(e.z) : int64_t(e.w);
        o.jv = j0 >= 0 && j0 < nodes && rt >= 0;
        int64_t const j = o.jv ? j0 : ic;
        load_rec(val + (o.jv ? rt : rdiag) * 576, o.jv ? int(j & 63) : lane, o.w, std::false_type{});
        o.z0 = x[3 * j], o.z1 = x[3 * j + 1], o.z2 = x[3 * j + 2];
        return o;
    };
    auto accumulate_pair = [&](pair_t const& o) {
        accumulate(o.v, o.dv ? o.x0 : XT(0), o.dv ? o.x1 : XT(0), o.dv ? o.x2 : XT(0), false);
        accumulate(o.w, o.jv ? o.z0 : XT(0), o.jv ? o.z1 : XT(0), o.jv ? o.z2 : XT(0), true);
    };
    // software-pipelined over two register sets: entry m + STEP's loads are issued before
    // entry m is accumulated (3 % faster at 128^3 in both precisions than a plain loop)
    int32_t m = STEP == 1 ? 0 : first;
    if (m + STEP < ne)
    {
        pair_t sa_ = fetch(m);
        for (; m + 2 * STEP < ne; m += 2 * STEP)
        {
            pair_t const sb = fetch(m + STEP);
            accumulate_pair(sa_);
            sa_ = fetch(m + 2 * STEP);
            accumulate_pair(sb);
        }
        accumulate_pair(sa_);
        m += STEP;
    }
    for (; m < ne; m += STEP) accumulate_pair(fetch(m));
    r0 = (a0 + b0) + (c0 + d0);
    r1 = (a1 + b1) + (c1 + d1);
    r2 = (a2 + b2) + (c2 + d2);
}

// The state a CG solve starts from, given r.r and r.z of the start (x = 0)
__device__ inline krylov_state cg_first_state(double rr, double rz, int criterion, double tol, int max_it)
{
    krylov_state s{};
    s.rz = rz;
    s.rr = rr;
    s.rhs2 = rr;
    s.it = 0;
    s.done = KRYLOV_RUNNING;
    if (criterion == NEON_STOP_RELATIVE)
    {
        s.threshold = fmax(tol * tol * rr, DBL_MIN);
        if (rr == 0.0 || rr < s.threshold) s.done = KRYLOV_CONVERGED;
    }
    else
    {
        s.threshold = 0.0;
        if (!(sqrt(rz) > tol)) s.done = KRYLOV_CONVERGED;
    }
    if (s.done == KRYLOV_RUNNING && max_it <= 0) s.done = KRYLOV_LIMIT;
    if (!isfinite(rr) || !isfinite(rz)) s.done = KRYLOV_NONFINITE;
    return s;
}

// End of a CG iteration: s <- its scalars, count and status from the new r.r and r.z; returns beta.
__device__ inline double cg_decide(krylov_state& s, double rr, double rz, int criterion, double tol, int max_it)
{
    int32_t it_new;
    int32_t done = KRYLOV_RUNNING;
    if (criterion == NEON_STOP_RELATIVE)
    {
        bool const conv = rr < s.threshold; // Eigen breaks before counting the iteration
        it_new = conv ? s.it : s.it + 1;
        if (conv)
            done = KRYLOV_CONVERGED;
        else if (it_new >= max_it)
            done = KRYLOV_LIMIT;
    }
    else
    {
        it_new = s.it + 1; // the CUDA loop counts at the top
        if (it_new >= max_it)
            done = KRYLOV_LIMIT;
        else if (!(sqrt(rz) > tol))
            done = KRYLOV_CONVERGED;
    }
    if (!isfinite(rr) || !isfinite(rz)) done = KRYLOV_NONFINITE;
    double const beta = rz / s.rz;
    s.rr = rr;
    s.rz = rz;
    s.beta = beta;
    s.it = it_new;
    s.done = done;
    return beta;
}

// The state a BiCGSTAB solve starts from (x = 0, r = r0 = b), given b.b
__host__ __device__ inline krylov_state bicg_first_state(double bb, int cuda_rule, double tol, int max_it)
{
    krylov_state s{};
    s.rz = bb; // r0 . r = b . b
    s.rr = bb;
    s.rhs2 = bb;
    s.aux0 = 1.0; // Eigen's rho_old, alpha, omega start at 1
    s.alpha = 1.0;
    s.omega = 1.0;
    s.aux1 = bb; // Eigen's |r0|^2
    if (cuda_rule)
    {
        s.aux0 = 0.0;
        s.alpha = s.omega = 0.0;
        if (!(sqrt(bb) > tol))
            s.done = KRYLOV_CONVERGED;
        else if (max_it <= 0)
            s.done = KRYLOV_LIMIT;
    }
    else
    {
        s.threshold = tol * tol * bb;
        if (bb == 0.0 || !(bb > s.threshold))
            s.done = KRYLOV_CONVERGED;
        else if (max_it <= 0)
            s.done = KRYLOV_LIMIT;
    }
    if (!(fabs(bb) <= DBL_MAX)) s.done = KRYLOV_NONFINITE;
    return s;
}

// The Eigen rule's restart test |rho| < eps^2 |r0|^2 and the scalars after a restart with |r|^2 = rr
// (the first one resets the iteration count)
__device__ inline bool bicg_restart_due(krylov_state const& s)
{
    return fabs(s.rz) < DBL_EPSILON * DBL_EPSILON * s.aux1;
}
__device__ inline void bicg_restarted(krylov_state& s, double rr)
{
    s.rz = rr;
    s.aux1 = rr;
    if (s.restarts++ == 0) s.it = 0;
    s.refine = 0;
}

// End of a BiCGSTAB iteration: s <- its scalars, count and status (s.refine: the CUDA rule's early
// exit; ts, tt, r0r and rr are then unused)
__device__ inline void bicg_decide(krylov_state& s, double ts, double tt, double r0r, double rr, int cuda_rule,
                                   double tol, int max_it)
{
    int32_t const k = s.it + 1;
    if (cuda_rule)
    {
        if (s.refine)
        {
            // ||s|| < tol: x += alpha p_hat, residual = ||s||^2, leave the loop
            s.rz = s.aux1 * s.aux1;
            s.done = k >= max_it ? KRYLOV_LIMIT : KRYLOV_CONVERGED;
        }
        else
        {
            s.omega = ts / tt;
            s.aux0 = s.rz;
            s.rz = r0r;
            if (s.omega == 0.0) // is_approx(omega, 0.0): an exact zero
                s.done = KRYLOV_BREAKDOWN;
            else if (!(sqrt(s.rz) > tol) || k >= max_it)
                s.done = k >= max_it ? KRYLOV_LIMIT : KRYLOV_CONVERGED;
            if (!isfinite(s.rz) && s.done != KRYLOV_BREAKDOWN) s.done = KRYLOV_NONFINITE;
        }
        s.rr = rr;
    }
    else
    {
        s.omega = tt > 0.0 ? ts / tt : 0.0;
        s.rr = rr;
        s.aux0 = s.rz; // rho_old for the next iteration
        s.rz = r0r;    // r0 . r, the next iteration's rho unless it restarts
        if (!(rr > s.threshold))
            s.done = KRYLOV_CONVERGED;
        else if (k >= max_it)
            s.done = KRYLOV_LIMIT;
        if (!isfinite(rr)) s.done = KRYLOV_NONFINITE;
    }
    s.it = k;
    s.refine = 0;
}
} // namespace neon_amd
