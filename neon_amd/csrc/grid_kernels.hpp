// Krylov iterations inside one resident grid: a launch runs a batch of whole iterations, its
// workgroups exchanging the dot products (and, with them, the published vector) through device
// memory instead of through kernel boundaries.
//
// What bounds the launch-per-phase loop on small and ordinary systems is not work but the chain
// of launches: four per CG iteration (five to thirteen in BiCGSTAB), each 2.5 to 6 us long at
// any size, plus vector passes that leave the chip between them.  Here a workgroup owns a fixed
// set of rows, keeps its part of the recurrence's vectors in LDS, and an iteration costs the
// matrix product plus two or three exchanges of 1.5 (32 workgroups) to 3 us (256 workgroups).
// Per FP64 CG iteration on neo-Hooke blocks, launches against grid: 375 dofs 20.0 -> 6.1 us,
// 27,783 24.6 -> 7.7, 59,049 26.7 -> 8.7, 117,912 31.9 -> 19.1, 311,469 48.6 -> 29.4, 680,943 72.9
// -> 55.7; with the launches' vector part in one of them (vector_iteration) 50^3 cells 56.7 -> 43.7,
// 64^3 88.3 -> 84.6.
//
// Visibility.  The only data that crosses workgroups are the exchanged scalars and the gathered
// vector p.  Both are written with agent-scope (write-through) stores; a wavefront waits for its
// stores before its workgroup publishes its scalars, and a workgroup reads others' entries of p only
// after it has seen every workgroup's scalars.  The caches of an XCD are not coherent with the
// other XCDs' stores, so no address of p may be read twice with different contents within one
// launch: every iteration of a launch writes p to a buffer of its own (the ring), and the
// launch boundary, which invalidates the caches, lets the ring be used again.  A workgroup's rows
// fill whole 128-byte lines of p, so no line is written by two workgroups.
//
// Progress.  The grid has at most one workgroup per compute unit and the host holds that many
// compute units for it against the other grids of the process (batch by batch where another solve
// waits for some), so all workgroups run at once as soon as ordinary kernels have left room.  Should
// another process keep some of them out, the waiting ones give up after a bounded time, raise the
// abort word and return; every workgroup checks that word when it starts, and the host then solves
// with the launch-per-phase loop, as it does the context's next solves for a while.
#pragma once

#include "spmv_layouts.hpp"

namespace neon_amd
{
constexpr int kGridThreads = 512;
constexpr int kGridWaves = kGridThreads / 64;
constexpr int kGridMaxBlocks = 256; // exchange slots
// 8-byte words per slot (32 bytes): two doubles, each in two words that carry the exchange's number
// in their upper halves, read and written 16 bytes at a time
constexpr int kGridSlotWords = 4;

struct grid_link
{
    uint64_t* slots;    // [2 parities][kGridMaxBlocks][kGridSlotWords]
    krylov_state* mark; // its `done` is the abort word
    uint64_t patience;  // ticks of the 100 MHz counter a wait may take (0: it gives up at once)
    uint32_t epoch;     // number of the launch's first exchange
};

// Rows of a block: `rounds` x (kGridWaves / wps) slices, wps wavefronts sharing one slice
// (sliced layouts), or a run of consecutive rows (CSR).
struct grid_shape
{
    int64_t n = 0;
    int32_t blocks = 0;    // of the grid
    int32_t per_xcd = 0;   // blocks per XCD
    int32_t rounds = 0;    // sliced layouts
    int32_t wps = 1;       // wavefronts per slice: 1, 4 or 8
    int32_t rows = 0;      // rows of a block (capacity)
    bool all = false;      // every vector of the recurrence in LDS
    int64_t lds = 0;       // bytes of dynamic LDS
};

// Sum over the wavefront in a fixed order, the total in every lane (DPP adds within and across
// the rows of 16 lanes, no LDS crossbar).
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v)
{
    int const lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
    int const hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
    return v + __hiloint2double(hi, lo);
}
__device__ inline double wave_total(double v)
{
    v = dpp_add<0x111, 0xf>(v); // row_shr:1
    v = dpp_add<0x112, 0xf>(v); // row_shr:2
    v = dpp_add<0x114, 0xf>(v); // row_shr:4
    v = dpp_add<0x118, 0xf>(v); // row_shr:8
    v = dpp_add<0x142, 0xa>(v); // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v); // row_bcast:31 into rows 2 and 3
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// The thread's index as a value the compiler cannot compute ahead: the unrolled vector phases' row
// addresses would otherwise all be kept in registers across the matrix product
__device__ inline int here(int tid)
{
    asm volatile("" : "+v"(tid));
    return tid;
}

__device__ inline void publish(double* p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Two tagged words at agent scope (past the caches of this XCD) in one access.  Each 8-byte half is
// written and read whole; the tag in each tells whether it has arrived.
typedef uint64_t word2 __attribute__((ext_vector_type(2)));
__device__ inline void store_words(uint64_t* p, uint64_t a, uint64_t b)
{
    word2 const q{a, b};
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(p), "v"(q) : "memory");
}
template <int NV>
__device__ inline void load_words(const uint64_t* p, word2 (&q)[NV])
{
    static_assert(NV == 1 || NV == 2);
    if constexpr (NV == 1)
        asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=&v"(q[0]) : "v"(p) : "memory");
    else
        asm volatile("global_load_dwordx4 %0, %2, off sc1\n\t"
                     "global_load_dwordx4 %1, %2, off offset:16 sc1\n\t"
                     "s_waitcnt vmcnt(0)"
                     : "=&v"(q[0]), "=&v"(q[1])
                     : "v"(p)
                     : "memory");
}

// The exchange of one grid launch by workgroups of WAVES wavefronts.  Every workgroup calls the same
// sequence of exchanges.
template <int WAVES = kGridWaves>
struct grid_exchange
{
    grid_link link;
    int blocks;
    double (*own)[2][WAVES]; // LDS [2 parities]: the wavefronts' sums
    double (*all)[2][WAVES]; // LDS [2 parities]: the sums of the slots each wavefront read
    int* bad;                     // LDS

    // v[k] <- the sum over the grid, in a fixed order, for the values given by every thread; also
    // a barrier: stores published before it are visible to every workgroup after it.  NV = 0:
    // only the barrier.  False when the grid has given up (the caller returns).
    template <int NV>
    __device__ __forceinline__ bool sum(double* v)
    {
        int const tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
        uint32_t const e = link.epoch++;
        int const par = int(e & 1);
        if constexpr (NV > 0)
        {
#pragma unroll
            for (int k = 0; k < NV; ++k)
            {
                double const s = wave_total(v[k]);
                if (lane == 0) own[par][k][wave] = s;
            }
        }
        // this wavefront's published stores are at the coherence point before the workgroup says so
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        double t[NV > 0 ? NV : 1];
        if constexpr (NV > 0)
        {
#pragma unroll
            for (int k = 0; k < NV; ++k)
            {
                t[k] = 0.0;
#pragma unroll
                for (int w = 0; w < WAVES; ++w) t[k] += own[par][k][w];
            }
        }
        if (blocks == 1)
        {
            if constexpr (NV > 0)
#pragma unroll
                for (int k = 0; k < NV; ++k) v[k] = t[k];
            return true;
        }
        uint64_t* const base = link.slots + size_t(par) * kGridMaxBlocks * kGridSlotWords;
        uint64_t const tag = uint64_t(e) << 32;
        if (tid == 0)
        {
            uint64_t* const mine = base + size_t(blockIdx.x) * kGridSlotWords;
            if constexpr (NV > 0)
            {
#pragma unroll
                for (int k = 0; k < NV; ++k)
                {
                    uint64_t const b = uint64_t(__double_as_longlong(t[k]));
                    store_words(mine + 2 * k, tag | (b & 0xffffffffull), tag | (b >> 32));
                }
            }
            else
                store_words(mine, tag, tag);
        }
        int const readers = (blocks + 63) / 64; // wavefronts that read slots
        if (wave < readers)
        {
            int const q = wave * 64 + lane;
            double got[NV > 0 ? NV : 1] = {};
            if (q < blocks)
            {
                const uint64_t* const src = base + size_t(q) * kGridSlotWords;
                word2 w[NV > 1 ? NV : 1];
                uint64_t const start = wall_clock64();
                for (uint32_t spin = 0;; ++spin)
                {
                    load_words(src, w);
                    bool seen = true;
#pragma unroll
                    for (int k = 0; k < (NV > 1 ? NV : 1); ++k)
                        seen = seen && uint32_t(w[k].x >> 32) == e && uint32_t(w[k].y >> 32) == e;
                    if (seen) break;
                    if ((spin & 255u) == 255u || link.patience == 0)
                    {
                        bool const late = wall_clock64() - start >= link.patience;
                        if (late)
                            __hip_atomic_store(&link.mark->done, int32_t(KRYLOV_ABORTED), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                        if (late || __hip_atomic_load(&link.mark->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
                        {
                            *bad = 1;
                            break;
                        }
                    }
                }
                if constexpr (NV > 0)
#pragma unroll
                    for (int k = 0; k < NV; ++k)
                        got[k] = __longlong_as_double(int64_t((w[k].x & 0xffffffffull) | (w[k].y << 32)));
            }
            if constexpr (NV > 0)
#pragma unroll
                for (int k = 0; k < NV; ++k)
                {
                    double const s = wave_total(got[k]);
                    if (lane == 0) all[par][k][wave] = s;
                }
        }
        __syncthreads();
        if (*bad) return false;
        if constexpr (NV > 0)
#pragma unroll
            for (int k = 0; k < NV; ++k)
            {
                v[k] = 0.0;
                for (int w = 0; w < readers; ++w) v[k] += all[par][k][w];
            }
        // the loads of the published vector stay behind the exchange
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        return true;
    }
};

// ------------------------------------------------------------------ the block's rows
// A layout gives a block's local rows (local index -> row of the system, -1 for none) and the
// product's entries for them.  Sliced layouts: local row 192 t + r is row r of the slice in local
// slot t = round * (kGridWaves / wps) + group; wavefronts group * wps ... share a slice's steps.
// XCD x (workgroups with id % 8 = x) takes one contiguous run of the layout's slice order and
// its blocks sweep it together, as the dispatch order of the one-launch product does.
template <typename VT>
struct grid_sym
{
    sym_matrix A;
    const VT* val;
    __device__ int32_t per_xcd() const { return A.slots / 8; }
    __device__ int32_t slice(int x, int32_t e) const { return A.sched[((e >> 2) * 8 + x) * 4 + (e & 3)]; }
    using head = sym_head;
    __device__ head load(int32_t s, int lane) const { return sym_load_head(A, s, lane); }
    template <int STEP, typename XT, typename AT, typename XV>
    __device__ void rows(XV x, head const& h, int lane, int32_t first, bool back, AT& r0, AT& r1, AT& r2) const
    {
        int64_t const i = int64_t(h.s) * 64 + lane;
        int64_t const row = 3 * (i < A.nodes ? i : int64_t(A.nodes) - 1);
        XT xo0 = XT(0), xo1 = XT(0), xo2 = XT(0);
        if (STEP == 1 || first == 0) xo0 = x[row], xo1 = x[row + 1], xo2 = x[row + 2];
        sym_slice_rows<STEP, VT, XT, AT>(A, val, x, h, lane, first, back, xo0, xo1, xo2, r0, r1, r2);
    }
    // A wavefront's share of slice s in registers: of the items (the diagonal record, then the
    // entries) those with index first, first + wps, ...; blocks a lane does not have are zero and
    // their column is the lane's own node
    template <int NP>
    struct kept
    {
        VT v[NP][9], w[NP][9];
        int32_t d[NP], t[NP]; // rows of x for the stored and for the transposed block
    };
    template <int NP>
    __device__ void keep(int32_t s, int lane, int first, int wps, kept<NP>& k) const
    {
        int64_t const i = int64_t(s) * 64 + lane;
        int64_t const ic = s >= 0 && i < A.nodes ? i : int64_t(A.nodes) - 1;
        int32_t const e0 = s >= 0 ? A.eptr[s] : 0, ne = s >= 0 ? A.eptr[s + 1] - e0 : -1;
#pragma unroll
        for (int u = 0; u < NP; ++u)
        {
            int const m = first + u * wps;
            k.d[u] = k.t[u] = int32_t(3 * ic);
#pragma unroll
            for (int q = 0; q < 9; ++q) k.v[u][q] = k.w[u][q] = VT(0);
            if (m > ne) continue;
            if (m == 0)
            {
                const VT* const rec = val + int64_t(A.rdiag[s]) * 576;
#pragma unroll
                for (int q = 0; q < 9; ++q) k.v[u][q] = rec[sell_pos<VT>(q, lane)];
                continue;
            }
            int4v const e = A.ent[e0 + m - 1];
            int64_t const off = e.x, up = i + off, dn = i - off;
            if (e.y >= 0 && up < A.nodes)
            {
                const VT* const rec = val + int64_t(e.y) * 576;
#pragma unroll
                for (int q = 0; q < 9; ++q) k.v[u][q] = rec[sell_pos<VT>(q, lane)];
                k.d[u] = int32_t(3 * up);
            }
            int64_t const sa = (int64_t(s) * 64 - off) >> 6;
            int32_t const rt = (dn >> 6) == sa ? e.z : e.w;
            if (dn >= 0 && dn < A.nodes && rt >= 0)
            {
                const VT* const rec = val + int64_t(rt) * 576;
#pragma unroll
                for (int q = 0; q < 9; ++q) k.w[u][q] = rec[sell_pos<VT>(q, int(dn & 63))];
                k.t[u] = int32_t(3 * dn);
            }
        }
    }
    template <int NP, typename XV, typename AT>
    __device__ static void apply(kept<NP> const& k, XV x, AT& r0, AT& r1, AT& r2)
    {
#pragma unroll
        for (int u = 0; u < NP; ++u)
        {
            AT const x0 = AT(x[k.d[u]]), x1 = AT(x[k.d[u] + 1]), x2 = AT(x[k.d[u] + 2]);
            AT const z0 = AT(x[k.t[u]]), z1 = AT(x[k.t[u] + 1]), z2 = AT(x[k.t[u] + 2]);
            r0 += (AT(k.v[u][0]) * x0 + AT(k.v[u][1]) * x1 + AT(k.v[u][2]) * x2)
                  + (AT(k.w[u][0]) * z0 + AT(k.w[u][3]) * z1 + AT(k.w[u][6]) * z2);
            r1 += (AT(k.v[u][3]) * x0 + AT(k.v[u][4]) * x1 + AT(k.v[u][5]) * x2)
                  + (AT(k.w[u][1]) * z0 + AT(k.w[u][4]) * z1 + AT(k.w[u][7]) * z2);
            r2 += (AT(k.v[u][6]) * x0 + AT(k.v[u][7]) * x1 + AT(k.v[u][8]) * x2)
                  + (AT(k.w[u][2]) * z0 + AT(k.w[u][5]) * z1 + AT(k.w[u][8]) * z2);
        }
    }
};

template <typename VT>
struct grid_sell
{
    sell_matrix A;
    const VT* val;
    // a lane's offset in the step of per-lane offsets `code`
    __device__ int64_t lane_offset(int32_t code, int lane) const
    {
        int64_t const at = int64_t(code) * 64 + lane;
        return A.soff16 ? int64_t(A.soff16[at]) : int64_t(A.soff32[at]);
    }
    __device__ int32_t per_xcd() const { return (A.slices + 7) / 8; }
    __device__ int32_t slice(int x, int32_t e) const
    {
        int32_t const s = x * per_xcd() + e;
        return s < A.slices ? s : -1;
    }
    struct head
    {
        int32_t node, exl, k0, ks;
        int32_t codes, excs; // of the first 64 steps, lane j holding step j's
    };
    __device__ head load(int32_t s, int lane) const
    {
        head h;
        h.node = A.snode[int64_t(s) * 64 + lane];
        h.exl = A.slane[s];
        h.k0 = A.sptr[s];
        h.ks = A.sptr[s + 1] - h.k0;
        h.codes = lane < h.ks ? A.scode[int64_t(h.k0) + lane] : 0;
        h.excs = lane < h.ks ? A.sexc[int64_t(h.k0) + lane] : 0;
        return h;
    }
    // Steps first, first + STEP, ...: four at a time, all their column offsets and then all their
    // operands requested before the first is used (a slice of per-lane offsets would otherwise
    // wait twice per step: 23 us for 180 slices of 24 steps, one wavefront per slice)
    template <int STEP, typename XT, typename AT, typename XV>
    __device__ void rows(XV x, head const& h, int lane, int32_t first, bool back, AT& r0, AT& r1, AT& r2) const
    {
        constexpr int U = 4, W = 16 / int(sizeof(VT));
        typedef VT vec_t __attribute__((ext_vector_type(W)));
        int64_t const nn = h.node >= 0 ? int64_t(h.node) : -1 - int64_t(h.node);
        int const ex0 = h.exl & 0xff, ex1 = (h.exl >> 8) & 0xff;
        int32_t const k0 = h.k0, ks = h.ks;
        // four accumulator sets, one for each of the four steps in flight, added pairwise
        AT a[U][3] = {};
        for (int32_t c = 0; c < ks; c += 64)
        {
            int32_t const c0 = back ? (ks - 1) / 64 * 64 - c : c;
            int32_t const cn = ks - c0 < 64 ? ks - c0 : 64;
            int64_t const base = int64_t(k0) + c0;
            bool const in = lane < cn;
            int32_t const codes = c0 == 0 ? h.codes : in ? A.scode[base + lane] : 0;
            int32_t const excs = c0 == 0 ? h.excs : in ? A.sexc[base + lane] : 0;
            bool const shared = __builtin_amdgcn_readlane(codes, 0) < 0;
            for (int32_t j0 = STEP == 1 ? 0 : first; j0 < cn; j0 += U * STEP)
            {
                int64_t m[U];
                bool on[U];
                int64_t rec[U];
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    int32_t const want = j0 + u * STEP;
                    on[u] = want < cn;
                    // past the end: step j0's operands again, x taken as zero
                    int32_t const j = back ? cn - 1 - (on[u] ? want : j0) : (on[u] ? want : j0);
                    rec[u] = base + j;
                    int32_t const code = __builtin_amdgcn_readlane(codes, j);
                    if (shared)
                    {
                        int32_t const e = __builtin_amdgcn_readlane(excs, j);
                        int64_t const o0 = int16_t(e & 0xffff), o1 = int16_t(uint32_t(e) >> 16);
                        m[u] = nn + (lane == ex0 ? o0 : (lane == ex1 ? o1 : shared_offset(code)));
                    }
                    else
                        m[u] = nn + lane_offset(code, lane);
                }
                VT v[U][9];
                XT xs[U][3];
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    const VT* p = val + rec[u] * 576;
#pragma unroll
                    for (int g = 0; g < 8 / W; ++g)
                    {
                        vec_t const q = *(reinterpret_cast<const vec_t*>(p + g * 64 * W) + lane);
#pragma unroll
                        for (int k = 0; k < W; ++k) v[u][g * W + k] = q[k];
                    }
                    v[u][8] = p[512 + lane];
#pragma unroll
                    for (int k = 0; k < 3; ++k) xs[u][k] = x[3 * m[u] + k];
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    AT const x0 = on[u] ? AT(xs[u][0]) : AT(0), x1 = on[u] ? AT(xs[u][1]) : AT(0),
                             x2 = on[u] ? AT(xs[u][2]) : AT(0);
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        a[u][i] += AT(v[u][3 * i]) * x0 + AT(v[u][3 * i + 1]) * x1 + AT(v[u][3 * i + 2]) * x2;
                }
            }
        }
        r0 = (a[0][0] + a[1][0]) + (a[2][0] + a[3][0]);
        r1 = (a[0][1] + a[1][1]) + (a[2][1] + a[3][1]);
        r2 = (a[0][2] + a[1][2]) + (a[2][2] + a[3][2]);
    }
    // as grid_sym's: the items are the slice's steps (at most 64 of them)
    template <int NP>
    struct kept
    {
        VT v[NP][9];
        int32_t d[NP];
    };
    template <int NP>
    __device__ void keep(int32_t s, int lane, int first, int wps, kept<NP>& k) const
    {
        int32_t const node = s >= 0 ? A.snode[int64_t(s) * 64 + lane] : 0;
        int64_t const nn = node >= 0 ? int64_t(node) : -1 - int64_t(node);
        int32_t const exl = s >= 0 ? A.slane[s] : 0xffff;
        int32_t const k0 = s >= 0 ? A.sptr[s] : 0, ks = s >= 0 ? A.sptr[s + 1] - k0 : 0;
#pragma unroll
        for (int u = 0; u < NP; ++u)
        {
            int const m = first + u * wps;
            k.d[u] = int32_t(3 * nn);
#pragma unroll
            for (int q = 0; q < 9; ++q) k.v[u][q] = VT(0);
            if (m >= ks) continue;
            int32_t const code = A.scode[int64_t(k0) + m], e = A.sexc[int64_t(k0) + m];
            int64_t off;
            if (code < 0)
                off = lane == (exl & 0xff) ? int64_t(int16_t(e & 0xffff))
                                           : (lane == ((exl >> 8) & 0xff) ? int64_t(int16_t(uint32_t(e) >> 16))
                                                                          : shared_offset(code));
            else
                off = lane_offset(code, lane);
            const VT* const rec = val + (int64_t(k0) + m) * 576;
#pragma unroll
            for (int q = 0; q < 9; ++q) k.v[u][q] = rec[sell_pos<VT>(q, lane)];
            k.d[u] = int32_t(3 * (nn + off));
        }
    }
    template <int NP, typename XV, typename AT>
    __device__ static void apply(kept<NP> const& k, XV x, AT& r0, AT& r1, AT& r2)
    {
#pragma unroll
        for (int u = 0; u < NP; ++u)
        {
            AT const x0 = AT(x[k.d[u]]), x1 = AT(x[k.d[u] + 1]), x2 = AT(x[k.d[u] + 2]);
            r0 += AT(k.v[u][0]) * x0 + AT(k.v[u][1]) * x1 + AT(k.v[u][2]) * x2;
            r1 += AT(k.v[u][3]) * x0 + AT(k.v[u][4]) * x1 + AT(k.v[u][5]) * x2;
            r2 += AT(k.v[u][6]) * x0 + AT(k.v[u][7]) * x1 + AT(k.v[u][8]) * x2;
        }
    }
};

// A block's rows on a sliced layout
template <typename LAY>
struct grid_sliced
{
    LAY lay;
    static constexpr bool kSliced = true;
    __device__ void hold(grid_shape const&, const int32_t*) const {}
    // the product's local row lr, after product()
    template <typename AT>
    __device__ AT result(grid_shape const& g, const AT* y, const AT* part, int lr) const
    {
        if (g.wps == 1) return y[lr];
        const AT* const p = part + (lr / 192 * g.wps) * 192 + lr % 192;
        AT s = p[0];
        for (int k = 1; k < g.wps; ++k) s += p[k * 192];
        return s;
    }

    // first_row: the slots' first rows (-1: none)
    __device__ void begin(grid_shape const& g, int32_t* first_row) const
    {
        int const x = blockIdx.x & 7, j = blockIdx.x >> 3;
        int const groups = kGridWaves / g.wps;
        int const slots = g.rounds * groups;
        for (int t = threadIdx.x; t < slots; t += kGridThreads)
        {
            int32_t const e = (t / groups * g.per_xcd + j) * groups + t % groups;
            int32_t const s = e < lay.per_xcd() ? lay.slice(x, e) : -1;
            first_row[t] = s < 0 ? -1 : s * 192;
        }
    }
    __device__ int64_t row(grid_shape const& g, const int32_t* first_row, int lr) const
    {
        int const t = lr / 192;
        int32_t const b = first_row[t];
        if (b < 0) return -1;
        int64_t const r = int64_t(b) + (lr - t * 192);
        return r < g.n ? r : -1;
    }
    template <int WPS, typename XT, typename AT, typename XV>
    __device__ void product_shared(grid_shape const& g, const int32_t* first_row, bool back, XV x, AT* y, AT* part) const
    {
        constexpr int groups = kGridWaves / WPS;
        int const lane = threadIdx.x & 63;
        int const wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
        int const grp = wave / WPS, w = wave % WPS;
        int const count = g.rounds * groups;
        for (int u = grp; u < count; u += groups)
        {
            int const t = back ? count - groups + 2 * grp - u : u;
            int32_t const b = __builtin_amdgcn_readfirstlane(first_row[t]);
            AT r0 = AT(0), r1 = AT(0), r2 = AT(0);
            if (b >= 0) lay.template rows<WPS, XT, AT>(x, lay.load(b / 192, lane), lane, w, back, r0, r1, r2);
            AT* const o = WPS == 1 ? y + t * 192 : part + (t * WPS + w) * 192;
            o[lane * 3] = r0;
            o[lane * 3 + 1] = r1;
            o[lane * 3 + 2] = r2;
        }
        __syncthreads();
    }
    // y[local rows] = A x (result() gives the rows); back: the slices and their items in the opposite order
    template <typename XT, typename AT, typename XV>
    __device__ void product(grid_shape const& g, const int32_t* first_row, bool back, XV x, AT* y, AT* part) const
    {
        switch (g.wps)
        {
        case 1: product_shared<1, XT, AT>(g, first_row, back, x, y, part); break;
        case 4: product_shared<4, XT, AT>(g, first_row, back, x, y, part); break;
        default: product_shared<8, XT, AT>(g, first_row, back, x, y, part); break;
        }
    }
};

// The same for one slice per WPS wavefronts (one round) whose share of the matrix, at most NP
// items per wavefront, stays in registers for the whole launch: an iteration then reads only the
// gathered vectors, which is most of a small product's time (the share's own loads wait for the
// slice's entry range, its entries and its records in turn).
template <typename LAY, int NP, int WPS>
struct grid_kept : grid_sliced<LAY>
{
    typename LAY::template kept<NP> mine;

    __device__ void hold(grid_shape const&, const int32_t* first_row)
    {
        int const lane = threadIdx.x & 63;
        int const wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
        int32_t const b = __builtin_amdgcn_readfirstlane(first_row[wave / WPS]);
        this->lay.template keep<NP>(b < 0 ? -1 : b / 192, lane, wave % WPS, WPS, mine);
    }
    template <typename XT, typename AT, typename XV>
    __device__ void product(grid_shape const&, const int32_t*, bool, XV x, AT*, AT* part) const
    {
        int const lane = threadIdx.x & 63;
        int const wave = threadIdx.x >> 6;
        AT r0 = AT(0), r1 = AT(0), r2 = AT(0);
        LAY::template apply<NP>(mine, x, r0, r1, r2);
        AT* const o = part + wave * 192;
        o[lane * 3] = r0;
        o[lane * 3 + 1] = r1;
        o[lane * 3 + 2] = r2;
        __syncthreads();
    }
    template <typename AT>
    __device__ AT result(grid_shape const&, const AT*, const AT* part, int lr) const
    {
        const AT* const p = part + (lr / 192 * WPS) * 192 + lr % 192;
        AT s = p[0];
#pragma unroll
        for (int k = 1; k < WPS; ++k) s += p[k * 192];
        return s;
    }
};

// A block's rows on the generic CSR layout: a run of g.rows consecutive rows (a multiple of 16),
// the blocks of an XCD adjacent.  Their entries are one contiguous span, taken in chunks of
// kCsrChunk: every thread loads its eight values and columns of a chunk (coalesced, the next
// chunk's while this one is summed), multiplies them with the gathered x into LDS, and four lanes
// add up each row's part of the chunk.  With lanes assigned to rows instead, as in
// spmv_csr_kernel, the dependent loads of one row pointer, its columns and x are paid once per
// four rows: 95 us against 37 us for the launch's 32 wavefronts per compute unit (7.6 M entries).
// A row with more than kCsrLong entries in a chunk is added up by a wavefront (four lanes take 20 us for
// a chunk of one row), in workgroups that have such rows: 20,000 rows, 64 of them full, 12.9 -> 1.3 ms
// per iteration; workgroups without keep the loop without the list (with it 4 % slower at 1 M rows).
constexpr int kCsrPerThread = 8;
constexpr int kCsrLong = 256;
static_assert(kCsrChunk == kGridThreads * kCsrPerThread);
template <typename VT>
struct grid_csr
{
    csr_matrix A;
    const VT* val;
    static constexpr bool kSliced = false;

    __device__ static int64_t first(grid_shape const& g)
    {
        int const b = blockIdx.x;
        int64_t const logical = (g.blocks & 7) == 0 ? int64_t(b & 7) * (g.blocks >> 3) + (b >> 3) : b;
        return logical * g.rows;
    }
    __device__ static int count(grid_shape const& g)
    {
        int64_t const left = g.n - first(g);
        return int(left < g.rows ? (left > 0 ? left : 0) : g.rows);
    }
    // `ptr`: the rows' pointers, count + 1 of them
    __device__ void begin(grid_shape const& g, int32_t* ptr) const
    {
        int const c = count(g);
        int64_t const r0 = c > 0 ? first(g) : 0;
        for (int q = threadIdx.x; q <= c; q += kGridThreads) ptr[q] = A.rp[r0 + q];
    }
    __device__ int64_t row(grid_shape const& g, const int32_t*, int lr) const
    {
        int64_t const r = first(g) + lr;
        return r < g.n ? r : -1;
    }
    // the next chunk's values and columns (-1: none)
    VT v[kCsrPerThread];
    int32_t col[kCsrPerThread];
    __device__ void load(int64_t c0, int64_t end)
    {
#pragma unroll
        for (int u = 0; u < kCsrPerThread; ++u)
        {
            int64_t const p = c0 + u * kGridThreads + int(threadIdx.x);
            bool const on = p < end;
            col[u] = on ? A.ci[p] : -1;
            v[u] = on ? val[p] : VT(0);
        }
    }
    bool any_long; // the block has rows of more than kCsrLong entries
    __device__ void hold(grid_shape const& g, const int32_t* ptr)
    {
        int const c = count(g);
        load(c > 0 ? ptr[0] : 0, c > 0 ? ptr[c] : 0);
        int found = 0;
        for (int q = threadIdx.x; q < c; q += kGridThreads) found |= ptr[q + 1] - ptr[q] > kCsrLong;
        any_long = __syncthreads_or(found) != 0;
    }
    template <typename AT>
    __device__ AT result(grid_shape const&, const AT* y, const AT*, int lr) const
    {
        return y[lr];
    }
    // a block of one chunk keeps it in registers; otherwise the last chunk's turn loads the first again
    template <bool LONG, typename XT, typename AT, typename XV>
    __device__ void chunks(grid_shape const& g, const int32_t* ptr, XV x, AT* y, AT* part)
    {
        __shared__ int next_row, longs, long_row[LONG ? kCsrChunk / kCsrLong : 1];
        int const c = count(g);
        int const tid = threadIdx.x;
        if (LONG && tid == 0) longs = 0;
        for (int q = tid; q < c; q += kGridThreads) y[q] = AT(0);
        int64_t const beg = c > 0 ? ptr[0] : 0, end = c > 0 ? ptr[c] : 0;
        int ra = 0; // the chunk's first row
        for (int64_t c0 = beg; c0 < end; c0 += kCsrChunk)
        {
            XT xs[kCsrPerThread];
#pragma unroll
            for (int u = 0; u < kCsrPerThread; ++u) xs[u] = col[u] >= 0 ? x[col[u]] : XT(0);
#pragma unroll
            for (int u = 0; u < kCsrPerThread; ++u) part[u * kGridThreads + tid] = AT(v[u]) * AT(xs[u]);
            int64_t const c1 = c0 + kCsrChunk < end ? c0 + kCsrChunk : end;
            if (end - beg > kCsrChunk) load(c1 < end ? c1 : beg, end);
            __syncthreads();
            int const sub = tid & 3;
            for (int q = ra + (tid >> 2); q < c; q += kGridThreads / 4)
            {
                int64_t const lo = ptr[q], hi = ptr[q + 1];
                if (lo >= c1) break;
                int const a = int((lo > c0 ? lo : c0) - c0), b = int((hi < c1 ? hi : c1) - c0);
                if (LONG && b - a > kCsrLong)
                {
                    if (sub == 0) long_row[atomicAdd(&longs, 1)] = q;
                }
                else
                {
                    AT s = AT(0);
                    for (int p = a + sub; p < b; p += 4) s += part[p];
                    s += __shfl_xor(s, 1, 64);
                    s += __shfl_xor(s, 2, 64);
                    if (sub == 0 && b > a) y[q] += s;
                }
                // the one row that holds the chunk's last entry
                if (sub == 0 && hi >= c1 && hi > lo) next_row = hi == c1 ? q + 1 : q;
            }
            __syncthreads();
            ra = next_row;
            if constexpr (LONG)
            {
                int const lane = tid & 63, listed = longs;
                for (int k = tid >> 6; k < listed; k += kGridWaves)
                {
                    int const q = long_row[k];
                    int64_t const lo = ptr[q], hi = ptr[q + 1];
                    int const a = int((lo > c0 ? lo : c0) - c0), b = int((hi < c1 ? hi : c1) - c0);
                    AT s = AT(0);
                    for (int p = a + lane; p < b; p += 64) s += part[p];
                    s = wave_total(s);
                    if (lane == 0) y[q] += s;
                }
                __syncthreads();
                if (tid == 0) longs = 0;
            }
        }
        __syncthreads();
    }
    template <typename XT, typename AT, typename XV>
    __device__ void product(grid_shape const& g, const int32_t* ptr, bool, XV x, AT* y, AT* part)
    {
        if (any_long)
            chunks<true, XT, AT>(g, ptr, x, y, part);
        else
            chunks<false, XT, AT>(g, ptr, x, y, part);
    }
};

// ------------------------------------------------------------------------ CG
// Up to `iters` iterations of cg64's Jacobi-PCG (the same recurrence, scalars and stopping rules
// as cg_update_xr_kernel and cg_update_p_kernel, the dot products summed in another fixed order).
// With b the launch starts the solve (x = 0, r = b, p = M^-1 r), else it continues the one in
// *st.  Ring buffer k holds the p of the launch's iteration k; x, r and p leave through global
// memory (p in buffer 0).  A p's place in LDS takes z = M^-1 r once A p is used.  ALL: x and M^-1
// are in LDS too; else they are read from global memory before the exchange of p.Ap, which waits for them.
// A thread handles the local rows tid, tid + kGridThreads, ... (at most kGridElems).
template <bool ALL>
constexpr int kGridElems = ALL ? 8 : 12;

template <typename ROWS, bool ALL>
__global__ __launch_bounds__(kGridThreads) void cg_grid_kernel(ROWS rows, grid_shape g, double* ring, int64_t stride,
                                                               const double* __restrict__ b, double* __restrict__ x,
                                                               double* __restrict__ r, const double* __restrict__ minv,
                                                               krylov_state* st, grid_link link, int iters,
                                                               int criterion, double tol, int max_it)
{
    constexpr int EL = kGridElems<ALL>;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double own[2][2][kGridWaves], all[2][2][kGridWaves];
    __shared__ int bad;
    int const tid = threadIdx.x;
    krylov_state s{};
    if (!b)
    {
        s = *st;
        if (s.done) return;
    }
    if (tid == 0) bad = __hip_atomic_load(&link.mark->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    double* const l_z = reinterpret_cast<double*>(smem); // A p, then z
    double* const l_r = l_z + g.rows;
    double* const l_p = l_r + g.rows;
    double* const l_m = l_p + g.rows;
    double* const l_x = l_m + (ALL ? g.rows : 0);
    double* const part = l_x + (ALL ? g.rows : 0);
    int32_t* const first_row =
        reinterpret_cast<int32_t*>(part + (!ROWS::kSliced ? kCsrChunk : g.wps > 1 ? g.rows * g.wps : 0));
    rows.begin(g, first_row);
    __syncthreads();
    grid_exchange<> ex{link, g.blocks, own, all, &bad};
    if (bad)
    {
        if (blockIdx.x == 0 && tid == 0) st->done = KRYLOV_ABORTED;
        return;
    }
    rows.hold(g, first_row);
    bool alive = true;
    double v[2] = {0.0, 0.0};
    for (int lr = tid; lr < g.rows; lr += kGridThreads)
    {
        int64_t const i = rows.row(g, first_row, lr);
        if (i < 0) continue;
        double const ri = b ? b[i] : r[i], mi = minv[i];
        double const pi = b ? mi * ri : ring[i];
        if (b)
        {
            publish(ring + i, pi);
            v[0] += ri * ri;
            v[1] += ri * pi;
            if constexpr (!ALL) x[i] = 0.0;
        }
        l_r[lr] = ri;
        l_p[lr] = pi;
        if constexpr (ALL)
        {
            l_m[lr] = mi;
            l_x[lr] = b ? 0.0 : x[i];
        }
    }
    if (b)
    {
        alive = ex.sum<2>(v);
        if (alive) s = cg_first_state(v[0], v[1], criterion, tol, max_it);
        if (s.done) iters = 0;
    }
    else
        __syncthreads(); // l_p whole before a lone workgroup gathers from it (the exchange is that barrier otherwise)
    for (int k = 0; alive && k < iters; ++k)
    {
        if (!ROWS::kSliced && g.blocks == 1) // local rows are the system's: p is gathered from LDS
            rows.template product<double, double>(g, first_row, false, static_cast<const double*>(l_p), l_z, part);
        else
            rows.template product<double, double>(g, first_row, (k & 1) != 0, ring + int64_t(k) * stride, l_z, part);
        v[0] = 0.0;
        int t = here(tid);
        double mi[ALL ? 1 : EL], xi[ALL ? 1 : EL];
#pragma unroll
        for (int e = 0; e < EL; ++e)
        {
            int const lr = t + e * kGridThreads;
            if (lr >= g.rows) break;
            int64_t const i = rows.row(g, first_row, lr);
            if (i < 0) continue;
            if constexpr (!ALL)
            {
                mi[e] = minv[i];
                xi[e] = x[i];
            }
            double const ap = rows.result(g, l_z, part, lr);
            if (!ROWS::kSliced || g.wps > 1) l_z[lr] = ap;
            v[0] += l_p[lr] * ap;
        }
        alive = ex.sum<1>(v);
        if (!alive) break;
        double const alpha = s.rz / v[0];
        v[0] = v[1] = 0.0;
        t = here(tid);
#pragma unroll
        for (int e = 0; e < EL; ++e)
        {
            int const lr = t + e * kGridThreads;
            if (lr >= g.rows) break;
            int64_t const i = rows.row(g, first_row, lr);
            if (i < 0) continue;
            double const ri = l_r[lr] - alpha * l_z[lr];
            double const zi = (ALL ? l_m[lr] : mi[ALL ? 0 : e]) * ri;
            l_r[lr] = ri;
            l_z[lr] = zi;
            v[0] += ri * ri;
            v[1] += ri * zi;
        }
        alive = ex.sum<2>(v);
        if (!alive) break;
        // x moves here, behind the exchange: its stores would have to reach memory before it
        double const beta = cg_decide(s, v[0], v[1], criterion, tol, max_it);
        bool const last = k + 1 == iters;
        double* const next = last ? ring : ring + int64_t(k + 1) * stride;
        t = here(tid);
#pragma unroll
        for (int e = 0; e < EL; ++e)
        {
            int const lr = t + e * kGridThreads;
            if (lr >= g.rows) break;
            int64_t const i = rows.row(g, first_row, lr);
            if (i < 0) continue;
            double const old = l_p[lr];
            double const pi = l_z[lr] + beta * old;
            l_p[lr] = pi;
            if (!s.done && (ROWS::kSliced || g.blocks > 1 || last)) publish(next + i, pi);
            if constexpr (ALL)
                l_x[lr] += alpha * old;
            else
                x[i] = xi[e] + alpha * old;
        }
        if (s.done) break;
        if (!last)
        {
            alive = ex.sum<0>(v);
            if (!alive) break;
        }
    }
    if (alive)
        for (int lr = tid; lr < g.rows; lr += kGridThreads)
        {
            int64_t const i = rows.row(g, first_row, lr);
            if (i < 0) continue;
            r[i] = l_r[lr];
            if constexpr (ALL) x[i] = l_x[lr];
        }
    if (blockIdx.x == 0 && tid == 0)
    {
        if (!alive) s.done = KRYLOV_ABORTED;
        *st = s;
    }
}

// p = z + beta p_old formed where it is gathered
struct gathered_p
{
    const double* z;
    const double* p_old;
    double beta;
    __device__ double operator[](int64_t i) const { return __builtin_fma(beta, p_old[i], z[i]); }
};

// The same for small blocks (at most kGridFew rows per thread), with two exchanges per iteration
// instead of three: the product forms p = z + beta p_old from the two published vectors where it
// gathers them, so no barrier has to follow beta, at twice the gathered entries (worth it while an
// exchange, 1.3 to 3 us, costs more than they do).  The vectors of the recurrence stay in
// registers.  Ring buffers 2 k and 2 k + 1 hold the z and the p of the launch's iteration k; the
// solve enters and leaves with p in buffer 0.
constexpr int kGridFew = 3;
template <typename ROWS>
__global__ __launch_bounds__(kGridThreads) void cg_grid_small_kernel(ROWS rows, grid_shape g, double* ring,
                                                                     int64_t stride, const double* __restrict__ b,
                                                                     double* __restrict__ x, double* __restrict__ r,
                                                                     const double* __restrict__ minv, krylov_state* st,
                                                                     grid_link link, int iters, int criterion,
                                                                     double tol, int max_it)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double own[2][2][kGridWaves], all[2][2][kGridWaves];
    __shared__ int bad;
    int const tid = threadIdx.x;
    krylov_state s{};
    if (!b)
    {
        s = *st;
        if (s.done) return;
    }
    if (tid == 0) bad = __hip_atomic_load(&link.mark->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    double* const Ap = reinterpret_cast<double*>(smem);
    double* const part = Ap + g.rows;
    int32_t* const first_row =
        reinterpret_cast<int32_t*>(part + (!ROWS::kSliced ? kCsrChunk : g.wps > 1 ? g.rows * g.wps : 0));
    rows.begin(g, first_row);
    __syncthreads();
    grid_exchange<> ex{link, g.blocks, own, all, &bad};
    if (bad)
    {
        if (blockIdx.x == 0 && tid == 0) st->done = KRYLOV_ABORTED;
        return;
    }
    rows.hold(g, first_row);
    bool alive = true;
    double v[2] = {0.0, 0.0};
    int64_t row[kGridFew];
    double ri[kGridFew], mi[kGridFew], pi[kGridFew], xi[kGridFew], zi[kGridFew];
#pragma unroll
    for (int e = 0; e < kGridFew; ++e)
    {
        int const lr = tid + e * kGridThreads;
        row[e] = lr < g.rows ? rows.row(g, first_row, lr) : -1;
        ri[e] = mi[e] = pi[e] = xi[e] = zi[e] = 0.0;
        if (row[e] < 0) continue;
        ri[e] = b ? b[row[e]] : r[row[e]];
        mi[e] = minv[row[e]];
        pi[e] = b ? mi[e] * ri[e] : ring[row[e]];
        xi[e] = b ? 0.0 : x[row[e]];
        zi[e] = pi[e];
        if (b)
        {
            publish(ring + row[e], pi[e]);
            v[0] += ri[e] * ri[e];
            v[1] += ri[e] * pi[e];
        }
    }
    if (b)
    {
        alive = ex.sum<2>(v);
        if (alive) s = cg_first_state(v[0], v[1], criterion, tol, max_it);
        if (s.done) iters = 0;
    }
    double beta = 0.0;
    for (int k = 0; alive && k < iters; ++k)
    {
        double* const z = ring + int64_t(2 * k) * stride;
        double* const p = z + stride;
        if (k > 0)
        {
#pragma unroll
            for (int e = 0; e < kGridFew; ++e)
            {
                if (row[e] < 0) continue;
                pi[e] = __builtin_fma(beta, pi[e], zi[e]);
                publish(p + row[e], pi[e]);
            }
        }
        // iteration 0: buffer 0 is p itself; iteration 1: its p_old is that buffer
        gathered_p const gp{z, k == 0 ? z : k == 1 ? ring : p - 2 * stride, beta};
        rows.template product<double, double>(g, first_row, (k & 1) != 0, gp, Ap, part);
        v[0] = 0.0;
        double ap[kGridFew];
#pragma unroll
        for (int e = 0; e < kGridFew; ++e)
        {
            ap[e] = row[e] >= 0 ? rows.result(g, Ap, part, tid + e * kGridThreads) : 0.0;
            v[0] += pi[e] * ap[e];
        }
        alive = ex.sum<1>(v);
        if (!alive) break;
        double const alpha = s.rz / v[0];
        v[0] = v[1] = 0.0;
        bool const last = k + 1 == iters;
#pragma unroll
        for (int e = 0; e < kGridFew; ++e)
        {
            if (row[e] < 0) continue;
            xi[e] += alpha * pi[e];
            ri[e] -= alpha * ap[e];
            zi[e] = mi[e] * ri[e];
            v[0] += ri[e] * ri[e];
            v[1] += ri[e] * zi[e];
            if (!last) publish(z + 2 * stride + row[e], zi[e]);
        }
        alive = ex.sum<2>(v);
        if (!alive) break;
        beta = cg_decide(s, v[0], v[1], criterion, tol, max_it);
        if (s.done) break;
    }
    if (alive)
#pragma unroll
        for (int e = 0; e < kGridFew; ++e)
        {
            if (row[e] < 0) continue;
            r[row[e]] = ri[e];
            x[row[e]] = xi[e];
            if (iters > 0) ring[row[e]] = __builtin_fma(beta, pi[e], zi[e]);
        }
    if (blockIdx.x == 0 && tid == 0)
    {
        if (!alive) s.done = KRYLOV_ABORTED;
        *st = s;
    }
}

// ------------------------------------------------------------------ BiCGSTAB
// Up to `iters` iterations of bicgstab64's Jacobi-BiCGSTAB with both stopping rules (the recurrence
// and scalars of the bicg_* kernels, the dot products summed in another fixed order): five
// exchanges per iteration (one carries only p_hat) in place of nine to thirteen launches.
// first: the launch starts the solve (x = 0, r = r0 = b, p = v = 0), else it continues the one in
// *st.  Ring buffers 3 k, 3 k + 1 and 3 k + 2 take p_hat, s_hat and, at a restart of the Eigen rule,
// x of the launch's iteration k.  All vectors are in LDS; x, r, r0, p and v leave through global
// memory.
constexpr int kGridBicgVectors = 8;
template <typename ROWS>
__global__ __launch_bounds__(kGridThreads) void bicg_grid_kernel(ROWS rows, grid_shape g, double* ring, int64_t stride,
                                                                 const double* __restrict__ b, double* __restrict__ x,
                                                                 double* __restrict__ r, double* __restrict__ r0,
                                                                 double* __restrict__ p, double* __restrict__ v,
                                                                 const double* __restrict__ minv, krylov_state* st,
                                                                 grid_link link, int first, int iters, int cuda_rule,
                                                                 double tol, int max_it)
{
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double own[2][2][kGridWaves], all[2][2][kGridWaves];
    __shared__ int bad;
    int const tid = threadIdx.x;
    krylov_state s{};
    if (!first)
    {
        s = *st;
        if (s.done) return;
    }
    if (tid == 0) bad = __hip_atomic_load(&link.mark->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    double* const l_y = reinterpret_cast<double*>(smem); // a product's rows
    double* const l_r = l_y + g.rows;                    // r, and s between the two products
    double* const l_r0 = l_r + g.rows;
    double* const l_p = l_r0 + g.rows;
    double* const l_v = l_p + g.rows;
    double* const l_x = l_v + g.rows;
    double* const l_m = l_x + g.rows;
    double* const l_b = l_m + g.rows;
    double* const part = l_b + g.rows;
    int32_t* const first_row =
        reinterpret_cast<int32_t*>(part + (!ROWS::kSliced ? kCsrChunk : g.wps > 1 ? g.rows * g.wps : 0));
    rows.begin(g, first_row);
    __syncthreads();
    grid_exchange<> ex{link, g.blocks, own, all, &bad};
    if (bad)
    {
        if (blockIdx.x == 0 && tid == 0) st->done = KRYLOV_ABORTED;
        return;
    }
    rows.hold(g, first_row);
    // f(local row, row) over the thread's rows
    auto each = [&](auto f) {
        for (int lr = tid; lr < g.rows; lr += kGridThreads)
        {
            int64_t const i = rows.row(g, first_row, lr);
            if (i >= 0) f(lr, i);
        }
    };
    double d[2] = {0.0, 0.0};
    each([&](int lr, int64_t i) {
        double const bi = b[i];
        l_b[lr] = bi;
        l_m[lr] = minv[i];
        l_r[lr] = first ? bi : r[i];
        l_r0[lr] = first ? bi : r0[i];
        l_p[lr] = first ? 0.0 : p[i];
        l_v[lr] = first ? 0.0 : v[i];
        l_x[lr] = first ? 0.0 : x[i];
        d[0] += bi * bi;
    });
    bool alive = true;
    if (first)
    {
        alive = ex.sum<1>(d);
        if (alive) s = bicg_first_state(d[0], cuda_rule, tol, max_it);
        if (s.done) iters = 0;
    }
    for (int k = 0; alive && k < iters; ++k)
    {
        double* const p_hat = ring + int64_t(3 * k) * stride;
        double* const s_hat = p_hat + stride;
        if (!cuda_rule && bicg_restart_due(s))
        {
            double* const xs = s_hat + stride;
            each([&](int lr, int64_t i) { publish(xs + i, l_x[lr]); });
            alive = ex.sum<0>(d);
            if (!alive) break;
            rows.template product<double, double>(g, first_row, false, xs, l_y, part);
            d[0] = 0.0;
            each([&](int lr, int64_t) {
                double const ri = l_b[lr] - rows.result(g, l_y, part, lr);
                l_r[lr] = ri;
                l_r0[lr] = ri;
                d[0] += ri * ri;
            });
            alive = ex.sum<1>(d);
            if (!alive) break;
            bicg_restarted(s, d[0]);
        }
        {
            bool const plain = cuda_rule && s.it == 0;
            double const beta = (s.rz / s.aux0) * (s.alpha / s.omega), omega = s.omega;
            each([&](int lr, int64_t i) {
                double const pi = plain ? l_r[lr] : l_r[lr] + beta * (l_p[lr] - omega * l_v[lr]);
                l_p[lr] = pi;
                publish(p_hat + i, l_m[lr] * pi);
            });
        }
        alive = ex.sum<0>(d);
        if (!alive) break;
        rows.template product<double, double>(g, first_row, false, p_hat, l_y, part);
        d[0] = 0.0;
        each([&](int lr, int64_t) {
            double const vi = rows.result(g, l_y, part, lr);
            l_v[lr] = vi;
            d[0] += l_r0[lr] * vi;
        });
        alive = ex.sum<1>(d);
        if (!alive) break;
        double const alpha = s.rz / d[0];
        d[0] = 0.0;
        each([&](int lr, int64_t i) {
            double const si = l_r[lr] - alpha * l_v[lr];
            l_r[lr] = si;
            publish(s_hat + i, l_m[lr] * si);
            d[0] += si * si;
        });
        alive = ex.sum<1>(d);
        if (!alive) break;
        s.alpha = alpha;
        s.aux1 = sqrt(d[0]);
        s.refine = cuda_rule && sqrt(d[0]) < tol ? 1 : 0;
        if (s.refine)
        {
            each([&](int lr, int64_t) { l_x[lr] += alpha * (l_m[lr] * l_p[lr]); });
            bicg_decide(s, 0.0, 0.0, 0.0, 0.0, cuda_rule, tol, max_it);
            break;
        }
        rows.template product<double, double>(g, first_row, true, s_hat, l_y, part);
        d[0] = d[1] = 0.0;
        each([&](int lr, int64_t) {
            double const ti = rows.result(g, l_y, part, lr);
            if (!ROWS::kSliced || g.wps > 1) l_y[lr] = ti;
            d[0] += ti * l_r[lr];
            d[1] += ti * ti;
        });
        alive = ex.sum<2>(d);
        if (!alive) break;
        double const ts = d[0], tt = d[1];
        double const omega = cuda_rule ? ts / tt : (tt > 0.0 ? ts / tt : 0.0);
        d[0] = d[1] = 0.0;
        each([&](int lr, int64_t) {
            double const ph = l_m[lr] * l_p[lr], sh = l_m[lr] * l_r[lr];
            if (cuda_rule)
            {
                // x = x + alpha p_hat + omega s_hat as two updates (the two cublasDaxpy calls)
                double const xi = l_x[lr] + alpha * ph;
                l_x[lr] = xi + omega * sh;
            }
            else
                l_x[lr] += alpha * ph + omega * sh; // x += (alpha y + w z)
            double const ri = l_r[lr] - omega * l_y[lr];
            l_r[lr] = ri;
            d[0] += l_r0[lr] * ri;
            d[1] += ri * ri;
        });
        alive = ex.sum<2>(d);
        if (!alive) break;
        bicg_decide(s, ts, tt, d[0], d[1], cuda_rule, tol, max_it);
        if (s.done) break;
    }
    if (alive)
        each([&](int lr, int64_t i) {
            x[i] = l_x[lr];
            r[i] = l_r[lr];
            r0[i] = l_r0[lr];
            p[i] = l_p[lr];
            v[i] = l_v[lr];
        });
    if (blockIdx.x == 0 && tid == 0)
    {
        if (!alive) s.done = KRYLOV_ABORTED;
        *st = s;
    }
}

// ------------------------------------------------------- the vector part of an iteration
// The scalars and vectors of one iteration between two products of the launch loops, in one launch
// in place of three (totals, r update, x and p update): the total of p.Ap from the product's partials,
// r -= alpha A p with r.z (and r.r), the exchange of those sums, and x += alpha p, p = z + beta p.  r
// stays in registers between the two halves, as do x and p (read before the exchange, which waits for
// them: 31 us at 1.6 M dofs, 102 MB that a copy moves in 17): 7 vector passes instead of 8 (FP32 on the
// Jacobi-scaled copy, z = r), 8 instead of 10 (FP64).  One workgroup per compute unit; a thread's
// elements past its kVectorKeep groups are read again.  DECIDE: the scalar rules of the loop, s <- the
// next state, returns beta.
constexpr int kVectorThreads = 1024;
constexpr int kVectorKeep = 3; // 16-byte groups of each vector that a thread keeps

template <typename T, bool PRECOND, bool RR, typename DECIDE>
__device__ __forceinline__ void vector_iteration(int64_t n, T* __restrict__ r, const T* __restrict__ Ap,
                                                 const T* __restrict__ minv, T* __restrict__ x, T* __restrict__ p,
                                                 const double* __restrict__ part_pAp, int npart,
                                                 const krylov_state* __restrict__ st, krylov_state* __restrict__ st_next,
                                                 grid_link link, DECIDE decide)
{
    constexpr int W = 16 / int(sizeof(T)), WAVES = kVectorThreads / 64;
    typedef T vec_t __attribute__((ext_vector_type(W)));
    __shared__ double own[2][2][WAVES], all[2][2][WAVES];
    __shared__ int bad;
    int const tid = threadIdx.x;
    krylov_state s = *st;
    if (s.done)
    {
        if (blockIdx.x == 0 && tid == 0) *st_next = s;
        return;
    }
    if (tid == 0) bad = __hip_atomic_load(&link.mark->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    double const alpha_d = s.rz / reduce_partials<kVectorThreads>(part_pAp, npart); // a barrier for `bad` too
    T const alpha = T(alpha_d);
    if (bad)
    {
        if (blockIdx.x == 0 && tid == 0)
        {
            s.done = KRYLOV_ABORTED;
            *st_next = s;
        }
        return;
    }
    grid_exchange<WAVES> ex{link, int(gridDim.x), own, all, &bad};
    int64_t beg, end;
    xcd_chunk_aligned<W>(n, beg, end);
    int64_t const full = beg + (end - beg) / W * W;
    double v[2] = {0.0, 0.0};
    // element of r -> its new value, its products into the sums
    auto half1 = [&](T ri, T api, T mi) {
        ri = ri - alpha * api;
        if constexpr (PRECOND)
        {
            T const zi = mi * ri;
            v[0] += double(ri) * double(zi);
            if constexpr (RR) v[1] += double(ri) * double(ri);
        }
        else
            v[0] += double(ri) * double(ri);
        return ri;
    };
    vec_t rk[kVectorKeep], xk[kVectorKeep], pk[kVectorKeep], mk[kVectorKeep];
#pragma unroll
    for (int g = 0; g < kVectorKeep; ++g)
    {
        int64_t const i = beg + (int64_t(g) * kVectorThreads + tid) * W;
        if (i >= full) break;
        rk[g] = *reinterpret_cast<const vec_t*>(r + i);
        vec_t const av = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(Ap + i));
        if constexpr (PRECOND) mk[g] = *reinterpret_cast<const vec_t*>(minv + i);
        xk[g] = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(x + i));
        pk[g] = *reinterpret_cast<const vec_t*>(p + i);
#pragma unroll
        for (int k = 0; k < W; ++k) rk[g][k] = half1(rk[g][k], av[k], PRECOND ? mk[g][k] : T(1));
    }
    for (int64_t i = beg + (int64_t(kVectorKeep) * kVectorThreads + tid) * W; i < full; i += kVectorThreads * W)
    {
        vec_t rv = *reinterpret_cast<const vec_t*>(r + i);
        vec_t const av = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(Ap + i));
        vec_t mv{};
        if constexpr (PRECOND) mv = *reinterpret_cast<const vec_t*>(minv + i);
#pragma unroll
        for (int k = 0; k < W; ++k) rv[k] = half1(rv[k], av[k], PRECOND ? mv[k] : T(1));
        *reinterpret_cast<vec_t*>(r + i) = rv;
    }
    // the last entries of the system, fewer than W
    for (int64_t i = full + tid; i < end; i += kVectorThreads) r[i] = half1(r[i], Ap[i], PRECOND ? minv[i] : T(1));
    if (!ex.template sum<RR ? 2 : 1>(v))
    {
        if (blockIdx.x == 0 && tid == 0)
        {
            s.done = KRYLOV_ABORTED;
            *st_next = s;
        }
        return;
    }
    T const beta = T(decide(s, v[1], v[0]));
    bool const more = s.done == KRYLOV_RUNNING;
#pragma unroll
    for (int g = 0; g < kVectorKeep; ++g)
    {
        int64_t const i = beg + (int64_t(g) * kVectorThreads + tid) * W;
        if (i >= full) break;
        *reinterpret_cast<vec_t*>(r + i) = rk[g];
        vec_t xv = xk[g], pv = pk[g];
#pragma unroll
        for (int k = 0; k < W; ++k)
        {
            xv[k] = xv[k] + alpha * pv[k];
            pv[k] = (PRECOND ? mk[g][k] * rk[g][k] : rk[g][k]) + beta * pv[k];
        }
        __builtin_nontemporal_store(xv, reinterpret_cast<vec_t*>(x + i));
        if (more) *reinterpret_cast<vec_t*>(p + i) = pv;
    }
    for (int64_t i = beg + (int64_t(kVectorKeep) * kVectorThreads + tid) * W; i < full; i += kVectorThreads * W)
    {
        vec_t const rv = *reinterpret_cast<const vec_t*>(r + i);
        vec_t xv = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(x + i));
        vec_t pv = *reinterpret_cast<const vec_t*>(p + i), mv{};
        if constexpr (PRECOND) mv = *reinterpret_cast<const vec_t*>(minv + i);
#pragma unroll
        for (int k = 0; k < W; ++k)
        {
            xv[k] = xv[k] + alpha * pv[k];
            pv[k] = (PRECOND ? mv[k] * rv[k] : rv[k]) + beta * pv[k];
        }
        __builtin_nontemporal_store(xv, reinterpret_cast<vec_t*>(x + i));
        if (more) *reinterpret_cast<vec_t*>(p + i) = pv;
    }
    for (int64_t i = full + tid; i < end; i += kVectorThreads)
    {
        T const pi = p[i];
        x[i] = x[i] + alpha * pi;
        if (more) p[i] = (PRECOND ? minv[i] * r[i] : r[i]) + beta * pi;
    }
    if (blockIdx.x == 0 && tid == 0) *st_next = s;
}

// FP64 CG (cg_update_xr_kernel and cg_update_p_kernel)
__global__ __launch_bounds__(kVectorThreads) void cg_vector_kernel(int64_t n, double* r, const double* Ap,
                                                                   const double* minv, double* x, double* p,
                                                                   const double* part_pAp, int npart,
                                                                   const krylov_state* st, krylov_state* st_next,
                                                                   grid_link link, int criterion, double tol,
                                                                   int max_it);
// mixed CG on the Jacobi-scaled copy, an iteration without a reliable update
// (mixed_update_xr_kernel<true, false> and mixed_update_p_kernel<true> with decided = 0)
__global__ __launch_bounds__(kVectorThreads) void mixed_vector_kernel(int64_t n, float* r, const float* Ap, float* x,
                                                                      float* p, const double* part_pAp, int npart,
                                                                      const krylov_state* st, krylov_state* st_next,
                                                                      grid_link link, int max_it);
} // namespace neon_amd
