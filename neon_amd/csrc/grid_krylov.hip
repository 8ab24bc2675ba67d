// Host side of the resident-grid Krylov loops (grid_kernels.hpp): which solves take them, the
// shape of their grids, and the compute units they hold.
#include "engine.hpp"
#include "grid_kernels.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>

namespace neon_amd
{
__global__ __launch_bounds__(kVectorThreads) void cg_vector_kernel(int64_t n, double* r, const double* Ap,
                                                                   const double* minv, double* x, double* p,
                                                                   const double* part_pAp, int npart,
                                                                   const krylov_state* st, krylov_state* st_next,
                                                                   grid_link link, int criterion, double tol,
                                                                   int max_it)
{
    vector_iteration<double, true, true>(n, r, Ap, minv, x, p, part_pAp, npart, st, st_next, link,
                                         [&](krylov_state& s, double rr, double rz) {
                                             return cg_decide(s, rr, rz, criterion, tol, max_it);
                                         });
}

__global__ __launch_bounds__(kVectorThreads) void mixed_vector_kernel(int64_t n, float* r, const float* Ap, float* x,
                                                                      float* p, const double* part_pAp, int npart,
                                                                      const krylov_state* st, krylov_state* st_next,
                                                                      grid_link link, int max_it)
{
    vector_iteration<float, false, false>(n, r, Ap, nullptr, x, p, part_pAp, npart, st, st_next, link,
                                          [&](krylov_state& s, double, double rz) {
                                              double const beta = rz / s.rz;
                                              int32_t const it = s.it + 1;
                                              s.done = it >= max_it ? KRYLOV_LIMIT : KRYLOV_RUNNING;
                                              if (!isfinite(rz)) s.done = KRYLOV_NONFINITE;
                                              s.rz = rz;
                                              s.it = it;
                                              s.refine = 0;
                                              return beta;
                                          });
}

namespace
{
constexpr int64_t kGridLds = 160 * 1024 - 1024; // LDS of a compute unit less the static arrays
} // namespace

// Compute units of each GPU that this process's resident grids may still take.  A grid's
// workgroups wait for each other, so two grids that together exceed the GPU must not be in flight at
// once; a solve waits here until the ones before it have left enough room, in the order of arrival.
class unit_pool
{
public:
    static unit_pool& of(int device)
    {
        static unit_pool pools[kDevices];
        return pools[device];
    }
    static constexpr int kDevices = 64;
    void take(int want, int units)
    {
        {
            std::unique_lock<std::mutex> lock(m_);
            uint64_t const ticket = arrived_++;
            cv_.wait(lock, [&] { return served_ == ticket && used_ + want <= units; });
            ++served_;
            used_ += want;
        }
        cv_.notify_all(); // the next in the queue may fit too
    }
    void give(int count)
    {
        {
            std::lock_guard<std::mutex> lock(m_);
            used_ -= count;
        }
        cv_.notify_all();
    }
    bool waited_for() const { return arrived_ != served_; }

private:
    std::mutex m_;
    std::condition_variable cv_;
    int used_ = 0;
    std::atomic<uint64_t> arrived_{0}, served_{0};
};

unit_hold::unit_hold(int device, int blocks, int units)
    : pool_(unit_pool::of(device)), count_(held(blocks, units)), units_(units)
{
    pool_.take(count_, units_);
}
unit_hold::~unit_hold() { pool_.give(count_); }
bool unit_hold::wanted() const { return pool_.waited_for(); }
void unit_hold::yield()
{
    pool_.give(count_);
    pool_.take(count_, units_);
}

namespace
{
// The vectors of a loop's recurrence: all of them in LDS, or the fewest that must be (0: all), and the
// most rows per thread in either case
struct vector_need
{
    int all, all_rows, least, least_rows;
};
constexpr vector_need kCgNeed{5, kGridElems<true>, 3, kGridElems<false>};
constexpr vector_need kBicgNeed{kGridBicgVectors, 64, 0, 0};

bool fit_lds(grid_shape& g, int64_t extra, vector_need need)
{
    for (bool all : {true, false})
    {
        if (!all && need.least == 0) break;
        int64_t const bytes = int64_t(g.rows) * 8 * (all ? need.all : need.least) + extra;
        if (bytes > kGridLds || g.rows > kGridThreads * (all ? need.all_rows : need.least_rows)) continue;
        g.all = all;
        g.lds = bytes;
        return true;
    }
    return false;
}

// Shape of a sliced layout's grid: per_xcd slices on each XCD's list with `mean` records or entries
// per slice, at most `most_items`.  Its cost is counted in items that a wavefront takes in turn, two
// more for each round (a slice's head and the sums of its shares); a wavefront that has a slice to
// itself waits for the longest slice.  Sharing a slice among wavefronts spreads few slices over all
// compute units and evens out slices of unequal length; without need it only adds rounds (41 x 40 x
// 38 cells, 1,050 slices: 14.4 us per product with one wavefront per slice, 15.1 with eight).
bool shape_sliced(grid_shape& g, int64_t n, int32_t per_xcd, double mean, int32_t most_items, int units,
                  vector_need need)
{
    int const most = std::min(units, kGridMaxBlocks) / 8; // blocks per XCD
    if (most < 1 || per_xcd < 1) return false;
    double best = 0.0;
    for (int wps : {1, 4, 8})
    {
        grid_shape t;
        int const groups = kGridWaves / wps;
        t.n = n;
        t.wps = wps;
        t.rounds = (per_xcd + groups * most - 1) / (groups * most);
        if (wps == 4 && t.rounds > 1) continue;
        // from four rounds on the launches' own dispatch spreads the slices better and the grid's
        // exchanges no longer outweigh that: 1,073,733 dofs 96.6 us per iteration against 105.1 by
        // launches, 1,215,672 dofs 130.8 against 123.0; at three rounds if they are not full or their
        // slices unequal (the items that every wavefront waits for against those there are): 815,409
        // dofs 82.0 against 79.6, long bars on the full copy 960,048 dofs 135 against 126, 1,026,027 dofs
        // 150 against 120; full ones on the full copy 1,029,000 dofs 151 against 157
        if (t.rounds > 3 && wps == 1) continue;
        if (t.rounds == 3 && wps == 1
            && t.rounds * (2.0 + most_items) > 1.4 * (2.0 + mean) * per_xcd / (groups * most))
            continue;
        t.per_xcd = std::min(most, (per_xcd + groups - 1) / groups);
        t.blocks = 8 * t.per_xcd;
        t.rows = t.rounds * groups * 192;
        double const cost = t.rounds * (2.0 + (wps == 1 ? most_items : mean / wps));
        int64_t const extra = (wps > 1 ? int64_t(t.rows) * wps * 8 : 0) + int64_t(t.rounds) * groups * 4;
        if (best > 0.0 && cost >= best) continue;
        if (!fit_lds(t, extra, need)) continue;
        best = cost;
        g = t;
    }
    return best > 0.0;
}

// Shape of a CSR grid: at least 64 rows per block.  A system of at most two chunks of entries takes
// one block, whose exchanges stay within the workgroup and which gathers p from LDS (210 rows, 3,952
// entries: 3.4 us per iteration against 5.6 with four blocks).
int64_t csr_rows(int64_t n, int64_t nnz, int units)
{
    int64_t const most = std::min(units, kGridMaxBlocks);
    int64_t const rows = nnz <= 2 * kCsrChunk && n <= 2 * kGridThreads ? n : std::max<int64_t>(64, (n + most - 1) / most);
    return (rows + 15) / 16 * 16;
}

bool shape_csr(grid_shape& g, int64_t n, int64_t nnz, int units, vector_need need)
{
    int64_t const rows = csr_rows(n, nnz, units);
    if (rows > 64 * kGridThreads) return false;
    g.n = n;
    g.rows = int32_t(rows);
    g.blocks = int32_t((n + rows - 1) / rows);
    return fit_lds(g, kCsrChunk * 8 + 4 * (rows + 1), need);
}

// Every solve sets the same limit: another thread may launch the kernel with more LDS than this one needs
template <typename K>
void allow_lds(K kernel)
{
    NEON_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       int(kGridLds)));
}

sym_matrix sym_of(linear_operator const& A)
{
    return sym_matrix{A.nodes,     A.slices,   A.sym_slots,
                      A.sym_records, A.sym_sched, A.sym_rdiag,
                      A.sym_eptr,  reinterpret_cast<const int4v*>(A.sym_ent),
                      A.sym_rslice, A.sym_roff};
}

sell_matrix sell_of(linear_operator const& A)
{
    return sell_matrix{A.nodes, A.slices, A.sptr, A.snode, A.slane, A.scode, A.sexc, A.soff16, A.soff32};
}

bool shape_of(grid_shape& g, linear_operator const& A, int units, vector_need need)
{
    if (A.node_block && A.sym)
        return shape_sliced(g, A.n, A.sym_slots / 8, 1.0 + A.sym_mean, 1 + A.sym_entries, units, need);
    if (A.node_block && A.sell)
        return shape_sliced(g, A.n, (A.slices + 7) / 8, A.sell_mean, A.sell_steps, units, need);
    return !A.node_block && !A.uneven && shape_csr(g, A.n, A.nnz, units, need);
}
} // namespace

int64_t krylov_engine::csr_block_rows(int64_t n, int64_t nnz) const { return csr_rows(n, nnz, std::max(grid_units_, 1)); }

// What the resident grids need beyond a solve's own vectors: with the engine, so that a solve in
// vectors of the caller's allocates nothing
void krylov_engine::grid_begin()
{
    NEON_CHECK_HIP(hipGetDevice(&grid_device_));
    int units = 0;
    NEON_CHECK_HIP(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, grid_device_));
    grid_slots_.resize(2 * size_t(kGridMaxBlocks) * kGridSlotWords);
    grid_clear();
    grid_units_ = grid_device_ < unit_pool::kDevices ? units : 0;
}

void krylov_engine::grid_clear()
{
    fill_zero(s_, int64_t(grid_slots_.size()), reinterpret_cast<double*>(grid_slots_.data()));
    fill_zero(s_, 2 * sizeof(krylov_state) / sizeof(double), reinterpret_cast<double*>(state_.data() + 2));
    grid_epoch = 1;
}

// The link for one launch of at most `exchanges` exchanges
grid_link krylov_engine::grid_next(uint32_t exchanges)
{
    if (grid_epoch > UINT32_MAX - exchanges - 1)
    {
        // the numbers start again: no slot may hold one of them (the solve's state stays)
        fill_zero(s_, int64_t(grid_slots_.size()), reinterpret_cast<double*>(grid_slots_.data()));
        grid_epoch = 1;
    }
    grid_link const l{grid_slots_.data(), state_.data() + 3, grid_patience_, grid_epoch};
    grid_epoch += exchanges;
    return l;
}

// Runs the launches of a resident grid: batch(true) starts the solve, batch(false) continues it
// from the state in state_[2], whose copies the host reads one launch behind (launches past the
// end return at once).  host_state_ holds the final state; false when the grid gave up (the
// state and vectors are then worthless).
template <typename Batch>
bool krylov_engine::grid_run(unit_hold& hold, Batch&& batch)
{
    auto const since = grid_clock::now();
    auto step = [&](bool first, int slot) {
        batch(first);
        NEON_CHECK_HIP(hipGetLastError());
        NEON_CHECK_HIP(hipMemcpyAsync(host_ring_ + 2 * slot, state_.data() + 2, 2 * sizeof(krylov_state),
                                      hipMemcpyDeviceToHost, s_));
        NEON_CHECK_HIP(hipEventRecord(ring_events_[slot], s_));
    };
    step(true, 0);
    int wait = 0;
    for (;; wait ^= 1)
    {
        if (hold.wanted())
        {
            // another solve's turn, once the launch in flight is through
            NEON_CHECK_HIP(hipEventSynchronize(ring_events_[wait]));
            if (host_ring_[2 * wait].done || host_ring_[2 * wait + 1].done) break;
            hold.yield();
        }
        step(false, wait ^ 1);
        NEON_CHECK_HIP(hipEventSynchronize(ring_events_[wait]));
        if (host_ring_[2 * wait].done || host_ring_[2 * wait + 1].done) break;
    }
    *host_state_ = host_ring_[2 * wait];
    if (!host_ring_[2 * wait + 1].done && host_state_->done != KRYLOV_ABORTED) return true;
    NEON_CHECK_HIP(hipStreamSynchronize(s_));
    grid_clear();
    grid_gave_up(since);
    return false;
}

int krylov_engine::vector_blocks(int64_t n, int width)
{
    if (!grid_units_ || grid_resting()) return 0;
    // at least one 16-byte group per thread, a multiple of 8 (the XCDs' shares) from 8 on
    int64_t const b = std::min<int64_t>((n + int64_t(kVectorThreads) * width - 1) / (int64_t(kVectorThreads) * width),
                                        std::min(grid_units_, kGridMaxBlocks));
    return int(b >= 8 ? b / 8 * 8 : b);
}

void krylov_engine::cg_vector(int blocks, int64_t n, double* r, const double* Ap, const double* minv, double* x,
                              double* p, const double* part, int npart, const krylov_state* st, krylov_state* next,
                              int criterion, double tol, int32_t max_it)
{
    cg_vector_kernel<<<blocks, kVectorThreads, 0, s_>>>(n, r, Ap, minv, x, p, part, npart, st, next, grid_next(1),
                                                        criterion, tol, max_it);
}

void krylov_engine::mixed_vector(int blocks, int64_t n, float* r, const float* Ap, float* x, float* p,
                                 const double* part, int npart, const krylov_state* st, krylov_state* next,
                                 int32_t max_it)
{
    mixed_vector_kernel<<<blocks, kVectorThreads, 0, s_>>>(n, r, Ap, x, p, part, npart, st, next, grid_next(1), max_it);
}

bool krylov_engine::vector_gave_up(grid_clock::time_point since)
{
    NEON_CHECK_HIP(hipMemcpyAsync(host_ring_, state_.data() + 3, sizeof(krylov_state), hipMemcpyDeviceToHost, s_));
    NEON_CHECK_HIP(hipStreamSynchronize(s_));
    if (!host_ring_[0].done) return false;
    grid_clear();
    grid_gave_up(since);
    return true;
}

bool krylov_engine::cg64_grid(const linear_operator& A, const double* b, double* x, const double* minv, int criterion,
                              double tol, int32_t max_it, const krylov_work* work, solve_result& out)
{
    if (prof && prof->enabled) return false; // per-launch timing needs the launches
    if (!grid_units_ || A.blocks_override > 0 || grid_resting()) return false;
    grid_shape g;
    if (!shape_of(g, A, grid_units_, kCgNeed)) return false;

    int64_t const n = A.n;
    int64_t const stride = (n + 31) / 32 * 32; // whole 128-byte lines
    double *r = nullptr, *ring = nullptr;
    int64_t buffers = 0;
    if (work)
    {
        r = work->r;
        ring = work->ring;
        buffers = work->ring_size / stride;
    }
    else
    {
        grid_r_.reserve(stride);
        buffers = std::clamp<int64_t>(kGridRing / stride, 8, 128);
        grid_ring_.reserve(buffers * stride);
        r = grid_r_.data();
        ring = grid_ring_.data();
    }
    // small blocks: two exchanges and two ring buffers per iteration
    bool const few = A.node_block ? g.wps > 1 && g.rounds == 1 : g.rows <= 256 && g.blocks > 1;
    int const iters = int(std::min<int64_t>(few ? buffers / 2 : buffers, 64));
    if (iters < 1) return false;
    krylov_state* st = state_.data() + 2;
    unit_hold hold(grid_device_, g.blocks, grid_units_);
    auto launch = [&](auto kernel, auto rows) {
        allow_lds(kernel);
        return grid_run(hold, [&, kernel](bool first) {
            kernel<<<g.blocks, kGridThreads, size_t(g.lds), s_>>>(rows, g, ring, stride, first ? b : nullptr, x, r, minv,
                                                                  st, grid_next(uint32_t(3 * iters + 2)), iters,
                                                                  criterion, tol, max_it);
        });
    };
    auto with = [&](auto rows) {
        if (few) return launch(cg_grid_small_kernel<decltype(rows)>, rows);
        if (g.all) return launch(cg_grid_kernel<decltype(rows), true>, rows);
        return launch(cg_grid_kernel<decltype(rows), false>, rows);
    };
    bool done = false;
    if (A.sym)
    {
        using lay = grid_sym<double>;
        lay const l{sym_of(A), A.s64};
        int const items = (1 + A.sym_entries + g.wps - 1) / g.wps; // of a wavefront
        if (few && g.wps == 8 && items <= 2)
            done = launch(cg_grid_small_kernel<grid_kept<lay, 2, 8>>, grid_kept<lay, 2, 8>{{l}, {}});
        else if (few && g.wps == 8 && items <= 4)
            done = launch(cg_grid_small_kernel<grid_kept<lay, 4, 8>>, grid_kept<lay, 4, 8>{{l}, {}});
        else if (few && g.wps == 4 && items <= 4)
            done = launch(cg_grid_small_kernel<grid_kept<lay, 4, 4>>, grid_kept<lay, 4, 4>{{l}, {}});
        else
            done = with(grid_sliced<lay>{l});
    }
    else if (A.sell)
    {
        using lay = grid_sell<double>;
        lay const l{sell_of(A), A.s64};
        int const items = (A.sell_steps + g.wps - 1) / g.wps;
        if (few && g.wps == 8 && items <= 4)
            done = launch(cg_grid_small_kernel<grid_kept<lay, 4, 8>>, grid_kept<lay, 4, 8>{{l}, {}});
        else if (few && g.wps == 4 && items <= 8)
            done = launch(cg_grid_small_kernel<grid_kept<lay, 8, 4>>, grid_kept<lay, 8, 4>{{l}, {}});
        else
            done = with(grid_sliced<lay>{l});
    }
    else
        done = with(grid_csr<double>{csr_matrix{int32_t(n), A.rp, A.ci}, A.v64, {}, {}, false});
    if (!done) return false;
    out = finish_solve(*host_state_, criterion);
    out.spmv = out.iterations + (criterion == NEON_STOP_RELATIVE && host_state_->done == KRYLOV_CONVERGED ? 1 : 0);
    return true;
}

bool krylov_engine::bicgstab64_grid(const linear_operator& A, const double* b, double* x, const double* minv,
                                    int criterion, double tol, int32_t max_it, const krylov_work* work,
                                    solve_result& out)
{
    if (prof && prof->enabled) return false;
    if (!grid_units_ || A.blocks_override > 0 || grid_resting()) return false;
    grid_shape g;
    if (!shape_of(g, A, grid_units_, kBicgNeed)) return false;
    int64_t const n = A.n;
    int64_t const stride = (n + 31) / 32 * 32; // whole 128-byte lines
    double *r, *r0, *p, *v, *ring;
    int64_t buffers;
    if (work)
    {
        r = work->r, r0 = work->r0, p = work->p, v = work->v;
        ring = work->bicg_ring;
        buffers = work->bicg_ring_size / stride;
    }
    else
    {
        grid_bicg_.reserve(4 * stride);
        r = grid_bicg_.data(), r0 = r + stride, p = r0 + stride, v = p + stride;
        buffers = std::clamp<int64_t>(kGridRing / stride, 12, 96);
        grid_ring_.reserve(buffers * stride);
        ring = grid_ring_.data();
    }
    int const iters = int(std::min<int64_t>(buffers / 3, 32));
    if (iters < 1) return false;
    int const cuda_rule = criterion == NEON_STOP_ABSOLUTE_PRECONDITIONED ? 1 : 0;
    krylov_state* st = state_.data() + 2;
    unit_hold hold(grid_device_, g.blocks, grid_units_);
    auto launch = [&](auto rows) {
        auto kernel = bicg_grid_kernel<decltype(rows)>;
        allow_lds(kernel);
        return grid_run(hold, [&, kernel](bool first) {
            kernel<<<g.blocks, kGridThreads, size_t(g.lds), s_>>>(rows, g, ring, stride, b, x, r, r0, p, v, minv, st,
                                                                  grid_next(uint32_t(7 * iters + 1)), first ? 1 : 0,
                                                                  iters, cuda_rule, tol, max_it);
        });
    };
    bool done = false;
    if (A.sym)
        done = launch(grid_sliced<grid_sym<double>>{{sym_of(A), A.s64}});
    else if (A.sell)
    {
        using lay = grid_sell<double>;
        lay const l{sell_of(A), A.s64};
        int const items = (A.sell_steps + g.wps - 1) / g.wps;
        if (g.rounds == 1 && g.wps == 8 && items <= 4)
            done = launch(grid_kept<lay, 4, 8>{{l}, {}});
        else if (g.rounds == 1 && g.wps == 4 && items <= 8)
            done = launch(grid_kept<lay, 8, 4>{{l}, {}});
        else
            done = launch(grid_sliced<lay>{l});
    }
    else
        done = launch(grid_csr<double>{csr_matrix{int32_t(n), A.rp, A.ci}, A.v64, {}, {}, false});
    if (!done) return false;
    out = finish_bicg(*host_state_, criterion);
    return true;
}
} // namespace neon_amd
