// Host-side engine of the MI355X implicit Newton step: device buffers, the
// device-resident mesh/constitutive state/tangent, and the Krylov drivers.  Everything
// here is called by the C ABI in capi.cpp and by the Newton driver in newton.cpp.
#pragma once

#include "common.hpp"
#include "neon_hip.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdint>
#include <memory>
#include <string>
#include <vector>

namespace neon_amd
{
struct krylov_state;

// device_array allocations of the process so far (a test holds the allocation-free solve to none)
extern std::atomic<int64_t> device_allocations;

template <typename T>
class device_array
{
public:
    device_array() = default;
    device_array(device_array const&) = delete;
    device_array& operator=(device_array const&) = delete;
    ~device_array() { release(); }

    void resize(size_t n)
    {
        if (n == count) return;
        release();
        if (n)
        {
            ++device_allocations;
            hipError_t const e = hipMalloc(reinterpret_cast<void**>(&ptr), n * sizeof(T));
            if (e != hipSuccess)
            {
                ptr = nullptr;
                throw status_error(e == hipErrorOutOfMemory ? NEON_OOM : NEON_HIP_ERROR,
                                   "hipMalloc of " + std::to_string(n * sizeof(T)) + " bytes failed");
            }
        }
        count = n;
    }
    // at least n entries (the contents are lost when it grows)
    void reserve(size_t n)
    {
        if (n > count) resize(n);
    }
    void release()
    {
        if (ptr) (void)hipFree(ptr);
        ptr = nullptr;
        count = 0;
    }
    T* data() const { return ptr; }
    size_t size() const { return count; }

private:
    T* ptr = nullptr;
    size_t count = 0;
};

// Event pairs around selected launches on one stream; elapsed times are summed per kernel
// class once the stream has been synchronised.
class kernel_profiler
{
public:
    ~kernel_profiler();
    bool enabled = false;
    // returns a token (< 0 when not recording)
    int begin(hipStream_t s, int cls);
    void end(hipStream_t s, int token);
    // accumulate pairs [0, pairs) whose launch ordinal < valid_launches (all if < 0), then clear
    void collect(int64_t valid_launches = -1);
    void read(int cls, bool reset, int64_t* count, double* ms);
    void discard() { pairs_ = 0; }
    void add(int cls, double ms)
    {
        if (!enabled) return;
        count_[cls] += 1;
        ms_[cls] += ms;
    }

private:
    static constexpr int kMaxPairs = 16384;
    std::vector<hipEvent_t> events_;
    std::vector<int> cls_;
    int pairs_ = 0;
    int64_t count_[NEON_KERNEL_CLASSES] = {};
    double ms_[NEON_KERNEL_CLASSES] = {};
};

struct solve_result
{
    int status = NEON_OK;
    int32_t iterations = 0;
    double error = 0.0;
    int64_t spmv = 0;
    int64_t refinements = 0;
};

struct sym_matrix; // krylov_kernels.hpp

// y = A x for a square matrix held on the device in one of two index layouts.
struct linear_operator
{
    int64_t n = 0;
    int64_t nnz = 0;     // generic CSR layout only
    bool uneven = false; // generic CSR layout: not for the resident grid (csr_grid_pays)
    bool node_block = false;
    // node-block layout
    int32_t nodes = 0;
    const int32_t* bptr = nullptr;
    const int32_t* bcol = nullptr;
    // generic CSR layout
    const int32_t* rp = nullptr;
    const int32_t* ci = nullptr;
    int lanes_per_row = 8;
    // node-block SpMV shape: lanes per block row of the CSR-order kernel (16 or 32),
    // nontemporal value loads, optional workgroup count
    int nb_lanes = 32;
    bool nb_nt = false;
    int blocks_override = 0;
    // the sliced layouts' slices in the opposite order (spmv_sell_kernel)
    int back = 0;
    // values
    const double* v64 = nullptr;
    const float* v32 = nullptr;
    // sliced copy of the node-block values (sell_matrix layout); the SpMV uses it when set
    bool sell = false;
    int32_t slices = 0;
    int32_t sell_steps = 0; // largest and mean number of steps of a slice
    double sell_mean = 0.0;
    const int32_t* sptr = nullptr;
    const int32_t* snode = nullptr;
    const int32_t* slane = nullptr;
    const int32_t* scode = nullptr;
    const int32_t* sexc = nullptr;
    const int16_t* soff16 = nullptr; // 16-bit per-lane offsets (used when set)
    const int32_t* soff32 = nullptr;
    const double* s64 = nullptr;
    const float* s32 = nullptr;
    // symmetric sliced copy (sym_matrix layout: diagonal and upper blocks); the SpMV uses it
    // when set, with its values at s64 / s32 and `slices` slices
    bool sym = false;
    int32_t sym_slots = 0;
    int64_t sym_records = 0;
    int32_t sym_entries = 0; // largest and mean number of entries of a slice
    double sym_mean = 0.0;
    const int32_t* sym_sched = nullptr;
    const int32_t* sym_rdiag = nullptr;
    const int32_t* sym_eptr = nullptr;
    const int32_t* sym_ent = nullptr; // 4 int32 per entry
    const int32_t* sym_rslice = nullptr;
    const int32_t* sym_roff = nullptr;

    int spmv_blocks() const;
    // FP64: y = A x (values v64); with part, also block partials of x.y (or w.y if w).
    // gate (with st): 1 runs only while st->refine is set, 2 only while it is clear
    void apply64(hipStream_t s, const double* x, double* y, double* part, const krylov_state* st, int gate = 0) const;
    // FP32 values/vectors, FP32 accumulation, FP64 partials of x.y
    void apply32(hipStream_t s, const float* x, float* y, double* part, const krylov_state* st) const;
    // r = b - A x in FP64 arithmetic from the stored values (v64 if set, else v32)
    // (skipped when st is given and the state is done, or, with gate, no reliable update is due)
    void residual64(hipStream_t s, const double* b, const double* x, double* r, const krylov_state* st = nullptr,
                    int gate = 0) const;
};

// Device work vectors of n entries each for the FP64 solvers, supplied by the caller instead of
// the engine's own (cg64 uses r, p, Ap; bicgstab64 r, p, r0, v, s, t, p_hat, s_hat).
struct krylov_work
{
    double *r = nullptr, *p = nullptr, *Ap = nullptr;
    double *r0 = nullptr, *v = nullptr, *s = nullptr, *t = nullptr, *p_hat = nullptr, *s_hat = nullptr;
    // the resident-grid loops' rings: CG's beside r, BiCGSTAB's beside r, p, r0 and v (doubles)
    double *ring = nullptr, *bicg_ring = nullptr;
    int64_t ring_size = 0, bicg_ring_size = 0;
};

struct grid_link; // grid_kernels.hpp
// Doubles of the ring that a resident grid's iterations publish their vectors to (64 MiB; at
// least 8 iterations' worth)
constexpr int64_t kGridRing = int64_t(1) << 23;
solve_result finish_solve(const krylov_state& s, int criterion);
solve_result finish_bicg(const krylov_state& s, int criterion);

// Device memory and a pinned buffer that the host-CSR solves of one context keep from call to call
// (a program solves many systems of one size; a small solve spent half its time on seven
// allocations and five pageable copies).  At most kCsrKept bytes stay after a call; the context
// frees the rest with it.
constexpr size_t kCsrKept = size_t(256) << 20;
constexpr size_t kCsrStage = size_t(256) << 10; // pinned
struct csr_space
{
    device_array<unsigned char> dev;
    unsigned char* stage = nullptr;
    csr_space();
    ~csr_space();
    csr_space(csr_space const&) = delete;
    csr_space& operator=(csr_space const&) = delete;
};

// Compute units of a GPU held for one solve's resident grids (grid_krylov.hip).  A solve with nothing
// in flight lets others have their turn with yield() while wanted(): it holds them for a batch of
// iterations at a time if another solve waits, for all of them otherwise.
class unit_pool;
class unit_hold
{
public:
    unit_hold(int device, int blocks, int units);
    ~unit_hold();
    unit_hold(unit_hold const&) = delete;
    unit_hold& operator=(unit_hold const&) = delete;
    bool wanted() const;
    void yield();
    // compute units held for `blocks` workgroups on a GPU of `units`: workgroups go to the 8 XCDs in turn,
    // whatever room these have, so counts are taken in whole turns; otherwise grids that fit by their
    // sum (250 and 6 workgroups, say) overfill an XCD, and each may wait for a compute unit the other has
    static constexpr int held(int blocks, int units)
    {
        int const whole = (blocks + 7) / 8 * 8;
        return whole <= units ? whole : units;
    }

private:
    unit_pool& pool_;
    int count_, units_;
};

class krylov_engine
{
public:
    csr_space csr;

    explicit krylov_engine(hipStream_t s);
    ~krylov_engine();

    // Jacobi inverse of the operator's diagonal (FP64 values).
    void jacobi64(const linear_operator& A, double* minv, int eigen_rule);

    // work: the caller's work vectors (nothing allocated), else the engine's own (grown to n)
    solve_result cg64(const linear_operator& A, const double* b, double* x, const double* minv, int criterion,
                      double tol, int32_t max_it, const krylov_work* work = nullptr);
    solve_result bicgstab64(const linear_operator& A, const double* b, double* x, const double* minv,
                            int criterion, double tol, int32_t max_it, const krylov_work* work = nullptr);
    // copy one device double to the host through the engine's pinned word (synchronises)
    double read_scalar(const double* d);
    // FP32 inner CG with FP64 reliable updates r = b - A x (relative rule only).
    solve_result cg_mixed(const linear_operator& A, const double* b, double* x, int criterion, double tol,
                          int32_t max_it);
    // same, for a node-block operator whose Jacobi inverse (FP64, from the FP32 diagonal) is given;
    // scaled: the Jacobi-scaled tangent D^-1/2 K D^-1/2 (minv positive, same layout as A), on
    // which the FP32 recurrence then runs without a preconditioner vector (A still gives the
    // FP64 residuals)
    solve_result cg_mixed_nb(const linear_operator& A, const double* b, double* x, const double* minv, double tol,
                             int32_t max_it, const linear_operator* scaled = nullptr);
    // every entry positive and finite (synchronises)
    bool all_positive(int64_t n, const double* v);

    double dot(int64_t n, const double* a, const double* b);
    // u += d, then out = u.u, d.d, f.f, r.r (synchronises)
    void step_norms(int64_t n, double* u, const double* d, const double* f, const double* r, double* out);

    hipStream_t stream() const { return s_; }
    int vec_blocks(int64_t n) const;
    // rows of a workgroup of the resident grid for a CSR system
    int64_t csr_block_rows(int64_t n, int64_t nnz) const;
    kernel_profiler* prof = nullptr;
    // iterations between convergence polls from the host
    int poll_every = 16;
    // ticks (100 MHz) that a resident grid's workgroups wait for each other before the solve falls
    // back to launches: another process may hold the compute units that some of them need
    void set_grid_patience(uint64_t ticks)
    {
        grid_patience_ = ticks;
        grid_rest_until_ = {};
    }
    int64_t grid_give_ups = 0;
    // the number of the next exchange (unique among those whose words the slots may still hold)
    uint32_t grid_epoch = 1;
    // reliable-update trigger of the mixed-precision CG: ||r32|| < delta ||r at last update||
#ifndef NEON_RELIABLE_DELTA
#define NEON_RELIABLE_DELTA 0.1
#endif
#ifndef NEON_REFINE_EVERY
#define NEON_REFINE_EVERY 8
#endif
    double reliable_delta = NEON_RELIABLE_DELTA;
    // the mixed CG tests the trigger (and, through the true residual, convergence) every this
    // many iterations
    int refine_every = NEON_REFINE_EVERY;

private:
    void ensure(int64_t n);
    void ensure_mixed(int64_t n);
    solve_result cg_mixed_run(const linear_operator& A, const double* b, double* x, double tol, int32_t max_it, int nb,
                              int ns, double* part_pAp, double* part_rr, double* part_rz, double* part_rr_t,
                              double* part_rz_t, krylov_state* st, float* minv, const linear_operator* scaled_op,
                              const double* minv64_scaled);
    hipStream_t s_;
    device_array<double> part_[6];
    device_array<krylov_state> state_;
    krylov_state* host_state_ = nullptr;
    // poll-ahead ring of run_batches and grid_run: two pinned state snapshots (of two states each
    // for grid_run) and their events
    krylov_state* host_ring_ = nullptr;
    hipEvent_t ring_events_[2] = {nullptr, nullptr};
    template <typename Batch>
    void run_batches(krylov_state* st, int64_t& launched, unit_hold* hold, Batch&& batch);
    // resident-grid loops (grid_krylov.hip): false when the solve does not qualify or its grid
    // gave up; the launch-per-phase loop then solves
    bool cg64_grid(const linear_operator& A, const double* b, double* x, const double* minv, int criterion, double tol,
                   int32_t max_it, const krylov_work* work, solve_result& out);
    bool bicgstab64_grid(const linear_operator& A, const double* b, double* x, const double* minv, int criterion,
                         double tol, int32_t max_it, const krylov_work* work, solve_result& out);
    // an iteration's vector part in one launch (vector_iteration): the workgroups for n entries (0:
    // not available) and the launches; vector_gave_up, after a loop with them that began at `since`:
    // whether one gave up (the loop then runs again without them)
    int vector_blocks(int64_t n, int width);
    void cg_vector(int blocks, int64_t n, double* r, const double* Ap, const double* minv, double* x, double* p,
                   const double* part, int npart, const krylov_state* st, krylov_state* next, int criterion, double tol,
                   int32_t max_it);
    void mixed_vector(int blocks, int64_t n, float* r, const float* Ap, float* x, float* p, const double* part,
                      int npart, const krylov_state* st, krylov_state* next, int32_t max_it);
    // A grid that gave up cost its solve the patience and the work so far, and what kept it out is
    // likely to be there for the next one too: solves take launches for kGridRest times as long as
    // was lost (at least kGridRest times 10 ms), so that a lasting cause costs 1 / kGridRest.
    static constexpr int kGridRest = 64;
    using grid_clock = std::chrono::steady_clock;
    bool grid_resting() const { return grid_clock::now() < grid_rest_until_; }
    void grid_gave_up(grid_clock::time_point since)
    {
        auto const now = grid_clock::now();
        grid_rest_until_ = now + kGridRest * std::max<grid_clock::duration>(now - since, std::chrono::milliseconds(10));
        ++grid_give_ups;
    }
    grid_clock::time_point grid_rest_until_{};
    uint64_t grid_patience_ = 100ull * 1000 * 1000;
    bool vector_gave_up(grid_clock::time_point since);
    void grid_begin();
    void grid_clear();
    grid_link grid_next(uint32_t exchanges);
    template <typename Batch>
    bool grid_run(unit_hold& hold, Batch&& batch);
    int grid_device_ = 0, grid_units_ = 0;
    device_array<uint64_t> grid_slots_;
    device_array<double> grid_ring_, grid_r_, grid_bicg_;
    double* host_scalar_ = nullptr;
    device_array<double> scalar_, norms_;
    int64_t n_ = 0, n_mixed_ = 0;
    device_array<double> r_, p_, Ap_;
    device_array<double> r0_, v_, s_vec_, t_, ph_, sh_;
    device_array<float> r32_, p32_, Ap32_, x32_, minv32_;
    device_array<double> x64_, r64_;
};

// Tangent value arrays extend this many entries past nnz (zeroed): SpMV kernels that stream a
// segment in 16-byte vectors may read up to one vector past its end.
constexpr int64_t kValuePad = 16;

// Shape of the node-block SpMV used by the Krylov solvers on a mesh tangent (the defaults
// are the fastest measured at 6.4M dofs on MI355X): lanes per block row, NEON_SPMV_* flags,
// workgroups for FP64 and FP32 values.
// constitutive_model::is_symmetric of each model id (only the J2 damage model's tangent is
// unsymmetric: small_strain_J2_plasticity_damage.hpp:44)
inline bool model_is_symmetric(int32_t model) { return (model & 0xff) != NEON_MODEL_J2_DAMAGE; }

struct spmv_config
{
    int lanes = 32;
    int flags = NEON_SPMV_SLICED | NEON_SPMV_NONTEMPORAL | NEON_SPMV_SYMMETRIC;
    int blocks64 = 0;
    int blocks32 = 0;
};

// Meshes of at most this many elements assemble through staged element blocks, 4,800 bytes each, which
// then stay in the 256 MB cache between the two launches: 8^3, 16^3, 25^3, 32^3 elements 24, 43, 91,
// 175 us (FP64) against 76, 90, 137, 233 us colour by colour.  Larger ones go colour by colour, which
// moves less in FP32 and needs no scratch: 40^3 elements 365 us (FP32 298) against 382 (361) staged.
constexpr int64_t kStageElements = int64_t(1) << 15;
struct qp_state; // element_kernels.hpp

// A sliced copy of at most this many bytes (a little under the 256 MB memory-side cache, which holds the
// vectors too) is read with plain loads, a larger one with nontemporal loads if the flags ask for
// them.  A solver reads the copy again in each iteration; nontemporal loads leave it in no L2, and
// whether the next cache holds it then depends on what else was there: after a staged assembly,
// whose blocks stay in the L2s, 14.4 us became 20.2 per FP32 product at 14^3 cells, 19.1 became 24.5 at
// 15^3.  Nontemporal against plain, us per product: FP32 copies of 3.3, 9, 67, 221, 267, 378, 887 MB
// 20.2 / 14.4, 23.3 / 15.3, 30.7 / 24.2, 45.4 / 39.9, 51.9 / 52.6, 87.6 / 92.4, 163.7 / 185.4; FP64
// copies of 18, 134, 229, 360, 534, 1,774 MB 27.2 / 16.4, 37.3 / 28.1, 46.3 / 38.8, 81.1 / 80.3, 113.1 /
// 116.5, 340.8 / 358.7.
constexpr size_t kStreamedCopy = size_t(240) << 20;

// Device-resident mesh: geometry, constitutive state, pattern, tangent and f_int.
class device_mesh
{
public:
    device_mesh(hipStream_t s, int32_t n_nodes, const double* X, int32_t n_elem, const int32_t* conn, int32_t model,
                const double* params, int32_t tangent_mode);

    int32_t nodes() const { return N_; }
    int32_t elements() const { return E_; }
    int64_t dofs() const { return 3ll * N_; }
    int64_t nnz() const { return nnz_; }
    int32_t model() const { return model_; }
    int32_t colours() const { return int32_t(colour_offsets_.size()) - 1; }

    void set_parameters(const double* params);
    void set_displacement_host(const double* u);
    // u (device) -> state; returns NEON_OK or the recoverable code.  dt is the time step of
    // the path-dependent models' rate equations: the step size at a load step's first update,
    // 0 at its Newton iterates
    int update_internal_variables(const double* u_dev, double dt = 0.0);
    // LATIN (latin_matrix.hpp): committed stress <- 0 (latin_reset) or <- current stress
    // (latin_commit); f <- the LATIN force at the current state with the committed
    // displacement u_old (device) and search direction s
    void latin_reset();
    void latin_commit();
    void latin_force(const double* u_dev, const double* u_old_dev, double s, double* f_dev);
    // ageing microsphere: the material's scission and recombination probabilities
    void set_ageing(double scission, double recombination);
    // ageing microsphere: network state, 11 per QP in QP order (host)
    void download_ageing_state(double* state);
    // J2 damage: the material constants; back stress (9 per QP, row-major), damage and energy
    // release rate (host, any may be null)
    void set_damage(const double* constants);
    void download_damage_state(double* back_stress, double* damage, double* energy);
    void save_internal_variables(bool converged);
    void assemble(const double* u_dev, int precision);
    void enforce_dirichlet(int32_t n_fixed, const int32_t* fixed_dev, double* b_dev, int precision);
    void pattern(int32_t* row_ptr, int32_t* col) const;
    void download(double* val, double* f_int, int precision_hint);
    void download_qp_state(double* sigma, double* D, double* detF, double* eps_p, double* ebar, double* vm);
    // operator over the assembled tangent (FP64 values, or FP32 values for mixed)
    linear_operator op(int precision) const;
    linear_operator op_base(int precision) const;
    // points A's SpMV at the sliced copy of the tangent (packed here when the tangent changed
    // since the last copy); index32: 32-bit per-lane offsets even where 16 bits fit
    void attach_sliced(linear_operator& A, int precision, bool index32 = false) const;
    // whether every per-lane offset of the sliced copy fits 16 bits
    bool sliced_index16() const { return soff16_ok_; }
    int32_t sliced_slices() const { return slices_; }
    int64_t sliced_steps() const { return sell_steps_; }
    // steps whose 64 lanes share one column offset
    int64_t sliced_shared_steps() const { return shared_steps_; }
    // the sliced copy is packed through LDS: nodes of at most 170 neighbours
    bool sliced_fits() const;
    // points A's SpMV at the symmetric sliced copy (diagonal and upper blocks; packed here when
    // the tangent changed since the last copy); only where symmetric_usable()
    // scale_minv (FP32 values only): attach D^-1/2 K D^-1/2 with D^-1 = scale_minv (positive)
    void attach_symmetric(linear_operator& A, int precision, const double* scale_minv = nullptr) const;
    // the solvers' operator is the symmetric copy (flags ask for it and the mesh allows it)
    bool symmetric_selected() const;
    // the symmetric FP32 copy of the Jacobi-scaled tangent (minv: the positive Jacobi inverse of
    // the FP32 diagonal), for the mixed solver
    linear_operator op_scaled(const double* minv) const;
    // a symmetric model and a pattern for which the symmetric copy pays (every slice needs at
    // most kMaxSymEntries offsets and the copy holds at most 3/4 of the full copy's steps)
    bool symmetric_usable() const;
    // the largest number of offsets (entries) of a slice (0 when the pattern does not qualify),
    // the symmetric copy's wave slots and records
    int32_t symmetric_offsets() const { return sym_ok_ ? sym_max_entries_ : 0; }
    int32_t symmetric_slots() const { return sym_slots_; }
    int64_t symmetric_records() const { return sym_records_; }
    // Jacobi inverse from the node-block diagonal
    void jacobi(double* minv, int eigen_rule, int precision);
    // consistent mass (density per element, host) in the pattern of K, FP64; Dirichlet rows and
    // columns zeroed with the diagonal kept; operator, Jacobi inverse and download
    void assemble_mass(const double* density);
    void enforce_dirichlet_mass(int32_t n_fixed, const int32_t* fixed_dev);
    linear_operator op_mass() const;
    void jacobi_mass(double* minv);
    void download_mass(double* val);
    // adjoint: grad (4 per element) = -lambda^T d f_int / d params at displacement u
    void parameter_gradient(const double* u_dev, const double* lambda_dev, double* grad_dev);

    // load-history checkpoints (J2 adjoint): u_n and the committed history h_{n-1} of every
    // converged step, kept on the device
    void clear_trajectory();
    void record_step();
    int32_t trajectory_steps() const { return int32_t(traj_u_.size()); }
    // u <- u_n, committed history <- h_{n-1}
    void restore_step(int32_t step);
    // J2 adjoint pieces at the state of restore_step + update_internal_variables:
    // rhs += B^T (dh/d eps)^T mu;  mu <- history adjoint of the step, grad += parameter adjoint
    void j2_adjoint_rhs(double* rhs);
    void j2_adjoint_history(const double* lambda, double* grad);
    void j2_adjoint_begin();
    int32_t tangent_mode() const { return tangent_mode_; }

    double* u() { return u_.data(); }
    double* f_int() { return fint_.data(); }
    hipStream_t stream() const { return s_; }
    bool has_k64() const { return k64_valid_; }
    bool has_k32() const { return k32_valid_; }

    // last assemble time split (ms) measured with events
    float last_assemble_ms = 0.0f;
    spmv_config spmv;
    // assembly grid: workgroups (one wavefront each) per compute unit and colour
    int assembly_blocks_per_cu = 128;
    int32_t max_degree() const { return max_degree_; }
    kernel_profiler* prof = nullptr;

private:
    void assemble_staged(const double* u_dev, qp_state const& st, bool fp64);
    void assemble_coloured(const double* u_dev, qp_state const& st, bool fp64);
    void build_sliced_pattern();
    void build_symmetric_pattern();
    sym_matrix sym_layout() const;
    hipStream_t s_;
    int32_t N_, E_, model_, tangent_mode_;
    int64_t nnz_ = 0;
    int32_t max_degree_ = 0;
    std::vector<int32_t> bptr_h_, bcol_h_;
    std::vector<int32_t> colour_offsets_;
    device_array<double> X_, u_, params_, fint_;
    device_array<int32_t> conn_, elems_, bptr_, bcol_, self_slot_, incp_, inc_;
    device_array<double> stage_; // staged assembly: element blocks, then element forces
    device_array<uint8_t> slots_;
    device_array<double> k64_, m64_;
    device_array<float> k32_;
    bool m64_valid_ = false;
    bool k64_valid_ = false, k32_valid_ = false;
    // sliced layout of the pattern (sell_matrix) and the sliced copies of the tangent
    int32_t slices_ = 0;
    int64_t sell_steps_ = 0, shared_steps_ = 0;
    device_array<int32_t> sptr_, snode_, slane_, scode_, sexc_, soff32_;
    device_array<int16_t> soff16_;
    bool soff16_ok_ = false;
    mutable device_array<double> s64_;
    mutable device_array<float> s32_;
    mutable bool s64_fresh_ = false, s32_fresh_ = false;
    // symmetric sliced layout: per-slice entries, records, the wave-slot schedule and the copies
    bool sym_ok_ = false;
    int32_t sym_slots_ = 0, sym_max_entries_ = 0;
    double sym_mean_entries_ = 0.0;
    int64_t sym_records_ = 0;
    device_array<int32_t> sym_sched_, sym_rdiag_, sym_eptr_, sym_ent_, sym_rslice_, sym_roff_;
    mutable device_array<double> y64_;
    mutable device_array<float> y32_, y32s_;
    mutable bool y64_fresh_ = false, y32_fresh_ = false, y32s_fresh_ = false;
    device_array<double> sigma_, coef_, detF_, eps_p_, ebar_, vm_, eps_p_old_, ebar_old_;
    device_array<double> age_, age_old_; // ageing microsphere: 11 x Q network state (SoA)
    device_array<double> sigma_old_;     // LATIN: committed stress (6 x Q)
    double scission_ = 0.0, recombination_ = 0.0, last_dt_ = 0.0;
    // J2 damage: back stress 6, damage 1, energy release rate 1 per QP (SoA) and the committed
    // back stress and damage; the material's constants (C, gamma, s_p, n_p, s_d, n_d)
    device_array<double> dmg_state_, dmg_state_old_;
    device_array<int32_t> yield_; // an update's yielding points: their count, then their numbers
    double damage_[6] = {1.0, 1.0, 1.0, 1.0, 1.0, 1.0};
    device_array<uint32_t> status_;
    std::vector<std::unique_ptr<device_array<double>>> traj_u_, traj_ep_, traj_eb_;
    device_array<double> mu_ep_, mu_eb_;
    uint32_t* status_host_ = nullptr;
};

void upload_hex8_tables();
void convert_to_float(hipStream_t s, int64_t n, const double* x, float* y);
void fill_zero(hipStream_t s, int64_t n, double* x);
void fill_ones(hipStream_t s, int64_t n, double* x);
void fill_ones(hipStream_t s, int64_t n, float* x);
} // namespace neon_amd

struct neon_context
{
    int device = 0;
    hipStream_t stream = nullptr;
    std::string error;
    neon_amd::krylov_engine* engine = nullptr;
    neon_amd::device_mesh* mesh = nullptr;
    neon_amd::kernel_profiler profiler;
};
