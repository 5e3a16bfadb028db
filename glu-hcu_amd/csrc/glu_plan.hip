// Plan construction (host) and the C-ABI of include/glu_hip.h.
//
// A plan uploads one sparsity pattern once: the Symbolic_Matrix arrays that
// LUonDevice copies on every call (src/numeric.cu:435-458), plus the tables
// this build adds — the CSR->CSC map, the per-update scatter map, work
// units and level schedules for the factorization and the four triangular
// sweeps, and (from an analysis) the permutation/scales and the structure of
// the original A for value refresh and FP64 refinement.
//
// Every index array is validated on the host before upload (pointer
// monotonicity, ranges, sorted unique rows, diagonal positions, CSR/CSC
// agreement, level permutation, fill closure); the kernels index without
// bounds checks and rely on it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <atomic>
#include <system_error>
#include <future>
#include <thread>
#include <vector>

#include "../../include/glu_hip.h"
#include "glu_dev.h"
#include "host/glu_host.h"

namespace glu {
namespace launch {
void pert(const FactorDev &F, const float *val, unsigned int *norm_bits, float *d_pert, hipStream_t st);
void factor_grid(const FactorDev &F, float *val, const float *d_pert, int lvl, uint32_t items, int perturb,
                 int threads, hipStream_t st);
void factor_phase(const PhaseDev &Ph, float *val, const float *d_pert, int perturb, int threads, hipStream_t st);
void factor_fused(const FactorDev &F, float *val, const float *d_pert, int l0, int l1, int perturb,
                  int threads, hipStream_t st);
void factor_divide(const FactorDev &F, float *val, const float *d_pert, uint32_t ndiv, int perturb, hipStream_t st);
void tri_grid(const TriDev &T, const float *lu, float *x, int lvl, uint32_t rows, hipStream_t st);
void tri_fused(const TriDev &T, const float *lu, float *x, int l0, int l1, int threads, hipStream_t st);
void perm_scale_f32(const float *in, float *out, const uint32_t *P, const double *S, int by_perm, uint32_t n,
                    hipStream_t st);
void perm_scale_f64(const double *in, float *out, const uint32_t *P, const double *S, int by_perm,
                    uint32_t n, hipStream_t st);
void update_x(const float *t, double *x, const uint32_t *P, const double *S, int by_perm, uint32_t n,
              hipStream_t st);
void refresh(const RefineDev &R, const double *ax, float *lu, uint32_t nnz_lu, int batch, hipStream_t st);
void residual(const RefineDev &R, const double *ax, const double *b, const double *x, double *r, uint32_t n,
              int transpose, int with_anorm, unsigned long long *norms, uint32_t lanes, hipStream_t st);
size_t batch_lds_bytes(int mode, uint32_t n);
void batch_same(const MatDesc *desc, int batch, const double *ax, const double *b, double *x, float *lu,
                float *lucsr, float *t32, double *r64, double *norms, double *kry, int32_t *iters, double *eta,
                double tol, int maxit, int perturb, int threads, int mode, size_t fact_lds, size_t ref_lds,
                int l0, hipStream_t st);
void batch_factor(const MatDesc *desc, int batch, const double *ax, float *lu, double *norms, int perturb,
                  int threads, size_t fact_lds, int l0, hipStream_t st);
void il_values(const RefineDev &R, const FactorDev &F, const double *ax, float *S, unsigned int *bits,
               double *pertd, uint32_t nnz, uint32_t n, int batch, int perturb, hipStream_t st);
void factor_grid_il(const FactorDev &F, float *S, const double *pertd, int lvl, uint32_t waves, int batch,
                    int perturb, hipStream_t st);
void il_to_rows(const float *S, float *lu, uint32_t nnz, int batch, hipStream_t st);
uint32_t il_items_per_wave();
uint32_t il_group();
void abft_cca(const FactorDev &F, const float *val, float *cca, int batch, hipStream_t st);
void abft_check(const FactorDev &F, const uint32_t *row_idx, const uint32_t *diag, const float *lu,
                const float *cca, float *ccl, float tol, int32_t *first_bad, float *max_diff, int batch,
                hipStream_t st);
void group_phases(const MatDesc *descs, const void *ios, const uint32_t *order, int count, const int32_t *l0,
                  const GroupLaunch &G, int perturb, int threads, hipStream_t st);
void batch_group(const MatDesc *descs, const void *ios, const uint32_t *order, int count, const int32_t *l0, double tol,
                 int maxit, int perturb, int threads, int mode, size_t fact_lds, size_t ref_lds, hipStream_t st);
void tri_df(const TriDev &T, const float *lu, float *x, int l0, int l1, uint32_t k0, uint32_t k1, uint32_t n,
            int threads, hipStream_t st);
size_t enable_lds();
void factor_window(const FactorDev &F, int w, uint32_t nslot, float *val, const float *d_pert, int perturb,
                   int threads, hipStream_t st);
void zero_u64(unsigned long long *p, int count, hipStream_t st);
void solve_one(const MatDesc *desc, const uint32_t *src, uint32_t nval, const float *lu, float *lucsr, const float *b,
               float *x, float *t32, uint32_t r0, int threads, int mode, size_t lds, int transpose, hipStream_t st);
void split_solve(const SplitDev &S, const float *b, const float *lu, float *lucsr, float *rhs, float *xg, hipStream_t st);
void split_precond(const SplitDev &S, const double *r, const float *lu, float *lucsr, float *rhs, float *xg,
                   hipStream_t st);
void refine_one(const MatDesc *desc, const uint32_t *src, uint32_t nval, const double *ax, const double *b, double *x,
                const float *lu, float *lucsr, float *t32, double *r64, double *norms, double *kry, int32_t *iters,
                double *eta, double tol, int maxit, int threads, size_t ref_lds, int transpose, hipStream_t st);
void copy_df(const uint32_t *src, uint32_t nval, const float *lu, float *lucsr, hipStream_t st);
void sweeps_df(const MatDesc *desc, const float *lucsr, float *t32, uint32_t r0, int threads, size_t lds,
               int transpose, hipStream_t st);
void adjoint_values(const RefineDev &R, const double *lam, const double *x, double *grad, uint32_t n,
                    hipStream_t st);
size_t matio_size();
uint32_t group_values();
}  // namespace launch
}  // namespace glu

using namespace glu;

// ---------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------

static thread_local std::string g_err;

static glu_status fail(glu_status s, const std::string &msg)
{
    g_err = msg;
    return s;
}

#define HIP_TRY(call)                                                                              \
    do {                                                                                           \
        hipError_t e_ = (call);                                                                    \
        if (e_ != hipSuccess) return fail(GLU_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

extern "C" const char *glu_last_error(void) { return g_err.c_str(); }

// f() with C++ exceptions as status codes (nothing may leave a C entry).
template <typename F>
static glu_status guarded(F f)
{
    try {
        return f();
    } catch (const std::bad_alloc &) {
        return fail(GLU_ERR_MEMORY, "out of host memory");
    } catch (const std::length_error &) {
        return fail(GLU_ERR_MEMORY, "a table is too large for host memory");
    } catch (const std::exception &e) {
        return fail(GLU_ERR_GENERAL, e.what());
    }
}

// ---------------------------------------------------------------------------
// analysis object
// ---------------------------------------------------------------------------

struct glu_analysis {
    Analysis an;
    Symbolic sym;
    std::vector<uint32_t> lu_from_dump;
    int64_t updates = 0;
};

static int64_t count_updates(const Symbolic &s)
{
    int64_t u = 0;
    for (uint32_t k = 0; k < s.n; ++k) {
        int64_t L = (int64_t)s.sym_c_ptr[k + 1] - s.l_col_ptr[k] - 1;
        int64_t U = (int64_t)s.csr_r_ptr[k + 1] - s.csr_diag_ptr[k] - 1;
        u += L * U;
    }
    return u;
}

extern "C" glu_status glu_analyze(uint32_t n, uint32_t nnz, const double *ax, const uint32_t *ai,
                                  const uint32_t *ap, glu_analysis **out)
{
    if (!out) return fail(GLU_ERR_ARGUMENT, "out is null");
    *out = nullptr;
    if (n == 0 || nnz == 0) return fail(GLU_ERR_EMPTY, "matrix is empty");
    if (!ax || !ai || !ap) return fail(GLU_ERR_ARGUMENT, "null array");
    std::unique_ptr<glu_analysis> a(new (std::nothrow) glu_analysis());
    if (!a) return fail(GLU_ERR_MEMORY, "out of host memory");
    std::string err;
    int rc;
    try {
        rc = analyze(n, nnz, ax, ai, ap, a->an, err);
        if (rc == kOk) {
            // Duplicates the reference's adjacency check lets through
            // (non-adjacent repeats in one column) are refused here.
            std::vector<uint32_t> stamp(n, UINT32_MAX);
            for (uint32_t c = 0; c < n && rc == kOk; ++c)
                for (uint32_t k = ap[c]; k < ap[c + 1]; ++k) {
                    if (stamp[ai[k]] == c) {
                        rc = kErrDuplicate;
                        err = "duplicate entry";
                        break;
                    }
                    stamp[ai[k]] = c;
                }
        }
        if (rc == kOk) {
            symbolic(n, a->an.ai.data(), a->an.ap.data(), a->sym);
            predict_lu(a->an.ai.data(), a->an.ap.data(), a->an.ax.data(), a->sym, &a->lu_from_dump);
            a->updates = count_updates(a->sym);
        }
    } catch (const std::bad_alloc &) {
        return fail(GLU_ERR_MEMORY, "out of host memory during analysis");
    }
    if (rc != kOk) return fail((glu_status)rc, err);
    *out = a.release();
    return GLU_OK;
}

// Independent patterns analysed on host threads (a work queue over the
// matrices); each item as glu_analyze.
extern "C" glu_status glu_analyze_many(int count, const uint32_t *n, const uint32_t *nnz,
                                       const double *const *ax, const uint32_t *const *ai,
                                       const uint32_t *const *ap, int threads, glu_analysis **out,
                                       glu_status *status)
{
    if (count <= 0 || !n || !nnz || !ax || !ai || !ap || !out || !status)
        return fail(GLU_ERR_ARGUMENT, "bad argument");
    for (int i = 0; i < count; ++i) out[i] = nullptr;
    int hw = (int)std::thread::hardware_concurrency();
    int nt = threads > 0 ? threads : (hw > 0 ? hw : 1);
    nt = std::max(1, std::min(nt, count));
    std::vector<std::string> msg(count);
    std::atomic<int> next(0);
    auto work = [&]() {
        for (int i = next.fetch_add(1); i < count; i = next.fetch_add(1)) {
            status[i] = glu_analyze(n[i], nnz[i], ax[i], ai[i], ap[i], out + i);
            if (status[i] != GLU_OK) msg[i] = glu_last_error();
        }
    };
    std::vector<std::thread> pool;
    try {
        pool.reserve(nt - 1);
        for (int t = 1; t < nt; ++t) pool.emplace_back(work);
    } catch (const std::exception &) {
        // fewer threads than asked for (none left, or no memory): the ones
        // that started share the queue with this thread
    }
    work();
    for (std::thread &t : pool) t.join();
    for (int i = 0; i < count; ++i)
        if (status[i] != GLU_OK) return fail(status[i], "matrix " + std::to_string(i) + ": " + msg[i]);
    return GLU_OK;
}

extern "C" void glu_analysis_destroy(glu_analysis *a) { delete a; }

extern "C" glu_status glu_analysis_info(const glu_analysis *a, int64_t info[8])
{
    if (!a || !info) return fail(GLU_ERR_ARGUMENT, "null argument");
    info[0] = a->sym.n;
    info[1] = a->an.nnz;
    info[2] = a->sym.nnz;
    info[3] = a->sym.num_lev;
    info[4] = a->updates;
    info[5] = info[6] = info[7] = 0;
    return GLU_OK;
}

template <typename T>
static glu_status copy_field(const std::vector<T> &v, void *dst, size_t bytes)
{
    if (bytes != v.size() * sizeof(T))
        return fail(GLU_ERR_ARGUMENT, "size mismatch: expected " + std::to_string(v.size() * sizeof(T)) +
                                          " bytes, got " + std::to_string(bytes));
    if (bytes) std::memcpy(dst, v.data(), bytes);
    return GLU_OK;
}

extern "C" glu_status glu_analysis_get(const glu_analysis *a, glu_field f, void *dst, size_t bytes)
{
    if (!a || (!dst && bytes)) return fail(GLU_ERR_ARGUMENT, "null argument");
    const Symbolic &s = a->sym;
    const Analysis &an = a->an;
    switch (f) {
    case GLU_F_SYM_C_PTR: return copy_field(s.sym_c_ptr, dst, bytes);
    case GLU_F_SYM_R_IDX: return copy_field(s.sym_r_idx, dst, bytes);
    case GLU_F_L_COL_PTR: return copy_field(s.l_col_ptr, dst, bytes);
    case GLU_F_CSR_R_PTR: return copy_field(s.csr_r_ptr, dst, bytes);
    case GLU_F_CSR_C_IDX: return copy_field(s.csr_c_idx, dst, bytes);
    case GLU_F_CSR_DIAG_PTR: return copy_field(s.csr_diag_ptr, dst, bytes);
    case GLU_F_VAL: return copy_field(s.val, dst, bytes);
    case GLU_F_LEVEL_PTR: return copy_field(s.level_ptr, dst, bytes);
    case GLU_F_LEVEL_IDX: return copy_field(s.level_idx, dst, bytes);
    case GLU_F_ROW_PERM: return copy_field(an.row_perm, dst, bytes);
    case GLU_F_ROW_PERM_INV: return copy_field(an.row_perm_inv, dst, bytes);
    case GLU_F_COL_PERM: return copy_field(an.col_perm, dst, bytes);
    case GLU_F_COL_PERM_INV: return copy_field(an.col_perm_inv, dst, bytes);
    case GLU_F_ROW_SCALE: return copy_field(an.row_scale, dst, bytes);
    case GLU_F_COL_SCALE_PERM: return copy_field(an.col_scale_perm, dst, bytes);
    case GLU_F_DUMP_AX: return copy_field(an.ax, dst, bytes);
    case GLU_F_DUMP_AI: return copy_field(an.ai, dst, bytes);
    case GLU_F_DUMP_AP: return copy_field(an.ap, dst, bytes);
    }
    return fail(GLU_ERR_ARGUMENT, "unknown field");
}

// ---------------------------------------------------------------------------
// plan
// ---------------------------------------------------------------------------

namespace {

constexpr int kGridThreads = 256;
constexpr int kDefaultFusedThreads = 1024;
constexpr int kDefaultKrylov = 2;         // FGMRES(2) cycles after the first solve
constexpr int kDefaultFuseUnits = 2048;   // lanes
constexpr uint32_t kCopyRange = 32768;    // slots (128 KB of LDS) per range of the batch value copy
constexpr int kMaxGroupSplit = 2;         // group members on the single-matrix path, at most

struct Segment {
    int l0, l1;      // levels [l0, l1)
    bool fused;
    uint32_t items;  // grid segments: items (factor) or rows (solve)
    uint32_t k0 = 0, k1 = 0;   // solve segments: dataflow tasks [k0, k1)
    int win = -1;              // factor segments: an LDS window
    int phase = -1;            // factor segments: a phase
};

struct TriHost {
    std::vector<uint32_t> rows, lvl_ptr, lvl_long;
    std::vector<uint32_t> len;     // entries of each row
    std::vector<uint32_t> tasks;   // dataflow task starts (+ end sentinel)
    std::vector<Segment> segs;
};

// Device arena: one allocation, 256-byte aligned sub-buffers.
struct Arena {
    std::vector<std::pair<size_t, size_t>> parts;  // offset, bytes
    size_t total = 0;
    size_t add(size_t bytes)
    {
        size_t off = total;
        total += (bytes + 255) & ~size_t(255);
        parts.push_back({off, bytes});
        return off;
    }
};

}  // namespace

struct glu_plan {
    int device = 0;
    uint32_t n = 0, nnz = 0, nnz_a = 0;
    int num_lev = 0;
    uint32_t ndiv = 0;           // division items of the factorization
    int64_t updates = 0;
    int64_t units = 0;
    int fused_threads = kDefaultFusedThreads;
    int fuse_units = kDefaultFuseUnits;
    bool has_scaling = false, has_refine = false;
    uint32_t a_nlong = 0, a_nlong_t = 0;   // long rows / columns of A
    uint32_t a_kmax = 0;                   // most entries in a row or a column of A

    std::vector<Segment> fsegs;
    std::vector<PhaseDev> phases;
    std::vector<std::vector<uint32_t>> phase_work;   // chunks of each phase's bins
    int phase_lev = 0;           // steps the phases cover
    size_t phase_out = 0;        // products of the largest (PhaseDev::out)
    TriHost tri[4];          // lo, up, tup, tlo
    bool tri_dataflow = false;   // fused solve segments run barrier-free
    int solve_df_opt = 0;        // glu_plan_opts.solve_dataflow
    size_t lds_cap = 0;          // dynamic LDS per workgroup (bytes)
    uint32_t df_nval = 0;        // values of the per-matrix sweep copy
    uint32_t tdf_nval = 0;       // the same for A' x = b
    float *d_tlucsr = nullptr;   // glu_refine's A' x = b value copy
    uint32_t t32_len = 0;        // floats of a matrix's sweep scratch (SolveDev::t32_len)
    uint64_t scratch_nval[2] = {0, 0};   // value copies the scratch limit of glu_refine_noalloc counts (A, A')
    uint32_t rhs_len[2] = {0, 0};        // lanes of the longer of the two sweeps' streams (A, A')
    // one matrix's sweeps outside the batch kernels (A, A'): value copy,
    // right-hand sides, vector by row; allocated on first use, never moved
    struct Single {
        float *buf = nullptr, *lucsr = nullptr, *rhs = nullptr, *xg = nullptr;
    } single[2];
    bool has_split = false;      // vector beyond LDS: split sweeps (split[0]: A, [1]: A')
    SplitDev split[2] = {};
    // LDS windows allowed (from the last level); windows hold narrow steps
    // only, so small orders get one whatever the cap, and n=500k MNA gains
    // up to ~16 (refactor 14.3 -> 12.4 ms; no change beyond)
    int max_windows = 64;
    uint32_t win_values = 0;     // values one window may stage (0: what LDS holds)
    int krylov = kDefaultKrylov;  // batch refinement: FGMRES restart length (0: plain)
    int nwin = 0;                // LDS windows of the factorization
    int win_steps = 0;           // steps they cover
    uint32_t win_nslot = 0;      // the largest window's values
    uint32_t copy_range = 0;     // slots the batch kernels' value copy stages in LDS at a time
    std::vector<uint32_t> win_slots;   // values of each window
    // batched kernels: steps [0, batch_grid_lev) run as one grid launch per
    // step over an interleaved copy of the batch (grid_waves: each one's
    // waves for one group of interleaved matrices: long merges one each,
    // other items il_items_per_wave() a wave)
    int batch_grid_opt = 0;      // glu_plan_opts.batch_grid_levels
    int batch_grid_lev = 0;
    std::vector<uint32_t> grid_waves;

    // hipGraph replay of the launch sequences (use_graph): one executable
    // graph per entry point, keyed on the buffers it was captured with
    struct GraphSlot {
        hipGraphExec_t exec = nullptr;
        const void *k[3] = {nullptr, nullptr, nullptr};
        int mode = -1;
    };
    bool use_graph = false;
    hipStream_t cap_stream = nullptr;
    GraphSlot g_factor, g_solve[2];

    char *d_arena = nullptr;
    size_t arena_bytes = 0;
    FactorDev F{};
    SolveDev S{};
    RefineDev R{};
    MatDesc *d_desc = nullptr;   // lives in the arena

    // scalars and single-matrix workspaces (also in the arena)
    unsigned int *d_norm_bits = nullptr;
    float *d_pert = nullptr;
    unsigned long long *d_norms = nullptr;
    float *d_t32 = nullptr;      // n
    const uint32_t *d_rowidx = nullptr, *d_diag = nullptr;   // sym_r_idx, l_col_ptr (arena)
    float *d_abft = nullptr;     // ABFT column sums of L, n per matrix (grown on demand)
    int abft_cap = 0;
    double *d_r64 = nullptr;     // n
    float *d_val = nullptr;      // nnz (glu_factor_host)

    // batch workspaces, grown on demand
    float *d_bt32 = nullptr;
    double *d_br64 = nullptr;
    float *d_blucsr = nullptr;   // sweep value copies, df_nval per matrix
    double *d_bnorms = nullptr;  // |A|_inf, |b|_inf per matrix
    char *d_rout = nullptr;      // glu_refine's iteration count and backward error (device)
    double *d_bkry = nullptr;    // Arnoldi vectors V, Z = M V, W = A Z: (3 krylov + 1) n per matrix
    int batch_cap = 0;
    double *d_fnorms = nullptr;  // glu_batch_factor: GESP value per matrix (2 doubles each)
    float *d_il = nullptr;       // interleaved batch values (groups of 16 matrices)
    unsigned int *d_il_bits = nullptr;   // per-matrix GESP maxima, zero between calls
    int il_cap = 0;              // matrices d_il, d_il_bits and d_fnorms hold

    ~glu_plan()
    {
        if (d_arena) (void)hipFree(d_arena);
        if (d_val) (void)hipFree(d_val);
        if (d_bt32) (void)hipFree(d_bt32);
        if (d_br64) (void)hipFree(d_br64);
        if (d_blucsr) (void)hipFree(d_blucsr);
        if (d_bkry) (void)hipFree(d_bkry);
        if (d_rout) (void)hipFree(d_rout);
        if (d_tlucsr) (void)hipFree(d_tlucsr);
        for (Single &q : single)
            if (q.buf) (void)hipFree(q.buf);
        if (d_abft) (void)hipFree(d_abft);
        if (d_bnorms) (void)hipFree(d_bnorms);
        if (d_fnorms) (void)hipFree(d_fnorms);
        if (d_il) (void)hipFree(d_il);
        if (d_il_bits) (void)hipFree(d_il_bits);
        for (GraphSlot *g : {&g_factor, &g_solve[0], &g_solve[1]})
            if (g->exec) (void)hipGraphExecDestroy(g->exec);
        if (cap_stream) (void)hipStreamDestroy(cap_stream);
    }
};

namespace {

// ------------------------- validation -----------------------------------

bool check_ptr(const uint32_t *p, uint32_t n, uint32_t total, std::string &err, const char *what)
{
    if (p[0] != 0 || p[n] != total) {
        err = std::string(what) + ": pointer array must start at 0 and end at the entry count";
        return false;
    }
    for (uint32_t i = 0; i < n; ++i)
        if (p[i] > p[i + 1]) {
            err = std::string(what) + ": pointer array not monotone";
            return false;
        }
    return true;
}

bool validate_pattern(const glu_pattern &P, std::string &err)
{
    const uint32_t n = P.n, nnz = P.nnz;
    if (!P.sym_c_ptr || !P.sym_r_idx || !P.l_col_ptr || !P.csr_r_ptr || !P.csr_c_idx || !P.csr_diag_ptr ||
        !P.level_ptr || !P.level_idx) {
        err = "null pattern array";
        return false;
    }
    if (nnz >= 0x80000000u) {
        err = "nnz(L+U) must be below 2^31";
        return false;
    }
    if (P.num_lev <= 0 || (uint32_t)P.num_lev > n) {
        err = "num_lev out of range";
        return false;
    }
    if (!check_ptr(P.sym_c_ptr, n, nnz, err, "sym_c_ptr") || !check_ptr(P.csr_r_ptr, n, nnz, err, "csr_r_ptr"))
        return false;
    for (uint32_t c = 0; c < n; ++c) {
        for (uint32_t p = P.sym_c_ptr[c]; p < P.sym_c_ptr[c + 1]; ++p) {
            if (P.sym_r_idx[p] >= n || (p > P.sym_c_ptr[c] && P.sym_r_idx[p] <= P.sym_r_idx[p - 1])) {
                err = "sym_r_idx out of range or not strictly ascending in column " + std::to_string(c);
                return false;
            }
        }
        const uint32_t d = P.l_col_ptr[c];
        if (d < P.sym_c_ptr[c] || d >= P.sym_c_ptr[c + 1] || P.sym_r_idx[d] != c) {
            err = "l_col_ptr does not point at the diagonal of column " + std::to_string(c);
            return false;
        }
    }
    // CSR must be the exact transpose of the CSC pattern.
    std::vector<uint32_t> cursor(P.csr_r_ptr, P.csr_r_ptr + n);
    for (uint32_t c = 0; c < n; ++c)
        for (uint32_t p = P.sym_c_ptr[c]; p < P.sym_c_ptr[c + 1]; ++p) {
            const uint32_t r = P.sym_r_idx[p];
            const uint32_t q = cursor[r]++;
            if (q >= P.csr_r_ptr[r + 1] || P.csr_c_idx[q] != c) {
                err = "CSR arrays are not the transpose of the CSC pattern";
                return false;
            }
        }
    for (uint32_t r = 0; r < n; ++r) {
        const uint32_t q = P.csr_diag_ptr[r];
        if (q < P.csr_r_ptr[r] || q >= P.csr_r_ptr[r + 1] || P.csr_c_idx[q] != r) {
            err = "csr_diag_ptr does not point at the diagonal of row " + std::to_string(r);
            return false;
        }
    }
    if (P.level_ptr[0] != 0 || (uint32_t)P.level_ptr[P.num_lev] != n) {
        err = "level_ptr must span 0..n";
        return false;
    }
    for (int l = 0; l < P.num_lev; ++l)
        if (P.level_ptr[l] > P.level_ptr[l + 1]) {
            err = "level_ptr not monotone";
            return false;
        }
    std::vector<int> level_of(n, -1);
    for (int l = 0; l < P.num_lev; ++l)
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) {
            const int k = P.level_idx[t];
            if (k < 0 || (uint32_t)k >= n || level_of[k] != -1) {
                err = "level_idx is not a permutation";
                return false;
            }
            level_of[k] = l;
        }
    // Dependencies of the right-looking update must sit in earlier levels
    // (src/symbolic.cc:115-130): otherwise two columns of one level race.
    for (uint32_t i = 0; i < n; ++i) {
        for (uint32_t p = P.sym_c_ptr[i]; p < P.l_col_ptr[i]; ++p) {
            const uint32_t r = P.sym_r_idx[p];
            if (P.l_col_ptr[r] + 1 != P.sym_c_ptr[r + 1] && level_of[r] >= level_of[i]) {
                err = "levels violate a column dependency";
                return false;
            }
        }
        for (uint32_t q = P.csr_r_ptr[i]; q < P.csr_diag_ptr[i]; ++q)
            if (level_of[P.csr_c_idx[q]] >= level_of[i]) {
                err = "levels violate a row dependency";
                return false;
            }
    }
    return true;
}

// --------------------------- tables -------------------------------------

struct Tables {
    std::vector<uint32_t> upos;        // CSR position -> CSC position
    // update map: target of (k, jj, ii) (its jj-th U and ii-th L entry) at
    // moff[k] + jj L(k) + ii (until the phases are built)
    std::vector<uint64_t> moff;
    std::vector<uint32_t> umap;
    // column tasks, by level: task t has lanes 64 t .. 64 t + 63 in cln
    // ({L position, pivot position, update count <= 4, 0}); the lane's e-th
    // update reads U value cup[256 t + 64 e + lane] and targets ctgt[same]
    std::vector<uint4> cln;
    std::vector<uint32_t> ctgt, cup;
    std::vector<uint32_t> ctask_ptr;   // [num_lev + 2]
    std::vector<uint32_t> ment, ment_ptr, ment_long, msrc_ptr;
    std::vector<MergeSrc> msrc;
    std::vector<uint2> dvd;            // division items, in CSC position order
    std::vector<uint32_t> dvd_ptr;     // [num_lev + 1]: items of the columns of levels < l (built by level)
};

// Runs work(worker, i) for i in [0, count) on up to `threads` host threads
// (the calling one included), items taken in increasing order from a shared
// counter.  The first exception thrown in any worker is rethrown here after
// every thread has finished.
template <typename Work>
void parallel_items(size_t count, unsigned threads, Work work)
{
    threads = (unsigned)std::max<size_t>(1, std::min<size_t>(threads, count));
    std::atomic<size_t> next(0);
    std::exception_ptr failure;
    std::mutex fail_mu;
    auto run = [&](unsigned worker) {
        try {
            for (size_t i = next.fetch_add(1); i < count; i = next.fetch_add(1)) work(worker, i);
        } catch (...) {
            std::lock_guard<std::mutex> lock(fail_mu);
            if (!failure) failure = std::current_exception();
            next.store(count);
        }
    };
    std::vector<std::thread> pool;
    try {
        pool.reserve(threads - 1);
        for (unsigned t = 1; t < threads; ++t) pool.emplace_back(run, t);
    } catch (const std::exception &) {
        // fewer threads than asked for: the ones that started share the work
    }
    run(0);
    for (std::thread &t : pool) t.join();
    if (failure) std::rethrow_exception(failure);
}

// Host threads for building plan tables: the cores available, at most 16.
unsigned table_threads()
{
    const unsigned hw = std::thread::hardware_concurrency();
    return std::max(1u, std::min(16u, hw ? hw : 1u));
}

// One level's factorization items (the level's slice of Tables).
struct LevelItems {
    std::vector<uint4> cln;
    std::vector<uint32_t> ctgt, cup;
    std::vector<uint32_t> ment, msrc_cnt;
    uint32_t ment_long = 0;
    std::vector<MergeSrc> msrc;
    std::vector<uint2> dvd;
};

// Lane items of the factorization, level by level.  For pivot column k of
// level l, every (i in L_k, j in U_k) update targets the CSC position of
// (i,j) in column j; the fill closure of the pattern guarantees it exists
// (checked).  Targets that two or more columns of the level update become
// merge entries whose sources keep the order in which level_idx lists the
// level's columns; all other updates are items.
// The update map is built per target column and the items per level, each
// on host threads; levels are then concatenated in order, so the tables do
// not depend on the thread count.
bool build_factor_tables(const glu_pattern &P, Tables &T, int64_t &updates, std::string &err)
{
    const uint32_t n = P.n, nnz = P.nnz;
    const int nl = P.num_lev;
    const unsigned threads = table_threads();
    T.upos.resize(nnz);
    std::vector<uint32_t> csc2csr(nnz);
    {
        std::vector<uint32_t> cursor(P.csr_r_ptr, P.csr_r_ptr + n);
        for (uint32_t c = 0; c < n; ++c)
            for (uint32_t p = P.sym_c_ptr[c]; p < P.sym_c_ptr[c + 1]; ++p) {
                const uint32_t q = cursor[P.sym_r_idx[p]]++;
                T.upos[q] = p;
                csc2csr[p] = q;
            }
    }
    // Scatter targets per (k, jj, ii), built per target column j (columns
    // write disjoint ranges of umap).
    std::vector<uint64_t> &moff = T.moff;
    moff.resize(n + 1);
    uint64_t off = 0;
    for (uint32_t k = 0; k < n; ++k) {
        moff[k] = off;
        const uint64_t L = P.sym_c_ptr[k + 1] - P.l_col_ptr[k] - 1;
        const uint64_t U = P.csr_r_ptr[k + 1] - P.csr_diag_ptr[k] - 1;
        off += L * U;
    }
    moff[n] = off;
    updates = (int64_t)off;
    std::vector<uint32_t> &umap = T.umap;
    try {
        umap.assign(off, 0);
    } catch (const std::bad_alloc &) {
        err = "update tables too large for host memory";
        return false;
    }
    {
        constexpr uint32_t kCols = 256;   // target columns per work item
        std::vector<std::vector<uint32_t>> stamps(threads), wheres(threads);
        std::atomic<uint32_t> bad_col(UINT32_MAX);
        parallel_items((n + kCols - 1) / kCols, threads, [&](unsigned w, size_t item) {
            std::vector<uint32_t> &stamp = stamps[w], &where = wheres[w];
            if (stamp.empty()) {
                stamp.assign(n, UINT32_MAX);
                where.assign(n, 0);
            }
            const uint32_t j1 = std::min<uint32_t>(n, (uint32_t)(item + 1) * kCols);
            for (uint32_t j = (uint32_t)item * kCols; j < j1; ++j) {
                for (uint32_t p = P.sym_c_ptr[j]; p < P.sym_c_ptr[j + 1]; ++p) {
                    stamp[P.sym_r_idx[p]] = j;
                    where[P.sym_r_idx[p]] = p;
                }
                for (uint32_t p = P.sym_c_ptr[j]; p < P.l_col_ptr[j]; ++p) {
                    const uint32_t k = P.sym_r_idx[p];
                    const uint32_t L = P.sym_c_ptr[k + 1] - P.l_col_ptr[k] - 1;
                    if (L == 0) continue;
                    const uint32_t jj = csc2csr[p] - P.csr_diag_ptr[k] - 1;
                    const uint64_t base = moff[k] + (uint64_t)jj * L;
                    const uint32_t l0 = P.l_col_ptr[k] + 1;
                    for (uint32_t ii = 0; ii < L; ++ii) {
                        const uint32_t i = P.sym_r_idx[l0 + ii];
                        if (stamp[i] != j) {
                            uint32_t none = UINT32_MAX;
                            bad_col.compare_exchange_strong(none, j);
                            return;
                        }
                        umap[base + ii] = where[i];
                    }
                }
            }
        });
        if (bad_col.load() != UINT32_MAX) {
            err = "pattern is not closed under fill (column " + std::to_string(bad_col.load()) + ")";
            return false;
        }
    }
    // Items per level, on host threads (each with its own marks over the
    // positions), heaviest levels first.
    std::vector<LevelItems> lv(nl);
    std::vector<uint64_t> lwork(nl, 0);
    for (int l = 0; l < nl; ++l)
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) {
            const uint32_t k = (uint32_t)P.level_idx[t];
            lwork[l] += (moff[k + 1] - moff[k]) + 1;
        }
    std::vector<int> lorder(nl);
    for (int l = 0; l < nl; ++l) lorder[l] = l;
    std::stable_sort(lorder.begin(), lorder.end(), [&](int a, int b) { return lwork[a] > lwork[b]; });
    struct Marks {
        std::vector<uint32_t> stamp, cnt, slot, touched;
    };
    std::vector<Marks> marks(threads);
    parallel_items((size_t)nl, threads, [&](unsigned w, size_t item) {
        const int l = lorder[item];
        Marks &M = marks[w];
        if (M.stamp.empty()) {
            M.stamp.assign(nnz, UINT32_MAX);
            M.cnt.assign(nnz, 0);
            M.slot.assign(nnz, 0);
        }
        LevelItems &out = lv[l];
        auto each_update = [&](auto f) {
            for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) {
                const uint32_t k = (uint32_t)P.level_idx[t];
                const uint32_t dpos = P.l_col_ptr[k];
                const uint32_t L = P.sym_c_ptr[k + 1] - dpos - 1;
                if (L == 0) continue;
                const uint32_t uf = P.csr_diag_ptr[k] + 1;
                const uint32_t U = P.csr_r_ptr[k + 1] - uf;
                for (uint32_t jj = 0; jj < U; ++jj) {
                    const uint32_t up = T.upos[uf + jj];
                    const uint64_t base = moff[k] + (uint64_t)jj * L;
                    for (uint32_t ii = 0; ii < L; ++ii) f(umap[base + ii], dpos + 1 + ii, up, dpos);
                }
            }
        };
        M.touched.clear();
        each_update([&](uint32_t tgt, uint32_t, uint32_t, uint32_t) {
            if (M.stamp[tgt] != (uint32_t)l) {
                M.stamp[tgt] = (uint32_t)l;
                M.cnt[tgt] = 0;
                M.touched.push_back(tgt);
            }
            ++M.cnt[tgt];
        });
        std::sort(M.touched.begin(), M.touched.end());
        // long merge entries (a wave each) first, then the rest
        std::vector<uint32_t> fillpos;
        for (int pass = 0; pass < 2; ++pass)
            for (uint32_t tgt : M.touched) {
                if (M.cnt[tgt] < 2 || (M.cnt[tgt] > kLongMerge) != (pass == 0)) continue;
                M.slot[tgt] = (uint32_t)out.ment.size();
                out.ment.push_back(tgt);
                out.msrc_cnt.push_back(M.cnt[tgt]);
                fillpos.push_back((uint32_t)out.msrc.size());
                out.msrc.resize(out.msrc.size() + M.cnt[tgt]);
                if (pass == 0) ++out.ment_long;
            }
        each_update([&](uint32_t tgt, uint32_t lpos, uint32_t up, uint32_t dpos) {
            if (M.cnt[tgt] >= 2) out.msrc[fillpos[M.slot[tgt]]++] = MergeSrc{lpos, up, dpos, 0};
        });
        // Column tasks: a lane takes one L entry A(i,k) of a pivot column
        // and up to four consecutive entries of its U list; lanes sharing a
        // U chunk are adjacent (they read the same U values), and tasks are
        // 64 lanes.  Merge targets are left to their merge entries (~0u).
        uint32_t used = 64;   // lanes used in the open task
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) {
            const uint32_t k = (uint32_t)P.level_idx[t];
            const uint32_t dpos = P.l_col_ptr[k];
            const uint32_t L = P.sym_c_ptr[k + 1] - dpos - 1;
            const uint32_t U = P.csr_r_ptr[k + 1] - P.csr_diag_ptr[k] - 1;
            if (!L || !U) continue;
            const uint32_t uf = P.csr_diag_ptr[k] + 1;
            for (uint32_t c0 = 0; c0 < U; c0 += 4) {
                const uint32_t nu = std::min<uint32_t>(4, U - c0);
                for (uint32_t ii = 0; ii < L; ++ii) {
                    if (used == 64) {
                        out.cln.resize(out.cln.size() + 64, make_uint4(0u, 0u, 0u, 0u));
                        out.ctgt.resize(out.ctgt.size() + 256, UINT32_MAX);
                        out.cup.resize(out.cup.size() + 256, 0u);
                        used = 0;
                    }
                    const size_t lane = out.cln.size() - 64 + used, slot0 = out.ctgt.size() - 256 + used;
                    out.cln[lane] = make_uint4(dpos + 1 + ii, dpos, nu, 0u);
                    for (uint32_t e = 0; e < nu; ++e) {
                        const uint32_t tgt = umap[moff[k] + (uint64_t)(c0 + e) * L + ii];
                        out.ctgt[slot0 + 64 * e] = M.cnt[tgt] >= 2 ? UINT32_MAX : tgt;
                        out.cup[slot0 + 64 * e] = T.upos[uf + c0 + e];
                    }
                    ++used;
                }
            }
        }
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) {
            const uint32_t k = (uint32_t)P.level_idx[t];
            const uint32_t dpos = P.l_col_ptr[k];
            for (uint32_t p = dpos + 1; p < P.sym_c_ptr[k + 1]; ++p)
                out.dvd.push_back(make_uint2(p, dpos | (p == dpos + 1 ? kFirstBit : 0u)));
        }
    });
    // concatenation in level order
    T.ctask_ptr.assign(nl + 2, 0);
    T.ment_ptr.assign(nl + 2, 0);
    T.ment_long.assign(nl + 1, 0);
    T.dvd_ptr.assign(nl + 1, 0);
    T.msrc_ptr.assign(1, 0);
    size_t ncln = 0, nment = 0, nmsrc = 0, ndvd = 0;
    for (const LevelItems &o : lv) {
        ncln += o.cln.size();
        nment += o.ment.size();
        nmsrc += o.msrc.size();
        ndvd += o.dvd.size();
    }
    T.cln.reserve(ncln);
    T.ctgt.reserve(ncln * 4);
    T.cup.reserve(ncln * 4);
    T.ment.reserve(nment);
    T.msrc_ptr.reserve(nment + 1);
    T.msrc.reserve(nmsrc);
    T.dvd.reserve(ndvd);
    for (int l = 0; l < nl; ++l) {
        LevelItems &o = lv[l];
        T.ctask_ptr[l] = (uint32_t)(T.cln.size() / 64);
        T.ment_ptr[l] = (uint32_t)T.ment.size();
        T.dvd_ptr[l] = (uint32_t)T.dvd.size();
        T.ment_long[l] = o.ment_long;
        T.cln.insert(T.cln.end(), o.cln.begin(), o.cln.end());
        T.ctgt.insert(T.ctgt.end(), o.ctgt.begin(), o.ctgt.end());
        T.cup.insert(T.cup.end(), o.cup.begin(), o.cup.end());
        T.ment.insert(T.ment.end(), o.ment.begin(), o.ment.end());
        for (uint32_t c : o.msrc_cnt) T.msrc_ptr.push_back(T.msrc_ptr.back() + c);
        T.msrc.insert(T.msrc.end(), o.msrc.begin(), o.msrc.end());
        T.dvd.insert(T.dvd.end(), o.dvd.begin(), o.dvd.end());
        o = LevelItems();
    }
    T.ctask_ptr[nl] = T.ctask_ptr[nl + 1] = (uint32_t)(T.cln.size() / 64);
    T.ment_ptr[nl] = T.ment_ptr[nl + 1] = (uint32_t)T.ment.size();
    T.dvd_ptr[nl] = (uint32_t)T.dvd.size();
    if (T.ctgt.size() >= UINT32_MAX || T.msrc.size() >= UINT32_MAX) {
        err = "more than 2^32 update items";
        return false;
    }
    return true;
}

// Level sets of one triangular sweep.  dir > 0: rows ascending, dependencies
// on smaller indices; dir < 0: descending.  deps(r, f) calls f(c) for each
// dependency c of row r; len(r) is the row's entry count.  Within a level,
// rows longer than kLongRow come first (lvl_long of them), then the rest,
// each group in increasing row order.

template <typename Deps, typename Len>
void tri_levels(uint32_t n, int dir, Deps deps, Len len, TriHost &H)
{
    std::vector<int> lev(n, 0);
    int nlev = 0;
    for (uint32_t t = 0; t < n; ++t) {
        const uint32_t r = dir > 0 ? t : n - 1 - t;
        int m = -1;
        deps(r, [&](uint32_t c) { m = std::max(m, lev[c]); });
        lev[r] = m + 1;
        nlev = std::max(nlev, m + 2);
    }
    H.lvl_ptr.assign(nlev + 1, 0);
    H.lvl_long.assign(nlev, 0);
    H.len.resize(n);
    for (uint32_t r = 0; r < n; ++r) H.len[r] = len(r);
    for (uint32_t r = 0; r < n; ++r) {
        ++H.lvl_ptr[lev[r] + 1];
        if (len(r) > kLongRow) ++H.lvl_long[lev[r]];
    }
    for (int l = 0; l < nlev; ++l) H.lvl_ptr[l + 1] += H.lvl_ptr[l];
    H.rows.assign(n, 0);
    std::vector<uint32_t> cur_long(H.lvl_ptr.begin(), H.lvl_ptr.end() - 1), cur_short(nlev);
    for (int l = 0; l < nlev; ++l) cur_short[l] = H.lvl_ptr[l] + H.lvl_long[l];
    for (uint32_t r = 0; r < n; ++r) {
        if (len(r) > kLongRow) H.rows[cur_long[lev[r]]++] = r;
        else H.rows[cur_short[lev[r]]++] = r;
    }
}

void make_segments(const std::vector<uint32_t> &work, uint32_t narrow, std::vector<Segment> &segs)
{
    segs.clear();
    const int nl = (int)work.size();
    int l = 0;
    while (l < nl) {
        if (work[l] > narrow) {
            segs.push_back(Segment{l, l + 1, false, work[l]});
            ++l;
            continue;
        }
        int e = l;
        while (e < nl && work[e] <= narrow) ++e;
        segs.push_back(Segment{l, e, true, 0});
        l = e;
    }
}

// Lanes a level needs: column tasks and long merge entries a wave each.
uint32_t level_lanes(const Tables &T, int l)
{
    const uint32_t nc = T.ctask_ptr[l + 1] - T.ctask_ptr[l];
    const uint32_t nm = T.ment_ptr[l + 1] - T.ment_ptr[l];
    const uint32_t ml = T.ment_long[l];
    return std::max({nc * 64, nm - ml, ml * 64});   // (divisions run after the last step)
}

// LDS windows: runs of consecutive steps whose items touch at most `budget`
// distinct CSC positions run inside one workgroup with those values staged
// in LDS (slots, in increasing position order) and the run's items rewritten
// to address slots.  A run shorter than kMinWindow steps stays in global
// memory (staging would cost more than it saves).
constexpr int kMinWindow = 6;

struct Window {
    int l0 = 0, l1 = 0;            // steps [l0, l1)
    std::vector<uint32_t> pos;     // slot -> CSC position
    std::vector<uint16_t> prog;    // chunks, 64 lanes of eight slots each, stream by stream (WinDev)
    std::vector<uint32_t> hdr;     // [chunks]
    std::vector<uint32_t> wptr;    // [waves + 1]: each wave's chunks
};

// The records {target, L, U, pivot of source 0}, {L, U, pivot of source 1,
// source count} of merge entries [e0, e1), positions through map.
template <typename Map>
void merge_records(const std::vector<uint32_t> &ment, const std::vector<uint32_t> &msrc_ptr,
                   const std::vector<MergeSrc> &msrc, uint32_t e0, uint32_t e1, Map map, std::vector<uint4> &out)
{
    for (uint32_t e = e0; e < e1; ++e) {
        const uint32_t s = msrc_ptr[e], cnt = msrc_ptr[e + 1] - s;
        const MergeSrc &a = msrc[s], &b = msrc[s + 1];
        out.push_back(make_uint4(map(ment[e]), map(a.lpos), map(a.upos), map(a.dpos)));
        out.push_back(make_uint4(map(b.lpos), map(b.upos), map(b.dpos), cnt));
    }
}

// The CSC positions the items of step l read or write, each once per call
// of f (duplicates possible).  Division items are not step items: they run
// after the last step, on the values in global memory.
template <typename F>
void step_positions(const Tables &T, int l, F f)
{
    for (uint32_t t = T.ctask_ptr[l]; t < T.ctask_ptr[l + 1]; ++t)
        for (uint32_t lane = 0; lane < 64; ++lane) {
            const uint4 &ln = T.cln[(size_t)t * 64 + lane];
            if (ln.z == 0) continue;
            f(ln.x), f(ln.y);
            for (uint32_t e = 0; e < ln.z; ++e) {
                const size_t q = 256 * (size_t)t + 64 * e + lane;
                f(T.cup[q]);
                if (T.ctgt[q] != UINT32_MAX) f(T.ctgt[q]);
            }
        }
    for (uint32_t e = T.ment_ptr[l]; e < T.ment_ptr[l + 1]; ++e) {
        f(T.ment[e]);
        for (uint32_t k = T.msrc_ptr[e]; k < T.msrc_ptr[e + 1]; ++k) {
            const MergeSrc &m = T.msrc[k];
            f(m.lpos), f(m.upos), f(m.dpos);
        }
    }
}

// Merge entries of up to kWinLaneMerge sources take a lane each (two sources
// a chunk), larger ones 16 lanes each (a chunk of 32 sources takes about two
// lane chunks' time).
constexpr uint32_t kWinLaneMerge = 4;

// The streams of one window or of one bin of a phase, step by step.  A step's
// single updates become column chunks (a lane: one L entry, up to three of
// its U entries; lanes that share U entries side by side).  Its chains of
// chunks go to the waves longest first, each to the wave with the least so
// far.
class WinBuilder {
public:
    struct Src {
        uint16_t l, u, d;
    };

    void begin(uint32_t nslot, uint32_t waves)
    {
        zero = nslot, one = nslot + 1, sink = nslot + 2;
        data.assign(waves, {});
        head.assign(waves, {});
        load.assign(waves, 0);
        clear();
    }
    // The single updates of one column: pivot slot d, its L entries' slots,
    // and {u, t} by L entry.
    void column(uint16_t d, size_t L, const uint16_t *l, const std::vector<std::vector<std::pair<uint16_t, uint16_t>>> &ut)
    {
        size_t longest = 0;
        for (size_t i = 0; i < L; ++i) longest = std::max(longest, ut[i].size());
        for (size_t r = 0; r < longest; r += 3)
            for (size_t i = 0; i < L; ++i) {
                if (ut[i].size() <= r) continue;
                uint16_t *e = lane(kWinCol, 10);
                e[0] = l[i];
                e[1] = d;
                for (size_t k = r; k < std::min(r + 3, ut[i].size()); ++k) {
                    e[2 + 2 * (k - r)] = ut[i][k].first;
                    e[3 + 2 * (k - r)] = ut[i][k].second;
                }
            }
    }
    // A merge entry and its sources in order.
    void merge(uint16_t t, const Src *src, uint32_t cnt)
    {
        merges.push_back(Merge{t, (uint32_t)srcs.size(), cnt});
        srcs.insert(srcs.end(), src, src + cnt);
    }
    // Up to two products of L entry l (pivot d): u[i] times it to place o[i].
    void product(uint16_t l, uint16_t d, uint32_t n, const uint16_t *u, const uint32_t *o)
    {
        uint16_t *e = lane(kWinOut, 10);
        e[0] = l;
        e[1] = d;
        for (uint32_t i = 0; i < n; ++i) {
            e[2 + i] = u[i];
            std::memcpy(e + 4 + 2 * i, &o[i], 4);
        }
    }
    void end_step(uint32_t step)
    {
        std::vector<Merge> one_lane, group;
        for (const Merge &m : merges) (m.cnt <= kWinLaneMerge ? one_lane : group).push_back(m);
        const auto most = [](const Merge &x, const Merge &y) { return x.cnt > y.cnt; };
        std::stable_sort(one_lane.begin(), one_lane.end(), most);
        std::stable_sort(group.begin(), group.end(), most);
        for (size_t i = 0; i < one_lane.size(); i += 64) {
            const uint32_t n = (one_lane[i].cnt + 1) / 2;
            chains.push_back(Chain{(uint32_t)kind.size(), n, 12 * n});
            for (uint32_t c = 0; c < n; ++c) {
                const size_t at = chunk(kWinMerge);
                for (size_t k = i; k < std::min(i + 64, one_lane.size()); ++k) {
                    const Merge &m = one_lane[k];
                    const uint32_t own = (m.cnt + 1) / 2;
                    if (c >= own) continue;   // this entry is done
                    uint16_t *e = &buf[at + 8 * (k - i)];
                    e[0] = m.t;
                    e[1] = (uint16_t)((c == 0 ? kWinFirst : 0) | (c + 1 == own ? kWinLast : 0));
                    for (uint32_t x = 2 * c; x < std::min(2 * c + 2, m.cnt); ++x) put(e + 2 + 3 * (x - 2 * c), srcs[m.first + x]);
                }
            }
        }
        for (size_t i = 0; i < group.size(); i += 4) {
            const uint32_t top = group[i].cnt, n = (top + 31) / 32;
            const bool half_last = top - 32 * (n - 1) <= 16;   // the last chunk uses 16 sources only
            chains.push_back(Chain{(uint32_t)kind.size(), n, 35 * n - (half_last ? 10 : 0)});
            for (uint32_t c = 0; c < n; ++c) {
                const size_t at = chunk(half_last && c + 1 == n ? kWinGroup1 : kWinGroup);
                for (size_t k = i; k < std::min(i + 4, group.size()); ++k) {
                    const Merge &m = group[k];
                    const uint32_t own = (m.cnt + 31) / 32;
                    if (c >= own) continue;
                    for (uint32_t ln = 0; ln < 16; ++ln) {
                        uint16_t *e = &buf[at + 8 * (16 * (k - i) + ln)];
                        e[6] = m.t;
                        e[7] = (uint16_t)((c == 0 ? kWinFirst : 0) | (c + 1 == own ? kWinLast : 0));
                        for (uint32_t x = 0; x < 2; ++x)
                            if (32 * c + 16 * x + ln < m.cnt) put(e + 3 * x, srcs[m.first + 32 * c + 16 * x + ln]);
                    }
                }
            }
        }
        std::stable_sort(chains.begin(), chains.end(), [](const Chain &x, const Chain &y) { return x.cost > y.cost; });
        std::fill(load.begin(), load.end(), 0);
        for (const Chain &c : chains) {
            const size_t to = std::min_element(load.begin(), load.end()) - load.begin();
            load[to] += c.cost;
            data[to].insert(data[to].end(), buf.begin() + 512 * (size_t)c.first, buf.begin() + 512 * (size_t)(c.first + c.count));
            for (uint32_t k = c.first; k < c.first + c.count; ++k) head[to].push_back(kind[k] << kWinKindShift | step);
        }
        clear();
    }
    void finish(Window &w) const
    {
        w.wptr.assign(1, 0);
        for (size_t v = 0; v < data.size(); ++v) {
            w.prog.insert(w.prog.end(), data[v].begin(), data[v].end());
            w.hdr.insert(w.hdr.end(), head[v].begin(), head[v].end());
            w.wptr.push_back((uint32_t)w.hdr.size());
        }
    }

private:
    struct Chain {   // chunks [first, first + count) of the step, run in order by one wave
        uint32_t first, count, cost;
    };
    struct Merge {
        uint16_t t;
        uint32_t first, cnt;
    };
    uint32_t zero = 0, one = 0, sink = 0;
    std::vector<std::vector<uint16_t>> data;   // per wave
    std::vector<std::vector<uint32_t>> head;
    std::vector<uint64_t> load;
    std::vector<uint16_t> buf;                 // the step's chunks
    std::vector<uint32_t> kind;
    std::vector<Chain> chains;
    std::vector<Merge> merges;
    std::vector<Src> srcs;
    uint32_t used = 64, open = 0;              // lanes used in the open chunk, its kind

    void clear()
    {
        buf.clear();
        kind.clear();
        chains.clear();
        merges.clear();
        srcs.clear();
        used = 64;
    }
    static void put(uint16_t *e, const Src &s) { e[0] = s.l, e[1] = s.u, e[2] = s.d; }
    // a chunk of kind kd whose lanes do nothing
    size_t chunk(uint32_t kd)
    {
        const size_t at = buf.size();
        buf.resize(at + 64 * 8);
        kind.push_back(kd);
        for (uint32_t ln = 0; ln < 64; ++ln) {
            const uint16_t z = (uint16_t)zero, o = (uint16_t)one, t = (uint16_t)(sink + ln);
            const uint16_t col[8] = {z, o, z, t, z, t, z, t};
            const uint16_t mrg[8] = {t, 0, z, z, o, z, z, o};
            const uint16_t grp[8] = {z, z, o, z, z, o, t, 0};
            const uint16_t out[8] = {z, o, z, z, 0xffff, 0xffff, 0xffff, 0xffff};
            std::copy_n(kd == kWinCol ? col : kd == kWinMerge ? mrg : kd == kWinOut ? out : grp, 8, &buf[at + 8 * ln]);
        }
        return at;
    }
    // the next lane of the open chunk of kind kd (one lane, one item)
    uint16_t *lane(uint32_t kd, uint32_t cost)
    {
        if (used == 64 || open != kd) {
            chains.push_back(Chain{(uint32_t)kind.size(), 1, cost});
            chunk(kd);
            used = 0;
            open = kd;
        }
        return &buf[buf.size() - 512 + 8 * used++];
    }
};

void make_window(const Tables &T, int a, int b, const std::vector<uint32_t> &slot_of_pos,
                 const std::vector<uint32_t> &pos, uint32_t waves, Window &w)
{
    w.l0 = a;
    w.l1 = b;
    w.pos = pos;
    auto slot = [&](uint32_t q) { return (uint16_t)slot_of_pos[q]; };
    WinBuilder B;
    B.begin((uint32_t)pos.size(), waves);
    std::vector<std::vector<std::pair<uint16_t, uint16_t>>> lists;   // a column's single updates {u, t} by L entry
    std::vector<uint16_t> lslot;
    std::vector<WinBuilder::Src> src;
    for (int l = a; l < b; ++l) {
        const size_t q1 = 64 * (size_t)T.ctask_ptr[l + 1];
        for (size_t q = 64 * (size_t)T.ctask_ptr[l]; q < q1;) {
            if (T.cln[q].z == 0) {
                ++q;
                continue;
            }
            // the lanes of one column: its L entries for each four U entries
            const size_t s = q;
            size_t e = s;
            while (e < q1 && T.cln[e].z && T.cln[e].y == T.cln[s].y) ++e;
            size_t L = 1;
            while (s + L < e && T.cln[s + L].x != T.cln[s].x) ++L;
            if (lists.size() < L) lists.resize(L);
            lslot.resize(L);
            for (size_t ii = 0; ii < L; ++ii) {
                lists[ii].clear();
                lslot[ii] = slot(T.cln[s + ii].x);
                for (size_t c = s + ii; c < e; c += L)
                    for (uint32_t k = 0; k < T.cln[c].z; ++k) {
                        const size_t at = 256 * (c / 64) + 64 * k + c % 64;
                        if (T.ctgt[at] != UINT32_MAX) lists[ii].push_back({slot(T.cup[at]), slot(T.ctgt[at])});
                    }
            }
            B.column(slot(T.cln[s].y), L, lslot.data(), lists);
            q = e;
        }
        for (uint32_t e = T.ment_ptr[l]; e < T.ment_ptr[l + 1]; ++e) {
            src.clear();
            for (uint32_t k = T.msrc_ptr[e]; k < T.msrc_ptr[e + 1]; ++k)
                src.push_back({slot(T.msrc[k].lpos), slot(T.msrc[k].upos), slot(T.msrc[k].dpos)});
            B.merge(slot(T.ment[e]), src.data(), (uint32_t)src.size());
        }
        B.end_step((uint32_t)(l - a));
    }
    B.finish(w);
}

// Windows chosen backward from the last step, so that the final run (the
// longest chain of short steps) is one window.  Apart from that final
// window, windows hold narrow steps only (at most `narrow` lanes): a window
// runs in one workgroup, so a wide step inside it would give up the grid's
// parallelism.
void choose_windows(const Tables &T, int num_lev, uint32_t nnz, uint32_t budget, uint32_t narrow, int max_windows,
                    uint32_t waves, std::vector<Window> &wins)
{
    wins.clear();
    if (budget == 0 || max_windows <= 0) return;
    std::vector<uint32_t> stamp(nnz, UINT32_MAX), slot_of_pos(nnz, UINT32_MAX);
    std::vector<uint32_t> fresh;
    int b = num_lev + 1;
    uint32_t gen = 0;
    while (b > 0 && (int)wins.size() < max_windows) {
        const uint32_t lim = b == num_lev + 1 ? UINT32_MAX : narrow;
        if (level_lanes(T, b - 1) > lim) {
            --b;
            continue;
        }
        ++gen;
        uint32_t count = 0;
        int a = b;
        while (a > 0 && level_lanes(T, a - 1) <= lim) {
            fresh.clear();
            step_positions(T, a - 1, [&](uint32_t q) {
                if (stamp[q] != gen) {
                    stamp[q] = gen;
                    fresh.push_back(q);
                }
            });
            if (count + fresh.size() > budget) {
                for (uint32_t q : fresh) stamp[q] = UINT32_MAX;
                break;
            }
            count += (uint32_t)fresh.size();
            --a;
        }
        if (b - a < kMinWindow) {
            b = a < b ? a : b - 1;   // too short: leave these steps in global memory
            continue;
        }
        std::vector<uint32_t> pos;
        for (int l = a; l < b; ++l)
            step_positions(T, l, [&](uint32_t q) {
                if (slot_of_pos[q] == UINT32_MAX) {
                    slot_of_pos[q] = 0;
                    pos.push_back(q);
                }
            });
        std::sort(pos.begin(), pos.end());
        for (uint32_t i = 0; i < pos.size(); ++i) slot_of_pos[pos[i]] = i;
        wins.emplace_back();
        make_window(T, a, b, slot_of_pos, pos, waves, wins.back());
        for (uint32_t q : pos) slot_of_pos[q] = UINT32_MAX;
        b = a;
    }
    std::reverse(wins.begin(), wins.end());
}

// A phase (PhaseDev): steps [l0, l1), the bins' streams (Window: entries and
// programs) and the products' assembly.
struct Phase {
    int l0 = 0, l1 = 0;
    std::vector<Window> bin;
    std::vector<uint2> grp;
    std::vector<uint32_t> tgt;
    std::vector<uint8_t> cnt;
    std::vector<AsmWave> wav;
    uint32_t nout = 0, nslot = 0;
};

constexpr uint32_t kPhaseWaves = 8;
constexpr uint32_t kPhaseBins = 512;       // two workgroups a CU
constexpr uint32_t kPhaseSlots = 19000;    // entries of a bin, at most (76 KB: two a CU)
constexpr int kMinPhase = 4;               // steps

// Whether steps gain from being a phase, estimated in us (measured over MNA,
// mesh and dense patterns).  A step as a launch of its own: 4.1, and 16 ns for
// each source of its longest merge entry and 20 ns per 1,000 lanes (4.2 to 5 on
// meshes and dense patterns, 13 where a rail's entry has 500 sources).  A phase:
// its two launches, 0.3 a step, the updates of the bin with the most at 1 ns
// (0.36 to 1.2 ns: one workgroup) or all of them at 8 ps (the whole card),
// and the longest entry's products at 3.5 ns.  What decides is how much of the
// work falls on one bin: the leading steps of a circuit fall apart into
// hundreds of components (n=200,003: 42 steps, 30 M updates over 512 bins,
// 292 us for about 700), a mesh's soon join into a few (a 300 x 300 mesh, all
// steps in 63 phases of 1 to 237 bins: 93 ms, as launches 9.7) and a dense
// pattern's are one (n=600: 29 ms, as launches 2.5).
struct StepCost {
    double us;
    uint64_t updates;
    uint32_t longest;      // sources of its longest merge entry
};

std::vector<StepCost> step_costs(const glu_pattern &P, const Tables &T, int limit)
{
    std::vector<StepCost> cost(limit);
    for (int l = 0; l < limit; ++l) {
        StepCost &c = cost[l];
        c.updates = 0;
        c.longest = 0;
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) c.updates += T.moff[P.level_idx[t] + 1] - T.moff[P.level_idx[t]];
        for (uint32_t e = T.ment_ptr[l]; e < T.ment_ptr[l + 1]; ++e) c.longest = std::max(c.longest, T.msrc_ptr[e + 1] - T.msrc_ptr[e]);
        c.us = 4.1 + 0.016 * c.longest + 2e-5 * level_lanes(T, l);
    }
    return cost;
}

constexpr double kEven = 5.0;

double phase_us(int steps, uint64_t updates, uint64_t most, uint64_t longest)
{
    return 10.0 + 0.3 * steps + std::max(1e-3 * (double)most, 8e-6 * (double)updates) + 3.5e-3 * (double)longest;
}

// The steps from l0 on that make a phase, at most to `limit` and as long as
// every component's entries fit a bin (of bin_slots): at least kMinPhase, as
// many as gain the most within kEven (the estimate errs on the bins' side:
// n=20,000 38 steps 605 us, the 37 it puts 2 us ahead 608).  Components of the columns of steps [l0, e):
// joined by entries of L or U between them.  Returns e (l0: none) and each
// column's component (UINT32_MAX: not in the phase).
int phase_end(const glu_pattern &P, const Tables &T, const std::vector<StepCost> &cost, int l0, int limit, uint32_t bin_slots,
              std::vector<uint32_t> &comp)
{
    const uint32_t n = P.n;
    std::vector<uint32_t> parent(n), ent(n);
    std::vector<uint64_t> work(n);
    std::vector<uint8_t> seen(n);
    auto find = [&](uint32_t r) {
        while (parent[r] != r) r = parent[r] = parent[parent[r]];
        return r;
    };
    // column k joins what it shares an entry with among the columns seen;
    // returns its component
    auto add = [&](uint32_t k) {
        seen[k] = 1;
        auto join = [&](uint32_t r) {
            if (!seen[r]) return;
            const uint32_t a = find(r), c = find(k);
            if (a == c) return;
            parent[a] = c;
            ent[c] += ent[a];
            work[c] += work[a];
        };
        for (uint32_t q = P.csr_r_ptr[k]; q < P.csr_r_ptr[k + 1]; ++q) join(P.csr_c_idx[q]);
        for (uint32_t q = P.sym_c_ptr[k]; q < P.sym_c_ptr[k + 1]; ++q) join(P.sym_r_idx[q]);
        return find(k);
    };
    auto reset = [&]() {
        for (uint32_t k = 0; k < n; ++k) {
            parent[k] = k;
            ent[k] = (P.sym_c_ptr[k + 1] - P.l_col_ptr[k]) + (P.csr_r_ptr[k + 1] - P.csr_diag_ptr[k] - 1);
            work[k] = T.moff[k + 1] - T.moff[k];
            seen[k] = 0;
        }
    };
    reset();
    int best = l0;
    double gain = 0.0, launches = 0.0;
    uint64_t updates = 0, most = 0, longest = 0;
    for (int e = l0; e < limit; ++e) {
        bool fits = true;
        for (int t = P.level_ptr[e]; t < P.level_ptr[e + 1]; ++t) {
            const uint32_t c = add((uint32_t)P.level_idx[t]);
            fits = ent[c] <= bin_slots && fits;
            most = std::max(most, work[c]);
        }
        if (!fits) break;
        launches += cost[e].us;
        updates += cost[e].updates;
        longest += cost[e].longest;
        const int steps = e + 1 - l0;
        const double g = launches - phase_us(steps, updates, std::max<uint64_t>(most, updates / kPhaseBins), longest);
        if (steps >= kMinPhase && g > 0.0 && g >= gain - kEven) best = e + 1;
        gain = std::max(gain, g);
    }
    reset();   // (without the steps after the best)
    for (int l = l0; l < best; ++l)
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) (void)add((uint32_t)P.level_idx[t]);
    comp.assign(n, UINT32_MAX);
    for (int l = l0; l < best; ++l)
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) comp[P.level_idx[t]] = find((uint32_t)P.level_idx[t]);
    return best;
}

// The streams and the assembly of the phase of steps [ph.l0, ph.l1) with the
// columns' components comp.  False: an update would cross components (the
// pattern's levels do not order it; the steps stay as they are).  The update
// map of the phase's columns, which nothing else reads from here on, is
// overwritten: updates of later entries get their products' places (kPlace).
constexpr uint32_t kPlace = 0x80000000u;   // (positions are below 2^31)

bool build_phase(const glu_pattern &P, Tables &T, const std::vector<int> &level_of,
                 const std::vector<uint32_t> &comp, uint32_t bin_slots, Phase &ph)
{
    const uint32_t n = P.n;
    const unsigned threads = table_threads();
    // components -> bins, largest first, each to the bin with the least work
    std::vector<uint32_t> id(n, UINT32_MAX), size;
    std::vector<uint64_t> work;
    uint64_t total = 0;
    for (uint32_t k = 0; k < n; ++k) {
        if (comp[k] == UINT32_MAX) continue;
        uint32_t &c = id[comp[k]];
        if (c == UINT32_MAX) {
            c = (uint32_t)size.size();
            size.push_back(0);
            work.push_back(0);
        }
        const uint32_t e = (P.sym_c_ptr[k + 1] - P.l_col_ptr[k]) + (P.csr_r_ptr[k + 1] - P.csr_diag_ptr[k] - 1);
        size[c] += e;
        work[c] += T.moff[k + 1] - T.moff[k] + e;
        total += T.moff[k + 1] - T.moff[k] + e;
    }
    std::vector<uint32_t> order(size.size()), bin_of(size.size());
    for (uint32_t c = 0; c < order.size(); ++c) order[c] = c;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return work[a] > work[b]; });
    const uint32_t nbin = (uint32_t)std::min<uint64_t>({(uint64_t)size.size(), kPhaseBins, total / 2048 + 1});
    std::vector<uint64_t> load(nbin, 0);
    std::vector<uint32_t> fill(nbin, 0);
    for (uint32_t c : order) {
        uint32_t to = UINT32_MAX;
        for (uint32_t b = 0; b < nbin; ++b)
            if (fill[b] + size[c] <= bin_slots && (to == UINT32_MAX || load[b] < load[to])) to = b;
        if (to == UINT32_MAX) {   // no room: one more bin
            to = (uint32_t)load.size();
            load.push_back(0);
            fill.push_back(0);
        }
        load[to] += work[c];
        fill[to] += size[c];
        bin_of[c] = to;
    }
    const uint32_t nb = (uint32_t)load.size();
    // columns of each bin by step, and the bin and slot of each entry it owns
    std::vector<std::vector<uint32_t>> cols(nb);
    for (int l = ph.l0; l < ph.l1; ++l)
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) {
            const uint32_t k = (uint32_t)P.level_idx[t];
            cols[bin_of[id[comp[k]]]].push_back(k);
        }
    std::vector<uint32_t> own(P.nnz, UINT32_MAX);   // bin of an entry
    std::vector<uint16_t> slot(P.nnz, 0);
    ph.bin.resize(nb);
    parallel_items(nb, threads, [&](unsigned, size_t b) {
        std::vector<uint32_t> &pos = ph.bin[b].pos;
        for (uint32_t k : cols[b]) {
            for (uint32_t p = P.l_col_ptr[k]; p < P.sym_c_ptr[k + 1]; ++p) pos.push_back(p);
            for (uint32_t q = P.csr_diag_ptr[k] + 1; q < P.csr_r_ptr[k + 1]; ++q) pos.push_back(T.upos[q]);
        }
        std::sort(pos.begin(), pos.end());
        for (uint32_t i = 0; i < pos.size(); ++i) {
            own[pos[i]] = (uint32_t)b;
            slot[pos[i]] = (uint16_t)i;
        }
    });
    // products per later entry: column j's pivots of the phase in schedule
    // order (step by step, a step's columns as level_idx lists them, the order
    // of every other path); cnt by position, then each product's place
    std::vector<uint32_t> cnt(P.nnz, 0);
    std::vector<uint32_t> csc2csr(P.nnz);
    for (uint32_t q = 0; q < P.nnz; ++q) csc2csr[T.upos[q]] = q;
    std::atomic<bool> crossed(false);
    std::vector<int> place_of(n);
    for (int t = 0; t < (int)n; ++t) place_of[P.level_idx[t]] = t;
    auto each_outside = [&](uint32_t j, bool in_order, std::vector<std::pair<int, uint32_t>> &ks, auto f) {
        ks.clear();
        for (uint32_t p = P.sym_c_ptr[j]; p < P.l_col_ptr[j]; ++p)
            if (comp[P.sym_r_idx[p]] != UINT32_MAX) ks.push_back({place_of[P.sym_r_idx[p]], p});
        if (in_order) std::sort(ks.begin(), ks.end());
        for (const auto &[at_place, p] : ks) {
            const uint32_t k = P.sym_r_idx[p], L = P.sym_c_ptr[k + 1] - P.l_col_ptr[k] - 1;
            const uint64_t at = T.moff[k] + (uint64_t)(csc2csr[p] - P.csr_diag_ptr[k] - 1) * L;
            for (uint32_t ii = 0; ii < L; ++ii) {
                const uint32_t t = T.umap[at + ii];
                if (own[t] == UINT32_MAX) f(at + ii, t);
                else if (own[t] != bin_of[id[comp[k]]]) crossed.store(true);
            }
        }
    };
    std::vector<std::vector<std::pair<int, uint32_t>>> scratch(threads);
    constexpr uint32_t kCols = 128;
    const size_t items = (n + kCols - 1) / kCols;
    parallel_items(items, threads, [&](unsigned w, size_t item) {
        for (uint32_t j = (uint32_t)item * kCols; j < std::min<uint32_t>(n, (uint32_t)(item + 1) * kCols); ++j)
            each_outside(j, false, scratch[w], [&](uint64_t, uint32_t t) { ++cnt[t]; });
    });
    if (crossed.load()) return false;
    // entries by product count: groups of 64 of about the same, waves for the rest
    std::vector<uint32_t> few, many, with(kAsmLane + 2, 0);   // with[c]: entries of more than c products, at most kAsmLane
    for (uint32_t p = 0; p < P.nnz; ++p)
        if (cnt[p] > kAsmLane) many.push_back(p);
        else if (cnt[p]) ++with[cnt[p] - 1];
    for (uint32_t c = kAsmLane; c-- > 0;) with[c] += with[c + 1];
    few.resize(with[0]);
    for (uint32_t p = 0; p < P.nnz; ++p)   // most products first, then by position
        if (cnt[p] && cnt[p] <= kAsmLane) few[with[cnt[p]]++] = p;
    std::stable_sort(many.begin(), many.end(), [&](uint32_t a, uint32_t b) { return cnt[a] > cnt[b]; });
    uint64_t out = 0;
    std::vector<uint32_t> next(P.nnz, UINT32_MAX);   // place of the entry's next product; kPlace: 64 apart
    for (size_t i = 0; i < few.size(); i += 64) {
        const uint32_t m = cnt[few[i]];
        ph.grp.push_back(make_uint2((uint32_t)out, m));
        for (size_t k = i; k < i + 64; ++k) {
            ph.tgt.push_back(k < few.size() ? few[k] : UINT32_MAX);
            ph.cnt.push_back(k < few.size() ? (uint8_t)cnt[few[k]] : 0);
            if (k < few.size()) next[few[k]] = kPlace | (uint32_t)(out + (k - i));
        }
        out += 64 * (uint64_t)m;
    }
    for (uint32_t p : many) {
        ph.wav.push_back(AsmWave{p, (uint32_t)out, cnt[p], 0});
        next[p] = (uint32_t)out;
        out += (cnt[p] + 63u) & ~63u;
    }
    if (out >= kPlace) return false;
    ph.nout = (uint32_t)out;
    parallel_items(items, threads, [&](unsigned w, size_t item) {
        for (uint32_t j = (uint32_t)item * kCols; j < std::min<uint32_t>(n, (uint32_t)(item + 1) * kCols); ++j)
            each_outside(j, true, scratch[w], [&](uint64_t at, uint32_t t) {
                T.umap[at] = kPlace | next[t];
                next[t] += (next[t] & kPlace) ? 64u : 1u;
            });
    });
    // each bin's program: its steps' inner updates, then all its products
    struct Marks {
        std::vector<uint32_t> stamp, count, first;
        uint32_t gen = 0;
    };
    std::vector<Marks> marks(threads);
    parallel_items(nb, threads, [&](unsigned wk, size_t b) {
        Marks &M = marks[wk];
        if (M.stamp.empty()) {   // by slot
            M.stamp.assign(0x10000, 0);
            M.count.assign(0x10000, 0);
            M.first.assign(0x10000, 0);
        }
        Window &w = ph.bin[b];
        w.l0 = 0;
        w.l1 = ph.l1 - ph.l0;
        WinBuilder B;
        B.begin((uint32_t)w.pos.size(), kPhaseWaves);
        std::vector<std::vector<std::pair<uint16_t, uint16_t>>> lists;
        std::vector<uint16_t> lslot, order;
        std::vector<WinBuilder::Src> src;
        size_t i = 0;
        for (int l = ph.l0; l < ph.l1; ++l) {
            size_t e = i;
            while (e < cols[b].size() && level_of[cols[b][e]] == l) ++e;
            if (e == i) continue;
            auto inner = [&](auto f) {   // f(column, jj, ii, L, target slot)
                for (size_t c = i; c < e; ++c) {
                    const uint32_t k = cols[b][c], L = P.sym_c_ptr[k + 1] - P.l_col_ptr[k] - 1;
                    if (L == 0) continue;
                    const uint32_t U = P.csr_r_ptr[k + 1] - P.csr_diag_ptr[k] - 1;
                    for (uint32_t jj = 0; jj < U; ++jj)
                        for (uint32_t ii = 0; ii < L; ++ii) {
                            const uint32_t t = T.umap[T.moff[k] + (uint64_t)jj * L + ii];
                            if (!(t & kPlace)) f(k, jj, ii, slot[t]);
                        }
                }
            };
            ++M.gen;
            order.clear();
            inner([&](uint32_t, uint32_t, uint32_t, uint16_t t) {
                if (M.stamp[t] != M.gen) {
                    M.stamp[t] = M.gen;
                    M.count[t] = 0;
                    order.push_back(t);
                }
                ++M.count[t];
            });
            uint32_t nsrc = 0;
            for (uint16_t t : order)
                if (M.count[t] >= 2) {
                    M.first[t] = nsrc;
                    nsrc += M.count[t];
                }
            src.resize(nsrc);
            // (the bin lists its columns in schedule order, so a merge entry's sources come in it)
            for (size_t c = i; c < e; ++c) {
                const uint32_t k = cols[b][c], dpos = P.l_col_ptr[k], L = P.sym_c_ptr[k + 1] - dpos - 1;
                if (L == 0) continue;
                const uint32_t U = P.csr_r_ptr[k + 1] - P.csr_diag_ptr[k] - 1;
                if (lists.size() < L) lists.resize(L);
                lslot.resize(L);
                for (uint32_t ii = 0; ii < L; ++ii) {
                    lists[ii].clear();
                    lslot[ii] = slot[dpos + 1 + ii];
                }
                for (uint32_t jj = 0; jj < U; ++jj) {
                    const uint16_t u = slot[T.upos[P.csr_diag_ptr[k] + 1 + jj]];
                    for (uint32_t ii = 0; ii < L; ++ii) {
                        const uint32_t q = T.umap[T.moff[k] + (uint64_t)jj * L + ii];
                        if (q & kPlace) continue;
                        const uint16_t t = slot[q];
                        if (M.count[t] >= 2) src[M.first[t]++] = {lslot[ii], u, slot[dpos]};
                        else lists[ii].push_back({u, t});
                    }
                }
                B.column(slot[dpos], L, lslot.data(), lists);
            }
            for (uint16_t t : order)
                if (M.count[t] >= 2) B.merge(t, &src[M.first[t] - M.count[t]], M.count[t]);
            B.end_step((uint32_t)(l - ph.l0));
            i = e;
        }
        for (uint32_t k : cols[b]) {
            const uint32_t dpos = P.l_col_ptr[k], L = P.sym_c_ptr[k + 1] - dpos - 1;
            const uint32_t U = P.csr_r_ptr[k + 1] - P.csr_diag_ptr[k] - 1;
            // two U entries a lane, the L entries side by side
            for (uint32_t jj = 0; jj < U; jj += 2)
                for (uint32_t ii = 0; ii < L; ++ii) {
                    uint16_t u[2];
                    uint32_t o[2], m = 0;
                    for (uint32_t x = jj; x < std::min(jj + 2, U); ++x) {
                        const uint32_t at = T.umap[T.moff[k] + (uint64_t)x * L + ii];
                        if (!(at & kPlace)) continue;
                        u[m] = slot[T.upos[P.csr_diag_ptr[k] + 1 + x]];
                        o[m++] = at & ~kPlace;
                    }
                    if (m) B.product(slot[dpos + 1 + ii], slot[dpos], m, u, o);
                }
        }
        B.end_step((uint32_t)(ph.l1 - ph.l0));
        B.finish(w);
    });
    for (const Window &w : ph.bin) ph.nslot = std::max<uint32_t>(ph.nslot, (uint32_t)w.pos.size());
    return true;
}

// The phases ahead of step `limit` (the first LDS window's), their bins of
// bin_slots entries at most.
void choose_phases(const glu_pattern &P, Tables &T, int limit, uint32_t bin_slots, std::vector<Phase> &phases)
{
    std::vector<int> level_of(P.n, 0);
    for (int l = 0; l < P.num_lev; ++l)
        for (int t = P.level_ptr[l]; t < P.level_ptr[l + 1]; ++t) level_of[P.level_idx[t]] = l;
    const std::vector<StepCost> cost = step_costs(P, T, limit);
    std::vector<uint32_t> comp;
    for (int l = 0; l < limit;) {
        const int e = phase_end(P, T, cost, l, limit, bin_slots, comp);
        if (e == l) break;
        Phase ph;
        ph.l0 = l;
        ph.l1 = e;
        if (!build_phase(P, T, level_of, comp, bin_slots, ph)) break;
        phases.push_back(std::move(ph));
        l = e;
    }
}

// Segments of the factorization schedule: windows (one workgroup each) and,
// between them, runs of global-memory steps split into fused and grid
// segments.
void factor_segments(glu_plan &p, const Tables &T, const std::vector<Phase> &phases, const std::vector<Window> &wins)
{
    p.fsegs.clear();
    int l = 0;
    for (size_t k = 0; k < phases.size(); ++k) {
        Segment s{phases[k].l0, phases[k].l1, false, 0};
        s.phase = (int)k;
        p.fsegs.push_back(s);
        l = phases[k].l1;
    }
    auto global_run = [&](int a, int b) {
        if (a >= b) return;
        std::vector<uint32_t> work(b - a);
        for (int q = a; q < b; ++q) work[q - a] = level_lanes(T, q);
        std::vector<Segment> segs;
        make_segments(work, (uint32_t)p.fuse_units, segs);
        for (Segment s : segs) {
            s.l0 += a;
            s.l1 += a;
            p.fsegs.push_back(s);
        }
    };
    for (size_t w = 0; w < wins.size(); ++w) {
        global_run(l, wins[w].l0);
        Segment s{wins[w].l0, wins[w].l1, true, 0};
        s.win = (int)w;
        p.fsegs.push_back(s);
        l = wins[w].l1;
    }
    global_run(l, p.num_lev + 1);
}

void tri_segments(glu_plan &p, TriHost &H)
{
    const int nlev = (int)H.lvl_ptr.size() - 1;
    std::vector<uint32_t> work(nlev);
    for (int l = 0; l < nlev; ++l) {
        const uint32_t rows = H.lvl_ptr[l + 1] - H.lvl_ptr[l];
        work[l] = (rows - H.lvl_long[l]) + H.lvl_long[l] * 64;   // lanes
    }
    make_segments(work, (uint32_t)p.fused_threads * 4, H.segs);
}

// Dataflow tasks of a sweep: in schedule order, each row with more than
// kDfLaneRow entries is a task of its own (a wave reads its entries at
// once), and consecutive shorter rows form tasks of up to 64 (one wave, a
// row per lane, every entry prefetched at the start), which may span
// levels.  No task crosses a segment boundary, so a fused segment runs
// tasks [k0, k1) by itself.
void tri_tasks(TriHost &H)
{
    H.tasks.clear();
    for (Segment &s : H.segs) {
        s.k0 = (uint32_t)H.tasks.size();
        uint32_t run = 0;   // rows in the open short task
        for (uint32_t q = H.lvl_ptr[s.l0]; q < H.lvl_ptr[s.l1]; ++q) {
            if (H.len[H.rows[q]] > kDfLaneRow) {
                H.tasks.push_back(q | kLongTask);
                run = 0;
                continue;
            }
            if (run == 0) H.tasks.push_back(q);
            run = run + 1 == 64 ? 0 : run + 1;   // a wave of rows
        }
        s.k1 = (uint32_t)H.tasks.size();
    }
    H.tasks.push_back(H.lvl_ptr.back());
}

// Task-contiguous layout of one sweep for the pipelined dataflow kernels
// (refinement sweeps of the batch).  entries(r, out) lists row r's
// {column, CSC position} pairs in the order the row consumes them; pivot
// (div sweeps) gives the CSC position of row r's divisor.
struct DfHost {
    std::vector<uint4> task;
    std::vector<uint2> rl;
    std::vector<uint32_t> idx, vpos;   // per slot
    std::vector<uint32_t> pvpos;       // per position: pivot CSC position (div)
};

// Lanes per row of a wave row: 16, 32 or 64 (longer rows take several
// passes of 64).
inline uint32_t df_group(uint32_t len) { return len <= 16 ? 16u : len <= 32 ? 32u : 64u; }

template <typename Entries, typename Pivot>
void build_df(const TriHost &H, Entries entries, bool div, Pivot pivot, bool long_lanes, DfHost &D)
{
    const uint32_t n = (uint32_t)H.rows.size();
    const int nlev = (int)H.lvl_ptr.size() - 1;
    std::vector<uint32_t> len(n);
    for (uint32_t r = 0; r < n; ++r) {
        std::vector<uint2> tmp;
        entries(r, tmp);
        len[r] = (uint32_t)tmp.size();
    }
    // Rows are taken a lane each (lane rows) or by groups of lanes (wave
    // rows).  Short rows (<= kDfK entries) are always lane rows.  With
    // long_lanes (orders whose sweep vector does not fit in LDS, where a
    // sweep is bound by the one workgroup's throughput), longer rows of up
    // to kDfLaneMax entries are lane rows too in a level with at least
    // kDfWideLevel of them: a lane walks its row kDfK entries at a time, 64
    // rows per task, where a wave would take 1 to 4 of them; in narrower
    // levels, which make up the sweep's critical path, they stay wave rows
    // (one memory round trip per row).  Measured: n=500k solve 55.7 ->
    // 34.6 ms, n=50k 2.57 -> 1.81 ms; the n=20k batch (vector in LDS) loses
    // 0.3 ms with them, so smaller orders keep wave rows.
    // Within each level (whose rows are independent) the short lane rows
    // are kept together, after the wave rows on even levels and before them
    // on odd ones, so that lane runs of adjacent levels meet and pack into
    // full tasks; long lane rows sit between the two, sorted by length so
    // that a task's rows have similar lengths (a task's slots are sized by
    // its longest row); wave rows are sorted by length so that rows sharing
    // a wave (16 or 32 lanes each) have the same lane count.
    std::vector<uint32_t> order(n);
    std::vector<uint8_t> lane_row(n);   // by position
    for (int l = 0; l < nlev; ++l) {
        std::vector<uint32_t> a, c, b;   // short lane rows, long lane rows, wave rows
        for (uint32_t q = H.lvl_ptr[l]; q < H.lvl_ptr[l + 1]; ++q) {
            const uint32_t r = H.rows[q];
            (len[r] <= kDfK ? a : len[r] <= kDfLaneMax ? c : b).push_back(r);
        }
        if (!long_lanes || c.size() < kDfWideLevel) {
            b.insert(b.end(), c.begin(), c.end());
            c.clear();
        }
        auto by_len = [&](uint32_t x, uint32_t y) { return len[x] < len[y]; };
        std::stable_sort(b.begin(), b.end(), by_len);
        std::stable_sort(c.begin(), c.end(), by_len);
        uint32_t q = H.lvl_ptr[l];
        auto put_rows = [&](auto first, auto last, uint8_t lane) {
            for (; first != last; ++first, ++q) {
                order[q] = *first;
                lane_row[q] = lane;
            }
        };
        if (l & 1) {
            put_rows(a.begin(), a.end(), 1);
            put_rows(c.begin(), c.end(), 1);
            put_rows(b.begin(), b.end(), 0);
        } else {
            put_rows(b.begin(), b.end(), 0);
            put_rows(c.rbegin(), c.rend(), 1);
            put_rows(a.begin(), a.end(), 1);
        }
    }
    std::vector<int> lev_of(n);
    for (int l = 0; l < nlev; ++l)
        for (uint32_t q = H.lvl_ptr[l]; q < H.lvl_ptr[l + 1]; ++q) lev_of[q] = l;
    std::vector<std::vector<uint2>> ent(n);
    D.rl.resize(n);
    for (uint32_t p = 0; p < n; ++p) {
        entries(order[p], ent[p]);
        D.rl[p] = make_uint2(order[p], (uint32_t)ent[p].size());
    }
    auto put = [&](const uint2 &e) {
        D.idx.push_back(e.x);
        D.vpos.push_back(e.y);
    };
    const uint2 pad = make_uint2(0u, UINT32_MAX);
    uint32_t p = 0;
    while (p < n) {
        const uint32_t base = (uint32_t)D.idx.size();
        const uint32_t p0 = p;
        if (!lane_row[p]) {
            // rows of one lane count and one level (no dependencies inside)
            const uint32_t gw = df_group((uint32_t)ent[p].size()), per = 64 / gw;
            uint32_t m = 0;
            while (p < n && p - p0 < per && lev_of[p] == lev_of[p0] && !lane_row[p] &&
                   df_group((uint32_t)ent[p].size()) == gw)
                m = std::max(m, (uint32_t)ent[p++].size());
            if (gw == 64) {   // padded to whole passes of 64 (every lane loads its slot)
                for (const uint2 &e : ent[p0]) put(e);
                while ((D.idx.size() - base) % 64) put(pad);
            } else {
                for (uint32_t g = 0; g < per; ++g)
                    for (uint32_t j = 0; j < gw; ++j)
                        put(p0 + g < p && j < ent[p0 + g].size() ? ent[p0 + g][j] : pad);
            }
            const uint32_t lg = gw == 16 ? 4u : gw == 32 ? 5u : 6u;
            D.task.push_back(make_uint4(base, p0, kLongTask | (lg << 24) | (p - p0), m));
            continue;
        }
        // lane rows, short and long ones in separate tasks
        const bool lng = ent[p].size() > kDfK;
        uint32_t m = 0;
        while (p < n && p - p0 < 64 && lane_row[p] && (ent[p].size() > kDfK) == lng)
            m = std::max(m, (uint32_t)ent[p++].size());
        for (uint32_t e = 0; e < m; ++e)
            for (uint32_t l = 0; l < 64; ++l) put(p0 + l < p && e < ent[p0 + l].size() ? ent[p0 + l][e] : pad);
        D.task.push_back(make_uint4(base, p0, p - p0, m));
    }
    // padding, so that the kernels' loads need no bounds tests: kDfK passes
    // of 64 slots after the last task, 64 positions after the last row
    for (uint32_t q = 0; q < kDfK * 64; ++q) put(pad);
    D.rl.resize(n + 64, make_uint2(0u, 0u));
    if (div) {
        D.pvpos.resize(n);
        for (uint32_t q = 0; q < n; ++q) D.pvpos[q] = pivot(order[q]);
    }
}

// Host check of a dataflow sweep table, before any launch.  Every load the
// sweep kernels issue stays inside the tables (a lane task's prefetch of
// kDfK slots per lane and its chunk refills, a wave task's slots, rows and
// pivots); every slot's value position is in the pattern or padding; every
// row runs exactly once; and every dependency of a row is finished by an
// earlier task or, in a lane task, by an earlier lane of the same task
// (the rows of a wave task never depend on each other).  Tasks are taken in
// order, so the lowest unfinished task always has its dependencies finished
// or inside itself: every ready-bit wait of the sweeps ends.
bool check_df(const DfHost &D, uint32_t n, uint32_t nnz, const char *name, std::string &err)
{
    const size_t nslots = D.idx.size();
    std::vector<uint8_t> done(n, 0);
    auto bad = [&](const std::string &what) {
        err = std::string(name) + " sweep table: " + what;
        return false;
    };
    if (D.rl.size() < (size_t)n + 64) return bad("row list not padded");
    for (size_t s = 0; s < nslots; ++s)
        if (D.vpos[s] != UINT32_MAX && D.vpos[s] >= nnz) return bad("value position out of range");
    for (size_t k = 0; k < D.task.size(); ++k) {
        const uint4 d = D.task[k];
        const uint32_t base = d.x, p0 = d.y, z = d.z, m = d.w;
        if ((size_t)p0 + 64 > D.rl.size()) return bad("task rows out of range");
        if (!(z & kLongTask)) {
            const uint32_t cnt = z;
            if (cnt > 64 || (size_t)base + (size_t)kDfK * 64 > nslots) return bad("lane task out of range");
            for (uint32_t lane = 0; lane < cnt; ++lane) {
                const uint32_t row = D.rl[p0 + lane].x, len = D.rl[p0 + lane].y;
                if (row >= n || len > m) return bad("lane row out of range");
                // a long lane row loads its entries kDfK at a time: up to the
                // end of its last chunk
                const size_t chunks = std::max<size_t>(1, (len + kDfK - 1) / kDfK);
                if (base + (chunks * kDfK - 1) * 64 + lane >= nslots) return bad("lane row slots out of range");
                for (uint32_t e = 0; e < len; ++e) {
                    const uint32_t dep = D.idx[base + (size_t)e * 64 + lane];
                    if (dep >= n || !done[dep]) return bad("row runs before its dependency");
                }
                if (done[row]) return bad("row runs twice");
                done[row] = 1;
            }
        } else {
            const uint32_t lg = (z >> 24) & 0x7fu, cnt = z & 0xffffffu, gw = 1u << lg;
            if (lg < 4 || lg > 6 || cnt == 0 || cnt * gw > 64) return bad("wave task shape");
            if ((size_t)base + 64 > nslots) return bad("wave task slots out of range");
            for (uint32_t g = 0; g < cnt; ++g) {
                const uint32_t row = D.rl[p0 + g].x, len = D.rl[p0 + g].y;
                if (row >= n || (gw < 64 && len > gw)) return bad("wave row out of range");
                if (gw == 64 && (cnt != 1 || (size_t)base + len > nslots)) return bad("wave row slots out of range");
                for (uint32_t j = 0; j < len; ++j) {
                    const uint32_t dep = D.idx[base + (size_t)gw * g + j];
                    if (dep >= n || !done[dep]) return bad("row runs before its dependency");
                }
            }
            for (uint32_t g = 0; g < cnt; ++g) {
                const uint32_t row = D.rl[p0 + g].x;
                if (done[row]) return bad("row runs twice");
                done[row] = 1;
            }
        }
    }
    for (uint32_t r = 0; r < n; ++r)
        if (!done[r]) return bad("a row never runs");
    return true;
}

// A sweep's streams (SwDev), from the dataflow table of the same sweep: its
// rows in schedule order, each row's entries, and whether the refinement sums
// the row's products (the rows that table gives a group of lanes).
struct SwHost {
    std::vector<uint4> meta;           // [lanes]
    std::vector<uint4> wave;           // by part and wave (SwDev)
    std::vector<uint32_t> hdr, first, lanes;   // chunks: header, first lane, lanes
    std::vector<uint32_t> row, rpos, vsrc;     // vsrc: CSC position of each value (~0: 0)
    std::vector<SwPart> part;
    std::vector<SwProd> prod;          // value index within this sweep
    uint32_t nwave = 0, per_lane = 4, nslot_max = 0;   // per_lane: values of a lane
};

// Rows of parts: part_of[r] (UINT32_MAX: not in this sweep), slot_of[r] and
// the part's row count.
struct SwParts {
    std::vector<uint32_t> part_of, slot_of, count;
};

constexpr uint32_t kSwEntries = 256;   // values of a chunk

// Lanes a row of len entries takes, four entries a lane (a summed row: at
// least the 16 entries whose sum is a fixed tree; 65 and more summed entries:
// chunks of its own).
inline uint32_t sw_lanes(uint32_t len, bool sum = false)
{
    uint32_t g = sum ? 4 : 1;
    while (4 * g < len) g *= 2;
    return g;
}

// Chunks go to the part's waves in turn, a level after the other; the rows of
// several chunks, which take their time but can start early, to waves of
// their own.  These run two such rows at a time, each chunk in a step where
// the wave has no other, and take their turn with the rest where no such row
// is under way (a wave with two chunks in a step is what every wave waits
// for.  Without: refinement of an 18^3 mesh, three solves, 2,643 us, 20^3
// 3,879, 10 dense blocks of 300 1,747 a solve; so 2,147, 3,282 and 1,596.
// Exact solve of the blocks 1,300 -> 945 us, n=50,000 374 -> 368).
void build_sw(const TriHost &H, const DfHost &D, uint32_t n, bool div, const SwParts &Q, uint32_t waves, SwHost &S)
{
    const uint32_t nparts = (uint32_t)Q.count.size();
    S.nwave = waves;
    S.per_lane = div ? 5 : 4;
    const uint32_t stride = kSwEntries + (div ? 64 : 0);   // of a chunk before its unused lanes go
    // by position: first entry's place in D, the step to the next, level, sum?
    struct Pos {
        uint32_t row, len, base, step, level, pivot;
        bool sum;
    };
    std::vector<std::vector<Pos>> rows(nparts);
    {
        std::vector<uint32_t> base(n), step(n);
        std::vector<uint8_t> sum(n);
        for (const uint4 &d : D.task) {
            const bool wave = (d.z & kLongTask) != 0;
            const uint32_t lg = (d.z >> 24) & 0x7fu, cnt = d.z & 0xffffffu;
            for (uint32_t k = 0; k < cnt; ++k) {
                base[d.y + k] = d.x + (wave ? k << lg : k);
                step[d.y + k] = wave ? 1 : 64;
                sum[d.y + k] = wave;
            }
        }
        uint32_t level = 0;
        for (uint32_t p = 0; p < n; ++p) {
            while (p >= H.lvl_ptr[level + 1]) ++level;
            const uint32_t r = D.rl[p].x;
            if (Q.part_of[r] != UINT32_MAX)
                rows[Q.part_of[r]].push_back(
                    Pos{r, D.rl[p].y, base[p], step[p], level, div ? D.pvpos[p] : 0u, sum[p] != 0});
        }
    }
    for (uint32_t part = 0; part < nparts; ++part) {
        std::vector<Pos> &R = rows[part];
        const uint32_t nslot = Q.count[part], zero = nslot, one = nslot + 1;
        S.nslot_max = std::max(S.nslot_max, nslot);
        SwPart P{(uint32_t)S.wave.size(), (uint32_t)S.row.size(), nslot, 0};
        S.row.resize(P.s0 + nslot);
        S.rpos.resize(P.s0 + nslot);
        auto is_long = [](const Pos &x) { return x.sum && x.len > 64; };
        // the part's chunks in schedule order
        std::vector<uint4> meta;
        std::vector<uint32_t> hdr, vsrc, wave, lanes, rpos(nslot);
        struct Prod {
            uint32_t chunk, at, vpos, col;
        };
        std::vector<Prod> prod;
        auto add = [&](uint32_t h) {
            hdr.push_back(h);
            meta.resize(meta.size() + 64, make_uint4(zero | zero << 16, zero | zero << 16, 0u, 0u));
            vsrc.resize(vsrc.size() + stride, UINT32_MAX);
            lanes.push_back(0);
        };
        auto put = [&](uint32_t lane, uint32_t e, const Pos &x, uint32_t k) {   // entry k of row x
            const size_t c = hdr.size() - 1, q = x.base + (size_t)k * x.step;
            const uint32_t col = D.idx[q], vp = D.vpos[q];
            uint32_t slot;
            if (Q.part_of[col] == part) {
                slot = Q.slot_of[col];
                vsrc[c * stride + 4 * lane + e] = vp;
            } else {
                slot = one;
                prod.push_back(Prod{(uint32_t)c, 4 * lane + e, vp, col});
            }
            uint4 &m = meta[64 * c + lane];
            uint32_t &w = e < 2 ? m.x : m.y;
            w = (e & 1) ? (w & 0xffffu) | slot << 16 : (w & 0xffff0000u) | slot;
        };
        std::vector<uint32_t> step_of(nslot, 0);   // a row's step
        auto ready = [&](const Pos &x, uint32_t k, uint32_t step, uint32_t before) {   // entry k of x: set that many steps before
            const uint32_t col = D.idx[x.base + (size_t)k * x.step];
            return Q.part_of[col] != part || step_of[Q.slot_of[col]] + before <= step;
        };
        // waves for the rows of several chunks, by their share of the work (a
        // chunk of 256 subtractions in order takes about 0.75 us, another
        // 0.2): at most three quarters
        size_t multi = 0;
        double rails = 0.0, rest = 1.0;
        for (const Pos &x : R) {
            const bool m = is_long(x) && x.len > kSwEntries;
            multi += m;
            (m ? rails : rest) += m ? 0.75 / kSwEntries * x.len : 0.2 / 64 * (is_long(x) ? 64 : sw_lanes(x.len, x.sum));
        }
        const uint32_t own = waves < 4 || !multi ? 0u
            : (uint32_t)std::min<size_t>(multi, std::max(1u, (uint32_t)std::min(0.75 * waves, waves * rails / (rails + rest) + 0.5)));
        uint32_t turn = 0, turn_long = 0;
        // the levels they are under way: from the first whose chunk can run, less the lead
        uint32_t own_from = UINT32_MAX, own_to = 0;
        if (own) {
            std::vector<uint32_t> level_of(nslot);
            for (const Pos &x : R) level_of[Q.slot_of[x.row]] = x.level;
            for (const Pos &x : R) {
                if (!is_long(x) || x.len <= kSwEntries) continue;
                uint32_t from = R[0].level;
                for (uint32_t k = 0; k < kSwEntries; ++k) {
                    const uint32_t col = D.idx[x.base + (size_t)k * x.step];
                    if (Q.part_of[col] == part) from = std::max(from, level_of[Q.slot_of[col]] + 1);
                }
                own_from = std::min(own_from, from);
                own_to = std::max(own_to, x.level);
            }
        }
        auto any_wave = [&](uint32_t level) {   // for a chunk of that level, in turn
            const uint32_t first = level + kSwLead < own_from || level > own_to ? 0u : own;
            return first + turn++ % (waves - first);
        };
        uint32_t used = 64;
        std::vector<uint32_t> track_step(2 * own, 0);   // the step a wave's open rows got to
        std::vector<std::vector<uint32_t>> taken(own);   // the steps of its newest 16 chunks
        for (size_t i = 0; i < R.size(); ++P.steps) {
            used = 64;
            size_t e = i;
            while (e < R.size() && R[e].level == R[i].level) ++e;
            // a level's rows are independent: long ones first, then by lanes,
            // down on even levels and up on odd ones (alignment costs least)
            const bool up = R[i].level & 1u;
            std::stable_sort(R.begin() + i, R.begin() + e, [&](const Pos &x, const Pos &y) {
                const bool lx = is_long(x), ly = is_long(y);
                if (lx != ly) return lx;
                if (lx) return false;
                const uint32_t a = 2 * sw_lanes(x.len, x.sum) + x.sum, b = 2 * sw_lanes(y.len, y.sum) + y.sum;
                return up ? a < b : a > b;
            });
            for (; i < e; ++i) {
                const Pos &x = R[i];
                const uint32_t slot = Q.slot_of[x.row];
                S.row[P.s0 + slot] = x.row;
                step_of[slot] = P.steps;
                if (is_long(x)) {
                    const uint32_t nc = (x.len + kSwEntries - 1) / kSwEntries;
                    // a row of several chunks: its chunks spread over the
                    // steps before its own, one of two rows a wave has open
                    const bool rail = nc > 1 && own;
                    const uint32_t track = rail ? turn_long++ % (2 * own) : 0u;
                    const uint32_t to = rail ? track % own : any_wave(x.level);
                    for (uint32_t c = 0; c < nc; ++c) {
                        const uint32_t left = std::min(x.len - c * kSwEntries, kSwEntries);
                        uint32_t at = P.steps;   // the row's step ends it
                        if (rail && c + 1 < nc) {
                            const uint32_t from = track_step[track], gap = (P.steps - from) / (nc - c);
                            at = std::min(from + std::min(std::max(gap, 1u), kSwLead), P.steps);
                            for (uint32_t k = 0; k < left; ++k) {
                                const uint32_t col = D.idx[x.base + (size_t)(c * kSwEntries + k) * x.step];
                                if (Q.part_of[col] == part) at = std::max(at, step_of[Q.slot_of[col]] + 1);
                            }
                            const std::vector<uint32_t> &T = taken[to];
                            uint32_t s = at;
                            while (s < P.steps && std::find(T.begin(), T.end(), s) != T.end()) ++s;
                            if (s < P.steps) at = s;
                        }
                        if (rail) {
                            track_step[track] = at;
                            if (taken[to].size() == 16) taken[to].erase(taken[to].begin());
                            taken[to].push_back(at);
                        }
                        uint32_t early = 0;   // leading entries set well before
                        while (early < left && ready(x, c * kSwEntries + early, at, kSwLead + 1)) ++early;
                        add(at | kSwLong | (c == 0 ? kSwFirst : 0u) | (c + 1 == nc ? kSwLast : 0u) |
                            (rail && track >= own ? kSwTrack : 0u) | early << kSwEarlyShift);
                        wave.push_back(to);
                        uint32_t bits[64] = {};
                        for (uint32_t k = 0; k < left; ++k) {
                            put(k % 64, k / 64, x, c * kSwEntries + k);
                            bits[k % 64] |= kSwEntry << (k / 64);
                        }
                        for (uint32_t lane = 0; lane < 64; ++lane) meta[64 * (hdr.size() - 1) + lane].z = slot | bits[lane] | left << kSwCountShift;
                        if (c == 0) rpos[slot] = 64 * (uint32_t)(hdr.size() - 1);
                        if (c + 1 == nc && div) vsrc[(hdr.size() - 1) * stride + kSwEntries] = x.pivot;
                        lanes.back() = std::min(left, 64u);
                    }
                    continue;
                }
                const uint32_t g = sw_lanes(x.len, x.sum);
                used = (used + g - 1) & ~(g - 1);
                if (used + g > 64) {
                    add(P.steps);
                    wave.push_back(any_wave(x.level));
                    used = 0;
                }
                const size_t c = hdr.size() - 1;
                hdr[c] |= x.sum ? kSwHasTree : kSwHasSeq;
                uint32_t early = 0;   // leading lanes whose entries are set two steps before
                while (early < g) {
                    bool all = true;
                    for (uint32_t k = 4 * early; k < std::min(4 * early + 4, x.len); ++k) all = all && ready(x, k, P.steps, 2);
                    if (!all) break;
                    ++early;
                }
                const uint32_t pre = early ? early - 1 : 0, rem = early ? g - early : g - 1;
                hdr[c] = (hdr[c] & ~(kSwPreMask << kSwPreShift | kSwRemMask << kSwRemShift)) |
                         std::max(pre, (hdr[c] >> kSwPreShift) & kSwPreMask) << kSwPreShift |
                         std::max(rem, (hdr[c] >> kSwRemShift) & kSwRemMask) << kSwRemShift;
                for (uint32_t lane = 0; lane < g; ++lane)
                    meta[64 * c + used + lane].z = slot | (uint32_t)__builtin_ctz(g) << 16 | (x.sum ? kSwTree : 0u) | kSwOn;
                for (uint32_t k = 0; k < x.len; ++k) put(used + k / 4, k % 4, x, k);
                rpos[slot] = 64 * (uint32_t)c + used;
                if (div)   // at the lane that stores the row: the last; a summed row's first too
                    for (uint32_t lane : {used + g - 1, x.sum ? used : used + g - 1})
                        vsrc[c * stride + kSwEntries + lane] = x.pivot;
                used += g;
                lanes.back() = used;
            }
        }
        // stream by stream
        std::vector<uint32_t> at(hdr.size());
        std::vector<std::vector<uint32_t>> stream(waves);
        for (size_t c = 0; c < hdr.size(); ++c) stream[wave[c]].push_back((uint32_t)c);
        for (uint32_t w = 0; w < waves; ++w) {
            std::stable_sort(stream[w].begin(), stream[w].end(),
                             [&](uint32_t a, uint32_t b) { return (hdr[a] & kSwStepMask) < (hdr[b] & kSwStepMask); });
            const size_t k0 = S.hdr.size();
            for (uint32_t c : stream[w]) {
                const uint32_t u = (std::max(lanes[c], 1u) + 3) & ~3u;
                at[c] = (uint32_t)S.hdr.size();
                S.hdr.push_back(hdr[c]);
                S.first.push_back((uint32_t)S.meta.size());
                S.lanes.push_back(u);
                const size_t m = 64 * (size_t)c, v = stride * (size_t)c;
                meta[m].w = hdr[c];
                S.meta.insert(S.meta.end(), meta.begin() + m, meta.begin() + m + u);
                S.vsrc.insert(S.vsrc.end(), vsrc.begin() + v, vsrc.begin() + v + 4 * u);
                if (div) S.vsrc.insert(S.vsrc.end(), vsrc.begin() + v + kSwEntries, vsrc.begin() + v + kSwEntries + u);
            }
            // a chunk names the one two after it (the last again)
            const size_t k1 = S.hdr.size();
            for (size_t k = k0; k < k1; ++k) {
                const size_t q = std::min(k + 2, k1 - 1);
                S.meta[S.first[k] + 1].w = S.first[q];
                S.meta[S.first[k] + 2].w = S.lanes[q];
            }
            const size_t q = std::min(k0 + 1, k1 - 1);
            S.wave.push_back(k0 == k1 ? make_uint4(0u, 0u, 0u, 0u)
                                      : make_uint4((uint32_t)(k1 - k0), S.first[k0], S.first[q], S.lanes[k0] | S.lanes[q] << 8));
        }
        for (uint32_t k = 0; k < nslot; ++k) S.rpos[P.s0 + k] = S.first[at[rpos[k] / 64]] + rpos[k] % 64;
        for (const Prod &q : prod) S.prod.push_back(SwProd{S.first[at[q.chunk]] * S.per_lane + q.at, q.vpos, q.col});
        S.part.push_back(P);
    }
}

// Host check of a sweep's streams before any launch: every slot and value
// position in range, every row of a part stored once, with its right-hand
// side at its first lane, a stream's steps in order, every entry's row in an
// earlier step than the entry (and two before where the chunk's header takes
// it ahead), the chunks of a long row together.
bool check_sw(const SwHost &S, uint32_t nnz, const char *name, std::string &err)
{
    auto bad = [&](const std::string &what) {
        err = std::string(name) + " sweep streams: " + what;
        return false;
    };
    const uint32_t nchunk = (uint32_t)S.hdr.size();
    if (S.first.size() != nchunk || S.lanes.size() != nchunk || S.vsrc.size() != S.per_lane * S.meta.size() ||
        S.wave.size() != S.part.size() * S.nwave || S.vsrc.size() > 0xffffffffull)
        return bad("sizes");
    for (uint32_t c = 0; c < nchunk; ++c)
        if (S.lanes[c] < 4 || S.lanes[c] > 64 || S.lanes[c] % 4 || S.first[c] % 4 ||
            (size_t)S.first[c] + S.lanes[c] > S.meta.size())
            return bad("chunk out of range");
    uint32_t k0 = 0, k1 = 0;   // a stream's chunks: the streams follow each other
    for (uint32_t v : S.vsrc)
        if (v != UINT32_MAX && v >= nnz) return bad("value position out of range");
    for (const SwProd &q : S.prod)
        if (q.val >= S.vsrc.size() || q.vpos >= nnz) return bad("product out of range");
    for (const SwPart &P : S.part) {
        if ((size_t)P.wp + S.nwave > S.wave.size() || (size_t)P.s0 + P.nslot > S.row.size() || P.nslot > 0xfffdu ||
            P.steps > kSwStepMask + 1)
            return bad("part out of range");
        std::vector<uint32_t> set(P.nslot + 2, 0);   // 1 + the row's step
        const uint32_t part_k0 = k1;
        for (uint32_t pass = 0; pass < 2; ++pass)
            for (uint32_t w = 0; w < S.nwave; ++w) {
                const uint4 d = S.wave[P.wp + w];
                k0 = w == 0 ? part_k0 : k1;
                if (d.x > nchunk - k0) return bad("stream out of range");
                k1 = k0 + d.x;
                for (uint32_t c = k0; c < k1; ++c) {
                    const uint32_t q = std::min(c + 2, k1 - 1), second = std::min(k0 + 1, k1 - 1), l = S.first[c];
                    if (S.meta[l].w != S.hdr[c] || S.meta[l + 1].w != S.first[q] || S.meta[l + 2].w != S.lanes[q] ||
                        d.y != S.first[k0] || d.z != S.first[second] || d.w != (S.lanes[k0] | S.lanes[second] << 8))
                        return bad("a chunk is misplaced");
                }
                uint32_t last = 0;
                bool open[2] = {false, false};   // in a long row
                uint32_t row_open[2] = {0, 0};
                for (uint32_t c = k0; c < k1; ++c) {
                    const uint32_t h = S.hdr[c], step = h & kSwStepMask;
                    if (step < last || step >= P.steps) return bad("step out of range");
                    last = step;
                    auto entry = [&](uint32_t lane, uint32_t e) {
                        const uint4 &m = S.meta[S.first[c] + lane];
                        const uint32_t v = e < 2 ? m.x : m.y;
                        return (e & 1) ? v >> 16 : v & 0xffffu;
                    };
                    for (uint32_t lane = 0; lane < S.lanes[c]; ++lane)
                        for (uint32_t e = 0; e < 4; ++e) {
                            if (entry(lane, e) > P.nslot + 1) return bad("slot out of range");
                            if (pass && set[entry(lane, e)] > step) return bad("an entry's row is not in an earlier step");
                        }
                    auto early = [&](uint32_t lane, uint32_t e) { return set[entry(lane, e)] < step || !set[entry(lane, e)]; };
                    auto store = [&](uint32_t slot) {
                        if (pass) return true;
                        const bool once = !set[slot];
                        set[slot] = step + 1;
                        return once;
                    };
                    if (h & kSwLong) {
                        const uint32_t z = S.meta[S.first[c]].z, slot = z & 0xffffu;
                        const uint32_t n_early = (h >> kSwEarlyShift) & kSwEarlyMask, count = z >> kSwCountShift;
                        const uint32_t tr = (h & kSwTrack) ? 1 : 0;
                        if (open[tr] ? (h & kSwFirst) || slot != row_open[tr] : !(h & kSwFirst)) return bad("a row's chunks are apart");
                        open[tr] = !(h & kSwLast);
                        row_open[tr] = slot;
                        if (slot >= P.nslot || count > kSwEntries || n_early > count || S.lanes[c] < std::min(count, 64u)) return bad("long row out of range");
                        for (uint32_t e = 0; e < n_early && pass; ++e)
                            if (set[entry(e % 64, e / 64)] && set[entry(e % 64, e / 64)] + kSwLead > step) return bad("an entry is taken before it is set");
                        if ((h & kSwFirst) && S.rpos[P.s0 + slot] != S.first[c]) return bad("right-hand side misplaced");
                        if ((h & kSwLast) && !store(slot)) return bad("a row runs twice");
                        continue;
                    }
                    const uint32_t pre = (h >> kSwPreShift) & kSwPreMask, rem = (h >> kSwRemShift) & kSwRemMask;
                    for (uint32_t lane = 0; lane < S.lanes[c];) {
                        const uint32_t z = S.meta[S.first[c] + lane].z, slot = z & 0xffffu, g = 1u << ((z >> 16) & 7u);
                        if (lane % g || lane + g > S.lanes[c] || g > 16) return bad("row lanes out of place");
                        if (z & kSwOn) {
                            if (slot >= P.nslot) return bad("row slot out of range");
                            if (S.rpos[P.s0 + slot] != S.first[c] + lane) return bad("right-hand side misplaced");
                            if (!store(slot)) return bad("a row runs twice");
                            uint32_t n_early = 0;   // lanes done a step ahead
                            while (n_early < std::min(g, pre + 1) && early(lane + n_early, 0) && early(lane + n_early, 1) &&
                                   early(lane + n_early, 2) && early(lane + n_early, 3))
                                ++n_early;
                            if (pass && (g - std::max(n_early, 1u) > rem || g - 1 > pre + rem)) return bad("a row is cut short");
                        }
                        lane += g;
                    }
                }
                if (open[0] || open[1]) return bad("a row does not end");
            }
        for (uint32_t k = 0; k < P.nslot; ++k)
            if (!set[k]) return bad("a row never runs");
    }
    return true;
}

// The split of an order whose vector does not fit in LDS.  A row's height is
// the longest chain of rows (entries of L or of U, either way) below it; the
// rows of height h and more are closed under the dependencies of the U
// sweeps, the others under those of the L sweeps, and fall into components
// that share no entry.  Of the heights tried, the one with the least
// estimated time: the tail's chunks on one workgroup and its chain, and the
// largest head part's.  Components go to parts largest first, each to the
// part with the least so far.
struct SwSplit {
    SwParts head, tail;
};

constexpr uint32_t kHeadWaves = 8;
constexpr uint32_t kHeadParts = 512;    // two workgroups a CU
constexpr uint32_t kHeadSlots = 16384;  // at most (64 KB of LDS)

// cap_slots: rows a workgroup's LDS holds.
bool choose_split(const glu_pattern &P, uint32_t cap_slots, uint32_t tail_waves, SwSplit &S)
{
    const uint32_t head_slots = std::min(cap_slots, kHeadSlots);
    const uint32_t n = P.n;
    std::vector<uint32_t> ht(n, 0), wgt(n);
    uint32_t top = 0;
    for (uint32_t r = 0; r < n; ++r) {
        uint32_t h = 0;
        for (uint32_t q = P.csr_r_ptr[r]; q < P.csr_diag_ptr[r]; ++q) h = std::max(h, ht[P.csr_c_idx[q]] + 1);
        for (uint32_t q = P.sym_c_ptr[r]; q < P.l_col_ptr[r]; ++q) h = std::max(h, ht[P.sym_r_idx[q]] + 1);
        ht[r] = h;
        top = std::max(top, h);
        // lanes of both sweeps
        const uint32_t l = P.csr_diag_ptr[r] - P.csr_r_ptr[r], u = P.csr_r_ptr[r + 1] - P.csr_diag_ptr[r] - 1;
        wgt[r] = (l > 64 ? l / 4 + 64 : sw_lanes(l)) + (u > 64 ? u / 4 + 64 : sw_lanes(u));
    }
    // components grow with h: one union-find over increasing heights
    std::vector<uint32_t> parent(n), rows_at(top + 2, 0), by_h(n);
    for (uint32_t r = 0; r < n; ++r) parent[r] = r, ++rows_at[ht[r] + 1];
    for (uint32_t h = 0; h <= top; ++h) rows_at[h + 1] += rows_at[h];
    {
        std::vector<uint32_t> cur(rows_at.begin(), rows_at.end() - 1);
        for (uint32_t r = 0; r < n; ++r) by_h[cur[ht[r]]++] = r;
    }
    std::vector<uint64_t> cw(wgt.begin(), wgt.end());
    std::vector<uint32_t> cn(n, 1);
    auto find = [&](uint32_t r) {
        while (parent[r] != r) r = parent[r] = parent[parent[r]];
        return r;
    };
    auto join = [&](uint32_t a, uint32_t b) {
        a = find(a), b = find(b);
        if (a == b) return a;
        if (cn[a] < cn[b]) std::swap(a, b);
        parent[b] = a;
        cw[a] += cw[b];
        cn[a] += cn[b];
        return a;
    };
    uint64_t total = 0, head_w = 0, max_w = 0;
    uint32_t max_n = 0, best_h = 0;
    for (uint32_t r = 0; r < n; ++r) total += wgt[r];
    double best = 0.0;
    std::vector<uint32_t> best_parent;
    constexpr double kChunk = 0.25, kHop = 0.2;   // us: a chunk of one wave, a hop of the chain
    uint32_t next_try = 4;
    for (uint32_t h = 1; h <= std::min(top, 512u); ++h) {   // rows of height < h in the head
        for (uint32_t k = rows_at[h - 1]; k < rows_at[h]; ++k) {
            const uint32_t r = by_h[k];
            head_w += wgt[r];
            uint32_t c = find(r);
            for (uint32_t q = P.csr_r_ptr[r]; q < P.csr_diag_ptr[r]; ++q) c = join(c, P.csr_c_idx[q]);
            for (uint32_t q = P.sym_c_ptr[r]; q < P.l_col_ptr[r]; ++q) c = join(c, P.sym_r_idx[q]);
            max_w = std::max(max_w, cw[c]);
            max_n = std::max(max_n, cn[c]);
        }
        if (h < next_try) continue;
        next_try = h + std::max(1u, h / 4);
        if (max_n > head_slots) break;
        const uint32_t tail = n - rows_at[h];
        if (tail > cap_slots) continue;
        const double head_chunks = std::max((double)max_w, (double)head_w / kHeadParts) / 64.0;
        const double t = (double)(total - head_w) / 64.0 / tail_waves * kChunk + 2.0 * (top + 1 - h) * kHop +
                         head_chunks / kHeadWaves * kChunk + 2.0 * h * kHop;
        if (best_h == 0 || t < best) {
            best = t;
            best_h = h;
            best_parent = parent;
        }
    }
    if (best_h == 0) return false;
    parent.swap(best_parent);
    S.head.part_of.assign(n, UINT32_MAX);
    S.head.slot_of.assign(n, 0);
    S.tail.part_of.assign(n, UINT32_MAX);
    S.tail.slot_of.assign(n, 0);
    S.tail.count.assign(1, 0);
    std::vector<uint32_t> comp(n, UINT32_MAX);
    std::vector<uint64_t> weight;
    std::vector<uint32_t> size;
    for (uint32_t r = 0; r < n; ++r) {
        if (ht[r] >= best_h) {
            S.tail.part_of[r] = 0;
            S.tail.slot_of[r] = S.tail.count[0]++;
            continue;
        }
        const uint32_t c = find(r);
        if (comp[c] == UINT32_MAX) {
            comp[c] = (uint32_t)weight.size();
            weight.push_back(0);
            size.push_back(0);
        }
        weight[comp[c]] += wgt[r];
        ++size[comp[c]];
    }
    std::vector<uint32_t> order(weight.size()), part(weight.size());
    for (uint32_t c = 0; c < order.size(); ++c) order[c] = c;
    std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return weight[a] > weight[b]; });
    const uint32_t nparts = (uint32_t)std::min<size_t>({weight.size(), kHeadParts, (size_t)(total / 1024 + 1)});
    std::vector<uint64_t> load(nparts, 0);
    std::vector<uint32_t> rows(nparts, 0);
    for (uint32_t c : order) {
        uint32_t to = UINT32_MAX;
        for (uint32_t k = 0; k < nparts; ++k)
            if (rows[k] + size[c] <= head_slots && (to == UINT32_MAX || load[k] < load[to])) to = k;
        if (to == UINT32_MAX) return false;
        load[to] += weight[c];
        rows[to] += size[c];
        part[c] = to;
    }
    S.head.count.assign(nparts, 0);
    for (uint32_t r = 0; r < n; ++r)
        if (ht[r] < best_h) {
            const uint32_t k = part[comp[find(r)]];
            S.head.part_of[r] = k;
            S.head.slot_of[r] = S.head.count[k]++;
        }
    return true;
}

struct Uploader {
    Arena arena;
    struct Item {
        size_t off;
        const void *src;
        size_t bytes;
    };
    std::vector<Item> items;
    template <typename T>
    size_t put(const T *src, size_t count)
    {
        size_t off = arena.add(count * sizeof(T));
        items.push_back(Item{off, src, count * sizeof(T)});
        return off;
    }
    template <typename T>
    size_t put(const std::vector<T> &v)
    {
        return put(v.data(), v.size());
    }
    size_t reserve(size_t bytes) { return arena.add(bytes); }
};

glu_status build_plan(const glu_pattern &P, const glu_analysis *a, const glu_plan_opts *opts, glu_plan **out)
{
    *out = nullptr;
    std::string err;
    if (P.n == 0 || P.nnz == 0) return fail(GLU_ERR_EMPTY, "matrix is empty");
    if (!validate_pattern(P, err)) return fail(GLU_ERR_INVALID, err);

    std::unique_ptr<glu_plan> p(new (std::nothrow) glu_plan());
    if (!p) return fail(GLU_ERR_MEMORY, "out of host memory");
    if (opts) {
        if (opts->block_threads) {
            if (opts->block_threads < 64 || opts->block_threads > 1024 || opts->block_threads % 64)
                return fail(GLU_ERR_ARGUMENT, "block_threads must be a multiple of 64 in [64, 1024]");
            p->fused_threads = opts->block_threads;
        }
        if (opts->fuse_units < 0) return fail(GLU_ERR_ARGUMENT, "fuse_units must be >= 0");
        if (opts->fuse_units) p->fuse_units = opts->fuse_units;
        p->use_graph = opts->use_graph != 0;
        if (opts->lds_windows < -1) return fail(GLU_ERR_ARGUMENT, "lds_windows must be >= -1");
        if (opts->lds_windows) p->max_windows = opts->lds_windows < 0 ? 0 : opts->lds_windows;
        if (opts->solve_dataflow < -1 || opts->solve_dataflow > 1)
            return fail(GLU_ERR_ARGUMENT, "solve_dataflow must be -1, 0 or 1");
        p->solve_df_opt = opts->solve_dataflow;
        if (opts->krylov < -1 || opts->krylov > kMaxKrylov)
            return fail(GLU_ERR_ARGUMENT, "krylov must be in [-1, 4]");
        if (opts->krylov) p->krylov = opts->krylov < 0 ? 0 : opts->krylov;
        if (opts->lds_window_values < 0) return fail(GLU_ERR_ARGUMENT, "lds_window_values must be >= 0");
        p->win_values = (uint32_t)opts->lds_window_values;
        if (opts->batch_grid_levels < -1) return fail(GLU_ERR_ARGUMENT, "batch_grid_levels must be >= -1");
        p->batch_grid_opt = opts->batch_grid_levels;
    }
    p->n = P.n;
    p->nnz = P.nnz;
    p->num_lev = P.num_lev;

    Tables T;
    try {
        if (!build_factor_tables(P, T, p->updates, err)) return fail(GLU_ERR_INVALID, err);
    } catch (const std::bad_alloc &) {
        return fail(GLU_ERR_MEMORY, "out of host memory building tables");
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(GLU_ERR_DEVICE, "no HIP device");
    HIP_TRY(hipGetDevice(&p->device));
    p->lds_cap = launch::enable_lds();
    std::vector<Window> wins;
    // (slots are 16-bit numbers)
    uint32_t budget = std::min<uint32_t>((uint32_t)(p->lds_cap / sizeof(float)), 0xffffu);
    budget -= std::min(budget, kWinExtra);
    const uint32_t bin_slots = std::min(budget, kPhaseSlots);
    if (p->win_values) budget = std::min(budget, p->win_values);
    // Built side by side on host threads: the windows, the four triangular
    // sweeps (L, U; U', L' for A' x = b: rows of U' are columns of U with the
    // pivot last, forward; rows of L' columns of L, backward: schedules,
    // dataflow tables and, when the sweep vector fits in LDS, their streams),
    // and, when it does not (then long lane rows in wide levels), the split.
    const uint32_t n = P.n;
    const bool long_lanes = launch::batch_lds_bytes(2, n) > p->lds_cap;
    const uint32_t wg_waves = (uint32_t)p->fused_threads / 64;
    DfHost dlo, dup, dtu, dtl;
    DfHost *const dfs[4] = {&dlo, &dup, &dtu, &dtl};
    const bool divs[4] = {false, true, true, false};
    const char *const names[4] = {"L", "U", "U'", "L'"};
    std::string errs[4];
    bool good[4] = {false, false, false, false}, split = false;
    SwSplit spl;
    SwHost sw[4], hd[4];   // streams of the whole order, or of the tail; of the head parts
    if (!long_lanes) {
        spl.tail.part_of.assign(n, 0);
        spl.tail.count.assign(1, n);
        spl.tail.slot_of.resize(n);
        for (uint32_t r = 0; r < n; ++r) spl.tail.slot_of[r] = r;
    }
    const auto sweep_tables = [&](int q) {
        TriHost &H = p->tri[q];
        const auto finish = [&](auto entries, auto pivot) {
            tri_segments(*p, H);
            tri_tasks(H);
            build_df(H, entries, divs[q], pivot, long_lanes, *dfs[q]);
            if (long_lanes) {
                good[q] = check_df(*dfs[q], n, P.nnz, names[q], errs[q]);
            } else {
                build_sw(H, *dfs[q], n, divs[q], spl.tail, wg_waves, sw[q]);
                good[q] = check_sw(sw[q], P.nnz, names[q], errs[q]);
            }
        };
        const auto no_pivot = [](uint32_t) { return 0u; };
        const auto diag = [&](uint32_t r) { return P.l_col_ptr[r]; };
        switch (q) {
        case 0:
            tri_levels(n, +1, [&](uint32_t r, auto f) {
                for (uint32_t k = P.csr_r_ptr[r]; k < P.csr_diag_ptr[r]; ++k) f(P.csr_c_idx[k]);
            }, [&](uint32_t r) { return P.csr_diag_ptr[r] - P.csr_r_ptr[r]; }, H);
            finish([&](uint32_t r, std::vector<uint2> &out) {
                for (uint32_t k = P.csr_r_ptr[r]; k < P.csr_diag_ptr[r]; ++k)
                    out.push_back(make_uint2(P.csr_c_idx[k], T.upos[k]));
            }, no_pivot);
            break;
        case 1:
            tri_levels(n, -1, [&](uint32_t r, auto f) {
                for (uint32_t k = P.csr_diag_ptr[r] + 1; k < P.csr_r_ptr[r + 1]; ++k) f(P.csr_c_idx[k]);
            }, [&](uint32_t r) { return P.csr_r_ptr[r + 1] - P.csr_diag_ptr[r] - 1; }, H);
            finish([&](uint32_t r, std::vector<uint2> &out) {
                for (uint32_t k = P.csr_r_ptr[r + 1]; k > P.csr_diag_ptr[r] + 1; --k)
                    out.push_back(make_uint2(P.csr_c_idx[k - 1], T.upos[k - 1]));
            }, diag);
            break;
        case 2:
            tri_levels(n, +1, [&](uint32_t r, auto f) {
                for (uint32_t k = P.sym_c_ptr[r]; k < P.l_col_ptr[r]; ++k) f(P.sym_r_idx[k]);
            }, [&](uint32_t r) { return P.l_col_ptr[r] - P.sym_c_ptr[r]; }, H);
            finish([&](uint32_t r, std::vector<uint2> &out) {
                for (uint32_t k = P.sym_c_ptr[r]; k < P.l_col_ptr[r]; ++k) out.push_back(make_uint2(P.sym_r_idx[k], k));
            }, diag);
            break;
        default:
            tri_levels(n, -1, [&](uint32_t r, auto f) {
                for (uint32_t k = P.l_col_ptr[r] + 1; k < P.sym_c_ptr[r + 1]; ++k) f(P.sym_r_idx[k]);
            }, [&](uint32_t r) { return P.sym_c_ptr[r + 1] - P.l_col_ptr[r] - 1; }, H);
            finish([&](uint32_t r, std::vector<uint2> &out) {
                for (uint32_t k = P.sym_c_ptr[r + 1]; k > P.l_col_ptr[r] + 1; --k)
                    out.push_back(make_uint2(P.sym_r_idx[k - 1], k - 1));
            }, no_pivot);
        }
    };
    // (the phases, the longest, beside all that comes before they are needed)
    std::vector<Phase> phases;
    const auto windows_and_phases = [&]() {
        choose_windows(T, P.num_lev, P.nnz, budget, (uint32_t)p->fuse_units, p->max_windows, wg_waves, wins);
        choose_phases(P, T, wins.empty() ? 0 : std::min(wins[0].l0, P.num_lev), bin_slots, phases);
    };
    std::future<void> factor_steps;   // (waits in its destructor, before what it works on goes)
    try {
        factor_steps = std::async(std::launch::async, windows_and_phases);
    } catch (const std::system_error &) {   // no thread to be had
        windows_and_phases();
    }
    parallel_items(long_lanes ? 5 : 4, table_threads(), [&](unsigned, size_t item) {
        if (item < 4)
            sweep_tables((int)item);
        else
            split = choose_split(P, (uint32_t)std::min<size_t>(std::max<size_t>(p->lds_cap / sizeof(float), 2), 0xffffu) - 2,
                                 wg_waves, spl);
    });
    for (int q = 0; q < 4; ++q)
        if (!good[q]) return fail(GLU_ERR_INVALID, errs[q]);
    if (split) {
        std::string werr[8];
        bool wgood[8] = {};
        parallel_items(8, table_threads(), [&](unsigned, size_t item) {
            const size_t q = item % 4;
            SwHost &h = item < 4 ? hd[q] : sw[q];
            build_sw(p->tri[q], *dfs[q], n, divs[q], item < 4 ? spl.head : spl.tail, item < 4 ? kHeadWaves : wg_waves, h);
            wgood[item] = check_sw(h, P.nnz, names[q], werr[item]);
        });
        for (int i = 0; i < 8; ++i)
            if (!wgood[i]) return fail(GLU_ERR_INVALID, werr[i]);
    }
    p->scratch_nval[0] = dlo.idx.size() + dup.idx.size() + n + 64;
    p->scratch_nval[1] = dtu.idx.size() + dtl.idx.size() + n + 64;
    for (int q = 0; q < 4; ++q)
        for (const SwHost *h : {&sw[q], &hd[q]}) p->rhs_len[q / 2] = std::max(p->rhs_len[q / 2], (uint32_t)h->meta.size());
    p->t32_len = long_lanes ? n : std::max({n, p->rhs_len[0], p->rhs_len[1]});
    // the value copies (CSC position of each value, ~0 for places without
    // one, which get 0) of A x = b and A' x = b; with the vector beyond LDS,
    // those of the dataflow tables (slots, then the pivots), and the split
    // sweeps' own beside them
    std::vector<uint32_t> df_vpos, tdf_vpos, spl_vpos[2];
    uint32_t sw_voff[4] = {0, 0, 0, 0}, hd_voff[4] = {0, 0, 0, 0}, tlo_voff = 0;
    auto append = [](std::vector<uint32_t> &to, const SwHost &h) {
        const uint32_t at = (uint32_t)to.size();
        to.insert(to.end(), h.vsrc.begin(), h.vsrc.end());
        return at;
    };
    if (!long_lanes) {
        for (int q = 0; q < 4; ++q) sw_voff[q] = append(q < 2 ? df_vpos : tdf_vpos, sw[q]);
    } else {
        df_vpos = dlo.vpos;
        df_vpos.insert(df_vpos.end(), dup.vpos.begin(), dup.vpos.end());
        df_vpos.insert(df_vpos.end(), dup.pvpos.begin(), dup.pvpos.end());
        df_vpos.resize(df_vpos.size() + 64, UINT32_MAX);   // pivot reads of the last positions' lanes
        tdf_vpos = dtu.vpos;   // U' slots, U' pivots (+64 pad), L' slots
        tdf_vpos.insert(tdf_vpos.end(), dtu.pvpos.begin(), dtu.pvpos.end());
        tdf_vpos.resize(tdf_vpos.size() + 64, UINT32_MAX);
        tlo_voff = (uint32_t)tdf_vpos.size();
        tdf_vpos.insert(tdf_vpos.end(), dtl.vpos.begin(), dtl.vpos.end());
        if (split)
            for (int q = 0; q < 4; ++q) {
                hd_voff[q] = append(spl_vpos[q / 2], hd[q]);
                sw_voff[q] = append(spl_vpos[q / 2], sw[q]);
            }
    }
    p->df_nval = (uint32_t)df_vpos.size();
    p->tdf_nval = (uint32_t)tdf_vpos.size();
    // The batch kernels build the copy in LDS, copy_range slots at a time:
    // per range, {CSC position, slot - range start} of its non-padding
    // slots in increasing position order (so that the reads sweep the
    // factors in order), then the range is written out whole.
    p->copy_range = std::min<uint32_t>({p->df_nval, kCopyRange, (uint32_t)(p->lds_cap / sizeof(float)) & ~63u});
    if (p->copy_range == 0) return fail(GLU_ERR_DEVICE, "no LDS for the batch value copy");
    std::vector<uint2> df_cpy;
    std::vector<uint32_t> df_cpy_ptr(1, 0);
    {
        std::vector<std::vector<uint2>> range((p->df_nval + p->copy_range - 1) / p->copy_range);
        parallel_items(range.size(), table_threads(), [&](unsigned, size_t i) {
            const uint32_t b = (uint32_t)i * p->copy_range, e = std::min<uint32_t>(p->df_nval, b + p->copy_range);
            for (uint32_t q = b; q < e; ++q)
                if (df_vpos[q] != UINT32_MAX) range[i].push_back(make_uint2(df_vpos[q], q - b));
            std::sort(range[i].begin(), range[i].end(),
                      [](const uint2 &x, const uint2 &y) { return x.x < y.x || (x.x == y.x && x.y < y.y); });
        });
        df_cpy.reserve(p->df_nval);
        for (const auto &r : range) {
            df_cpy.insert(df_cpy.end(), r.begin(), r.end());
            df_cpy_ptr.push_back((uint32_t)df_cpy.size());
        }
    }

    // Refinement / refresh tables from the analysis.
    std::vector<uint32_t> a_rptr, a_cidx, a_src, lu_src, lu_col, a_rows, a_cols;
    std::vector<double> rs_col, a_rs, a_cs;
    std::vector<uint32_t> a_dst, lu_fill, df_rsrc, tdf_rsrc;
    std::vector<double> df_rscale, tdf_rscale;
    std::vector<uint2> sp_chunk[2], sp_rl[2], sp_ent[2];
    const Analysis *an = a ? &a->an : nullptr;
    if (an) {
        const uint32_t nnz_a = an->nnz;
        p->nnz_a = nnz_a;
        // CSR of the caller's A (rows = caller rows), remembering each
        // entry's position in the caller's CSC value array.
        a_rptr.assign(n + 1, 0);
        for (uint32_t k = 0; k < nnz_a; ++k) ++a_rptr[an->in_ai[k] + 1];
        for (uint32_t i = 0; i < n; ++i) a_rptr[i + 1] += a_rptr[i];
        a_cidx.resize(nnz_a);
        a_src.resize(nnz_a);
        std::vector<uint32_t> cur(a_rptr.begin(), a_rptr.end() - 1);
        for (uint32_t c = 0; c < n; ++c)
            for (uint32_t k = an->in_ap[c]; k < an->in_ap[c + 1]; ++k) {
                const uint32_t q = cur[an->in_ai[k]]++;
                a_cidx[q] = c;
                a_src[q] = k;
            }
        lu_src.resize(P.nnz);
        for (uint32_t q = 0; q < P.nnz; ++q) {
            const uint32_t d = a->lu_from_dump[q];
            lu_src[q] = (d == UINT32_MAX) ? UINT32_MAX : an->src_pos[d];
        }
        rs_col.resize(n);
        for (uint32_t c = 0; c < n; ++c) rs_col[c] = an->row_scale[an->row_perm[c]];
        lu_col.resize(P.nnz);
        for (uint32_t c = 0; c < n; ++c)
            for (uint32_t q = P.sym_c_ptr[c]; q < P.sym_c_ptr[c + 1]; ++q) lu_col[q] = c;
        // the inverse map: every caller value lands on exactly one LU position
        a_dst.assign(nnz_a, UINT32_MAX);
        a_rs.assign(nnz_a, 0.0);
        a_cs.assign(nnz_a, 0.0);
        for (uint32_t q = 0; q < P.nnz; ++q) {
            const uint32_t k = lu_src[q];
            if (k == UINT32_MAX) continue;
            if (k >= nnz_a || a_dst[k] != UINT32_MAX) return fail(GLU_ERR_INVALID, "value map is not one-to-one");
            a_dst[k] = q;
            a_rs[k] = rs_col[lu_col[q]];
            a_cs[k] = an->col_scale_perm[P.sym_r_idx[q]];
        }
        for (uint32_t k = 0; k < nnz_a; ++k)
            if (a_dst[k] == UINT32_MAX) return fail(GLU_ERR_INVALID, "a value of A has no LU position");
        for (uint32_t q = 0; q < P.nnz; ++q)
            if (lu_src[q] == UINT32_MAX) lu_fill.push_back(q);
        // rows / columns of A with more than kLongRow entries first
        auto long_first = [&](const uint32_t *ptr, std::vector<uint32_t> &order, uint32_t &nlong) {
            order.clear();
            for (uint32_t i = 0; i < n; ++i)
                if (ptr[i + 1] - ptr[i] > kLongRow) order.push_back(i);
            nlong = (uint32_t)order.size();
            for (uint32_t i = 0; i < n; ++i)
                if (ptr[i + 1] - ptr[i] <= kLongRow) order.push_back(i);
        };
        long_first(a_rptr.data(), a_rows, p->a_nlong);
        long_first(an->in_ap.data(), a_cols, p->a_nlong_t);
        for (uint32_t i = 0; i < n; ++i)
            p->a_kmax = std::max({p->a_kmax, a_rptr[i + 1] - a_rptr[i], an->in_ap[i + 1] - an->in_ap[i]});
        // short rows of A and A' for the products in one workgroup
        for (int t = 0; t < 2; ++t) {
            const uint32_t *ptr = t ? an->in_ap.data() : a_rptr.data();
            std::vector<uint32_t> rows;
            for (uint32_t i = 0; i < n; ++i)
                if (ptr[i + 1] - ptr[i] <= kLongRow) rows.push_back(i);
            for (size_t i = 0; i < rows.size(); i += 64) {
                uint32_t m = 1;
                for (size_t k = i; k < std::min(i + 64, rows.size()); ++k) m = std::max(m, ptr[rows[k] + 1] - ptr[rows[k]]);
                const size_t base = sp_ent[t].size();
                sp_chunk[t].push_back(make_uint2((uint32_t)base, m));
                sp_ent[t].resize(base + 64 * (size_t)m, make_uint2(0u, 0u));
                for (size_t k = i; k < i + 64; ++k) {
                    if (k >= rows.size()) {
                        sp_rl[t].push_back(make_uint2(0u, ~0u));
                        continue;
                    }
                    const uint32_t r = rows[k], len = ptr[r + 1] - ptr[r];
                    sp_rl[t].push_back(make_uint2(r, len));
                    for (uint32_t e = 0; e < len; ++e)
                        sp_ent[t][base + 64 * (size_t)e + (k - i)] =
                            t ? make_uint2(ptr[r] + e, an->in_ai[ptr[r] + e])
                              : make_uint2(a_src[ptr[r] + e], a_cidx[ptr[r] + e]);
                }
            }
        }
        // the first sweeps' right-hand sides by row
        df_rsrc.resize(n);
        df_rscale.resize(n);
        tdf_rsrc.resize(n);
        tdf_rscale.resize(n);
        for (uint32_t q = 0; q < n; ++q) {
            const uint32_t t = an->row_perm[q];
            df_rsrc[q] = an->col_perm[q];
            df_rscale[q] = an->col_scale_perm[q];
            tdf_rsrc[q] = t;
            tdf_rscale[q] = an->row_scale[t];
        }
        p->has_scaling = p->has_refine = true;
    }

    std::vector<uint2> cln2(T.cln.size());   // {L position, pivot position} per lane
    for (size_t q = 0; q < T.cln.size(); ++q) cln2[q] = make_uint2(T.cln[q].x, T.cln[q].y);
    std::vector<uint4> mrec;
    merge_records(T.ment, T.msrc_ptr, T.msrc, 0, (uint32_t)T.ment.size(), [](uint32_t q) { return q; }, mrec);

    // ---------------- upload everything into one arena ------------------
    if (factor_steps.valid()) factor_steps.get();
    p->nwin = (int)wins.size();
    for (const Window &w : wins) {
        p->win_steps += w.l1 - w.l0;
        p->win_nslot = std::max<uint32_t>(p->win_nslot, (uint32_t)w.pos.size());
        p->win_slots.push_back((uint32_t)w.pos.size());
    }
    T.umap = std::vector<uint32_t>();
    factor_segments(*p, T, phases, wins);
    p->units = (int64_t)(T.cln.size() / 64);
    // The batched kernels' leading grid steps: those ahead of the first LDS
    // window with at least a workgroup's worth of lanes per matrix (a
    // narrower step takes one pass of the per-matrix workgroup anyway).
    {
        const int lim = std::min({wins.empty() ? P.num_lev : std::min(wins[0].l0, P.num_lev),
                                  p->batch_grid_opt < 0 ? 0 : p->batch_grid_opt > 0 ? p->batch_grid_opt : INT32_MAX});
        const uint32_t per_wave = launch::il_items_per_wave();
        for (int l = 0; l < lim && level_lanes(T, l) >= (uint32_t)p->fused_threads; ++l) {
            const uint32_t ml = T.ment_long[l], nm = T.ment_ptr[l + 1] - T.ment_ptr[l];
            const uint32_t items = (T.ctask_ptr[l + 1] - T.ctask_ptr[l]) * 64 + (nm - ml) +
                                   (l > 0 ? T.dvd_ptr[l] - T.dvd_ptr[l - 1] : 0u);   // + previous step's divisions
            p->grid_waves.push_back(ml + (items + per_wave - 1) / per_wave);
        }
        p->batch_grid_lev = (int)p->grid_waves.size();
    }
    // Division items: those of the columns of each of the batched kernels'
    // grid steps but the last run with the next grid step (kept step by
    // step); the rest run in one pass after the last step (the single path
    // runs them all there).  Each step's items, and the rest, are in
    // position order: a wave's items are then consecutive L entries of a
    // column (each column's first entry first) and read and write whole
    // lines.
    {
        const auto by_pos = [](const uint2 &a, const uint2 &b) { return a.x < b.x; };
        const int early = std::max(p->batch_grid_lev - 1, 0);
        for (int l = 0; l < early; ++l)
            std::sort(T.dvd.begin() + T.dvd_ptr[l], T.dvd.begin() + T.dvd_ptr[l + 1], by_pos);
        std::sort(T.dvd.begin() + T.dvd_ptr[early], T.dvd.end(), by_pos);
    }


    Uploader U;
    const size_t o_colptr = U.put(P.sym_c_ptr, n + 1);
    std::vector<uint32_t> gcols;   // columns of the pattern, long ones first (GESP sums)
    gcols.reserve(n);
    for (int pass = 0; pass < 2; ++pass) {
        for (uint32_t c = 0; c < n; ++c)
            if ((P.sym_c_ptr[c + 1] - P.sym_c_ptr[c] > kLongRow) == (pass == 0)) gcols.push_back(c);
        if (pass == 0) p->F.ngl = (uint32_t)gcols.size();
    }
    const size_t o_gcols = U.put(gcols);
    const size_t o_rowidx = U.put(P.sym_r_idx, P.nnz);
    const size_t o_diag = U.put(P.l_col_ptr, n);
    const size_t o_crptr = U.put(P.csr_r_ptr, n + 1);
    const size_t o_ccidx = U.put(P.csr_c_idx, P.nnz);
    const size_t o_cdiag = U.put(P.csr_diag_ptr, n);
    const size_t o_upos = U.put(T.upos);
    const size_t o_cptr = U.put(T.ctask_ptr);
    const size_t o_cln = U.put(cln2);
    const size_t o_ctgt = U.put(T.ctgt);
    const size_t o_cup = U.put(T.cup);
    const size_t o_ment = U.put(T.ment);
    const size_t o_mptr = U.put(T.ment_ptr);
    const size_t o_mlong = U.put(T.ment_long);
    const size_t o_msptr = U.put(T.msrc_ptr);
    const size_t o_msrc = U.put(T.msrc);
    const size_t o_mrec = U.put(mrec);
    const size_t o_dvd = U.put(T.dvd);
    const size_t o_dptr = U.put(T.dvd_ptr);
    p->ndiv = (uint32_t)T.dvd.size();
    std::vector<size_t> o_wpos(wins.size()), o_wprog(wins.size()), o_whdr(wins.size()), o_wptr(wins.size());
    for (size_t w = 0; w < wins.size(); ++w) {
        o_wpos[w] = U.put(wins[w].pos);
        o_wprog[w] = U.put(wins[w].prog);
        o_whdr[w] = U.put(wins[w].hdr);
        o_wptr[w] = U.put(wins[w].wptr);
    }
    struct PhaseOff {
        std::vector<size_t> pos, prog, hdr, wptr;
        size_t bin, grp, tgt, cnt, wav;
    };
    std::vector<PhaseOff> o_ph(phases.size());
    size_t most_out = 0;
    for (size_t k = 0; k < phases.size(); ++k) {
        PhaseOff &o = o_ph[k];
        for (const Window &w : phases[k].bin) {
            o.pos.push_back(U.put(w.pos));
            o.prog.push_back(U.put(w.prog));
            o.hdr.push_back(U.put(w.hdr));
            o.wptr.push_back(U.put(w.wptr));
        }
        o.grp = U.put(phases[k].grp);
        o.tgt = U.put(phases[k].tgt);
        o.cnt = U.put(phases[k].cnt);
        o.wav = U.put(phases[k].wav);
        o.bin = U.reserve(sizeof(WinDev) * phases[k].bin.size());
        most_out = std::max<size_t>(most_out, phases[k].nout);
    }
    const size_t o_out = U.reserve(sizeof(float) * most_out);
    p->phase_out = most_out;
    const size_t o_wdev = U.reserve(sizeof(WinDev) * std::max<size_t>(wins.size(), 1));
    struct SwOff {
        size_t meta, wave, part, row, rpos, prod;
    };
    SwOff o_sw[4], o_hd[4];
    for (int q = 0; q < 4; ++q)
        for (int k = 0; k < 2; ++k) {
            SwHost &h = k ? hd[q] : sw[q];
            if (h.prod.size())   // product values count from the copy's start
                for (SwProd &e : h.prod) e.val += k ? hd_voff[q] : sw_voff[q];
            (k ? o_hd : o_sw)[q] = SwOff{U.put(h.meta), U.put(h.wave), U.put(h.part),
                                         U.put(h.row), U.put(h.rpos), U.put(h.prod)};
        }
    const size_t o_spl[2] = {U.put(spl_vpos[0]), U.put(spl_vpos[1])};
    if (!long_lanes) dlo = dup = dtu = dtl = DfHost();   // (not uploaded: the streams replace them)
    const size_t o_dlo_task = U.put(dlo.task), o_dlo_rl = U.put(dlo.rl), o_dlo_idx = U.put(dlo.idx);
    const size_t o_dup_task = U.put(dup.task), o_dup_rl = U.put(dup.rl), o_dup_idx = U.put(dup.idx);
    const size_t o_dtu_task = U.put(dtu.task), o_dtu_rl = U.put(dtu.rl), o_dtu_idx = U.put(dtu.idx);
    const size_t o_dtl_task = U.put(dtl.task), o_dtl_rl = U.put(dtl.rl), o_dtl_idx = U.put(dtl.idx);
    const size_t o_tdfsrc = U.put(tdf_vpos);
    const size_t o_dfsrc = U.put(df_vpos);
    const size_t o_dfcpy = U.put(df_cpy), o_dfcptr = U.put(df_cpy_ptr);
    size_t o_trows[4], o_tptr[4], o_tlong[4], o_ttask[4];
    for (int s = 0; s < 4; ++s) {
        o_trows[s] = U.put(p->tri[s].rows);
        o_tptr[s] = U.put(p->tri[s].lvl_ptr);
        o_tlong[s] = U.put(p->tri[s].lvl_long);
        o_ttask[s] = U.put(p->tri[s].tasks);
    }
    size_t o_spc[2] = {0, 0}, o_spr[2] = {0, 0}, o_spe[2] = {0, 0};
    size_t o_rsrc = 0, o_rscale = 0, o_trsrc = 0, o_trscale = 0;
    size_t o_rp = 0, o_rpi = 0, o_cp = 0, o_cpi = 0, o_rs = 0, o_csp = 0;
    size_t o_arptr = 0, o_acidx = 0, o_asrc = 0, o_acptr = 0, o_aridx = 0, o_lusrc = 0, o_rscol = 0;
    size_t o_lucol = 0, o_arows = 0, o_acols = 0, o_adst = 0, o_ars = 0, o_acs = 0, o_lufill = 0;
    if (an) {
        for (int t = 0; t < 2; ++t) {
            o_spc[t] = U.put(sp_chunk[t]);
            o_spr[t] = U.put(sp_rl[t]);
            o_spe[t] = U.put(sp_ent[t]);
        }
        o_rsrc = U.put(df_rsrc);
        o_rscale = U.put(df_rscale);
        o_trsrc = U.put(tdf_rsrc);
        o_trscale = U.put(tdf_rscale);
        o_rp = U.put(an->row_perm);
        o_rpi = U.put(an->row_perm_inv);
        o_cp = U.put(an->col_perm);
        o_cpi = U.put(an->col_perm_inv);
        o_rs = U.put(an->row_scale);
        o_csp = U.put(an->col_scale_perm);
        o_arptr = U.put(a_rptr);
        o_acidx = U.put(a_cidx);
        o_asrc = U.put(a_src);
        o_acptr = U.put(an->in_ap);
        o_aridx = U.put(an->in_ai);
        o_lusrc = U.put(lu_src);
        o_rscol = U.put(rs_col);
        o_lucol = U.put(lu_col);
        o_arows = U.put(a_rows);
        o_acols = U.put(a_cols);
        o_adst = U.put(a_dst);
        o_lufill = U.put(lu_fill);
        o_ars = U.put(a_rs);
        o_acs = U.put(a_cs);
    }
    const size_t o_desc = U.reserve(sizeof(MatDesc));
    const size_t o_normbits = U.reserve(sizeof(unsigned int));
    const size_t o_pert = U.reserve(sizeof(float));
    const size_t o_norms = U.reserve(4 * sizeof(unsigned long long));
    const size_t o_t32 = U.reserve(sizeof(float) * n);
    const size_t o_r64 = U.reserve(sizeof(double) * n);

    HIP_TRY(hipMalloc(&p->d_arena, U.arena.total));
    p->arena_bytes = U.arena.total;
    // large parts as they are, runs of small ones (a phase has a few per bin)
    // gathered into one copy each
    {
        constexpr size_t kSmall = 1u << 20, kRun = 32u << 20;
        std::vector<char> run;
        size_t at = 0;
        auto flush = [&]() -> hipError_t {
            const hipError_t e = run.empty() ? hipSuccess
                                             : hipMemcpy(p->d_arena + at, run.data(), run.size(), hipMemcpyHostToDevice);
            run.clear();
            return e;
        };
        for (auto &it : U.items) {
            if (!it.bytes) continue;
            if (it.bytes >= kSmall || (!run.empty() && it.off + it.bytes - at > kRun)) HIP_TRY(flush());
            if (it.bytes >= kSmall) {
                HIP_TRY(hipMemcpy(p->d_arena + it.off, it.src, it.bytes, hipMemcpyHostToDevice));
                continue;
            }
            if (run.empty()) at = it.off;
            run.resize(it.off + it.bytes - at);   // (reserved parts in between are filled later)
            std::memcpy(run.data() + (it.off - at), it.src, it.bytes);
        }
        HIP_TRY(flush());
    }
    HIP_TRY(hipMemset(p->d_arena + o_normbits, 0, sizeof(unsigned int)));

    char *A = p->d_arena;
    auto u32p = [&](size_t o) { return reinterpret_cast<const uint32_t *>(A + o); };
    FactorDev &F = p->F;
    F.col_ptr = u32p(o_colptr);
    F.gcols = u32p(o_gcols);
    F.ctask_ptr = u32p(o_cptr);
    F.cln = reinterpret_cast<const uint2 *>(A + o_cln);
    F.ctgt = u32p(o_ctgt);
    F.cup = u32p(o_cup);
    F.ment = u32p(o_ment);
    F.ment_ptr = u32p(o_mptr);
    F.ment_long = u32p(o_mlong);
    F.msrc_ptr = u32p(o_msptr);
    F.msrc = reinterpret_cast<const MergeSrc *>(A + o_msrc);
    F.mrec = reinterpret_cast<const uint4 *>(A + o_mrec);
    F.dvd = reinterpret_cast<const uint2 *>(A + o_dvd);
    F.dvd_ptr = u32p(o_dptr);
    const uint32_t *upos_d = u32p(o_upos);
    (void)upos_d;
    F.num_lev = P.num_lev;
    F.n = n;
    F.nnz = P.nnz;
    for (size_t k = 0; k < phases.size(); ++k) {
        const PhaseOff &o = o_ph[k];
        std::vector<WinDev> wd;
        for (size_t b = 0; b < phases[k].bin.size(); ++b) {
            const Window &x = phases[k].bin[b];
            WinDev d{};
            d.l0 = x.l0;
            d.l1 = x.l1;
            d.nslot = (uint32_t)x.pos.size();
            d.nwave = (uint32_t)x.wptr.size() - 1;
            d.pos = u32p(o.pos[b]);
            d.prog = reinterpret_cast<const uint4 *>(A + o.prog[b]);
            d.hdr = u32p(o.hdr[b]);
            d.wptr = u32p(o.wptr[b]);
            wd.push_back(d);
        }
        HIP_TRY(hipMemcpy(A + o.bin, wd.data(), sizeof(WinDev) * wd.size(), hipMemcpyHostToDevice));
        PhaseDev d{};
        d.bin = reinterpret_cast<const WinDev *>(A + o.bin);
        d.grp = reinterpret_cast<const uint2 *>(A + o.grp);
        d.tgt = u32p(o.tgt);
        d.cnt = reinterpret_cast<const uint8_t *>(A + o.cnt);
        d.wav = reinterpret_cast<const AsmWave *>(A + o.wav);
        d.out = reinterpret_cast<float *>(A + o_out);
        d.nbin = (uint32_t)wd.size();
        d.ngrp = (uint32_t)phases[k].grp.size();
        d.nwav = (uint32_t)phases[k].wav.size();
        d.nslot = phases[k].nslot;
        p->phases.push_back(d);
        p->phase_work.emplace_back();
        for (const Window &w : phases[k].bin) p->phase_work.back().push_back((uint32_t)w.hdr.size());
        p->phase_lev = phases[k].l1;
    }
    {
        std::vector<WinDev> wd(wins.size());
        for (size_t w = 0; w < wins.size(); ++w) {
            const Window &x = wins[w];
            WinDev &d = wd[w];
            d.l0 = x.l0;
            d.l1 = x.l1;
            d.nslot = (uint32_t)x.pos.size();
            d.nwave = (uint32_t)x.wptr.size() - 1;
            d.pos = u32p(o_wpos[w]);
            d.prog = reinterpret_cast<const uint4 *>(A + o_wprog[w]);
            d.hdr = u32p(o_whdr[w]);
            d.wptr = u32p(o_wptr[w]);
        }
        if (!wd.empty())
            HIP_TRY(hipMemcpy(A + o_wdev, wd.data(), sizeof(WinDev) * wd.size(), hipMemcpyHostToDevice));
        F.win = reinterpret_cast<const WinDev *>(A + o_wdev);
        F.nwin = (int32_t)wins.size();
        F.win_nslot = p->win_nslot;
    }

    auto tri = [&](int s, const uint32_t *beg, uint32_t begoff, const uint32_t *end, const uint32_t *idx,
                   const uint32_t *vpos, const uint32_t *dpos, int desc) {
        TriDev t{};
        t.beg = beg;
        t.begoff = begoff;
        t.end = end;
        t.idx = idx;
        t.vpos = vpos;
        t.dpos = dpos;
        t.desc = desc;
        t.rows = u32p(o_trows[s]);
        t.lvl_ptr = u32p(o_tptr[s]);
        t.lvl_long = u32p(o_tlong[s]);
        t.nlev = (int)p->tri[s].lvl_ptr.size() - 1;
        t.dtask = u32p(o_ttask[s]);
        t.ntask = (uint32_t)p->tri[s].tasks.size() - 1;
        return t;
    };
    const uint32_t *colptr = u32p(o_colptr), *rowidx = u32p(o_rowidx), *diag = u32p(o_diag);
    p->d_rowidx = rowidx;
    p->d_diag = diag;
    const uint32_t *crptr = u32p(o_crptr), *ccidx = u32p(o_ccidx), *cdiag = u32p(o_cdiag);
    SolveDev &S = p->S;
    S.lo = tri(0, crptr, 0, cdiag, ccidx, upos_d, nullptr, 0);
    S.up = tri(1, cdiag, 1, crptr + 1, ccidx, upos_d, diag, 1);
    S.tup = tri(2, colptr, 0, diag, rowidx, nullptr, diag, 0);
    S.tlo = tri(3, diag, 1, colptr + 1, rowidx, nullptr, nullptr, 0);
    // the same L and U sweeps, pipelined, over the per-matrix value copy
    auto df = [&](const DfHost &h, size_t ot, size_t orl, size_t oi, int div, uint32_t voff) {
        DfDev d{};
        d.task = reinterpret_cast<const uint4 *>(A + ot);
        d.rl = reinterpret_cast<const uint2 *>(A + orl);
        d.idx = u32p(oi);
        d.ntask = (uint32_t)h.task.size();
        d.nslots = (uint32_t)h.idx.size();
        d.div = div;
        d.voff = voff;
        return d;
    };
    auto swd = [&](const SwHost &h, const SwOff &o, bool div, uint32_t voff) {
        SwDev d{};
        d.meta = reinterpret_cast<const uint4 *>(A + o.meta);
        d.wave = reinterpret_cast<const uint4 *>(A + o.wave);
        d.part = reinterpret_cast<const SwPart *>(A + o.part);
        d.row = u32p(o.row);
        d.rpos = u32p(o.rpos);
        d.prod = reinterpret_cast<const SwProd *>(A + o.prod);
        d.nprod = (uint32_t)h.prod.size();
        d.nwave = h.nwave;
        d.voff = voff;
        d.div = div;
        return d;
    };
    if (!long_lanes)
        for (int q = 0; q < 4; ++q) S.sw[q] = swd(sw[q], o_sw[q], divs[q], sw_voff[q]);
    S.t32_len = p->t32_len;
    p->has_split = split;
    if (split)
        for (int t = 0; t < 2; ++t) {
            SplitDev &d = p->split[t];
            for (int k = 0; k < 2; ++k) {
                d.head[k] = swd(hd[2 * t + k], o_hd[2 * t + k], divs[2 * t + k], hd_voff[2 * t + k]);
                d.tail[k] = swd(sw[2 * t + k], o_sw[2 * t + k], divs[2 * t + k], sw_voff[2 * t + k]);
            }
            d.src = u32p(o_spl[t]);
            d.nval = (uint32_t)spl_vpos[t].size();
            d.parts = (uint32_t)hd[2 * t].part.size();
            d.head_slots = std::max(hd[2 * t].nslot_max, hd[2 * t + 1].nslot_max);
            d.tail_slots = sw[2 * t].nslot_max;
        }
    S.lo_df = df(dlo, o_dlo_task, o_dlo_rl, o_dlo_idx, 0, 0);
    S.up_df = df(dup, o_dup_task, o_dup_rl, o_dup_idx, 1, (uint32_t)dlo.idx.size());
    S.tup_df = df(dtu, o_dtu_task, o_dtu_rl, o_dtu_idx, 1, 0);
    S.tlo_df = df(dtl, o_dtl_task, o_dtl_rl, o_dtl_idx, 0, tlo_voff);
    S.tdf_src = u32p(o_tdfsrc);
    S.tdf_nval = p->tdf_nval;
    S.df_src = u32p(o_dfsrc);
    S.df_nval = p->df_nval;
    S.df_cpy = reinterpret_cast<const uint2 *>(A + o_dfcpy);
    S.df_cpy_ptr = u32p(o_dfcptr);
    S.df_cpy_range = p->copy_range;
    p->tri_dataflow = p->solve_df_opt >= 0 && p->lds_cap >= 4 * (size_t)((n + 31) / 32);
    if (an) {
        S.df_rsrc = u32p(o_rsrc);
        S.df_rscale = reinterpret_cast<const double *>(A + o_rscale);
        S.tdf_rsrc = u32p(o_trsrc);
        S.tdf_rscale = reinterpret_cast<const double *>(A + o_trscale);
        p->split[0].rsrc = S.df_rsrc;
        p->split[0].rscale = S.df_rscale;
        p->split[1].rsrc = S.tdf_rsrc;
        p->split[1].rscale = S.tdf_rscale;
        S.row_perm = u32p(o_rp);
        S.row_perm_inv = u32p(o_rpi);
        S.col_perm = u32p(o_cp);
        S.col_perm_inv = u32p(o_cpi);
        S.row_scale = reinterpret_cast<const double *>(A + o_rs);
        S.col_scale_perm = reinterpret_cast<const double *>(A + o_csp);
        RefineDev &R = p->R;
        for (int t = 0; t < 2; ++t) {
            R.sp[t].chunk = reinterpret_cast<const uint2 *>(A + o_spc[t]);
            R.sp[t].rl = reinterpret_cast<const uint2 *>(A + o_spr[t]);
            R.sp[t].ent = reinterpret_cast<const uint2 *>(A + o_spe[t]);
            R.sp[t].nchunk = (uint32_t)sp_chunk[t].size();
        }
        R.a_rptr = u32p(o_arptr);
        R.a_cidx = u32p(o_acidx);
        R.a_src = u32p(o_asrc);
        R.a_cptr = u32p(o_acptr);
        R.a_ridx = u32p(o_aridx);
        R.lu_src = u32p(o_lusrc);
        R.row_idx = rowidx;
        R.lu_col = u32p(o_lucol);
        R.a_rows = u32p(o_arows);
        R.a_cols = u32p(o_acols);
        R.a_nlong = p->a_nlong;
        R.a_nlong_t = p->a_nlong_t;
        R.rs_col = reinterpret_cast<const double *>(A + o_rscol);
        R.a_dst = u32p(o_adst);
        R.lu_fill = u32p(o_lufill);
        R.nfill = (uint32_t)lu_fill.size();
        R.a_rs = reinterpret_cast<const double *>(A + o_ars);
        R.a_cs = reinterpret_cast<const double *>(A + o_acs);
        R.csp = S.col_scale_perm;
        R.nnz_a = p->nnz_a;
    }
    MatDesc md{};
    md.f = F;
    md.s = S;
    md.r = p->R;
    md.n = n;
    md.nnz = P.nnz;
    md.krylov = (uint32_t)p->krylov;
    md.a_kmax = p->a_kmax;
    p->d_desc = reinterpret_cast<MatDesc *>(A + o_desc);
    HIP_TRY(hipMemcpy(p->d_desc, &md, sizeof(MatDesc), hipMemcpyHostToDevice));
    p->d_norm_bits = reinterpret_cast<unsigned int *>(A + o_normbits);
    p->d_pert = reinterpret_cast<float *>(A + o_pert);
    p->d_norms = reinterpret_cast<unsigned long long *>(A + o_norms);
    p->d_t32 = reinterpret_cast<float *>(A + o_t32);
    p->d_r64 = reinterpret_cast<double *>(A + o_r64);
    *out = p.release();
    return GLU_OK;
}

glu_pattern pattern_of(const Symbolic &s)
{
    glu_pattern P{};
    P.n = s.n;
    P.nnz = s.nnz;
    P.num_lev = s.num_lev;
    P.sym_c_ptr = s.sym_c_ptr.data();
    P.sym_r_idx = s.sym_r_idx.data();
    P.l_col_ptr = s.l_col_ptr.data();
    P.csr_r_ptr = s.csr_r_ptr.data();
    P.csr_c_idx = s.csr_c_idx.data();
    P.csr_diag_ptr = s.csr_diag_ptr.data();
    P.level_ptr = s.level_ptr.data();
    P.level_idx = s.level_idx.data();
    return P;
}

glu_status run_factor(glu_plan *p, float *d_val, int perturb, hipStream_t st)
{
    if (perturb) launch::pert(p->F, d_val, p->d_norm_bits, p->d_pert, st);
    for (const Segment &s : p->fsegs) {
        if (s.phase >= 0)
            launch::factor_phase(p->phases[s.phase], d_val, p->d_pert, perturb, (int)kPhaseWaves * 64, st);
        else if (s.win >= 0)
            launch::factor_window(p->F, s.win, p->win_slots[s.win], d_val, p->d_pert, perturb, p->fused_threads, st);
        else if (s.fused)
            launch::factor_fused(p->F, d_val, p->d_pert, s.l0, s.l1, perturb, p->fused_threads, st);
        else
            launch::factor_grid(p->F, d_val, p->d_pert, s.l0, s.items, perturb, kGridThreads, st);
    }
    launch::factor_divide(p->F, d_val, p->d_pert, p->ndiv, perturb, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("factor launch: ") + hipGetErrorString(e));
    return GLU_OK;
}

void run_tri(glu_plan *p, const TriDev &T, const TriHost &H, const float *lu, float *x, hipStream_t st)
{
    for (const Segment &s : H.segs) {
        if (s.fused && p->tri_dataflow)
            launch::tri_df(T, lu, x, s.l0, s.l1, s.k0, s.k1, p->n, p->fused_threads, st);
        else if (s.fused)
            launch::tri_fused(T, lu, x, s.l0, s.l1, p->fused_threads, st);
        else
            launch::tri_grid(T, lu, x, s.l0, s.items, st);
    }
}

// t (scaled, permuted) -> LU sweeps in place
void run_sweeps(glu_plan *p, const float *lu, float *t, int transpose, hipStream_t st)
{
    if (!transpose) {
        run_tri(p, p->S.lo, p->tri[0], lu, t, st);
        run_tri(p, p->S.up, p->tri[1], lu, t, st);
    } else {
        run_tri(p, p->S.tup, p->tri[2], lu, t, st);
        run_tri(p, p->S.tlo, p->tri[3], lu, t, st);
    }
}

// Rows whose values a one-workgroup sweep with ready bits of `bits` bytes
// keeps in the rest of `cap` bytes of LDS: the last ones, when they are at
// least a quarter of the n rows, else none.
uint32_t split_rows(uint32_t n, size_t bits, size_t cap)
{
    const size_t keep = cap > bits ? std::min<size_t>(n, (cap - bits) / sizeof(float)) : 0;
    return 4 * keep >= n ? (uint32_t)keep : 0u;
}

// The richest sweep mode of the batch kernels whose LDS fits order n:
// 2 = ready bits and correction vector in LDS, 1 = ready bits only,
// 0 = level-synchronous sweeps.
int sweep_mode(uint32_t n, size_t cap)
{
    for (int mode = 2; mode > 0; --mode)
        if (launch::batch_lds_bytes(mode, n) <= cap) return mode;
    return 0;
}

glu_status ensure_batch(glu_plan *p, int batch)
{
    if (batch <= p->batch_cap) return GLU_OK;
    if (p->d_bt32) (void)hipFree(p->d_bt32);
    if (p->d_br64) (void)hipFree(p->d_br64);
    if (p->d_blucsr) (void)hipFree(p->d_blucsr);
    if (p->d_bnorms) (void)hipFree(p->d_bnorms);
    if (p->d_bkry) (void)hipFree(p->d_bkry);
    p->d_bkry = nullptr;
    p->d_bt32 = nullptr;
    p->d_br64 = nullptr;
    p->d_blucsr = nullptr;
    p->d_bnorms = nullptr;
    p->batch_cap = 0;
    HIP_TRY(hipMalloc(&p->d_bt32, sizeof(float) * (size_t)p->t32_len * batch));
    HIP_TRY(hipMalloc(&p->d_br64, sizeof(double) * (size_t)p->n * batch));
    HIP_TRY(hipMalloc(&p->d_blucsr, sizeof(float) * (size_t)p->df_nval * batch));
    HIP_TRY(hipMalloc(&p->d_bnorms, 2 * sizeof(double) * (size_t)batch));
    if (p->krylov)
        HIP_TRY(hipMalloc(&p->d_bkry, sizeof(double) * (3 * (size_t)p->krylov + 1) * p->n * (size_t)batch));
    p->batch_cap = batch;
    return GLU_OK;
}

// Is the caller capturing a graph on st?
bool capturing(hipStream_t st)
{
    hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &c) == hipSuccess) return c != hipStreamCaptureStatusNone;
    (void)hipGetLastError();   // (the null stream beside a capture: the launches report it)
    return false;
}

// The buffers of one matrix's sweeps (p->single[transpose]).
glu_status ensure_single(glu_plan *p, int transpose)
{
    glu_plan::Single &q = p->single[transpose];
    if (q.buf) return GLU_OK;
    const size_t nval = p->has_split ? p->split[transpose].nval : transpose ? p->tdf_nval : p->df_nval;
    const size_t rhs = p->has_split ? p->rhs_len[transpose] : p->t32_len;
    const size_t a = (nval + 63) & ~(size_t)63, b = (rhs + 63) & ~(size_t)63;
    HIP_TRY(hipMalloc(&q.buf, sizeof(float) * (a + b + p->n)));
    q.lucsr = q.buf;
    q.rhs = q.buf + a;
    q.xg = q.rhs + b;
    return GLU_OK;
}

}  // namespace

extern "C" glu_status glu_plan_create(const glu_pattern *pat, const glu_plan_opts *opts, glu_plan **out)
{
    if (!pat || !out) return fail(GLU_ERR_ARGUMENT, "null argument");
    return guarded([&] { return build_plan(*pat, nullptr, opts, out); });
}

extern "C" glu_status glu_plan_create_from_analysis(const glu_analysis *a, const glu_plan_opts *opts,
                                                    glu_plan **out)
{
    if (!a || !out) return fail(GLU_ERR_ARGUMENT, "null argument");
    glu_pattern P = pattern_of(a->sym);
    return guarded([&] { return build_plan(P, a, opts, out); });
}

extern "C" void glu_plan_destroy(glu_plan *p) { delete p; }

extern "C" glu_status glu_plan_info(const glu_plan *p, int64_t info[12])
{
    if (!p || !info) return fail(GLU_ERR_ARGUMENT, "null argument");
    info[0] = p->n;
    info[1] = p->nnz;
    info[2] = p->nnz_a;
    info[3] = p->num_lev;
    info[4] = p->updates;
    info[5] = (int64_t)p->fsegs.size();
    info[6] = (int64_t)p->arena_bytes;
    info[7] = p->units;
    info[8] = p->nwin;
    info[9] = p->win_steps;
    info[10] = p->win_nslot;
    info[11] = p->batch_grid_lev;
    return GLU_OK;
}

namespace {

// Replays slot's graph on st, capturing `issue` (which enqueues the launch
// sequence on the stream it is given) first when the slot is empty or was
// captured for other buffers / another mode.
template <typename Issue>
glu_status replay(glu_plan *p, glu_plan::GraphSlot &slot, const void *k0, const void *k1, const void *k2, int mode,
                  hipStream_t st, Issue issue)
{
    if (!slot.exec || slot.k[0] != k0 || slot.k[1] != k1 || slot.k[2] != k2 || slot.mode != mode) {
        if (slot.exec) {
            HIP_TRY(hipStreamSynchronize(st));   // the old graph may still run
            HIP_TRY(hipGraphExecDestroy(slot.exec));
            slot.exec = nullptr;
        }
        if (!p->cap_stream) HIP_TRY(hipStreamCreateWithFlags(&p->cap_stream, hipStreamNonBlocking));
        HIP_TRY(hipStreamBeginCapture(p->cap_stream, hipStreamCaptureModeThreadLocal));
        glu_status s = issue(p->cap_stream);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(p->cap_stream, &g);
        if (s != GLU_OK) {
            if (g) (void)hipGraphDestroy(g);
            return s;
        }
        if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("graph capture: ") + hipGetErrorString(e));
        e = hipGraphInstantiate(&slot.exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            slot.exec = nullptr;
            return fail(GLU_ERR_DEVICE, std::string("graph instantiate: ") + hipGetErrorString(e));
        }
        slot.k[0] = k0;
        slot.k[1] = k1;
        slot.k[2] = k2;
        slot.mode = mode;
    }
    HIP_TRY(hipGraphLaunch(slot.exec, st));
    return GLU_OK;
}

}  // namespace

extern "C" glu_status glu_factor(glu_plan *p, float *d_val, int perturb, void *stream)
{
    if (!p || !d_val) return fail(GLU_ERR_ARGUMENT, "null argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (!p->use_graph) return run_factor(p, d_val, perturb, st);
    return replay(p, p->g_factor, d_val, nullptr, nullptr, perturb ? 1 : 0, st,
                  [&](hipStream_t cs) { return run_factor(p, d_val, perturb, cs); });
}

extern "C" glu_status glu_factor_host(glu_plan *p, float *h_val, int perturb)
{
    if (!p || !h_val) return fail(GLU_ERR_ARGUMENT, "null argument");
    if (!p->d_val) HIP_TRY(hipMalloc(&p->d_val, sizeof(float) * p->nnz));
    HIP_TRY(hipMemcpy(p->d_val, h_val, sizeof(float) * p->nnz, hipMemcpyHostToDevice));
    glu_status s = run_factor(p, p->d_val, perturb, nullptr);
    if (s != GLU_OK) return s;
    HIP_TRY(hipDeviceSynchronize());
    HIP_TRY(hipMemcpy(h_val, p->d_val, sizeof(float) * p->nnz, hipMemcpyDeviceToHost));
    return GLU_OK;
}

extern "C" glu_status glu_solve(glu_plan *p, const float *d_lu, const float *d_b, float *d_x, int transpose,
                                void *stream)
{
    if (!p || !d_lu || !d_b || !d_x) return fail(GLU_ERR_ARGUMENT, "null argument");
    if (!p->has_scaling) return fail(GLU_ERR_ARGUMENT, "plan has no permutation/scaling (create it from an analysis)");
    hipStream_t st = static_cast<hipStream_t>(stream);
    transpose = transpose ? 1 : 0;
    // mode 2: one workgroup, the vector in LDS (A x = b and A' x = b);
    // 1: the split sweeps, or (A x = b) one workgroup with the ready bits in
    // LDS; 0: level by level.  All give the reference's arithmetic.
    int mode = p->tri_dataflow ? sweep_mode(p->n, launch::enable_lds()) : 0;
    if (mode == 1 && !p->has_split && transpose) mode = 0;
    // the other modes' buffers come with their first call; in a capture, which
    // cannot allocate, that call runs level by level
    if (mode != 0 && !p->single[transpose].buf && capturing(st)) mode = 0;
    const bool split = mode == 1 && p->has_split;
    if (mode != 0) {
        glu_status s = ensure_single(p, transpose);   // (before any graph capture)
        if (s != GLU_OK) return s;
    }
    auto issue = [&](hipStream_t s) {
        const SolveDev &S = p->S;
        const glu_plan::Single &q = p->single[transpose];
        if (split) {
            const SplitDev &d = p->split[transpose];
            launch::copy_df(d.src, d.nval, d_lu, q.lucsr, s);
            launch::split_solve(d, d_b, d_lu, q.lucsr, q.rhs, q.xg, s);
            if (!transpose)
                launch::perm_scale_f32(q.xg, d_x, S.row_perm_inv, S.row_scale, 0, p->n, s);
            else
                launch::perm_scale_f32(q.xg, d_x, S.col_perm_inv, S.col_scale_perm, 1, p->n, s);
        } else if (mode != 0) {
            // mode 1: the LDS the ready bits leave free holds the last rows
            // (r0..n-1) when they are a quarter of the rows or more
            const size_t bits = launch::batch_lds_bytes(mode, p->n), cap = launch::enable_lds();
            const uint32_t keep = mode == 1 ? split_rows(p->n, bits, cap) : 0u;
            launch::solve_one(p->d_desc, transpose ? S.tdf_src : S.df_src, transpose ? p->tdf_nval : p->df_nval, d_lu,
                              q.lucsr, d_b, d_x, q.rhs, keep ? p->n - keep : UINT32_MAX, p->fused_threads, mode,
                              bits + sizeof(float) * keep, transpose, s);
        } else if (!transpose) {
            launch::perm_scale_f32(d_b, p->d_t32, S.col_perm, S.col_scale_perm, 0, p->n, s);
            run_sweeps(p, d_lu, p->d_t32, 0, s);
            launch::perm_scale_f32(p->d_t32, d_x, S.row_perm_inv, S.row_scale, 0, p->n, s);
        } else {
            launch::perm_scale_f32(d_b, p->d_t32, S.row_perm, S.row_scale, 1, p->n, s);
            run_sweeps(p, d_lu, p->d_t32, 1, s);
            launch::perm_scale_f32(p->d_t32, d_x, S.col_perm_inv, S.col_scale_perm, 1, p->n, s);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("solve launch: ") + hipGetErrorString(e));
        return GLU_OK;
    };
    if (!p->use_graph) return issue(st);
    return replay(p, p->g_solve[transpose], d_lu, d_b, d_x, mode, st, issue);
}

extern "C" glu_status glu_refresh(glu_plan *p, const double *d_ax, float *d_lu, int batch, void *stream)
{
    if (!p || !d_ax || !d_lu || batch <= 0) return fail(GLU_ERR_ARGUMENT, "bad argument");
    if (!p->has_refine) return fail(GLU_ERR_ARGUMENT, "plan has no analysis");
    launch::refresh(p->R, d_ax, d_lu, p->nnz, batch, static_cast<hipStream_t>(stream));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("refresh launch: ") + hipGetErrorString(e));
    return GLU_OK;
}

static double bits_to_double(unsigned long long b)
{
    double d;
    std::memcpy(&d, &b, sizeof d);
    return d;
}

namespace {

// Plain iterative refinement driven from the host, one preconditioner
// solve per iteration: x = 0, r = b; then t = float(r scaled into the
// factors' frame), the two sweeps on t, x += t scaled back, r = b - A x with
// |r|, |x| (and |A|, |b| on the first pass), eta on the host.  The FP64 work
// runs in grid kernels; the sweeps run in one workgroup over the
// sweep-layout copy `lucsr` (dataflow, ready bits in LDS) or, when lucsr is
// null, level by level over the factors; with `rhs`, they are the split
// sweeps (right-hand sides in rhs, lucsr their copy, t32 the vector by row).
glu_status refine_host_loop(glu_plan *p, const double *d_ax, const float *d_lu, const double *d_b, double *d_x,
                            double tol, int maxit, int transpose, float *lucsr, float *rhs, float *t32, double *r64,
                            unsigned long long *norms, int *h_iters, double *h_eta, hipStream_t st)
{
    const SolveDev &S = p->S;
    const uint32_t n = p->n;
    // the sweeps keep the results of the last rows in the LDS their ready
    // bits leave free (rows r0..n-1), when that is a quarter of the rows or
    // more (below that the test per access costs more than it saves)
    const size_t bits = launch::batch_lds_bytes(1, n), cap = launch::enable_lds();
    const uint32_t keep = split_rows(n, bits, cap), r0 = keep ? n - keep : UINT32_MAX;
    HIP_TRY(hipMemsetAsync(d_x, 0, sizeof(double) * n, st));
    HIP_TRY(hipMemcpyAsync(r64, d_b, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
    double anorm = 0.0, bnorm = 0.0, eta = 0.0;
    int it = 0;
    for (;;) {
        if (rhs)
            launch::split_precond(p->split[transpose ? 1 : 0], r64, d_lu, lucsr, rhs, t32, st);
        else if (!transpose)
            launch::perm_scale_f64(r64, t32, S.col_perm, S.col_scale_perm, 0, n, st);
        else
            launch::perm_scale_f64(r64, t32, S.row_perm, S.row_scale, 1, n, st);
        if (rhs)
            ;   // the split sweeps scaled the residual themselves
        else if (lucsr)
            launch::sweeps_df(p->d_desc, lucsr, t32, r0, p->fused_threads, bits + sizeof(float) * keep, transpose, st);
        else
            run_sweeps(p, d_lu, t32, transpose, st);
        if (!transpose)
            launch::update_x(t32, d_x, S.row_perm_inv, S.row_scale, 0, n, st);
        else
            launch::update_x(t32, d_x, S.col_perm_inv, S.col_scale_perm, 1, n, st);
        launch::zero_u64(norms, 4, st);
        const uint32_t nl = transpose ? p->a_nlong_t : p->a_nlong;
        launch::residual(p->R, d_ax, d_b, d_x, r64, n, transpose, it == 0, norms, (n - nl) + nl * 64, st);
        HIP_TRY(hipGetLastError());
        unsigned long long nb[4];
        HIP_TRY(hipMemcpyAsync(nb, norms, sizeof nb, hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        if (it == 0) {
            anorm = bits_to_double(nb[2]);
            bnorm = bits_to_double(nb[3]);
        }
        const double rn = bits_to_double(nb[0]), xn = bits_to_double(nb[1]);
        eta = rn / (anorm * xn + bnorm);
        ++it;
        if (!(eta > tol) || it >= maxit) break;
    }
    if (h_iters) *h_iters = it;
    if (h_eta) *h_eta = eta;
    if (!(eta == eta)) return fail(GLU_ERR_NUMERIC, "refinement produced NaN");
    return GLU_OK;
}

// The one-workgroup refinement (sweeps, FGMRES and the products with A in
// one workgroup; sweep vector and ready bits in LDS), then its iteration
// count and eta read back.
glu_status refine_one_wg(glu_plan *p, const double *d_ax, const float *d_lu, const double *d_b, double *d_x,
                         double tol, int maxit, int transpose, float *lucsr, float *t32, double *r64,
                         double *bnorms, double *kry, char *out16, int *h_iters, double *h_eta,
                         hipStream_t st)
{
    const uint32_t n = p->n;
    int32_t *d_it = reinterpret_cast<int32_t *>(out16);
    double *d_eta = reinterpret_cast<double *>(out16 + 8);
    launch::refine_one(p->d_desc, transpose ? p->S.tdf_src : p->S.df_src, transpose ? p->tdf_nval : p->df_nval, d_ax, d_b,
                       d_x, d_lu, lucsr, t32, r64,
                       bnorms, kry, d_it, d_eta, tol, maxit, p->fused_threads, launch::batch_lds_bytes(2, n),
                       transpose, st);
    HIP_TRY(hipGetLastError());
    int32_t it = 0;
    double eta = 0.0;
    HIP_TRY(hipMemcpyAsync(&it, d_it, sizeof it, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(&eta, d_eta, sizeof eta, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (h_iters) *h_iters = it;
    if (h_eta) *h_eta = eta;
    if (!(eta == eta)) return fail(GLU_ERR_NUMERIC, "refinement produced NaN");
    return GLU_OK;
}

}  // namespace

extern "C" glu_status glu_refine(glu_plan *p, const double *d_ax, const float *d_lu, const double *d_b,
                                 double *d_x, double tol, int maxit, int transpose, int *h_iters, double *h_eta,
                                 void *stream)
{
    if (!p || !d_ax || !d_lu || !d_b || !d_x || maxit <= 0) return fail(GLU_ERR_ARGUMENT, "bad argument");
    if (!p->has_refine) return fail(GLU_ERR_ARGUMENT, "plan has no analysis");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint32_t n = p->n;
    // 2: the sweep vector fits in LDS -> everything in one workgroup (FGMRES,
    // plan.krylov); 1: only the ready bits fit -> dataflow sweeps in one
    // workgroup, FP64 work across the grid (plain refinement); 0: level by
    // level.
    const int mode = sweep_mode(n, launch::enable_lds());
    if (mode == 1 && p->has_split) {
        glu_status s = ensure_single(p, transpose ? 1 : 0);
        if (s != GLU_OK) return s;
        const glu_plan::Single &q = p->single[transpose ? 1 : 0];
        const SplitDev &d = p->split[transpose ? 1 : 0];
        launch::copy_df(d.src, d.nval, d_lu, q.lucsr, st);
        return refine_host_loop(p, d_ax, d_lu, d_b, d_x, tol, maxit, transpose, q.lucsr, q.rhs, q.xg, p->d_r64,
                                p->d_norms, h_iters, h_eta, st);
    }
    float *lucsr = nullptr;
    if (mode != 0) {
        glu_status s = ensure_batch(p, 1);
        if (s != GLU_OK) return s;
        lucsr = p->d_blucsr;
        if (transpose) {
            if (!p->d_tlucsr) HIP_TRY(hipMalloc(&p->d_tlucsr, sizeof(float) * p->tdf_nval));
            lucsr = p->d_tlucsr;
        }
    }
    if (mode == 2) {
        if (!p->d_rout) HIP_TRY(hipMalloc(&p->d_rout, 16));
        return refine_one_wg(p, d_ax, d_lu, d_b, d_x, tol, maxit, transpose, lucsr, p->d_bt32, p->d_br64,
                             p->d_bnorms, p->d_bkry, p->d_rout, h_iters, h_eta, st);
    }
    if (mode == 1)
        launch::copy_df(transpose ? p->S.tdf_src : p->S.df_src, transpose ? p->tdf_nval : p->df_nval, d_lu, lucsr, st);
    return refine_host_loop(p, d_ax, d_lu, d_b, d_x, tol, maxit, transpose, lucsr, nullptr, p->d_t32, p->d_r64,
                            p->d_norms, h_iters, h_eta, st);
}

// ---------------------------------------------------------------------------
// glu_refine_noalloc: glu_refine's one-workgroup path with its scratch in a
// file-scope device array instead of plan buffers grown on first use.
// ---------------------------------------------------------------------------

namespace {

constexpr size_t kScratchBytes = GLU_NOALLOC_SCRATCH_BYTES / 2 * (size_t)5;   // see noalloc_layout
constexpr int kScratchDevices = 64;

// One copy per device, held until the process ends.  Host code never uses
// this name as an address: each device's copy is reached through the
// pointer hipGetSymbolAddress gives for it (scratch_base).
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

std::mutex g_scratch_mu;
unsigned char *g_scratch_ptr[kScratchDevices] = {};

// The calling thread's current device's copy of `scratch`, looked up once
// per device (with that device current).
glu_status scratch_base(unsigned char **out)
{
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kScratchDevices) return fail(GLU_ERR_DEVICE, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(GLU_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = static_cast<unsigned char *>(ptr);
    }
    *out = g_scratch_ptr[dev];
    return GLU_OK;
}

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// The scratch of glu_refine_noalloc in sweep mode `mode` (t: A' x = b): sweep
// value copy, right-hand sides and vector, residual, norms (one-workgroup
// path: FP64 |b| slots, FGMRES vectors, iteration count + eta; grid path: the
// four norm words).  limit: what GLU_NOALLOC_SCRATCH_BYTES counts, the same
// with the dataflow tables' slots in the copy and no right-hand sides.
//
// Every order within the limit fits kScratchBytes.  One workgroup (mode 2): a
// sweep's streams have at most (slots + 64 n) / 3 lanes (the most by slots: a
// row of 65 entries, 128 slots and 64 lanes, and one of 320, 320 and 128), so
// with 4 and 5 values a lane and the right-hand sides the layout takes at most
// 2 limit + 207.4 n floats, and n <= 39,718 (the vector and the ready bits in
// 160 KB): 160 MiB.  Split sweeps (mode 1) take the split's copy when it
// fits, else the one workgroup's, which is what the limit counts (the same
// bits).
struct NoallocLayout {
    bool split = false;
    uint32_t nval = 0;
    size_t val = 0, rhs = 0, t32 = 0, r64 = 0, norms = 0, kry = 0, out = 0, bytes = 0, limit = 0;
};

NoallocLayout noalloc_layout(const glu_plan &p, int mode, int t)
{
    const size_t n = p.n, kry = mode == 2 && p.krylov ? sizeof(double) * (3 * (size_t)p.krylov + 1) * n : 0;
    NoallocLayout L;
    L.split = mode == 1 && p.has_split;
    for (;;) {
        size_t off = 0;
        auto take = [&](size_t bytes) {
            const size_t o = off;
            off = align256(off + bytes);
            return o;
        };
        L.nval = L.split ? p.split[t].nval : t ? p.tdf_nval : p.df_nval;
        L.val = take(sizeof(float) * (size_t)L.nval);
        L.rhs = take(L.split ? sizeof(float) * (size_t)p.rhs_len[t] : 0);
        L.t32 = take(sizeof(float) * (mode == 2 ? std::max<size_t>(p.rhs_len[t], n) : n));
        L.r64 = take(sizeof(double) * n);
        L.norms = take(4 * sizeof(unsigned long long));
        L.kry = take(kry);
        L.out = take(16);
        L.bytes = off;
        if (!L.split || L.bytes <= kScratchBytes) break;
        L.split = false;
    }
    L.limit = align256(sizeof(float) * (size_t)p.scratch_nval[t]) + align256(sizeof(float) * n) +
              align256(sizeof(double) * n) + align256(4 * sizeof(unsigned long long)) + align256(kry) + align256(16);
    return L;
}

}  // namespace

extern "C" glu_status glu_refine_noalloc(glu_plan *p, const double *d_ax, const float *d_lu, const double *d_b,
                                         double *d_x, double tol, int maxit, int transpose, int *h_iters,
                                         double *h_eta, void *stream)
{
    if (!p || !d_ax || !d_lu || !d_b || !d_x || maxit <= 0) return fail(GLU_ERR_ARGUMENT, "bad argument");
    if (!p->has_refine) return fail(GLU_ERR_ARGUMENT, "plan has no analysis");
    const uint32_t n = p->n;
    const int mode = sweep_mode(n, launch::enable_lds());
    if (mode == 0)
        return fail(GLU_ERR_ARGUMENT, "order " + std::to_string(n) +
                                          " is beyond the dataflow sweeps (their ready bits exceed LDS): "
                                          "use glu_refine");
    const int t = transpose ? 1 : 0;
    const NoallocLayout L = noalloc_layout(*p, mode, t);
    if (L.limit > GLU_NOALLOC_SCRATCH_BYTES || L.bytes > kScratchBytes)
        return fail(GLU_ERR_ARGUMENT, "refinement needs " + std::to_string(L.limit) + " bytes of scratch; the static " +
                                          "scratch holds " + std::to_string(GLU_NOALLOC_SCRATCH_BYTES) + ": use glu_refine");
    unsigned char *base = nullptr;
    glu_status s = scratch_base(&base);
    if (s != GLU_OK) return s;
    hipStream_t st = static_cast<hipStream_t>(stream);
    float *lucsr = reinterpret_cast<float *>(base + L.val);
    float *t32 = reinterpret_cast<float *>(base + L.t32);
    double *r64 = reinterpret_cast<double *>(base + L.r64);
    if (mode == 2)   // as glu_refine: everything in one workgroup
        return refine_one_wg(p, d_ax, d_lu, d_b, d_x, tol, maxit, transpose, lucsr, t32, r64,
                             reinterpret_cast<double *>(base + L.norms),
                             p->krylov ? reinterpret_cast<double *>(base + L.kry) : nullptr,
                             reinterpret_cast<char *>(base + L.out), h_iters, h_eta, st);
    // as glu_refine: the split sweeps, or both sweeps in one workgroup
    launch::copy_df(L.split ? p->split[t].src : transpose ? p->S.tdf_src : p->S.df_src, L.nval, d_lu, lucsr, st);
    return refine_host_loop(p, d_ax, d_lu, d_b, d_x, tol, maxit, transpose, lucsr,
                            L.split ? reinterpret_cast<float *>(base + L.rhs) : nullptr, t32, r64,
                            reinterpret_cast<unsigned long long *>(base + L.norms), h_iters, h_eta, st);
}

extern "C" glu_status glu_adjoint_values(glu_plan *p, const double *d_lam, const double *d_x, double *d_grad_ax,
                                         void *stream)
{
    if (!p || !d_lam || !d_x || !d_grad_ax) return fail(GLU_ERR_ARGUMENT, "null argument");
    if (!p->has_refine) return fail(GLU_ERR_ARGUMENT, "plan has no analysis");
    launch::adjoint_values(p->R, d_lam, d_x, d_grad_ax, p->n, static_cast<hipStream_t>(stream));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("adjoint launch: ") + hipGetErrorString(e));
    return GLU_OK;
}

namespace {

// Scratch of the interleaved steps for `batch` matrices (grown on demand;
// the GESP maxima start at zero and every call leaves them so).
glu_status ensure_il(glu_plan *p, int batch)
{
    if (p->batch_grid_lev == 0 || batch <= p->il_cap) return GLU_OK;
    for (void *q : {(void *)p->d_il, (void *)p->d_il_bits, (void *)p->d_fnorms})
        if (q) (void)hipFree(q);
    p->d_il = nullptr;
    p->d_il_bits = nullptr;
    p->d_fnorms = nullptr;
    p->il_cap = 0;
    const size_t padded = ((size_t)batch + launch::il_group() - 1) / launch::il_group() * launch::il_group();
    HIP_TRY(hipMalloc(&p->d_il, sizeof(float) * padded * p->nnz));
    HIP_TRY(hipMalloc(&p->d_il_bits, sizeof(unsigned int) * (size_t)batch));
    HIP_TRY(hipMalloc(&p->d_fnorms, 2 * sizeof(double) * (size_t)batch));
    HIP_TRY(hipMemset(p->d_il_bits, 0, sizeof(unsigned int) * (size_t)batch));
    p->il_cap = batch;
    return GLU_OK;
}

// The batched kernels' first steps: the values of every matrix into the
// interleaved copy (with each GESP value in norms[2 m]); steps
// [0, batch_grid_lev) as one grid launch each; the factors so far into
// d_lu.  The per-matrix workgroups go on from there (with a right-hand
// side, from |b|_inf into norms[2 m + 1], x = 0 and r = b).
void batch_grid_steps(glu_plan *p, int batch, const double *d_ax, float *d_lu, double *norms, int perturb,
                      hipStream_t st)
{
    if (p->batch_grid_lev == 0) return;
    launch::il_values(p->R, p->F, d_ax, p->d_il, p->d_il_bits, norms, p->nnz, p->n, batch, perturb, st);
    for (int l = 0; l < p->batch_grid_lev; ++l)
        launch::factor_grid_il(p->F, p->d_il, norms, l, p->grid_waves[l], batch, perturb, st);
    launch::il_to_rows(p->d_il, d_lu, p->nnz, batch, st);
}

}  // namespace

extern "C" glu_status glu_batch_solve(glu_plan *p, int batch, const double *d_ax, const double *d_b, double *d_x,
                                      float *d_lu, double tol, int maxit, int32_t *d_iters, double *d_eta,
                                      unsigned flags, void *stream)
{
    if (!p || batch <= 0 || !d_ax || !d_b || !d_x || !d_lu || !d_iters || !d_eta || maxit <= 0)
        return fail(GLU_ERR_ARGUMENT, "bad argument");
    if (!p->has_refine) return fail(GLU_ERR_ARGUMENT, "plan has no analysis");
    glu_status s = ensure_batch(p, batch);
    if (s == GLU_OK) s = ensure_il(p, batch);
    if (s != GLU_OK) return s;
    const size_t cap = launch::enable_lds();
    const int mode = sweep_mode(p->n, cap);
    const int perturb = (int)(flags & 1u);
    hipStream_t st = static_cast<hipStream_t>(stream);
    batch_grid_steps(p, batch, d_ax, d_lu, p->d_bnorms, perturb, st);
    launch::batch_same(p->d_desc, batch, d_ax, d_b, d_x, d_lu, p->d_blucsr, p->d_bt32, p->d_br64, p->d_bnorms,
                       p->d_bkry, d_iters, d_eta, tol, maxit, perturb, p->fused_threads, mode,
                       sizeof(float) * std::max(p->win_nslot + kWinExtra, p->copy_range), launch::batch_lds_bytes(mode, p->n),
                       p->batch_grid_lev, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("batch launch: ") + hipGetErrorString(e));
    return GLU_OK;
}

extern "C" glu_status glu_batch_factor(glu_plan *p, int batch, const double *d_ax, float *d_lu, unsigned flags,
                                       void *stream)
{
    if (!p || batch <= 0 || !d_ax || !d_lu) return fail(GLU_ERR_ARGUMENT, "bad argument");
    if (!p->has_refine) return fail(GLU_ERR_ARGUMENT, "plan has no analysis");
    (void)launch::enable_lds();
    const int perturb = (int)(flags & 1u);
    hipStream_t st = static_cast<hipStream_t>(stream);
    glu_status s = ensure_il(p, batch);
    if (s != GLU_OK) return s;
    batch_grid_steps(p, batch, d_ax, d_lu, p->d_fnorms, perturb, st);
    launch::batch_factor(p->d_desc, batch, d_ax, d_lu, p->d_fnorms, perturb, p->fused_threads,
                         sizeof(float) * (p->win_nslot + kWinExtra), p->batch_grid_lev, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("batch factor launch: ") + hipGetErrorString(e));
    return GLU_OK;
}

extern "C" glu_status glu_abft_sums(glu_plan *p, int batch, const float *d_val, float *d_cca, void *stream)
{
    if (!p || batch <= 0 || !d_val || !d_cca) return fail(GLU_ERR_ARGUMENT, "bad argument");
    if (batch > 65535) return fail(GLU_ERR_ARGUMENT, "batch above 65535");
    launch::abft_cca(p->F, d_val, d_cca, batch, static_cast<hipStream_t>(stream));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("abft launch: ") + hipGetErrorString(e));
    return GLU_OK;
}

extern "C" glu_status glu_abft_check(glu_plan *p, int batch, const float *d_lu, const float *d_cca, float tol,
                                     int32_t *d_first_bad, float *d_max_diff, void *stream)
{
    if (!p || batch <= 0 || !d_lu || !d_cca || !d_first_bad || !d_max_diff || !(tol >= 0.f))
        return fail(GLU_ERR_ARGUMENT, "bad argument");
    if (batch > 65535) return fail(GLU_ERR_ARGUMENT, "batch above 65535");
    if (batch > p->abft_cap) {
        if (p->d_abft) (void)hipFree(p->d_abft);
        p->d_abft = nullptr;
        p->abft_cap = 0;
        HIP_TRY(hipMalloc(&p->d_abft, sizeof(float) * (size_t)p->n * batch));
        p->abft_cap = batch;
    }
    launch::abft_check(p->F, p->d_rowidx, p->d_diag, d_lu, d_cca, p->d_abft, tol, d_first_bad, d_max_diff, batch,
                       static_cast<hipStream_t>(stream));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("abft launch: ") + hipGetErrorString(e));
    return GLU_OK;
}

// ---------------------------------------------------------------------------
// uneven groups
// ---------------------------------------------------------------------------

struct MatIOHost {            // mirrors the device-side MatIO layout
    const double *ax;
    const double *b;
    double *x;
    float *lu;
    float *t32;
    double *r64;
    float *lucsr;
    double *norms;
    double *kry;
    int32_t *iters;
    double *eta;
};

struct glu_group {
    std::vector<glu_plan *> plans;
    MatDesc *d_descs = nullptr;
    MatIOHost *d_ios = nullptr;
    uint32_t *d_order = nullptr;
    char *d_items = nullptr;       // the leading launches' items and phases, l0
    int32_t *d_l0 = nullptr;       // by member: steps its phases cover
    GroupLaunch lead[kMaxGroupSplit + 1];   // by the number of members split off
    float *d_t32 = nullptr;
    double *d_r64 = nullptr;
    float *d_lucsr = nullptr;
    float *d_prod = nullptr;       // the phases' products, a range a member
    double *d_norms = nullptr;
    double *d_kry = nullptr;
    std::vector<size_t> voff;   // per-matrix offset into d_r64
    std::vector<size_t> toff;   // per-matrix offset into d_t32
    std::vector<size_t> koff;   // per-matrix offset into d_kry (~0: plain refinement)
    std::vector<size_t> foff;   // per-matrix offset into d_lucsr
    std::vector<uint32_t> order;   // members, heaviest first (d_order)
    int threads = kDefaultFusedThreads;
    int split_req = -1;            // heaviest members on the single-matrix path (-1: automatic)
    hipStream_t aux[kMaxGroupSplit] = {};
    hipEvent_t ev_in = nullptr, ev_aux[kMaxGroupSplit] = {};
    ~glu_group()
    {
        for (int j = 0; j < kMaxGroupSplit; ++j) {
            if (aux[j]) (void)hipStreamDestroy(aux[j]);
            if (ev_aux[j]) (void)hipEventDestroy(ev_aux[j]);
        }
        if (ev_in) (void)hipEventDestroy(ev_in);
        if (d_lucsr) (void)hipFree(d_lucsr);
        if (d_prod) (void)hipFree(d_prod);
        if (d_norms) (void)hipFree(d_norms);
        if (d_kry) (void)hipFree(d_kry);
        if (d_descs) (void)hipFree(d_descs);
        if (d_ios) (void)hipFree(d_ios);
        if (d_order) (void)hipFree(d_order);
        if (d_items) (void)hipFree(d_items);
        if (d_t32) (void)hipFree(d_t32);
        if (d_r64) (void)hipFree(d_r64);
    }
};

namespace {

glu_status group_create(glu_plan *const *plans, int count, glu_group **out)
{
    if (!plans || count <= 0 || !out) return fail(GLU_ERR_ARGUMENT, "bad argument");
    *out = nullptr;
    if (launch::matio_size() != sizeof(MatIOHost)) return fail(GLU_ERR_GENERAL, "MatIO layout mismatch");
    std::unique_ptr<glu_group> g(new glu_group());
    std::vector<MatDesc> descs(count);
    std::vector<std::pair<int64_t, uint32_t>> work(count);
    size_t vtot = 0, ttot = 0, ftot = 0, ktot = 0;
    for (int i = 0; i < count; ++i) {
        glu_plan *p = plans[i];
        if (!p || !p->has_refine) return fail(GLU_ERR_ARGUMENT, "every plan must come from an analysis");
        g->plans.push_back(p);
        descs[i].f = p->F;
        descs[i].s = p->S;
        descs[i].r = p->R;
        descs[i].n = p->n;
        descs[i].nnz = p->nnz;
        descs[i].krylov = (uint32_t)p->krylov;
        descs[i].a_kmax = p->a_kmax;
        g->koff.push_back(p->krylov ? ktot : ~(size_t)0);
        ktot += (3 * (size_t)p->krylov + 1) * p->n * (p->krylov != 0);
        g->voff.push_back(vtot);
        vtot += p->n;
        g->toff.push_back(ttot);
        ttot += p->t32_len;
        g->foff.push_back(ftot);   // (whole lines: the sweeps load 16 bytes a lane)
        ftot += ((size_t)p->df_nval + 63) & ~(size_t)63;
        g->threads = std::max(g->threads, p->fused_threads);
        // heaviest first: levels dominate the latency, updates the work
        work[i] = {-(int64_t)(p->num_lev + p->tri[0].lvl_ptr.size() + p->tri[1].lvl_ptr.size()) * 64 - p->updates,
                   (uint32_t)i};
    }
    std::sort(work.begin(), work.end());
    std::vector<uint32_t> &order = g->order;
    order.resize(count);
    for (int i = 0; i < count; ++i) order[i] = work[i].second;
    HIP_TRY(hipMalloc(&g->d_descs, sizeof(MatDesc) * count));
    HIP_TRY(hipMalloc(&g->d_ios, sizeof(MatIOHost) * count));
    HIP_TRY(hipMalloc(&g->d_order, sizeof(uint32_t) * count));
    HIP_TRY(hipMalloc(&g->d_t32, sizeof(float) * ttot));
    HIP_TRY(hipMalloc(&g->d_r64, sizeof(double) * vtot));
    HIP_TRY(hipMalloc(&g->d_lucsr, sizeof(float) * ftot));
    HIP_TRY(hipMalloc(&g->d_norms, 2 * sizeof(double) * count));
    if (ktot) HIP_TRY(hipMalloc(&g->d_kry, sizeof(double) * ktot));
    // The leading launches (for every number of members that may be split
    // off): blocks of values, then bins (those with the most work first) and
    // assembly blocks of each phase round.  A member's products go to a range
    // of its own: a plan may be several members, and is in use outside the
    // group (a split-off member's factorization, glu_factor on another stream).
    {
        std::vector<int32_t> l0(count, 0);
        std::vector<size_t> poff(count, 0);
        size_t ptot = 0;
        for (int i = 0; i < count; ++i) {
            l0[i] = plans[i]->phases.size() <= kGroupRounds ? plans[i]->phase_lev : 0;
            poff[i] = ptot;
            if (l0[i]) ptot += (plans[i]->phase_out + 63) & ~(size_t)63;
        }
        if (ptot) HIP_TRY(hipMalloc(&g->d_prod, sizeof(float) * ptot));
        std::vector<PhaseDev> ph[kGroupRounds];
        for (uint32_t r = 0; r < kGroupRounds; ++r) {
            ph[r].resize(count);
            for (int i = 0; i < count; ++i)
                if (l0[i] && r < plans[i]->phases.size()) {
                    ph[r][i] = plans[i]->phases[r];
                    ph[r][i].out = g->d_prod + poff[i];
                }
        }
        std::vector<uint2> items;
        size_t first[kMaxGroupSplit + 1][1 + 2 * kGroupRounds];
        for (int sp = 0; sp <= kMaxGroupSplit; ++sp) {
            GroupLaunch &G = g->lead[sp];
            G.threads = kPhaseWaves * 64;
            std::vector<uint32_t> mem(order.begin() + std::min(sp, count), order.end());
            first[sp][0] = items.size();
            for (uint32_t m : mem)
                for (uint32_t b = 0; l0[m] && b * (uint64_t)launch::group_values() < plans[m]->nnz; ++b)
                    items.push_back(make_uint2(m, b));
            G.nvalues = (uint32_t)(items.size() - first[sp][0]);
            for (uint32_t r = 0; r < kGroupRounds; ++r) {
                first[sp][1 + 2 * r] = items.size();
                for (uint32_t m : mem)
                    if (l0[m] && r < plans[m]->phases.size()) {
                        G.rounds = std::max(G.rounds, r + 1);
                        G.nslot[r] = std::max(G.nslot[r], ph[r][m].nslot);
                        for (uint32_t b = 0; b < ph[r][m].nbin; ++b) items.push_back(make_uint2(m, b));
                    }
                std::stable_sort(items.begin() + first[sp][1 + 2 * r], items.end(), [&](const uint2 &a, const uint2 &b) {
                    return plans[a.x]->phase_work[r][a.y] > plans[b.x]->phase_work[r][b.y];
                });
                G.nbin[r] = (uint32_t)(items.size() - first[sp][1 + 2 * r]);
                first[sp][2 + 2 * r] = items.size();
                for (uint32_t m : mem)
                    if (l0[m] && r < plans[m]->phases.size())
                        for (uint32_t w = 0; w < ph[r][m].nwav + ph[r][m].ngrp; w += 4) items.push_back(make_uint2(m, w));
                G.nasm[r] = (uint32_t)(items.size() - first[sp][2 + 2 * r]);
            }
        }
        const size_t o_items = sizeof(PhaseDev) * count * kGroupRounds, o_l0 = o_items + sizeof(uint2) * items.size();
        HIP_TRY(hipMalloc(&g->d_items, o_l0 + sizeof(int32_t) * count));
        for (uint32_t r = 0; r < kGroupRounds; ++r)
            HIP_TRY(hipMemcpy(g->d_items + sizeof(PhaseDev) * count * r, ph[r].data(), sizeof(PhaseDev) * count,
                              hipMemcpyHostToDevice));
        if (!items.empty())
            HIP_TRY(hipMemcpy(g->d_items + o_items, items.data(), sizeof(uint2) * items.size(), hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(g->d_items + o_l0, l0.data(), sizeof(int32_t) * count, hipMemcpyHostToDevice));
        g->d_l0 = reinterpret_cast<int32_t *>(g->d_items + o_l0);
        const uint2 *it = reinterpret_cast<const uint2 *>(g->d_items + o_items);
        for (int sp = 0; sp <= kMaxGroupSplit; ++sp) {
            GroupLaunch &G = g->lead[sp];
            G.values = it + first[sp][0];
            for (uint32_t r = 0; r < kGroupRounds; ++r) {
                G.phase[r] = reinterpret_cast<const PhaseDev *>(g->d_items) + (size_t)count * r;
                G.bins[r] = it + first[sp][1 + 2 * r];
                G.asms[r] = it + first[sp][2 + 2 * r];
            }
        }
    }
    HIP_TRY(hipMemcpy(g->d_descs, descs.data(), sizeof(MatDesc) * count, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(g->d_order, order.data(), sizeof(uint32_t) * count, hipMemcpyHostToDevice));
    *out = g.release();
    return GLU_OK;
}

}  // namespace

extern "C" glu_status glu_group_create(glu_plan *const *plans, int count, glu_group **out)
{
    return guarded([&] { return group_create(plans, count, out); });
}

extern "C" void glu_group_destroy(glu_group *g) { delete g; }

extern "C" glu_status glu_group_set_split(glu_group *g, int count)
{
    if (!g || count < -1 || count > kMaxGroupSplit) return fail(GLU_ERR_ARGUMENT, "split count must be -1..2");
    g->split_req = count;
    return GLU_OK;
}

namespace {

glu_status group_solve(glu_group *g, const double *const *d_ax, const double *const *d_b, double *const *d_x,
                       float *const *d_lu, double tol, int maxit, int32_t *d_iters, double *d_eta, unsigned flags,
                       void *stream)
{
    if (!g || !d_ax || !d_b || !d_x || !d_lu || !d_iters || !d_eta || maxit <= 0)
        return fail(GLU_ERR_ARGUMENT, "bad argument");
    const int count = (int)g->plans.size();
    std::vector<MatIOHost> ios(count);
    for (int i = 0; i < count; ++i) {
        if (!d_ax[i] || !d_b[i] || !d_x[i] || !d_lu[i]) return fail(GLU_ERR_ARGUMENT, "null matrix pointer");
        ios[i] = MatIOHost{d_ax[i], d_b[i], d_x[i], d_lu[i], g->d_t32 + g->toff[i], g->d_r64 + g->voff[i],
                           g->d_lucsr + g->foff[i], g->d_norms + 2 * i,
                           g->koff[i] == ~(size_t)0 ? nullptr : g->d_kry + g->koff[i], d_iters + i, d_eta + i};
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    HIP_TRY(hipMemcpyAsync(g->d_ios, ios.data(), sizeof(MatIOHost) * count, hipMemcpyHostToDevice, st));
    const size_t cap = launch::enable_lds();
    const int perturb = (int)(flags & 1u);
    // The heaviest members (as many as asked; automatic: one in a group of
    // four or more) run on the single-matrix path on streams of their own,
    // alongside the fused launch of the rest: the grid factorization on the
    // CUs the fused launch leaves idle, then the one-workgroup refinement,
    // the same kernel the fused launch runs (same workgroup size and restart
    // length), so the results are the same bits.  Only members whose
    // refinement keeps its vector in LDS qualify, and one member of a plan
    // (that path works in the plan's scratch; the fused launch in the group's).
    int want = g->split_req >= 0 ? g->split_req : (count >= 4 ? 1 : 0);
    want = std::min(want, count - 1);
    int nsplit = 0;
    const auto apart = [&](const glu_plan *p) {   // not a split-off member's plan
        for (int j = 0; j < nsplit; ++j)
            if (g->plans[g->order[j]] == p) return false;
        return true;
    };
    while (nsplit < want && sweep_mode(g->plans[g->order[nsplit]]->n, cap) == 2 && apart(g->plans[g->order[nsplit]]))
        ++nsplit;
    if (nsplit > 0) {
        if (!g->ev_in) HIP_TRY(hipEventCreateWithFlags(&g->ev_in, hipEventDisableTiming));
        HIP_TRY(hipEventRecord(g->ev_in, st));
    }
    for (int j = 0; j < nsplit; ++j) {
        const uint32_t m = g->order[j];
        glu_plan *p = g->plans[m];
        glu_status s = ensure_batch(p, 1);
        if (s != GLU_OK) return s;
        if (!g->aux[j]) HIP_TRY(hipStreamCreateWithFlags(&g->aux[j], hipStreamNonBlocking));
        if (!g->ev_aux[j]) HIP_TRY(hipEventCreateWithFlags(&g->ev_aux[j], hipEventDisableTiming));
        hipStream_t as = g->aux[j];
        HIP_TRY(hipStreamWaitEvent(as, g->ev_in, 0));
        launch::refresh(p->R, d_ax[m], d_lu[m], p->nnz, 1, as);
        s = run_factor(p, d_lu[m], perturb, as);
        if (s != GLU_OK) return s;
        launch::refine_one(p->d_desc, p->S.df_src, p->df_nval, d_ax[m], d_b[m], d_x[m], d_lu[m], p->d_blucsr, p->d_bt32,
                           p->d_br64, p->d_bnorms, p->d_bkry, d_iters + m, d_eta + m, tol, maxit, g->threads,
                           launch::batch_lds_bytes(2, p->n), 0, as);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventRecord(g->ev_aux[j], as));
    }
    size_t nmax = 0, tmax = 0;
    for (int i = nsplit; i < count; ++i) {
        const glu_plan *p = g->plans[g->order[i]];
        nmax = std::max<size_t>(nmax, p->n);
        tmax = std::max<size_t>(tmax, sizeof(float) * (p->win_nslot + kWinExtra));
    }
    const int mode = sweep_mode((uint32_t)nmax, cap);
    // ready bits only for the largest order: each matrix whose vector fits
    // keeps it in LDS too (the launch's LDS: the largest such need)
    size_t ref_lds = launch::batch_lds_bytes(mode, (uint32_t)nmax);
    if (mode == 1)
        for (int i = nsplit; i < count; ++i) {
            const glu_plan *p = g->plans[g->order[i]];
            const size_t full = launch::batch_lds_bytes(2, p->n);
            ref_lds = std::max(ref_lds, full <= cap ? full : launch::batch_lds_bytes(1, p->n));
        }
    launch::group_phases(g->d_descs, g->d_ios, g->d_order + nsplit, count - nsplit, g->d_l0, g->lead[nsplit], perturb,
                         g->threads, st);
    launch::batch_group(g->d_descs, g->d_ios, g->d_order + nsplit, count - nsplit, g->d_l0, tol, maxit, perturb,
                        g->threads, mode, tmax, ref_lds, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GLU_ERR_DEVICE, std::string("group launch: ") + hipGetErrorString(e));
    for (int j = 0; j < nsplit; ++j) HIP_TRY(hipStreamWaitEvent(st, g->ev_aux[j], 0));
    // ios is read by the kernel from device memory; the host copy may go.
    HIP_TRY(hipStreamSynchronize(st));
    return GLU_OK;
}

}  // namespace

extern "C" glu_status glu_group_solve(glu_group *g, const double *const *d_ax, const double *const *d_b,
                                      double *const *d_x, float *const *d_lu, double tol, int maxit,
                                      int32_t *d_iters, double *d_eta, unsigned flags, void *stream)
{
    return guarded([&] { return group_solve(g, d_ax, d_b, d_x, d_lu, tol, maxit, d_iters, d_eta, flags, stream); });
}
