/*
 * rchol.h -- C ABI of the MI355X randomized-Cholesky preconditioner + PCG.
 *
 * One handle owns one HIP stream and all device memory it allocates.  Handles
 * are not thread-safe: use one host thread per handle.  Every entry point
 * returns RC_OK (0) or a negative rc_status; rc_last_error() gives the text.
 * Nothing in the library calls exit() or assert().
 *
 * The reference exposes this path as two CLIs and two C++ templates; each
 * entry point below names the reference interface it replaces:
 *   driver.cu:2148-2157 / driver_physics.cu:2120-2129   GPU CLI
 *     `driver <mtx> <num_blocks> <check_solve> <tol>`
 *   driver_local.cpp:1325-1347                           CPU CLI
 *     `driver <mtx> <threads> <out_prefix> [1]`
 *   driver.cu:1551-1552   factorization_driver<int,double>(processor, num_blocks, check_solve, tol)
 *   solver.hpp:236-238    prepare_and_solve(laplacian, rowptr, val, colind, diag, tol, physics, nnz, removal)
 *   pre_process.hpp:322-417  sparse_matrix_processor<int,double>(path)
 *   write_graph.jl:43-95, 328-414  orderings and the SDDM ground append (offline Julia)
 */
#ifndef RCHOL_H
#define RCHOL_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct rc_handle_s *rc_handle_t;

typedef enum {
    RC_OK = 0,
    RC_ERR_ARG = -1,          /* bad argument                                    */
    RC_ERR_IO = -2,           /* file could not be opened / written              */
    RC_ERR_FORMAT = -3,       /* malformed Matrix Market / factor dump           */
    RC_ERR_NOT_DOMINANT = -4, /* SDDM input is not diagonally dominant           */
    RC_ERR_STATE = -5,        /* call out of order (e.g. solve before factor)    */
    RC_ERR_HIP = -6,          /* HIP runtime error                               */
    RC_ERR_POOL = -7,         /* fill/output pool exhausted even after regrowth  */
    RC_ERR_TIMEOUT = -8,      /* a device-side bounded wait expired              */
    RC_ERR_BREAKDOWN = -9,    /* PCG breakdown: p'Ap <= 0 or not finite          */
    RC_ERR_NO_DEVICE = -10,   /* no HIP device / library built without one       */
    RC_ERR_NOMEM = -11,       /* host or device allocation failed                */
    RC_ERR_NOT_SYMMETRIC = -12,/* Laplacian pattern or values not symmetric      */
    RC_ERR_MAXIT = -13        /* PCG hit maxit before the stop rule held (info)  */
} rc_status;

/* Input kinds of rc_load_mtx / rc_set_csc. */
enum {
    RC_INPUT_LAPLACIAN = 0,  /* graph Laplacian or adjacency (driver.cu)                        */
    RC_INPUT_GROUNDED = 1,   /* Laplacian whose LAST vertex is an appended ground; factor it,
                                then drop the ground from L and A (driver_physics.cu:1945-2090) */
    RC_INPUT_SDDM = 2        /* raw SDDM; the ground vertex is appended after ordering
                                (write_graph.jl:367-383), then handled as GROUNDED              */
};

/* Orderings (write_graph.jl:46-78, 333-365).  LEARNED uses the graph network
 * when weights are loaded and falls back to NNZ_SORT otherwise.  ND is nested
 * dissection (write_graph.jl:71-75 uses Metis; this one bisects by BFS level
 * structures: both halves first, the separator last, recursively). */
enum { RC_ORDER_AS_IS = 0, RC_ORDER_NNZ_SORT = 1, RC_ORDER_RANDOM = 2, RC_ORDER_AMD = 3, RC_ORDER_LEARNED = 4,
       RC_ORDER_ND = 5 };

/* PCG stop rules: REFERENCE = sqrt(r'z / r0'z0) <= tol (solver.hpp:536);
 * TRUE_RESIDUAL = ||r_k|| / ||b|| <= tol on the recurrence residual. */
enum { RC_STOP_REFERENCE = 0, RC_STOP_TRUE_RESIDUAL = 1 };

/* Right-hand sides generated by the library (solver.hpp:29-61, 419-444). */
enum {
    RC_RHS_ZERO_SUM_UNIFORM = 0, /* U[0,1) from std::mt19937(seed), minus the mean (reference)   */
    RC_RHS_NORMAL = 1,           /* N(0,1) by Box-Muller over Philox4x32-10(seed)                */
    RC_RHS_NORMAL_PROJECTED = 2  /* N(0,1), mean removed per connected component                 */
};

typedef struct {
    int device;              /* HIP device ordinal (default 0); -1 = host-only handle:
                                input, ordering, RHS and rc_get_prepared_csc work, every
                                device entry point returns RC_ERR_NO_DEVICE             */
    uint64_t seed;           /* elimination sampling seed (default 1)                   */
    int num_blocks;          /* elimination workgroups; 0 = sized to occupancy. The
                                reference's argv[2] (driver.cu:2157)                    */
    int factor_precision;    /* 64 (default) or 32: factor storage + triangular solves  */
    int stop_rule;           /* RC_STOP_REFERENCE (default)                             */
    int maxit;               /* default 300 (solver.hpp:483)                            */
    double pool_factor;      /* initial fill-pool capacity / nnz(lower A); default 4.0   */
    int verbose;             /* 1: print reference-style progress lines to stdout       */
    int host_threads;        /* host threads of the input path (Matrix Market parse,
                                orderings); 0 = all hardware threads. The reference
                                CPU driver's <threads> (driver_local.cpp:1330)          */
} rc_options;

typedef struct {
    int64_t n;               /* columns factored (incl. ground)                         */
    int64_t nnz_lower;       /* strict-lower nnz of the factored Laplacian              */
    int64_t nnz_factor;      /* sum_k (d_k + 1): the reference's "factor nnz"           */
    int64_t fills;           /* sum_k max(d_k - 1, 0)                                   */
    int64_t max_degree;      /* max_k d_k                                               */
    int32_t nlevels;         /* depth of the triangular-solve DAG                       */
    int32_t zero_pivots;     /* D_k == 0 (one per connected component)                  */
    double factor_ms;        /* elimination kernel (hipEvent)                           */
    double assemble_ms;      /* compaction, transpose, level analysis (hipEvent)        */
    double bytes_factor;     /* algorithmic bytes of the elimination                    */
    int32_t pool_regrowths;  /* times the pools were regrown and the kernel rerun       */
    double prepare_ms;       /* ordering applied, ground append/trim, lower slice and
                                dependency counts (device), when this factor did it;
                                0 when the prepared system was reused                  */
} rc_factor_stats;

typedef struct {
    int32_t iterations;
    int32_t converged;       /* 1 if the stop rule held before maxit                    */
    double rel_res_true;     /* ||A x - b|| / ||b|| (solver.hpp:549-569)                */
    double rel_res_precond;  /* sqrt(r'z / r0'z0) at exit                               */
    double pcg_ms;           /* PCG loop (hipEvent)                                     */
    double setup_ms;         /* per-solve setup before the loop                         */
    double err_vs_oracle;    /* ||x - x_ref||_A / ||x_ref||_A when a reference x is set;
                                -1 otherwise                                            */
} rc_solve_stats;

/* ---------------- handle ---------------- */
void rc_default_options(rc_options *opt);
int rc_create(rc_handle_t *h, const rc_options *opt);
int rc_destroy(rc_handle_t h);
const char *rc_last_error(rc_handle_t h);
const char *rc_status_string(int status);

/* ---------------- input (pre_process.hpp:322-417) ---------------- */
/* Matrix Market coordinate real/integer/pattern, general or symmetric. */
int rc_load_mtx(rc_handle_t h, const char *path, int input_kind);
/* Triplets as read from a Matrix Market file (0-based); copied in. */
int rc_set_triplets(rc_handle_t h, int n, int64_t m, const int *rows, const int *cols,
                    const double *vals, int input_kind);
/* Size of the loaded system as the user sees it (ground excluded). */
int rc_get_size(rc_handle_t h, int64_t *n, int64_t *nnz);

/* ---------------- ordering (write_graph.jl) ---------------- */
int rc_order(rc_handle_t h, int method, uint64_t seed);
/* perm[new] = old, length = rc_get_size n. */
int rc_get_permutation(rc_handle_t h, int *perm);
/* Explicit ordering perm[new] = old over the loaded vertices (ground
 * excluded) -- the reference reads pre-permuted files; this takes the
 * permutation instead.  Used by the ordering network's trainer. */
int rc_set_permutation(rc_handle_t h, const int *perm);

/* ---------------- row locality of the sweeps (no reference counterpart) ----
 * The triangular sweeps store each level's rows contiguously; inside a level
 * they follow the input numbering (RC_LOCALITY_INPUT, default) or a recursive
 * bisection order of the input graph (RC_LOCALITY_BISECTION: every subgraph of
 * the bisection, a compact region, holds contiguous positions), which puts the
 * dependencies that one chunk of rows gathers into fewer cache lines; the SpMV
 * then visits its 64-row tiles in the bisection order of their first rows.  The
 * order depends on the graph only: it is computed on the host once per loaded
 * matrix (at rc_order / rc_set_permutation, or here if a matrix is ordered)
 * and changes neither the factor nor the iterates beyond summation order.
 * In a batch every system is bisected on its own and keeps its row range.
 * rc_get_locality writes rank[user vertex] (the input numbering when off) and
 * the seconds the last bisection took. */
enum { RC_LOCALITY_INPUT = 0, RC_LOCALITY_BISECTION = 1 };
int rc_set_locality(rc_handle_t h, int mode);
int rc_get_locality(rc_handle_t h, int *rank, double *seconds);

/* ---------------- ordering network (no reference counterpart) ----------------
 * Three message-passing layers (hidden 64, bfloat16 weights, FP32 accumulate)
 * on (log degree, log weighted degree); RC_ORDER_LEARNED eliminates vertices
 * in descending score.  Weights: float32, rc_gnn_weight_count() values. */
int64_t rc_gnn_weight_count(void);
int rc_set_gnn_weights(rc_handle_t h, const float *w, int64_t count);
/* Scores of the loaded vertices (GPU forward pass). */
int rc_gnn_scores(rc_handle_t h, const float *w, float *scores);
/* dw = d(sum_v dscores[v] * score[v]) / dw (GPU forward + backward pass). */
int rc_gnn_gradient(rc_handle_t h, const float *w, const float *dscores, float *dw);

/* The ordered (and, for SDDM input, ground-appended) Laplacian that rc_factor
 * eliminates, as CSC (both triangles, rows sorted).  This is the matrix the
 * reference's offline preprocessing writes (write_graph.jl:80-91, 386-398:
 * mmwrite of G_new).  Query sizes with NULL arrays.  Works on host-only
 * handles (device = -1). */
int rc_get_prepared_csc(rc_handle_t h, int64_t *n, int64_t *nnz, int64_t *colptr, int *rowind, double *val);
int rc_write_prepared_mtx(rc_handle_t h, const char *path);

/* ---------------- factor (driver.cu:1551-1897) ---------------- */
int rc_factor(rc_handle_t h, rc_factor_stats *st);
/* Incomplete Cholesky IC(0) of the same prepared matrix instead of the
 * randomized elimination (no reference function: the context preconditioner
 * of the reference's comparisons, MATLAB ichol in experiment/ichol_*_test.m).
 * L D L^T with L on the pattern of the lower triangle; every solve entry
 * point then runs with it. */
int rc_factor_ic0(rc_handle_t h, rc_factor_stats *st);
/* Factor as the reference's CSR of L^T with the unit diagonal first in every
 * row (driver.cu:1310-1548, driver_local.cpp:881-956), values -w/S, in the
 * solve numbering (ground removed for grounded inputs).  Query sizes with
 * NULL arrays. */
int rc_get_factor(rc_handle_t h, int64_t *n, int64_t *nnz, int64_t *rowptr, int *colind,
                  double *val, double *diag);
/* <prefix>l_sol.mtx + <prefix>sol_diag.txt (driver_local.cpp:958-988). */
int rc_dump_factor(rc_handle_t h, const char *prefix);
/* Read a factor dump back and use it as the preconditioner
 * (experiment/independent_cg.cpp:277-332). */
int rc_load_factor(rc_handle_t h, const char *prefix);

/* ---------------- solve (solver.hpp:236-593) ---------------- */
/* Change the PCG stop rule (RC_STOP_*) and, when maxit > 0, the iteration
 * limit of later solves on this handle (solver.hpp:483, 493, 536); the
 * factor is kept. */
int rc_set_solve_options(rc_handle_t h, int stop_rule, int maxit);
/* b, x in the numbering of the loaded matrix (ground excluded). */
int rc_solve(rc_handle_t h, const double *b, double *x, double tol, rc_solve_stats *st);
/* k <= 64 right-hand sides sharing the factor (no counterpart in the
 * reference, which solves one RHS per run; for many right-hand sides on one factor).
 * B and X are column-major n x k in the loaded numbering; st has k entries.
 * Every right-hand side runs its own PCG (own scalars and stop test); a
 * converged one is frozen while the others continue. */
int rc_solve_multi(rc_handle_t h, int k, const double *B, double *X, double tol, rc_solve_stats *st);
/* Resident form of rc_solve_multi (used by the benchmark so that the RHS are
 * in HBM before the timed region): rc_set_rhs_multi uploads B (column-major,
 * n x k), rc_solve_multi_resident runs the k PCGs on them (st has k entries),
 * rc_get_solution_multi copies X back (column-major). */
int rc_set_rhs_multi(rc_handle_t h, int k, const double *B);
int rc_solve_multi_resident(rc_handle_t h, double tol, rc_solve_stats *st);
int rc_get_solution_multi(rc_handle_t h, double *X);
/* Per-right-hand-side statistics of the last multi-RHS solve (k entries). */
int rc_get_multi_stats(rc_handle_t h, rc_solve_stats *st);

/* Several resident solves in one launch sequence (no counterpart in the
 * reference, which solves one system per process run): handles[i] holds a
 * factored system and a resident right-hand side -- rc_set_rhs (one system,
 * or one RHS per system of a batch) or rc_set_rhs_multi, whichever was called
 * last.  Every member's PCG runs with its own scalars and stop test; two
 * iterations of every member are captured into one hipGraph on the first
 * handle's stream and launched until all members are done, so a large
 * multi-RHS system and a batch of small Laplacians advance together.  st has
 * `count` entries (the member's worst right-hand side / system); per-RHS and
 * per-system details via rc_get_multi_stats / rc_get_batch_stats; solutions
 * via rc_get_solution / rc_get_solution_multi.  All handles on one device;
 * errors are reported on handles[0]. */
int rc_solve_group(int count, const rc_handle_t *handles, double tol, rc_solve_stats *st);
/* Generate a right-hand side of the given kind in the loaded numbering. */
int rc_make_rhs(rc_handle_t h, int kind, uint64_t seed, double *b);
/* Optional reference solution for err_vs_oracle (copied in; NULL clears). */
int rc_set_reference_solution(rc_handle_t h, const double *x_ref);

/* Resident-input solve (no counterpart in the reference; used by the
 * benchmark so that the timed region starts with the RHS already in HBM):
 * rc_set_rhs uploads and permutes b, rc_solve_resident runs the PCG on it,
 * rc_get_solution copies x back in the loaded numbering. */
int rc_set_rhs(rc_handle_t h, const double *b);
int rc_solve_resident(rc_handle_t h, double tol, rc_solve_stats *st);
int rc_get_solution(rc_handle_t h, double *x);

/* Allocation-free solve (no counterpart in the reference: for callers that
 * cannot allocate device memory -- code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc).  Same PCG as rc_solve on a
 * factored single system, but b_dev and x_dev are DEVICE pointers (n doubles
 * each, the loaded numbering) and every work vector, scalar and counter of the
 * solve lives in a fixed workspace of 64 MiB per GPU (a __device__ array held
 * until the process ends), so nothing is allocated: systems needing more
 * (about 1.0 M rows with an FP64 factor, 1.2 M with FP32) return RC_ERR_ARG.
 * Batches return RC_ERR_ARG.  All calls on one GPU share that workspace and
 * it keeps the last call's contents: calls that overlap on one GPU (two host
 * threads, or two handles on one device used concurrently) race. */
int rc_solve_noalloc(rc_handle_t h, const double *b_dev, double *x_dev, double tol, rc_solve_stats *st);

/* ---------------- batched systems (no reference counterpart) ----------------
 * The reference factors and solves one Laplacian per process run (driver.cu:
 * 2148-2157, one .mtx per call of the test scripts); these entry points take
 * nsys independent Laplacians at once.  System s has sys_n[s] vertices and
 * sys_m[s] triplets with system-local 0-based indices; the triplet arrays are
 * the systems' arrays concatenated.  The batch is held as one block-diagonal
 * Laplacian (rows of system s at offsets[s] .. offsets[s+1]-1), so rc_order,
 * rc_factor, rc_make_rhs, rc_set_rhs, rc_get_solution work on it unchanged;
 * rc_solve / rc_solve_resident / rc_solve_batch run one PCG per system (own
 * alpha, beta, r'z, stop test and iteration count) in shared launches. */
int rc_set_batch(rc_handle_t h, int nsys, const int *sys_n, const int64_t *sys_m,
                 const int *rows, const int *cols, const double *vals);
/* Number of systems (1 for a handle without a batch) and offsets[nsys+1]. */
int rc_get_batch(rc_handle_t h, int *nsys, int64_t *offsets);
/* Solve with one RHS per system (b, x in the block-diagonal numbering);
 * per_system has nsys entries (may be NULL). */
int rc_solve_batch(rc_handle_t h, const double *b, double *x, double tol, rc_solve_stats *per_system);
/* Per-system statistics of the last solve of a batch (nsys entries). */
int rc_get_batch_stats(rc_handle_t h, rc_solve_stats *per_system);

/* ---------------- measurement ---------------- */
/* Kernel ids for rc_time_kernel. */
enum { RC_KERNEL_SPMV = 0, RC_KERNEL_TRSV_FWD = 1, RC_KERNEL_TRSV_BWD = 2, RC_KERNEL_PCG_ITER = 3,
       RC_KERNEL_COPY = 4, RC_KERNEL_MULTI_SPMM = 5, RC_KERNEL_MULTI_TRSV_FWD = 6, RC_KERNEL_MULTI_TRSV_BWD = 7 };
/* Launch one PCG kernel `reps` times on the handle's stream between two
 * hipEvents and return the mean ms per launch and its algorithmic bytes.
 * RC_KERNEL_COPY is a plain 1 GiB device-to-device copy (2 GiB moved) that
 * calibrates the achievable bandwidth and the HBM byte counters.  The
 * RC_KERNEL_MULTI_* ids time the k-right-hand-side SpMM and sweeps of the last
 * multi-RHS solve (they overwrite its vectors: fetch its solution first). */
int rc_time_kernel(rc_handle_t h, int kernel, int reps, double *ms_per_launch, double *bytes_per_launch);

/* ---------------- autotuner (no reference counterpart) ----------------
 * The reference's thread-block count is a command-line argument (driver.cu:
 * 2157).  rc_autotune times both triangular sweeps for every candidate launch
 * configuration (start of the dense tail, by estimate or by a level width
 * limit, x persistent sweep grid) on the factored structure and keeps the
 * fastest for this handle (later factors of the same handle reuse it).  Needs rc_factor and rc_set_rhs
 * first; the RHS and the factor are unchanged.  reps <= 0 means 5. */
typedef struct {
    int32_t tail_max_rows;    /* width limit of the chosen tail (0 = no tail)          */
    int32_t sweep_blocks;     /* chosen persistent sweep grid                          */
    int32_t configs_tried;
    double sweeps_ms_before;  /* forward + backward sweep before tuning                */
    double sweeps_ms_after;   /* ... with the chosen configuration                     */
} rc_tune_stats;
int rc_autotune(rc_handle_t h, int reps, rc_tune_stats *st);

#ifdef __cplusplus
}
#endif
#endif
