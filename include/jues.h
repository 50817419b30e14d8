/*
 * libjues_hip -- C ABI for JuES's correlation hot path on MI355X (gfx950).
 *
 * Conventions
 *   - Every array is COLUMN-MAJOR (Fortran order) with 0-based indices, i.e.
 *     exactly the memory a Julia Array{Float64,N} hands to ccall.
 *     A Julia T2[i,j,a,b] (o x o x v x v) is element i + o*(j + o*(a + v*b)).
 *   - Host pointers are only read/written during the call; the library keeps no
 *     host pointer after it returns.  Device state lives in a jues_ctx.
 *   - Calls are synchronous with respect to the host.  A jues_ctx is not
 *     thread-safe: use one per host thread.
 *   - Every call returns a jues_status; on error jues_last_error() describes it.
 *
 * Reference interfaces (paths relative to the JuES.jl tree) are cited on each
 * entry point.  The reference has no FFI of its own; these entry points replace
 * the bodies of the Julia functions named there (see the ccall stubs in
 * jues.jl_amd/julia/JuESHip.jl).
 */
#ifndef JUES_H
#define JUES_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct jues_ctx jues_ctx;

typedef enum {
    JUES_OK = 0,
    JUES_NOT_CONVERGED = 1,  /* iteration limit reached; results hold the last iterate */
    JUES_NONFINITE = 2,      /* a NaN/Inf appeared (e.g. a zero orbital-energy denominator) */
    JUES_OOM = 3,            /* device allocation failed */
    JUES_BAD_ARG = 4,        /* invalid sizes, strings, null pointers, missing integrals */
    JUES_HIP_ERROR = 5       /* a HIP runtime call failed */
} jues_status;

typedef enum {
    JUES_FP64 = 0,        /* plain form: every contraction in FP64 MFMA */
    JUES_FP32_MIXED = 1,  /* contractions in FP32 MFMA (FP32 accumulate); energies,
                             denominators, DIIS and the final refinement in FP64 */
    JUES_FP16X3_MIXED = 2 /* as FP32_MIXED, but the ring, particle-particle ladder and
                             hole-hole GEMMs run on FP16 MFMA with each FP32 operand split
                             into hi + lo halves under a power-of-two scale (three products,
                             FP32 accumulate; ~2^-21 relative per product).  Below o v = 1900 they
                             run in FP32 MFMA, which is faster there and more precise */
} jues_prec;

/* Which reference RCCSD equations to follow.  They differ only in the T1 exchange
 * term of Fae: mRCCSD.jl:140 contracts t1[m,f] with <me|af>, RCCSD.jl:189 with
 * <ma|ef>.  Every other term is identical. */
typedef enum {
    JUES_CCSD_MRCCSD = 0,  /* CoupledCluster/mRCCSD.jl (the module the reference test uses) */
    JUES_CCSD_RCCSD = 1    /* CoupledCluster/RCCSD.jl */
} jues_ccsd_eqs;

/* Initial T2 guess.  MP2 and OVOV are the first-order amplitudes of the equations
 * iterated first, so under coupling continuation they carry that lambda (c/N). */
typedef enum {
    JUES_GUESS_ZERO = 0,   /* t = 0, as mRCCD.jl:245 */
    JUES_GUESS_MP2 = 1,    /* t = <ij|ab>/D, as mRCCSD.jl:66 */
    JUES_GUESS_OVOV = 2,   /* t = (ij|ab)/D, as RCCD.jl:145-160 */
    JUES_GUESS_USER = 3    /* t = T2_inout on entry (warm start) */
} jues_guess;

/* Particle-particle ladder integrals <ab|ef>. */
typedef enum {
    JUES_LADDER_AUTO = 0,       /* stored when they fit in device memory, else recomputed (needs factors) */
    JUES_LADDER_STORED = 1,     /* packed V+/V- built once and kept (o^0 v^4 / 2 elements) */
    JUES_LADDER_RECOMPUTE = 2   /* rebuilt from the 3-index factors every iteration in slabs, as
                                   DF-RCCD.jl:198-215 contracts bvv . bvv; never stored */
} jues_ladder;

/* How a fast stage (FP32_MIXED / FP16X3_MIXED) hands over to FP64. */
typedef enum {
    JUES_REFINE_RESTART = 0,  /* FP64 iterations from the fast stage's amplitudes with a fresh DIIS
                                 history, until e_conv / r_conv (at most refine_maxit) */
    JUES_REFINE_DEFECT = 1    /* defect correction (RCCD; RCCSD falls back to RESTART): an FP64
                                 iteration at t0 keeps its numerator R0 = <ij|ab> + S + L, and the fast
                                 stage then solves D t = lambda (R0 + [R(t) - R(t0)]) with the bracket
                                 formed from d = t - t0, so that its rounding scales with |d|, not
                                 |t|; repeated until an FP64 iteration meets e_conv / r_conv, at most
                                 refine_maxit FP64 iterations */
} jues_refine;

/* Options; jues_cc_default_opts() fills the defaults noted here.
 * Names mirror CoupledCluster.jl:36-43 (cc_max_iter, cc_e_conv, cc_max_rms, diis). */
typedef struct {
    int32_t maxit;            /* cc_max_iter, default 100 */
    double e_conv;            /* |E_k - E_{k-1}| threshold, default 1e-10 */
    double r_conv;            /* ||t_new - t_old||_2 threshold, default 1e-9 */
    int32_t diis;             /* 1 = DIIS (mRCCD.jl:171-203), 0 = plain Jacobi (RCCD.jl:55-74) */
    int32_t diis_max;         /* (t, error) pairs kept; mRCCD.jl's max_diis=6 keeps 5. default 5 */
    int32_t guess;            /* jues_guess, default JUES_GUESS_MP2 */
    int32_t ccsd_eqs;         /* jues_ccsd_eqs, default JUES_CCSD_MRCCSD */
    int32_t fcn;              /* frozen core: drop the first fcn occupied orbitals (get_eri's fcn) */
    /* FP32_MIXED / FP16X3_MIXED: the fast stage stops once ||dt||_2 < fp32_r_conv (or it
     * stalls); FP64 refinement iterations then run to e_conv / r_conv, at most refine_maxit. */
    double fp32_r_conv;       /* default 1e-5 */
    int32_t refine_maxit;     /* default 60 */
    int32_t verbose;          /* print one line per iteration to stderr */
    /* Coupling continuation.  Every residual term carries exactly one integral, so the
     * equations for integrals scaled by lambda are t = lambda R(t) / D.  With
     * continuation = N > 1 the solver converges lambda = c/N, 2c/N, ..., c (c = coupling)
     * in turn, each warm-started from the previous amplitudes with a fresh DIIS history;
     * the result is the lambda = c solution on the branch connected to lambda -> 0.
     * Energies are those of the lambda-scaled integrals. */
    double coupling;          /* c, default 1.0 */
    int32_t continuation;     /* N, default 1 (no continuation) */
    int32_t ladder;           /* jues_ladder, default JUES_LADDER_AUTO */
    int32_t refine;           /* jues_refine, default JUES_REFINE_RESTART */
} jues_cc_opts;

/* Per-iteration record passed to the optional callback. */
typedef struct {
    int32_t iter;             /* 1-based */
    int32_t stage;            /* 0 = FP64, 1 = the fast stage of FP32_MIXED, 2 = that of FP16X3_MIXED */
    double energy;            /* correlation energy of the Jacobi update t_new */
    double delta_e;           /* energy - previous energy */
    double rnorm;             /* ||t_new - t_old||_2 (T1 and T2 together for CCSD) */
    int32_t diis_size;        /* number of DIIS pairs used this iteration */
    double ms;                /* device time of the iteration (HIP events on the ctx stream) */
    double coupling;          /* lambda of the equations iterated (1 unless continuation is used) */
} jues_iter_info;

typedef void (*jues_iter_cb)(void* user, const jues_iter_info* info);

/* ---- context -------------------------------------------------------------- */
jues_status jues_create(jues_ctx** ctx, int device);
void jues_destroy(jues_ctx* ctx);
const char* jues_last_error(const jues_ctx* ctx);
void jues_cc_default_opts(jues_cc_opts* opts);
/* Bytes of device memory currently held by the library: integrals, scratch, and the blocks that
 * each context keeps for its next buffers (at most a sixteenth of the device's memory). */
size_t jues_device_bytes(const jues_ctx* ctx);
/* Release all device buffers held by the context, kept blocks included (keeps the stream). */
jues_status jues_release(jues_ctx* ctx);

/* ---- AO integrals (the Wfn.ao_eri carrier, Backend/Wavefunction.jl:87) ------
 * Exactly one representation is current; setting one drops the other.
 * dense: g[mu,nu,lam,sig], n^4, chemist order (mu fastest), copied to the device.
 * factors: B[mu,nu,P], n x n x naux, with (mu nu|lam sig) = sum_P B[mu,nu,P] B[lam,sig,P];
 *          the dense tensor is never formed (configs whose n^4 does not fit). */
jues_status jues_set_ao_eri(jues_ctx* ctx, const double* gao, int n);
jues_status jues_set_ao_factors(jues_ctx* ctx, const double* B, int n, int naux);

/* ---- Density fitting (Backend/DF.jl:30-58) ------------------------------------
 * Takes the pair setup_df returns (DF.jl:48-50): the three-index integrals
 * pqP[mu,nu,P] (n x n x naux) and the metric's inverse square root
 * Jpqh[P,Q] = (P|Q)^(-1/2) (naux x naux), and forms
 * b[mu,nu,Q] = sum_P pqP[mu,nu,P] Jpqh[P,Q] (make_bmunu, DF.jl:52-58) on the
 * device; b becomes the current AO factors, so every entry point below then runs
 * the DF route: jues_rmp2 is do_df_rmp2 (MollerPlesset/DF-RMP2.jl:1-46) and
 * jues_rccd with the recomputed ladder is do_df_rccd's bvv.bvv contraction
 * (CoupledCluster/DF-RCCD.jl:207).  jues_get_ao_factors copies the current
 * factors back (n and naux must match). */
jues_status jues_set_df_integrals(jues_ctx* ctx, const double* pqP, const double* Jpqh, int n, int naux);
jues_status jues_get_ao_factors(jues_ctx* ctx, double* B, int n, int naux);

/* ---- Transformation.tei_transform (Backend/Transformation.jl:39-93) ----------
 * out[p,q,r,s] = sum C1[mu,p] C2[nu,q] C3[lam,r] C4[sig,s] g[mu,nu,lam,sig]
 * (chemist order, out is d1 x d2 x d3 x d4).  C_k is n x d_k.  Uses the dense AO
 * tensor if set, else the factors.  FP32_MIXED runs the quarter GEMMs in FP32. */
jues_status jues_tei_transform(jues_ctx* ctx, int prec,
                               const double* C1, int d1, const double* C2, int d2,
                               const double* C3, int d3, const double* C4, int d4,
                               int n, double* out);

/* ---- IntegralTransformation.get_eri (Backend/IntegralTransformation.jl:38-101) --
 * eri_string: 4 chars from {o,O,v,V}; notation: "phys" (default when NULL) or "chem".
 * As the reference (:52-68), upper-case letters take the alpha orbitals, O -> Cao
 * (n x nalpha) and V -> Cav (n x nvira), lower-case letters the beta ones, o -> Cbo
 * (n x nbeta) and v -> Cbv (n x nvirb); for a restricted reference pass the alpha arrays
 * twice.  A block the string does not name may be NULL.  fcn drops the first fcn
 * columns of either occupied block.  out has the dimensions the letters name (nalpha -
 * fcn, nbeta - fcn, nvira or nvirb), in the requested notation.  prec: JUES_FP64 or
 * JUES_FP32_MIXED (quarter GEMMs in FP32). */
jues_status jues_get_eri(jues_ctx* ctx, int prec, const char* eri_string, const char* notation,
                         const double* Cao, int nalpha, const double* Cav, int nvira,
                         const double* Cbo, int nbeta, const double* Cbv, int nvirb, int n, int fcn,
                         double* out);

/* ---- MollerPlesset.do_rmp2 (MollerPlesset/RMP2.jl:11-45) ----------------------
 * E = sum_{ijab} <ij|ab>(2<ij|ab> - <ij|ba>) / (e_i + e_j - e_a - e_b). eps has n = o+v entries. */
jues_status jues_rmp2(jues_ctx* ctx, int prec, const double* Cocc, int o, const double* Cvir,
                      int v, int n, const double* eps, double* E);

/* ---- Allocation-free RMP2 (no reference counterpart) -----------------------------
 * For callers that cannot allocate device memory: code under HIP graph capture, tight
 * serving loops, harnesses that forbid hipMalloc.  The FP64 RMP2 energy of jues_rmp2 (same
 * inputs, prec must be JUES_FP64) from the context's AO factors, which must already be set
 * (jues_set_ao_factors / jues_set_df_integrals allocate; this call does not).  Every device
 * intermediate lives in one static array of JUES_NOALLOC_SCRATCH_BYTES per GPU, which each
 * GPU the library runs on holds until the process ends; the call makes no hipMalloc/hipFree
 * and touches no context scratch.  It needs, in 8-byte elements with each region rounded up
 * to 256 bytes, n*o + n*v + (o+v) + (o*v+1) + max(n*min(o,v), o*v)*naux + o*v*naux + o*v*v
 * (one occupied index's slab of (ia|jb)); larger problems return JUES_BAD_ARG with the byte
 * count (o=60, v=340, n=400, naux=1200 needs 483 MB and fits).  Calls on one GPU share the
 * array: calls that overlap on one GPU (two threads, two contexts) race. */
#define JUES_NOALLOC_SCRATCH_BYTES (512ull << 20)
jues_status jues_rmp2_noalloc(jues_ctx* ctx, int prec, const double* Cocc, int o, const double* Cvir,
                              int v, int n, const double* eps, double* E);

/* MP2 adjoint (no reference counterpart; the reverse rule of jues_rmp2 for a
 * ChainRulesCore rrule).  C is the full n x n matrix [Cocc Cvir] (o occupied
 * columns first), eps the n orbital energies (occupied first).  Outputs, each may be
 * NULL: dE_dC (n x n), dE_dg (n^4, only with a dense AO tensor) and dE_deps (n).
 * Every entry of C, g and eps is an independent variable.  With AO factors the
 * gradient takes the factor route (dL = 2 G L through L = Co^T B_P Cv; no n^2 o v
 * intermediate); with a dense AO tensor the call recomputes the half-transformed
 * integrals it needs (the forward transform's and (mu a|j sig)), storing nothing
 * between calls. */
jues_status jues_rmp2_grad(jues_ctx* ctx, int prec, const double* C, int o, int n,
                           const double* eps, double* E, double* dE_dC, double* dE_dg,
                           double* dE_deps);

/* ---- CoupledCluster.{RCCD,mRCCD}.do_rccd (RCCD.jl:33-83, mRCCD.jl:38-118) ------
 * Converges the closed-shell CCD equations of RCCD.jl:134-303.  T2_inout (o x o x v x v,
 * Julia order) may be NULL; when given it receives the final amplitudes, and with
 * guess == JUES_GUESS_USER it also supplies the starting amplitudes.  These have
 * t[i,j,a,b] = t[j,i,b,a], as every iterate has: the packed ladders read one of the two
 * and the ring terms their half-sum. */
jues_status jues_rccd(jues_ctx* ctx, int prec, const jues_cc_opts* opts,
                      const double* Cocc, int o, const double* Cvir, int v, int n,
                      const double* eps, double* E, double* T2_inout,
                      jues_iter_cb cb, void* user);

/* ---- CoupledCluster.{RCCSD,mRCCSD}.do_rccsd (RCCSD.jl:33-101, mRCCSD.jl:35-101) --
 * T1_inout is o x v.  opts->ccsd_eqs selects the reference module's equations. */
jues_status jues_rccsd(jues_ctx* ctx, int prec, const jues_cc_opts* opts,
                       const double* Cocc, int o, const double* Cvir, int v, int n,
                       const double* eps, double* E, double* T1_inout, double* T2_inout,
                       jues_iter_cb cb, void* user);

/* ---- AutoRCCSD.do_rccsd (CoupledCluster/AutoRCCSD.jl:193-300) -----------------
 * Closed-shell CCSD driven by the full MO Fock matrix `fock` ((o + v) x (o + v) over
 * [Cocc | Cvir], e.g. from jues_get_fock): the resolvents take its diagonal and the
 * off-diagonal blocks f_oo, f_vv, f_ov enter the residuals (AutoRCCSD.jl:76-132) and
 * the energy 2 f_ia t_ia (:39-51), so non-canonical and non-Hartree-Fock references
 * are handled.  The equations are those of the RCCSD.jl set (opts->ccsd_eqs), the
 * MP2 guess adds T1 = f_ia / d_ia (:249), and options, precision and outputs are as
 * for jues_rccsd (coupling must be 1, continuation 1). */
jues_status jues_rccsd_fock(jues_ctx* ctx, int prec, const jues_cc_opts* opts, const double* Cocc, int o,
                            const double* Cvir, int v, int n, const double* fock, double* E, double* T1_inout,
                            double* T2_inout, jues_iter_cb cb, void* user);

/* ---- MollerPlesset.do_ump2 (MollerPlesset/UMP2.jl:12-79) ------------------------
 * Unrestricted MP2 on a UHF reference: alpha-alpha and beta-beta pairs i > j, a > b
 * of <ij||ab>^2 / D, and alpha-beta pairs of (ia|JB)^2 / D.  Cao (n x na), Cav
 * (n x va), Cbo (n x nb), Cbv (n x vb); epsa (na + va) and epsb (nb + vb) hold the
 * occupied energies first.  nb may be 0 (then Cbo may be NULL). */
jues_status jues_ump2(jues_ctx* ctx, int prec, const double* Cao, int na, const double* Cav, int va,
                      const double* Cbo, int nb, const double* Cbv, int vb, int n, const double* epsa,
                      const double* epsb, double* E);

/* ---- IntegralTransformation.get_fock (Backend/IntegralTransformation.jl:119-141) --
 * f[p,q] = sum C[mu,p] C[nu,q] (h[mu,nu] + 2 (mu nu|lam sig) D[lam,sig] - (mu lam|nu sig) D[lam,sig]),
 * D = Co Co^T, for the m columns of C (n x m) and the o columns of Co (n x o), from
 * the context's AO integrals (dense or factors) and the core Hamiltonian hao (n x n);
 * f is m x m.  The reference's spin keyword selects (C, Co) = (Ca, Cao) or (Cb, Cbo). */
jues_status jues_get_fock(jues_ctx* ctx, const double* hao, const double* C, int m, const double* Co, int o, int n,
                          double* f);

/* ---- PerturbativeTriples.compute_pT (CoupledCluster/PerturbativeTriples.jl:35-138) ----
 * Et = (T) correction from the CCSD amplitudes T1 (o x v), T2 (o x o x v x v) and the
 * integral arrays AutoRCCSD.jl:295-297 passes: Vvvvo (v x v x v x o), Vvooo (v x o x o x o),
 * Vvovo (v x o x v x o), with fo (o) and fv (v) the diagonal Fock elements.  The loop of
 * :79-133 (i >= j >= k, a >= b >= c, weights (2-d_ij-d_jk)/(1+d_ab+d_bc)) runs on the
 * device; FP32_MIXED forms W in FP32 MFMA and sums the energy in FP64.
 * jues_rccsd_pT builds the same three blocks on the device from the context's AO
 * integrals (dense or factors) and canonical orbitals, fo/fv = eps (AutoRCCSD.jl:294-300).
 * verbose != 0 prints one progress line per occupied orbital i to stderr, as :81 does. */
jues_status jues_compute_pT(jues_ctx* ctx, int prec, const double* T1, const double* T2, const double* Vvvvo,
                            const double* Vvooo, const double* Vvovo, const double* fo, const double* fv, int o,
                            int v, int verbose, double* Et);
jues_status jues_rccsd_pT(jues_ctx* ctx, int prec, const double* Cocc, int o, const double* Cvir, int v, int n,
                          const double* eps, const double* T1, const double* T2, int verbose, double* Et);

/* ---- stepwise solver (the same loop as jues_rccd / jues_rccsd, split so that a
 * caller can time iterations with every input already resident on the device) ----
 * method: 0 = RCCD, 1 = RCCSD.  setup builds the MO integral blocks on the device and
 * the starting amplitudes; iterate runs up to nsteps iterations in the given stage
 * precision (JUES_FP64 or JUES_FP32_MIXED), stopping early only if stop_on_conv is set
 * and the convergence test passes.  info receives the last iteration's record. */
jues_status jues_cc_setup(jues_ctx* ctx, int method, int prec, const jues_cc_opts* opts,
                          const double* Cocc, int o, const double* Cvir, int v, int n,
                          const double* eps, const double* T1_init, const double* T2_init);
jues_status jues_cc_iterate(jues_ctx* ctx, int stage_prec, int nsteps, int stop_on_conv,
                            jues_iter_info* info, int* converged);
/* Reset the DIIS history (e.g. at the FP32 -> FP64 hand-over). */
jues_status jues_cc_reset_diis(jues_ctx* ctx);
/* Defect-correction refinement (JUES_REFINE_DEFECT) of the resident RCCD state: at most
 * max_anchors FP64 iterations, each (unless it meets e_conv / r_conv, or is the last)
 * followed by at most inner_maxit iterations of the correction equation in inner_prec
 * (JUES_FP32_MIXED, JUES_FP16X3_MIXED, or JUES_FP64, where the bracket is exact), which stop
 * once ||dt||_2 < max(r_conv / 10, kappa ||dt||_2 of the FP64 iteration) or stall, kappa being
 * about what one FP64 iteration can contract with that inner form (1e-5 FP32, 1e-3 split-FP16, 0 FP64).  info receives the last FP64 iteration's record;
 * converged is set when it met the convergence test; n_fp64 (may be null) receives the
 * number of FP64 iterations run. */
jues_status jues_cc_refine(jues_ctx* ctx, int inner_prec, int max_anchors, int inner_maxit,
                           jues_iter_info* info, int* converged, int* n_fp64);
jues_status jues_cc_get(jues_ctx* ctx, double* E, double* T1_out, double* T2_out);

/* Accumulated device time per kernel class since the last reset (HIP events on
 * the ctx stream).  names/ms/flops/bytes arrays of length cap; returns the count. */
int jues_kernel_stats(jues_ctx* ctx, const char** names, double* ms, double* calls,
                      double* flops, double* bytes, int cap);
void jues_kernel_stats_reset(jues_ctx* ctx, int enable);

/* Raw MFMA GEMM (column-major): C = alpha*op(A)*op(B) + beta*C, on device copies of
 * host arrays.  Exposed for the GEMM unit tests; prec selects FP64 or FP32 MFMA, or
 * JUES_FP16X3_MIXED for the split-FP16 GEMM. */
jues_status jues_gemm_test(jues_ctx* ctx, int prec, char transa, char transb, int M, int N,
                           int K, double alpha, const double* A, int lda, const double* B,
                           int ldb, double beta, double* C, int ldc);

/* Two independent products C_i = alpha*A_i*op(B_i) + beta*C_i (A_i not transposed, op the
 * same for both) in one launch of the MFMA GEMM kernel, as the coupled-cluster ladders use
 * it; device copies of host arrays, FP64 or FP32 (prec).  Exposed for the GEMM unit tests. */
jues_status jues_gemm_pair_test(jues_ctx* ctx, int prec, char transb, int M0, int N0, int K0,
                                const double* A0, int lda0, const double* B0, int ldb0, double* C0,
                                int ldc0, int M1, int N1, int K1, const double* A1, int lda1,
                                const double* B1, int ldb1, double* C1, int ldc1, double alpha,
                                double beta);

#ifdef __cplusplus
}
#endif
#endif /* JUES_H */
