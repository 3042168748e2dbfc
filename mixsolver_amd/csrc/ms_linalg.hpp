// ms_linalg.hpp -- device Krylov solvers on SELL-64 matrices.
#pragma once
#include "ms_common.hpp"

namespace ms {

struct KS {              // device-resident solver scalars (one per solve)
  double bnrm, rz, pap, alpha, beta, res, rho, omega, snrm, tt, rr;
  double rmax, delta;    // reliable updates: largest sloppy |r| since the last update, trigger ratio
  double sigma, scale;   // FP32 iteration runs on r/sigma; scale = sigma_old/sigma_new at an update
  double cnu;            // coarse part of r.z: (Z^T r) . E^-1 (Z^T r)
  double tol;
  int it, ierr, done, maxit;  // done: 0 running, 1 finished, 2 paused for a reliable update
  int coarse;            // coarse correction active
  int ru;                // reliable update requested for this iteration
  int nru;               // reliable updates performed
  int pup;               // a p update is pending for the next product (fused p update)
  // two-launch PCG (k_cg_ps / k_cg_xr): r.z of the last two iterations, the
  // parity of the iteration under way, and whether r comes from a reliable
  // update (its residual is not tested again)
  double rz2[2];
  int par, trig;
};

struct SolveResult {
  int it = 0, ierr = 0;
  double res = 0.0;
  int outer = 0;          // refinement cycles / reliable updates (mixed precision)
  int stalled = 0;        // mixed precision: the solve ran or finished in FP64 after an FP32 stall
  int it32 = 0, it64 = 0; // iterations run in FP32 and in FP64 (it32 + it64 = it, bar the exhaustion count)
};

// Stall guard of the mixed-precision PCG: the FP32 iteration gives way to
// FP64 when its residual has not halved over this many iterations (default
// 1024; checked at the end of each 16-iteration chunk).
void set_stall_window(int iters);
int stall_window();
// in-loop timing of the mixed PCG's FP32 SpMV (the last launch of every
// 16-iteration chunk; measurement only)
void set_spmv_probe(bool on);
void read_spmv_probe(long long *launches, double *ms, long long *rows);

// average duration (ms) of a device-to-device copy of `bytes` (read + write)
double time_copy(long long bytes, int reps);
double time_stream(long long bytes, int kind, int reps);

// Matrix-free product with the reduced matrix S = D1 - B^T D0^-1 B of a
// two-colour system (rows [0,n0) colour 0, [n0,n0+n1) colour 1 of the full
// matrix A), for the FP32 inner iterations of the reduced solve: two
// launches over A's rows instead of one over the formed S.  w holds, in A's
// slices and in the order of mf_pos, -a_kj / a_kk off the diagonal and (row sum) / a_kk on it for
// the colour-0 rows, -a_ij and the row sum for the colour-1 rows; hx holds
// (h_k, x_ref_k) per colour-0 row between the two launches.
struct MatFree {
  int n0 = 0, n1 = 0;
  const SellPattern *A = nullptr;
  float *w = nullptr;
  float2 *hx = nullptr;
  const int *agg1 = nullptr;   // aggregate of every colour-1 row (coarse space), for the fused p update
  const unsigned short *c16 = nullptr;   // A's columns in 16 bits, in w's order (k_mf_cols)
  const int *win = nullptr;              // their windows, 16 per slice
};
// the pending p update p = r/d + nu[agg] + beta p, applied inside the next
// matrix-free product instead of its own launch (MIXSOLVER_P_FUSED=1;
// default off: the neighbours' r, d, aggregate and p gathered by the product
// cost more than the launch they save, 15.87 against 17.68 PISO steps/s at
// 2M cells)
bool p_fused_enabled();
void set_p_fused(bool on);
// arguments of the fused p update (beta from the solver state)
struct PUp {
  const float *r, *dg;
  const int *agg1;
  const double *nu;
};
// the reduced solve's FP32 iterations apply S matrix-free (default on;
// MIXSOLVER_SCHUR_MF=0 or ms_set_schur_matfree(0) forms S for them too)
bool schur_matfree_enabled();
void set_schur_matfree(bool on);

// Preconditioner kinds used internally.
enum PcKind { PC_JACOBI = 0, PC_NATURAL_IC0 = 1, PC_NATURAL_ILU0 = 2, PC_DILU = 3 };

// ms_levels.hip: the natural-order factor packed in the order of the
// level-scheduled sweeps, and their application
template <class T>
struct LevelFactor {
  DBuf<T> vf, vb, df, db;   // forward / backward entries and diagonals, step order
  void pack(const SellPattern &P, const T *F, bool ic0);
  DBuf<T> xf, xb;           // vectors in level order (SellPattern::sweep_ordered)
  // F: the factor in the matrix's layout, read where it is not packed
  void apply(const SellPattern &P, bool ic0, const T *F, const T *in, T *out, const int *done);
};
struct DiagFactor {   // work arrays of factor_levels: entries and diagonal in step order, factor's diagonal
  DBuf<double> lo, up, dg, d;
};
void factor_levels(const SellPattern &P, double *F, bool ic0, int *flag, DiagFactor &D);

class Krylov {
 public:
  explicit Krylov(const SellPattern *pat);
  ~Krylov();
  // FP64 solvers with the reference recurrences (mod_uns_linsolver_mpi.f90):
  // x is the initial guess on entry.  Returns reference it/res/ierr.
  // coarse: add the aggregate coarse correction of pat->coarse to the
  // preconditioner (PCG only).
  // reuse: the matrix values are those of the previous solve with the same
  // preconditioner (e.g. the second PISO corrector): its set-up (FP32 copy,
  // preconditioner, coarse inverse) is kept.
  SolveResult pcg(const double *val, const double *b, double *x, double tol, int maxit, PcKind pc,
                  bool coarse = false, bool reuse = false);
  // coarse: add the aggregate coarse correction Z E^-1 Z^T to the
  // preconditioner (the p' matrix is symmetric, so E is)
  SolveResult bicgstab(const double *val, const double *b, double *x, double tol, int maxit, PcKind pc,
                       bool coarse = false);
  // Mixed precision.  PCG: FP32 matrix, preconditioner and Krylov vectors
  // with FP32 accumulation, FP64 solution and reliable updates of the true
  // FP64 residual.  BiCGSTAB: FP32 inner solves inside FP64 iterative
  // refinement.  res is the FP64 true relative residual.
  SolveResult mixed(const double *val, const double *b, double *x, double tol, int maxit, PcKind pc,
                    int solver, double inner_tol, bool coarse = false, bool reuse = false);
  void spmv(const double *val, const double *x, double *y);
  // average duration (ms) of the PCG SpMV+dot kernel on matrix val, measured
  // with HIP events on the library stream over `reps` launches; fp32 selects
  // the FP32 difference-form kernel of the mixed path.
  double time_spmv(const double *val, bool fp32, int reps, bool cold = false);
  long long launches = 0;
  bool fp32_stalled() const { return fp32_stalled_; }
  // the FP32 SpMV of the mixed PCG applies this operator instead of val32
  void set_matfree(const MatFree *m) { mf_ = m; }
  bool matfree_on() const { return mf_ && schur_matfree_enabled(); }

  const SellPattern *pat;
  int n;
  struct HostState {   // pinned page for the solver state, and its events
    int dev = 0;
    void *pin = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
  };

 private:
  static HostState borrow_host_state();
  static void give_back_host_state(const HostState &h);
  HostState host_;
  int setup_pc64(PcKind pc, const double *val);
  void setup_pc32(PcKind pc, const double *val);
  // staged: the launch that formed `in` has done the first stage (Jacobi's
  // quotient, DILU's first colour)
  template <class T> void apply_pc(PcKind pc, const T *val, const T *fac, const T *dg, const T *in, T *out,
                                   const int *done, bool staged = false);
  template <class T> KS read_state(KS *d);
  bool small_system() const;
  // two-launch PCG (no coarse space): its vectors and partial arrays
  template <class T> struct Cg2 {
    PcKind pc = PC_JACOBI;
    int mode = 0, G = 0, nrz = 0;   // grid; r.z partials in rz
    T *r = nullptr, *z = nullptr, *p0 = nullptr, *p1 = nullptr, *q = nullptr, *dg = nullptr;
    T *rr = nullptr, *rz = nullptr, *pq = nullptr, *swp = nullptr;
  };
  template <class T> Cg2<T> cg2(PcKind pc);
  template <class T> void cg2_precond(const Cg2<T> &c, const T *val, const T *fac);
  template <class T> void cg2_start(const Cg2<T> &c, const T *val, const T *fac);
  template <class T, bool MIXED, class X>
  void cg2_iteration(const Cg2<T> &c, const T *val, const T *fac, X *x, hipEvent_t e0, hipEvent_t e1);
  // PCG with a coarse space: vectors, partial arrays, chunk sums
  template <class T> struct Cx {
    int mode = 0, G = 0, nrz = 0, ncn = 0, cw = 0;   // grid; r.z partials; coarse parts of r.z; coarse workgroups
    T *r = nullptr, *z = nullptr, *p = nullptr, *q = nullptr, *dg = nullptr;
    T *rr = nullptr, *rz = nullptr, *csum = nullptr, *pq = nullptr;
  };
  template <class T> Cx<T> cx(PcKind pc);
  template <class T, bool MIXED> void cx_p(const Cx<T> &c, int what);
  template <class T, bool MIXED> void cx_direction(const Cx<T> &c, const T *val, int what);
  template <class T, bool MIXED> void cx_restart(const Cx<T> &c, const T *val, const double *r64, bool direction);
  template <class T, bool MIXED, class X> void cx_update(const Cx<T> &c, const T *val, X *x, bool ride);
  SolveResult bicg32(PcKind pc, int maxit, int window, bool coarse);
  template <class T> void coarse_apply(T *out, KS *st);
  template <class T> struct Parts {   // one or two arrays of n partials
    int n;
    const T *a, *b;
  };
  template <class T> Parts<T> parts_for(int readers, int m, const T *a, const T *b, const KS *st);
  // BiCGSTAB: vectors, solution, preconditioner, partials and state
  template <class T> struct Bi {
    T *r, *r0, *p, *v, *s, *t, *ph, *sh, *x;
    const T *dg, *fac;
    T *part;
    KS *st;
  };
  template <class T> void bi_start(const Bi<T> &w);
  template <class T> void bi_iteration(const Bi<T> &w, PcKind pc, const T *val, bool coarse);
  template <class T> KS bi_state(const Bi<T> &w);
  void ensure32();
  void coarse_setup(const double *val);   // E = Z^T A Z and its inverse

  DBuf<double> r_, r0_, p_, q_, z_, s_, t_, ph_, sh_, fac_, dg_, part_, prz_;   // prz_: DILU sweep partials
  DBuf<float> val32_, r32_, r032_, p32_, q32_, z32_, s32_, t32_, ph32_, sh32_, x32_, fac32_, dg32_, part32_, prz32_;
  DBuf<KS> st_, st32_;
  DBuf<double> cnu_split_;   // c.nu parts of k_cx_coarse
  DBuf<int> flag_;
  LevelFactor<double> lev_;
  LevelFactor<float> lev32_;
  DiagFactor diag_;
  CoarseMat cm_;             // E, E^-1 and nu of the coarse space for the current matrix
  DBuf<double> co_part_;     // chunk sums of a BiCGSTAB coarse correction
  const MatFree *mf_ = nullptr;
  // q = op p with the fused p.q partials; start / stop events (may be null)
  // bracket the product's launches
  void spmv32(const double *val64, const float *v32, float *p, float *q, KS *st, float *part, hipEvent_t e0,
              hipEvent_t e1, const PUp *pu = nullptr);
  void *hpin_ = nullptr;
  hipEvent_t state_ev_[2] = {nullptr, nullptr};   // the two pipelined chunk states (mixed PCG)
  void *state_slot(int slot) const { return (char *)hpin_ + 1024 * (slot + 1); }
  int nblk_;
  bool have32_ = false;
  struct SetupKey {
    const double *val = nullptr;
    int pc = -1, fp32 = -1, coarse = -1;
    bool operator==(const SetupKey &o) const {
      return val == o.val && pc == o.pc && fp32 == o.fp32 && coarse == o.coarse;
    }
  } last_;   // the set-up the preconditioner buffers currently hold
  // captured 16-iteration chunk of the mixed PCG: valid while the kernels'
  // arguments (buffers, preconditioner, coarse mode) are those of the key
  struct ChunkKey {
    const void *v32 = nullptr, *fac = nullptr, *dg = nullptr, *nu = nullptr;
    int pc = -1, coarse = -1, fused = -1, len = 0, mf = 0, pf = 0;
    bool operator==(const ChunkKey &o) const {
      return v32 == o.v32 && fac == o.fac && dg == o.dg && nu == o.nu && pc == o.pc && coarse == o.coarse &&
             fused == o.fused && len == o.len && mf == o.mf && pf == o.pf;
    }
  } chunk_key_;
  hipGraphExec_t chunk_exec_ = nullptr;
  bool fp32_stalled_ = false;   // the mixed PCG stalled on this system: FP64 PCG from then on
};

}  // namespace ms
