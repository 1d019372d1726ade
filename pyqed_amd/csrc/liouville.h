// Shared by the Liouville-space entry points: the register form for N <= 16 (liouville_small.hip).
#pragma once

#include "common.h"

namespace pqa {

constexpr int kSmallN = 16;

struct LiouvilleRun {
  int N, nterm, n_inst, n_obs;
  int64_t nsteps, save_every;
  double dt;
  const double2* A;      // [nterm][N][N]
  const double* field;   // [n_inst][nsteps][nterm - 1]
  double2* rho;          // [n_inst][N], advanced in place (adjoint: read)
  const double2* obs;
  double2* obs_out;
  double2* rho_out;
  // adjoint
  const double2* rhoT_bar;
  double* grad_field;
  double2* grad_A;
  double2* rho0_bar;
  double2* ckpt;         // states at the starts of the segments, [n_inst][nsegs + 1][N], then scratch of one
                         // segment's states, [groups][seg][N]
  int64_t seg;           // steps per segment
};

LiouvilleRun forward_run(int N, int nterm, const void* A, int n_inst, void* rho, const double* field, int64_t nsteps, double dt,
                         int n_obs, const void* obs, void* obs_out, void* rho_out, int64_t save_every);
LiouvilleRun adjoint_run(int N, int nterm, const void* A, int n_inst, const void* rho0, const double* field, int64_t nsteps,
                         double dt, int64_t seg, const void* rhoT_bar, double* grad_field, void* grad_A, void* rho0_bar,
                         void* ckpt);
// Does the register form take these sizes (N and the LDS of its generators and gradient rows)?
bool small_fits(int N, int nterm, bool grad_A);
// Segment length with which a run of N <= 16 is cut along time, or 0 where it stays one chain per instance.
int64_t small_split(int N, int nterm, int n_inst, int64_t nsteps, bool adjoint);
// Workspace of a cut run: segment propagators and the states (and adjoint states, gradients) at their ends.
int64_t small_split_bytes(int N, int nterm, int n_inst, int64_t nsteps, int64_t seg, bool adjoint);

int small_forward(const LiouvilleRun& r, hipStream_t st);
int small_forward_split(const LiouvilleRun& r, void* work, hipStream_t st);
int small_adjoint(const LiouvilleRun& r, hipStream_t st);
int small_adjoint_split(const LiouvilleRun& r, void* work, hipStream_t st);

// dv/dt = A v for one vector of N <= 1024 elements by powers of the RK4 step matrix (propagator.hip): nsteps
// steps in place, kRowSeg rows at a time; every `every` steps the first n_out elements go to out + slot out_stride
// (out may be NULL).  Weak: a program linked without propagator.hip has no such runs (power_size).
constexpr int64_t kRowSeg = 1024;
// complex elements of the matrices: seven and the powers
inline int64_t power_matrix_elems(int N, int levels) { return (int64_t)(7 + levels) * N * N; }
inline int64_t power_vector_bytes(int N) { return 16 * (power_matrix_elems(N, 7) + kRowSeg * N); }
__attribute__((weak)) int power_vector(int N, const double2* A, double2* v, int64_t nsteps, double dt, double2* out, int n_out,
                                       int64_t out_stride, int64_t every, void* work, hipStream_t st);

}  // namespace pqa
