// krylov.hpp -- internal interfaces of the Krylov layer.
#pragma once

#include <cmath>
#include <memory>

#include "common.hpp"

struct tnlmi_spmv_plan;
struct tnlmi_preconditioner;

namespace tnlmi {

// The matrix operator of a solver: y = A x with FP64 vectors and
// accumulation, through the matrix's own format kernels or its split plan.
struct Operator
{
   const tnlmi_matrix* A;
   const tnlmi_spmv_plan* plan;
   int64_t rows;
   void apply( const double* x, double* y, hipStream_t s ) const;
};

// x = M^{-1} b (identity when P is NULL)
void precond_apply( const tnlmi_preconditioner* P, int64_t n, const double* b, double* x, hipStream_t s );

// The preconditioner's kind and, for the Diagonal one, its diagonal d (x = b / d).
tnlmi_precond_kind precond_kind( const tnlmi_preconditioner* P );
const double* precond_diagonal( const tnlmi_preconditioner* P );

// ---------------------------------------------------------- solver state

// IterativeSolver.hpp:98-143
struct Stop
{
   tnlmi_solver_state* st;
   int64_t it = 0;
   double res = 0;
   bool check() const
   {
      return ! ( std::isnan( res ) || it > st->max_iterations
                 || ( res > st->divergence_residue && it >= st->min_iterations )
                 || ( res < st->convergence_residue && it >= st->min_iterations ) );
   }
   bool next()
   {
      const bool r = check();
      it++;
      return r;
   }
   bool converged() const
   {
      if( std::isnan( res ) )
         return false;
      if( res > st->divergence_residue && it > st->min_iterations )
         return false;
      if( it >= st->max_iterations )
         return false;
      if( res > st->convergence_residue )
         return false;
      return true;
   }
};

// pinned host mirror of a few device scalars
struct HostScalars
{
   double* h = nullptr;
   HostScalars() { TNLMI_HIP( hipHostMalloc( (void**) &h, 64 * sizeof( double ), hipHostMallocDefault ) ); }
   ~HostScalars()
   {
      if( h )
         (void) hipHostFree( h );
   }
   // synchronous read of k device scalars starting at d
   const double* read( const double* d, int k, hipStream_t s )
   {
      TNLMI_HIP( hipMemcpyAsync( h, d, k * sizeof( double ), hipMemcpyDeviceToHost, s ) );
      TNLMI_HIP( hipStreamSynchronize( s ) );
      return h;
   }
};

// CG with fused kernels for no or Diagonal preconditioning (fused_cg.hip).
// residue_kind 0: TNL's residue sqrt((r, z)) / ||M^-1 b||; 1: the recurrence
// residual ||r|| / ||b|| (the true-residual stopping rule of the mixed solvers).
// column_codes: 8-bit column codes for a column-major Ellpack / SlicedEllpack
// matrix of few distinct column offsets (as the mixed solver's inner matrix), in
// the launches per iteration that use no row masks.
void fused_cg_solve( const Operator& A, const tnlmi_preconditioner* M, const double* b, double* x,
                     tnlmi_solver_state* st, hipStream_t s, int residue_kind = 0, bool column_codes = false );

// ---- solvers whose iterations run in one resident launch (krylov_resident.hip)

// An FP64 matrix's rows as column-major Ellpack slots: its own, or a copy of a
// CSR matrix's with short rows of about one length.
struct EllSlots
{
   int64_t n = 0, stride = 0;
   int32_t w = 0;
   const int32_t* cols = nullptr;
   const double* vals = nullptr;
};
// how many doubles the copy takes (0: none is made).  It has a place in a work array
// of the solve: an allocation of its own, of more than 64 MB, would take 0.3 ms
int64_t ell_copy_values( const Operator& A );
// false: the matrix has no such slots, more rows than a resident launch takes, or
// more lines * rows of far columns than `far` (fused_cg.hip)
// room: ell_copy_values( A ) doubles, or NULL (then no copy is made)
bool ell_slots( const Operator& A, double far, double* room, EllSlots& out, hipStream_t s );

// BiCGStab's iterations from an admitted one on (sc: the solver's scalars).
// Returns what ended them, or kResidentNot when nothing was launched.
enum ResidentEnd { kResidentNot, kResidentStopped, kResidentMore, kResidentRestart, kResidentLate, kResidentZeroPivot };

struct ResidentState  // on the device, and its host copy
{
   double res, beta, normb, beta_ratio;
   int64_t it;
   int32_t end, cycles, m, pad;
};

struct ResidentBicgstab
{
   EllSlots A;
   const double *d, *rast;  // Jacobi diagonal (or NULL); the shadow residual
   double *r, *p, *Ap, *x, *sc;
   double b_norm, eps2;
};
class Resident;  // work space of a solve
// pub0, pub1: n values each that the solve does not use otherwise
std::shared_ptr< Resident > resident_work( double* pub0, double* pub1, hipStream_t s );
ResidentEnd resident_bicgstab( Resident& w, const ResidentBicgstab& a, Stop& S, hipStream_t s );

struct ResidentGmres
{
   EllSlots A;
   const double *d, *b;
   double *r, *V, *x;
   int64_t ld;
   bool classical;
   int passes, rmin, rmax, dmin, dmax;
   double normb;
};
// whole cycles from S, beta and r on; x, r, beta, S, cycles and beta_ratio as they end
ResidentEnd resident_gmres( Resident& w, const ResidentGmres& a, Stop& S, double& beta, double& beta_ratio, int& cycles,
                            int& m, hipStream_t s );

}  // namespace tnlmi
