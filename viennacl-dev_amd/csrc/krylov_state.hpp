// krylov_state.hpp -- the device-resident record of a Krylov solve (scalars, flags, counters) and the
// partial-sum slots that its kernels share.
#pragma once

#include "device.hpp"

namespace vclhip {

enum : uint32_t {
  kFlagDone = 1u,       // every kernel of the solve returns at once
  kFlagFinishing = 2u,  // BiCGStab: the final vector update is pending, everything else stops
  // Mixed-precision CG.  An iteration that asks for an FP64 correction sets Pause (the remaining
  // iterations of the chunk return at once) and clears NoPause (the correction kernels at the end of
  // the chunk run).  The correction clears TailIdle while it refreshes the FP32 state.
  kFlagPause = 4u,
  kFlagNoPause = 8u,
  kFlagTailIdle = 16u,
};

constexpr uint32_t kSlots = 8;  // partial-sum slots of kMaxPartials doubles each
struct KState {
  double alpha, beta, omega;
  double rr;        // CG: <r,r> or <r,M^-1 r>;  BiCGStab: <r,r0*>
  double nrs;       // CG: norm of the right-hand side squared;  BiCGStab: ||b||
  double res;       // BiCGStab residual-norm estimate
  double ap_r0;     // BiCGStab <Ap,r0*> of the current iteration
  double tol, abs_tol;
  double* history;  // device array or null
  uint32_t history_len;
  uint32_t iter, max_iters;
  uint32_t flags;
  uint32_t converged;
  uint32_t final_mode;        // BiCGStab: 0 full update, 1 converged (x only), 2 last iteration (full)
  uint32_t rr_from_partials;  // BiCGStab: <r,r0*> comes from the previous vector update's partials
  uint32_t breakdown;
  // mixed-precision CG
  double rr2;       // FP32 recursive <r,r>
  double rr_ref;    // <r,r> after the last FP64 correction (reliable update)
  float inner, initial;  // reference schedule: FP32 <r,r> and its value at the last restart
  float inner_tol;
  uint32_t updates;      // FP64 corrections done
  uint32_t iter2[2];     // CG, compact mode: iteration count, read from [k & 1] and written to the other
};

__host__ __device__ __forceinline__ double* slot_ptr(double* part, uint32_t slot) { return part + slot * kMaxPartials; }
__host__ __device__ __forceinline__ const double* slot_ptr(const double* part, uint32_t slot)
{
  return part + slot * kMaxPartials;
}

__device__ __forceinline__ void record_history(KState* st, uint32_t iter, double v)
{
  if (st->history && iter >= 1 && iter <= st->history_len) st->history[iter - 1] = v;
}

}  // namespace vclhip
