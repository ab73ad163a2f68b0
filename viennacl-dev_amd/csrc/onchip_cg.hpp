// onchip_cg.hpp -- CG on a DIA operator in one launch: every vector of the solve lives in the
// registers and LDS of the CUs and only boundary rows and inner products travel between them.
#pragma once

#include <functional>
#include <optional>

#include "krylov_state.hpp"
#include "solver.hpp"

namespace vclhip {

// What a solve that stands right after cg_setup_kernel hands over: x = 0, r, p and A p of the first
// direction in memory, the scalars in *st.
template <typename T>
struct OnchipCg {
  uint32_t n;
  DiaDev<T> dia;
  bool jacobi;
  bool wide;  // the vector kernels' 16-byte packs (their partial sums' grouping)
  T* x;
  T* r;
  T* p;
  T* Ap;
  const T* d;
  KState* st;
  // The mixed solver: enqueues the FP64 correction, whose kernels return at once unless the iterations
  // ended asking for one.  The solve then goes on until the correction says that it is done.
  std::function<int()> after;
};

enum class Onchip { kNo, kDeferred, kDone, kAborted };

// For as long as it lives, a solve that runs by launches of its own: another thread's solve then leaves
// the one-launch mode out if that took more than a quarter of the device.  Not made for a solve that was
// left out itself (two of them would keep each other from it).
class LaunchedSolve {
 public:
  LaunchedSolve();
  ~LaunchedSolve();
  LaunchedSolve(const LaunchedSolve&) = delete;
  LaunchedSolve& operator=(const LaunchedSolve&) = delete;

 private:
  int dev_ = -1;
};

// Runs the iterations to the end if the system fits; where other threads' solves hold the CUs it waits for
// its turn.  kNo: it does not fit; kDeferred: another thread's LaunchedSolve needs the device.  Nothing was
// launched then and the solve stands as before.
// kAborted: the workgroups could not all run at once within the wait limit; the vectors and *st are
// then undefined and the caller starts over with the other modes.  kDone: x is written and *fin is the final state.
template <typename T>
int onchip_cg(const OnchipCg<T>& c, Workspace& ws, hipStream_t s, KState* fin, Onchip* outcome);

}  // namespace vclhip
