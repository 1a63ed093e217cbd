// Host-side launchers shared between translation units of libdgami.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dgami {

// Workspace slots (see workspace() in dgami_internal.hpp); one purpose each.
enum WorkspaceSlot {
  WS_GK = 0,         // two-point object in [nb][nb][nv][nk] layout
  WS_GR = 1,         // its momentum-space FFT
  WS_SIGMA_PART = 2, // per-frequency-chunk partial self-energies
  WS_LADDER = 3,     // ladder matrices / factors (large-n path)
  WS_LADDER_AUX = 4, // pivots, inverse pivots and interchange maps of WS_LADDER
  WS_DC = 5,         // double-counting kernel operands
  WS_PAIR = 6,       // Eliashberg matvec intermediates
  WS_MISC = 7,
  WS_MIXED = 8,      // mixed-precision factors (slots 8 and 9)
  WS_MIXED_VEC = 10, // refinement vectors
  WS_TRI = 11,       // inverse diagonal blocks of the triangular factors
  WS_TRI_VEC = 12,   // complex64 right-hand sides of the triangular sweeps
  WS_SELFCONS = 13,  // Hartree-Fock transforms
  WS_MU = 14,        // chemical-potential secant: per-k occupations and the secant state
  WS_LADDER_G32 = 15, // complex64 scaled vertex of the fused first block of the blocked LU
  // work issued on the library's extra stream k (1..MAX_EXTRA_STREAMS) uses its own slots:
  // slot + k * WS_STREAM_STRIDE
  WS_STREAM_STRIDE = 16,
  // slots of the shared-vertex ladder (beyond the extra streams' ranges; offset by the stride there too)
  WS_SHARED_VEC = 64,   // Krylov basis and iterates; then the matrices of the problems left to the LU
  WS_SHARED = 65,       // mean matrices, their inverses and the q-dependent part; then those LUs' pivots
  WS_SHARED_STATE = 66, // per-column Hessenberg factors and states, list of unconverged problems
};
constexpr int MAX_EXTRA_STREAMS = 3;

// The library's extra stream k of the current device (created on first use, default priority,
// not blocking the null stream): fork makes it wait for the work queued so far on `caller`,
// join makes `caller` wait for the work queued on it, so that a captured caller stream takes
// the forked work into its graph.
int extra_stream_fork(hipStream_t caller, int k, hipStream_t* out);
int extra_stream_join(hipStream_t caller, int k);

// The extra streams of one call: 1, 2, ... forked one after the other, and all joined by join() or,
// where the call ends in an error, by the destructor: what they still do on the caller's arrays is
// then ordered before whatever the caller puts on its stream next.
class ExtraStreamSet {
 public:
  explicit ExtraStreamSet(hipStream_t caller) : caller_(caller) {}
  ExtraStreamSet(const ExtraStreamSet&) = delete;
  ExtraStreamSet& operator=(const ExtraStreamSet&) = delete;
  ~ExtraStreamSet() { (void)join(); }
  int fork(hipStream_t* out) {
    const int rc = extra_stream_fork(caller_, count_ + 1, out);
    if (rc == 0) ++count_;
    return rc;
  }
  int join() {
    int rc = 0;
    for (; count_ > 0; --count_) {
      const int r = extra_stream_join(caller_, count_);
      if (rc == 0) rc = r;
    }
    return rc;
  }

 private:
  hipStream_t caller_;
  int count_ = 0;
};

int launch_fft_grid(const double2* in, double2* out, int64_t batch, int nx, int ny, int nz, int sign, double scale,
                    hipStream_t stream);
int launch_ref2_to_gk(const double2* in, double2* out, int nk, int nb, int nv_in, int v0, int nv, hipStream_t stream);

}  // namespace dgami
