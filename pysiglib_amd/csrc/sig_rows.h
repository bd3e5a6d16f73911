// Sweeps for many channels (more than 32), forward at degrees 3 .. 7, backward 3 .. 6.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sig_registry.h"

namespace sigamd {

// whether the backward / forward sweeps serve (element size, augmented dimension, degree)
bool rows_bwd_supported(size_t elem_bytes, uint64_t d, uint64_t degree);
bool rows_fwd_supported(size_t elem_bytes, uint64_t d, uint64_t degree);

// whether a launch for `batch` paths fits the grid limits (to be checked before anything is enqueued)
bool rows_fits(size_t elem_bytes, uint64_t d, uint64_t degree, uint64_t batch);

// whole-path sweeps (p.nseg must be 1, p.inc holds increments); p.d is the augmented dimension.  The backward ones add the
// increment gradient into p.dzinc in double precision whatever the element type (zeroed by the caller).
template <typename T>
hipError_t launch_rows_bwd(const BwdParams& p, int degree);
hipError_t launch_rows_fwd_f64(const FwdParams& p, int degree);

// single precision on the matrix units (sig_rows_mfma.hip)
bool rows_bwd_mfma_supported(uint64_t d);
hipError_t launch_rows_bwd_mfma(const BwdParams& p, int degree);
hipError_t launch_rows_fwd_mfma(const FwdParams& p, int degree);

}  // namespace sigamd
