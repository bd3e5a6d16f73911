// Forward sweeps of few channels to high degrees, double precision (sig_heads.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sigamd {

struct HeadsParams {
    const void* inc;        // increments [paths][L + 2][D], with a chunk of slack past the last row
    void* table;            // scratch: (paths * L + 1) * HeadsEntry::row elements, at a multiple of 64 bytes
    void* out;              // one row per (path, segment)
    int64_t paths, L;       // L < 2^30
    int64_t out_stride;
    int scalar;
    int nseg;
    int64_t lseg;
    int* nonfinite;
    hipStream_t stream;
};

struct HeadsEntry {
    int D, N;
    int row;                // elements of the table per step
    int blocks;             // blocks per (path, segment)
    int64_t most_blocks;    // of a launch, which numbers its threads with 32 bits
    int resident;           // blocks of a compute unit
    int step_ns, lone_ns;   // duration of a step: so many blocks on every compute unit; a block or less
    hipError_t (*launch)(const HeadsParams&);
};

// null: no such sweep
const HeadsEntry* heads_entry(uint64_t d, uint64_t degree);

}  // namespace sigamd
